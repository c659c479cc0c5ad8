// launch_check.cpp -- a launch folded by rows_per_launch stays within the 32-bit
// thread count of a dispatch and wastes less than one row of it.
#include <cstdio>
#include <initializer_list>

#include "../../cpp_projects_amd/csrc/launch_limits.hpp"

int main() {
    const int64_t blocks[] = {1, 7, 8, 64, 1024, 16383, 16777215, 16777216};
    for (int64_t b : blocks)
        for (int64_t threads : {64, 256, 1024}) {
            const int64_t n = sps::rows_per_launch(b, threads);
            if (n * b * threads > 0xffffffffLL || (n + 1) * b * threads <= 0xffffffffLL) {
                std::printf("FAILED: %lld blocks of %lld threads, %lld rows\n", (long long)b, (long long)threads, (long long)n);
                return 1;
            }
        }
    // 8192 channels x 2^20 samples: 1024 blocks of 256 threads a row, some 24000 rows of state 0
    if (sps::rows_per_launch(1024, 256) != 16383) return 1;
    std::printf("launch check ok\n");
    return 0;
}
