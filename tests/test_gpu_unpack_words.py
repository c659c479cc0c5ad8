"""GUPPI blocks of an odd number of bins: one load a sample, as with even ones."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch_cuda():
    import torch

    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    return torch


def best_us(torch, fn, n=9, calls=20):
    fn()
    ts = []
    for _ in range(n):
        a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        a.record()
        for _ in range(calls):
            fn()
        b.record()
        torch.cuda.synchronize()
        ts.append(a.elapsed_time(b) * 1e3 / calls)
    return min(ts)


def test_odd_bins_take_one_load_a_sample(torch_cuda):
    """Against the same samples one byte further on, which have to be read byte
    by byte: equal blocks, in 0.87 of the time (1.00 when both read bytes)."""
    from cpp_projects_amd import unpack

    torch = torch_cuda
    npol, nchan, nbin, nfft, nov = 4, 128, 65535, 4, 4096
    n = (nbin - 2 * nov) * nfft
    buf = torch.randint(-128, 128, (nchan * n * npol + 4,), dtype=torch.int8, device="cuda")
    buf[1:] = buf[:-1].clone()
    whole = buf[1: 1 + nchan * n * npol]
    aligned = whole.clone()
    out = [torch.empty(unpack.out_size(nbin, nfft, npol, nchan), dtype=torch.complex64, device="cuda") for _ in "ab"]

    def run(x, o):
        return best_us(torch, lambda: unpack.unpack_chunk_guppi(x, n, nov, nbin, nfft, npol, nchan, o))

    assert any(run(aligned, out[0]) < 0.95 * run(whole, out[1]) for _ in range(5))
    assert torch.equal(torch.view_as_real(out[0]), torch.view_as_real(out[1]))
