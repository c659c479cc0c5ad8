"""Autotuner over what callers can set on the merge passes (staging mode, group
shape, schedule).  The launches take up to six iterations each whatever is set,
so there is nothing to choose: the interface stays for callers that store its
choice, and returns what the handle has."""

DEFAULT_SHAPES = ((6144, 16, 16), (5120, 16, 16), (7168, 16, 16), (6144, 16, 32), (6144, 16, 64), (7168, 16, 32),
                  (5120, 16, 32), (6144, 32, 32), (8192, 32, 16), (9216, 32, 16), (8192, 64, 16))


def candidate_schedules(n, max_depth=3):
    c = set()
    for d in range(1, max_depth + 1):
        s = [d] * (n // d)
        r = n - sum(s)
        if r:
            c.add(tuple(s + [r]))
            c.add(tuple([r] + s))
        else:
            c.add(tuple(s))
    for big in range(2, max_depth + 1):
        for kb in range(0, n // big + 1):
            rem = n - big * kb
            for small in range(1, big):
                if rem % small == 0:
                    c.add(tuple([big] * kb + [small] * (rem // small)))
                    c.add(tuple([small] * (rem // small) + [big] * kb))
    # passes of depth 1 only pay off at the ends of a schedule: keep at most two
    return sorted(s for s in c if sum(s) == n and all(1 <= d <= max_depth for d in s) and s.count(1) <= 2)


def tune_search(search, run_once, reps=2, log=None, modes=(0, 1, 3, 4), shapes=DEFAULT_SHAPES):
    """Times `search` (a SingleBeamSearch) as it is set, run_once() issuing one
    search step, and returns ({"staged": mode, "shape": None, "schedule": list},
    [(ms, mode, None, schedule)]): the schedule that it has and the least mode
    that takes it.  modes and shapes name candidates that no longer differ, so
    none of them is tried and the handle keeps its settings."""
    sched = [int(d) for d in search.get_schedule()]
    mode = 1 if max(sched, default=0) > 3 else 0
    search.enable_timing(True)
    try:
        run_once()  # builds the pass tables
        tot = 0.0
        for _ in range(reps):
            run_once()
            tot += sum(search.stage_times_ms())
    finally:
        search.enable_timing(False)
    ms = tot / max(reps, 1)
    if log:
        log(f"[tune] {sched}: {ms:.3f} ms")
    return {"staged": mode, "shape": None, "schedule": sched}, [(ms, mode, None, tuple(sched))]
