"""The work that a user of this framework has it do, as measurable cases.

Every case goes through the public Python entry points (the same C ABI calls
that the C++ classes make).  Sizes come from cpp_projects_amd/workloads.py,
the tests and bench.py, or are generic; the band is 1200-1600 MHz throughout.

Kinds:
* ``fdmt``      one transform: FDMTGPU.execute (f32 or u8 waterfall, running
                mean or RESTRICT init);
* ``search``    one beam: SingleBeamSearch.run and its sorted candidates,
                optionally the clustering leg;
* ``batch``     several ragged beams replayed as one graph, then each beam's
                sorted candidates;
* ``grad``      the differentiable path: transform, boxcar S/N map, and both
                adjoints;
* ``coherent``  raw 8-bit voltages to intensity waterfalls: unpack, forward
                FFT, one waterfall per coherent DM;
* ``chunk``     those waterfalls to clustered candidates: one search over the
                legacy CFdmt plan per coherent DM, then gather and clustering;
* ``dropin``    the reference's own call sequence step by step (statistics and
                normalisation, CFdmt of mask and data, S/N division, gathers,
                clustering).
"""
import ctypes
import math

import numpy as np
import torch

from cpp_projects_amd import unpack, workloads
from cpp_projects_amd.batch import BatchSearch, Beam
from cpp_projects_amd.coherent import CoherentChunk
from cpp_projects_amd.fdmt import SPS_INIT_MEAN, SPS_INIT_RESTRICT, CFdmtGpu, FDMTGPU
from cpp_projects_amd.search import (SPS_NORM_GLOBAL, SPS_NORM_PER_CHANNEL, SingleBeamSearch, boxcar_snr,
                                     boxcar_snr_adjoint, clusterization, fdmt_normalization,
                                     statistical_preprocessing)

F_MIN, F_MAX = workloads.F_MIN, workloads.F_MAX
DEV = "cuda"


def listed():
    c = workloads.COHERENT
    return [
        # the smallest call a caller makes (the smoke test's size): launch latency
        dict(name="fdmt_small_f32", kind="fdmt", nch=128, ns=2048, dt_max=127, dtype="f32", restrict=False),
        # an ordinary transform off every power of two, straight from an 8-bit detected waterfall
        dict(name="fdmt_ragged_u8", kind="fdmt", nch=1000, ns=50021, dt_max=799, dtype="u8", restrict=False),
        # the small end-to-end search with its clustering leg (the plain CPU workload's size and bins)
        dict(name="search_512_f32", kind="search", nch=512, ns=1 << 15, dt_max=511, dtype="f32", q=5, norm="global",
             tuned="", npulses=3, rfi=0.0, cap=1 << 20, cluster=32),
        # the benchmark's single 8-bit beam, with the schedule the package ships for it
        dict(name="search_4096_u8", kind="search", nch=4096, ns=1 << 18, dt_max=4095, dtype="u8", q=8, norm="global",
             tuned="single", npulses=8, rfi=0.0, cap=1 << 25, cluster=0),
        # a beam of odd length with per-channel normalisation and nothing tuned
        dict(name="search_ragged_f32", kind="search", nch=2048, ns=100003, dt_max=2047, dtype="f32", q=8,
             norm="channel", tuned="", npulses=3, rfi=0.0, cap=1 << 23, cluster=0),
        # the large share's channel count and interference on the longest rows that fit several times over
        dict(name="search_8192_f32", kind="search", nch=8192, ns=1 << 17, dt_max=8191, dtype="f32", q=9,
             norm="global", tuned="large", npulses=6, rfi=0.1, cap=1 << 25, cluster=0),
        # eight ragged beams of the batch workload's short half as one captured graph
        dict(name="batch_8_f32", kind="batch", beams="1024x44001,2048x19004,4096x16384,1024x65536,2048x30002,"
             "4096x27001,1024x20480,2048x61440", npulses=2, workers=4),
        # forward and backward of the differentiable path
        dict(name="grad_1024_f32", kind="grad", nch=1024, ns=1 << 16, dt_max=1023, w=16),
        # the coherent front-end's workload: GUPPI bytes to one waterfall per coherent DM
        dict(name="coherent_guppi", kind="coherent", layout="guppi", npol=c["npol"], nchan=c["nchan"],
             len_sft=c["len_sft"], nbin=c["nbin"], nfft=c["nfft"], nov=c["noverlap"], ndm=len(c["dms"])),
        # LOFAR's layout with sub-bands that are no power of two (the three-step path)
        dict(name="coherent_lofar", kind="coherent", layout="lofar", npol=4, nchan=20, len_sft=12, nbin=12288, nfft=9,
             nov=1536, ndm=3),
        # a chunk's waterfalls to its clustered candidates, as the chunk pipeline runs them
        dict(name="chunk_search", kind="chunk", rows=2048, cols=24576, imaxdt=32, ndm=8, wnd=4, npulses=4),
        # a reference caller that keeps its own step-by-step sequence
        dict(name="dropin_chain", kind="dropin", rows=1024, cols=20000, imaxdt=64, q=4, wnd=8, npulses=3),
    ]


def _logint(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _length(rng, lo, hi):
    """A row length, spread over its logarithm: odd, a multiple of 4, or a power of two."""
    n = _logint(rng, lo, hi)
    how = rng.randrange(3)
    if how == 0:
        return n | 1
    if how == 1:
        return max(4, n & ~3)
    return 1 << max(4, n.bit_length() - 1)


def draw(rng):
    kind = rng.choice(["fdmt", "fdmt", "search", "search", "search", "batch", "grad", "coherent", "chunk", "dropin"])
    if kind == "fdmt":
        nch = _logint(rng, 64, 4096)
        ns = _length(rng, 2048, min(1 << 18, (1 << 28) // nch))
        return dict(kind=kind, nch=nch, ns=ns, dt_max=min(ns // 2, _logint(rng, max(8, nch // 4), nch)),
                    dtype=rng.choice(["f32", "u8"]), restrict=rng.random() < 0.2)
    if kind == "search":
        nch = rng.choice([256, 512, 1024, 2048, 4096, _logint(rng, 200, 4096)])
        ns = _length(rng, 1 << 14, min(1 << 18, (1 << 29) // nch))
        return dict(kind=kind, nch=nch, ns=ns, dt_max=min(ns // 2, nch - 1), dtype=rng.choice(["u8", "f32"]),
                    q=rng.randrange(3, 10), norm=rng.choice(["global", "global", "channel"]),
                    tuned=rng.choice(["", "nch"]), npulses=rng.randrange(0, 4), rfi=rng.choice([0.0, 0.0, 0.1]),
                    cap=1 << 22, cluster=rng.choice([0, 0, 16, 32]))
    if kind == "batch":
        beams = [f"{rng.choice([1024, 2048, 4096])}x{_length(rng, 1 << 14, 1 << 15)}" for _ in range(rng.randrange(2, 9))]
        return dict(kind=kind, beams=",".join(beams), npulses=rng.randrange(0, 4), workers=rng.choice([1, 2, 4]))
    if kind == "grad":
        nch = _logint(rng, 64, 1024)
        ns = _length(rng, 2048, 1 << 16)
        return dict(kind=kind, nch=nch, ns=ns, dt_max=min(ns // 2, nch - 1), w=_logint(rng, 1, 64))
    if kind == "coherent":
        layout = rng.choice(["guppi", "lofar"])
        len_sft = rng.choice([8, 12, 16, 20, 32, 64])
        mbin = rng.choice([128, 256, 512, 1024, 2048, 4096, 384, 1000])
        if len_sft * mbin > 1 << 16:
            mbin = 512
        return dict(kind=kind, layout=layout, npol=rng.choice([2, 4]), nchan=rng.randrange(4, 33), len_sft=len_sft,
                    nbin=len_sft * mbin, nfft=rng.randrange(2, 17), nov=len_sft * (mbin // rng.choice([4, 8, 16])),
                    ndm=rng.randrange(1, 9))
    if kind == "chunk":
        imaxdt = rng.choice([8, 16, 32, 64])
        return dict(kind=kind, rows=imaxdt * rng.randrange(8, 65), cols=_length(rng, 4096, 24576), imaxdt=imaxdt,
                    ndm=rng.randrange(1, 9), wnd=4, npulses=rng.randrange(1, 5))
    return dict(kind="dropin", rows=_logint(rng, 256, 1024), cols=_length(rng, 4096, 20000),
                imaxdt=rng.choice([16, 32, 64]), q=rng.randrange(2, 6), wnd=rng.choice([4, 8, 16]),
                npulses=rng.randrange(0, 4))


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed) & 0x7FFFFFFF)
    return g


def _pulse_track(nch, sweep):
    """Delay in samples of every channel (row 0 the lowest frequency) of a pulse with this sweep."""
    f = F_MIN + (F_MAX - F_MIN) / nch * np.arange(nch, dtype=np.float64)
    return np.round((f ** -2 - F_MAX ** -2) / (F_MIN ** -2 - F_MAX ** -2) * sweep).astype(np.int64)


def _inject(x, rng, npulses, max_sweep, max_width, sigma):
    """Adds dispersed pulses of S/N 10 to 30 to a waterfall of this noise level, in place."""
    nch, ns = x.shape
    flat = x.view(-1)
    for _ in range(npulses):
        sweep = int(rng.integers(0, max_sweep + 1))
        width = float(rng.uniform(1.0, max_width))
        snr = float(rng.uniform(10.0, 30.0))
        t0 = int(rng.integers(0, max(1, ns - sweep)))
        half = int(math.ceil(3 * width))
        offs = torch.arange(-half, half + 1, device=DEV)
        t = t0 + torch.from_numpy(_pulse_track(nch, sweep)).to(DEV)[:, None] + offs[None, :]
        ok = (t >= 0) & (t < ns)
        idx = (torch.arange(nch, device=DEV)[:, None] * ns + t)[ok]
        amp = sigma * snr / math.sqrt(nch * max(width, 1.0)) * torch.exp(-0.5 * (offs.float() / width) ** 2)
        flat[idx] += amp[None, :].expand_as(t)[ok]
    return x


def _waterfall(nch, ns, dtype, seed, npulses, max_sweep, max_width, rfi=0.0):
    """Detected noise with a few pulses: f32 N(0, 1), or u8 clip(round(N(128, 16)))."""
    rng = np.random.default_rng(seed)
    x = torch.empty((nch, ns), dtype=torch.float32, device=DEV).normal_(generator=_gen(seed))
    if rfi > 0:
        bad = torch.from_numpy(np.sort(rng.choice(nch, int(round(rfi * nch)), replace=False))).to(DEV)
        x[bad] *= 5.0
    _inject(x, rng, npulses, max_sweep, max_width, 1.0)
    if dtype == "f32":
        return x
    return x.mul_(16.0).add_(128.0).round_().clamp_(0, 255).to(torch.uint8)


def _search_input(case, seed):
    return _waterfall(case["nch"], case["ns"], case["dtype"], seed, case["npulses"], case["dt_max"],
                      float(1 << min(case["q"], 6)), case["rfi"])


def _beams(case):
    return [tuple(int(v) for v in b.split("x")) for b in case["beams"].split(",")]


def _beam_input(case, seed, i, nch, ns):
    return _waterfall(nch, ns, "f32", seed * 64 + i, case["npulses"], nch - 1, 16.0)


def _chunk_waterfall(case, seed, i):
    """Intensities as the coherent front-end detects them (two polarisations: Gamma(2)), with pulses."""
    g = _gen(seed * 64 + i)
    x = torch.empty((case["rows"], case["cols"]), dtype=torch.float32, device=DEV).exponential_(generator=g)
    x += torch.empty_like(x).exponential_(generator=g)
    return _inject(x, np.random.default_rng(seed * 64 + i), case["npulses"], case["imaxdt"] - 1, 4.0, math.sqrt(2.0))


def _raw_size(case):
    return (case["nbin"] - 2 * case["nov"]) * case["nfft"]


def _raw(case, seed):
    n = case["nchan"] * _raw_size(case) * case["npol"]
    v = torch.empty(n, dtype=torch.float32, device=DEV)
    v.normal_(0.0, 20.0, generator=_gen(seed))
    return v.round_().clamp_(-127, 127).to(torch.int8)


def _dms(case):
    return [25.0 * i for i in range(case["ndm"])]


def _coherent_tsamp():
    return workloads.COHERENT["tsamp"]


# ---------------------------------------------------------------------------
# what a user's program has in hand
# ---------------------------------------------------------------------------
def _tuned_config(case):
    if case["tuned"] == "single":
        return workloads.SINGLE_BEAM_TUNED
    if case["tuned"] == "large":
        return workloads.LARGE_TUNED
    if case["tuned"] == "nch":
        return workloads.BATCH_TUNED.get(case["nch"])
    return None


def prepare(case, seed):
    kind = case["kind"]
    st = {"case": case}
    if kind == "fdmt":
        st["x"] = _waterfall(case["nch"], case["ns"], case["dtype"], seed, 2, case["dt_max"], 16.0)
        st["f"] = FDMTGPU(F_MIN, F_MAX, case["nch"], case["ns"], 1.0, case["dt_max"],
                          init_mode=SPS_INIT_RESTRICT if case["restrict"] else SPS_INIT_MEAN)
        st["out"] = torch.empty(st["f"].output_shape(), dtype=torch.float32, device=DEV)
    elif kind == "search":
        st["x"] = _search_input(case, seed)
        s = SingleBeamSearch(F_MIN, F_MAX, case["nch"], case["ns"], case["dt_max"], in_dtype=case["dtype"],
                             norm_mode=SPS_NORM_GLOBAL if case["norm"] == "global" else SPS_NORM_PER_CHANNEL,
                             box_q=case["q"], threshold=6.0, cand_capacity=case["cap"])
        t = _tuned_config(case)
        if t is not None:
            s.set_staged(t["staged"])
            s.set_group_shape(*t["shape"])
            s.set_schedule(t["schedule"])
        st["s"] = s
        st["dmt"] = torch.empty((s.ndt, case["ns"]), dtype=torch.float32, device=DEV)
        st["cands"] = torch.zeros((case["cap"], 4), dtype=torch.int32, device=DEV)
        st["count"] = torch.zeros(1, dtype=torch.int64, device=DEV)
        st["bins"] = torch.tensor(workloads.PLAIN_CPU["bins"], dtype=torch.int32, device=DEV)
        st["delegates"] = np.zeros((5, MAX_DELEGATES), np.int64)
    elif kind == "batch":
        beams = []
        for i, (nch, ns) in enumerate(_beams(case)):
            x = _beam_input(case, seed, i, nch, ns)
            cands = torch.zeros((1 << 21, 4), dtype=torch.int32, device=DEV)
            count = torch.zeros(1, dtype=torch.int64, device=DEV)
            dmt = torch.empty((nch, ns), dtype=torch.float32, device=DEV)
            beams.append(Beam(F_MIN, F_MAX, nch, ns, nch - 1, x, cands, count, dmt))
        b = BatchSearch(beams, in_dtype="f32", box_q=8, threshold=6.0, nworkers=case["workers"])
        for i, (nch, ns) in enumerate(_beams(case)):
            t = workloads.BATCH_TUNED[nch]
            b.set_staged(i, t["staged"])
            b.set_group_shape(i, *t["shape"])
            b.set_schedule(i, t["schedule"])
        st["b"] = b
    elif kind == "grad":
        nch, ns = case["nch"], case["ns"]
        st["x"] = _waterfall(nch, ns, "f32", seed, 2, case["dt_max"], 16.0)
        st["f"] = FDMTGPU(F_MIN, F_MAX, nch, ns, 1.0, case["dt_max"])
        shape = st["f"].output_shape()
        st["g"] = torch.empty(shape, device=DEV).normal_(generator=_gen(seed + 1))
        for k in ("y", "snr", "gy"):
            st[k] = torch.empty(shape, dtype=torch.float32, device=DEV)
        st["gx"] = torch.empty((nch, ns), dtype=torch.float32, device=DEV)
    elif kind == "coherent":
        st["raw"] = _raw(case, seed)
        st["cc"] = CoherentChunk(F_MIN, F_MAX, case["npol"], case["nchan"], case["len_sft"], case["nbin"],
                                 case["nfft"], case["nov"], _coherent_tsamp())
        st["blocks"] = torch.empty(unpack.out_size(case["nbin"], case["nfft"], case["npol"], case["nchan"]),
                                   dtype=torch.complex64, device=DEV)
        st["wf"] = [torch.empty((st["cc"].rows, st["cc"].cols), dtype=torch.float32, device=DEV)
                    for _ in range(case["ndm"])]
    elif kind == "chunk":
        rows, cols, L = case["rows"], case["cols"], case["imaxdt"]
        st["wf"] = [_chunk_waterfall(case, seed, i) for i in range(case["ndm"])]
        st["s"] = SingleBeamSearch(F_MIN, F_MAX, rows, cols, L - 1, in_dtype="f32", box_q=0, threshold=1e30,
                                   cand_capacity=0, cfdmt_imaxdt=L)
        st["img"] = torch.empty((case["ndm"] * L, cols), dtype=torch.float32, device=DEV)
        st["cands"] = torch.empty((1, 4), dtype=torch.int32, device=DEV)
        st["count"] = torch.zeros(1, dtype=torch.int64, device=DEV)
        st["thr"] = torch.tensor([6.0], dtype=torch.float32, device=DEV)
        st["bins"] = torch.tensor([2, 1, 2], dtype=torch.int32, device=DEV)
        st.update(_records())
    elif kind == "dropin":
        rows, cols, L = case["rows"], case["cols"], case["imaxdt"]
        st["raw"] = _chunk_waterfall(case, seed, 0)
        st["x"] = torch.empty_like(st["raw"])
        st["mask"] = torch.empty_like(st["raw"])
        st["buff"] = torch.empty(2 * rows + 4, dtype=torch.float32, device=DEV)
        st["f"] = CFdmtGpu(F_MIN, F_MAX, rows, cols, L)
        for k in ("y", "ynorm", "snr"):
            st[k] = torch.empty((L, cols), dtype=torch.float32, device=DEV)
        st["thr"] = torch.tensor([6.0], dtype=torch.float32, device=DEV)
        st["bins"] = torch.tensor([2, 1, 2], dtype=torch.int32, device=DEV)
        st.update(_records())
    return st


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def run(st):
    case = st["case"]
    kind = case["kind"]
    if kind == "fdmt":
        st["f"].execute(st["x"], st["x"].numel(), st["out"], st["out"].numel())
        return st["out"]
    if kind == "search":
        s = st["s"]
        s.run(st["x"], st["dmt"], st["cands"], st["count"])
        _, n = s.candidates(st["dmt"], st["cands"], st["count"])
        out = {"image": st["dmt"], "candidates": st["cands"], "n": n}
        if case["cluster"]:
            dele, sizes, out["gathered"] = s.cluster(st["dmt"], case["cluster"], st["bins"])
            k = min(len(dele), MAX_DELEGATES)
            st["delegates"][:4, :k] = np.ascontiguousarray(dele[:k]).view(np.int32).reshape(k, 4).T
            st["delegates"][4, :k] = sizes[:k]
            out["delegates"], out["groups"] = st["delegates"], len(dele)
        return out
    if kind == "batch":
        b = st["b"]
        b.launch()
        counts = [b.sort_candidates(i) for i in range(len(b.beams))]
        return {"images": [beam.d_dmt for beam in b.beams], "candidates": [beam.d_cands for beam in b.beams],
                "counts": counts}
    if kind == "grad":
        f, w = st["f"], case["w"]
        rows, cols = f.output_shape()
        f.execute(st["x"], st["x"].numel(), st["y"], st["y"].numel())
        boxcar_snr(st["y"], rows, cols, w, st["snr"])
        boxcar_snr_adjoint(st["g"], rows, cols, w, st["gy"])
        f.adjoint(st["gy"], st["gx"])
        return {"y": st["y"], "snr": st["snr"], "gy": st["gy"], "gx": st["gx"]}
    if kind == "coherent":
        up = unpack.unpack_chunk_guppi if case["layout"] == "guppi" else unpack.unpack_chunk_lofar
        up(st["raw"], _raw_size(case), case["nov"], case["nbin"], case["nfft"], case["npol"], case["nchan"],
           st["blocks"])
        st["cc"].forward(st["blocks"])
        for dm, wf in zip(_dms(case), st["wf"]):
            st["cc"].waterfall(st["blocks"], dm, wf)
        return st["wf"]
    if kind == "chunk":
        L = case["imaxdt"]
        for i, wf in enumerate(st["wf"]):
            st["s"].run(wf, st["img"][i * L:(i + 1) * L], st["cands"], st["count"])
        return {"image": st["img"], **_gather_and_cluster(st, st["img"])}
    rows, cols, L = case["rows"], case["cols"], case["imaxdt"]
    st["x"].copy_(st["raw"])
    statistical_preprocessing.calc_fdmt_inputs(st["x"], rows, cols, st["buff"], st["mask"])
    st["f"].process_image(st["mask"], st["ynorm"], False)
    st["f"].process_image(st["x"], st["y"], False)
    fdmt_normalization(st["y"], st["ynorm"], L * cols, st["snr"])
    pow2, npow2 = clusterization.gather_candidates_in_dynamicalArray(st["snr"], L, cols, st["thr"], case["q"])
    _keep(st["pow2"], pow2)
    return {"x": st["x"], "mask": st["mask"], "y": st["y"], "ynorm": st["ynorm"], "snr": st["snr"],
            "pow2": st["pow2"], "npow2": npow2, **_gather_and_cluster(st, st["snr"])}


# what a program keeps of results whose number it does not know beforehand: buffers of its own, zeros past the end
MAX_CANDIDATES, MAX_DELEGATES = 1 << 20, 1 << 16


def _records():
    r = {k: torch.zeros((MAX_CANDIDATES, 4), dtype=torch.int32, device=DEV) for k in ("pow2", "heap")}
    r["dele"] = torch.zeros(MAX_CANDIDATES, dtype=torch.int32, device=DEV)
    r["sizes"] = torch.zeros(MAX_CANDIDATES, dtype=torch.int64, device=DEV)
    return r


def _keep(buf, t):
    n = min(len(t), len(buf))
    buf[:n].copy_(t[:n])


def _gather_and_cluster(st, img):
    ok, cands, n = clusterization.gather_candidates_in_heap_with_plan(img, img.shape[0], img.shape[1], st["thr"],
                                                                      st["case"]["wnd"])
    groups = 0
    if ok:
        dele, sizes = clusterization.cluster(cands, n, st["bins"])
        groups = len(dele)
        _keep(st["heap"], cands)
        _keep(st["dele"], dele)
        _keep(st["sizes"], sizes)
    return {"candidates": st["heap"], "n": n, "delegates": st["dele"], "group_sizes": st["sizes"], "groups": groups}


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def _search_work(nch, ns, ndt, elem, q):
    merges = math.ceil(math.log2(max(nch, 2)))
    return elem * nch * ns + 4.0 * ndt * ns, float(ns) * ndt * (merges + q + 1)


def work(case):
    kind = case["kind"]
    if kind == "fdmt":
        nch, ns, ndt = case["nch"], case["ns"], case["dt_max"] + 1
        b, f = _search_work(nch, ns, ndt, 1 if case["dtype"] == "u8" else 4, 0)
    elif kind == "search":
        b, f = _search_work(case["nch"], case["ns"], case["dt_max"] + 1, 1 if case["dtype"] == "u8" else 4, case["q"])
    elif kind == "batch":
        parts = [_search_work(nch, ns, nch, 4, 8) for nch, ns in _beams(case)]
        b, f = sum(p[0] for p in parts), sum(p[1] for p in parts)
    elif kind == "grad":
        nch, ns, ndt = case["nch"], case["ns"], case["dt_max"] + 1
        b1, f1 = _search_work(nch, ns, ndt, 4, 0)
        # transform, its S/N map, the upstream gradient, both adjoints' outputs
        b, f = b1 + 4.0 * ns * (3 * ndt + nch), 2 * f1 + 2.0 * ns * ndt
    elif kind == "coherent":
        spectra = case["nfft"] * case["nchan"] * (case["npol"] // 2) * case["nbin"]
        msamp = case["nfft"] * (case["nbin"] // case["len_sft"] - 2 * (case["nov"] // case["len_sft"]))
        wf = case["nchan"] * case["len_sft"] * msamp
        fwd = 5.0 * spectra * math.log2(case["nbin"])
        inv = 5.0 * spectra * math.log2(case["nbin"] / case["len_sft"])
        b = case["nchan"] * _raw_size(case) * case["npol"] + 4.0 * wf * case["ndm"]
        f = fwd + case["ndm"] * (inv + 9.0 * spectra)
    else:
        n = case["rows"] * case["cols"]
        ndm = case.get("ndm", 1)
        img = case["imaxdt"] * case["cols"]
        merges = math.ceil(math.log2(case["rows"]))
        b = ndm * (4.0 * n + 4.0 * img)
        f = ndm * (8.0 * n + 2.0 * merges * img)
        if kind == "dropin":
            b += 8.0 * n + 8.0 * img
    return {"bytes": float(b), "flops": float(f)}


# ---------------------------------------------------------------------------
# the same outputs in 64 bits, in plain torch and numpy
# ---------------------------------------------------------------------------
_powf = ctypes.CDLL("libm.so.6").powf
_powf.restype = ctypes.c_float
_powf.argtypes = [ctypes.c_float, ctypes.c_float]
_f32 = np.float32


def _inv2(f):
    return _f32(_powf(float(f), -2.0))


def _ratio(a0, a1, b0, b1):
    return (_inv2(a0) - _inv2(a1)) / (_inv2(b0) - _inv2(b1))


def _scaled(r, dt):
    return np.floor((np.asarray(dt, _f32) * r).astype(np.float64) + 0.5).astype(np.int64)


def _nearest(g, v):
    """Index of the entry of the sorted g nearest to each v, the larger entry on ties."""
    i = np.searchsorted(g, v)
    last = len(g) - 1
    j = np.minimum(i, last)
    left = (i <= last) & (j > 0) & (v - g[np.maximum(j - 1, 0)] < g[j] - v)
    return np.where(left, j - 1, j)


def _plan(nch, dt_max):
    """(init dts per channel, per iteration (tail, head, offset) rows): the integer tables of the transform."""
    fmin, fmax = _f32(F_MIN), _f32(F_MAX)
    df = (fmax - fmin) / _f32(nch)
    half = df / _f32(2)

    def grid(fs, fe):
        return np.arange(0, int(_scaled(_ratio(fs, fe, fmin, fmax), dt_max)) + 1, dtype=np.int64)

    grids = []
    for c in range(nch):
        fs = df * _f32(c) + fmin
        grids.append(grid(fs, fs + df))
    init, iters = grids, []
    top_grid, top, bot = grids[-1], df, df
    while len(grids) > 1:
        odd = len(grids) % 2 == 1
        ncur = len(grids) // 2 + odd
        row = np.concatenate([[0], np.cumsum([len(g) for g in grids])])
        top = top if odd else top + bot
        bot = bot * _f32(2)
        new, tail, head, off = [], [], [], []
        for s in range(ncur):
            fs = bot * _f32(s) + fmin
            if s == ncur - 1 and odd:
                g = top_grid
                new.append(g)
                tail.append(row[2 * s] + _nearest(grids[2 * s], g))
                head.append(np.full(len(g), -1))
                off.append(np.zeros(len(g), np.int64))
                continue
            fe = fs + (top if s == ncur - 1 else bot)
            fm = fs + bot / _f32(2)
            g = grid(fs, fe)
            if s == ncur - 1:
                top_grid = g
            lo, hi = _scaled(_ratio(fs, fm - half, fs, fe), g), _scaled(_ratio(fs, fm + half, fs, fe), g)
            new.append(g)
            tail.append(row[2 * s] + _nearest(grids[2 * s], lo))
            head.append(row[2 * s + 1] + _nearest(grids[2 * s + 1], g - hi))
            off.append(hi)
        iters.append((np.concatenate(tail), np.concatenate(head), np.concatenate(off)))
        grids = new
    return init, iters


def _cplan(nch, imaxdt):
    """The legacy plan's tables, laid out as _plan's."""
    fmin, fmax = _f32(F_MIN), _f32(F_MAX)

    def delta(f0, f1):
        return int(math.ceil((1.0 / float(f0 * f0) - 1.0 / float(f1 * f1))
                             / (1.0 / float(fmin * fmin) - 1.0 / float(fmax * fmax)) * (imaxdt - 1.0)))

    def delay(a, b):
        return _f32(1.0 / float(a * a) - 1.0 / float(b * b))

    d = delta(fmin, fmin + (fmax - fmin) / _f32(nch))
    rows = [d + 1] * nch
    freq = [fmin + _f32(i) * (fmax - fmin) / _f32(nch) for i in range(nch)] + [fmax]
    iters = []
    while len(rows) > 1:
        q = len(rows)
        cs = np.concatenate([[0], np.cumsum(rows)])
        nr, nf, tail, head, off = [], [], [], [], []
        for i in range(q // 2):
            a, b, c = freq[2 * i], freq[2 * i + 1], freq[2 * i + 2]
            n = delta(a, c) + 1
            j = np.arange(n, dtype=_f32)
            j0 = (delay(a, b) / delay(a, c) * j).astype(np.int64)
            j1 = (delay(b, c) / delay(a, c) * j).astype(np.int64)
            tail.append(cs[2 * i] + j0)
            head.append(cs[2 * i + 1] + j1)
            off.append(j0)
            nr.append(n)
            nf.append(a)
        if q % 2:
            n = rows[-1]
            tail.append(cs[q - 1] + np.arange(n))
            head.append(np.full(n, -1))
            off.append(np.zeros(n, np.int64))
            nr.append(n)
            nf.append(freq[q - 1])
        iters.append((np.concatenate(tail), np.concatenate(head), np.concatenate(off)))
        rows, freq = nr, nf + [fmax]
    return [np.arange(d + 1, dtype=np.int64)] * nch, iters


def _live(plan, out_rows):
    """Per state, the rows some delivered output depends on."""
    init, iters = plan
    flags = [None] * (len(iters) + 1)
    n = sum(len(g) for g in init) if not iters else len(iters[-1][0])
    flags[-1] = np.arange(n) < out_rows
    for i in range(len(iters) - 1, -1, -1):
        tail, head, _ = iters[i]
        prev = np.zeros(len(iters[i - 1][0]) if i else sum(len(g) for g in init), bool)
        prev[tail[flags[i + 1]]] = True
        h = head[flags[i + 1]]
        prev[h[h >= 0]] = True
        flags[i] = prev
    return flags


def _init64(x, init, mode):
    n = x.shape[1]
    s = torch.zeros((sum(len(g) for g in init), n), dtype=torch.float64, device=x.device)
    r = 0
    for c, g in enumerate(init):
        prev = None
        for k, d in enumerate(g):
            d = int(d)
            row = s[r]
            if d >= n:
                pass
            elif mode == "restrict" and k > 0:
                dp = int(g[k - 1])
                row[d:] = prev[d:] * ((dp + 1.0) + x[c, :n - d]) / (d + 1.0)
            elif k == 0:
                for j in range(d + 1):
                    row[d:] += x[c, j:n - d + j]
                row[d:] /= d + 1.0
            else:
                dp = int(g[k - 1])
                acc = prev[d:] * (dp + 1.0)
                for j in range(d - dp):
                    acc += x[c, j:n - d + j]
                row[d:] = acc / (d + 1.0)
            prev = row
            r += 1
    return s


def _fdmt64(x, plan, out_rows, mode="mean"):
    init, iters = plan
    flags = _live(plan, out_rows)
    s = _init64(x, init, mode)
    n = x.shape[1]
    for i, (tail, head, off) in enumerate(iters):
        new = torch.empty((len(tail), n), dtype=torch.float64, device=x.device)
        for r in np.nonzero(flags[i + 1])[0]:
            new[r].copy_(s[int(tail[r])])
            h, o = int(head[r]), int(off[r])
            if h >= 0 and o < n:
                new[r, o:] += s[h, :n - o]
        s = new
    return s[:out_rows]


def _fdmt64_adjoint(g, plan):
    init, iters = plan
    n = g.shape[1]
    for i in range(len(iters) - 1, -1, -1):
        tail, head, off = iters[i]
        prev = len(iters[i - 1][0]) if i else sum(len(v) for v in init)
        p = torch.zeros((prev, n), dtype=torch.float64, device=g.device)
        for r in range(len(tail)):
            p[int(tail[r])] += g[r]
            h, o = int(head[r]), int(off[r])
            if h >= 0 and o < n:
                p[h, :n - o] += g[r, o:]
        g = p
    gx = torch.zeros((len(init), n), dtype=torch.float64, device=g.device)
    r = 0
    for c, gr in enumerate(init):
        for d in gr:
            d = int(d)
            if d < n:  # sample i enters the means at t = i .. i + d (t >= d)
                v = g[r, d:] / (d + 1.0)
                for j in range(d + 1):
                    gx[c, j:n - d + j] += v
            r += 1
    return gx


def _stats64(x, mode):
    """(mean, std, keep) per row, the reference's cleaning rule (rows over 4 sigma from the mean variance go)."""
    m = x.mean(1)
    v = (x * x).mean(1) - m * m
    vm, vs = v.mean(), torch.sqrt((v * v).mean() - v.mean() ** 2)
    drop = (v - vm).abs() > 4.0 * vs
    if mode == "channel":
        drop |= ~(v > 0)
        return m, torch.sqrt(v), ~drop
    mean = m.mean()
    sd = torch.sqrt((v + m * m).mean() - mean * mean)
    return mean.expand_as(m), sd.expand_as(m), ~drop


def _normalise64(x, mode):
    m, s, keep = _stats64(x, mode)
    xn = x.sub_(m[:, None]).div_(s[:, None])
    xn[~keep] = 0.0
    return xn, keep


def _extent(plan):
    init, iters = plan
    e = np.concatenate(init)
    for tail, head, off in iters:
        e = np.maximum(e[tail], np.where(head >= 0, e[np.maximum(head, 0)] + off, 0))
    return int(e.max())


def _snr64(x, plan, out_rows, mode):
    """S/N image of a raw waterfall: normalise, transform, divide by sqrt(transform of the keep mask + 1e-8)."""
    n = x.shape[1]
    xn, keep = _normalise64(x.double(), mode)
    L = min(n, _extent(plan) + 1)
    nrm = _fdmt64(keep.double()[:, None].expand(-1, L).contiguous(), plan, out_rows)
    img = _fdmt64(xn, plan, out_rows)
    img[:, :L] /= torch.sqrt(nrm + 1e-8)
    img[:, L:] /= torch.sqrt(nrm[:, -1:] + 1e-8)
    return img


def _boxcar64(img, w):
    n = img.shape[1]
    out = torch.zeros_like(img)
    if w <= n:
        cs = torch.nn.functional.pad(torch.cumsum(img, 1), (1, 0))
        out[:, :n - w + 1] = (cs[:, w:] - cs[:, :-w]) / math.sqrt(w)
    return out


def _boxcar64_adjoint(g, w):
    n = g.shape[1]
    if w > n:
        return torch.zeros_like(g)
    k = g.clone()
    k[:, n - w + 1:] = 0.0
    cs = torch.nn.functional.pad(torch.cumsum(k, 1), (w, 0))
    return (cs[:, w:] - cs[:, :-w]) / math.sqrt(w)


def _unpack64(case, raw):
    nbin, nfft, nov, npol, nchan = case["nbin"], case["nfft"], case["nov"], case["npol"], case["nchan"]
    nsamp = _raw_size(case)
    if case["layout"] == "guppi":
        v = raw.view(nchan, nsamp, npol).permute(2, 0, 1)  # [component][chan][samp]
    else:
        v = raw.view(npol, nsamp, nchan).permute(0, 2, 1)
    v = v.double()
    v = torch.complex(v[0::2].contiguous(), v[1::2].contiguous())
    step = nbin - 2 * nov
    v = torch.nn.functional.pad(v, (nov, nov + nbin))
    return torch.stack([v[..., f * step:f * step + nbin] for f in range(nfft)], 1)  # [pol][fft][chan][bin]


def _waterfall64(case, spec, dm):
    nchan, ls, nbin = case["nchan"], case["len_sft"], case["nbin"]
    mbin = nbin // ls
    bw = float(_f32(F_MAX) - _f32(F_MIN))
    bw_sub, bw_chan = bw / nchan, bw / nchan / ls
    dev = spec.device
    bf = -0.5 * bw_chan + (torch.arange(mbin, dtype=torch.float64, device=dev) + 0.5) * bw_chan / mbin
    taper = 1.0 / torch.sqrt(1.0 + (bf / (0.47 * bw_chan)) ** 80.0)
    c = torch.arange(nchan, dtype=torch.float64, device=dev)[:, None, None]
    k = torch.arange(ls, dtype=torch.float64, device=dev)[None, :, None]
    f0 = (F_MIN + bw_sub * (0.5 + c) + bw_chan * (k - ls / 2.0 + 0.5)).float().double()  # the definition's float centre
    r = bf / f0
    delay = dm * r * r / (f0 + bf) * 4.148808e9
    ph = -torch.frac(delay) * 2.0 * math.pi
    fac = torch.polar(taper / nbin * torch.ones_like(ph), ph).reshape(nchan, nbin)
    x = spec * torch.roll(fac, nbin // 2, 1)
    x = torch.fft.ifft(x.reshape(*x.shape[:-1], ls, mbin), norm="forward").reshape(x.shape)
    p = (x.real ** 2 + x.imag ** 2).sum(0) / nbin / nbin  # [fft][chan][bin]
    del x
    p = torch.roll(p, nbin // 2, -1).reshape(case["nfft"], nchan, ls, mbin)
    ov = case["nov"] // ls
    p = p[..., ov:mbin - ov]
    wf = p.flip(1, 2).permute(1, 2, 0, 3).reshape(nchan * ls, -1)
    rows, msamp = wf.shape
    foff = (float(_f32(F_MAX)) - float(_f32(F_MIN))) / rows
    tsamp = float(_f32(ls) * _f32(_coherent_tsamp()))
    out = torch.empty_like(wf)
    for row in range(rows):
        fr = (rows - 1 - row) * foff + F_MIN
        d = 4.148808e3 * dm * (1.0 / (F_MIN * F_MIN) - 1.0 / (fr * fr))
        out[row] = torch.roll(wf[row], int(math.floor(d / tsamp + 0.5)) % msamp)
    return out


# whole numbers have no value in 64 bits of their own
_NO_CLUSTERS = dict.fromkeys(("candidates", "n", "delegates", "group_sizes", "groups"))


def exact(case, seed):
    kind = case["kind"]
    if kind == "fdmt":
        x = _waterfall(case["nch"], case["ns"], case["dtype"], seed, 2, case["dt_max"], 16.0)
        return _fdmt64(x.double(), _plan(case["nch"], case["dt_max"]), case["dt_max"] + 1,
                       "restrict" if case["restrict"] else "mean")
    if kind == "search":
        img = _snr64(_search_input(case, seed), _plan(case["nch"], case["dt_max"]), case["dt_max"] + 1, case["norm"])
        out = {"image": img, "candidates": None, "n": None}
        if case["cluster"]:
            out.update(gathered=None, delegates=None, groups=None)
        return out
    if kind == "batch":
        images = [_snr64(_beam_input(case, seed, i, nch, ns), _plan(nch, nch - 1), nch, "global")
                  for i, (nch, ns) in enumerate(_beams(case))]
        none = [None] * len(images)
        return {"images": images, "candidates": none, "counts": none}
    if kind == "grad":
        x = _waterfall(case["nch"], case["ns"], "f32", seed, 2, case["dt_max"], 16.0)
        plan = _plan(case["nch"], case["dt_max"])
        ndt = case["dt_max"] + 1
        g = torch.empty((ndt, case["ns"]), device=DEV).normal_(generator=_gen(seed + 1)).double()
        y = _fdmt64(x.double(), plan, ndt)
        gy = _boxcar64_adjoint(g, case["w"])
        return {"y": y, "snr": _boxcar64(y, case["w"]), "gy": gy, "gx": _fdmt64_adjoint(gy, plan)}
    if kind == "coherent":
        spec = torch.fft.fft(_unpack64(case, _raw(case, seed)))
        return [_waterfall64(case, spec, dm) for dm in _dms(case)]
    if kind == "chunk":
        plan = _cplan(case["rows"], case["imaxdt"])
        img = torch.cat([_snr64(_chunk_waterfall(case, seed, i), plan, case["imaxdt"], "global")
                         for i in range(case["ndm"])])
        return {"image": img, **_NO_CLUSTERS}
    plan = _cplan(case["rows"], case["imaxdt"])
    xn, keep = _normalise64(_chunk_waterfall(case, seed, 0).double(), "global")
    mask = keep.double()[:, None].expand(-1, case["cols"]).contiguous()
    y, ynorm = _fdmt64(xn, plan, case["imaxdt"]), _fdmt64(mask, plan, case["imaxdt"])
    return {"x": xn, "mask": mask, "y": y, "ynorm": ynorm, "snr": y / torch.sqrt(ynorm + 1e-8), "pow2": None,
            "npow2": None, **_NO_CLUSTERS}
