"""The work a program has this library do, as cases to measure.

Pairs come from the library's seeded generator (gasal2_amd.synth_batch): 150 x
250 bp short reads, the full-feature batch (100-300 bp queries, flanked and
diverged targets, N bases, half the queries reverse-complemented), uneven
lengths (50-5000 bp) and seed extensions (100-250 bp).  A case goes through one
of the library's entries:

  resident  gasal2_run_resident on a storage whose batch was uploaded once; the
            outputs are the storage's device arrays
  device    gasal2_aln_noalloc on the caller's device arrays and stream
  call      gasal_aln_async on a filled host batch, polled until the results
            are on the host: what a GASAL2 program does per batch
  stream    the multi-storage driver (gasal2_stream_align) over a set of pairs
            in host memory

Every state owns its storage, so states alternate as the storages of a program
with several HIP streams do.
"""
import ctypes as C
import math

import numpy as np
import torch

import gasal2_amd as g

SHORT, FULL, UNEVEN, SEED = 1, 2, 3, 4          # workloads of the generator
BASES = {SHORT: (150, 250), FULL: (200, 250), UNEVEN: (510, 510), SEED: (175, 175)}   # mean bases per pair
CIGAR = {SHORT: 256, FULL: 256, UNEVEN: 2048}   # bytes that hold a pair's CIGAR
CELLS = {SHORT: 37.5e3, FULL: 53.3e3, UNEVEN: 424e3, SEED: 30.6e3}                    # mean Lq * Lt per pair

MODES = {
    "local": (g.LOCAL, g.WITHOUT_START),
    "local_start": (g.LOCAL, g.WITH_START),
    "local_tb": (g.LOCAL, g.WITH_TB),
    "global": (g.GLOBAL, g.WITHOUT_START),
    "global_tb": (g.GLOBAL, g.WITH_TB),
    "semi": (g.SEMI_GLOBAL, g.WITHOUT_START),
    "semi_start": (g.SEMI_GLOBAL, g.WITH_START),
    "banded": (g.BANDED, g.WITHOUT_START),
    "ksw": (g.KSW, g.WITHOUT_START),
}


def _case(name, entry, mode, pairs, workload, **kw):
    c = {"entry": entry, "mode": mode, "pairs": pairs, "workload": workload, "second": False, "packed": False,
         "head": "TARGET", "tail": "TARGET", "k_band": 0, "w": -1, "zdrop": 0, "scores": "1,4,6,1"}
    c.update(kw)
    return dict(c, name=name) if name else c


def listed():
    return [
        # a pipeline stage inside a larger GPU program: a few thousand reads
        # already on the device, captured or called in a loop
        _case("device_local_start_2k", "device", "local_start", 2000, SHORT),
        # an interactive caller: one small batch, host to host
        _case("call_local_tb_64", "call", "local_tb", 64, FULL),
        # score-only filtering of short reads, one moderate batch
        _case("short_local_10k", "resident", "local", 10_000, SHORT),
        # every feature at once: ends, starts, second best, CIGAR
        _case("full_local_tb_second", "resident", "local_tb", 300_000, FULL, second=True),
        # whole-sequence comparison of mixed lengths up to 5 kbp, scores
        _case("uneven_global", "resident", "global", 20_000, UNEVEN),
        # whole-sequence alignments (CIGAR), an odd count
        _case("full_global_tb", "resident", "global_tb", 100_001, FULL),
        # reads placed inside their targets, packed host input
        _case("full_semi_start", "resident", "semi_start", 300_000, FULL, packed=True),
        # tile-banded extension
        _case("seed_banded", "resident", "banded", 500_000, SEED, k_band=32),
        # seed extension, the reference's KSW form
        _case("seed_ksw", "resident", "ksw", 500_000, SEED),
        # mixed lengths up to 5 kbp, score and ends
        _case("uneven_local", "resident", "local", 100_000, UNEVEN),
        # mixed lengths with tracebacks: the largest
        _case("uneven_local_tb", "resident", "local_tb", 50_000, UNEVEN),
        # production throughput: host pairs in, results and CIGARs out
        _case("stream_local_tb_second", "stream", "local_tb", 200_000, FULL, second=True),
    ]


def draw(rng):
    entry = rng.choice(["resident"] * 6 + ["device", "call"])
    if entry == "device":
        mode = rng.choice(["local", "local_start", "global", "semi", "semi_start"])
    elif entry == "call":
        mode = rng.choice(["local", "local_tb", "global_tb", "semi_start"])
    else:
        mode = rng.choice(sorted(MODES))
    if mode in ("banded", "ksw"):
        workload = SEED
    elif entry == "resident":
        workload = rng.choice([SHORT, FULL, UNEVEN])
    else:
        workload = rng.choice([SHORT, FULL])
    cells = {"resident": (1e8, 1.2e10), "device": (3e6, 8e7), "call": (1e6, 1e8)}[entry]
    if mode in ("global_tb", "ksw"):
        cells = (cells[0], min(cells[1], 5e9))
    if workload == UNEVEN and mode not in ("local", "local_tb"):   # a few hundred to a few thousand long pairs
        cells = (cells[0], 1e9)
    lo, hi = math.log(cells[0]), math.log(cells[1])
    kw = {"second": mode in ("local", "local_start", "local_tb", "semi", "semi_start") and
          workload != UNEVEN and rng.random() < 0.3,
          "packed": rng.random() < 0.25, "scores": rng.choice(["1,4,6,1", "1,4,6,1", "2,3,5,2"])}
    if mode.startswith("semi"):
        kw["head"], kw["tail"] = (rng.choice(["NONE", "QUERY", "TARGET", "BOTH"]) for _ in range(2))
    if mode == "banded":
        kw["k_band"] = 8 * rng.randint(2, 8)
    if mode == "ksw" and rng.random() < 0.4:
        kw["w"], kw["zdrop"] = rng.choice([20, 50, 100]), rng.choice([0, 100])
    pairs = int(math.exp(rng.uniform(lo, hi)) / CELLS[workload]) | 1
    return _case(None, entry, mode, pairs, workload, **kw)


def _params(case):
    algo, start = MODES[case["mode"]]
    return g.Parameters(algo=algo, start_pos=start, secondBest=g.TRUE if case["second"] else g.FALSE,
                        isReverseComplement=case["workload"] == FULL, isPacked=case["packed"], k_band=case["k_band"],
                        semiglobal_skipping_head=getattr(g, case["head"]),
                        semiglobal_skipping_tail=getattr(g, case["tail"]))


def _outputs(case):
    """The result arrays the mode writes, by the names of the library's result struct."""
    mode = case["mode"]
    keys = ["aln_score"]
    if not mode.startswith("global"):
        keys += ["query_batch_end", "target_batch_end"]
    if mode in ("local_start", "local_tb", "semi_start"):
        keys += ["query_batch_start", "target_batch_start"]
    return keys


def prepare(case, seed):
    # the same lengths and mutations for a seed every time, other pairs for another
    batch = g.synth_batch(case["workload"], seed, case["pairs"])
    scores = tuple(int(v) for v in case["scores"].split(","))
    params = _params(case)
    mq, mt = int(batch.qlen.max()), int(batch.tlen.max())
    g.set_ksw_extension(case["w"], case["zdrop"])
    st = {"case": case, "params": params, "batch": batch, "keys": _outputs(case), "scores": scores}
    if case["entry"] == "device":
        g.set_n_code(g.N_CODE_DEFAULT)
        g.set_n_penalty(1)
        g.gasal_copy_subst_scores(g.gasal_subst_scores(*scores))
        on_gpu = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
        as_i32 = lambda a: on_gpu(a.astype(np.int32))
        seqs = [batch.packed_words(True), batch.packed_words(False)] if case["packed"] else [batch.q, batch.t]
        st["in"] = [on_gpu(a) for a in seqs] + [as_i32(a) for a in (batch.qoff, batch.toff, batch.qlen, batch.tlen)] + \
                   [on_gpu(a) for a in (batch.qop, batch.top)]
        st["out"] = [torch.zeros(batch.n, dtype=torch.int32, device="cuda") for _ in range(8)]
        st["max"] = (mq, mt)
        return st
    if case["entry"] == "stream":
        st["pairs"] = g.PairSet.from_batch(batch, pack=case["packed"])
        st["stream"] = g.Stream(params, 50_000, 3, mq, mt)
        return st
    st["aligner"] = a = g.Aligner(params, mq, mt, batch.n, scores=scores, n_penalty=1)
    if case["entry"] == "resident":
        a.load(batch, per_pair=False)
        st["stream"] = torch.cuda.ExternalStream(a.s.str)
    elif params.start_pos == g.WITH_TB:   # the padded query bytes' pair and place in it, to read CIGARs out of the query layout
        words = 8 * ((batch.qlen.astype(np.int64) + 7) // 8)
        st["owner"] = np.repeat(np.arange(batch.n), words)
        st["place"] = np.arange(len(batch.q)) - batch.qoff.astype(np.int64)[st["owner"]]
    return st


class _DeviceArray:
    """A device array of a storage, for torch.as_tensor; it keeps the storage."""

    def __init__(self, owner, address, shape, typestr):
        self.owner = owner
        self.__cuda_array_interface__ = {"data": (address, False), "shape": shape, "typestr": typestr, "version": 3}


def _view(owner, address, shape, typestr="<i4"):
    return torch.as_tensor(_DeviceArray(owner, address, shape, typestr), device="cuda")


def _resident_views(st):
    """The storage's result arrays as tensors (they stay where they are while the batch stays)."""
    a, n = st["aligner"], st["batch"].n
    address = lambda p: C.cast(p, C.c_void_p).value
    res = a.s.device_cpy.contents
    out = {k: _view(a, address(getattr(res, k)), (n,)) for k in st["keys"]}
    if st["params"].secondBest:
        second = a.s.device_cpy_second.contents
        out.update({"second_" + k: _view(a, address(getattr(second, k)), (n,))
                    for k in ("aln_score", "query_batch_end", "target_batch_end")})
    if st["params"].start_pos == g.WITH_TB:
        _, _, _, n_ops, cigar, cap = a.result_views()
        width = CIGAR[st["case"]["workload"]]
        out["n_ops"] = _view(a, n_ops, (n,))
        st["slots"] = _view(a, cigar, (n, cap), "|u1")[:, :width]
        st["column"] = torch.arange(width, dtype=torch.int32, device="cuda")
    return out


def run(st):
    case, params = st["case"], st["params"]
    if case["entry"] == "device":
        ptr = lambda t: C.c_void_p(t.data_ptr())
        b, out = st["batch"], st["out"]
        if g.lib().gasal2_aln_noalloc(ptr(st["in"][0]), ptr(st["in"][1]), len(b.q), len(b.t), *map(ptr, st["in"][2:]), b.n,
                                      *st["max"], *map(ptr, out), None, params.native(),
                                      C.c_void_p(torch.cuda.current_stream().cuda_stream)) != 0:
            raise RuntimeError("gasal2_aln_noalloc rejected the batch")
        keep = len(st["keys"])
        return out[:keep] + (out[5:] if params.secondBest else [])
    if case["entry"] == "stream":
        res, _ = st["pairs"].align(params, scores=st["scores"], n_penalty=1, cigar_cap=256, stream=st["stream"])
        return {k: v for k, v in res.items()}
    a = st["aligner"]
    if case["entry"] == "call":
        qb, tb, n = a.fill(st["batch"], per_pair=False)
        a.align_filled(qb, tb, n, poll_s=0)
        res = a._collect(n, qb)
        out = {k: v for k, v in res.items() if v is not None and k != "cigar_qlayout"}
        if params.algo == g.GLOBAL:
            out = {k: out[k] for k in ("score", "n_ops") if k in out}
        if "n_ops" in out:   # the written bytes of every CIGAR
            at = np.flatnonzero(st["place"] < out["n_ops"][st["owner"]])
            out["cigar"] = np.zeros((n, 8 * 64), np.uint8)
            out["cigar"][st["owner"][at], st["place"][at]] = res["cigar_qlayout"][at]
        return out
    a.run_resident()
    if "views" not in st:
        st["views"] = _resident_views(st)
    out = dict(st["views"])
    if "n_ops" in out:   # the written bytes of every CIGAR slot, on the storage's stream
        with torch.cuda.stream(st["stream"]):
            out["cigar"] = st["slots"] * (st["column"] < out["n_ops"][:, None])
    return out


def work(case):
    """Bytes: each base read once as it is stored, each result written once.
    flops: integer operations of the recurrence (11 a cell, 16 where the path
    is kept too), over the cells the mode is defined on."""
    n, (bq, bt) = case["pairs"], BASES[case["workload"]]
    cells = CELLS[case["workload"]]
    if case["mode"] == "banded":
        cells = min(cells, (case["k_band"] + 20.0) * bt)
    if case["w"] >= 0:
        cells = min(cells, (2.0 * case["w"] + 1.0) * bt)
    tb = case["mode"].endswith("_tb")
    outputs = 4 * (len(_outputs(case)) + (3 if case["second"] else 0)) + (4 + 40 if tb else 0)
    return {"bytes": n * ((bq + bt) * (0.5 if case["packed"] else 1.0) + 16 + outputs),
            "flops": n * cells * (16 if tb else 11) * (2 if case["mode"] in ("local_start", "semi_start") else 1)}


def exact(case, seed):
    """LOCAL scores of small batches from the textbook recurrence in int64 (no
    other output has a value that does not depend on tie-breaking)."""
    n = case["pairs"]
    if not case["mode"].startswith("local") or case["workload"] != SHORT or n * CELLS[SHORT] > 1e8:
        return None
    match, mismatch, gap_open, gap_extend = (int(v) for v in case["scores"].split(","))
    b = g.synth_batch(case["workload"], seed, n)
    rows, cols = int(b.qlen.max()), int(b.tlen.max())
    lay = lambda buf, off, ln, width: np.stack([np.pad(buf[o:o + l], (0, width - l)) for o, l in zip(off, ln)], axis=1)
    q, t = lay(b.q, b.qoff, b.qlen, rows), lay(b.t, b.toff, b.tlen, cols)   # padding: 0, equal to no base
    h, e, best = np.zeros((cols + 1, n), np.int64), np.full((cols + 1, n), -10**9), np.zeros(n, np.int64)
    for i in range(rows):
        s = np.where(q[i] == t, match, -mismatch)
        s = np.where((q[i] == ord("N")) | (t == ord("N")), -1, s)
        s = np.where((q[i] == 0) | (t == 0), -10**6, s)
        diag, f = h[0].copy(), np.full(n, -10**9)
        for j in range(1, cols + 1):
            e[j] = np.maximum(e[j] - gap_extend, h[j] - gap_open - gap_extend)
            f = np.maximum(f - gap_extend, h[j - 1] - gap_open - gap_extend)
            v = np.maximum(np.maximum(diag + s[j - 1], 0), np.maximum(e[j], f))
            diag = h[j].copy()
            h[j] = v
            best = np.maximum(best, v)
    if case["entry"] == "device":
        return [best]
    return {"score" if case["entry"] == "call" else "aln_score": best}
