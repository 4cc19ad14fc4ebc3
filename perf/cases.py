"""Timed cases of the Top-K SpMV paths: what a program that searches resident
matrices calls, over the sizes it meets.

A case is one matrix and one call on it:

  call "lowbit"  one query through the low-bit two-stage search
                 (GpuMatrix.topk_lowbit, or a Plan of it);
       "host"    the same from host arrays (GpuMatrix.topk_lowbit_host);
       "batch"   nq queries in one call (GpuMatrix.topk_lowbit_batch, or a Plan
                 of it), each with its own K when mixed;
       "fp32"    one query through the plain FP32 CSR Top-K
                 (GpuMatrix.topk_fp32, or a Plan of it);
       "serve"   nq requests submitted to a Server and waited for.

Matrices: rows x cols with distinct uniform columns, row lengths uniform in
[lo, hi] or power-law (gamma shape 0.5 with mean lo, at most hi), values
|N(0,1)| (N(0,1) for signed packets), L2-normalised rows except the largest
matrix.  Queries are N(0,1).  All of it is drawn from the seed, on the GPU.

torch is imported first: the library then shares its HIP runtime, and tensors
can be passed where it takes device memory.
"""
import math

import numpy as np
import torch

import acceles_amd as acc

MIXED_K = (1, 8, 16, 32, 50, 75, 100)


def _case(name, call, rows, cols, lo, hi, **more):
    c = {"name": name, "call": call, "rows": rows, "cols": cols, "deg": "uniform", "lo": lo, "hi": hi, "l2norm": True,
         "bits": 8, "signed": False, "split": 32, "ck": 512, "nq": 1, "k": 100, "mixed": False, "plan": False}
    c.update(more)
    return c


def listed():
    return [
        # a lookup in a small corpus from host arrays: the drop-in call of a program without device memory of its own
        _case("host_20k", "host", 20000, 500, 40, 100),
        # interactive search of an embedding corpus, one query at a time
        _case("lowbit_400k", "lowbit", 400000, 500, 40, 100),
        # the same with fewer bits per value and a captured launch sequence, a short result list, ragged sizes
        _case("lowbit_1m_4bit", "lowbit", 999983, 250, 20, 60, bits=4, k=32, plan=True),
        # a corpus far beyond the caches: the streaming pass is all of it
        _case("lowbit_20m", "lowbit", 20000000, 1024, 10, 30, l2norm=False, split=64, ck=1024),
        # a few users at once
        _case("batch8_400k", "batch", 400000, 500, 40, 100, nq=8, mixed=True),
        # the throughput configuration: batches of Top-100 queries replayed from a plan
        _case("batch100_400k", "batch", 400000, 500, 40, 100, nq=100, plan=True),
        # one fused launch of many queries of mixed K on a large matrix
        _case("batch256_2m", "batch", 2000000, 900, 30, 90, nq=256, mixed=True, plan=True),
        # signed embeddings at 6 bits, an odd batch
        _case("batch41_1m_signed6", "batch", 1000000, 500, 40, 80, bits=6, signed=True, nq=41, mixed=True),
        # exact search of a small corpus
        _case("fp32_100k", "fp32", 100000, 500, 50, 90, plan=True),
        # exact search of a large one
        _case("fp32_2m", "fp32", 2000000, 900, 30, 90),
        # exact search over power-law rows with a long result list (re-ranking)
        _case("fp32_5m_gamma", "fp32", 4999999, 1024, 20, 1024, deg="gamma", l2norm=False, k=500),
        # a burst of requests of mixed K at the request loop
        _case("serve_400k", "serve", 400000, 500, 40, 100, nq=200, mixed=True),
    ]


def draw(rng):
    def log_int(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    call = rng.choice(("host", "lowbit", "lowbit", "batch", "batch", "batch", "fp32", "fp32", "serve"))
    rows = log_int(20000, 400000 if call == "serve" else 1500000)
    cols = rng.randint(200, 1024)
    lo = rng.randint(10, 50)
    hi = lo + rng.randint(10, 50)
    c = _case("", call, rows, cols, lo, hi)
    del c["name"]
    if rng.random() < 0.2:
        c.update(deg="gamma", lo=rng.randint(15, 40), hi=cols)
    if call == "fp32":
        c["k"] = log_int(1, 500)
    else:
        bits, signed = rng.choice(((8, False), (8, False), (4, False), (6, True)))
        split = rng.choice((16, 32, 64))
        c.update(bits=bits, signed=signed, split=split, ck=split * rng.choice((8, 16, 24)), k=rng.randint(1, 100))
    if call == "batch":
        c.update(nq=log_int(2, 256), mixed=rng.random() < 0.5)
    if call == "serve":
        c.update(nq=log_int(20, 200), mixed=True)
    if call not in ("host", "serve"):
        c["plan"] = rng.random() < 0.5
    if c["mixed"]:
        c["k"] = 100
    c["k"] = min(c["k"], c["ck"])
    return c


# ---- inputs ---------------------------------------------------------------

def _matrix(case, seed):
    """(ptr, idx, val) of the case's matrix as numpy arrays."""
    rows, cols = case["rows"], case["cols"]
    g = torch.Generator(device="cuda").manual_seed(seed)
    if case["deg"] == "gamma":
        # Gamma(1/2) with mean lo is lo times a squared N(0,1)
        d = torch.randn(rows, generator=g, device="cuda").square() * case["lo"]
        d = d.round().clamp(1, case["hi"])
    else:
        d = torch.randint(case["lo"], case["hi"] + 1, (rows,), generator=g, device="cuda").float()
    # draws with replacement that leave about d distinct columns
    d = (-cols * torch.log1p(-(d / cols).clamp(max=0.95))).round().clamp(min=1).long()
    key = torch.repeat_interleave(torch.arange(rows, device="cuda"), d)
    key.mul_(cols).add_(torch.randint(0, cols, key.shape, generator=g, device="cuda"))
    key = torch.unique_consecutive(key.sort().values)
    ptr = torch.searchsorted(key, torch.arange(rows + 1, device="cuda") * cols).cpu().numpy()
    idx = key.remainder_(cols).int().cpu().numpy()
    del key
    val = torch.randn(len(idx), generator=g, device="cuda")
    if not case["signed"]:
        val.abs_()
    val = val.cpu().numpy()
    if case["l2norm"]:
        s = np.sqrt(np.add.reduceat(val.astype(np.float64) ** 2, ptr[:-1]))
        val = (val / np.repeat(s, np.diff(ptr))).astype(np.float32)
    torch.cuda.empty_cache()
    return ptr, idx, val


def _queries(case, seed):
    x = np.random.default_rng(seed + 1).standard_normal((case["nq"], case["cols"])).astype(np.float32)
    if case["mixed"]:
        ks = np.random.default_rng(seed + 2).choice(MIXED_K, case["nq"])
        ks = np.minimum(ks, case["k"])
    else:
        ks = np.full(case["nq"], case["k"])
    return x, ks.astype(np.int32)


def prepare(case, seed):
    ptr, idx, val = _matrix(case, seed)
    csr = acc.CSRMatrix.from_arrays(case["rows"], case["cols"], ptr, idx, val)
    x, ks = _queries(case, seed)
    st = {"call": case["call"], "ck": case["ck"], "k": case["k"], "ks": ks, "plan": None}
    packed = None
    if case["call"] != "fp32":
        packed = csr.pack(bits=case["bits"], split=case["split"], is_signed=case["signed"])
    if case["call"] == "serve":
        st["server"] = acc.Server(max_batch=256, slots=4, ck=case["ck"], memory_budget=8 << 30)
        st["matrix"] = st["server"].add_matrix(csr, packed)
        st["x"] = list(x)
        return st
    m = st["m"] = acc.GpuMatrix(csr, packed)
    if case["call"] == "host":
        st["x"] = x[0]
        return st
    st["x"] = torch.from_numpy(x).cuda()
    st["out"] = torch.zeros((case["nq"], case["k"], 2), dtype=torch.int32, device="cuda")
    st["result"] = {"value": st["out"].view(torch.float32)[..., 0], "row": st["out"][..., 1]}
    if case["plan"]:
        kind = {"lowbit": acc.PLAN_LOWBIT, "batch": acc.PLAN_LOWBIT_BATCH, "fp32": acc.PLAN_FP32}[case["call"]]
        st["plan"] = acc.Plan(m, kind, st["x"], ks, case["ck"], st["out"], case["k"])
    return st


def run(st):
    call = st["call"]
    if call == "serve":
        srv, m, ks = st["server"], st["matrix"], st["ks"]
        tickets = [srv.submit(m, x, k) for x, k in zip(st["x"], ks)]
        got = np.zeros((len(ks), st["k"]), acc.ELEMENT_DTYPE)
        for i, t in enumerate(tickets):
            got[i, :ks[i]] = srv.wait(t, ks[i])
        return {"value": got["value"], "row": got["index"]}
    if call == "host":
        got = st["m"].topk_lowbit_host(st["x"], st["k"], st["ck"])
        return {"value": got["value"], "row": got["index"]}
    if st["plan"] is not None:
        st["plan"].launch()
    elif call == "lowbit":
        st["m"].topk_lowbit(st["x"], st["k"], st["ck"], st["out"])
    elif call == "batch":
        st["m"].topk_lowbit_batch(st["x"], st["ks"], st["ck"], st["out"], st["k"])
    else:
        st["m"].topk_fp32(st["x"], st["k"], st["out"])
    return st["result"]


# ---- what a pass cannot do without ----------------------------------------

def work(case):
    mean = case["lo"] if case["deg"] == "gamma" else (case["lo"] + case["hi"]) / 2
    nnz, nq = case["rows"] * mean, case["nq"]
    ends = nq * (case["cols"] * 4 + case["k"] * 8)
    if case["call"] == "fp32":
        return {"bytes": nnz * 8 + case["rows"] * 4 + ends, "flops": 2 * nnz}
    # one pass over the packed entries for all queries, and the candidates' FP32 rows
    entry = (max(case["cols"] - 1, 1).bit_length() + case["bits"]) / 8
    rescored = nq * case["ck"] * mean
    return {"bytes": nnz * entry + rescored * 8 + ends, "flops": 2 * (nnz * nq + rescored)}


# ---- the same in 64 bits --------------------------------------------------

def _quantized(v, bits, signed):
    """q = rint(M * (v / max|v|)) in float32, half to even."""
    M = (1 << bits) - 1
    M = M // 2 if signed else M
    s = np.abs(v).max()
    return np.clip(np.rint(np.float32(M) * (v / s)), -M - 1, M)


def _all_scores(ptr, idx, val, cols, x):
    """A x for queries x (nq, cols) in float64: (nq, rows) on the GPU, from dense blocks of rows."""
    rows = len(ptr) - 1
    step = max(1, (1 << 27) // cols)
    xt = torch.from_numpy(np.ascontiguousarray(x.T, dtype=np.float64)).cuda()
    out = torch.empty((len(x), rows), dtype=torch.float64, device="cuda")
    for r0 in range(0, rows, step):
        r1 = min(rows, r0 + step)
        b, e = ptr[r0], ptr[r1]
        dense = torch.zeros((r1 - r0) * cols, dtype=torch.float64, device="cuda")
        r = torch.repeat_interleave(torch.arange(r1 - r0, device="cuda"), torch.from_numpy(np.diff(ptr[r0:r1 + 1])).cuda())
        dense[r * cols + torch.from_numpy(idx[b:e]).cuda()] = torch.from_numpy(val[b:e]).cuda().double()
        out[:, r0:r1] = (dense.view(r1 - r0, cols) @ xt).T
    return out


def exact(case, seed):
    ptr, idx, val = _matrix(case, seed)
    x, ks = _queries(case, seed)
    rows, cols, nq = case["rows"], case["cols"], case["nq"]
    if case["call"] == "fp32":
        top = torch.topk(_all_scores(ptr, idx, val, cols, x), case["k"]).values.cpu().numpy()
    else:
        # stage 1 in whole numbers: the best M rows of each partition, the lower row on ties
        q = _quantized(val, case["bits"], case["signed"])
        xq = np.stack([_quantized(v, 8, True) for v in x])
        split, M = case["split"], case["ck"] // case["split"]
        size = rows // split
        cand = []
        for q0 in range(0, nq, 64):
            s = _all_scores(ptr, idx, q, cols, xq[q0:q0 + 64]).long()
            s.mul_(1 << 31).add_(rows - 1 - torch.arange(rows, device="cuda"))
            rest = s[:, size * (split - 1):]
            parts = [torch.topk(rest, min(M, rest.shape[1])).values]
            if split > 1:
                head = s[:, :size * (split - 1)].reshape(len(s), split - 1, size)
                parts.append(torch.topk(head, min(M, size)).values.flatten(1))
            cand.append(rows - 1 - torch.cat(parts, 1).remainder(1 << 31))
            del s, rest
        cand = torch.cat(cand).cpu().numpy()
        # stage 2: their rows against the query
        top = np.empty((nq, case["k"]))
        for i in range(nq):
            b = ptr[cand[i]]
            n = ptr[cand[i] + 1] - b
            at = np.repeat(b - np.concatenate(([0], np.cumsum(n)[:-1])), n) + np.arange(n.sum())
            p = val[at].astype(np.float64) * x[i].astype(np.float64)[idx[at]]
            # a zero closes the list: reduceat gives an empty row its next row's first product
            starts = np.concatenate(([0], np.cumsum(n)[:-1]))
            y = np.where(n > 0, np.add.reduceat(np.concatenate((p, [0.0])), starts), 0.0)
            top[i] = np.sort(y)[::-1][:case["k"]]
    torch.cuda.empty_cache()
    if case["call"] == "host":
        return {"value": top[0], "row": None}
    if case["call"] != "fp32":
        top = np.where(np.arange(case["k"]) < ks[:, None], top, 0.0)
    return {"value": top, "row": None}
