"""The work that performance is measured on: what a program using this library has it do.

Every case goes through the public entry points (the C ABI as ``tomos_amd._capi`` binds it, and
``tomos_amd.autograd``).  The sizes are those of the repository's benchmark and tests, or generic
ones between them: 20,000 x 200 (plain LSQR on one small problem) to 2,000,000 x 1000 (the headline
solve), 64 uneven problems of 20,000..200,000 x 64..512 (here a batch of 20, so that every
gradient comes back as an output of its own), GEMMs up to 8192^3, CSR with 5..50 entries per row.

Matrices are column-major as in the C ABI: a contiguous torch tensor of shape (n, ld) is an m x n
matrix with leading dimension ld >= m.  A leading dimension equal to an odd m is what
``Dense::create_strided`` gives a C++ caller; ``tomos_amd.autograd`` and the benchmark pad to 64.
"""
import ctypes
import math

import numpy as np
import torch

from tomos_amd import _capi as C
from tomos_amd import autograd

TYPES = {"f32": C.F32, "f16": C.F16, "bf16": C.BF16, "fp32_16": C.FP32_16, "fp32_bf16": C.FP32_BF16}
TIERS = {"default": C.TIER_DEFAULT, "exact": C.TIER_EXACT, "materialize": C.TIER_MATERIALIZE}
PACKS = {"fp32_16": C.PACK_FP32_16, "fp32_bf16": C.PACK_FP32_BF16}
UNPACKS = {"fp32_16": C.DECODE_FP32_16_EXACT, "fp32_bf16": C.DECODE_FP32_BF16_EXACT}
DEV = "cuda"


def listed():
    return [
        # one step's products u = A v, z = A^T u of a small plain LSQR: launches and latency
        {"name": "gemv_20000x200", "kind": "gemv", "type": "fp32_bf16", "tier": "default", "m": 20000, "n": 200,
         "ld": 20000},
        # the published GEMV size, per-iteration tier of the FP32_16 format
        {"name": "gemv_1000000x1000_half", "kind": "gemv", "type": "fp32_16", "tier": "default", "m": 1000000,
         "n": 1000, "ld": 1000000},
        # restart residual and its transposed product: exact values, FP64 vectors, odd sizes, no padding
        {"name": "gemv_131071x501_exact", "kind": "gemv", "type": "fp32_16", "tier": "exact", "m": 131071, "n": 501,
         "ld": 131071},
        # storing an FP32 matrix in planes and reading it back
        {"name": "pack_500000x301", "kind": "pack", "type": "fp32_16", "m": 500000, "n": 301},
        # the preconditioner of an ordinary problem: CountSketch, QR, R^-1 (odd rows, no padding)
        {"name": "precond_250001x300", "kind": "precond", "type": "fp32_16", "m": 250001, "n": 300, "ld": 250001,
         "factor": 4, "kappa": 100.0},
        # the headline: preconditioner and solve to 1e-6
        {"name": "lsqr_2000000x1000", "kind": "lsqr", "type": "fp32_bf16", "m": 2000000, "n": 1000, "ld": 2000000,
         "factor": 4, "kappa": 1e6},
        # one differentiable least-squares layer fitting noisy data, forward and backward
        {"name": "lstsq_60000x300", "kind": "lstsq", "problems": 1, "m": 60000, "n": 300, "kappa": 1e3,
         "noise": 1e-3},
        # a batch of uneven differentiable problems with consistent right-hand sides, forward and backward
        {"name": "lstsq_batch20", "kind": "lstsq", "problems": 20, "m": 200000, "n": 512, "kappa": 1e4, "noise": 0.0},
        # both operands packed, 3-term split on the matrix cores
        {"name": "split_8192", "kind": "split", "type": "fp32_bf16", "m": 8192, "n": 8192, "k": 8192},
        # mm_apply's default tier on ragged sizes (A^T B, a block of right-hand sides)
        {"name": "mm_3001x1501x6001", "kind": "mm", "type": "fp32_16", "tier": "default", "ta": 1, "tb": 0, "m": 3001,
         "n": 1501, "k": 6001},
        # sparse LSQR at the tall shape, 50 entries per row
        {"name": "csr_2000000x1000", "kind": "csr", "m": 2000000, "n": 1000, "row": 50},
        # a dense Gaussian sketch
        {"name": "gaussian_2000x131072", "kind": "gaussian", "type": "f32", "m": 2000, "n": 131072},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["gemv", "gemv", "pack", "precond", "lsqr", "lstsq", "split", "mm", "csr", "gaussian"])
    if kind == "gemv":
        t = rng.choice(["f32", "f16", "bf16", "fp32_16", "fp32_16", "fp32_bf16", "fp32_bf16"])
        m, n = _log(rng, 5000, 1000000), _log(rng, 20, 1000)
        ld = m if rng.random() < 0.5 else (m + 63) // 64 * 64
        return {"kind": kind, "type": t, "tier": rng.choice(["default", "exact"]), "m": m, "n": n, "ld": ld}
    if kind == "pack":
        return {"kind": kind, "type": rng.choice(sorted(PACKS)), "m": _log(rng, 5000, 500000), "n": _log(rng, 20, 300)}
    if kind in ("precond", "lsqr"):
        t = rng.choice(["fp32_16", "fp32_bf16", "f32"])
        n = _log(rng, 40, 1000)
        m = max(_log(rng, 20000, 1000000), 20 * n)
        ld = m if kind == "precond" and rng.random() < 0.5 else (m + 63) // 64 * 64
        return {"kind": kind, "type": t, "m": m, "n": n, "ld": ld, "factor": rng.choice([4, 8]),
                "kappa": 100.0 if t == "fp32_16" else 10.0 ** rng.randint(2, 5)}
    if kind == "lstsq":
        p = rng.choice([1, 1, 2, 7, 16])
        noise = rng.choice([0.0, 1e-3]) if p == 1 else 0.0
        return {"kind": kind, "problems": p, "m": _log(rng, 5000, 60000 if noise else 180000),
                "n": _log(rng, 16, 300 if noise else 500), "kappa": 10.0 ** rng.randint(1, 4), "noise": noise}
    if kind in ("split", "mm"):
        c = {"kind": kind, "type": rng.choice(sorted(PACKS)), "m": _log(rng, 200, 8000), "n": _log(rng, 60, 8000),
             "k": _log(rng, 200, 8000)}
        if kind == "mm":
            c.update(tier=rng.choice(["default", "default", "materialize"]), ta=rng.randint(0, 1), tb=rng.randint(0, 1))
        return c
    if kind == "csr":
        return {"kind": kind, "m": _log(rng, 20000, 2000000), "n": _log(rng, 50, 4000), "row": rng.randint(5, 50)}
    return {"kind": kind, "type": rng.choice(["f32", "f32", "f16", "bf16"]), "m": _log(rng, 100, 4000),
            "n": _log(rng, 2000, 65000)}


# ---------------------------------------------------------------- inputs (plain torch, from the seed alone)
def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _matrix(g, m, n, ld, kappa=None, spread=0, dtype=torch.float32):
    """m x n column-major in an (n, ld) tensor: N(0,1), columns scaled log-spaced 1..1/kappa, or every
    entry by 2^k, k uniform in -spread..spread; the padding rows are zero."""
    a = torch.randn((n, ld), generator=g, device=DEV)
    if ld > m:
        a[:, m:] = 0
    if kappa is not None and n > 1:
        a *= torch.logspace(0, -math.log10(kappa), n, dtype=torch.float64, device=DEV).float()[:, None]
    if spread:
        a = torch.ldexp(a, torch.randint(-spread, spread + 1, a.shape, generator=g, device=DEV, dtype=torch.int32))
    return a.to(dtype)


def _rows(x, c0, c1):
    return x[c0:c1].double()


def _a_x(a, m, x):
    """A x in FP64 from the (n, ld) tensor, summed in a fixed order."""
    y = torch.zeros(m, dtype=torch.float64, device=DEV)
    step = max(1, int(2e8) // max(1, m))
    for j in range(0, a.shape[0], step):
        y += (_rows(a, j, j + step)[:, :m] * x[j:j + step, None]).sum(0)
    return y


def _at_y(a, m, y):
    step = max(1, int(2e8) // max(1, m))
    return torch.cat([(_rows(a, j, j + step)[:, :m] * y).sum(1) for j in range(0, a.shape[0], step)])


def _p(t):
    return ctypes.c_void_p(t.data_ptr()) if t is not None else None


def _stream():
    return ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)


def _bytes(n):
    return torch.empty(max(int(n), 1), dtype=torch.uint8, device=DEV)


def _store(kind, a, m):
    """The (n, ld) FP32 tensor in the storage type: (A or its hi plane, lo plane or None)."""
    if kind == "f32":
        return a, None
    if kind in ("f16", "bf16"):
        return a.to(torch.float16 if kind == "f16" else torch.bfloat16), None
    n, ld = a.shape
    wh, wr = torch.zeros_like(a, dtype=torch.int16), torch.zeros_like(a, dtype=torch.int16)
    C.call("tomos_pack", PACKS[kind], m, n, _p(a), ld, _p(wh), _p(wr), ld, _stream())
    return wh, wr


def _shapes(case, seed):
    """The shapes (m, n, kappa) of a batch: up to the case's, uneven, the same for every seed."""
    r = np.random.default_rng(case["m"] * 1009 + case["n"])
    out = [(case["m"], case["n"], case["kappa"])]
    for _ in range(case["problems"] - 1):
        n = int(r.integers(max(1, case["n"] // 8), case["n"] + 1))
        m = int(r.integers(max(4 * n, case["m"] // 10), max(4 * n, case["m"]) + 1))
        out.append((m, n, 10.0 ** r.uniform(1, math.log10(case["kappa"]))))
    return out


def _lstsq_inputs(case, seed):
    g = _gen(seed)
    out = []
    for m, n, kappa in _shapes(case, seed):
        at = _matrix(g, m, n, m, kappa)
        xt = torch.randn(n, generator=g, device=DEV, dtype=torch.float64)
        b = _a_x(at, m, xt)
        noise = torch.randn(m, generator=g, device=DEV, dtype=torch.float64)
        b = b + noise * (case["noise"] * b.norm() / noise.norm())
        out.append((at.t().contiguous(), b, torch.randn(n, generator=g, device=DEV, dtype=torch.float64)))
        del at
    return out


def _solve_inputs(case, seed):
    g = _gen(seed)
    m, n, ld = case["m"], case["n"], case["ld"]
    a = _matrix(g, m, n, ld, case["kappa"])
    xt = torch.randn(n, generator=g, device=DEV, dtype=torch.float64)
    return a, xt


def _csr_inputs(case, seed):
    g = _gen(seed)
    m, n, row = case["m"], case["n"], case["row"]
    # ragged rows: 1..row entries, the tall benchmark shape has them all
    full = m >= 2000000
    ln = torch.full((m,), row, device=DEV) if full else torch.randint(1, row + 1, (m,), generator=g, device=DEV)
    ci = torch.randint(0, n, (m, row), generator=g, device=DEV, dtype=torch.int32)
    v = torch.randn((m, row), generator=g, device=DEV)
    xt = torch.randn(n, generator=g, device=DEV, dtype=torch.float64)
    rp = torch.zeros(m + 1, dtype=torch.int32, device=DEV)
    rp[1:] = torch.cumsum(ln, 0).int()
    keep = torch.arange(row, device=DEV)[None, :] < ln[:, None]
    b = torch.empty(m, dtype=torch.float64, device=DEV)
    for i in range(0, m, 200000):
        s = slice(i, i + 200000)
        b[s] = (v[s].double() * xt[ci[s].long()] * keep[s]).sum(1)
    if full:
        return v.reshape(-1), ci.reshape(-1), rp, b, xt
    return v[keep], ci[keep], rp, b, xt


def prepare(case, seed):
    k = case["kind"]
    st = {"case": case}
    if k == "gemv":
        g = _gen(seed)
        m, n, ld = case["m"], case["n"], case["ld"]
        vt = torch.float64 if case["tier"] == "exact" else torch.float32
        a = _matrix(g, m, n, ld, spread=8 if case["type"] != "f16" else 2)
        st["a"], st["wr"] = _store(case["type"], a, m)
        st["x"] = torch.randn(n, generator=g, device=DEV, dtype=vt)
        st["w"] = torch.randn(m, generator=g, device=DEV, dtype=vt)
        st["y"], st["z"] = torch.empty(m, dtype=vt, device=DEV), torch.empty(n, dtype=vt, device=DEV)
        st["vt"] = C.F64 if vt == torch.float64 else C.F32
        t, tier = TYPES[case["type"]], TIERS[case["tier"]]
        st["nb"] = max(C.lib().tomos_gemv_scratch_size(t, tier, tr, m, n) for tr in (0, 1))
        st["scratch"] = _bytes(st["nb"])
    elif k == "pack":
        m, n = case["m"], case["n"]
        st["a"] = _matrix(_gen(seed), m, n, m, spread=8)
        st["wh"] = torch.zeros((n, m), dtype=torch.int16, device=DEV)
        st["wr"] = torch.zeros((n, m), dtype=torch.int16, device=DEV)
        st["back"] = torch.empty((n, m), device=DEV)
    elif k in ("precond", "lsqr"):
        m, n, s = case["m"], case["n"], case["factor"] * case["n"]
        a, xt = _solve_inputs(case, seed)
        st["a"], st["wr"] = _store(case["type"], a, m)
        st["sketch"] = torch.empty((n, s), dtype=torch.float64, device=DEV)
        st["nb"] = C.lib().tomos_countsketch_scratch_size(m, n, s)
        st["scratch"] = _bytes(st["nb"])
        if k == "lsqr":
            st["b"] = _a_x(a, m, xt)
            st["x"] = torch.empty(n, dtype=torch.float64, device=DEV)
            o = C.LsqrOptions(TYPES[case["type"]], C.TIER_DEFAULT, C.TIER_EXACT, C.F32, C.F64, C.F64, 1e-6, 1e-6, 8, 40,
                              8, 1, 1)
            st["opt"] = o
            st["ab"] = C.lib().tomos_lsqr_arena_size(ctypes.byref(o), m, n)
            st["sb"] = C.lib().tomos_lsqr_scratch_size(ctypes.byref(o), m, n)
            st["arena"], st["lscratch"] = _bytes(st["ab"]), _bytes(st["sb"])
    elif k == "lstsq":
        ins = _lstsq_inputs(case, seed)
        st["a"] = [a.requires_grad_() for a, _, _ in ins]
        st["b"] = [b.requires_grad_() for _, b, _ in ins]
        st["g"] = [g for _, _, g in ins]
    elif k == "split":
        g = _gen(seed)
        m, n, kk = case["m"], case["n"], case["k"]
        st["a"], st["aw"] = _store(case["type"], _matrix(g, m, kk, m), m)
        st["b"], st["bw"] = _store(case["type"], _matrix(g, kk, n, kk), kk)
        st["c"] = torch.empty((n, m), device=DEV)
        st["nb"] = C.lib().tomos_gemm_split_scratch_size(m, n, kk)
        st["scratch"] = _bytes(st["nb"])
    elif k == "mm":
        g = _gen(seed)
        m, n, kk = case["m"], case["n"], case["k"]
        ar, ac = (kk, m) if case["ta"] else (m, kk)
        br, bc = (n, kk) if case["tb"] else (kk, n)
        st["a"], st["wr"] = _store(case["type"], _matrix(g, ar, ac, ar), ar)
        st["b"] = _matrix(g, br, bc, br)
        st["c"] = torch.empty((n, m), device=DEV)
    elif k == "csr":
        st["v"], st["ci"], st["rp"], st["b"], _ = _csr_inputs(case, seed)
        m, n, nnz = case["m"], case["n"], st["v"].numel()
        o = C.LsqrOptions(C.F32, C.TIER_DEFAULT, C.TIER_DEFAULT, C.F32, C.F64, -1, 1e-6, 1e-6, 200, 1, 8, 0)
        st["opt"], st["nnz"] = o, nnz
        st["ab"] = C.lib().tomos_lsqr_arena_size(ctypes.byref(o), m, n)
        st["sb"] = C.lib().tomos_lsqr_csr_scratch_size(ctypes.byref(o), C.INDEX_INT32, m, n, nnz)
        st["arena"], st["scratch"] = _bytes(st["ab"]), _bytes(st["sb"])
        st["x"] = torch.empty(n, dtype=torch.float64, device=DEV)
    else:
        dt = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}[case["type"]]
        st["out"] = torch.empty((case["n"], case["m"]), dtype=dt, device=DEV)
        st["seed"] = int(seed) * 7919 + 17
    return st


# ---------------------------------------------------------------- one pass
def _precondition(st):
    c = st["case"]
    m, n, s = c["m"], c["n"], c["factor"] * c["n"]
    C.call("tomos_countsketch_apply", TYPES[c["type"]], C.TIER_EXACT, m, n, _p(st["a"]), _p(st["wr"]), c["ld"], s,
           _p(st["sketch"]), s, _p(st["scratch"]), st["nb"], _stream())
    C.call("tomos_sketch_qr_precond_f64", s, n, _p(st["sketch"]), s, _stream())
    return st["sketch"][:, :n]


def run(st):
    c = st["case"]
    k = c["kind"]
    if k == "gemv":
        t, tier = TYPES[c["type"]], TIERS[c["tier"]]
        for tr, x, y in ((0, st["x"], st["y"]), (1, st["w"], st["z"])):
            C.call("tomos_gemv", t, tier, tr, 1.0, c["m"], c["n"], _p(st["a"]), _p(st["wr"]), c["ld"], st["vt"], _p(x), 0.0,
                   st["vt"], _p(y), _p(st["scratch"]), st["nb"], _stream())
        return {"y": st["y"], "z": st["z"]}
    if k == "pack":
        m, n = c["m"], c["n"]
        C.call("tomos_pack", PACKS[c["type"]], m, n, _p(st["a"]), m, _p(st["wh"]), _p(st["wr"]), m, _stream())
        C.call("tomos_unpack", UNPACKS[c["type"]], m, n, _p(st["wh"]), _p(st["wr"]), m, _p(st["back"]), m, _stream())
        return {"wh": st["wh"], "wr": st["wr"], "back": st["back"]}
    if k == "precond":
        return {"rinv": _precondition(st)}
    if k == "lsqr":
        rinv = _precondition(st)
        s = c["factor"] * c["n"]
        C.call("tomos_lsqr_solve", ctypes.byref(st["opt"]), c["m"], c["n"], _p(st["a"]), _p(st["wr"]), c["ld"], _p(st["b"]),
               _p(st["x"]), _p(st["sketch"]), s, _p(st["arena"]), st["ab"], _p(st["lscratch"]), st["sb"], None, None, 0,
               None, _stream())
        return {"x": st["x"], "rinv": rinv}
    if k == "lstsq":
        if c["problems"] == 1:
            xs = [autograd.lstsq(st["a"][0], st["b"][0])]
        else:
            xs = autograd.lstsq_batched(st["a"], st["b"])
        grads = torch.autograd.grad(xs, st["a"] + st["b"], st["g"])
        p = c["problems"]
        return {"x": [x.detach() for x in xs], "grad_a": list(grads[:p]), "grad_b": list(grads[p:])}
    if k == "split":
        m, n, kk = c["m"], c["n"], c["k"]
        C.call("tomos_gemm_split", TYPES[c["type"]], m, n, kk, 1.0, _p(st["a"]), _p(st["aw"]), m, _p(st["b"]), _p(st["bw"]),
               kk, 0.0, _p(st["c"]), m, _p(st["scratch"]), st["nb"], _stream())
        return {"c": st["c"]}
    if k == "mm":
        m, n, kk = c["m"], c["n"], c["k"]
        C.call("tomos_gemm", TYPES[c["type"]], TIERS[c["tier"]], c["ta"], c["tb"], 1.0, m, n, kk, _p(st["a"]),
               _p(st["wr"]), kk if c["ta"] else m, _p(st["b"]), n if c["tb"] else kk, 0.0, _p(st["c"]), m, _stream())
        return {"c": st["c"]}
    if k == "csr":
        C.call("tomos_lsqr_solve_csr", ctypes.byref(st["opt"]), C.INDEX_INT32, c["m"], c["n"], st["nnz"], _p(st["v"]),
               _p(st["rp"]), _p(st["ci"]), -1, None, _p(st["b"]), _p(st["x"]), None, 1, _p(st["arena"]), st["ab"],
               _p(st["scratch"]), st["sb"], None, None, 0, None, _stream())
        return {"x": st["x"]}
    C.call("tomos_gaussian_fill", TYPES[c["type"]], c["m"], c["n"], _p(st["out"]), c["m"], st["seed"], _stream())
    return {"out": st["out"]}


# ---------------------------------------------------------------- what a pass cannot do without
def _esz(case, exact=False):
    t = case["type"]
    return 4 if t == "f32" or (exact and t in PACKS) else 2


def work(case):
    k, m, n = case["kind"], case["m"], case["n"]
    mn = float(m) * n
    if k == "gemv":  # the two products read A once each
        v = 8 if case["tier"] == "exact" else 4
        return {"bytes": 2 * (_esz(case, case["tier"] == "exact") * mn + v * (m + n)), "flops": 4 * mn}
    if k == "pack":
        return {"bytes": 16 * mn, "flops": 0}
    if k == "precond":
        s = case["factor"] * n
        return {"bytes": _esz(case, True) * mn + 8.0 * n * n, "flops": mn + 2.0 * s * n * n - n ** 3 / 3}
    if k == "lsqr":
        # A once for the sketch, b, and a solve of at least 16 iterations on the per-iteration plane
        # (2 products each) with two exact residuals
        s = case["factor"] * n
        return {"bytes": 3 * _esz(case, True) * mn + 16 * _esz(case) * mn + 8.0 * m + 8.0 * n,
                "flops": 16 * 4 * mn + 2.0 * s * n * n}
    if k == "lstsq":  # A and b in, x, grad_A and grad_b out; 2 x 16 Krylov steps of two products
        byts = flops = 0.0
        for mi, ni, _ in _shapes(case, 0):
            byts += 8.0 * mi * ni + 16.0 * mi
            flops += 32 * 4.0 * mi * ni
        return {"bytes": byts, "flops": flops}
    if k == "split":
        return {"bytes": 4.0 * (m + n) * case["k"] + 4 * mn, "flops": 6 * mn * case["k"]}
    if k == "mm":
        t = 3 if case["tier"] == "materialize" else 1
        return {"bytes": ((4.0 if t == 3 else 2.0) * m + 4.0 * n) * case["k"] + 4 * mn, "flops": t * 2 * mn * case["k"]}
    if k == "csr":  # values and columns in, b in, x out
        nnz = float(m) * (case["row"] if m >= 2000000 else (case["row"] + 1) / 2)
        return {"bytes": 8 * nnz + 4.0 * m + 8.0 * m + 8.0 * n, "flops": 4 * 4 * nnz}
    return {"bytes": (4 if case["type"] == "f32" else 2) * mn, "flops": 0}


def tolerance(case):
    k = case["kind"]
    if k == "pack":
        return "exact"
    if k == "gemv":  # FP64 sums of FP64 vectors, or FP32 sums
        return {"rel": 1e-13, "max": 1e-12} if case["tier"] == "exact" else {"rel": 1.5e-6, "max": 1.5e-5}
    if k == "precond":
        return {"rel": 1e-6, "max": 1e-4}
    if k == "lsqr":  # stops at relres 1e-6 with kappa up to 1e6; other sum orders move x by 1e-6
        return {"rel": 1e-4, "max": 1e-3}
    if k == "lstsq":  # grad_A is FP32
        return {"rel": 1e-8, "max": 5e-7}
    if k in ("split", "mm"):  # FP32 accumulation over k
        return {"rel": 3e-6, "max": 3e-5}
    if k == "csr":
        return {"rel": 2e-6, "max": 2e-5}
    return {"rel": 4e-7, "max": 4e-6} if case["type"] == "f32" else {"rel": 2e-4, "max": 1e-2}


# ---------------------------------------------------------------- the same in 64 bits, plain torch
def _stored(kind, a, exact):
    """The values that the storage type's tier multiplies by, from the FP32 matrix."""
    if kind == "f32" or (exact and kind in PACKS):
        return a
    if kind in ("f16", "bf16"):
        return a.to(torch.float16 if kind == "f16" else torch.bfloat16).float()
    out = torch.empty_like(a)
    step = max(1, int(1e8) // a.shape[1])
    for j in range(0, a.shape[0], step):
        u = a[j:j + step].contiguous().view(torch.int32)
        if kind == "fp32_bf16":  # the upper 16 bits
            out[j:j + step] = (u & -65536).view(torch.float32)
            continue
        # nearest-even to 9 fraction bits; below 2^-14 cut to a multiple of 2^-24
        r = ((u + 0x1FFF + ((u >> 14) & 1)) & -16384).view(torch.float32)
        low = torch.trunc(r * 2.0 ** 24) * 2.0 ** -24
        out[j:j + step] = torch.where(r.abs() < 2.0 ** -14, low, r)
    return out


def _i64(u):
    return u - (1 << 64) if u >= 1 << 63 else u


def _mix(z):
    """SplitMix64's output function on int64 tensors (wrapping products, logical shifts)."""
    z = (z ^ ((z >> 30) & ((1 << 34) - 1))) * _i64(0xbf58476d1ce4e5b9)
    z = (z ^ ((z >> 27) & ((1 << 37) - 1))) * _i64(0x94d049bb133111eb)
    return z ^ ((z >> 31) & ((1 << 33) - 1))


_GOLDEN = _i64(0x9e3779b97f4a7c15)


def _dense(a, b, g):
    """x, grad_A, grad_b of x = argmin |A x - b| with upstream g: CholeskyQR twice, in FP64."""
    a = a.detach().double()
    eye = torch.eye(a.shape[1], dtype=torch.float64, device=DEV)
    inv = lambda r: torch.linalg.solve_triangular(r, eye, upper=True)  # noqa: E731
    d = a.norm(dim=0)
    r1 = inv(torch.linalg.cholesky((a / d).t() @ (a / d), upper=True)) / d[:, None]
    q = a @ r1
    r2 = inv(torch.linalg.cholesky(q.t() @ q, upper=True))
    q, r = q @ r2, r1 @ r2
    x = r @ (q.t() @ b)
    x = x + r @ (q.t() @ (b - a @ x))
    w = r @ (r.t() @ g)
    gb = q @ (r.t() @ g)
    return x, torch.outer(b - a @ x, w) - torch.outer(gb, x), gb


def exact(case, seed):
    k, m, n = case["kind"], case["m"], case["n"]
    if k == "gemv":
        g = _gen(seed)
        vt = torch.float64 if case["tier"] == "exact" else torch.float32
        a = _matrix(g, m, n, case["ld"], spread=8 if case["type"] != "f16" else 2)
        a = _stored(case["type"], a, case["tier"] == "exact")
        x = torch.randn(n, generator=g, device=DEV, dtype=vt).double()
        w = torch.randn(m, generator=g, device=DEV, dtype=vt).double()
        return {"y": _a_x(a, m, x), "z": _at_y(a, m, w)}
    if k == "pack":
        return {"wh": None, "wr": None, "back": _matrix(_gen(seed), m, n, m, spread=8).double()}
    if k == "precond":
        return None  # R's row signs are the implementation's
    if k == "lsqr":
        return {"x": _solve_inputs(case, seed)[1], "rinv": None}  # R's row signs are the implementation's
    if k == "lstsq":
        got = [_dense(*t) for t in _lstsq_inputs(case, seed)]
        return {"x": [t[0] for t in got], "grad_a": [t[1] for t in got], "grad_b": [t[2] for t in got]}
    if k == "split":
        g = _gen(seed)
        a, b = _matrix(g, m, case["k"], m).double(), _matrix(g, case["k"], n, case["k"]).double()
        return {"c": b @ a}
    if k == "mm":
        g = _gen(seed)
        ar, ac = (case["k"], m) if case["ta"] else (m, case["k"])
        br, bc = (n, case["k"]) if case["tb"] else (case["k"], n)
        full = case["tier"] == "materialize"
        a, b = _stored(case["type"], _matrix(g, ar, ac, ar), full), _matrix(g, br, bc, br)
        if not full:
            b = b.to(torch.float16 if case["type"] == "fp32_16" else torch.bfloat16)
        a, b = a.double(), b.double()  # (columns, rows): op(A) is a.t() unless transposed
        return {"c": (b.t() if case["tb"] else b) @ (a.t() if case["ta"] else a)}
    if k == "csr":
        return {"x": _csr_inputs(case, seed)[4]}
    half = (m + 1) // 2
    st_seed = int(seed) * 7919 + 17
    out = torch.empty((n, 2 * half), dtype=torch.float64, device=DEV)
    step = max(1, int(5e7) // half)
    for j in range(0, n, step):
        p = torch.arange(j * half, min(n, j + step) * half, dtype=torch.int64, device=DEV)
        z = _mix((p + 1) * _GOLDEN + st_seed)
        u1 = (((z >> 41) & ((1 << 23) - 1)).double() + 0.5) * 2.0 ** -23
        u2 = ((z >> 8) & 0xFFFFFF).double() * 2.0 ** -24
        r = torch.sqrt(-2.0 * torch.log(u1))
        out[j:j + step, 0::2] = (r * torch.cos(2 * math.pi * u2)).reshape(-1, half)
        out[j:j + step, 1::2] = (r * torch.sin(2 * math.pi * u2)).reshape(-1, half)
    return {"out": out[:, :m]}
