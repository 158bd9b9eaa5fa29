"""GPU GEMV parity against the CPU oracle tiers and an FP64 numpy reference.

Tolerances:
  * FAST / EXACT tiers and every F64 GEMV accumulate in FP64 over the same
    decoded values as the oracle: |gpu - oracle| <= 1e-12 * (|A||x|)_i + tiny.
  * DEFAULT tier (FP32 accumulation): |gpu - oracle_fp64acc| <= 2e-6 * (|A||x|)_i.
  * The reference's own tier tolerances vs the exact product
    (test/core/matrix/test_fp32_16.cpp:178-182, 1015-1016): pure_half
    0.15|ref|+0.15 elementwise on U[-8,8] data, L2-rel < 5e-2 at 140000 x 100;
    accurate 1e-3|ref|+1e-4 and L2-rel < 1e-3.
"""
import numpy as np
import pytest

from tests import hipcall as H
from tomos_amd import _capi as C

pytestmark = pytest.mark.gpu

FORMATS = {
    C.FP32_16: (C.PACK_FP32_16, {C.TIER_DEFAULT: 1, C.TIER_FAST: 1, C.TIER_EXACT: 0}),
    C.FP32_BF16: (C.PACK_FP32_BF16, {C.TIER_DEFAULT: 5, C.TIER_FAST: 5, C.TIER_EXACT: 4}),
}


def data(m, n, seed, wide=False):
    rng = np.random.default_rng(seed)
    A = rng.standard_normal((m, n))
    if wide:
        A *= 2.0 ** rng.integers(-8, 9, (m, n))
    return np.asfortranarray(A.astype(np.float32))


def check_close(got, exp, scale, rtol):
    err = np.abs(got.astype(np.float64) - exp.astype(np.float64))
    bound = rtol * scale + 1e-30
    assert np.all(err <= bound), (np.max(err / bound), np.argmax(err / bound))


@pytest.mark.parametrize("a_type", [C.FP32_16, C.FP32_BF16])
@pytest.mark.parametrize("tier", [C.TIER_DEFAULT, C.TIER_FAST, C.TIER_EXACT])
@pytest.mark.parametrize("trans", [0, 1])
@pytest.mark.parametrize("shape", [(3000, 70, 3000), (2999, 33, 2999), (1000, 257, 1008), (5, 5, 5)])
def test_packed_gemv_vs_oracle(capi, orc, a_type, tier, trans, shape):
    m, n, lda = shape
    print("gemv", a_type, tier, trans, shape, flush=True)
    A = data(m, n, seed=m + n + trans, wide=True)
    variant, decs = FORMATS[a_type]
    wh, wr = H.pack(variant, A, ld=lda)
    rng = np.random.default_rng(7)
    rows, cols = (n, m) if trans else (m, n)
    x = rng.standard_normal(cols).astype(np.float32)
    y0 = rng.standard_normal(rows).astype(np.float32)
    for alpha, beta in [(1.0, 0.0), (-0.75, 0.7)]:
        got = H.gemv(a_type, tier, trans, alpha, m, n, wh, wr, lda, x, beta, y0)
        ehh, err_ = orc.pack(variant, A)
        dec = decs[tier]
        exp = orc.mv_packed(dec, trans, alpha, ehh, err_, m, x, beta, y0)
        Adec = orc.unpack(dec, ehh, err_).astype(np.float64)
        scale = np.abs(alpha) * (np.abs(Adec.T if trans else Adec) @ np.abs(x.astype(np.float64)))
        scale += np.abs(beta) * np.abs(y0.astype(np.float64))
        rtol = 3e-5 if tier == C.TIER_DEFAULT else 1e-6  # y is stored in FP32
        check_close(got, exp, scale + 1e-30, rtol)


@pytest.mark.parametrize("trans", [0, 1])
@pytest.mark.parametrize("xy", [(C.F32, C.F32), (C.F64, C.F32), (C.F32, C.F64), (C.F64, C.F64)])
def test_plain_gemv_types(capi, trans, xy):
    m, n = 4100, 130
    A = data(m, n, 11)
    x_type, y_type = xy
    rng = np.random.default_rng(5)
    rows, cols = (n, m) if trans else (m, n)
    x = rng.standard_normal(cols)
    y0 = rng.standard_normal(rows)
    Ad = H.dev(A)
    A64 = A.astype(np.float64)
    ref = 0.5 * ((A64.T if trans else A64) @ x.astype(np.float32 if x_type == C.F32 else np.float64)) + 2.0 * y0.astype(np.float32 if y_type == C.F32 else np.float64)
    scale = 0.5 * (np.abs(A64.T if trans else A64) @ np.abs(x)) + 2.0 * np.abs(y0)
    for tier, rtol in [(C.TIER_DEFAULT, 3e-5), (C.TIER_EXACT, 1e-12 if y_type == C.F64 else 1e-7)]:
        got = H.gemv(C.F32, tier, trans, 0.5, m, n, Ad, None, m, x, 2.0, y0, x_type, y_type)
        check_close(got, ref, scale, rtol)
    A2 = H.dev(A64)
    got = H.gemv(C.F64, C.TIER_DEFAULT, trans, 0.5, m, n, A2, None, m, x, 2.0, y0, x_type, y_type)
    check_close(got, ref, scale, 1e-12 if y_type == C.F64 else 1e-7)


def test_gemv_explicit_scratch_and_small_square(capi):
    # small square (R^-1 shape class): exercises the column-split path
    n = 1000
    rng = np.random.default_rng(1)
    R = np.triu(rng.standard_normal((n, n)))
    x = rng.standard_normal(n)
    Rd = H.dev(R)
    for trans in (0, 1):
        got = H.gemv(C.F64, C.TIER_DEFAULT, trans, 1.0, n, n, Rd, None, n, x, 0.0, None,
                     C.F64, C.F64, scratch="explicit")
        ref = (R.T if trans else R) @ x
        check_close(got, ref, np.abs(R.T if trans else R) @ np.abs(x), 1e-13)


def test_reference_tier_tolerances_small(capi, orc):
    """test_fp32_16.cpp:178-182 style: 5x5, U[-8,8], trans x beta grid."""
    rng = np.random.default_rng(101)
    for trial in range(3):
        A = rng.uniform(-8, 8, (5, 5)).astype(np.float32)
        x = rng.uniform(-8, 8, 5).astype(np.float32)
        y0 = rng.uniform(-8, 8, 5).astype(np.float32)
        wh, wr = H.pack(C.PACK_FP32_16, A)
        for trans in (0, 1):
            for beta in (0.0, 0.7):
                ref = (A.T.astype(np.float64) if trans else A.astype(np.float64)) @ x + beta * y0
                ph = H.gemv(C.FP32_16, C.TIER_DEFAULT, trans, 1.0, 5, 5, wh, wr, 5, x, beta, y0)
                fa = H.gemv(C.FP32_16, C.TIER_FAST, trans, 1.0, 5, 5, wh, wr, 5, x, beta, y0)
                ex = H.gemv(C.FP32_16, C.TIER_EXACT, trans, 1.0, 5, 5, wh, wr, 5, x, beta, y0)
                assert np.all(np.abs(ph - ref) <= 0.15 * np.abs(ref) + 0.15)
                assert np.all(np.abs(fa - ref) <= 0.05 * np.abs(ref) + 0.05)
                assert np.all(np.abs(ex - ref) <= 1e-3 * np.abs(ref) + 1e-4)


def test_reference_large_shape_l2(capi):
    """test_fp32_16.cpp:924-1017: 140000 x 100 and the ragged 140001 lead dim."""
    for m in (140000, 140001):
        n = 100
        rng = np.random.default_rng(m)
        A = rng.uniform(-8, 8, (m, n)).astype(np.float32, order="F")
        x = rng.uniform(-8, 8, n).astype(np.float32)
        u = rng.uniform(-8, 8, m).astype(np.float32)
        wh, wr = H.pack(C.PACK_FP32_16, A)
        A64 = A.astype(np.float64)
        for trans, vec in ((0, x), (1, u)):
            ref = (A64.T if trans else A64) @ vec.astype(np.float64)
            ph = H.gemv(C.FP32_16, C.TIER_DEFAULT, trans, 1.0, m, n, wh, wr, m, vec)
            ex = H.gemv(C.FP32_16, C.TIER_EXACT, trans, 1.0, m, n, wh, wr, m, vec)
            l2 = lambda g: np.linalg.norm(g - ref) / np.linalg.norm(ref)
            assert l2(ph) < 5e-2 and l2(ex) < 1e-3, (m, trans, l2(ph), l2(ex))


def bf16_bits_rne(A32):
    """Round-to-nearest-even FP32 -> bf16 bits (finite inputs)."""
    u = np.asarray(A32, dtype=np.float32).view(np.uint32).astype(np.uint64)
    r = (u + 0x7FFF + ((u >> 16) & 1)) >> 16
    return r.astype(np.uint16)


@pytest.mark.parametrize("a_type", [C.F16, C.BF16])
@pytest.mark.parametrize("trans", [0, 1])
@pytest.mark.parametrize("shape", [(3000, 70, 3000), (2999, 33, 2999), (1000, 257, 1008)])
def test_native_16bit_gemv(capi, a_type, trans, shape):
    """Native IEEE half / bf16 storage: the stored values times x, FP32
    accumulation (DEFAULT) or FP64 (FAST, EXACT), against FP64 numpy."""
    m, n, lda = shape
    A = data(m, n, 17 + m)
    if a_type == C.F16:
        bits = A.astype(np.float16).view(np.uint16)
        A_used = A.astype(np.float16).astype(np.float64)
    else:
        bits = bf16_bits_rne(A)
        A_used = (bits.astype(np.uint32) << 16).view(np.float32).astype(np.float64)
    store = np.zeros((lda, n), np.uint16, order="F")
    store[:m] = bits
    Ad = H.dev(store)
    rng = np.random.default_rng(3)
    rows, cols = (n, m) if trans else (m, n)
    x = rng.standard_normal(cols)
    y0 = rng.standard_normal(rows)
    op = A_used.T if trans else A_used
    ref = 1.5 * (op @ x) - 0.5 * y0
    scale = 1.5 * (np.abs(op) @ np.abs(x)) + 0.5 * np.abs(y0)
    for tier, rtol in [(C.TIER_DEFAULT, 3e-6), (C.TIER_FAST, 1e-12), (C.TIER_EXACT, 1e-12)]:
        got = H.gemv(a_type, tier, trans, 1.5, m, n, Ad, None, lda, x, -0.5, y0, C.F64, C.F64)
        check_close(got, ref, scale, rtol)


# The edges of the kernels' ranges: fewer rows than a vector, the last vector
# of a column moved back over its neighbour's rows, columns on odd addresses,
# one column, fewer columns than column groups, both sides of the whole-column
# limit (128 KB a column) and of the column-split rules.
EDGE = [(1, 1, 1), (7, 3, 7), (8, 1, 8), (9, 40, 9), (129, 66, 131), (4097, 9, 4099), (65535, 5, 65535),
        (65536, 3, 65536), (65537, 67, 65537), (32769, 33, 32777), (300, 300, 300)]


@pytest.mark.parametrize("a_type", [C.F32, C.F64, C.F16, C.BF16, C.FP32_16, C.FP32_BF16])
@pytest.mark.parametrize("shape", EDGE)
def test_gemv_edges(capi, orc, a_type, shape):
    """Every tier and direction against FP64 products of the stored values.
    The matrix holds every word class of FP32_16 (subnormal and overflowing
    half words, saturated words), one Inf in the last row (rows next to it
    are read twice) and padding rows of NaN.  Bounds as in the tests above:
    n eps |A||x| is 65537 * 6e-8 = 4e-3 at worst for FP32 sums in one chain
    and 300 * 6e-8 = 2e-5 in the chains used here; FP64 7e-12 and 3e-14."""
    m, n, lda = shape
    rng = np.random.default_rng(m * 7 + n)
    A = data(m, n, m + 3 * n, wide=True)
    k = rng.integers(0, m * n, 3)
    A.flat[k] = np.array([3e4, -2e-9, 1e-6], np.float32)  # large, saturated, subnormal half
    inf_at = (m - 1, n - 1)
    if a_type in FORMATS:
        variant, decs = FORMATS[a_type]
        A[inf_at] = np.inf  # FP32_16: a saturated overflow word
        ehh, err_ = orc.pack(variant, A)
        sh, sr = np.full((lda, n), 0x7FFF, np.uint16, order="F"), np.full((lda, n), 0x7FFF, np.uint16, order="F")
        sh[:m], sr[:m] = ehh, err_
        a, wr = H.dev(sh), H.dev(sr)
        value = {t: orc.unpack(decs[t], ehh, err_).astype(np.float64) for t in decs}
    else:
        dt = {C.F32: np.float32, C.F64: np.float64, C.F16: np.float16}.get(a_type)
        A[inf_at] = np.inf
        if a_type == C.BF16:
            st = bf16_bits_rne(A)
            v = (st.astype(np.uint32) << 16).view(np.float32).astype(np.float64)
            pad = np.uint16(0x7FFF)
        else:
            st = A.astype(dt)
            v, pad = st.astype(np.float64), np.nan
        store = np.full((lda, n), pad, st.dtype, order="F")
        store[:m] = st
        a, wr = H.dev(store), None
        value = {t: v for t in (C.TIER_DEFAULT, C.TIER_FAST, C.TIER_EXACT)}
    for trans in (0, 1):
        rows, cols = (n, m) if trans else (m, n)
        x = rng.standard_normal(cols)
        y0 = rng.standard_normal(rows)
        for tier, rtol in ((C.TIER_DEFAULT, 3e-5), (C.TIER_FAST, 1e-12), (C.TIER_EXACT, 1e-12)):
            print("edge", a_type, shape, trans, tier, flush=True)
            op = value[tier].T if trans else value[tier]
            with np.errstate(invalid="ignore"):
                ref = 1.5 * (op @ x) - 0.5 * y0
                scale = 1.5 * (np.abs(op) @ np.abs(x)) + 0.5 * np.abs(y0)
            got = H.gemv(a_type, tier, trans, 1.5, m, n, a, wr, lda, x, -0.5, y0, C.F64, C.F64)
            fin = np.isfinite(ref)
            assert np.array_equal(got[~fin], ref[~fin], equal_nan=True)
            check_close(got[fin], ref[fin], scale[fin], rtol)


@pytest.mark.parametrize("a_type", [C.F32, C.F64, C.BF16, C.FP32_16, C.FP32_BF16])
@pytest.mark.parametrize("m,n", [(1, 4097), (3, 9000), (9, 4103), (300, 5001), (1025, 4100), (2050, 8193), (12300, 8200)])
def test_gemv_t_many_columns(capi, orc, a_type, m, n):
    """A^T x of many short columns (a wave owns 8): fewer rows than a vector,
    the last vector moved back over its neighbour's rows with an Inf beside
    it, column counts around the wave's 8, both sides of the rules on a
    column's bytes.  Products of small integers, |sum| < 2^24: exact."""
    rng = np.random.default_rng(m + n)
    A = rng.integers(-8, 9, (m, n)).astype(np.float32)
    A[m - 1, n // 2] = np.inf
    x = rng.integers(-8, 9, m).astype(np.float64)
    x[m - 1] = 2.0
    lda = m + 3
    store = np.full((lda, n), np.nan, np.float32, order="F")
    store[:m] = A
    if a_type in FORMATS:
        wh, wr = H.pack(FORMATS[a_type][0], store)
    else:
        st = store.astype(np.float64) if a_type == C.F64 else bf16_bits_rne(store) if a_type == C.BF16 else store
        wh, wr = H.dev(st), None
    with np.errstate(invalid="ignore"):
        ref = A.T.astype(np.float64) @ x
    for tier in (C.TIER_DEFAULT, C.TIER_FAST, C.TIER_EXACT):
        print("many columns", a_type, m, n, tier, flush=True)
        got = H.gemv(a_type, tier, 1, 1.0, m, n, wh, wr, lda, x, 0.0, None, C.F64, C.F64)
        fin = np.isfinite(ref)
        assert np.array_equal(got[fin], ref[fin])
        assert np.array_equal(got[~fin], ref[~fin])


def test_gemv_t_beyond_one_grid(capi):
    """More column groups than the wave kernel's grid holds, and more columns
    than a launch of 512 threads for every four has work items for (2^32)."""
    n = (1 << 25) + 5
    A = (np.arange(n) % 251).astype(np.float32).reshape(1, n)
    got = H.gemv(C.F32, C.TIER_DEFAULT, 1, 1.0, 1, n, H.dev(A), None, 1, np.array([3.0]))
    assert np.array_equal(got, 3.0 * A[0])


@pytest.mark.parametrize("a_type", [C.F32, C.F64, C.BF16, C.FP32_16])
@pytest.mark.parametrize("n", [1, 5, 64, 300, 2000])
def test_gemv_t_in_place(capi, a_type, n):
    """y = A^T x with y over x (a square A): every product before any store."""
    rng = np.random.default_rng(n)
    A, x = rng.integers(-8, 9, (n, n)).astype(np.float32), rng.integers(-8, 9, n).astype(np.float64)
    if a_type == C.FP32_16:
        wh, wr = H.pack(C.PACK_FP32_16, A)
    else:
        wh, wr = H.dev(A.astype(np.float64) if a_type == C.F64 else bf16_bits_rne(A) if a_type == C.BF16 else A), None
    xd = H.dev(x)
    for tier in (C.TIER_DEFAULT, C.TIER_EXACT):
        C.call("tomos_memcpy_htod", xd.ptr, x.ctypes.data, x.nbytes, None)
        C.call("tomos_gemv", a_type, tier, 1, 1.0, n, n, wh.ptr, wr.ptr if wr else None, n, C.F64, xd.ptr, 0.0, C.F64,
               xd.ptr, None, 0, None)
        assert np.array_equal(xd.to_numpy(np.float64, (n,)), A.T.astype(np.float64) @ x)


@pytest.mark.parametrize("a_type", [C.F32, C.F64, C.BF16, C.FP32_16, C.FP32_BF16])
@pytest.mark.parametrize("m,n", [(1, 300001), (7, 90001), (130, 33333), (300, 20011), (1000, 6007), (4099, 3001)])
def test_gemv_n_wide(capi, orc, a_type, m, n):
    """A x of a wide matrix, whose columns are split over the grid: fewer rows
    than a vector, ragged rows and columns, an Inf, beta != 0, the caller's
    scratch of exactly the advertised size.  Entries are +-1 or 0 and |x| <= 8,
    so every sum stays below 2^24: exact."""
    rng = np.random.default_rng(m + n)
    A, x = rng.integers(-1, 2, (m, n)).astype(np.float32), rng.integers(-8, 9, n).astype(np.float64)
    A[m - 1, n - 1], x[n - 1] = np.inf, 2.0
    y0 = rng.integers(-8, 9, m).astype(np.float64)
    if a_type in FORMATS:
        wh, wr = H.pack(FORMATS[a_type][0], A)
    else:
        wh, wr = H.dev(A.astype(np.float64) if a_type == C.F64 else bf16_bits_rne(A) if a_type == C.BF16 else A), None
    with np.errstate(invalid="ignore"):
        ref = 2.0 * (A.astype(np.float64) @ x) - y0
    for tier in (C.TIER_DEFAULT, C.TIER_FAST, C.TIER_EXACT):
        print("wide", a_type, m, n, tier, flush=True)
        got = H.gemv(a_type, tier, 0, 2.0, m, n, wh, wr, m, x, -1.0, y0, C.F64, C.F64, scratch="explicit")
        assert np.array_equal(got, ref)


@pytest.mark.parametrize("a_type", [C.F32, C.BF16, C.FP32_16])
def test_gemv_n_error_of_fp32_sums(capi, orc, a_type):
    """FP32 sums of the DEFAULT tier run over at most L = 32 columns here and
    meet in FP64.  A rounding is 2^-24 / sqrt(3) rms of its partial sum at most,
    partial sums grow as sqrt(k), so a chain's error is 2^-24 sqrt(L^2 / 6)
    terms and the whole sum's, relative, 2^-24 sqrt(L / 6) = 1.38e-7."""
    m, n = 60000, 1000
    rng = np.random.default_rng(1)
    A, x = rng.standard_normal((m, n), dtype=np.float32), rng.standard_normal(n).astype(np.float32)
    if a_type == C.FP32_16:
        wh, wr = H.pack(C.PACK_FP32_16, A)
        A = orc.unpack(orc.DEC16_HALF, *orc.pack(C.PACK_FP32_16, A)).astype(np.float32)
    else:
        st = bf16_bits_rne(A) if a_type == C.BF16 else A
        wh, wr = H.dev(st), None
        A = (st.astype(np.uint32) << 16).view(np.float32) if a_type == C.BF16 else A
    got = H.gemv(a_type, C.TIER_DEFAULT, 0, 1.0, m, n, wh, wr, m, x, 0.0, None, C.F32, C.F64)
    ref = A.astype(np.float64) @ x.astype(np.float64)
    assert np.linalg.norm(got - ref) <= 2.0 ** -24 * np.sqrt(32 / 6) * np.linalg.norm(ref)


@pytest.mark.parametrize("n", [17, 64, 300, 2000])
def test_gemv_n_in_place(capi, n):
    """y = A x with y over x (a square A): every product before any store."""
    rng = np.random.default_rng(n)
    A, x = rng.integers(-8, 9, (n, n)).astype(np.float32), rng.integers(-8, 9, n).astype(np.float64)
    wh, xd = H.dev(A), H.dev(x)
    for tier in (C.TIER_DEFAULT, C.TIER_EXACT):
        C.call("tomos_memcpy_htod", xd.ptr, x.ctypes.data, x.nbytes, None)
        C.call("tomos_gemv", C.F32, tier, 0, 1.0, n, n, wh.ptr, None, n, C.F64, xd.ptr, 0.0, C.F64, xd.ptr, None, 0, None)
        assert np.array_equal(xd.to_numpy(np.float64, (n,)), A.astype(np.float64) @ x)
