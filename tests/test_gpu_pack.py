"""GPU pack / decode: bit-exact against the CPU oracle encoders/decoders.

Inputs: a strided sweep of 2^26 fp32 bit patterns (every 64-pattern block of
the 2^32 space, every exponent, signs, zeros, subnormals, Inf, NaN) plus all
2^16 wh words for the wh-only decoders.
"""
import ctypes

import numpy as np
import pytest

from tests import hipcall as H
from tomos_amd import _capi as C

pytestmark = pytest.mark.gpu


def sweep_bits(n_log2=26, seed=0):
    i = np.arange(1 << n_log2, dtype=np.uint64)
    rng = np.random.default_rng(seed)
    low = rng.integers(0, 1 << (32 - n_log2), size=i.size, dtype=np.uint64)
    bits = ((i << np.uint64(32 - n_log2)) | low).astype(np.uint32)
    return bits.view(np.float32)


ENCODERS = [
    (C.PACK_FP32_16, 0), (C.PACK_FP32_16_CLAMPED, 1), (C.PACK_FP32_16_TRUNCATED, 2),
    (C.PACK_FP32_BF16, 3), (C.PACK_FP32_BF16_ROUNDED, 4),
]


@pytest.mark.parametrize("variant,orc_variant", ENCODERS)
def test_pack_bit_exact_sweep(capi, orc, variant, orc_variant):
    print("pack sweep variant", variant, flush=True)
    v = sweep_bits()
    m = 1 << 13
    n = v.size // m
    A = v.reshape(n, m).T  # (m, n) view
    wh, wr = H.pack(variant, A)
    gh = H.from_dev16(wh, m, n)
    gr = H.from_dev16(wr, m, n)
    eh, er = orc.pack(orc_variant, A)
    assert np.array_equal(gh, eh), np.argwhere(gh != eh)[:5]
    assert np.array_equal(gr, er), np.argwhere(gr != er)[:5]


@pytest.mark.parametrize("ld_pad", [0, 5, 8])
def test_pack_strided_and_ragged(capi, orc, ld_pad):
    rng = np.random.default_rng(3)
    m, n = 1001, 7
    A = (rng.standard_normal((m, n)) * 2.0 ** rng.integers(-30, 30, (m, n))).astype(np.float32)
    ld = m + ld_pad
    for variant in range(5):
        wh, wr = H.pack(variant, A, ld=ld)
        gh = H.from_dev16(wh, ld, n)[:m]
        gr = H.from_dev16(wr, ld, n)[:m]
        eh, er = orc.pack(variant, A)
        assert np.array_equal(gh, eh) and np.array_equal(gr, er), variant


DECODERS = [
    C.DECODE_FP32_16_EXACT, C.DECODE_FP32_16_HALF, C.DECODE_FP32_16_HALF_FAST,
    C.DECODE_FP32_16_BF16, C.DECODE_FP32_BF16_EXACT, C.DECODE_FP32_BF16_HI,
    C.DECODE_FP32_BF16_EXACT_ROUNDED, C.DECODE_FP32_16_EXACT_TRUNCATED,
]


@pytest.mark.parametrize("dec", DECODERS)
def test_unpack_bit_exact(capi, orc, dec):
    print("unpack decoder", dec, flush=True)
    v = sweep_bits(22, seed=dec)
    m = 1 << 11
    n = v.size // m
    A = v.reshape(n, m).T
    enc = {0: 0, 1: 0, 2: 0, 3: 0, 4: 3, 5: 3, 6: 4, 7: 2}[dec]
    eh, er = orc.pack(enc, A)
    dh, dr = H.dev(eh), H.dev(er)
    out = H.DeviceBuffer(m * n * 4)
    C.call("tomos_unpack", dec, m, n, dh.ptr, dr.ptr, m, out.ptr, m, None)
    got = out.to_numpy(np.float32, (m, n)).view(np.uint32)
    exp = orc.unpack(dec, eh, er).view(np.uint32)
    assert np.array_equal(got, exp), np.argwhere(got != exp)[:5]


@pytest.mark.parametrize("dec,fn", [
    (C.DECODE_FP32_16_HALF, "orc_fp32_16_half_only"),
    (C.DECODE_FP32_16_HALF_FAST, "orc_fp32_16_half_only_fast"),
    (C.DECODE_FP32_16_BF16, "orc_fp32_16_bf16_only"),
])
def test_decode_wh_all_words(capi, orc, dec, fn):
    words = np.arange(1 << 16, dtype=np.uint16)
    d = H.dev(words)
    out = H.DeviceBuffer(words.nbytes)
    C.call("tomos_decode_wh", dec, words.size, d.ptr, out.ptr, None)
    got = out.to_numpy(np.uint16, (words.size,))
    f = getattr(orc.lib(), fn)
    exp = np.array([f(int(w)) for w in words], dtype=np.uint16)
    if dec == C.DECODE_FP32_16_BF16:
        # control=0 words whose fp16 value is NaN (exponent field 31, never
        # produced by the encoders) may differ only in the NaN payload
        nan = ((words & 1) == 0) & (((words >> 10) & 0x1F) == 0x1F) & ((words & 0x3FF) != 0)
        assert np.array_equal(got[~nan], exp[~nan])
        assert np.all((got[nan] & 0x7F80) == 0x7F80) and np.all((got[nan] & 0x7F) != 0)
    else:
        assert np.array_equal(got, exp)


@pytest.mark.parametrize("m,n", [(1, 1), (7, 3), (8, 2), (9, 5), (2047, 2), (2049, 3)])
@pytest.mark.parametrize("pad", [0, 1, 8])
def test_unpack_runs_and_remainders(capi, orc, m, n, pad):
    """Every decoder on rows that end inside a run of 8, columns without
    padding (one long column), at odd and at aligned leading dimensions; words
    of every class, saturated ones among them; nothing is written past row m."""
    rng = np.random.default_rng(m + pad)
    A = (rng.standard_normal((m, n)) * 2.0 ** rng.integers(-34, 34, (m, n))).astype(np.float32)
    ld = m + pad
    for variant, decs in ((0, (0, 1, 2, 3)), (2, (7,)), (3, (4, 5)), (4, (6,))):
        eh, er = orc.pack(variant, A)
        sh, sr = np.full((ld, n), 0x7FFF, np.uint16, order="F"), np.full((ld, n), 0x7FFF, np.uint16, order="F")
        sh[:m], sr[:m] = eh, er
        wh, wr = H.dev(sh), H.dev(sr)
        for dec in decs:
            print("unpack", variant, dec, m, n, pad, flush=True)
            out = H.dev(np.full((ld, n), -7.0, np.float32))
            C.call("tomos_unpack", dec, m, n, wh.ptr, wr.ptr, ld, out.ptr, ld, None)
            got = out.to_numpy(np.float32, (ld, n))
            exp = orc.unpack(dec, eh, er)
            assert np.array_equal(got[:m].view(np.uint32), np.ascontiguousarray(exp).astype(np.float32).view(np.uint32)), dec
            assert np.all(got[m:] == -7.0)


@pytest.mark.parametrize("m,n,pad_src,pad_dst,shift", [(1, 1, 0, 0, 0), (7, 65, 0, 3, 1), (128, 64, 0, 0, 0),
                                                        (129, 63, 5, 7, 2), (127, 66, 1, 1, 3), (300, 3, 0, 4, 1),
                                                        (260, 200, 2, 0, 0)])
def test_pack_rows_equals_pack(capi, orc, m, n, pad_src, pad_dst, shift):
    """A row-major source packs to the same words as its columns, at tile
    edges and remainders, odd leading dimensions and a source at any element;
    nothing is written past row m or column n."""
    rng = np.random.default_rng(m * n)
    A = (rng.standard_normal((m, n)) * 2.0 ** rng.integers(-34, 34, (m, n))).astype(np.float32)
    A.flat[::7] = rng.choice(np.array([0.0, -0.0, np.inf, -np.inf, np.nan, 1e-45, 65520.0], np.float32), A.flat[::7].size)
    lds, ld = n + pad_src, m + pad_dst
    flat = np.full(shift + m * lds, 3.0, np.float32)
    flat[shift:].reshape(m, lds)[:, :n] = A
    src = H.dev(flat)
    cols = H.dev(np.asfortranarray(A))
    for variant in range(5):
        print("pack_rows", variant, m, n, lds, ld, shift, flush=True)
        outs = []
        for entry in ("tomos_pack_rows", "tomos_pack"):
            wh, wr = (H.dev(np.full(ld * (n + 1), 0x1234, np.uint16)) for _ in range(2))
            rows = entry == "tomos_pack_rows"
            C.call(entry, variant, m, n, src.ptr + 4 * shift if rows else cols.ptr, lds if rows else m, wh.ptr, wr.ptr,
                   ld, None)
            outs.append([x.to_numpy(np.uint16, (ld * (n + 1),)) for x in (wh, wr)])
        assert np.array_equal(outs[0][0], outs[1][0]) and np.array_equal(outs[0][1], outs[1][1]), variant
    assert C.lib().tomos_pack_rows(0, m, n, ctypes.c_void_p(src.ptr), n - 1, ctypes.c_void_p(src.ptr),
                                   ctypes.c_void_p(src.ptr), ld, None) == 1


@pytest.mark.parametrize("m", [1, 7, 8, 9, 16, 17, 100, 1024, 1025])
@pytest.mark.parametrize("n", [2, 31, 257])
def test_short_padded_columns(capi, orc, m, n):
    """Several columns a block: row counts around the powers of two that halve
    a column's share of the block, column counts that leave part of one, odd
    leading dimensions; nothing is written past row m."""
    rng = np.random.default_rng(m * n)
    A = (rng.standard_normal((m, n)) * 2.0 ** rng.integers(-30, 30, (m, n))).astype(np.float32)
    lds, ld = m + 3, m + 5
    src = np.full((lds, n), 5.0, np.float32, order="F")
    src[:m] = A
    print("short columns", m, n, flush=True)
    for variant, dec in ((0, 0), (3, 4)):
        eh, er = orc.pack(variant, A)
        wh, wr = H.dev(np.full((ld, n), 0x1111, np.uint16)), H.dev(np.full((ld, n), 0x1111, np.uint16))
        sd = H.dev(src)
        C.call("tomos_pack", variant, m, n, sd.ptr, lds, wh.ptr, wr.ptr, ld, None)
        gh, gr = H.from_dev16(wh, ld, n), H.from_dev16(wr, ld, n)
        assert np.array_equal(gh[:m], eh) and np.array_equal(gr[:m], er)
        assert np.all(gh[m:] == 0x1111) and np.all(gr[m:] == 0x1111)
        out = H.dev(np.full((lds, n), -7.0, np.float32))
        C.call("tomos_unpack", dec, m, n, wh.ptr, wr.ptr, ld, out.ptr, lds, None)
        got = out.to_numpy(np.float32, (lds, n))
        assert np.array_equal(got[:m].view(np.uint32), orc.unpack(dec, eh, er).astype(np.float32).view(np.uint32))
        assert np.all(got[m:] == -7.0)
