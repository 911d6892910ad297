"""The prefill's product on fp16 planes (csrc/split_gemm.hip) by itself: split_rows,
split_decode and split_gemm called through their symbols, against 64-bit products of the
decoded weights and, where a row is not finite, against the fp32 product
(csdr_dense_linear_ex) in value and in which outputs are infinite or NaN.

Bars. A plane pair holds a value to 2^-23 of itself, and with lo at 2^12 times its size that
holds down to 2^-27 of the row's largest value; the left-out lo . lo term is at most 2^-22 of a
product; products are exact and sums fp32. So the relative L2 error is a few 2^-24, like an fp32
product's: 1e-6 leaves room for the order of the sums, and it may not be more than the fp32
matrix-core product's own error on the same inputs.
"""
import ctypes as C

import numpy as np
import pytest

from conftest import rel_l2

pytestmark = pytest.mark.gpu

PLAIN, RMS_NORM, SILU_MUL = 0, 1, 2


class Planes(C.Structure):
    _fields_ = [("hi", C.c_void_p), ("lo", C.c_void_p), ("inv", C.c_void_p), ("ld", C.c_int)]


def _symbols():
    from cortexsdr_amd import _lib

    lib = _lib.load()
    P, I = C.c_void_p, C.c_int
    rows = lib._ZN4csdr10split_rowsENS_7SplitOpEPfPKfS3_iiifRKNS_11SplitPlanesEP12ihipStream_t
    rows.argtypes = [I, P, P, P, I, I, I, C.c_float, P, P]
    dec = lib._ZN4csdr12split_decodeEiPKPK9csdr_hsdbPKNS_11SplitPlanesEP12ihipStream_t
    dec.argtypes = [I, P, P, P]
    gemm = lib._ZN4csdr10split_gemmEiPKNS_11SplitPlanesEPKiRS1_iPKPfPKPKfiP12ihipStream_t
    gemm.argtypes = [I, P, P, P, I, P, P, I, P]
    return _lib, lib, rows, dec, gemm


def _planes(gpu, rows, ld):
    hi = gpu.empty(rows, ld, dtype=gpu.float16, device="cuda")
    lo = gpu.empty_like(hi)
    inv = gpu.empty(rows, device="cuda")
    return Planes(hi.data_ptr(), lo.data_ptr(), inv.data_ptr(), ld), (hi, lo, inv)


def split_product(gpu, segs, x, splits=1, bias=None, op=PLAIN, x2=None, eps=0.0):
    """[op(x) . W^T (+ bias)] of the segments, x (M x C) fp32 on the device."""
    L, lib, rows, dec, gemm = _symbols()
    M, Cc = x.shape
    ld = (Cc + 63) // 64 * 64
    st = int(gpu.cuda.current_stream().cuda_stream)
    xp, keep = _planes(gpu, M, ld)
    n = len(segs)
    assert 1 <= n <= 3 and all(s.cols == Cc for s in segs)
    L.check(rows(op, x.data_ptr(), x2.data_ptr() if x2 is not None else None, None, 0, M, Cc, eps,
                 C.addressof(xp), st))
    wp = (Planes * n)()
    keeps = []
    for i, s in enumerate(segs):
        wp[i], k = _planes(gpu, s.rows, ld)
        keeps.append(k)
    L.check(dec(n, (C.c_void_p * n)(*[s._h.value for s in segs]), wp, st))
    ys = [gpu.full((splits, M, s.rows), float("nan"), device="cuda") for s in segs]
    R = (C.c_int * n)(*[s.rows for s in segs])
    bp = (C.c_void_p * n)(*[b.data_ptr() if b is not None else None for b in bias]) if bias else None
    L.check(gemm(n, wp, R, C.addressof(xp), M, (C.c_void_p * n)(*[y.data_ptr() for y in ys]), bp,
                 splits, st))
    gpu.cuda.synchronize()
    del keep, keeps
    return [y.sum(0) for y in ys]


def randn(gpu, *shape):
    g = gpu.Generator(device="cuda").manual_seed(sum(shape))
    return gpu.randn(*shape, generator=g, device="cuda")


def fp32_product(gpu, w, x):
    L, lib, *_ = _symbols()
    y = gpu.empty(x.shape[0], w.shape[0], device="cuda")
    L.check(lib.csdr_dense_linear_ex(w.data_ptr(), w.shape[0], w.shape[1], x.data_ptr(),
                                     x.shape[0], y.data_ptr(), None, 0,
                                     int(gpu.cuda.current_stream().cuda_stream)))
    return y


def segment(R, Cc, K=96, nnz=8, seed=3, D=None, edge=None, coef=None, sigma=0.1):
    from cortexsdr_amd import formats, synth
    from cortexsdr_amd.hsdr import HsdbSegment

    rng = np.random.default_rng(seed)
    if D is None:
        D = synth.dictionary(K, 64, seed)
    n = R * (Cc // 64)
    idx = rng.integers(0, D.shape[0], (n, nnz)).astype(np.uint16)
    if coef is None:
        coef = (rng.standard_normal((n, nnz)) * sigma).astype(np.float16)
    ce = Cc % 64
    if ce and edge is None:
        edge = (rng.standard_normal((R, ce)) * 0.1).astype(np.float32)
    return HsdbSegment(formats.pack_hsdb(R, Cc, D, idx, coef, edge=edge))


def check64(gpu, segs, x, ys, label):
    for s, y in zip(segs, ys):
        w = s.decompress()
        want = (x.double() @ w.double().T).cpu().numpy()
        err = rel_l2(y.cpu().numpy(), want)
        err32 = rel_l2(fp32_product(gpu, w, x).cpu().numpy(), want)
        print(f"{label} R={s.rows}: {err:.2e} (fp32 matrix cores {err32:.2e})")
        assert err <= 1e-6
        # (a tenth for the draw of the inputs; below 1e-7 both are the last bits of a few sums)
        assert err <= max(1.1 * err32, 1e-7)


# tiles per decoding thread 1, 2, 5, 11 and 16 (up to 256 tiles), edge strips, one to three
# matrices, every tile of the product (few rows: 64 x 32 and 64 x 64; 4864 and more: 128 x 64),
# parts of the contraction, row buffers past 60 KiB of LDS (15,361 columns on)
@pytest.mark.parametrize("Cc,Rs,M,nnz,splits", [
    (100, (37,), 8, 4, 1), (1000, (70, 5, 5), 33, 8, 2), (1024, (130,), 65, 16, 4),
    (2048, (66, 3), 9, 6, 3), (896, (896, 128, 128), 300, 8, 1), (896, (4864, 4864), 70, 8, 1),
    (4864, (896,), 140, 8, 8), (5120, (40,), 20, 8, 8), (5184, (33,), 12, 4, 1),
    (11008, (65, 31), 17, 8, 8), (11264, (20,), 40, 16, 7), (11300, (70,), 9, 3, 1),
    (15361, (34,), 10, 8, 8), (16384, (66,), 66, 8, 8),
])
def test_against_64_bits(gpu, Cc, Rs, M, nnz, splits):
    segs = [segment(R, Cc, nnz=nnz, seed=Cc + i) for i, R in enumerate(Rs)]
    g = gpu.Generator(device="cuda").manual_seed(Cc * 31 + M)
    x = gpu.randn(M, Cc, generator=g, device="cuda")
    ys = split_product(gpu, segs, x, splits)
    check64(gpu, segs, x, ys, f"C={Cc} M={M} slots={nnz} parts={splits}")
    if splits == 1:
        bias = [gpu.randn(R, generator=g, device="cuda") for R in Rs]
        for y, yb, b in zip(ys, split_product(gpu, segs, x, 1, bias), bias):
            assert gpu.equal(yb, y + b)


@pytest.mark.parametrize("op", [RMS_NORM, SILU_MUL])
def test_row_ops(gpu, op):
    M, Cc, eps = 21, 1100, 1e-5
    seg = segment(90, Cc)
    x = randn(gpu, M, Cc)
    x2 = randn(gpu, Cc) if op == RMS_NORM else randn(gpu, M + 1, Cc)[1:]
    xd = x.double()
    if op == RMS_NORM:
        t = xd / (xd.square().mean(1, keepdim=True) + eps).sqrt() * x2.double()
    else:
        t = gpu.nn.functional.silu(xd) * x2.double()
    want = t @ seg.decompress().double().T
    y = split_product(gpu, [seg], x, op=op, x2=x2, eps=eps)[0]
    assert rel_l2(y.cpu().numpy(), want.cpu().numpy()) <= 1e-6


@pytest.mark.parametrize("ratio", [2.0 ** 8, 2.0 ** 16, 2.0 ** 24, 2.0 ** 27])
def test_rows_of_mixed_magnitude(gpu, ratio):
    """One value of a row `ratio` times the others, met by zeros in the other operand: what is
    left is the rest's product, to fp32's precision. x's large values stand where every atom is
    zero, W's (edge strip) where x is."""
    from cortexsdr_amd import synth

    D = synth.dictionary(96, 64, 5)
    D[:, 7] = 0.0
    R, Cc, M = 70, 896 + 32, 40
    rng = np.random.default_rng(9)
    edge = rng.standard_normal((R, 32)).astype(np.float32) * 0.1
    edge[:, 11] *= np.float32(ratio)
    seg = segment(R, Cc, D=D, edge=edge)
    x = randn(gpu, M, Cc)
    x[:, 7] *= ratio
    x[:, 64 + 7] = -ratio
    x[:, 896 + 11] = 0.0
    check64(gpu, [seg], x, split_product(gpu, [seg], x), f"ratio={ratio:g}")


@pytest.mark.parametrize("xs,ws", [(2.0 ** -118, 1.0), (2.0 ** 118, 2.0 ** -20), (2.0 ** -125, 2.0 ** 13),
                                   (1e-30, 1e4)])
def test_rows_of_extreme_magnitude(gpu, xs, ws):
    """Whole rows near the ends of fp32's range: no overflow or underflow on the way to results
    that fp32 holds."""
    R, Cc, M = 66, 640 + 16, 20
    rng = np.random.default_rng(2)
    # the edge strip carries W's scale (coefficients are fp16); atoms' coefficients zero
    edge = (rng.standard_normal((R, 16)) * ws).astype(np.float32)
    seg = segment(R, Cc, edge=edge, coef=np.zeros((R * 10, 8), np.float16))
    x = randn(gpu, M, Cc) * xs
    check64(gpu, [seg], x, split_product(gpu, [seg], x), f"x={xs:g} w={ws:g}")


@pytest.mark.parametrize("splits", [1, 4])
def test_rows_that_are_not_finite(gpu, splits):
    """NaN and infinities in rows of X, in coefficients and in the edge strip, beside finite
    rows: the outputs are those of the fp32 product, infinite and NaN where its are."""
    R, Cc, M = 70, 1000, 40
    rng = np.random.default_rng(4)
    edge = (rng.standard_normal((R, 40)) * 0.1).astype(np.float32)
    edge[3, 5], edge[9, 0], edge[20, 39] = np.inf, np.nan, -np.inf
    coef = (rng.standard_normal((R * 15, 8)) * 0.1).astype(np.float16)
    coef[15 * 33 + 2, 1] = np.inf
    seg = segment(R, Cc, edge=edge, coef=coef)
    x = randn(gpu, M, Cc)
    x[2, 17], x[5, 999], x[6, 0] = float("inf"), float("nan"), -float("inf")
    x[11] = 0.0          # a zero row against infinite weights: NaN
    x[12, 960 + 5] = 0.0
    got = split_product(gpu, [seg], x, splits)[0].cpu().numpy()
    want = fp32_product(gpu, seg.decompress(), x).cpu().numpy()
    assert np.array_equal(np.isnan(got), np.isnan(want))
    assert np.array_equal(np.isinf(got), np.isinf(want))
    assert np.array_equal(got[np.isinf(got)], want[np.isinf(want)])
    ok = np.isfinite(want)
    assert ok.sum() > R * M // 2 and not ok.all()
    assert rel_l2(got[ok], want[ok]) <= 1e-6
