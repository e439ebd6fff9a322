"""Linears on quantized weights at 17 rows and more (gemm_quant.hip): edges of the
32-row tiles, K slices, the fused epilogues, and the shapes it leaves to the
general tile kernel, against the oracle.  test_gpu_linear_tiles.py has the other
tiles."""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

import oracle
import spec_blocks as sb
from gpu_util import call, carrier, dev, f16_dev, f16_host, host, lws, ptr, stream, torch

pytestmark = pytest.mark.gpu

QTYPES = [8, 12, 14]


def _f16(a):
    return np.asarray(a, np.float32).astype(np.float16).astype(np.float32)


def _tol(W, X, ref):
    """FP16 output rounding (2^-11, doubled), 2^-14 of the dot-product mass for
    the FP32 sums and 2^-11 of it for the weights' rounding to FP16."""
    mass = np.abs(X.astype(np.float64)) @ np.abs(W.astype(np.float64)).T
    return 2.0 ** -10 * np.abs(ref) + (2.0 ** -14 + 2.0 ** -11) * mass + 1e-6


def _case(t, M, N, K, seed=0):
    rng = np.random.default_rng(seed + 1000 * t + M + N + K)
    raw, W = sb.random_matrix(rng, t, N, K)
    return carrier(t, raw, N, K), W, _f16(rng.standard_normal((M, K)))


def _linear(t, car, X, N, bias=None, ws=True, shift=0):
    M, K = X.shape
    x = torch().zeros(M * K + shift, dtype=torch().int16, device="cuda")
    x[shift:] = f16_dev(X).reshape(-1).view(torch().int16)
    y = torch().full((M * N,), -1, dtype=torch().int16, device="cuda")
    b = f16_dev(bias) if bias is not None else None
    w = lws() if ws else (None, C.c_size_t(0))
    call("bx_linear_f16", t, ptr(car), ptr(b), ptr(x[shift:]), ptr(y), M, N, K, *w, stream())
    return f16_host(y).reshape(M, N)


@pytest.mark.parametrize("t", QTYPES)
@pytest.mark.parametrize("M,N,K", [(17, 1, 256), (32, 127, 768), (33, 130, 2560), (64, 129, 512), (65, 260, 1024),
                                   (97, 3, 6144), (129, 258, 4096), (200, 2050, 768), (300, 513, 3072)])
def test_quant_tiles_vs_oracle(t, M, N, K):
    """Partial row and column tiles, odd columns (scalar stores, odd scale
    counts), one block of K and many; with the workspace (K slices) and
    without (one slice); a second launch gives the same bits."""
    print(f"[quant tiles] t={t} M={M} N={N} K={K}", flush=True)
    car, W, X = _case(t, M, N, K)
    bias = _f16(np.random.default_rng(1).standard_normal(N))
    ref = oracle.linear(W, X) + bias
    tol = _tol(W, X, ref)
    got = _linear(t, car, X, N, bias)
    assert np.all(np.abs(got - ref) <= tol), float((np.abs(got - ref) / tol).max())
    assert np.array_equal(got, _linear(t, car, X, N, bias))
    one = _linear(t, car, X, N, bias, ws=False)
    assert np.all(np.abs(one - ref) <= tol), float((np.abs(one - ref) / tol).max())


@pytest.mark.parametrize("t", QTYPES)
@pytest.mark.parametrize("M", [37, 512])
def test_quant_tiles_multiply_the_dequantized_weights(t, M):
    """Rows that pick one element of K each return the weights themselves: the
    bits of bx_dequant_to_f16, also of weights near zero (blocks whose scale
    times code all but cancels the minimum among them)."""
    print(f"[quant weights] t={t} M={M}", flush=True)
    N, K = 300, 512
    rng = np.random.default_rng(60 + t)
    raw = bytearray(sb.random_matrix(rng, t, N, K)[0])
    if t == 12:   # d and dmin such that d * sc * q passes close to dmin * m
        blocks = np.frombuffer(raw, np.uint8).reshape(-1, 144)
        blocks[::2, 0:4] = np.array([0.0101, 0.0477], np.float16).view(np.uint8)
    car = carrier(t, bytes(raw), N, K)
    W = torch().empty(N * K, dtype=torch().int16, device="cuda")
    call("bx_dequant_to_f16", t, ptr(car), ptr(W), N, K, stream())
    W = f16_host(W).reshape(N, K)
    for k0 in range(0, K, M):
        X = np.zeros((M, K), np.float32)
        n = min(M, K - k0)
        X[np.arange(n), k0 + np.arange(n)] = 1
        got = _linear(t, car, X, N)
        assert np.array_equal(got[:n], W[:, k0:k0 + n].T), int((got[:n] != W[:, k0:k0 + n].T).sum())


@pytest.mark.parametrize("t", QTYPES)
def test_quant_tiles_misaligned_x_takes_the_general_kernel(t):
    """Rows that do not start on 16 bytes: the copies of 16 bytes do not take
    them; the result stays."""
    M, N, K = 150, 300, 512
    car, W, X = _case(t, M, N, K)
    ref = oracle.linear(W, X)
    for shift in (0, 2, 4):
        got = _linear(t, car, X, N, shift=shift)
        assert np.all(np.abs(got - ref) <= _tol(W, X, ref)), shift


@pytest.mark.parametrize("t", QTYPES)
def test_quant_tiles_infinite_and_nan_rows_stay_in_their_rows(t):
    """A row of X with an infinity or a NaN (and the rows that repeat the last
    one to fill a tile) changes its own outputs only."""
    M, N, K = 70, 140, 512
    car, W, X = _case(t, M, N, K)
    clean = _linear(t, car, X, N)
    bad = X.copy()
    bad[5, 7], bad[M - 1, 300] = np.inf, np.nan
    got = _linear(t, car, bad, N)
    keep = [m for m in range(M) if m not in (5, M - 1)]
    assert np.array_equal(got[keep], clean[keep])
    assert np.isnan(got[M - 1]).all() and not np.isfinite(got[5]).any()


@pytest.mark.parametrize("t", QTYPES)
@pytest.mark.parametrize("M,K,Ns", [(130, 6144, (257, 130, 130)), (200, 1024, (384, 127, 127))])
def test_quant_fused_epilogues_vs_oracle(t, M, K, Ns):
    """q / k / v in one launch, the residual add and SwiGLU, where the tiles
    are few enough to split K."""
    print(f"[quant fused] t={t} M={M} K={K}", flush=True)
    cars, Ws = zip(*[_case(t, M, n, K, seed=i)[:2] for i, n in enumerate(Ns)])
    X = _case(t, M, Ns[0], K)[2]
    # projections of magnitude about 8, so that gate * up stays in FP16's range
    X = _f16(X * (8 / max(np.abs(oracle.linear(W, X)).max() for W in Ws)))
    x = f16_dev(X)
    refs = [oracle.linear(W, X) for W in Ws]
    ys = [torch().empty(M * n, dtype=torch().int16, device="cuda") for n in Ns]
    call("bx_linear_group_f16", t, 3, (C.c_void_p * 3)(*[ptr(c) for c in cars]), (C.c_void_p * 3)(*[ptr(y) for y in ys]),
         (C.c_int * 3)(*Ns), ptr(x), M, K, *lws(), stream())
    for y, W, n, ref in zip(ys, Ws, Ns, refs):
        assert np.all(np.abs(f16_host(y).reshape(M, n) - ref) <= _tol(W, X, ref))
    H0 = np.random.default_rng(3).standard_normal((M, Ns[0])).astype(np.float32)
    H = dev(H0)
    call("bx_linear_residual_f16", t, ptr(cars[0]), ptr(x), ptr(H), M, Ns[0], K, *lws(), stream())
    assert np.all(np.abs(host(H).reshape(M, -1) - H0 - refs[0]) <= _tol(Ws[0], X, refs[0]) + 2.0 ** -22 * np.abs(H0))
    act = torch().empty(M * Ns[1], dtype=torch().int16, device="cuda")
    call("bx_linear_swiglu_f16", t, ptr(cars[1]), ptr(cars[2]), ptr(x), ptr(act), M, Ns[1], K, *lws(), stream())
    g, u = refs[1].astype(np.float64), refs[2].astype(np.float64)
    sg = 1 / (1 + np.exp(-g))
    ref = g * sg * u
    # each factor's own error, and the roundings of g, silu(g), u and the product
    tol = (np.abs(u) * 1.1 * _tol(Ws[1], X, g) + np.abs(g * sg) * _tol(Ws[2], X, u) +
           _tol(Ws[1], X, g) * _tol(Ws[2], X, u) * 1.1 + 2.0 ** -9 * np.abs(ref) + 1e-6)
    got = f16_host(act).reshape(M, Ns[1])
    assert np.all(np.abs(got - ref) <= tol), float((np.abs(got - ref) / tol).max())


@pytest.mark.parametrize("t", QTYPES)
@pytest.mark.parametrize("M,K,N", [(128, 2048, 2048), (128, 1024, 3072), (160, 1024, 3072), (300, 2048, 1024), (511, 4096, 130),
                                   (200, 1280, 258), (150, 6144, 300), (129, 768, 98), (140, 14336, 64)])
def test_quant_residual_and_swiglu_have_the_bits_of_the_separate_ops(t, M, K, N):
    """Both add an output's K slices in the order of the plain launch, whatever
    tiles they take."""
    print(f"[quant fused bits] t={t} M={M} K={K} N={N}", flush=True)
    rng = np.random.default_rng(M + K)
    ws = [carrier(t, sb.random_blocks(rng, t, N * K // sb.QK[t])[0], N, K) for _ in range(2)]
    x = f16_dev(rng.standard_normal((M, K)) * 0.02)
    sep = [torch().empty(M * N, dtype=torch().int16, device="cuda") for _ in range(3)]
    for w, y in zip(ws, sep):
        call("bx_linear_f16", t, ptr(w), None, ptr(x), ptr(y), M, N, K, *lws(), stream())
    assert np.isfinite(f16_host(sep[0])).all()
    H0 = rng.standard_normal((M, N)).astype(np.float32)
    H = dev(H0)
    call("bx_linear_residual_f16", t, ptr(ws[0]), ptr(x), ptr(H), M, N, K, *lws(), stream())
    assert np.array_equal(host(H).reshape(M, -1), H0 + f16_host(sep[0]).reshape(M, -1))
    call("bx_linear_swiglu_f16", t, ptr(ws[0]), ptr(ws[1]), ptr(x), ptr(sep[2]), M, N, K, *lws(), stream())
    call("bx_silu_f16", ptr(sep[0]), ptr(sep[0]), M * N, stream())
    call("bx_mul_f16", ptr(sep[0]), ptr(sep[1]), M * N, stream())
    assert np.array_equal(host(sep[2]), host(sep[0]))
