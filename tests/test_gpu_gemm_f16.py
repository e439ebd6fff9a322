"""Linears on FP16 weights at 17 rows and more (gemm_f16.hip): the epilogues at
partial tiles, and operands and shapes it leaves to the general kernels.
test_gpu_linear_tiles.py has every tile shape."""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

from gpu_util import call, dev, f16_dev, f16_host, host, lws, ptr, stream, torch

pytestmark = pytest.mark.gpu


def _f16(a):
    return np.asarray(a, np.float32).astype(np.float16).astype(np.float32)


def _tol(W, X, ref):
    """FP16 output rounding (2^-11, doubled) and 2^-14 of the dot-product mass
    for the FP32 sums."""
    mass = np.abs(X.astype(np.float64)) @ np.abs(W.astype(np.float64)).T
    return 2.0 ** -10 * np.abs(ref) + 2.0 ** -14 * mass + 1e-6


def _rand(M, N, K, n=1):
    rng = np.random.default_rng(M + N + K)
    return _f16(rng.standard_normal((M, K))), [_f16(rng.standard_normal((N, K)) * 0.05) for _ in range(n)]


def _ref(X, W):
    return X.astype(np.float64) @ W.astype(np.float64).T


# on 256 CUs: 64 x 64 tiles of gemm_f16.hip and (from 128 rows, K to 1024) of
# gemm.hip, 128 x 128 (one and two workgroups per CU) and 256 x 256, partial tiles
SHAPES = [(17, 1, 64), (63, 65, 128), (65, 130, 192), (129, 2049, 64), (385, 4100, 640), (700, 4097, 448),
          (2049, 1025, 512), (1100, 9000, 320), (1281, 12295, 256)]


@pytest.mark.parametrize("M,N,K", SHAPES)
def test_f16_tiles(M, N, K):
    print(f"[f16 tiles] M={M} N={N} K={K}", flush=True)
    X, (W,) = _rand(M, N, K)
    bias = _f16(np.random.default_rng(1).standard_normal(N))
    ref = _ref(X, W) + bias
    tol = _tol(W, X, ref)
    w, b, x = f16_dev(W), f16_dev(bias), f16_dev(X)
    y = torch().full((M * N + 8,), -1, dtype=torch().int16, device="cuda")
    call("bx_linear_f16", 1, ptr(w), ptr(b), ptr(x), ptr(y), M, N, K, *lws(), stream())
    got = f16_host(y[:M * N]).reshape(M, N)
    assert np.all(np.abs(got - ref) <= tol), float((np.abs(got - ref) / tol).max())
    assert (host(y[M * N:]) == -1).all()    # nothing past the output
    H0 = np.random.default_rng(2).standard_normal((M, N)).astype(np.float32)
    if M >= 128:
        H = dev(H0)
        call("bx_linear_residual_f16", 1, ptr(w), ptr(x), ptr(H), M, N, K, *lws(), stream())
        # the same projection rounded to FP16, then one FP32 add
        plain = torch().empty(M * N, dtype=torch().int16, device="cuda")
        call("bx_linear_f16", 1, ptr(w), None, ptr(x), ptr(plain), M, N, K, *lws(), stream())
        assert np.array_equal(host(H).reshape(M, N), H0 + f16_host(plain).reshape(M, N))


@pytest.mark.parametrize("M,F,K", [(128, 33, 64), (200, 1000, 192), (520, 3072, 128), (777, 4099, 64)])
def test_f16_swiglu_and_group_equal_the_separate_ops(M, F, K):
    X, (Wg, Wu) = _rand(M, F, K, 2)
    x, g, u = f16_dev(X), f16_dev(Wg), f16_dev(Wu)
    new = lambda: torch().empty(M * F, dtype=torch().int16, device="cuda")
    act, yg, yu, sep = new(), new(), new(), [new(), new()]
    call("bx_linear_swiglu_f16", 1, ptr(g), ptr(u), ptr(x), ptr(act), M, F, K, *lws(), stream())
    call("bx_linear_group_f16", 1, 2, (C.c_void_p * 2)(ptr(g), ptr(u)), (C.c_void_p * 2)(ptr(yg), ptr(yu)),
         (C.c_int * 2)(F, F), ptr(x), M, K, *lws(), stream())
    for w, y in zip((g, u), sep):
        call("bx_linear_f16", 1, ptr(w), None, ptr(x), ptr(y), M, F, K, *lws(), stream())
    assert np.array_equal(host(yg), host(sep[0])) and np.array_equal(host(yu), host(sep[1]))
    call("bx_silu_f16", ptr(sep[0]), ptr(sep[0]), M * F, stream())
    call("bx_mul_f16", ptr(sep[0]), ptr(sep[1]), M * F, stream())
    assert np.array_equal(host(act), host(sep[0]))


@pytest.mark.parametrize("xs,ws,ys", [(2, 0, 0), (0, 4, 0), (0, 0, 1), (0, 0, 4)])
def test_f16_tiles_misaligned_operands(xs, ws, ys):
    """Operands off a 16-byte boundary (elements xs, ws) take the general
    kernel; an output off it (ys) takes narrower stores."""
    M, N, K = 150, 200, 128
    X, (W,) = _rand(M, N, K)
    x, w = (torch().zeros(a.size + 8, dtype=torch().int16, device="cuda") for a in (X, W))
    x[xs:xs + X.size] = f16_dev(X).reshape(-1).view(torch().int16)
    w[ws:ws + W.size] = f16_dev(W).reshape(-1).view(torch().int16)
    y = torch().full((M * N + 16,), -1, dtype=torch().int16, device="cuda")
    call("bx_linear_f16", 1, ptr(w[ws:]), None, ptr(x[xs:]), ptr(y[ys:]), M, N, K, *lws(), stream())
    ref = _ref(X, W)
    got = f16_host(y[ys:ys + M * N].clone()).reshape(M, N)
    assert np.all(np.abs(got - ref) <= _tol(W, X, ref))
    assert (host(y[:ys]) == -1).all() and (host(y[ys + M * N:]) == -1).all()
