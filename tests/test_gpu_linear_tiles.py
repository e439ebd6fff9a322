"""Every tile of the 17-row-and-up linears, at partial tiles and several steps of
K: plain launches against float64, residual and SwiGLU launches against the
separate ops bit for bit."""
from __future__ import annotations

import pytest

import tile_cases as tc
from gpu_util import call, lws, ptr, stream, torch

pytestmark = pytest.mark.gpu

# bytes of a block, its elements, and where its FP16 scales sit
BLOCK = {8: (34, 32, (0,)), 12: (144, 256, (0, 2)), 14: (210, 256, (208,))}


def _weight(t, N, K, gen):
    """(carrier, float64 values) of random codes with scales near 0.0001."""
    T = torch()
    if t == 1:
        w = T.randn(N, K, generator=gen, device="cuda", dtype=T.float16) * 0.05
        return w, w.double()
    size, elems, scales = BLOCK[t]
    raw = T.randint(0, 256, (N * K // elems, size), generator=gen, device="cuda", dtype=T.uint8)
    for at in scales:
        d = (T.rand(len(raw), generator=gen, device="cuda") + 0.5) * 1e-4
        raw[:, at:at + 2] = d.half().view(T.uint8).reshape(-1, 2)
    car = T.empty_like(raw)
    call("bx_repack_gguf_rows", t, ptr(raw), ptr(car), N, K, stream())
    w = T.empty(N, K, dtype=T.float32, device="cuda")
    call("bx_dequant_to_f32", t, ptr(car), ptr(w), N, K, stream())
    return car, w.double()


@pytest.mark.parametrize("t,form,rows,cols,more,M,N,K", tc.params())
def test_tile(t, form, rows, cols, more, M, N, K):
    print(f"[tile] t={t} form={form} {rows}x{cols} ({more}) M={M} N={N} K={K}", flush=True)
    T = torch()
    kernel, r, c, s = tc.plan(t, form, N, M, K)
    assert (kernel, r, c, s if t == 1 else min(s, 2)) == (2 if t == 1 else 3, rows, cols, more)
    gen = T.Generator(device="cuda").manual_seed(M + N + K + t)
    x = T.randn(M, K, generator=gen, device="cuda", dtype=T.float16)
    ws = [_weight(t, N, K, gen) for _ in range(2 if form else 1)]
    # one value past the output, which stays
    out = [T.full((M * N + 1,), -1, dtype=T.int16, device="cuda") for _ in range(3)]
    for (w, _), y in zip(ws, out):
        call("bx_linear_f16", t, ptr(w), None, ptr(x), ptr(y), M, N, K, *lws(), stream())
    plain = out[0][:-1].view(T.float16).reshape(M, N)
    assert bool(T.isfinite(plain).all())
    if form == 0:
        W, X = ws[0][1], x.double()
        want = X @ W.t().contiguous()
        # FP16 rounding of the result (2^-11, doubled), of the weights (2^-11 of the
        # dot product's mass) and the FP32 sums (2^-14 of it)
        mass = X.abs() @ W.abs().t().contiguous()
        tol = 2.0 ** -10 * want.abs() + (2.0 ** -14 + (0 if t == 1 else 2.0 ** -11)) * mass + 1e-6
        assert bool(((plain.double() - want).abs() <= tol).all()), float(((plain.double() - want).abs() / tol).max())
        bias = T.randn(N, generator=gen, device="cuda", dtype=T.float16)
        call("bx_linear_f16", t, ptr(ws[0][0]), ptr(bias), ptr(x), ptr(out[1]), M, N, K, *lws(), stream())
        got = out[1][:-1].view(T.float16).reshape(M, N).double()
        tol += 2.0 ** -10 * bias.double().abs()
        assert bool(((got - want - bias.double()).abs() <= tol).all())
        if M >= 128:
            H0 = T.randn(M, N, generator=gen, device="cuda")
            H = H0.clone()
            call("bx_linear_residual_f16", t, ptr(ws[0][0]), ptr(x), ptr(H), M, N, K, *lws(), stream())
            assert T.equal(H, H0 + plain.float())
    else:
        call("bx_linear_swiglu_f16", t, ptr(ws[0][0]), ptr(ws[1][0]), ptr(x), ptr(out[2]), M, N, K, *lws(), stream())
        call("bx_silu_f16", ptr(out[0]), ptr(out[0]), M * N, stream())
        call("bx_mul_f16", ptr(out[0]), ptr(out[1]), M * N, stream())
        assert T.equal(out[2][:-1], out[0][:-1])
    assert all(int(y[-1]) == -1 for y in out)
