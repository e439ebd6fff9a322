"""Shapes that reach every tile of the 17-row-and-up linears (gemm_quant.hip,
gemm_f16.hip) on 256 CUs, with partial tiles in rows and columns: per type family
{(form, tile rows, tile columns, K slices or workgroups per CU): (M, N, K)}.
form 0: plain and residual launches; 2: SwiGLU.  K slices: 1, or 2 for any split."""
from __future__ import annotations

import ctypes as C

QUANT = {
    (0, 32, 128, 1): (17, 65, 768), (0, 32, 128, 2): (17, 65, 1280),
    (0, 64, 128, 1): (97, 8195, 768), (0, 64, 128, 2): (1500, 129, 4096),
    (0, 96, 128, 1): (129, 12289, 768), (0, 96, 128, 2): (65, 6145, 4096),
    (0, 128, 128, 1): (200, 12289, 768), (0, 128, 128, 2): (97, 8195, 4096),
    (0, 64, 256, 1): (385, 8195, 768), (0, 96, 256, 1): (450, 8195, 768), (0, 128, 256, 1): (385, 12289, 768),
    (2, 32, 128, 1): (129, 65, 768), (2, 32, 128, 2): (129, 65, 1280),
    (2, 64, 128, 1): (1700, 257, 768), (2, 64, 128, 2): (1025, 129, 2048),
    (2, 96, 128, 1): (200, 5000, 768), (2, 96, 128, 2): (1500, 129, 4096),
    (2, 128, 128, 1): (200, 6145, 768), (2, 128, 128, 2): (300, 1025, 4096),
    (2, 32, 256, 1): (129, 6145, 768), (2, 32, 256, 2): (900, 65, 1280),
    (2, 64, 256, 1): (129, 8195, 768), (2, 64, 256, 2): (129, 2600, 4096),
    (2, 96, 256, 1): (129, 12289, 768), (2, 96, 256, 2): (1700, 257, 4096),
    (2, 128, 256, 1): (200, 10001, 768),
}
# Q6_K: its decode is slower, its columns even here (one scale of a pair each), no
# 128 x 256 tile; 32 x 256 SwiGLU tiles are taken with K slices only
Q6_K = {
    **{k: (m, n + n % 2, kk) for k, (m, n, kk) in QUANT.items() if k[1:3] != (128, 256)},
    (0, 64, 128, 2): (1025, 130, 4096), (0, 96, 128, 2): (65, 6146, 2048),
    (2, 64, 128, 2): (1025, 66, 2048), (2, 96, 128, 1): (129, 6146, 768), (2, 96, 128, 2): (1025, 130, 4096),
    (2, 128, 128, 2): (385, 514, 4096), (2, 32, 256, 2): (513, 66, 2048), (2, 64, 256, 2): (1281, 200, 4096),
    (2, 96, 256, 2): (450, 1300, 2048),
}
del Q6_K[2, 32, 256, 1]
F16 = {
    (0, 64, 64, 1): (17, 65, 320), (0, 128, 64, 1): (65, 8195, 320), (0, 128, 128, 1): (129, 12289, 320),
    (0, 128, 128, 2): (385, 8195, 320), (0, 256, 128, 1): (385, 12289, 2112), (0, 256, 256, 1): (900, 8195, 320),
    (2, 64, 64, 1): (129, 65, 1088), (2, 128, 64, 1): (129, 3000, 1088), (2, 128, 128, 1): (129, 6145, 320),
    (2, 128, 128, 2): (129, 8195, 320), (2, 256, 128, 1): (129, 12289, 2112), (2, 256, 256, 1): (385, 8195, 320),
}
CASES = {8: QUANT, 12: QUANT, 14: Q6_K, 1: F16}


def plan(t: int, form: int, N: int, M: int, K: int, have_ws: int = 1) -> tuple:
    """(kernel, tile rows, tile columns, K slices or workgroups per CU) of a launch."""
    from brolm_amd import _native
    out = (C.c_int * 4)()
    _native.bx_check(_native.hip().bx_linear_plan(t, form, 1, (C.c_int * 1)(N), M, K, have_ws, out), "linear_plan")
    return tuple(out)


def params():
    return [(t, *key, *shape) for t, cases in CASES.items() for key, shape in cases.items()]
