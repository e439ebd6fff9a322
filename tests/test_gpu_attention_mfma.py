"""Attention of 16 and more query rows against float64: each way the rows, heads
and keys are dealt to wavefronts and workgroups, with remainders in all three."""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _exact(q, K, V, n_q, n_kv, hd, causal):
    import torch
    L, n = q.shape[0], K.shape[0]
    q = torch.from_numpy(q).double().view(L, n_kv, n_q // n_kv, hd).permute(1, 2, 0, 3)
    K = torch.from_numpy(K).double().view(n, n_kv, 1, hd).permute(1, 2, 3, 0)
    V = torch.from_numpy(V).double().view(n, n_kv, 1, hd).permute(1, 2, 0, 3)
    s = q @ K / hd ** 0.5
    if causal:
        s = s.masked_fill(torch.ones(L, n, dtype=torch.bool).triu(n - L + 1), float("-inf"))
    return (s.softmax(-1) @ V).permute(2, 0, 1, 3).reshape(L, n_q * hd).numpy()


@pytest.mark.parametrize("offset", [0, 1])   # 1: operands 2 bytes off the 16-byte grid
@pytest.mark.parametrize("L,keys,n_q,n_kv,hd,causal", [
    # one tile of keys in 16-row fragments: 64 keys, then 128, wavefronts without a row
    (16, 16, 4, 4, 64, 1), (31, 33, 4, 2, 128, 1), (33, 64, 6, 2, 128, 0), (64, 64, 16, 2, 128, 1), (17, 32, 2, 1, 64, 1),
    (300, 47, 6, 3, 64, 0), (16, 65, 4, 2, 128, 1), (32, 100, 7, 7, 64, 1), (128, 128, 4, 1, 128, 1), (65, 127, 3, 1, 64, 0),
    (113, 113, 2, 2, 64, 1), (50, 97, 5, 5, 128, 0),
    # keys of a tile over two wavefronts: one row to a few tiles, wavefronts without a row
    (16, 130, 4, 2, 128, 1), (64, 256, 8, 1, 64, 0),
    (129, 129, 7, 1, 128, 1), (700, 701, 16, 2, 128, 1), (600, 1, 16, 2, 64, 0),
    # over four, and then over workgroups too
    (300, 300, 8, 2, 128, 1), (257, 257, 8, 8, 64, 0), (17, 1500, 8, 2, 128, 1), (65, 1023, 4, 4, 64, 1),
    (40, 900, 24, 3, 128, 0), (17, 20000, 16, 8, 64, 1), (128, 1025, 32, 8, 128, 1),
    # two heads sharing a tile; an odd group, which cannot
    (1100, 1100, 16, 2, 128, 1), (1216, 1216, 15, 5, 64, 1),
    # a wavefront to each 32 rows: four, two and one head to a tile
    (1100, 1100, 32, 8, 128, 1), (1057, 1200, 32, 16, 64, 1), (1000, 999, 35, 5, 128, 0)])
def test_attention_rows(L, keys, n_q, n_kv, hd, causal, offset):
    import torch
    from brolm_amd import _native as nat
    print(f"[attention rows] L={L} keys={keys} {n_q}/{n_kv} hd={hd} causal={causal} offset={offset}", flush=True)
    rng = np.random.default_rng(L + 7 * keys + n_q)
    host = [rng.standard_normal((r, n * hd)).astype(np.float16) for r, n in ((L, n_q), (keys, n_kv), (keys, n_kv))]
    devs = []
    for x in host:
        buf = torch.zeros(x.size + 8, dtype=torch.float16, device="cuda")
        buf[offset:offset + x.size] = torch.from_numpy(x.reshape(-1)).cuda()
        devs.append(buf)
    out = torch.full((L * n_q * hd + 16,), -7.0, dtype=torch.float16, device="cuda")
    hip = nat.hip()
    # the workspace ends in a guard: the split path stays inside it
    nb = int(hip.bx_attention_workspace_bytes(L, n_q, hd, keys))
    ws = torch.full((nb // 4 + 64,), 3.0, dtype=torch.float32, device="cuda")
    p = [C.c_void_p(t.data_ptr() + 2 * offset) for t in (*devs, out)]
    st = C.c_void_p(torch.cuda.current_stream().cuda_stream)
    if causal:
        rc = hip.bx_attention_decode_f16(p[0], p[1], p[2], L, keys, n_q, n_kv, hd, C.c_float(0.0), 0, p[3],
                                         C.c_void_p(ws.data_ptr()), st)
    else:
        rc = hip.bx_attention_gqa_f16(p[0], p[1], p[2], L, keys, n_q, n_kv, hd, 0, p[3], C.c_void_p(ws.data_ptr()), st)
    assert rc == 0, nat.hip_error()
    got = out.cpu().numpy()
    assert (got[:offset] == -7).all() and (got[offset + L * n_q * hd:] == -7).all()
    assert (ws[nb // 4:] == 3).all()
    got = got[offset:offset + L * n_q * hd].astype(np.float64).reshape(L, -1)
    want = _exact(host[0].astype(np.float32), host[1].astype(np.float32), host[2].astype(np.float32), n_q, n_kv, hd,
                  causal)
    # the weights, summing to 1, are rounded to FP16 (2^-11 each at most) and so
    # is the result; scores and sums are FP32 (below 1e-5 here)
    tol = 2.0 ** -11 * (np.abs(host[2]).max() + np.abs(want)) + 1e-5
    assert (np.abs(got - want) <= tol).all(), float((np.abs(got - want) / tol).max())


def test_attention_two_streams_with_their_own_workspaces():
    """Calls on two streams at once, keys shared out over workgroups (records in the
    workspace): each gives the bits it gives alone."""
    import torch
    from brolm_amd import _native as nat
    hip = nat.hip()
    L, keys, n_q, n_kv, hd, reps = 40, 2040, 16, 8, 128, 6
    rng = np.random.default_rng(5)
    nb = int(hip.bx_attention_workspace_bytes(L, n_q, hd, keys))
    ops = [[torch.from_numpy(rng.standard_normal((r, n * hd)).astype(np.float16)).cuda()
            for r, n in ((L, n_q), (keys, n_kv), (keys, n_kv))] for _ in range(2)]
    wss = [torch.empty(nb, dtype=torch.uint8, device="cuda") for _ in range(2)]

    def run(i, out, stream):
        p = [C.c_void_p(t.data_ptr()) for t in (*ops[i], out, wss[i])]
        assert hip.bx_attention_decode_f16(*p[:3], L, keys, n_q, n_kv, hd, C.c_float(0.0), 0, p[3], p[4],
                                           C.c_void_p(stream.cuda_stream)) == 0, nat.hip_error()

    outs = [[torch.zeros(L, n_q * hd, dtype=torch.float16, device="cuda") for _ in range(reps)] for _ in range(2)]
    alone = [torch.zeros(L, n_q * hd, dtype=torch.float16, device="cuda") for _ in range(2)]
    for i in range(2):
        run(i, alone[i], torch.cuda.current_stream())
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    for r in range(reps):
        for i in range(2):
            run(i, outs[i][r], streams[i])
    torch.cuda.synchronize()
    for i in range(2):
        assert float(alone[i].float().abs().max()) > 0
        for r in range(reps):
            assert torch.equal(outs[i][r], alone[i]), (i, r)
