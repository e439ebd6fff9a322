"""The tiles that the 17-row-and-up linears choose (bx_linear_plan), without a
device: 256 CUs are assumed."""
from __future__ import annotations

import pytest

import tile_cases as tc


@pytest.mark.parametrize("t", list(tc.CASES))
def test_cases_reach_every_tile(t):
    """Each listed shape runs the tile it is listed for, and the list has every
    tile that a plan can choose (Q6_K has no 128 x 256, its raw blocks leave no LDS
    for it; 32 x 256 is for SwiGLU alone)."""
    for (form, rows, cols, more), (M, N, K) in tc.CASES[t].items():
        kernel, r, c, s = tc.plan(t, form, N, M, K)
        assert (kernel, r, c) == (2 if t == 1 else 3, rows, cols), (t, form, M, N, K)
        assert (s if t == 1 else min(s, 2)) == more, (t, form, M, N, K, s)
        assert M % rows and (N % cols if form == 0 else N % (cols // 2)), (M, N)
    tiles = {(f, r, c) for f, r, c, _ in tc.CASES[t]}
    if t == 1:
        shapes = {(64, 64, 1), (128, 64, 1), (128, 128, 1), (128, 128, 2), (256, 128, 1), (256, 256, 1)}
        assert set(tc.CASES[t]) == {(f, *s) for f in (0, 2) for s in shapes}
    else:
        every = {(f, r, c) for f in (0, 2) for r in (32, 64, 96, 128) for c in (128, 256)} - {(0, 32, 256)}
        assert tiles == every - ({(0, 128, 256), (2, 128, 256)} if t == 14 else set())


def test_plan_follows_the_dispatch():
    """Which kernel takes a launch: the GEMVs to 16 rows, the general tiles where K
    or an odd Q6_K block count leaves no whole copies, one K slice without a
    workspace, and the SwiGLU launch in the slices of the plain one."""
    assert tc.plan(12, 0, 2048, 16, 2048)[0] == 0
    assert tc.plan(12, 0, 2048, 17, 2048)[0] == 3
    assert tc.plan(8, 0, 2048, 200, 2080)[0] == 1
    assert tc.plan(14, 0, 129, 200, 768)[0] == 1 and tc.plan(14, 0, 130, 200, 768)[0] == 3
    assert tc.plan(1, 0, 2048, 200, 1040)[0] == 1
    assert tc.plan(1, 0, 1000, 200, 768)[0] == 1 and tc.plan(1, 0, 1000, 100, 768)[0] == 2
    assert tc.plan(1, 0, 1024, 200, 2048)[0] == 2
    for t in (8, 12, 14):
        assert tc.plan(t, 0, 2048, 128, 6144)[3] > 1
        assert tc.plan(t, 0, 2048, 128, 6144, have_ws=0)[3] == 1
        for M in (128, 160, 300, 511, 1025):
            for N in (66, 130, 1024, 3072, 6144):
                for K in (768, 2048, 4096, 14336):
                    assert tc.plan(t, 2, N, M, K)[3] == tc.plan(t, 0, N, M, K)[3], (t, M, N, K)
