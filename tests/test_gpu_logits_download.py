"""Logits on their way to the host: pieces converted by several threads, calls
beyond the pinned staging's size, and steps that keep their logits buffer."""
from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def model(tmp_path_factory):
    import brolm_amd as ba
    ba.init()
    path = str(tmp_path_factory.mktemp("dl") / "wide.gguf")
    ba.write_synth_qwen3(ba.SynthSpec(vocab=70001, hidden=256, intermediate=256, layers=2, n_q=4, n_kv=2, head_dim=64,
                                      seed=5), path)
    m = ba.Qwen3Model(ba.Qwen3Config.from_gguf(path))
    m.load_weights(path)
    m.allocate_cache(128)
    yield m
    m.close()


def _fp16_values(a):
    return np.array_equal(a, a.astype(np.float16).astype(np.float32))


def test_large_downloads_hold_every_row(model):
    """64 rows of 70,001 logits (4.48 M values, two rounds of staging, four
    pieces each) against the same rows computed and downloaded in smaller
    calls (one piece; three pieces).  2e-2: the model tolerance between two
    splits of a prompt; rows of other tokens differ by more."""
    import brolm_amd as ba
    ids = ba.prompt_ids(64, 70001, 9)
    model.reset_cache()
    full = model.forward(ids)
    assert _fp16_values(full)
    model.reset_cache()
    rows = [model.forward(ids[:7]), model.forward(ids[7:40]), model.forward(ids[40:])]
    assert all(_fp16_values(r) for r in rows)
    parts = np.concatenate(rows)
    assert np.abs(full - parts).max() <= 2e-2
    # the bound tells rows apart
    assert min(np.abs(full[i] - full[i - 1]).max() for i in range(1, 64)) > 0.2


def test_one_row_downloads_follow_their_step(model):
    """Steps that reuse the handle's logits row: each call returns its own
    step's logits, whatever ran before, and the greedy tokens agree."""
    import brolm_amd as ba
    ids = ba.prompt_ids(9, 70001, 3)
    model.reset_cache()
    model.forward_last(ids[:8])
    a = model.forward_last([ids[8]])
    model.truncate_cache(8)
    other = model.forward_last([int(ids[0])])
    model.truncate_cache(8)
    b = model.forward_last([ids[8]])
    model.truncate_cache(8)
    assert np.array_equal(a, b) and not np.array_equal(a, other)
    assert model.decode_greedy(ids[8], 1) == [int(a.argmax())]
