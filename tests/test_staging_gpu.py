"""Decode steps that read their inputs from pinned host memory by themselves, and write their tokens there."""
import gc

import numpy as np
import pytest
import torch

from drtc_amd.engine.decode_runner import DecodeRunner
from drtc_amd.models import TINY_LLAMA, TransformerLM

pytestmark = pytest.mark.gpu


def _runner(seed=3, **kw):
    m = TransformerLM(TINY_LLAMA, "cuda", seed=seed)
    return DecodeRunner(m, m.new_cache(64, 4), 4, 8, **kw)


def _launch(r, ids, at, blocks):
    """A greedy step: row i's token ids[i] at position at[i], its cache blocks in blocks[i]."""
    n, at = len(ids), np.asarray(at, np.int32)
    rows = np.zeros((n, r.max_blocks), np.int32)
    for row, b in zip(rows, blocks):
        row[:len(b)] = b
    slots = rows[np.arange(n), at // 32].astype(np.int64) * 32 + at % 32
    return r.launch(n, np.asarray(ids, np.int32), at, at + 1, slots, rows, np.zeros(n, np.float32), np.zeros(n, np.int32),
                    np.ones(n, np.float32))


def test_a_runner_that_goes_waits_for_its_steps(hipk):
    r = _runner()
    for at in range(2):
        r.wait(_launch(r, [5], [at], [[1]]))
    torch.cuda._sleep(100_000_000)
    _launch(r, [6], [2], [[1]])
    events = list(r.events)
    assert not events[0].query()
    del r
    gc.collect()
    assert all(e.query() for e in events)
