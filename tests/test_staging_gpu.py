"""Decode steps that read their inputs from pinned host memory by themselves, and write their tokens there."""
import gc

import numpy as np
import pytest
import torch

from drtc_amd import ops
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


@pytest.mark.parametrize("rows,columns,per", [(1, 1, 32), (1, 700, 32), (1, 40000, 1), (15, 64, 32), (17, 1100, 8), (300, 65, 32),
                                              (1024, 16, 32), (1024, 600, 32), (1500, 130, 1), (9000, 200, 3)])
def test_table_rows_by_their_lengths(hipk, rows, columns, per):
    """Every word that a row's length asks for, none beyond the columns that go ahead of the lengths (4096 words of all
    rows, 16 of each at least), nothing outside; lengths of 0, of whole blocks and past the table."""
    rng = np.random.default_rng(rows)
    need = rng.integers(0, columns + 1, rows)
    need[::7] = rng.integers(0, min(columns, 20) + 1, len(need[::7]))
    need[rows // 2] = columns
    lengths = np.maximum(0, per * need - rng.integers(0, per, rows))
    lengths[rows // 3] = per * columns + 5
    need = np.minimum(-(-lengths // per), columns)
    words = 3 + rows + 2 + rows * columns + 1  # gaps of words that stay
    at_len, at_tab = 3, 3 + rows + 2
    host = torch.zeros(4 * words, dtype=torch.uint8, pin_memory=True)
    h = host.numpy().view(np.int32)
    h[:] = rng.integers(1, 1 << 30, words)
    h[at_len:at_len + rows] = lengths
    dst = torch.full((4 * words,), 255, dtype=torch.uint8, device="cuda")
    ops.StageRows(dst, host, [(0, 4), (8, 8)], (4 * at_tab, rows, columns, 4 * at_len, per))()
    got = dst.cpu().numpy().view(np.int32)
    table, want = got[at_tab:-1].reshape(rows, columns), h[at_tab:-1].reshape(rows, columns)
    at, ahead = np.arange(columns), max(16, 4096 // rows)
    assert ((table == want) | (at >= need[:, None])).all()
    assert ((table == -1) | (at < np.maximum(need, ahead)[:, None])).all()
    assert got[0] == h[0] and (got[1:at_tab] == -1).all() and got[-1] == -1
    with pytest.raises(AssertionError):
        ops.StageRows(dst, host, [], (4 * at_tab + 8, rows, columns, 4 * at_len, per))


def test_a_step_reads_the_blocks_that_its_contexts_have(hipk):
    """Of block tables as wide as long models' only the contexts' blocks cross the bus, with a graph and without; the tokens
    are the narrow tables'."""
    m = TransformerLM(TINY_LLAMA, "cuda", seed=3)
    n = 1000
    ids, blocks, tokens = np.arange(n) % 400, [[1 + i] for i in range(n)], []
    for width, graphs in ((1, True), (1024, True), (1024, False)):
        r = DecodeRunner(m, m.new_cache(n + 1, 4), 1024, width, use_graphs=graphs)
        if graphs:
            r.capture(r.bucket(n))
        r.bt.fill_(7)
        tokens.append(np.stack([r.wait(_launch(r, ids, np.full(n, at), blocks)) for at in range(3)]))
        assert (r.bt[:n, :1].cpu().numpy() == blocks).all()
        assert (r.bt[:, 16:] == 7).all()
    assert all((t == tokens[0]).all() for t in tokens)


@pytest.mark.parametrize("between", ["raised", "eager"])
def test_a_turn_passed_over(hipk, between):
    """Between steps of a graph a launch that raises with its set chosen, or a step without a graph: the next replay reads
    its own set, not the other one's positions, slots and tokens."""
    tokens = []
    for passed in (False, True):
        r, got = _runner(), []
        for at in range(6):
            if passed and at in (2, 3):
                if between == "raised":
                    with pytest.raises(ValueError):
                        r.launch(1, np.array([9], np.int32), np.zeros(3, np.int32), *[None] * 6)
                else:
                    graphs, r._graphs, r.use_graphs = r._graphs, {}, False
            got.append(r.wait(_launch(r, [5 + at], [at], [[1]])).tolist())
            assert int(r.positions[0]) == at and int(r.slots[0]) == 32 + at
            if not r.use_graphs:
                r._graphs, r.use_graphs = graphs, True
        tokens.append(got)
    assert tokens[0] == tokens[1]
