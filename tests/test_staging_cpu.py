"""Decode staging: what of it can be checked without a GPU."""
import gc
import os
import re
import subprocess
import weakref

import pytest
import torch

from drtc_amd import _build


@pytest.mark.skipif(not os.path.exists(_build.HIPCC), reason="no hipcc")
def test_the_turn_has_arrived_before_a_workgroup_counts_itself(tmp_path):
    """step_stage_kernel, as compiled: no read of whose turn it is (the only load at agent scope) is under way at the
    workgroup's first barrier, behind which the workgroup counts and the last one gives the turn away.  The barrier itself
    waits for no load."""
    src, asm = os.path.join(_build.CSRC, "kernels", "sampling.hip"), tmp_path / "sampling.s"
    subprocess.run([_build.HIPCC, "--offload-arch=gfx950", "-O3", "-std=c++17", "-ffp-contract=fast", "-Xclang", "-target-feature",
                    "-Xclang", "-packed-fp32-ops", "--offload-device-only", "-S", src, "-o", str(asm)], check=True,
                   capture_output=True)
    text = asm.read_text()
    body = text[re.search(r"^\w*step_stage_kernel\w*:", text, re.M).end():]
    under_way, looked = False, 0
    for line in body[:body.index("s_endpgm")].splitlines():
        op = line.split(";")[0].strip()
        if op.startswith("global_load") and re.search(r"\bsc1\b", op) and not re.search(r"\bsc0\b", op):
            under_way, looked = True, looked + 1
        elif op.startswith("s_waitcnt") and re.search(r"vmcnt\(0\)", op):
            under_way = False
        elif op.startswith("s_barrier"):
            assert looked and not under_way
            return
    raise AssertionError("no barrier")


@pytest.mark.parametrize("recording", [False, True])
def test_pinned_buffers_outlive_the_steps_of_a_runner(monkeypatch, recording):
    """A runner that goes with steps under way keeps the buffers that their kernels address until the steps' events have
    gone by, which are not waited for while a graph is recorded."""
    from drtc_amd.engine import decode_runner
    from drtc_amd.models import TINY_LLAMA, TransformerLM

    m = TransformerLM(TINY_LLAMA, "cpu", seed=1)
    seen = []

    class Event:
        def synchronize(self):
            seen.append(all(b() is not None for b in buffers))

    def runner():
        r = decode_runner.DecodeRunner(m, m.new_cache(4, 4), 4, 8)
        r.events[:] = [Event(), Event()]
        return r

    r = runner()
    buffers = [weakref.ref(t) for t in (*r.h_stage, *r.h_out)]
    monkeypatch.setattr(torch.cuda, "is_initialized", lambda: recording)
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: recording)
    del r
    gc.collect()
    if recording:
        assert not seen and all(b() is not None for b in buffers)
        monkeypatch.undo()
        r = runner()
        del r
        gc.collect()
    assert seen == [True] * (4 if recording else 2) and not decode_runner._retired
    assert all(b() is None for b in buffers)


def test_runners_that_go_while_another_is_waited_for():
    """As from another thread, or the collector during the wait: each one's buffers until its own steps are over."""
    from drtc_amd.engine import decode_runner

    class Buffer:
        pass

    order, buffers = [], [Buffer(), Buffer()]
    alive = [weakref.ref(b) for b in buffers]

    class Event:
        def __init__(self, i, nested=None):
            self.i, self.nested = i, nested

        def synchronize(self):
            if self.nested:
                nested, self.nested = self.nested, None
                decode_runner._retire(*nested)
            order.append((self.i, alive[self.i]() is not None))

    held = (buffers.pop(),)
    decode_runner._retire([Event(0, ([Event(1)], held))], (buffers.pop(),))
    assert order == [(1, True), (0, True)] and alive[0]() is None and not decode_runner._retired
    del held
    gc.collect()
    assert alive[1]() is None
