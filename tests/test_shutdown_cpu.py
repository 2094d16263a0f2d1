"""Product shutdown without aborts.

SIGTERM to the deployed processes must end them in order and with exit code 0 within 10 s,
with no "terminate called" abort from a thread left inside native code at interpreter exit:

* ``python -m drtc_amd.llm.server --backend scripted``;
* ``python -m drtc_amd.llm.server --backend engine`` with the engine in the server process
  (a tiny model on the CPU: the EngineLoop thread, its in-flight requests and the RPC
  handlers blocked on them);
* a 3-node Raft cluster of ``python -m drtc_amd.server.node`` processes.

And in process: EngineLoop.stop() fails what is still queued (callers return), joins its
thread and leaves the engine closed; WorkerPool.close() joins its threads.
"""
import os
import signal
import subprocess
import sys
import threading
import time

import grpc
import pytest

from drtc_amd.protos import llm_pb, make_stub, raft_pb, LLM_SERVICE, RAFT_SERVICE

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _free_port():
    import socket

    s = socket.socket()
    s.bind(("127.0.0.1", 0))
    p = s.getsockname()[1]
    s.close()
    return p


def _popen(args, env=None):
    env = dict(os.environ, PYTHONPATH=ROOT + os.pathsep + os.environ.get("PYTHONPATH", ""),
               **(env or {}))
    return subprocess.Popen([sys.executable, "-m", *args], env=env, stdout=subprocess.DEVNULL,
                            stderr=subprocess.PIPE, start_new_session=True)


def _sigterm_and_wait(p, limit=10.0):
    t0 = time.time()
    p.send_signal(signal.SIGTERM)
    try:
        rc = p.wait(timeout=limit)
    except subprocess.TimeoutExpired:
        os.killpg(p.pid, signal.SIGKILL)
        p.wait()
        raise AssertionError(f"no exit within {limit} s of SIGTERM")
    err = p.stderr.read().decode(errors="replace")
    return rc, time.time() - t0, err


def _wait_llm(port, timeout=120.0):
    stub = make_stub(grpc.insecure_channel(f"127.0.0.1:{port}"), LLM_SERVICE)
    t_end = time.time() + timeout
    while True:
        try:
            return stub, stub.GetSmartReply(llm_pb.SmartReplyRequest(
                request_id="probe", recent_messages=[llm_pb.Message(sender="a", content="hi")]),
                timeout=30)
        except grpc.RpcError:
            if time.time() > t_end:
                raise
            time.sleep(0.2)


def test_llm_server_scripted_exits_cleanly_on_sigterm():
    port = _free_port()
    p = _popen(["drtc_amd.llm.server", "--backend", "scripted", "--port", str(port),
                "--log-level", "INFO"])
    try:
        _, r = _wait_llm(port)
        assert len(r.suggestions) == 3
        rc, dt, err = _sigterm_and_wait(p)
    finally:
        if p.poll() is None:
            os.killpg(p.pid, signal.SIGKILL)
    assert rc == 0, err[-2000:]
    assert "terminate called" not in err and "shutting down" in err
    assert dt < 10


@pytest.mark.parametrize("where", ["cpu", pytest.param("gpu", marks=pytest.mark.gpu)])
def test_llm_server_engine_backend_exits_cleanly_with_requests_in_flight(where):
    """The in-process engine backend (EngineLoop thread) on a tiny model - on the CPU, and on
    the GPU with HIP kernels and hipGraph decode: SIGTERM arrives while clients still wait on
    generations; the server stops the RPC front-end, stops and drains the engine (the waiting
    handlers return their fallback), synchronizes the device and exits 0."""
    port = _free_port()
    p = _popen(["drtc_amd.llm.server", "--backend", "engine", "--model", "tiny-llama",
                "--in-process", "--max-batch", "4", "--max-model-len", "512",
                "--port", str(port), "--log-level", "INFO"]
               + (["--no-graphs"] if where == "cpu" else []),
               env={"CUDA_VISIBLE_DEVICES": ""} if where == "cpu" else None)
    try:
        stub, r = _wait_llm(port, timeout=180)
        assert len(r.suggestions) == 3
        # keep the engine busy: more concurrent generations than batch slots
        errs = []

        def call():
            try:
                stub.GetLLMAnswer(llm_pb.LLMRequest(request_id="q", query="what now?",
                                                    context=["a", "b"]), timeout=60)
            except grpc.RpcError as e:  # cancelled by the server's stop: fine
                errs.append(e.code())

        ts = [threading.Thread(target=call) for _ in range(12)]
        for t in ts:
            t.start()
        time.sleep(0.5)
        rc, dt, err = _sigterm_and_wait(p)
        for t in ts:
            t.join(timeout=20)
    finally:
        if p.poll() is None:
            os.killpg(p.pid, signal.SIGKILL)
    assert rc == 0, err[-3000:]
    assert "terminate called" not in err and "Traceback" not in err, err[-3000:]
    assert dt < 10


@pytest.mark.slow
def test_raft_cluster_nodes_exit_cleanly_on_sigterm(tmp_path):
    ports = {i: _free_port() for i in (1, 2, 3)}
    addrs = {i: f"127.0.0.1:{p}" for i, p in ports.items()}
    peers = ",".join(f"{i}={a}" for i, a in addrs.items())
    procs = {i: _popen(["drtc_amd.server.node", "--node-id", str(i), "--port", str(ports[i]),
                        "--peers", peers, "--data-root", str(tmp_path), "--llm", "",
                        "--election-timeout", "0.4,0.8", "--heartbeat", "0.04",
                        "--bcrypt-rounds", "4", "--log-level", "WARNING"])
             for i in ports}
    try:
        t_end = time.time() + 60
        leader = None
        while leader is None and time.time() < t_end:
            for i, a in addrs.items():
                try:
                    r = make_stub(grpc.insecure_channel(a), RAFT_SERVICE).GetLeaderInfo(
                        raft_pb.GetLeaderRequest(), timeout=0.5)
                    if r.is_leader:
                        leader = i
                except grpc.RpcError:
                    pass
            time.sleep(0.1)
        assert leader is not None
        for a in addrs.values():  # every node is up (signal handlers installed) before SIGTERM
            while True:
                try:
                    make_stub(grpc.insecure_channel(a), RAFT_SERVICE).GetLeaderInfo(
                        raft_pb.GetLeaderRequest(), timeout=0.5)
                    break
                except grpc.RpcError:
                    assert time.time() < t_end
                    time.sleep(0.1)
        stub = make_stub(grpc.insecure_channel(addrs[leader]), RAFT_SERVICE)
        t_end = time.time() + 30
        while True:  # the default users arrive through the log after the first election
            r = stub.Login(raft_pb.LoginRequest(username="alice", password="alice123"), timeout=10)
            if r.success or time.time() > t_end:
                break
            time.sleep(0.1)
        assert r.success
        # SIGTERM all three together (a cluster shutdown), then check each
        for p in procs.values():
            p.send_signal(signal.SIGTERM)
        results = {}
        for i, p in procs.items():
            results[i] = _sigterm_and_wait(p) if p.poll() is None else (p.returncode, 0.0, "")
    finally:
        for p in procs.values():
            if p.poll() is None:
                os.killpg(p.pid, signal.SIGKILL)
    for i, (rc, dt, err) in results.items():
        assert rc == 0, (i, err[-2000:])
        assert "terminate called" not in err and "Traceback" not in err, (i, err[-2000:])
        assert dt < 10


def test_engine_loop_stop_fails_queued_requests_and_closes_the_engine():
    from drtc_amd.engine import LLMEngine, Request, SamplingParams
    from drtc_amd.engine.engine import EngineLoop, _LIVE_LOOPS
    from drtc_amd.models import TINY_LLAMA, TransformerLM

    m = TransformerLM(TINY_LLAMA, "cpu", seed=1)
    eng = LLMEngine(m, max_batch=2, max_model_len=256, num_blocks=64, use_graphs=False)
    loop = EngineLoop(eng, burst_gap_s=0).start()
    assert loop in _LIVE_LOOPS
    reqs = [loop.submit(Request(list(range(1, 30)), SamplingParams.greedy(200, ignore_eos=True)))
            for _ in range(6)]
    time.sleep(0.3)
    assert loop.stop(timeout=10)
    assert not loop.thread.is_alive() and loop not in _LIVE_LOOPS
    assert all(r.wait(1.0) for r in reqs)  # nobody is left waiting
    reasons = {r.finish_reason for r in reqs}
    assert reasons <= {"length", "error: shutdown"} and "error: shutdown" in reasons
    assert eng.closed and not eng.running and not eng.waiting and eng.alloc.num_used == 0
    with pytest.raises(RuntimeError):
        eng.add_request(Request([1, 2, 3], SamplingParams.greedy(2)))
    assert loop.stop() is True  # idempotent


def test_worker_pool_close_joins_threads_and_fails_waiters():
    from drtc_amd.engine import SamplingParams
    from drtc_amd.llm.backends import WorkerPool

    pool = WorkerPool("tiny-llama", ["cpu"], dict(max_batch=2, max_model_len=256, num_blocks=32,
                                                  use_graphs=False), hb_interval=0.2)
    # more long requests than the replica's two slots: some are still queued at close()
    subs = [pool.submit(0, list(range(1, 20)), SamplingParams.greedy(120, ignore_eos=True))
            for _ in range(6)]
    pool.close()
    assert all(not p.is_alive() for p in pool.procs)
    assert all(not t.is_alive() for t in pool._threads)
    for _, ev, slot in subs:  # nobody is left waiting
        assert ev.wait(1.0) and slot
    pool.close()  # idempotent
