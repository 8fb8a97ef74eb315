"""Cyclic garbage collection stays out of a graph capture (model_executor/hip_graph_runner.py)."""
import contextlib
import gc
import types
import weakref

import pytest
import torch

from semi_pd_amd import _lib
from semi_pd_amd.model_executor import hip_graph_runner as runner


class _Node:
    pass


def _dead_cycle():
    a, b = _Node(), _Node()
    a.other, b.other = b, a
    return weakref.ref(a)


def test_nothing_is_collected_inside_and_the_setting_comes_back():
    assert gc.isenabled()
    with pytest.raises(KeyError):
        with runner.without_cycle_collection():
            dead = _dead_cycle()
            keep = [_Node() for _ in range(20 * gc.get_threshold()[0])]      # (collections of the youngest objects fall due many times)
            assert dead() is not None and not gc.isenabled()
            with runner.without_cycle_collection():                            # (another thread's capture, begun and ended meanwhile)
                pass
            assert not gc.isenabled()
            raise KeyError
    assert gc.isenabled()
    gc.collect()
    assert dead() is None and keep
    gc.disable()
    try:
        with runner.without_cycle_collection():
            pass
        assert not gc.isenabled()
    finally:
        gc.enable()


@pytest.fixture
def collecting(monkeypatch):
    """Captures on a host without a device: [(what, was the collector on)] of what happens in and around them."""
    seen = []

    @contextlib.contextmanager
    def graph(g, **kw):
        seen.append(("begin", gc.isenabled()))
        yield
        seen.append(("end", gc.isenabled()))

    class Lib:
        def semipd_stream_abort_capture(self, stream):
            seen.append(("abort", gc.isenabled()))

        semipd_clear_last_error = semipd_stream_create = lambda self, *a: 0

    stream = types.SimpleNamespace(wait_stream=lambda other: None)
    monkeypatch.setattr(torch.cuda, "graph", graph)
    monkeypatch.setattr(torch.cuda, "CUDAGraph", lambda: types.SimpleNamespace(pool=lambda: None))
    monkeypatch.setattr(torch.cuda, "ExternalStream", lambda *a, **k: stream)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda *a: stream)
    monkeypatch.setattr(torch.cuda, "stream", lambda s: contextlib.nullcontext())
    monkeypatch.setattr(torch.cuda, "synchronize", lambda *a: None)
    monkeypatch.setattr(_lib, "load", Lib)
    monkeypatch.setattr(runner, "_PARKED", [])
    return seen


def _runner(step):
    """A runner whose model step is `step`, in front of its captures."""
    r = runner.HipGraphRunner.__new__(runner.HipGraphRunner)
    r.mr = types.SimpleNamespace(req_to_token_pool=None, token_to_kv_pool=None, sampler=None,
                                 attn_backend=types.SimpleNamespace(init_forward_metadata_capture_cuda_graph=lambda *a: None),
                                 model=types.SimpleNamespace(forward=step))
    r.input_ids = r.req_pool_indices = r.seq_lens = r.out_cache_loc = r.positions = r.state_indices = torch.zeros(4, dtype=torch.int64)
    r.graphs, r.outputs, r.pool, r._cus, r._raw_stream = {}, {}, None, 0, None
    r.stream, r._stream_finalizer = torch.cuda.current_stream(), types.SimpleNamespace(detach=lambda: None)
    return r


def test_a_capture_runs_without_collection(collecting):
    out = types.SimpleNamespace(next_token_ids=torch.zeros(2), next_token_logits=None)
    _runner(lambda *a: (collecting.append(("step", gc.isenabled())), out)[1])._capture_one(2)
    assert collecting == [("step", True)] * 2 + [("begin", False), ("step", False), ("end", False)] and gc.isenabled()


def test_a_capture_that_fails_is_gone_before_collection_comes_back(collecting):
    out, runs = types.SimpleNamespace(next_token_ids=torch.zeros(2), next_token_logits=None), []

    def step(*a):
        runs.append(None)
        if len(runs) == 3:
            raise RuntimeError("refused")
        return out

    with pytest.raises(RuntimeError, match="refused"):
        _runner(step)._capture_one(2)
    assert collecting == [("begin", False), ("abort", False)] and gc.isenabled()


def test_the_recovery_s_capture_runs_without_collection(collecting):
    runner.recover_after_failed_capture("cpu")
    assert collecting == [("begin", False), ("end", False)] and gc.isenabled()
