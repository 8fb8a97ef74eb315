"""Cyclic garbage collection stays out of a graph capture (model_executor/hip_graph_runner.py)."""
import gc
import inspect
import weakref

import pytest

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


def test_captures_run_without_collection():
    source = inspect.getsource(runner.HipGraphRunner._capture_one)
    assert "with without_cycle_collection(), torch.cuda.graph(" in source
