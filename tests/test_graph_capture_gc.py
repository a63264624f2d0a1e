"""A captured outer step and Python's cyclic garbage collector: a CUDAGraph
collected while a stream is capturing ends the process (its destructor
synchronises the device), so the runners are freed by their reference count
and captures hold the collector off."""
import gc
import weakref


def test_nested_step_is_no_cycle(pkg):
    on = gc.isenabled()
    gc.disable()
    try:
        ns = pkg.step.NestedStep([], [3], feedback=False)
        assert ns.order == [0, 0, 0]
        ref = weakref.ref(ns)
        del ns
        assert ref() is None
    finally:
        if on:
            gc.enable()


def test_no_collection_restores_the_collector(pkg):
    on = gc.isenabled()
    with pkg.step.no_collection():
        assert not gc.isenabled()
    assert gc.isenabled() == on
    gc.disable()
    try:
        with pkg.step.no_collection():
            assert not gc.isenabled()
        assert not gc.isenabled()
    finally:
        if on:
            gc.enable()
