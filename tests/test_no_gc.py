"""_lib.no_gc: the garbage collector stays off while any thread captures a
graph, however their captures overlap, and ends as it was."""
import gc
import threading

import pytest


@pytest.mark.parametrize("enabled", [True, False])
def test_overlapping_threads(enabled):
    from fluids2d_amd._lib import no_gc
    was = gc.isenabled()
    inside, leave = threading.Event(), threading.Event()
    seen = []

    def second():
        with no_gc():
            inside.set()
            leave.wait(30)
            seen.append(gc.isenabled())  # the first has left meanwhile
    t = threading.Thread(target=second)
    try:
        gc.enable() if enabled else gc.disable()
        with no_gc():
            t.start()
            assert inside.wait(30)
            assert not gc.isenabled()
        assert not gc.isenabled()
        leave.set()
        t.join(30)
        assert seen == [False] and gc.isenabled() == enabled
        with pytest.raises(ValueError), no_gc(), no_gc():
            raise ValueError
        assert gc.isenabled() == enabled
    finally:
        leave.set()
        gc.enable() if was else gc.disable()
