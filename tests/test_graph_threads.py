"""The pause of the garbage collector around captures, with several threads (no GPU)."""
import gc
import threading

import pytest


@pytest.mark.parametrize("was", [True, False])
def test_collector_stays_off_until_the_last_capture_ends(was):
    from jztree_amd.graph import _no_collection
    before = gc.isenabled()
    (gc.enable if was else gc.disable)()
    first_in, second_in, first_out = threading.Event(), threading.Event(), threading.Event()
    seen = []

    def first():
        with _no_collection():
            first_in.set()
            assert second_in.wait(10)
        seen.append(gc.isenabled())  # the second is still in
        first_out.set()

    try:
        t = threading.Thread(target=first)
        t.start()
        assert first_in.wait(10)
        with _no_collection():
            second_in.set()
            assert first_out.wait(10)
            seen.append(gc.isenabled())
        t.join()
        assert seen == [False, False] and gc.isenabled() == was
        with pytest.raises(ValueError):
            with _no_collection():
                raise ValueError
        assert gc.isenabled() == was
    finally:
        (gc.enable if before else gc.disable)()
