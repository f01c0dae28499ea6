"""A step is captured with cyclic garbage collection off: an unreachable older graph freed in between would synchronize
the device inside the capture."""
import contextlib
import gc

import pytest
import torch


@pytest.mark.parametrize("on", [True, False])
def test_no_collection_during_a_capture(monkeypatch, on):
    from leankv_amd.engine import _capture

    monkeypatch.setattr(torch.cuda, "graph", lambda graph, stream=None: contextlib.nullcontext())
    freed = []

    class Old:
        def __init__(self):
            self.me = self

        def __del__(self):
            freed.append(1)

    old = gc.get_threshold(), gc.isenabled()
    try:
        (gc.enable if on else gc.disable)()
        with pytest.raises(ValueError):
            with _capture(None, None):
                gc.set_threshold(1, 1, 1)
                Old()
                [[] for _ in range(1000)]
                assert not freed
                raise ValueError  # a failed capture restores the setting too
        assert gc.isenabled() is on
        gc.collect()
        assert freed
    finally:
        gc.set_threshold(*old[0])
        (gc.enable if old[1] else gc.disable)()


def test_no_collection_while_another_thread_captures(monkeypatch):
    """The first capture to end leaves the collector off for the one still running."""
    import threading

    from leankv_amd.engine import _capture

    monkeypatch.setattr(torch.cuda, "graph", lambda graph, stream=None: contextlib.nullcontext())
    first_in, second_in, first_out = threading.Event(), threading.Event(), threading.Event()

    def first():
        with _capture(None, None):
            first_in.set()
            second_in.wait(10)
        first_out.set()

    was = gc.isenabled()
    try:
        gc.enable()
        t = threading.Thread(target=first)
        t.start()
        assert first_in.wait(10)
        with _capture(None, None):
            second_in.set()
            assert first_out.wait(10)
            assert not gc.isenabled()
        assert gc.isenabled()
        t.join(10)
    finally:
        (gc.enable if was else gc.disable)()
