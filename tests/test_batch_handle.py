"""The native batch behind a Batch and its frame lives as long as either: the frame's
handle is the batch's, which a frame taken from a released Batch still uses."""
import ctypes as C
import gc

import pytest

import tileink_amd as tk
from tileink_amd import _abi


class _Library:
    """Stands in for the native library: counts what is created and destroyed."""

    def __init__(self):
        self.destroyed = []

    def tk_batch_create(self, context, scenes, count, out):
        C.cast(out, C.POINTER(C.c_void_p))[0] = 0x1000
        return 0

    def tk_batch_frame(self, batch):
        return 0x2000

    def tk_batch_destroy(self, batch):
        self.destroyed.append(("batch", batch.value))

    def tk_frame_destroy(self, frame):
        self.destroyed.append(("frame", frame.value))


class _Context:
    handle = C.c_void_p(1)


@pytest.mark.parametrize("last", ["frame", "batch"])
def test_the_native_batch_outlives_both_holders(monkeypatch, last):
    library = _Library()
    monkeypatch.setattr(tk, "lib", lambda: library)
    gc.disable()  # released by reference count alone, as before
    try:
        batch = tk.Batch(_Context(), [_abi.Scene()])
        frame = batch.frame
        assert frame._h.value == 0x2000
        if last == "frame":
            del batch
            assert library.destroyed == []
            del frame
        else:
            del frame
            assert library.destroyed == []
            del batch
        assert library.destroyed == [("batch", 0x1000)]
    finally:
        gc.enable()


def test_a_failed_creation_destroys_nothing(monkeypatch):
    library = _Library()
    library.tk_batch_create = lambda *a: _abi.TK_ERR_INVALID
    library.tk_last_error = lambda: b"refused"
    monkeypatch.setattr(tk, "lib", lambda: library)
    with pytest.raises(tk.TileinkError):
        tk.Batch(_Context(), [_abi.Scene()])
    gc.collect()
    assert library.destroyed == []
