"""A context's handle keeps the context alive as long as the handle is held (no GPU needed)."""

import ctypes
import gc

from heraclespp_amd import hydro


def test_handle_keeps_its_context_alive(monkeypatch):
    destroyed = []

    class _Lib:
        def hclpp_set_stream(self, h, stream):
            return 0

        def hclpp_ctx_destroy(self, h):
            destroyed.append(h.value)

    class _Stream:
        cuda_stream = 0

    monkeypatch.setattr(hydro, "lib", lambda: _Lib())
    monkeypatch.setattr(hydro.torch.cuda, "current_stream", lambda: _Stream())
    c = hydro.Context.__new__(hydro.Context)
    c._h = ctypes.c_void_p(4096)
    h = c.handle
    del c
    gc.collect()
    assert h.value == 4096 and not destroyed
    del h
    gc.collect()
    assert destroyed == [4096]
