"""Control blocks and streams, without a GPU: which block Extractor.ctl_for hands out.

A forward returns while its count kernel may still be using its control block, so two streams must
never share one; a capture needs a block whose memory outlives it."""
import ctypes

import pytest
import torch

from diso_amd import _lib, engine

CPU = torch.device("cpu")
FLAGS = _lib.FLAG_VIRTUAL_PAD


@pytest.fixture
def on(monkeypatch):
    """Sets the handle of the current stream and whether it is capturing."""
    now = {"stream": 0, "capturing": False}
    monkeypatch.setattr(engine, "_stream", lambda device: ctypes.c_void_p(now["stream"]))
    monkeypatch.setattr(engine, "_capturing", lambda: now["capturing"], raising=False)
    return lambda stream, capturing=False: now.update(stream=stream, capturing=capturing)


def test_each_stream_has_its_own_block(on):
    ex = engine.Extractor(_lib.MC, torch.float32)
    seen = {}
    for handle in (0, 0x1000, 0x2000, 0x1000, 0):
        on(handle)
        ctl = ex.ctl_for(CPU, (8, 9, 10), FLAGS)
        assert ctl.numel() >= _lib.lib().diso_ctl_bytes(8, 9, 10, FLAGS) and not ctl.any()
        assert seen.setdefault(handle, ctl) is ctl  # and keeps it
    assert len({c.data_ptr() for c in seen.values()}) == 3


def test_capture_uses_a_block_that_outlives_it(on):
    ex = engine.Extractor(_lib.DMC, torch.float32)
    args = (CPU, (8, 8, 8), FLAGS)
    on(0x2000, capturing=True)
    assert not ex.ctl_for(*args).any() and not ex._ctl  # cleared by the replays alone: not kept
    on(0x1000)
    warm = ex.ctl_for(*args)
    on(0x2000, capturing=True)
    assert ex.ctl_for(*args) is warm
    on(0x2000)  # the same stream outside the capture
    assert ex.ctl_for(*args) is not warm
    on(0x2000, capturing=True)  # which may now be dropped; the captured one not
    assert ex.ctl_for(*args, capturing=True) is warm
    for handle in range(1, 200):
        on(0x10000 * handle)
        ex.ctl_for(*args)
        assert len(ex._ctl) <= 64
    on(0x3000, capturing=True)
    assert ex.ctl_for(*args) is warm
