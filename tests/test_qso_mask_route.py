"""When the quasar draw goes through the mask of candidates, as measured."""
import pytest

from saclaymocks_amd import qso


@pytest.mark.parametrize("shape,mask", [((160, 2560, 1536), True), ((40, 512, 512), True), ((10, 800, 1200), True),
                                        ((40, 400, 300), False), ((10, 300, 300), False), ((2, 3, 7), False)])
def test_mask_pays(shape, mask):
    assert qso.mask_pays(*shape) == mask


def test_drawer_follows_the_rule(monkeypatch):
    """The scratch buffer that launch hands to the library."""
    seen = []

    class Library:
        def smk_qso_draw_scratch(self, *args):
            seen.append((args[-3], args[-2]))
            return 0

    monkeypatch.setattr(qso._lib, "lib", lambda: Library())
    monkeypatch.setattr(qso._lib, "stream_ptr", lambda stream: None)
    monkeypatch.setattr(qso._lib, "ptr", lambda t: None if t is None else id(t))
    import ctypes
    import types

    import torch
    for shape in ((160, 2560, 1536), (10, 300, 300)):
        d = object.__new__(qso.Drawer)
        d.setup = types.SimpleNamespace(nx=shape[0], ny=shape[1], nz=shape[2])
        d.prm = type("P", (ctypes.Structure,), {"_fields_": [("rsd", ctypes.c_int)]})()
        d.records, d.count, d.capacity = torch.zeros(1), torch.zeros(1), 1
        d.scratch = torch.zeros(64, dtype=torch.uint8)
        d.launch(None, None, None)
        assert seen[-1] == ((id(d.scratch), 64) if qso.mask_pays(*shape) else (None, 0))
