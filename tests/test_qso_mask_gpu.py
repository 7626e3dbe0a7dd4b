"""The draw through the mask of candidate cells (smk_qso_draw_scratch) against
the draw that looks at every cell (smk_qso_draw): the same records, whatever
the cells' place in the words, blocks, chunks and columns, for fields with
infinities and NaN, and where every cell is a candidate."""
import ctypes

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _draw(d, p, vel, seed, scratch_bytes):
    """The records, sorted by key, with scratch_bytes of scratch (None: without)."""
    from saclaymocks_amd import _lib, qso
    n = d.setup.nx * d.setup.ny * d.setup.nz
    rec = torch.zeros((n, qso.RECORD.itemsize), dtype=torch.uint8, device=d.dev)
    count = torch.zeros(1, dtype=torch.int64, device=d.dev)
    args = [ctypes.byref(d.prm)] + [_lib.ptr(a) for a in (*p, *vel)]
    tail = [ctypes.c_uint64(seed), _lib.ptr(rec), n, _lib.ptr(count)]
    if scratch_bytes is None:
        _lib.check(_lib.lib().smk_qso_draw(*args, *tail, None), "smk_qso_draw")
    else:
        scratch = torch.full((scratch_bytes,), 0xff, dtype=torch.uint8, device=d.dev)
        _lib.check(_lib.lib().smk_qso_draw_scratch(*args, *tail, _lib.ptr(scratch), scratch_bytes, None), "draw")
    k = int(count.item())
    out = rec[:k].cpu().numpy().view(qso.RECORD)[:, 0]
    return out[np.argsort(out["key"])]


@pytest.mark.parametrize("shape", [(2, 3, 7), (3, 5, 63), (2, 33, 130), (1, 70, 1025), (5, 7, 2100)])
@pytest.mark.parametrize("mode", ["rsd", "zfix", "randoms", "wide", "all"])
def test_mask_draws_the_same(cuda, shape, mode):
    from saclaymocks_amd import qso
    nx, ny, nz = shape
    print(f"[qso mask] {shape} {mode}", flush=True)
    s = qso.DrawSetup(nx, ny, nz, ny, 700.0 / max(ny, nz), 700.0 / max(ny, nz), 700.0 / max(ny, nz), 0, 1, dmax=0,
                      sigma=(0.9, 1.0, 1.1), dra=80.0, ddec=80.0, rsd=mode == "rsd", randoms=mode == "randoms",
                      zfix=2.0 if mode == "zfix" else None)
    # one cell in ten passes the first condition, or every one; the others take half
    s.norm, s.density_max = (10.0 if mode == "all" else 0.05), max(s.dn_cell.max(), 1e-30)
    rng = np.random.default_rng(nz + ny)
    p = [torch.from_numpy(rng.normal(0, 4.0 if mode == "wide" else sg, shape).astype(np.float32)).to(cuda)
         for sg in s.sigma]
    for a, bad in zip(p, (float("inf"), float("nan"), -float("inf"))):
        a.view(-1)[::17] = bad
    vel = [torch.from_numpy(rng.normal(0, 400, shape).astype(np.float32)).to(cuda) for _ in range(3)]
    d = qso.Drawer(s)
    want = _draw(d, p, vel, 11, None)
    got = _draw(d, p, vel, 11, d.scratch.numel())
    assert len(got) == len(want) and got.tobytes() == want.tobytes(), (shape, mode, len(got), len(want))
    if nx * ny * nz > 4000:
        assert len(want) > 0
    with pytest.raises(ValueError):
        _draw(d, p, vel, 11, d.scratch.numel() - 8)
