"""The 2D BP in tiles with staged footprints and the angles split over a
group's waves, against the gathering BP.  Both round a tap's coordinate t
< 512 three times (3 * 2^-24 * 512 < 1e-4 texels); the sinogram (50 texels
or more, windowed to zero at its ends) changes by about 0.1 of its mean per
texel, so the two differ by less than 1e-5.
Tiles that the slice does not fill, the three tile shapes, fewer angles than
waves, detectors that only part of the slice projects onto, footprints of one
texel and of nearly a staged row; a slice that no footprint fits, few angles
and a source inside the slice keep the gather's floats."""
import numpy as np
import pytest

from conftest import rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("geom,w,h,na,nd,du,same", [
    ("par", 1, 1, 9, 3, 1.0, False),
    ("par", 33, 17, 15, 60, 0.9, False),
    ("fan", 65, 50, 131, 120, 1.1, False),
    ("fbp", 16, 200, 70, 301, 1.0, False),
    ("par", 60, 45, 33, 400, 0.1, False),
    ("fan", 300, 257, 40, 50, 4.0, False),
    ("par", 520, 516, 30, 500, 1.2, False),
    ("fbp", 513, 528, 70, 400, 2.9, False),
    ("par", 2050, 2040, 34, 480, 6.0, False),
    ("fan", 2049, 2033, 33, 500, 9.0, False),
    ("par", 64, 64, 7, 96, 1.0, True),
    ("par", 40, 40, 20, 500, 0.05, True),
    ("inside", 64, 64, 20, 96, 1.0, True),
])
def test_tiles_match_gather(monkeypatch, geom, w, h, na, nd, du, same):
    import torch

    import astra
    ang = np.linspace(0.05, 0.05 + 2 * np.pi, na, endpoint=False)
    vg = astra.create_vol_geom(h, w)
    m = max(w, h)
    if geom == "par":
        pg = astra.create_proj_geom("parallel", du, nd, ang)
    else:
        pg = astra.create_proj_geom("fanflat", du, nd, ang, 0.3 * m if geom == "inside" else 2.0 * m, 0.5 * m)
    k = np.arange(nd)
    y = (1.0 + 0.3 * np.sin(0.2 * k[None] + 3 * ang[:, None])) * np.sin(np.pi * (k[None] + 0.5) / nd) ** 2
    if nd < 40:
        y[:] = 1.0
    y = torch.from_numpy(y.astype(np.float32)).cuda()
    pid = astra.create_projector("cuda", pg, vg)
    out = []
    try:
        for lds in ("0", None):
            if lds:
                monkeypatch.setenv("ASTRA_AMD_BP2D_LDS", lds)
            else:
                monkeypatch.delenv("ASTRA_AMD_BP2D_LDS")
            x = torch.full((h, w), float("nan"), device="cuda")
            if geom == "fbp":
                from astra import _core, _lib
                _core.bp(astra.projector.get(pid), y, x, _lib.MODE_SET, fbp_weighted=True)
            else:
                astra.experimental.direct_BP2D(pid, x, y)
            out.append(x.cpu().numpy())
    finally:
        astra.projector.delete(pid)
    if same:
        np.testing.assert_array_equal(out[0], out[1])
    else:
        assert rel_l2(out[1], out[0]) <= 1e-5
    assert np.abs(out[0]).max() > 0
