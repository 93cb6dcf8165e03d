"""The 2D FP with slice rows staged in LDS against the gathering FP: the same
samples in the same order, so the same floats.  Slices and detectors around a
wave's 64 detectors and a chunk's 16 slices, one, two and three angles per
wave (by the number of waves), rays along both axes in one wave, detectors
wide enough that a chunk exceeds its buffer, sub-rays, infinities, and a
source next to or on the detector's line, whose rays run along the slices
(positions that round by texels, or are NaN)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("geom,w,h,na,nd,du,ss", [
    ("par", 1, 1, 1, 1, 1.0, 1),
    ("par", 64, 17, 5, 65, 0.9, 1),
    ("par", 33, 40, 401, 700, 0.06, 1),
    ("par", 40, 31, 1501, 705, 0.05, 1),
    ("par", 300, 15, 9, 130, 3.5, 2),
    ("fan", 16, 200, 7, 63, 2.5, 1),
    ("fan", 97, 64, 400, 720, 0.3, 1),
    ("fan", 24, 33, 1501, 705, 0.1, 1),
    ("wide", 130, 129, 30, 300, 2.0, 3),
    ("steep", 200, 210, 6, 64, 0.9, 1),
    ("steep", 97, 300, 6, 200, 0.1, 2),
])
def test_staged_equals_gather(monkeypatch, geom, w, h, na, nd, du, ss):
    import torch

    import astra
    ang = np.linspace(0.05, 0.05 + 2 * np.pi, na, endpoint=False)
    vg = astra.create_vol_geom(h, w)
    if geom == "par":
        pg = astra.create_proj_geom("parallel", du, nd, ang)
    elif geom == "steep":
        gaps = [1e-1, 1e-3, 1e-4, 1e-5, 0.0, 3.0]
        pg = astra.create_proj_geom("fanflat_vec", nd, np.array([[3.3, 7.5, 3.0, 7.5 - g, du, 0.0] for g in gaps]))
    else:
        sod = max(w, h) * (0.8 if geom == "wide" else 2.0)
        pg = astra.create_proj_geom("fanflat", du, nd, ang, sod, 0.1 * sod)
    pid = astra.create_projector("cuda", pg, vg, options={"DetectorSuperSampling": ss})
    gen = torch.Generator().manual_seed(w + 7 * nd)
    vol = torch.randn(h, w, generator=gen).cuda()
    if w > 60:
        vol[h // 2, w // 3] = float("inf")
    out = []
    try:
        for lds in ("0", "1"):
            monkeypatch.setenv("ASTRA_AMD_FP2D_LDS", lds)
            y = torch.full((na, nd), float("nan"), device="cuda")
            astra.experimental.direct_FP2D(pid, vol, y)
            out.append(y.cpu().numpy())
    finally:
        astra.projector.delete(pid)
    np.testing.assert_array_equal(out[0], out[1])
    assert np.abs(np.nan_to_num(out[0], posinf=0, neginf=0)).max() > 0
