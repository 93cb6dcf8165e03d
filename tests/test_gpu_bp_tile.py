"""The 3D BP's two forms beside the gather: angles split over a workgroup's
waves (small volumes) against the FP64 oracle, with fewer angles than waves
and volumes that do not fill a tile (rel-L2 <= 1e-5), and staged footprints
(large volumes), which give the gather's floats, on ragged volumes, angle
counts around the footprint group of 128, and detectors that only part of
the volume projects onto."""
import numpy as np
import pytest

from conftest import rel_l2

pytestmark = pytest.mark.gpu


def _geom(kind, nx, ny, nz, na, nu, nv, sod, odd):
    import astra
    vg = astra.create_vol_geom(ny, nx, nz)
    ang = np.linspace(0.1, 0.1 + 2 * np.pi, na, endpoint=False)
    if kind == "par3d":
        return vg, astra.create_proj_geom("parallel3d", 1.1, 0.9, nv, nu, ang), ang
    return vg, astra.create_proj_geom("cone", 1.2, 1.1, nv, nu, ang, sod, odd), ang


@pytest.mark.parametrize("na", [1, 3, 4, 6])
@pytest.mark.parametrize("kind,n", [("cone", (9, 17, 5)), ("par3d", (8, 7, 3)), ("cone", (1, 1, 1))])
def test_split_bp(kind, n, na):
    import astra
    import torch
    from oracle import geometry as OG, proj3d as O3
    nx, ny, nz = n
    nu, nv = 21, 13
    vg, pg, ang = _geom(kind, nx, ny, nz, na, nu, nv, 60.0, 30.0)
    if kind == "par3d":
        vec, vs = OG.normalise_3d(OG.gen_par3d_projections(ang, nu, nv, 1.1, 0.9), kind, vg)
        bp = O3.par3d_bp
    else:
        vec, vs = OG.normalise_3d(OG.gen_cone_projections(ang, nu, nv, 60.0, 30.0, 1.2, 1.1), kind, vg)
        bp = O3.cone_bp
    y = np.random.default_rng(nx + na).random((nv, na, nu), dtype=np.float32)
    pid = astra.create_projector("cuda3d", pg, vg)
    vol = torch.full((nz, ny, nx), float("nan"), dtype=torch.float32, device="cuda")
    astra.experimental.direct_BP3D(pid, vol, torch.from_numpy(y).cuda())
    astra.projector3d.delete(pid)
    assert rel_l2(vol.cpu().numpy(), bp(y.astype(np.float64), vec, (nz, ny, nx), vs)) <= 1e-5


@pytest.mark.parametrize("case", [("cone", 161, 170, 159, 5, 190, 200, 400.0, 200.0),
                                  ("cone", 176, 160, 150, 130, 100, 60, 300.0, 150.0),
                                  ("cone", 168, 168, 168, 7, 300, 300, 130.0, 300.0),
                                  ("par3d", 165, 163, 161, 3, 240, 170, 0, 0)],
                         ids=["ragged", "small_detector_130_angles", "near_source", "par3d"])
def test_tile_bp_equals_gather(case, monkeypatch):
    import astra
    import torch
    kind, nx, ny, nz, na, nu, nv, sod, odd = case
    vg, pg, _ = _geom(kind, nx, ny, nz, na, nu, nv, sod, odd)
    g = torch.Generator(device="cuda").manual_seed(3)
    y = torch.rand((nv, na, nu), generator=g, device="cuda")
    pid = astra.create_projector("cuda3d", pg, vg)
    out = {}
    for lds in ("0", "1", None):  # gather, tiles, the one the rule takes
        monkeypatch.setenv("ASTRA_AMD_BP3D_LDS", lds) if lds else monkeypatch.delenv("ASTRA_AMD_BP3D_LDS")
        out[lds] = torch.full((nz, ny, nx), float("nan"), dtype=torch.float32, device="cuda")
        astra.experimental.direct_BP3D(pid, out[lds], y)
    astra.projector3d.delete(pid)
    assert float(out["0"].abs().max()) > 0
    assert torch.equal(out["0"], out["1"]) and torch.equal(out["0"], out[None])
