"""The 3D FP over columns of rays (detectors whose v axis is the z axis)
against the FP64 oracle, at the edges of its tiles: rows that do not fill a
block of 64, one row, one slice, one column, thin volumes, rays above and
below the volume and a shifted (helical) source, each number of rays per
lane, and spacings whose windows need one more block of rows or leave the
kernel (the gather takes those).  One projection: rel-L2 <= 1e-5."""
import numpy as np
import pytest

from conftest import rel_l2

pytestmark = pytest.mark.gpu

# kind, (nx, ny, nz), angles, nu, nv, du, dv, sod, odd
CASES = {
    "small_65_rows": ("cone", (31, 28, 40), 24, 37, 65, 1.0, 1.0, 120.0, 60.0),
    "small_1_row": ("cone", (20, 23, 9), 11, 30, 1, 1.0, 1.0, 90.0, 40.0),
    "one_slice": ("cone", (26, 26, 1), 16, 33, 17, 1.0, 0.8, 100.0, 50.0),
    "one_column": ("cone", (17, 19, 30), 9, 1, 70, 1.5, 1.1, 80.0, 30.0),
    "one_voxel_wide": ("par3d", (1, 24, 33), 10, 29, 50, 1.0, 1.0, 0, 0),
    "rays_off_volume": ("cone", (24, 24, 12), 12, 40, 200, 1.2, 1.2, 90.0, 45.0),
    "wide_rows": ("cone", (24, 24, 60), 12, 40, 130, 1.0, 2.2, 120.0, 20.0),
    "too_wide_rows": ("cone", (24, 24, 60), 12, 40, 90, 1.0, 4.5, 120.0, 10.0),
    "par3d_129_rows": ("par3d", (33, 30, 90), 14, 45, 129, 1.1, 0.9, 0, 0),
    "rays_1": ("cone", (12, 12, 70), 300, 56, 64, 1.0, 1.5, 60.0, 5.0),
    "rays_3": ("cone", (14, 12, 150), 300, 66, 192, 1.0, 1.0, 200.0, 60.0),
    "rays_3_par": ("par3d", (12, 14, 190), 300, 64, 190, 1.0, 1.0, 0, 0),
    "rays_4": ("cone", (12, 13, 200), 300, 60, 251, 1.0, 1.0, 260.0, 80.0),
}


@pytest.mark.parametrize("name", list(CASES))
def test_cols_fp(name):
    import astra
    from oracle import geometry as OG, proj3d as O3
    kind, (nx, ny, nz), na, nu, nv, du, dv, sod, odd = CASES[name]
    vg = astra.create_vol_geom(ny, nx, nz)
    ang = np.linspace(0.1, 0.1 + 2 * np.pi, na, endpoint=False)
    if kind == "par3d":
        pg = astra.create_proj_geom("parallel3d", du, dv, nv, nu, ang)
        vec = OG.gen_par3d_projections(ang, nu, nv, du, dv)
    else:
        pg = astra.create_proj_geom("cone", du, dv, nv, nu, ang, sod, odd)
        vec = OG.gen_cone_projections(ang, nu, nv, sod, odd, du, dv)
    _check(pg, vg, vec, kind, (nx, ny, nz), nu, nv)


def test_cols_fp_helical():
    """Source and detector move along z from angle to angle; anisotropic voxels."""
    import astra
    from oracle import geometry as OG
    nx, ny, nz, na, nu, nv = 22, 25, 48, 30, 41, 77
    vg = astra.create_vol_geom(ny, nx, nz, -11, 11, -12.5, 12.5, -30, 30)
    rows = []
    for i, a in enumerate(np.linspace(0, 4 * np.pi, na, endpoint=False)):
        z = 40.0 * (i / na - 0.5)
        c, s = np.cos(a), np.sin(a)
        rows.append([90 * s, -90 * c, z, -45 * s, 45 * c, z, 1.1 * c, 1.1 * s, 0, 0, 0, 0.9])
    rows = np.array(rows)
    pg = astra.create_proj_geom("cone_vec", nv, nu, rows)
    _check(pg, vg, OG.conevec_from_astra(rows, nu, nv), "cone", (nx, ny, nz), nu, nv)


def test_groups_of_both_forms_share_one_buffer():
    """Upright detectors in the x-group, tilted ones in the y-group: the
    columns' and the gather's copies of the volume use one buffer in turn, no
    more scratch than the job splitter counts."""
    import astra
    import torch
    from astra import _lib, composite
    from oracle import geometry as OG
    nx, ny, nz, nu, nv = 44, 40, 72, 50, 65
    vg = astra.create_vol_geom(ny, nx, nz)
    rows = []
    for a in np.linspace(0.1, 0.1 + 2 * np.pi, 60, endpoint=False):
        c, s = np.cos(a), np.sin(a)
        t = 0.0 if abs(s) > abs(c) else 0.1
        rows.append([130 * s, -130 * c, 0, -60 * s, 60 * c, 0, c, s, 0, -t * s, t * c, 1.0])
    rows = np.array(rows)
    pg = astra.create_proj_geom("cone_vec", nv, nu, rows)
    torch.cuda.synchronize()
    base, _ = _lib.scratch_usage(reset_peak=True)
    _check(pg, vg, OG.conevec_from_astra(rows, nu, nv), "cone", (nx, ny, nz), nu, nv)
    _, peak = _lib.scratch_usage()
    assert peak - base <= composite._fp_scratch((nz, ny, nx)) + 65536  # tickets, allocation grain


def _check(pg, vg, vec, kind, n, nu, nv):
    import astra
    import torch
    from oracle import geometry as OG, proj3d as O3
    nx, ny, nz = n
    vec, vs = OG.normalise_3d(vec, kind, vg)
    vol = np.random.default_rng(nx + nv).random((nz, ny, nx), dtype=np.float32)
    pid = astra.create_projector("cuda3d", pg, vg)
    proj = torch.full((nv, len(vec), nu), float("nan"), dtype=torch.float32, device="cuda")
    astra.experimental.direct_FP3D(pid, torch.from_numpy(vol).cuda(), proj)
    fp = O3.par3d_fp if kind == "par3d" else O3.cone_fp
    want = fp(vol.astype(np.float64), vec, nu, nv, vs)
    got = proj.cpu().numpy()
    astra.projector3d.delete(pid)
    assert np.abs(want).max() > 0
    assert rel_l2(got, want) <= 1e-5
