"""The transpose of the column FP (adj3d_cols.hip) against the FP64 oracle's
exact transpose, at the edges of its tiles: volumes that do not fill 4
slices, 8 rows or 64 z, one z or two per lane, one row or column of the
detector, columns that miss the volume, and spacings whose candidates do not
fit a wave's window (the general gather takes those).  rel-L2 <= 1e-5."""
import numpy as np
import pytest

from conftest import rel_l2

pytestmark = pytest.mark.gpu

# kind, (nx, ny, nz), angles, nu, nv, du, dv, sod, odd
CASES = {
    "ragged": ("cone", (13, 18, 21), 13, 26, 31, 1.0, 1.0, 70.0, 35.0),
    "one_slice": ("cone", (12, 12, 1), 10, 18, 6, 1.0, 1.0, 60.0, 30.0),
    "z_65": ("cone", (9, 10, 65), 8, 20, 100, 1.0, 1.0, 120.0, 60.0),
    "z_131": ("par3d", (8, 9, 131), 7, 15, 140, 1.0, 1.0, 0, 0),
    "one_detector_row": ("cone", (11, 9, 8), 9, 21, 1, 1.0, 1.0, 50.0, 20.0),
    "one_detector_column": ("cone", (10, 11, 9), 9, 1, 17, 1.4, 1.0, 50.0, 20.0),
    "detector_off_volume": ("cone", (10, 10, 30), 9, 60, 12, 1.3, 1.0, 50.0, 20.0),
    "close_rows": ("cone", (8, 8, 20), 6, 14, 60, 1.0, 0.4, 60.0, 20.0),
    "too_close_rows": ("cone", (8, 8, 24), 6, 14, 90, 1.0, 0.15, 40.0, 40.0),
    "wide_rows_and_columns": ("par3d", (14, 12, 33), 9, 7, 9, 2.6, 3.7, 0, 0),
}


@pytest.mark.parametrize("name", list(CASES))
def test_adj_cols(name):
    import astra
    import torch
    from astra import autograd as AG
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
    vec, vs = OG.normalise_3d(vec, kind, vg)
    y = np.random.default_rng(nx + nv).random((nv, na, nu), dtype=np.float32)
    pid = astra.create_projector("cuda3d", pg, vg)
    got = AG.back_project(torch.from_numpy(y).cuda(), pid).cpu().numpy()
    astra.projector3d.delete(pid)
    T = O3.par3d_fp_T if kind == "par3d" else O3.cone_fp_T
    want = T(y.astype(np.float64), vec, (nz, ny, nx), vs)
    assert np.abs(want).max() > 0
    assert rel_l2(got, want) <= 1e-5
