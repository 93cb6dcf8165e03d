"""The par3d BP that back projects each detector row in 2D and interpolates
between the row images, against the gathering BP.  Both round a tap's
coordinates (t < 512) a few times, 1e-4 texels at most; the projections
change by about 0.1 of their mean per texel: rel-L2 <= 1e-5.  Ragged tiles,
rows in several chunks, slices off the detector, both weights, non-cubic
voxels, and the update mode of SIRT; a tilted detector, few angles and more
than 1.5 rows a slice keep the other forms (equal floats with 3D tiles)."""
import numpy as np
import pytest

from conftest import rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny,nz,na,nu,nv,dv,kern,win,same", [
    (100, 97, 200, 17, 150, 130, 1.0, "default", None, False),
    (48, 45, 920, 16, 60, 300, 3.1, "default", None, False),      # three chunks of rows
    (130, 65, 120, 40, 150, 90, 0.8, "2d_weighting", None, False),
    (96, 96, 300, 20, 140, 120, 1.0, "default", (2.0, 1.0), False),  # slices above and below the detector
    (100, 97, 400, 15, 150, 130, 1.0, "default", None, True),
    (100, 97, 400, 20, 150, 450, 0.45, "default", None, True),
    (100, 97, 400, 20, 150, 130, None, "default", None, True),
])
def test_flat_matches(monkeypatch, nx, ny, nz, na, nu, nv, dv, kern, win, same):
    import torch

    import astra
    ang = np.linspace(0.1, 0.1 + np.pi, na, endpoint=False)
    if win:
        vg = astra.create_vol_geom(ny, nx, nz, -nx * win[1] / 2, nx * win[1] / 2, -ny * win[1] / 2, ny * win[1] / 2,
                                   -nz * win[0] / 2, nz * win[0] / 2)
    else:
        vg = astra.create_vol_geom(ny, nx, nz)
    pg = astra.create_proj_geom("parallel3d", 1.1, dv or 1.0, nv, nu, ang)
    if dv is None:  # the detector leans
        pg = astra.geom_2vec(pg)
        pg["Vectors"][:, 9] = 0.02
    pid = astra.create_projector("cuda3d", pg, vg, options={"ProjectionKernel": kern})
    k, r = np.arange(nu), np.arange(nv)
    y = (1 + 0.3 * np.sin(0.2 * k + 3 * ang[:, None])) * np.sin(np.pi * (k + 0.5) / nu) ** 2
    y = (y[None] * (1 + 0.3 * np.cos(0.2 * r))[:, None, None] * np.sin(np.pi * (r + 0.5) / nv)[:, None, None] ** 2)
    y = torch.from_numpy(y.astype(np.float32)).cuda()
    out = []
    try:
        for lds in ("1" if same else "0", None):
            if lds:
                monkeypatch.setenv("ASTRA_AMD_BP3D_LDS", lds)
            else:
                monkeypatch.delenv("ASTRA_AMD_BP3D_LDS")
            x = torch.full((nz, ny, nx), float("nan"), device="cuda")
            astra.experimental.direct_BP3D(pid, x, y)
            out.append(x.cpu().numpy())
            if kern == "default" and not same:
                v = torch.full((nz, ny, nx), 0.1, device="cuda")
                d, p = astra.data3d.link("-vol", vg, v), astra.data3d.link("-sino", pg, y)
                cfg = astra.astra_dict("SIRT3D_CUDA")
                cfg.update(ReconstructionDataId=d, ProjectionDataId=p, option={"MinConstraint": 0.0})
                a = astra.algorithm.create(cfg)
                astra.algorithm.run(a, 2)
                astra.algorithm.delete(a)
                astra.data3d.delete([d, p])
                out.append(v.cpu().numpy())
    finally:
        astra.projector3d.delete(pid)
    h = len(out) // 2
    for got, ref in zip(out[h:], out[:h]):
        if same:
            np.testing.assert_array_equal(got, ref)
        else:
            assert rel_l2(got, ref) <= 1e-5
        assert np.abs(ref).max() > 0
