"""The host rules that choose a kernel's form, called in the library itself:
no GPU is needed, a geometry's sizes and bounds are filled in by hand."""
import ctypes
import os
import shutil
import subprocess

import numpy as np
import pytest

from oracle import geometry as OG, proj3d as O3

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "astra-toolbox_amd", "csrc")
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")

DRIVER = r"""
#include "internal.hpp"
#include "forms3d.hpp"
using namespace amx;
static void fill(Geom3D &g, const unsigned *n) {
    g.kind = ASTRA_AMD_GEOM_CONE;
    g.nx = n[0]; g.ny = n[1]; g.nz = n[2]; g.na = n[3]; g.nu = n[4]; g.nv = n[5];
    g.dir_count.assign(3, 0);
}
// n: nx ny nz na nu nv; an equal part of the angles in the x- and the y-group
extern "C" int cols_rays(const unsigned *n, double spread, double typical, double slope) {
    Geom3D g;
    fill(g, n);
    g.dir_count[0] = g.dir_count[1] = (int)n[3] / 2;
    for (int k = 0; k < 2; ++k) {
        g.cols[k].ok = true;
        g.cols[k].spread = spread;
        g.cols[k].typical = typical;
        g.cols[k].slope = slope;
    }
    return fp3d_cols_rays(g, 0);
}
// bytes of the FP's volume copies; ok: the groups that columns can serve
extern "C" size_t fp_scratch(const unsigned *n, int ok, int *rays) {
    Geom3D g;
    fill(g, n);
    g.dir_count[0] = g.dir_count[1] = (int)n[3] / 2;
    for (int k = 0; k < 2; ++k) {
        g.cols[k].ok = (ok >> k) & 1;
        g.cols[k].spread = g.cols[k].typical = 1.0;
    }
    const FPForms f = fp3d_forms(g, 1);
    for (int k = 0; k < 3; ++k) rays[k] = f.rays[k];
    return f.bytes;
}
extern "C" size_t matched_scratch(const unsigned *n, int kind, int ok, unsigned ss) {
    Geom3D g;
    fill(g, n);
    g.kind = kind;
    g.dir_count[0] = g.dir_count[1] = (int)n[3] / 2;
    for (int k = 0; k < 2; ++k) {
        g.cols[k].ok = (ok >> k) & 1;
        g.cols[k].spread = g.cols[k].typical = g.cols[k].closest = 1.0;
    }
    const MatchedForms f = matched_forms(g, ss);
    return f.tables + f.geo + f.sums;
}
// ang: na rows of BP3DAngle
extern "C" int tiles_fit(const unsigned *n, const BP3DAngle *ang, double *miss) {
    Geom3D g;
    fill(g, n);
    g.tile_miss = bp3d_tile_miss(0, g.nx, g.ny, g.nz, g.nu, g.nv, ang, g.na);
    *miss = g.tile_miss;
    return bp3d_tiles_fit(g);
}
"""


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    from astra import _lib
    _lib.load()
    cxx = shutil.which("g++") or shutil.which("clang++")
    if cxx is None:
        pytest.skip("no host compiler")
    d = tmp_path_factory.mktemp("rules")
    (d / "rules.cpp").write_text(DRIVER)
    so = str(d / "rules.so")
    r = subprocess.run([cxx, "-O1", "-std=c++17", "-w", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__",
                        "-I" + CSRC, "-I" + os.path.join(ROCM, "include"), str(d / "rules.cpp"), "-o", so,
                        _lib.LIB_PATH, "-Wl,-rpath," + os.path.dirname(_lib.LIB_PATH)],
                       capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stderr
    lib = ctypes.CDLL(so)
    lib.fp_scratch.restype = lib.matched_scratch.restype = ctypes.c_size_t
    return lib


def cols_rays(rules, shape, level=False):
    """Rays per lane for unit pixels: a circular cone (source at 2 n,
    detector at n, magnification 1.5) or level parallel rays."""
    n = (ctypes.c_uint * 6)(*shape)
    nv = shape[5]
    b = (1.0, 1.0, 0.0) if level else (1.0, 1.0 / 1.5, nv / (6.0 * shape[0]))
    return rules.cols_rays(n, *(ctypes.c_double(x) for x in b))


# (nx, ny, nz, angles, columns, rows)
@pytest.mark.parametrize("shape", [
    (64, 64, 8, 720, 80, 10), (128, 128, 16, 400, 160, 20), (512, 512, 8, 60, 700, 16), (512, 512, 6, 360, 700, 8),
    (1024, 1024, 1, 360, 1024, 1), (256, 256, 1, 24, 384, 1), (256, 256, 12, 90, 332, 16), (512, 512, 12, 24, 665, 16)])
@pytest.mark.parametrize("level", [False, True], ids=["cone", "level"])
def test_few_rows_take_the_gather(rules, shape, level):
    """A column wave holds 64 rows: detectors of a few rows and many columns
    are the gather's (measured 1.2 to 10 times faster)."""
    assert cols_rays(rules, shape, level) == 0


@pytest.mark.parametrize("shape, rays", [
    ((64, 64, 64, 90, 96, 96), 2), ((64, 64, 1, 30, 96, 1), 1), ((64, 64, 48, 90, 83, 64), 1),
    ((128, 128, 48, 90, 166, 64), 1), ((256, 256, 96, 24, 332, 128), 2), ((512, 512, 512, 720, 768, 768), 4),
    # the shapes whose values are checked with 1, 3 and 4 rays per lane
    ((12, 12, 70, 300, 56, 64), 1), ((14, 12, 150, 300, 66, 192), 3), ((12, 13, 200, 300, 60, 251), 4)])
def test_columns_where_they_are_faster(rules, shape, rays):
    assert cols_rays(rules, shape) == rays


@pytest.mark.parametrize("shape, rays", [
    ((400, 391, 130, 300, 513, 140), 3), ((12, 14, 190, 300, 64, 190), 3), ((512, 512, 48, 90, 665, 64), 1), ((256, 256, 48, 360, 332, 64), 0),
    ((512, 512, 48, 360, 665, 64), 0)])
def test_level_rays(rules, shape, rays):
    """64 rows of a full chip: one ray per lane up to 32768 waves."""
    assert cols_rays(rules, shape, level=True) == rays


@pytest.mark.parametrize("slope, rays", [(8.0, 2), (10.0, 2), (10.1, 0), (15.0, 0)])
def test_steep_rays_take_the_gather(rules, slope, rays):
    """A chunk's window of rows holds the outermost rays' heights with 0.01
    rows to spare; |a| n + |c| of 8 x 10^4 rounds by half of that in fp32."""
    n = (ctypes.c_uint * 6)(64, 64, 64, 90, 96, 96)
    assert rules.cols_rays(n, *(ctypes.c_double(x) for x in (0.5, 0.4, slope))) == rays


# n^3 volume, angles, columns = rows, pixel, source and detector distance;
# share of blocks and angles whose footprint exceeds the staged tile, counted
# over all of them (every eleventh angle)
@pytest.mark.parametrize("n, na, nu, du, sod, odd, share, fits", [
    (256, 180, 384, 1.0, 1000.0, 500.0, 0.0, True),
    (256, 180, 590, 0.65, 1000.0, 500.0, 0.014, True),
    (256, 180, 698, 0.55, 1000.0, 500.0, 0.43, False),
    (256, 180, 768, 0.5, 1000.0, 500.0, 0.81, False),
    (256, 180, 960, 0.4, 1000.0, 500.0, 1.0, False),
    (256, 180, 512, 1.2, 260.0, 300.0, 0.23, False),
    (512, 720, 768, 1.0, 1000.0, 500.0, 0.0, True),
    (1024, 1440, 1536, 1.0, 1000.0, 500.0, 0.11, True)])
def test_bp_tiles_only_where_footprints_fit(rules, n, na, nu, du, sod, odd, share, fits):
    """A footprint that is not staged costs two gathers an update: detectors
    of fine pixels keep the gather from pairs (measured 1.2 to 1.6 times faster)."""
    vecs, vs = OG.normalise_3d(OG.gen_cone_projections(np.linspace(0, 2 * np.pi, na, endpoint=False), nu, nu, sod, odd,
                                                       du, du), "cone", OG.vol_geom_3d(n, n, n))
    c = np.zeros((na, 3, 4), np.float32)
    for a in range(na):
        u, v, d = O3.cone_bp_params(vecs[a], "default", vs)
        c[a] = np.array([np.add(u, 1.5 * np.asarray(d)), np.add(v, 1.5 * np.asarray(d)), d])
    miss = ctypes.c_double()
    got = rules.tiles_fit((ctypes.c_uint * 6)(n, n, n, na, nu, nu), c.ctypes.data_as(ctypes.c_void_p),
                          ctypes.byref(miss))
    assert abs(miss.value - share) <= 0.07 and bool(got) == fits


@pytest.mark.parametrize("ok", [0, 1, 2, 3])
@pytest.mark.parametrize("shape", [(600, 200, 400, 720, 900, 500), (64, 48, 50, 90, 96, 96), (3, 700, 300, 200, 900, 400),
                                   (1, 1, 500, 100, 5, 700)])
def test_fp_scratch_is_what_the_planner_counts(rules, shape, ok):
    """Groups of different forms use one buffer in turn."""
    from astra import composite
    rays = (ctypes.c_int * 3)()
    got = rules.fp_scratch((ctypes.c_uint * 6)(*shape), ok, rays)
    assert all(not r or (ok >> k) & 1 for k, r in enumerate(rays))
    assert 0 < got <= composite._fp_scratch(shape[2::-1])


@pytest.mark.parametrize("ss", [1, 3])
@pytest.mark.parametrize("ok", [0, 1, 3])
@pytest.mark.parametrize("shape", [(256, 256, 256, 360, 384, 384), (600, 200, 400, 720, 900, 500),
                                   (400, 400, 300, 4, 128, 100), (64, 48, 50, 90, 96, 96), (64, 48, 50, 90, 96, 1),
                                   (20, 20, 20, 2, 3000, 3000)])
def test_matched_scratch_is_what_the_planner_counts(rules, shape, ok, ss):
    from astra import _lib, composite
    nx, ny, nz, na, nu, nv = shape
    for kind in (_lib.GEOM_CONE, _lib.GEOM_PAR3D):
        got = rules.matched_scratch((ctypes.c_uint * 6)(*shape), kind, ok, ss)
        assert 0 < got <= composite._matched_scratch((nz, ny, nx), (nv, na, nu), ss)
    assert got >= (nx * ny * nz * 4 if ok and ss == 1 else 0)
