"""The staged BPs take every tap from the texels they staged, at LDS addresses
that nothing checks: the footprint of a tile has to hold the taps of all its
lanes, those past the edge of the volume included.

These CPU tests compile the kernels' own text -- `bp_footprint` and
`bp_tile_angle` of csrc/bp3d_tile.hip, `bp2d_footprint`, `bp2d_angle` and the
lines of `bp2d_wave` that choose corners and clamps in csrc/proj2d_dev.hpp --
for the host, with a checked pointer in the place of the LDS address, and
run every lane of every tile over whole geometries.  Planted mistakes (the
footprint of the block's first z slice, of the tile's first row, of the part
of a tile inside the slice) must be caught.
"""
import ctypes
import math
import os
import re
import shutil
import subprocess

import numpy as np
import pytest

from oracle import geometry as OG, proj3d as O3

f32 = np.float32
CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "astra-toolbox_amd", "csrc")

PRELUDE = r"""
#include <algorithm>
#include <cmath>
#include <cstddef>
#include <cstdint>
#include <vector>
using std::max;
using std::min;
#define __device__
#define __host__
#define __forceinline__ inline
constexpr int kPad = 2;
typedef int __amdgpu_buffer_rsrc_t;
struct float4 { float x, y, z, w; };
static float4 make_float4(float x, float y, float z, float w) { return {x, y, z, w}; }
struct BP2DAngle { float num[3], den[3], w, pad_; };
struct BP3DAngle { float nu[4], nv[4], dn[4]; };
static float med3(float x, float lo, float hi) {  // v_med3_f32: NaN gives the least of the others
    return std::isnan(x) ? std::min(lo, hi) : std::min(std::max(x, lo), hi);
}
static float clamp_pad(float p, float hi) { return med3(p, 0.5f, hi); }
static float frac(float p) { return p - std::floor(p); }
static float lerp(float a, float b, float w) { return std::fma(w, b - a, a); }
static float bilerp_pairs(float4 q, float w1, float w2) {
    return lerp(std::fma(w2, q.y, q.x), std::fma(w2, q.w, q.z), w1);
}
static unsigned cvt_u32(float x) {  // v_cvt_u32_f32
    return !(x > 0.f) ? 0u : x >= 4294967040.f ? 0xffffffffu : (unsigned)x;
}
static unsigned mul24(unsigned a, unsigned b) { return (a & 0xffffff) * (b & 0xffffff); }
static float load_b32(int, int, int, int) { return 0.f; }
// a vote of a wave's lanes, each with an angle of its own
static bool others_fit = true;
static bool __all(bool x) { return x && others_fit; }
// LDS pointer: counts the reads outside the staged texels [base, end)
static unsigned lds_base, lds_end;
static long outside;
struct Lds {
    unsigned a;
    explicit Lds(size_t x) : a((unsigned)x) {}
    float operator[](int i) const {
        const unsigned p = a + 4u * (unsigned)i;
        if (p < lds_base || p >= lds_end) ++outside;
        return 0.f;
    }
};
"""

SUBST = [
    (r"typedef const __attribute__\(\(address_space\(3\)\)\) float \*lptr;", "typedef Lds lptr;"),
    (r"\(unsigned\)(t|pu|pv)\b", r"cvt_u32(\1)"),
    (r"__builtin_amdgcn_fmed3f", "med3"),
    (r"__builtin_amdgcn_rcpf\(", "(1.f / "),
    (r"__builtin_amdgcn_raw_buffer_load_b32", "load_b32"),
    (r"__int_as_float", ""),
    (r"__umul24", "mul24"),
    (r"__builtin_amdgcn_sched_barrier\(0\);", ""),
    (r"__builtin_isfinite", "std::isfinite"),
    (r'asm(?: volatile)?\("".*?\);', ""),
]


def source(name):
    return open(os.path.join(CSRC, name)).read()


def part(text, first, last, include_last=False):
    """`text` from the marker `first` to the marker `last`."""
    a = text.index(first)
    b = text.index(last, a) + (len(last) if include_last else 0)
    return text[a:b]


def host(text):
    for pat, rep in SUBST:
        text = re.sub(pat, rep, text, flags=re.S)
    return text


def harness_2d():
    src = source("proj2d_dev.hpp")
    code = part(src, "constexpr int kBp2KA", "// Sums over the angles [alo, ahi)")
    corners = part(src, "    const float fx = (X0 + lane % LX)", "    const unsigned step")
    call = re.search(r"pk = (\w+\()ang\[.*?\]\);\n", src).group(1) + "c)"
    choose = part(src, "            if (f >> 30)", "k * step, rs, acc);", True)
    whole = "Y1 = Y0 + 64 / LX * TY - 1;"  # the corners of the first try
    assert corners.count(whole) == 1
    corners = corners.replace(whole, whole + """
        if (plant == 1) Y1 = Y0;
        if (plant == 2) X1 = min(X1, (int)w - 1), Y1 = min(Y1, (int)h - 1);
""")
    return host(code) + r"""
template <int KIND, int LX, int TX, int TY>
long run2d(unsigned w, unsigned h, unsigned na, unsigned nd, const BP2DAngle *ang, int plant, long *staged) {
    outside = 0;
    others_fit = plant != 3;
    lds_base = 1u << 28;
    for (int Y0 = 0; Y0 < (int)h; Y0 += 64 / LX * TY)
        for (int X0 = 0; X0 < (int)w; X0 += LX * TX)
            for (unsigned a = 0; a < na; ++a) {
                const BP2DAngle c = ang[a];
                for (int lane = 0; lane < 64; ++lane) {
                    """ + host(corners) + r"""
                    const int f = """ + call + r""";
                    if (!(f >> 20)) break;
                    if (lane == 0) ++*staged;
                    lds_end = lds_base + 4u * ((f >> 20) & 0x3ff);
                    const unsigned at = lds_base - 4u * (f & 0xfffff), k = 0, step = 0;
                    const int rs = 0;
                    float acc[TY][TX] = {};
                    """ + host(choose) + r"""
                }
            }
    return outside;
}
extern "C" long check2d(int kind, int form, unsigned w, unsigned h, unsigned na, unsigned nd, const BP2DAngle *ang,
                        int plant, long *staged) {
#define FORM(i, LX, TX, TY)                                                              \
    if (form == i) return kind == 0 ? run2d<0, LX, TX, TY>(w, h, na, nd, ang, plant, staged) \
                                    : run2d<1, LX, TX, TY>(w, h, na, nd, ang, plant, staged);
    FORM(0, 8, 2, 2) FORM(1, 8, 4, 2) FORM(2, 8, 4, 4) FORM(3, 64, 1, 2) FORM(4, 64, 1, 4) FORM(5, 64, 1, 8)
    return -1;
}
"""


def harness_3d():
    src = source("bp3d_tile.hip")
    code = part(src, "constexpr int kTileRows", "}  // namespace") + \
        part(src, "struct BPFoot {", "// Barrier that orders LDS only") + \
        part(src, "template <int KIND, int ZS, bool CLIP>", "// The same from memory")
    kernel = part(src, "void bp3d_tile_kernel(BPArgs A)", "// ---", False)
    place = part(kernel, "    const unsigned tiles_x", "    const unsigned lds")
    ray = part(kernel, "            const float un =", "            const float wgt")
    zs = re.search(r"constexpr int kTileZ = (\d+);", source("proj3d_dev.hpp")).group(1)
    return host(code) + "constexpr int ZS = " + zs + r""";
struct Dim { unsigned x, y; };
struct BPArgs { unsigned nx, ny, nz, nu, nv; };
// one block of the launch at one angle; -1: not staged
extern "C" long check3d(unsigned nx, unsigned ny, unsigned nz, unsigned nu, unsigned nv, const float *coef,
                        unsigned bx, unsigned by, unsigned bz, int plant) {
    constexpr int KIND = 0;
    const BPArgs A{nx, ny, nz, nu, nv};
    const Dim blockIdx{by * ((nx + 15) / 16) + bx, bz};
    BP3DAngle c;
    std::copy(coef, coef + 12, &c.nu[0]);
    outside = 0;
    lds_base = 1u << 28;
    for (int wave = 0; wave < 4; ++wave)
        for (int lane = 0; lane < 64; ++lane) {
            """ + host(place).replace("const float cz0", "float cz0") + r"""
            (void)active; (void)plane;
            const BPFoot f = bp_footprint<KIND>(c, cx0, cx1, cy0, cy1, cz0, plant ? cz0 : cz1, hiu, hiv,
                                                (int)pitch, (int)prow);
            if (f.w == 0) return -1;
            """ + host(ray) + r"""
            // f.h rows of f.w staged texels, kTilePitch apart; a column outside its row can lie in
            // another one: checked apart below
            const unsigned at = lds_base + (unsigned)f.at;
            lds_end = lds_base + 4u * ((f.h - 1) * kTilePitch + f.w);
            float acc[ZS] = {};
            f.inner ? bp_tile_angle<KIND, ZS, false>(c.nv[2], un, vn, fr, 1.f, hiu, hiv, at, acc)
                    : bp_tile_angle<KIND, ZS, true>(c.nv[2], un, vn, fr, 1.f, hiu, hiv, at, acc);
            const float pu = clamp_pad(un * fr, hiu);
            if ((int)pu < f.u0 || (int)pu + 1 > f.u0 + f.w - 1) ++outside;
        }
    return outside;
}
"""


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    cxx = shutil.which("g++") or shutil.which("clang++")
    if cxx is None:
        pytest.skip("no host compiler")
    d = tmp_path_factory.mktemp("footprints")
    out = {}
    for name, text in (("2d", harness_2d()), ("3d", harness_3d())):
        cpp, so = d / (name + ".cpp"), d / (name + ".so")
        cpp.write_text(PRELUDE + text)
        r = subprocess.run([cxx, "-O2", "-std=c++17", "-mfma", "-ffp-contract=off", "-shared", "-fPIC", str(cpp),
                            "-o", str(so)], capture_output=True, text=True, timeout=120)
        assert r.returncode == 0, r.stderr
        out[name] = ctypes.CDLL(str(so))
        getattr(out[name], "check" + name).restype = ctypes.c_long
    return out


def bp3d_coeffs(vec, vs):
    """The kernel's float32 BP3DAngle (csrc/geometry.cpp cone_bp_coeffs):
    DevConeParams with the texel-centre offset and the padding folded in."""
    nu, nv, dn = O3.cone_bp_params(vec, "default", vs)
    return np.array([[nu[k] + 1.5 * dn[k] for k in range(4)], [nv[k] + 1.5 * dn[k] for k in range(4)], dn],
                    dtype=f32)


def check3d(lib, shape, na, nu, nv, sod, odd, angle_step=1, plant=False):
    nz, ny, nx = shape
    ang = np.linspace(0, 2 * np.pi, na, endpoint=False)
    vecs, vs = OG.normalise_3d(OG.gen_cone_projections(ang, nu, nv, sod, odd, 1.0, 1.0), "cone",
                               OG.vol_geom_3d(ny, nx, nz))
    bad = staged = 0
    pick = lambda n: sorted({0, n // 3, n // 2, n - 1})
    for a in range(0, na, angle_step):
        c = bp3d_coeffs(vecs[a], vs)
        p = c.ctypes.data_as(ctypes.c_void_p)
        for bx in pick((nx + 15) // 16):
            for by in pick((ny + 15) // 16):
                for bz in pick((nz + 15) // 16):
                    r = lib["3d"].check3d(nx, ny, nz, nu, nv, p, bx, by, bz, int(plant))
                    staged += r >= 0
                    bad += max(r, 0)
    assert staged > 0
    return bad


def test_bp3d_taps_inside_staged_footprint_512(lib):
    """The benchmarked cone geometry (512^3, 768^2, SOD 1000, ODD 500),
    corner / edge / centre blocks at every 6th of the 720 angles."""
    assert check3d(lib, (512, 512, 512), 720, 768, 768, 1000.0, 500.0, angle_step=6) == 0


def test_bp3d_taps_inside_staged_footprint_near_source(lib):
    assert check3d(lib, (48, 48, 48), 24, 96, 96, 40.0, 400.0) == 0


def test_bp3d_taps_inside_staged_footprint_ragged(lib):
    """Blocks cut by the volume's faces, a source near them."""
    assert check3d(lib, (19, 47, 33), 60, 80, 72, 45.0, 60.0) == 0


def test_bp3d_planted_first_slice_footprint_is_caught(lib):
    """A footprint from the block's first z slice only misses taps."""
    assert check3d(lib, (64, 64, 64), 36, 96, 96, 150.0, 100.0, plant=True) > 0


def bp2d_coeffs(kind, w, h, nd, na, sod, odd):
    """The kernel's BP2DAngle (csrc/geometry.cpp angle2d_params), float32."""
    ang = np.linspace(0.2, 0.2 + 2 * np.pi, na, endpoint=False)
    vg = OG.vol_geom_2d(h, w)
    if kind == "par":
        vecs, _ = OG.normalise_2d(OG.gen_par_projections(ang, nd, 1.1), "parallel", vg)
    else:
        vecs, _ = OG.normalise_2d(OG.gen_fan_projections(ang, nd, sod, odd, 1.3), "fan", vg)
    out = np.zeros((na, 8), f32)
    for a in range(na):
        p = [float(x) for x in vecs[a]]
        if kind == "par":
            rx, ry, dsx, dsy, ux, uy = p
            d = ux * ry - uy * rx
            out[a, :7] = [(dsy * rx - dsx * ry) / d + 1.5, ry / d, -rx / d, 1, 0, 0, 1]
        else:
            sx, sy, dsx, dsy, ux, uy = p
            smdx, smdy = sx - dsx, sy - dsy
            det2 = lambda ax, ay, bx, by: ax * by - ay * bx
            sc = math.sqrt(ux * ux + uy * uy) / det2(ux, uy, smdx, smdy)
            nc, nx, ny = sc * det2(sx, sy, dsx, dsy), sc * smdy, -sc * smdx
            dc, dx, dy = sc * det2(ux, uy, sx, sy), sc * uy, -sc * ux
            out[a, :7] = [nc + 1.5 * dc, nx + 1.5 * dx, ny + 1.5 * dy, dc, dx, dy, 1]
    return out


# pixels of a tile: bp2d_tile_kernel's 16 x 16, 32 x 16, 32 x 32 and the
# batched kernels' 64 columns of 2, 4, 8 rows
FORMS = {"16x16": 0, "32x16": 1, "32x32": 2, "rows2": 3, "rows4": 4, "rows8": 5}


def check2d(lib, kind, form, w, h, nd, na, sod, odd, plant=0):
    c = bp2d_coeffs(kind, w, h, nd, na, sod, odd)
    staged = ctypes.c_long(0)
    bad = lib["2d"].check2d(0 if kind == "par" else 1, FORMS[form], w, h, na, nd,
                            c.ctypes.data_as(ctypes.c_void_p), plant, ctypes.byref(staged))
    assert bad >= 0 and staged.value > 0
    return bad


RAGGED = {"par": ("par", 130, 70, 200, 45, 0, 0), "fan": ("fan", 129, 97, 190, 60, 500.0, 300.0),
          "fan_near": ("fan", 96, 96, 200, 50, 60.0, 400.0),
          "par_cut": ("par", 65, 33, 40, 30, 0, 0), "fan_cut": ("fan", 70, 41, 64, 48, 44.0, 20.0)}


@pytest.mark.parametrize("form", FORMS)
@pytest.mark.parametrize("case", RAGGED)
def test_bp2d_taps_inside_staged_footprint(lib, case, form):
    kind, w, h, nd, na, sod, odd = RAGGED[case]
    assert check2d(lib, kind, form, w, h, nd, na, sod, odd) == 0
    # an angle beside it whose whole tile's interval is too long
    assert check2d(lib, kind, form, w, h, nd, na, sod, odd, plant=3) == 0


def test_bp2d_planted_first_row_footprint_is_caught(lib):
    assert check2d(lib, "fan", "32x32", 128, 96, 190, 60, 500.0, 300.0, plant=1) > 0


def test_bp2d_planted_cut_corners_are_caught(lib):
    """Lanes past the edge of a slice against the footprint of those inside."""
    assert check2d(lib, "par", "32x32", 130, 70, 200, 45, 0, 0, plant=2) > 0


@pytest.mark.parametrize("case", [("par", 1024, 1024, 1536, 8, 0, 0), ("fan", 512, 512, 768, 12, 1024.0, 512.0)],
                         ids=["par1024", "fan512"])
def test_bp2d_taps_inside_staged_footprint_batched_sizes(lib, case):
    """Slices of the batched workload's sizes (fan: source-origin 2N,
    origin-detector N), 8 rows per thread."""
    kind, w, h, nd, na, sod, odd = case
    assert check2d(lib, kind, "rows8", w, h, nd, na, sod, odd) == 0


def fan_wave(src, det0, u, n, w, h):
    """Float32 (a, c) of `ray2d` for n rays along the rows (V): position
    a s + c at slice s, from a source and detector pixels det0 + k u."""
    k = np.arange(n)
    p0, p1 = det0[0] + k * u[0], det0[1] + k * u[1]
    with np.errstate(all="ignore"):
        a = -(src[0] - p0) / (src[1] - p1)
        c = a * (-0.5 * h + 0.5) + p0 + p1 * a + 0.5 * w - 0.5 + 2
    return a.astype(f32), c.astype(f32), src[1] - p1


def fp2d_rule():
    """The staged 2D FP's margin and its limit of |a| n + |c|."""
    src = source("proj2d_dev.hpp")
    margin = re.search(r"plo = cvt_floor\(clamp_pad\(tmin - ([\d.]+)f", src).group(1)
    limit = re.search(r"!\(fmaf\(fabsf\(R\[j\]\.a\), \(float\)nsl, fabsf\(R\[j\]\.c\)\) < (\w+)f\)", src)
    return float(margin), float(limit.group(1)) if limit else np.inf


def outside_interval(a, c, den, h, hi, margin, limit):
    """Samples of a staged wave whose texel is not between those of its first
    and last ray; 0 where the wave is not staged."""
    if not ((den > 0).all() or (den < 0).all() or (den >= 0).all()):
        return 0
    with np.errstate(all="ignore"):
        if limit < np.inf and not (np.abs(a) * f32(h) + np.abs(c) < limit).all():
            return 0
        s = np.arange(h, dtype=f32)[:, None]
        t = (a.astype(np.float64) * s + c).astype(f32)  # one fused multiply-add
    ends = t[:, [0, -1]]
    lo = np.fmin.reduce(ends, axis=1, keepdims=True, initial=f32(np.inf))
    hi_ = np.fmax.reduce(ends, axis=1, keepdims=True, initial=f32(-np.inf))
    clamp = lambda x: np.fmin(np.fmax(x, f32(0.5)), f32(hi))
    plo, phi = np.floor(clamp(lo - f32(margin))), np.floor(clamp(hi_ + f32(margin)))
    q = np.floor(np.where(np.isnan(t), 0, clamp(t)))  # NaN converts to texel 0
    return int(np.count_nonzero((q < plo) | (q > phi)))


@pytest.mark.parametrize("gap", [100.0, 3.0, 1e-1, 1e-3, 1e-4, 1e-5, 0.0])
def test_fp2d_positions_inside_staged_interval(gap):
    """Rays of a fan whose source is `gap` pixels from its detector's line,
    down to on it: the steeper they are, the more their positions round."""
    margin, limit = fp2d_rule()
    bad = 0
    for w, h, v in ((512, 512, 7.5), (1024, 900, -300.5), (97, 2000, 0.25)):
        for du in (1.0, 0.1, 0.013):
            a, c, den = fan_wave((3.3, v), (3.3 - 20 * du, v - gap), (du, 0.0), 64, w, h)
            bad += outside_interval(a, c, den, h, w + 2.5, margin, limit)
            a, c, den = fan_wave((3.3, v), (3.3 - 20 * du, v - gap), (du, -gap / 80), 64, w, h)
            bad += outside_interval(a, c, den, h, w + 2.5, margin, limit)
    assert bad == 0


def test_fp2d_planted_steep_rays_are_caught():
    a, c, den = fan_wave((3.3, 7.5), (-16.7, 7.5 - 1e-5), (1.0, 0.0), 64, 512, 512)
    assert outside_interval(a, c, den, 512, 514.5, fp2d_rule()[0], np.inf) > 0
