// Device code shared by the 3D forward projectors (proj3d.hip, fp3d_cols.hip):
// launch arguments, the XCD-aware work map, the FP64 ray setup and the
// output epilogue.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdlib>

#include "devutil.hpp"
#include "forms3d.hpp"
#include "internal.hpp"

namespace amx {

struct FPArgs {
    const float *volp;  // padded slice-major copy of this group
    unsigned n0, n1, n2;
    const FP3DAngle *ang;
    const int *alist;  // angle indices of this direction group
    unsigned nu, nv, na;
    float fs1, fs2, osc;
    float *out;
    int mode;
    const float *rb;  // OUT_RESID: b in the output layout
    const float *rw;  // OUT_RESID: weights in the output layout (may be NULL)
    int padded_out;   // write [a][v+2][u+2] instead of [v][a][u]
    // workgroup map (fp_map): detector tiles, angles per block, the range
    // [lfirst, lfirst + lcount) of alist covered by this launch, and the
    // part [xfirst[x], xfirst[x + 1]) of that range taken by XCD x
    unsigned tiles, ablk, lfirst, lcount;
    unsigned xfirst[9];
    unsigned ss;  // rays per detector pixel and dimension (DetectorSuperSampling)
};

// Workgroup -> (detector tile, angle) map.  Workgroups are handed out
// round-robin over the 8 XCDs (workgroup L runs on XCD L % 8), and each XCD
// has its own L2.  XCD x takes the angles [xfirst[x], xfirst[x + 1]) of the
// launch's range (an eighth of them), cut into equal blocks of at most
// `ablk` angles, in the order (angle block, tile, angle within block); no
// block spans two XCDs.  The workgroups resident on one XCD at a time are
// then a few neighbouring tiles, each over a block of consecutive angles,
// which start together and march through the same slices at the same
// time: rays of neighbouring angles sample nearly the same voxels, so they
// share the XCD's L2 instead of each fetching the volume from HBM.
// Workgroups beyond their XCD's range return at once.  (A single range cut
// into blocks across the XCDs left the last XCD with the partial block and
// the others with 48 of every 45 angles' work: 48.7 vs 42.7 ms per group
// launch at 512^3 / 720 x 768^2.)
__device__ __forceinline__ bool fp_map_L(const FPArgs &A, unsigned L, unsigned &tile, int &angle) {
    const unsigned x = L & 7u, q = L >> 3;
    const unsigned first = A.xfirst[x], count = A.xfirst[x + 1] - first;
    if (count == 0) return false;
    const unsigned nblk = (count + A.ablk - 1) / A.ablk;
    const unsigned bsz = (count + nblk - 1) / nblk;  // angles per block
    const unsigned span = bsz * A.tiles;             // items per full block
    const unsigned blk = q / span;
    const unsigned b0 = blk * bsz;
    if (b0 >= count) return false;
    const unsigned bs = min(bsz, count - b0);
    const unsigned r = q - blk * span;
    if (r >= bs * A.tiles) return false;
    tile = r / bs;
    angle = A.alist[A.lfirst + first + b0 + r % bs];
    return true;
}

__device__ __forceinline__ bool fp_map(const FPArgs &A, unsigned &tile, int &angle) {
    return fp_map_L(A, blockIdx.x, tile, angle);
}

// One thread per ray; a 256-thread workgroup covers a 16 x 16 detector tile
// of one angle, each wave a 16 u x 4 v sub-tile.  Ray setup runs in FP64;
// the slice loop is wave-uniform over the union of the lanes' clipped slice
// ranges, so the slice base address is scalar and every fetch is one
// 16-byte load with a 32-bit vector offset.
// (u, v): detector coordinates of the ray relative to pixel (0, 0)'s centre
// (fractional for sub-rays).
// GK: GEO_PAR3D, GEO_CONE (flat detector) or GEO_CYL (cylindrical detector:
// pixel centre on the cylinder, cuda/3d/cone_cyl.cu:243-258).
enum { GEO_PAR3D = 0, GEO_CONE = 1, GEO_CYL = 2 };

// The ray of detector coordinates (u, v) in the group's slice frame:
// texel coordinate - 0.5 along axes 1, 2 at slice s = a_k s + c_k, and the
// slices [lo, hi] where it can touch the volume.
template <int GK>
__device__ __forceinline__ void fp3d_ray_line(const FP3DAngle &G, unsigned nu, unsigned nv,
                                              unsigned n0, unsigned n1, unsigned n2, double u,
                                              double v, double &a1, double &a2, double &c1,
                                              double &c2, int &lo, int &hi) {
    constexpr bool CONE = GK != GEO_PAR3D;
    double P[3], d[3];
    if (GK == GEO_CYL) {
        const double th = (u - 0.5 * nu + 0.5) * G.dth;
        const double fv = v - 0.5 * nv + 0.5;
        const double ct = cos(th), st = sin(th);
        for (int k = 0; k < 3; ++k) P[k] = G.p0[k] + ct * G.u[k] + st * G.b[k] + fv * G.v[k];
    } else {
        for (int k = 0; k < 3; ++k) P[k] = G.p0[k] + u * G.u[k] + v * G.v[k];
    }
    for (int k = 0; k < 3; ++k) d[k] = CONE ? (G.s[k] - P[k]) : G.s[k];
    const double *B = CONE ? G.s : P;
    a1 = d[1] / d[0];
    a2 = d[2] / d[0];
    // texel coordinate - 0.5 at slice s: a_k (s - n0/2 + 0.5 - B0) + B_k + n_k/2 - 0.5
    const double base = -0.5 * n0 + 0.5 - B[0];
    c1 = a1 * base + B[1] + 0.5 * n1 - 0.5;
    c2 = a2 * base + B[2] + 0.5 * n2 - 0.5;
    lo = 0;
    hi = (int)n0 - 1;
    clip_range(a1, c1, (double)n1, (int)n0, lo, hi);
    clip_range(a2, c2, (double)n2, (int)n0, lo, hi);
}

template <int GK>
__device__ __forceinline__ void fp3d_ray(const FPArgs &A, const FP3DAngle &G, double u, double v,
                                         float &a1f, float &a2f, float &c1f, float &c2f,
                                         float &scale, int &lo, int &hi) {
    double a1, a2, c1, c2;
    fp3d_ray_line<GK>(G, A.nu, A.nv, A.n0, A.n1, A.n2, u, v, a1, a2, c1, c2, lo, hi);
    a1f = (float)a1;
    a2f = (float)a2;
    c1f = (float)(c1 + kPad);  // padded texel coordinates
    c2f = (float)(c2 + kPad);
    scale = (float)(sqrt(a1 * a1 * A.fs1 + a2 * a2 * A.fs2 + 1.0) * A.osc);
}

// Write the value of ray (u, v) at `angle` in the launch's mode.
__device__ __forceinline__ void fp3d_store(const FPArgs &A, int u, int v, int angle, float val) {
    size_t idx = ((size_t)v * A.na + angle) * A.nu + u;
    size_t oidx = A.padded_out
                      ? ((size_t)angle * (A.nv + 2 * kPad) + (v + kPad)) * (A.nu + 2 * kPad) + u + kPad
                      : idx;
    if (A.mode == OUT_ADD) {
        A.out[oidx] += val;
    } else if (A.mode == OUT_SET) {
        A.out[oidx] = val;
    } else if (A.mode == OUT_RESID) {  // (b + val) * w
        float r = A.rb[idx] + val;
        if (A.rw) r *= A.rw[oidx];
        A.out[oidx] = r;
    } else if (A.mode == OUT_RATIO) {
        A.out[oidx] = em_ratio(A.rb[idx], val);
    } else {  // OUT_ADDMUL: (out + val) * w
        float r = A.out[oidx] + val;
        if (A.rw) r *= A.rw[oidx];
        A.out[oidx] = r;
    }
}

// ------------------------------------------------------------- BP --------
struct BPArgs {
    const float *pp;  // padded angle-major projections
    unsigned nu, nv, na;
    const BP3DAngle *ang;
    const float *aw;  // par3d per-angle weights
    unsigned nx, ny, nz;
    float osc;
    float *vol;
    int mode;
    const float *uw;  // OUT_UPDATE: per-voxel weights (may be NULL)
    float lo, hi;     // OUT_UPDATE: clamp
    const float *pre; // bp3d_kernel: BP of earlier angle chunks, added before the epilogue (or NULL)
};

// Epilogue of a column of ZS voxels: scale, add the earlier chunks, write
// in the launch's mode.
// Every load of the column (earlier chunks, old values, weights) is issued
// before the first store, so the column's read-modify-write costs one
// memory round trip, not one per voxel (the compiler cannot reorder a load
// of vol after a store to vol by itself).  Z0 is the workgroup's, so the
// bounds tests are uniform.
template <int ZS>
__device__ __forceinline__ void bp_column_store(const BPArgs &A, int X, int Y, int Z0,
                                                const float (&acc)[ZS]) {
    const int nzr = min(ZS, (int)A.nz - Z0);
    const size_t plane = (size_t)A.ny * A.nx;
    const size_t base = ((size_t)Z0 * A.ny + Y) * A.nx + X;
    const bool old = A.mode != OUT_SET;
    const bool wts = (A.mode == OUT_EMUPD || A.mode == OUT_UPDATE) && A.uw;
    float pv[ZS], ov[ZS], wv[ZS];
#pragma unroll
    for (int i = 0; i < ZS; ++i) {
        pv[i] = 0.f;
        ov[i] = 0.f;
        wv[i] = 1.f;
        if (i < nzr) {
            const size_t idx = base + i * plane;
            if (A.pre) pv[i] = A.pre[idx];
            if (old) ov[i] = A.vol[idx];
            if (wts) wv[i] = A.uw[idx];
        }
    }
#pragma unroll
    for (int i = 0; i < ZS; ++i) {
        if (i < nzr) {
            float val = acc[i] * A.osc;
            if (A.pre) val += pv[i];
            float out;
            if (A.mode == OUT_ADD) out = ov[i] + val;
            else if (A.mode == OUT_SET) out = val;
            else if (A.mode == OUT_EMUPD) out = ov[i] * (val * wv[i]);
            else out = fminf(fmaxf(fmaf(wv[i], val, ov[i]), A.lo), A.hi);  // OUT_UPDATE
            A.vol[base + i * plane] = out;
        }
    }
}

// ------------------------------------------------------------ launch -----
// Most angles per block of the FP workgroup map (fp_map): an XCD's range
// is cut into equal blocks of at most this many angles.
// ASTRA_AMD_FP3D_ANGLE_BLOCK overrides the default 64 (1..64; read at every
// call).  Measured at 512^3 / 720 x 768^2 (45 angles per XCD and group),
// ms per group launch: 16: 43.5, 23: 42.9, 32 (blocks of 32 and 13): 44.0,
// 45 or 64 (one block): 42.8, 42.7.
inline unsigned fp_angle_block() {
    const char *e = std::getenv("ASTRA_AMD_FP3D_ANGLE_BLOCK");
    const long x = e ? std::strtol(e, nullptr, 10) : 0;
    return (x >= 1 && x <= 64) ? (unsigned)x : 64u;
}

// Split the angles [first, first + count) of a group's list over the 8
// XCDs in equal counts: xfirst[x] is the first angle of XCD x (relative to
// `first`), xfirst[8] = count.  (Splitting by an estimated cost per angle
// -- samples, or cache lines fetched -- measured slower at 512^3 / 720 x
// 768^2: 44.5-45.9 against 43.8-44.3 ms per group launch; the per-angle time
// varies less with the angle than either estimate.)
inline void xcd_split(unsigned count, unsigned (&xfirst)[9]) {
    for (unsigned x = 0; x <= 8; ++x) xfirst[x] = (unsigned)((size_t)count * x / 8);
}

// 16 x 16 detector tiles of one angle
inline unsigned fp_tiles(const FPArgs &A) { return ((A.nu + 15) / 16) * ((A.nv + 15) / 16); }

// Launch `kern` over `count` angles of one direction group, `tiles`
// workgroups each, in as many launches as the 2^32 work-item limit of one
// grid requires.
template <typename K>
void fp_group_launches(FPArgs A, unsigned tiles, unsigned count, K kern, hipStream_t s) {
    A.tiles = tiles;
    A.ablk = fp_angle_block();
    const size_t max_groups = (1u << 24) - 8;  // 256 threads each
    AMX_REQUIRE((size_t)A.tiles * 16 <= max_groups, "fp3d: detector too large for one launch");
    // at most max_groups / tiles - 8 angles per launch: 8 XCD ranges of
    // ceil(count / 8) angles fit
    const unsigned per_launch = (unsigned)(max_groups / A.tiles - 8);
    for (unsigned first = 0; first < count; first += per_launch) {
        A.lfirst = first;
        A.lcount = std::min(count - first, per_launch);
        xcd_split(A.lcount, A.xfirst);
        const size_t groups = (size_t)8 * ((A.lcount + 7) / 8) * A.tiles;
        kern(A, (unsigned)groups);
        AMX_LAUNCHED();
    }
}

// Flat parallel BP (bp3d_flat.hip)
void bp3d_flat_launch(const Geom3D &g, const BPArgs &A, const BP2DAngle *ang, hipStream_t s);
// Column FP (fp3d_cols.hip)
size_t fp3d_cols_bytes(const Geom3D &g);
void fp3d_cols_copy(const Geom3D &g, const float *vol, float *cols, hipStream_t s);
void fp3d_cols_launch(const Geom3D &g, int grp, int rays, FPArgs A, const float *cols, hipStream_t s);

// Its transpose (adj3d_cols.hip)
void adj3d_cols_launch(const Geom3D &g, int grp, const FPArgs &A, const float *proj, const float4 *geo,
                       float4 *q0, float2 *q1, float *yw, float *out, hipStream_t s);
void adj3d_cols_add(const Geom3D &g, const float *cols, float *vol, hipStream_t s);

// BP with staged detector footprints (bp3d_tile.hip): from the padded single
// layout, angles [0, A.na), U and the denominator constant along z; `kind` as
// bp3d_kernel's, kTileZ voxels of a column per thread.
constexpr int kTileZ = 16;
void bp3d_tile_launch(int kind, const BPArgs &A, hipStream_t s);

}  // namespace amx
