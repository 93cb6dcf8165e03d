// Voxel-driven 3D back projection with detector footprints staged in LDS.
//
// bp3d_kernel (proj3d.hip) reads every bilinear tap as one 16-byte gather,
// which the texture-address path serves at 16 clocks per wave and CU whatever
// its width.  Here a workgroup (16 x 16 columns of ZS voxels) copies, per
// angle, the rectangle of the projection that its block projects into from
// the padded single layout to LDS -- coalesced dword loads, which that path
// serves in 4 clocks -- and takes the taps from there: two LDS instructions
// of 4 clocks per update.  No pair copy of the projections is made.
//
// Taps, weights and the order of the sums are those of bp3d_kernel<KIND, ZS, true>
// (the pair plane's stored row difference is the difference taken here), so
// both give the same floats.  Like that form it needs U and the denominator
// constant along z; with a reciprocal and a second coordinate per update the
// VALU bounds both forms, and the gather is the faster one (BP of 200 x 187 x
// 150 / 180 x 260 x 230 with a tilted detector: 0.81 ms, staged 0.85 to 0.95).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>

#include "proj3d_dev.hpp"

namespace amx {

namespace {
constexpr int kTileRows = 48;         // tallest footprint (texel rows)
constexpr int kTileCols = 64;         // widest footprint (texel columns)
constexpr int kTilePitch = 72;        // LDS row pitch
constexpr int kTileSlots = kTileRows / 4;
constexpr int kFpGroup = 128;         // angles whose footprints are held at once
}  // namespace

// Texels (u0, v0) .. of the padded plane that the block's taps read: w columns
// and h rows; w = 0: not staged.  u and v are linear-fractional in the voxel
// position, so their extremes over the block are at its corners (the clamp
// to the padded range is monotone), widened by one texel on each side, far
// beyond the fp32 rounding of the taps.  inner: no tap of the block reaches
// the clamp.
struct BPFoot {
    short u0, v0, w, h;
    int at;     // byte offset of texel (0, 0) of the plane from the tile's start
    int inner;
};

__host__ __device__ inline float foot_clamp(float p, float hi) { return fminf(fmaxf(p, 0.5f), hi); }

template <int KIND>
__host__ __device__ BPFoot bp_footprint(const BP3DAngle &c, float x0, float x1, float y0, float y1, float z0,
                               float z1, float hiu, float hiv, int pitch, int prow) {
    float umin = INFINITY, umax = -INFINITY, vmin = INFINITY, vmax = -INFINITY;
    float dmin = INFINITY, dmax = -INFINITY;
    for (int j = 0; j < 8; ++j) {
        const float x = (j & 1) ? x1 : x0, y = (j & 2) ? y1 : y0, z = (j & 4) ? z1 : z0;
        const float un = fmaf(y, c.nu[1], fmaf(x, c.nu[0], c.nu[3]));
        const float dn = fmaf(y, c.dn[1], fmaf(x, c.dn[0], c.dn[3]));
        const float vn = fmaf(z, c.nv[2], fmaf(y, c.nv[1], fmaf(x, c.nv[0], c.nv[3])));
        dmin = fminf(dmin, dn);
        dmax = fmaxf(dmax, dn);
        const float fr = (KIND == 2) ? 1.f : 1.f / dn;
        umin = fminf(umin, un * fr);
        umax = fmaxf(umax, un * fr);
        vmin = fminf(vmin, vn * fr);
        vmax = fmaxf(vmax, vn * fr);
    }
    BPFoot f{0, 0, 0, 0, 0, 0};
    const bool sign_ok = (KIND == 2) || dmin > 0.f || dmax < 0.f;
    const bool finite = __builtin_isfinite(umin) && __builtin_isfinite(umax) &&
                        __builtin_isfinite(vmin) && __builtin_isfinite(vmax);
    if (!sign_ok || !finite) return f;
    f.inner = umin > 1.5f && umax < hiu - 1.f && vmin > 1.5f && vmax < hiv - 1.f;
    umin = foot_clamp(umin, hiu);
    umax = foot_clamp(umax, hiu);
    vmin = foot_clamp(vmin, hiv);
    vmax = foot_clamp(vmax, hiv);
    // taps: texels floor(u), floor(u) + 1 of rows floor(v), floor(v) + 1
    const int u0 = std::max(0, (int)umin - 1), u1 = std::min(pitch - 1, (int)umax + 2);
    const int v0 = std::max(0, (int)vmin - 1), v1 = std::min(prow - 1, (int)vmax + 2);
    const int w = u1 - u0 + 1, h = v1 - v0 + 1;
    if (w < 2 || h < 2 || w > kTileCols || h > kTileRows) return f;
    f.u0 = (short)u0;
    f.v0 = (short)v0;
    f.w = (short)w;
    f.h = (short)h;
    f.at = -4 * (u0 + v0 * kTilePitch);
    return f;
}

// Barrier that orders LDS only: loads from memory stay in flight across it.
__device__ __forceinline__ void lds_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// The coefficients of an angle as scalar loads (constant address space: the
// barriers' fences would make them vector loads, and waiting for those would
// wait for the staged loads in flight too).
__device__ __forceinline__ BP3DAngle scalar_angle(const BP3DAngle *p) {
    typedef const __attribute__((address_space(4))) float *cptr;
    const cptr q = (cptr)(size_t)first_lane_ptr(p);
    BP3DAngle c;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        c.nu[i] = q[i];
        c.nv[i] = q[4 + i];
        c.dn[i] = q[8 + i];
    }
    return c;
}
__device__ __forceinline__ float scalar_float(const float *p) {
    return *(const __attribute__((address_space(4))) float *)(size_t)first_lane_ptr(p);
}

// One angle's updates of a column from the staged tile at LDS byte address
// `at` (of texel (0, 0) of the plane); CLIP: coordinates are clamped to the
// padded range (an angle whose footprint reaches it).
template <int KIND, int ZS, bool CLIP>
__device__ __forceinline__ void bp_tile_angle(float dv, float un, float vn, float fr, float wgt, float hiu,
                                              float hiv, unsigned at, float (&acc)[ZS]) {
    typedef const __attribute__((address_space(3))) float *lptr;
    constexpr int G = 4;  // updates whose taps are in flight
    const float pu = CLIP ? clamp_pad(un * fr, hiu) : un * fr;
    const float wu = frac(pu);
    const unsigned col = at + ((unsigned)pu << 2);
#pragma unroll
    for (int g = 0; g < ZS; g += G) {
        float p00[G], p01[G], p10[G], p11[G], wv[G];
#pragma unroll
        for (int i = 0; i < G; ++i) {
            const float pv = CLIP ? clamp_pad(vn * fr, hiv) : vn * fr;
            wv[i] = frac(pv);
            const lptr q = (lptr)(size_t)(__umul24((unsigned)pv, kTilePitch * 4u) + col);
            p00[i] = q[0];
            p01[i] = q[1];
            p10[i] = q[kTilePitch];
            p11[i] = q[kTilePitch + 1];
            vn += dv;
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < G; ++i) {
            const float4 q = make_float4(p00[i], p10[i] - p00[i], p01[i], p11[i] - p01[i]);
            acc[g + i] = fmaf(wgt, bilerp_pairs(q, wu, wv[i]), acc[g + i]);
        }
    }
}

// The same from memory (an angle whose footprint is not staged).
template <int KIND, int ZS>
__device__ __forceinline__ void bp_global_angle(const float *pl, unsigned pitch, float dv, float un, float vn,
                                                float fr, float wgt, float hiu, float hiv, float (&acc)[ZS]) {
    const float pu = clamp_pad(un * fr, hiu);
#pragma unroll
    for (int i = 0; i < ZS; ++i) {
        const float pv = clamp_pad(vn * fr, hiv);
        const unsigned o = pair_idx(pu, pv, pitch) << 2;
        const float2 a = ld2b(pl, o), b = ld2b(pl, o + pitch * 4u);
        const float4 q = make_float4(a.x, b.x - a.x, a.y, b.y - a.y);
        acc[i] = fmaf(wgt, bilerp_pairs(q, frac(pu), frac(pv)), acc[i]);
        vn += dv;
    }
}

// A.pp: padded single layout [angle][v + 4][u + 4].  A wave is 8 x 8 columns, so
// that its taps of one z lie in few texels.  Two tiles: while angle a is
// sampled from one, angle a + 1 is written to the other from registers, and
// the loads of angle a + 2 are in flight; one barrier per angle.
//
// What bounds it: VALU (13 instructions per update, 0.99 per clock and CU)
// and LDS (two read2_b32, 80 % busy).  Measured at 512^3 / 720 x 768^2: 39 ms
// against 48 for the gather.  Row pitch 72: neighbouring rows start 8 banks
// apart (pitch 65: 54 ms, 64 and 96: 57 and 64, 76 and 80: 44 and 45).  48
// rows leave LDS for 5 workgroups per CU
// (56 rows and 8 updates in flight, 4 workgroups: 44 ms; 40 rows, 6: 45 ms).
template <int KIND, int ZS>
__global__ __launch_bounds__(256, 5) void bp3d_tile_kernel(BPArgs A) {
    __shared__ float tile[2][kTileRows * kTilePitch];
    __shared__ BPFoot foots[kFpGroup];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const unsigned tiles_x = (A.nx + 15) / 16;
    const int X0 = (blockIdx.x % tiles_x) * 16, Y0 = (blockIdx.x / tiles_x) * 16;
    const int X = X0 + (wave & 1) * 8 + (lane & 7), Y = Y0 + (wave >> 1) * 8 + (lane >> 3);
    const int Z0 = blockIdx.y * ZS;
    const bool active = X < (int)A.nx && Y < (int)A.ny;
    const float hx = 0.5f * A.nx - 0.5f, hy = 0.5f * A.ny - 0.5f, hz = 0.5f * A.nz - 0.5f;
    // columns past the volume repeat its last one and write nothing
    const float fx = min(X, (int)A.nx - 1) - 0.5f * A.nx + 0.5f;
    const float fy = min(Y, (int)A.ny - 1) - 0.5f * A.ny + 0.5f;
    const float fz = Z0 - 0.5f * A.nz + 0.5f;
    const float cx0 = X0 - hx, cx1 = min(X0 + 15, (int)A.nx - 1) - hx;
    const float cy0 = Y0 - hy, cy1 = min(Y0 + 15, (int)A.ny - 1) - hy;
    const float cz0 = Z0 - hz, cz1 = (Z0 + ZS - 1) - hz;
    const unsigned pitch = A.nu + 2 * kPad, prow = A.nv + 2 * kPad;
    const size_t plane = (size_t)prow * pitch;  // texels per angle
    const float hiu = (float)A.nu + 2.5f, hiv = (float)A.nv + 2.5f;
    const unsigned lds = (unsigned)(size_t)(__attribute__((address_space(3))) float *)&tile[0][0];
    float acc[ZS];
#pragma unroll
    for (int i = 0; i < ZS; ++i) acc[i] = 0.f;

    float g[kTileSlots];
    // this thread's texels of a footprint: column lane of rows wave + 4 k
    auto fetch = [&](unsigned a, const BPFoot &f) {
        const int h = __builtin_amdgcn_readfirstlane(f.h), v0 = __builtin_amdgcn_readfirstlane(f.v0);
        const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
            const_cast<float *>(first_lane_ptr(A.pp + a * plane)), (short)0, -1, 0x00020000);
        const int off = min((int)f.u0 + lane, (int)pitch - 1) * 4;
        int so = (v0 + wave) * (int)pitch * 4;
#pragma unroll
        for (int k = 0; k < kTileSlots; ++k, so += 16 * (int)pitch)
            if (wave + 4 * k < h) g[k] = __int_as_float(__builtin_amdgcn_raw_buffer_load_b32(rs, off, so, 0));
    };
    auto put = [&](const BPFoot &f, int slot) {
        const int h = __builtin_amdgcn_readfirstlane(f.h);
        float *t = &tile[slot][wave * kTilePitch + lane];
#pragma unroll
        for (int k = 0; k < kTileSlots; ++k)
            if (wave + 4 * k < h) t[4 * k * kTilePitch] = g[k];
    };

    for (unsigned g0 = 0; g0 < A.na; g0 += kFpGroup) {
        const unsigned gn = min((unsigned)kFpGroup, A.na - g0);
        __syncthreads();  // the previous group's footprints and tiles are no longer read
        if (tid < (int)gn)
            foots[tid] = bp_footprint<KIND>(A.ang[g0 + tid], cx0, cx1, cy0, cy1, cz0, cz1, hiu, hiv,
                                                (int)pitch, (int)prow);
        __syncthreads();
        fetch(g0, foots[0]);
        put(foots[0], 0);
        if (gn > 1) fetch(g0 + 1, foots[1]);
        lds_barrier();
        for (unsigned k = 0; k < gn; ++k) {
            if (k + 1 < gn) put(foots[k + 1], (k + 1) & 1);
            if (k + 2 < gn) fetch(g0 + k + 2, foots[k + 2]);
            const BP3DAngle c = scalar_angle(A.ang + g0 + k);
            const BPFoot f = foots[k];
            // nu[2] == dn[2] == 0
            const float un = fmaf(fy, c.nu[1], fmaf(fx, c.nu[0], c.nu[3]));
            const float vn = fmaf(fz, c.nv[2], fmaf(fy, c.nv[1], fmaf(fx, c.nv[0], c.nv[3])));
            const float dn = fmaf(fy, c.dn[1], fmaf(fx, c.dn[0], c.dn[3]));
            const float fr = (KIND == 2) ? 1.f : __builtin_amdgcn_rcpf(dn);
            const float wgt = (KIND == 0) ? fr * fr : (KIND == 1 ? fr : scalar_float(A.aw + g0 + k));
            float dv = c.nv[2];
            asm volatile("" : "+v"(dv));  // a vector register: its additions then issue at twice the rate
            if (__builtin_amdgcn_readfirstlane(f.w)) {
                const unsigned at = __builtin_amdgcn_readfirstlane(f.at) + lds +
                                    (k & 1) * (unsigned)(kTileRows * kTilePitch * 4);
                if (__builtin_amdgcn_readfirstlane(f.inner))
                    bp_tile_angle<KIND, ZS, false>(dv, un, vn, fr, wgt, hiu, hiv, at, acc);
                else
                    bp_tile_angle<KIND, ZS, true>(dv, un, vn, fr, wgt, hiu, hiv, at, acc);
            } else {
                bp_global_angle<KIND, ZS>(first_lane_ptr(A.pp + (g0 + k) * plane), pitch, dv, un, vn, fr, wgt,
                                          hiu, hiv, acc);
            }
            lds_barrier();  // angle k's tile is read, angle k + 1's is written
        }
    }
    if (active) bp_column_store<ZS>(A, X, Y, Z0, acc);
}

// ------------------------------------------------------------ launch -----
// Share of the (block, angle) pairs whose footprint is not staged, from 5 blocks
// along each axis at 16 angles.
float bp3d_tile_miss(int kind, unsigned nx, unsigned ny, unsigned nz, unsigned nu, unsigned nv,
                     const BP3DAngle *ang, unsigned na) {
    auto pick = [](unsigned n, unsigned i, unsigned of) { return n > of ? (2 * i + 1) * n / (2 * of) : i; };
    const unsigned bx = (nx + 15) / 16, by = (ny + 15) / 16, bz = (nz + kTileZ - 1) / kTileZ;
    const float hx = 0.5f * nx - 0.5f, hy = 0.5f * ny - 0.5f, hz = 0.5f * nz - 0.5f;
    const float hiu = (float)nu + 2.5f, hiv = (float)nv + 2.5f;
    const int pitch = nu + 2 * kPad, prow = nv + 2 * kPad;
    unsigned all = 0, miss = 0;
    for (unsigned a = 0; a < std::min(na, 16u); ++a)
        for (unsigned k = 0; k < std::min(bz, 5u); ++k)
            for (unsigned j = 0; j < std::min(by, 5u); ++j)
                for (unsigned i = 0; i < std::min(bx, 5u); ++i) {
                    const BP3DAngle &c = ang[pick(na, a, 16)];
                    const int X0 = pick(bx, i, 5) * 16, Y0 = pick(by, j, 5) * 16, Z0 = pick(bz, k, 5) * kTileZ;
                    const float x0 = X0 - hx, x1 = std::min(X0 + 15, (int)nx - 1) - hx;
                    const float y0 = Y0 - hy, y1 = std::min(Y0 + 15, (int)ny - 1) - hy;
                    const float z0 = Z0 - hz, z1 = (Z0 + kTileZ - 1) - hz;
                    const BPFoot f = kind == 2 ? bp_footprint<2>(c, x0, x1, y0, y1, z0, z1, hiu, hiv, pitch, prow)
                                               : bp_footprint<0>(c, x0, x1, y0, y1, z0, z1, hiu, hiv, pitch, prow);
                    ++all;
                    miss += f.w == 0;
                }
    return (float)miss / all;
}

// An update whose footprint is not staged reads two 8-byte gathers where
// bp3d_kernel reads one of 16 bytes, each at the texture path's 16 clocks: the
// tiles are the faster form up to a share of about an eighth.  Measured at 180
// angles, share, gather and tiles in ms: 256^3 on pixels of 1 / 0.7 / 0.65 /
// 0.6 / 0.55 / 0.5 (magnification 1.5) 0: 1.52 and 1.30, 0: 1.67 and 1.46,
// 0.02: 1.78 and 1.52, 0.19: 1.93 and 1.98, 0.48: 2.36 and 2.76, 0.85: 2.85
// and 4.08; sources at 300 and 260 from its axis 0.14: 1.90 and 1.88, 0.24:
// 2.08 and 2.12; 512^3 on 1536^2 pixels of 0.5 0.80: 21.1 and 33.1.
bool bp3d_tiles_fit(const Geom3D &g) { return g.tile_miss <= 0.125f; }

void bp3d_tile_launch(int kind, const BPArgs &A, hipStream_t s) {
    constexpr int ZS = kTileZ;
    const dim3 grid(((A.nx + 15) / 16) * ((A.ny + 15) / 16), (A.nz + ZS - 1) / ZS);
    if (kind == 0) bp3d_tile_kernel<0, ZS><<<grid, 256, 0, s>>>(A);
    else if (kind == 1) bp3d_tile_kernel<1, ZS><<<grid, 256, 0, s>>>(A);
    else bp3d_tile_kernel<2, ZS><<<grid, 256, 0, s>>>(A);
    AMX_LAUNCHED();
}

}  // namespace amx
