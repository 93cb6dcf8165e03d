// 3D forward projection for detectors whose v axis is the volume's z axis
// (circular and helical cone beams, parallel beams about z): the rays of one
// detector column share their path through the slice planes, and only
// their height z differs.
//
// The gather of proj3d.hip (one 16-byte load per sample) is bound by the
// texture-address path, which serves 4 lanes per clock for every load wider
// than a dword, and issues 16 VALU instructions per sample.  Here a wave
// takes 64 R consecutive v of one column u at one angle, so the in-slice
// coordinate y(s) and its weight are the wave's: per slice the wave loads the
// two z rows around y(s) with coalesced dword loads (served 16 lanes per
// clock), interpolates them across y once per z (not once per ray), leaves
// the interpolated row in LDS and takes every ray's two taps from there.
// Loads, LDS and VALU then each take about 8 to 9 clocks per 64 samples
// and CU, against 16 for the gather.
//
// The copy of the volume is [y + 4][x + 4][z] (z fastest, a zero border of two
// columns around x and y); the x- and the y-group march through the same
// copy.  Rows have no border along z: every row is its own buffer resource,
// and loads outside [0, nz) are out of its range and return 0.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>

#include "proj3d_dev.hpp"

namespace amx {

namespace {
constexpr int kSl = 4;              // slices per chunk
constexpr int kPerBlock = 64 / kSl; // chunks per block of 64 precomputed slices
constexpr int kWaves = 4;           // columns u per workgroup, a wave each
}  // namespace

// vol [z][y][x] -> cols [y + 2][x + 2][z]: a (z, x) transpose of 64 x 64
// tiles per y.  grid = (x tiles, z tiles, ny + 4); border columns are 0.
__global__ __launch_bounds__(256) void cols_copy(const float *__restrict__ vol,
                                                 float *__restrict__ cols, unsigned nx,
                                                 unsigned ny, unsigned nz) {
    __shared__ float tile[64][65];
    const unsigned px = nx + 2 * kPad;
    const int x0 = blockIdx.x * 64, z0 = blockIdx.y * 64;  // padded x, z origin
    const unsigned yp = blockIdx.z;
    const int y = (int)yp - kPad;
    const int tx = threadIdx.x & 63, ty = threadIdx.x >> 6;
    const bool yin = y >= 0 && y < (int)ny;
    const int x = x0 + tx - kPad;
    float v[16];
#pragma unroll
    for (int k = 0; k < 16; ++k) {
        const int z = z0 + ty + 4 * k;
        v[k] = (yin && x >= 0 && x < (int)nx && z < (int)nz) ? vol[((size_t)z * ny + y) * nx + x] : 0.f;
    }
#pragma unroll
    for (int k = 0; k < 16; ++k) tile[ty + 4 * k][tx] = v[k];
    __syncthreads();
    const unsigned z = z0 + tx;
    if (z >= nz) return;
#pragma unroll
    for (int k = 0; k < 16; ++k) {
        const unsigned xp = x0 + ty + 4 * k;
        if (xp < px) cols[((size_t)yp * px + xp) * nz + z] = tile[tx][ty + 4 * k];
    }
}

struct FPCols {
    const float *cols;  // [y + 4][x + 4][z]
    unsigned row_b;     // bytes of a z row
    unsigned s_step;    // rows from slice s to s + 1
    unsigned y_step;    // rows from in-slice index y to y + 1
    unsigned tiles_u;   // workgroups along u
};

__device__ __forceinline__ int floor_i32(float x) {  // exact for |x| < 2^31
    int r;
    asm("v_cvt_flr_i32_f32 %0, %1" : "=v"(r) : "v"(x));
    return r;
}

// One wave: rays (u, v0 + 64 r + lane), r < R, of one angle; a workgroup is
// kWaves consecutive u of one block of 64 R rows v.
// Per chunk of kSl slices the rows [zb, zb + 64 nb) are loaded, nb <= R + 1
// blocks of 64 (the host checks that no chunk needs more); the loads of the
// next chunk are in flight while this one is sampled.  The slice
// parameters (row of the copy, weight across y, z range) are computed for 64
// slices at a time, one per lane, and read back with v_readlane.
// A wave writes and reads its own part of LDS only, in program order.
//
// What bounds it: VALU (7 instructions per sample and 2 per interpolated row)
// and L1 misses (TCP_PENDING_STALL 45 % of the cycles): neighbouring u share
// one of their two rows, so the waves of a workgroup are paced by a barrier
// per chunk, and 4 waves per SIMD are faster than more.  Measured at 512^3 /
// 720 x 768^2: 35 ms per group launch against 42 for the gather; without the
// pacing 39, with 8 waves per workgroup 45, with 8 slices per chunk 37.
template <int GK, int R>
__global__ __launch_bounds__(64 * kWaves, 4) void fp3d_cols_kernel(FPArgs A, FPCols C) {
    constexpr int NB = R + 1;  // blocks of rows: R in flight, one more where a chunk needs it
    __shared__ float buf[kWaves][kSl][64 * NB];
    __shared__ int range[2][kWaves];
    unsigned tile;
    int angle;
    if (!fp_map(A, tile, angle)) return;  // uniform over the workgroup
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int v0 = (int)(tile / C.tiles_u) * 64 * R;
    // waves past the detector repeat its last column and write nothing
    const int u1 = (int)(tile % C.tiles_u) * kWaves + wave;
    const int u = min(u1, (int)A.nu - 1);
    const FP3DAngle &G = A.ang[angle];
    const unsigned rstep_b = C.y_step * C.row_b;
    const float hi1 = (float)A.n1 + 2.5f;
    const unsigned lds = (unsigned)(size_t)(__attribute__((address_space(3))) float *)&buf[wave][0][0];
    const int vlast = min(v0 + 64 * R, (int)A.nv) - 1;  // last ray of the wave

    // ray setup: c = a s + c along both in-slice axes (fp3d_ray_line)
    constexpr bool CONE = GK != GEO_PAR3D;
    const double P0 = G.p0[0] + u * G.u[0], P1 = G.p0[1] + u * G.u[1];
    const double d0 = CONE ? G.s[0] - P0 : G.s[0], d1 = CONE ? G.s[1] - P1 : G.s[1];
    const double B0 = CONE ? G.s[0] : P0, B1 = CONE ? G.s[1] : P1;
    const double base = -0.5 * A.n0 + 0.5 - B0;
    const double inv0 = 1.0 / d0;
    const double a1 = d1 * inv0, c1 = a1 * base + B1 + 0.5 * A.n1 - 0.5;
    const float a1f = (float)a1, c1f = (float)(c1 + kPad);
    float a2f[R], c2f[R], scale[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int v = min(v0 + 64 * r + lane, vlast);
        const double P2 = G.p0[2] + u * G.u[2] + v * G.v[2];
        const double d2 = CONE ? G.s[2] - P2 : G.s[2], B2 = CONE ? G.s[2] : P2;
        const double a2 = d2 * inv0;
        a2f[r] = (float)a2;
        c2f[r] = (float)(a2 * base + B2 + 0.5 * A.n2 - 0.5);
        scale[r] = (float)(sqrt(a1 * a1 * A.fs1 + a2 * a2 * A.fs2 + 1.0) * A.osc);
    }
    int slo = 0, shi = (int)A.n0 - 1;
    clip_range(a1, c1, (double)A.n1, (int)A.n0, slo, shi);
    // the workgroup's waves take the union of their slices together
    if (lane == 0) {
        range[0][wave] = max(slo, 0);
        range[1][wave] = min(shi, (int)A.n0 - 1);
    }
    __syncthreads();
    slo = range[0][0];
    shi = range[1][0];
#pragma unroll
    for (int i = 1; i < kWaves; ++i) {
        slo = min(slo, range[0][i]);
        shi = max(shi, range[1][i]);
    }
    slo = __builtin_amdgcn_readfirstlane(slo);
    shi = __builtin_amdgcn_readfirstlane(shi);
    // the outermost rays bound every ray's height at every slice
    const float aF = __shfl(a2f[0], 0, 64), cF = __shfl(c2f[0], 0, 64);
    const float aL = __shfl(a2f[R - 1], 63, 64), cL = __shfl(c2f[R - 1], 63, 64);

    unsigned prow = 0;
    float pfy = 0.f;
    int plo = 0, phi = 0;
    // parameters of slices s0 + lane.  The last chunk runs up to kSl - 1
    // slices past shi, where y is clamped into the zero border, or into
    // the border behind the last slice
    auto params = [&](int s0) {
        const int s = s0 + lane;
        const float sf = (float)s;
        const float y = clamp_pad(fmaf(a1f, sf, c1f), hi1);
        pfy = frac(y);
        prow = (unsigned)y * C.y_step + (unsigned)(min(s, (int)A.n0 + 1) + kPad) * C.s_step;
        const float zF = fmaf(aF, sf, cF), zL = fmaf(aL, sf, cL);
        // 0.01: far beyond the rounding of the rays in between
        plo = floor_i32(fminf(zF, zL) - 0.01f);
        phi = floor_i32(fmaxf(zF, zL) + 0.01f) + 1;
    };
    float p0[kSl][R], p1[kSl][R], fy[kSl];
    // a descriptor per row: the range check compares the offset with
    // num_records - soffset, so the row must be in the base
    __amdgpu_buffer_rsrc_t r0[kSl], r1[kSl];
    int zb = 0, nb = 0;
    auto lane_off = [&](int b) {
        // a z below 0 is an offset beyond every row: kept out of the
        // instruction's immediate, which would wrap it back
        int off = (zb + lane + 64 * b) * 4;
        asm volatile("" : "+v"(off));
        return off;
    };
    auto ld = [&](__amdgpu_buffer_rsrc_t r, int off) {
        return __int_as_float(__builtin_amdgcn_raw_buffer_load_b32(r, off, 0, 0));
    };
    auto issue = [&](int k) {
        const int q = (k % kPerBlock) * kSl;
        if (q == 0) params(slo + k * kSl);
        const int lo = min(__builtin_amdgcn_readlane(plo, q), __builtin_amdgcn_readlane(plo, q + kSl - 1));
        const int hi = max(__builtin_amdgcn_readlane(phi, q), __builtin_amdgcn_readlane(phi, q + kSl - 1));
        zb = lo;
        // rays wholly above or below the volume read nothing
        nb = (hi < 0 || lo >= (int)A.n2) ? 0 : (hi - lo + 64) >> 6;
        if (nb == 0) return;
#pragma unroll
        for (int i = 0; i < kSl; ++i) {
            const unsigned row = __builtin_amdgcn_readlane(prow, q + i);
            char *p = const_cast<char *>(reinterpret_cast<const char *>(C.cols)) + (size_t)row * C.row_b;
            r0[i] = __builtin_amdgcn_make_buffer_rsrc(p, (short)0, (int)C.row_b, 0x00020000);
            r1[i] = __builtin_amdgcn_make_buffer_rsrc(p + rstep_b, (short)0, (int)C.row_b, 0x00020000);
            fy[i] = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(pfy), q + i));
        }
#pragma unroll
        for (int b = 0; b < R; ++b) {
            if (b > 0 && nb <= b) break;
            const int off = lane_off(b);
#pragma unroll
            for (int i = 0; i < kSl; ++i) {
                p0[i][b] = ld(r0[i], off);
                p1[i][b] = ld(r1[i], off);
            }
        }
    };

    float acc[R][2];
#pragma unroll
    for (int r = 0; r < R; ++r) acc[r][0] = acc[r][1] = 0.f;
    const int chunks = (shi - slo + kSl) / kSl;  // <= 0: the column misses the volume
    if (chunks > 0) issue(0);
    for (int k = 0; k < chunks; ++k) {
        const int zk = zb, nk = nb;
        if (nk) {
#pragma unroll
            for (int b = 0; b < R; ++b) {
                if (b > 0 && nk <= b) break;
#pragma unroll
                for (int i = 0; i < kSl; ++i)
                    buf[wave][i][64 * b + lane] = fmaf(fy[i], p1[i][b] - p0[i][b], p0[i][b]);
            }
            if (nk > R) {
                const int off = lane_off(R);
#pragma unroll
                for (int i = 0; i < kSl; ++i) {
                    const float q0 = ld(r0[i], off), q1 = ld(r1[i], off);
                    buf[wave][i][64 * R + lane] = fmaf(fy[i], q1 - q0, q0);
                }
            }
        }
        // pacing only: the waves' loads of neighbouring rows meet in L1
        __builtin_amdgcn_s_barrier();
        if (k + 1 < chunks) issue(k + 1);
        if (!nk) continue;
        // LDS address of (slice i, z = 0); the taps of a group of samples
        // are all in flight before the first is used
        const float sf = (float)(slo + k * kSl);
        const unsigned at = __builtin_amdgcn_readfirstlane(lds - 4u * (unsigned)zk);
        constexpr int kGroup = R == 3 ? 6 : R == 1 ? 4 : 8;  // samples in flight
#pragma unroll
        for (int g = 0; g < kSl * R; g += kGroup) {
            float t0[kGroup], t1[kGroup], w[kGroup];
#pragma unroll
            for (int e = 0; e < kGroup; ++e) {
                const int i = (g + e) / R, r = (g + e) % R;
                const float z = fmaf(a2f[r], sf + (float)i, c2f[r]);
                const unsigned o = ((unsigned)floor_i32(z) << 2) + (at + i * (64 * NB * 4));
                const __attribute__((address_space(3))) float *q =
                    (const __attribute__((address_space(3))) float *)(size_t)o;
                t0[e] = q[0];
                t1[e] = q[1];
                w[e] = frac(z);
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int e = 0; e < kGroup; ++e) {
                const int i = (g + e) / R, r = (g + e) % R;
                acc[r][i & 1] += fmaf(w[e], t1[e] - t0[e], t0[e]);
            }
        }
    }
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int v = v0 + 64 * r + lane;
        if (u1 < (int)A.nu && v < (int)A.nv) fp3d_store(A, u, v, angle, (acc[r][0] + acc[r][1]) * scale[r]);
    }
}

// ------------------------------------------------------------ launch -----
size_t fp3d_cols_bytes(const Geom3D &g) {
    return (size_t)(g.nx + 2 * kPad) * (g.ny + 2 * kPad) * g.nz * sizeof(float);
}

void fp3d_cols_copy(const Geom3D &g, const float *vol, float *cols, hipStream_t s) {
    dim3 grid((g.nx + 2 * kPad + 63) / 64, (g.nz + 63) / 64, g.ny + 2 * kPad);
    cols_copy<<<grid, 256, 0, s>>>(vol, cols, g.nx, g.ny, g.nz);
    AMX_LAUNCHED();
}

namespace {
// Rows one chunk of group `grp` can need with r rays per lane: the rays'
// spread, their drift over the chunk, and the two taps with the margins of
// params().  Steeper rays' heights, up to 4000 slices times their slope, round
// by more than those margins in fp32.
bool fits(const ColsBound &b, int r) {
    return b.slope <= 10.0 && (64 * r - 1) * b.spread + (kSl - 1) * b.slope + 3.1 <= 64.0 * (r + 1);
}
double waves(const Geom3D &g, int grp, int r) {
    return (double)g.nu * g.dir_count[grp] * ((g.nv + 64 * r - 1) / (64 * r));
}
// Rays per lane of a group whose launch does not fill the chip; 0: it does,
// or columns do not serve it.
int small_rays(const Geom3D &g, int grp) {
    const ColsBound &b = g.cols[grp];
    const int r = !b.ok || !g.dir_count[grp] ? 0 : g.nv > 64 && fits(b, 2) ? 2 : fits(b, 1) ? 1 : 0;
    return r && waves(g, grp, r) < 16384.0 ? r : 0;
}
}  // namespace

// Rays per lane of the column FP for direction group `grp`, 0: the gather.
//
// A column wave holds 64 R rows whatever the detector has, so the waves to
// count are nu x angles x blocks of 64 R rows.  From 16384 of them on the chip is
// full and the cost is the time per 64 rows of a column, relative to the
// gather with its 16-row tiles, times the columns' blocks: measured at 512^3 /
// 768 rows (43 ms per group launch for the gather; 43, 36, 35 with 2, 3, 4 rays
// per lane; one ray per lane repeats the slice's work for each 64 rows) and at
// 256^3 / 384 rows.
//
// Below, a launch is its copies, a chain of n slices per wave and what its
// waves add to that: the time of an FP in us, fitted to 320 shapes (n x n x nz
// with n 32 to 512, 6 to 360 angles, 1 to 128 rows, cone and parallel).  The
// gather's waves are 4 x 16 rays and end at once where none is on the
// detector; its pair copies cost 0.6 us per 10^6 voxels and group more.  The
// groups that do not fill the chip are decided together: one in each form
// pays for the copies of both.  Gather and columns: 64^2 x 6 / 90 x 83 x 8
// 73 and 49, 256^2 x 12 / 90 x 332 x 16 164 and 382, 512^2 x 12 / 24 x 665 x
// 16 208 and 538, x 48 / 24 x 665 x 64 673 and 551, 64^2 x 72 / 90 x 83 x 96
// 120 and 59.  Over 688 shapes, 288 of them not in the fit, the form taken is
// at most 1.09 times slower than the gather (geometric mean 0.74).
int fp3d_cols_rays(const Geom3D &g, int grp) {
    const ColsBound &b = g.cols[grp];
    if (!b.ok) return 0;
    if (const int r0 = small_rays(g, grp)) {
        const double rows = g.nv > 12 ? 4.0 * ((g.nv + 15) / 16) : (g.nv + 3) / 4;
        double cols = 0.0, gather = 0.0;
        for (int k = 0; k < 2; ++k) {
            const int r = small_rays(g, k);
            if (!r) continue;
            const double n = 0.5 * (k == 0 ? g.nx : g.ny);
            const bool level = g.cols[k].slope == 0.0;
            const double chain = level ? 0.34 : 0.32, each = (level ? 65e-6 : 85e-6) * (r == 2 ? 1.2 : 1.0);
            cols += 7.5 + n * (chain + each * waves(g, k, r));
            gather += 26.5 + n * (0.25 + 98e-6 * ((g.nu + 15) / 16) * rows * g.dir_count[k]) +
                      0.6e-6 * g.nx * g.ny * g.nz;
        }
        return cols < 0.96 * gather ? r0 : 0;
    }
    const bool level = b.slope == 0.0;  // rays that do not climb
    const double per64[5] = {1.0, 1.2, 1.0, 0.84, 0.82};
    // Rays that do not climb keep their rows over all slices: the few rows past
    // a window's last full block cost next to nothing, and the gather gains
    // nothing from its smaller tiles (par3d, gather and columns: 400 x 397 x 130 / 300 x
    // 513 x 140 4.5 and 3.3 ms, 256 x 253 x 100 / 120 x 300 x 100 0.80 and
    // 0.58, 300 x 297 x 64 / 200 x 350 x 64 0.94 and 0.92, 300 x 297 x 290 /
    // 200 x 350 x 200 with rows 1.5 apart 2.7 and 3.4).  With one ray per lane
    // that holds up to about 32768 waves: 512^2 x 48 / 90 x 665 x 64 (29925) 1.49
    // and 1.27, 256^2 x 48 / 360 x 332 x 64 (59760) 0.98 and 1.15 ms.
    const double base = per64[0] * ((g.nv + 15) / 16) / 4.0;
    double best = INFINITY;
    int rays = 0;
    for (int r : {1, 2, 3, 4}) {
        if (!fits(b, r)) continue;
        // rows per ray beyond one cost their loads and interpolation
        const double rows = ((64 * r - 1) * b.typical + 3.0) / 64.0;
        const double blocks = (level ? rows : std::ceil(rows)) / r;
        const double cost = (per64[r] + 0.5 * std::max(0.0, blocks - 1.0)) * r * ((g.nv + 64 * r - 1) / (64 * r));
        const double limit = level && (r > 1 || waves(g, grp, r) < 32768.0) ? 1.25 * base : base;
        if (cost < std::min(best, limit)) {
            best = cost;
            rays = r;
        }
    }
    return rays;
}

void fp3d_cols_launch(const Geom3D &g, int grp, int rays, FPArgs A, const float *cols, hipStream_t s) {
    FPCols C{};
    C.cols = cols;
    C.row_b = g.nz * sizeof(float);
    const unsigned px = g.nx + 2 * kPad;
    C.s_step = grp == 0 ? 1 : px;
    C.y_step = grp == 0 ? px : 1;
    const unsigned vb = (g.nv + 64 * rays - 1) / (64 * rays);
    C.tiles_u = (g.nu + kWaves - 1) / kWaves;
    fp_group_launches(A, C.tiles_u * vb, (unsigned)g.dir_count[grp], [&](const FPArgs &a, unsigned groups) {
        const bool cone = g.kind == ASTRA_AMD_GEOM_CONE;
        if (rays == 1)
            cone ? fp3d_cols_kernel<GEO_CONE, 1><<<groups, 64 * kWaves, 0, s>>>(a, C)
                 : fp3d_cols_kernel<GEO_PAR3D, 1><<<groups, 64 * kWaves, 0, s>>>(a, C);
        else if (rays == 2)
            cone ? fp3d_cols_kernel<GEO_CONE, 2><<<groups, 64 * kWaves, 0, s>>>(a, C)
                 : fp3d_cols_kernel<GEO_PAR3D, 2><<<groups, 64 * kWaves, 0, s>>>(a, C);
        else if (rays == 3)
            cone ? fp3d_cols_kernel<GEO_CONE, 3><<<groups, 64 * kWaves, 0, s>>>(a, C)
                 : fp3d_cols_kernel<GEO_PAR3D, 3><<<groups, 64 * kWaves, 0, s>>>(a, C);
        else
            cone ? fp3d_cols_kernel<GEO_CONE, 4><<<groups, 64 * kWaves, 0, s>>>(a, C)
                 : fp3d_cols_kernel<GEO_PAR3D, 4><<<groups, 64 * kWaves, 0, s>>>(a, C);
    }, s);
}

}  // namespace amx
