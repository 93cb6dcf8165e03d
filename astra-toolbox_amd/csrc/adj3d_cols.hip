// Exact transpose of the 3D forward projection for detectors whose v axis is
// the volume's z axis (the geometries of fp3d_cols.hip).
//
// A ray (u, v) of an angle samples slice s at in-slice position y(u, s) and
// height z(u, v, s) = zm(u, s) + (v - vm) dz(u, s): y does not depend on v, and
// zm and dz are linear in s.  The transpose therefore splits into
//     T(u, s; z) = sum_v y'(u, v) (1 - |z(u, v, s) - z|)+      (y' = y x weight)
//     x[s][J][z] = sum over angles and u of (1 - |y(u, s) - J|)+ T(u, s; z),
// where T is computed once per (angle, u, slice) and added to the two rows J
// around y(u, s).  The general gather (proj3d.hip) evaluates every candidate
// ray of every voxel: about 25 rays and 70 VALU instructions a voxel and
// angle, against 2 / (distance in u) times (2 / dz + 1) candidates here.
//
// A wave owns one slice s, kRows rows J and 64 R consecutive z (a lane each)
// and sums them over all angles in its part of LDS: no atomics, the same
// sums in the same order on every run.  u ascends, so the rows under y(u, s)
// move one at a time and the two live sums are kept in registers until
// their row is left.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>

#include "proj3d_dev.hpp"

namespace amx {

namespace {
constexpr int kRows = 8;  // rows J of a wave
constexpr int kWin = 5;    // blocks of 64 v in a wave's window
}  // namespace

// Per (angle of the chunk, u): y = q0.x s + q0.y (as the FP rounds them; padded
// row coordinate), zm = q0.z s + q0.w, dz = q1.x s + q1.y.
template <int GK>
__global__ __launch_bounds__(256) void adj_rays_kernel(FPArgs A, float4 *__restrict__ q0,
                                                       float2 *__restrict__ q1) {
    const unsigned i = blockIdx.x * 256 + threadIdx.x;
    if (i >= A.lcount * A.nu) return;
    const unsigned li = i / A.nu, u = i - li * A.nu;
    const FP3DAngle &G = A.ang[A.alist[A.lfirst + li]];
    constexpr bool CONE = GK != GEO_PAR3D;
    const double vm = 0.5 * ((double)A.nv - 1.0);
    const double P0 = G.p0[0] + u * G.u[0], P1 = G.p0[1] + u * G.u[1];
    const double P2 = G.p0[2] + u * G.u[2] + vm * G.v[2];
    const double d0 = CONE ? G.s[0] - P0 : G.s[0], d1 = CONE ? G.s[1] - P1 : G.s[1];
    const double d2 = CONE ? G.s[2] - P2 : G.s[2];
    const double base = -0.5 * A.n0 + 0.5 - (CONE ? G.s[0] : P0);
    const double inv0 = 1.0 / d0;
    const double a1 = d1 * inv0, c1 = a1 * base + (CONE ? G.s[1] : P1) + 0.5 * A.n1 - 0.5;
    const double a2 = d2 * inv0, c2 = a2 * base + (CONE ? G.s[2] : P2) + 0.5 * A.n2 - 0.5;
    const double g = CONE ? -G.v[2] * inv0 : 0.0, k = CONE ? g * base : G.v[2];
    q0[i] = make_float4((float)a1, (float)(c1 + kPad), (float)a2, (float)c2);
    q1[i] = make_float2((float)g, (float)k);
}

// y'[angle of the chunk][u][v] = proj[v][angle][u] x the ray's distance weight: a
// (v, u) transpose of 64 x 64 tiles.  grid = (u tiles, v tiles, angles).
template <int GK>
__global__ __launch_bounds__(256) void adj_weigh_kernel(FPArgs A, const float *__restrict__ proj,
                                                        float *__restrict__ yw) {
    __shared__ float tile[64][65];
    const unsigned li = blockIdx.z;
    const int angle = A.alist[A.lfirst + li];
    const FP3DAngle &G = A.ang[angle];
    const unsigned u0 = blockIdx.x * 64, v0 = blockIdx.y * 64;
    const unsigned tx = threadIdx.x & 63, ty = threadIdx.x >> 6;
    float x[16];
#pragma unroll
    for (int k = 0; k < 16; ++k) {
        const unsigned v = v0 + ty + 4 * k, u = u0 + tx;
        x[k] = (v < A.nv && u < A.nu) ? proj[((size_t)v * A.na + angle) * A.nu + u] : 0.f;
    }
    constexpr bool CONE = GK != GEO_PAR3D;
    const double u = u0 + tx;
    const double d0 = CONE ? G.s[0] - (G.p0[0] + u * G.u[0]) : G.s[0];
    const double d1 = CONE ? G.s[1] - (G.p0[1] + u * G.u[1]) : G.s[1];
    const double inv0 = 1.0 / d0, a1 = d1 * inv0;
#pragma unroll
    for (int k = 0; k < 16; ++k) {
        const double v = v0 + ty + 4 * k;
        const double a2 = (CONE ? G.s[2] - (G.p0[2] + u * G.u[2] + v * G.v[2]) : G.s[2]) * inv0;
        tile[ty + 4 * k][tx] = x[k] * (float)(sqrt(a1 * a1 * A.fs1 + a2 * a2 * A.fs2 + 1.0) * A.osc);
    }
    __syncthreads();
    const unsigned v = v0 + tx;
    if (v >= A.nv) return;
#pragma unroll
    for (int k = 0; k < 16; ++k) {
        const unsigned uo = u0 + ty + 4 * k;
        if (uo < A.nu) yw[((size_t)li * A.nu + uo) * A.nv + v] = tile[tx][ty + 4 * k];
    }
}

struct AdjCols {
    const float4 *q0;   // [angle of chunk][u]
    const float2 *q1;
    const float *yw;    // [angle of chunk][u][v]
    const float4 *geo;  // [angle of chunk][3]: u = geo[0].(W, 1) / geo[2].(W, 1)
    unsigned count;     // angles in the chunk
    unsigned nu, nv, n0, n1, n2;
    unsigned s_step, y_step;  // rows of `out` per slice, per J
    float *out;               // [row][z], += the chunk's contribution
};

// grid = (slices / 4, row tiles, z tiles); 4 waves: 4 consecutive slices.
// What bounds it: VALU issue (0.7 instructions per clock and CU) with LDS
// behind it (a read per candidate, 34 %).  8 rows per wave: LDS lets 28 waves
// per CU run.  FP and gradient at 256^3 / 360 x 384^2 (two of these launches)
// take 16.6 ms, 18.4 with 12 rows, 19.3 with 16, 22.9 with one z per lane, and
// 42.4 with the general gather.
template <int R>
__global__ __launch_bounds__(256, 4) void adj_cols_kernel(AdjCols M) {
    __shared__ float acc_all[4][kRows][64 * R];
    __shared__ float win_all[4][64 * kWin];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int s = blockIdx.x * 4 + wave;
    if (s >= (int)M.n0) return;  // no barrier follows
    const int ya = blockIdx.y * kRows, zb = blockIdx.z * 64 * R;
    float(*acc)[64 * R] = acc_all[wave];
    float *win = win_all[wave];
#pragma unroll
    for (int j = 0; j < kRows; ++j)
#pragma unroll
        for (int r = 0; r < R; ++r) acc[j][64 * r + lane] = 0.f;
    const float sf = (float)s, vm = 0.5f * ((float)M.nv - 1.f);
    const float w0 = sf - 0.5f * M.n0 + 0.5f;
    const float wa = (float)(ya - 1) - 0.5f * M.n1 + 0.5f, wb = wa + (float)(kRows + 1);
    float z[R];
#pragma unroll
    for (int r = 0; r < R; ++r) z[r] = (float)(zb + lane + 64 * r);

    for (unsigned a = 0; a < M.count; ++a) {
        // u whose y(u, s) can lie in (ya - 1, ya + kRows): y is monotone in u
        const float4 gu = M.geo[3 * a], gd = M.geo[3 * a + 2];
        const float ua = fmaf(gu.x, w0, fmaf(gu.y, wa, gu.w)) / fmaf(gd.x, w0, fmaf(gd.y, wa, gd.w));
        const float ub = fmaf(gu.x, w0, fmaf(gu.y, wb, gu.w)) / fmaf(gd.x, w0, fmaf(gd.y, wb, gd.w));
        const float um = (float)M.nu - 1.f;
        const int ulo = __builtin_amdgcn_readfirstlane((int)fminf(fmaxf(ceilf(fminf(ua, ub) - 0.05f), 0.f), um + 1.f));
        const int uhi = __builtin_amdgcn_readfirstlane((int)fmaxf(fminf(floorf(fmaxf(ua, ub) + 0.05f), um), -1.f));
        float lo[R], hi[R];  // sums of rows cur and cur + 1
#pragma unroll
        for (int r = 0; r < R; ++r) lo[r] = hi[r] = 0.f;
        int cur = -1000000;
        auto flush = [&](int row, const float (&x)[R]) {
            const int j = row - ya;
            if (j < 0 || j >= kRows) return;
#pragma unroll
            for (int r = 0; r < R; ++r) acc[j][64 * r + lane] += x[r];
        };
        for (int u0 = ulo; u0 <= uhi; u0 += 64) {
            // parameters of u0 + lane
            const unsigned ui = a * M.nu + (unsigned)min(u0 + lane, (int)M.nu - 1);
            const float4 q0 = M.q0[ui];
            const float2 q1 = M.q1[ui];
            const float y = fmaf(q0.x, sf, q0.y);
            const int pJ = (int)floorf(y) - kPad;
            const float pf = frac(y);
            const float pz = fmaf(q0.z, sf, q0.w), pd = fmaf(q1.x, sf, q1.y);
            const float pr = 1.f / pd;
            const int n = min(64, uhi - u0 + 1);

            // column i: its first candidates and its window of y', loads in flight
            float g[kWin], e[R], dz = 0.f;
            int at[R], nb = 0, nk = 0;
            auto rl = [](float x, int i) { return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), i)); };
            auto issue = [&](int i) {
                const float zm = rl(pz, i), rd = rl(pr, i);
                dz = rl(pd, i);
                const float h = fabsf(rd) + 0.01f;  // far beyond fp32 rounding of the candidates
                nk = __builtin_amdgcn_readfirstlane((int)(2.f * h)) + 1;  // candidates of a z
                int vs[R];
#pragma unroll
                for (int r = 0; r < R; ++r) {
                    const float v = ceilf(fmaf(z[r] - zm, rd, vm) - h);
                    vs[r] = (int)v;
                    e[r] = fmaf(v - vm, dz, zm - z[r]);  // z(v) - z
                }
                const int first = __builtin_amdgcn_readlane(vs[0], 0), last = __builtin_amdgcn_readlane(vs[R - 1], 63);
                const int start = min(first, last);
                const int len = max(first, last) + nk - start;
                // columns whose rays all miss these z have nothing to load
                nb = (start >= (int)M.nv || start + len <= 0) ? 0 : min((len + 63) >> 6, kWin);
                if (nb == 0) return;
#pragma unroll
                for (int r = 0; r < R; ++r) at[r] = vs[r] - start;
                // its own resource, so that a v outside [0, nv) reads 0 (kept
                // out of the immediate offset, which would wrap it back)
                const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
                    const_cast<float *>(M.yw + (size_t)(a * M.nu + (unsigned)(u0 + i)) * M.nv), (short)0,
                    (int)(M.nv * 4u), 0x00020000);
#pragma unroll
                for (int b = 0; b < kWin; ++b) {
                    if (b > 0 && nb <= b) break;
                    int off = (start + lane + 64 * b) * 4;
                    asm volatile("" : "+v"(off));
                    g[b] = __int_as_float(__builtin_amdgcn_raw_buffer_load_b32(rs, off, 0, 0));
                }
            };
            issue(0);
            for (int i = 0; i < n; ++i) {
                const int J = __builtin_amdgcn_readlane(pJ, i);
                const float f = rl(pf, i);
                const int ck = nk, cb = nb;
                const float cd = dz;
                float ce[R];
                int ca[R];
#pragma unroll
                for (int r = 0; r < R; ++r) {
                    ce[r] = e[r];
                    ca[r] = at[r];
                }
                if (cb) {
#pragma unroll
                    for (int b = 0; b < kWin; ++b) {
                        if (b > 0 && cb <= b) break;
                        win[64 * b + lane] = g[b];
                    }
                }
                if (i + 1 < n) issue(i + 1);
                if (cb == 0 || J < ya - 1 || J >= ya + kRows) continue;
                if (J != cur) {
                    if (J == cur + 1) {
                        flush(cur, lo);
#pragma unroll
                        for (int r = 0; r < R; ++r) {
                            lo[r] = hi[r];
                            hi[r] = 0.f;
                        }
                    } else if (J == cur - 1) {
                        flush(cur + 1, hi);
#pragma unroll
                        for (int r = 0; r < R; ++r) {
                            hi[r] = lo[r];
                            lo[r] = 0.f;
                        }
                    } else {
                        flush(cur, lo);
                        flush(cur + 1, hi);
#pragma unroll
                        for (int r = 0; r < R; ++r) lo[r] = hi[r] = 0.f;
                    }
                    cur = J;
                }
                float T[R];
#pragma unroll
                for (int r = 0; r < R; ++r) T[r] = 0.f;
                int k = 0;
                for (; k + 1 < ck; k += 2) {
                    float x0[R], x1[R];
#pragma unroll
                    for (int r = 0; r < R; ++r) {
                        x0[r] = win[ca[r] + k];
                        x1[r] = win[ca[r] + k + 1];
                    }
#pragma unroll
                    for (int r = 0; r < R; ++r) {
                        T[r] = fmaf(x0[r], tent(ce[r]), T[r]);
                        ce[r] += cd;
                        T[r] = fmaf(x1[r], tent(ce[r]), T[r]);
                        ce[r] += cd;
                    }
                }
                if (k < ck) {
#pragma unroll
                    for (int r = 0; r < R; ++r) T[r] = fmaf(win[ca[r] + k], tent(ce[r]), T[r]);
                }
#pragma unroll
                for (int r = 0; r < R; ++r) {
                    lo[r] = fmaf(1.f - f, T[r], lo[r]);
                    hi[r] = fmaf(f, T[r], hi[r]);
                }
            }
        }
        flush(cur, lo);
        flush(cur + 1, hi);
    }
#pragma unroll 4
    for (int j = 0; j < kRows; ++j) {
        if (ya + j >= (int)M.n1) break;
        float *o = M.out + ((size_t)s * M.s_step + (size_t)(ya + j) * M.y_step) * M.n2;
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const unsigned zi = zb + lane + 64 * r;
            if (zi < M.n2) o[zi] += acc[j][64 * r + lane];
        }
    }
}

// vol [z][y][x] += cols [y][x][z]; grid = (x tiles, z tiles, ny)
__global__ __launch_bounds__(256) void cols_add(const float *__restrict__ cols, float *__restrict__ vol,
                                                unsigned nx, unsigned ny, unsigned nz) {
    __shared__ float tile[64][65];
    const unsigned x0 = blockIdx.x * 64, z0 = blockIdx.y * 64, y = blockIdx.z;
    const unsigned tx = threadIdx.x & 63, ty = threadIdx.x >> 6;
    float v[16], o[16];
#pragma unroll
    for (int k = 0; k < 16; ++k) {
        const unsigned x = x0 + ty + 4 * k, z = z0 + tx;
        v[k] = (x < nx && z < nz) ? cols[((size_t)y * nx + x) * nz + z] : 0.f;
    }
#pragma unroll
    for (int k = 0; k < 16; ++k) tile[ty + 4 * k][tx] = v[k];
    __syncthreads();
    const unsigned x = x0 + tx;
    if (x >= nx) return;
#pragma unroll
    for (int k = 0; k < 16; ++k) {
        const unsigned z = z0 + ty + 4 * k;
        o[k] = z < nz ? vol[((size_t)z * ny + y) * nx + x] : 0.f;
    }
#pragma unroll
    for (int k = 0; k < 16; ++k) {
        const unsigned z = z0 + ty + 4 * k;
        if (z < nz) vol[((size_t)z * ny + y) * nx + x] = o[k] + tile[tx][ty + 4 * k];
    }
}

// ------------------------------------------------------------ launch -----
namespace {
// z per lane: a wave's window of v has to hold the candidates of its 64 R z
int adj_z_per_lane(const ColsBound &b, unsigned nz) {
    if (!b.ok || !(b.closest > 0.0)) return 0;
    auto fits = [&](int r) {
        return (64 * r - 1) / b.closest + 2.0 / b.closest + 5.0 <= 64.0 * kWin;
    };
    if (nz > 64 && fits(2)) return 2;
    return fits(1) ? 1 : 0;
}
}  // namespace

bool adj3d_cols_ok(const Geom3D &g, int grp) { return adj_z_per_lane(g.cols[grp], g.nz) > 0; }

// out [y][x][z] += the transpose of the angles [A.lfirst, A.lfirst + A.lcount)
// of direction group grp; `geo` as matched_geo_kernel writes it.
void adj3d_cols_launch(const Geom3D &g, int grp, const FPArgs &A, const float *proj, const float4 *geo,
                       float4 *q0, float2 *q1, float *yw, float *out, hipStream_t s) {
    const bool cone = g.kind == ASTRA_AMD_GEOM_CONE;
    const unsigned rb = (A.lcount * A.nu + 255) / 256;
    const dim3 wg((A.nu + 63) / 64, (A.nv + 63) / 64, A.lcount);
    if (cone) {
        adj_rays_kernel<GEO_CONE><<<rb, 256, 0, s>>>(A, q0, q1);
        adj_weigh_kernel<GEO_CONE><<<wg, 256, 0, s>>>(A, proj, yw);
    } else {
        adj_rays_kernel<GEO_PAR3D><<<rb, 256, 0, s>>>(A, q0, q1);
        adj_weigh_kernel<GEO_PAR3D><<<wg, 256, 0, s>>>(A, proj, yw);
    }
    AMX_LAUNCHED();
    AdjCols M{};
    M.q0 = q0;
    M.q1 = q1;
    M.yw = yw;
    M.geo = geo;
    M.count = A.lcount;
    M.nu = A.nu; M.nv = A.nv;
    M.n0 = A.n0; M.n1 = A.n1; M.n2 = A.n2;
    M.s_step = grp == 0 ? 1 : g.nx;
    M.y_step = grp == 0 ? g.nx : 1;
    M.out = out;
    const int r = adj_z_per_lane(g.cols[grp], g.nz);
    const dim3 grid((A.n0 + 3) / 4, (A.n1 + kRows - 1) / kRows, (A.n2 + 64 * r - 1) / (64 * r));
    if (r == 2)
        adj_cols_kernel<2><<<grid, 256, 0, s>>>(M);
    else
        adj_cols_kernel<1><<<grid, 256, 0, s>>>(M);
    AMX_LAUNCHED();
}

void adj3d_cols_add(const Geom3D &g, const float *cols, float *vol, hipStream_t s) {
    const dim3 grid((g.nx + 63) / 64, (g.nz + 63) / 64, g.ny);
    cols_add<<<grid, 256, 0, s>>>(cols, vol, g.nx, g.ny, g.nz);
    AMX_LAUNCHED();
}

}  // namespace amx
