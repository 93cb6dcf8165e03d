// Device code shared by the single-slice 2D projectors (proj2d.hip) and the
// batched 2D SIRT (batch2d.hip): per-ray forward projection, per-pixel back
// projection, and the output epilogues.
//
// Sampling semantics follow cuda/2d/par_fp.cu:53-200, cuda/2d/fan_fp.cu:55-193,
// cuda/2d/par_bp.cu:52-87 and cuda/2d/fan_bp.cu:57-103.
#pragma once

#include <hip/hip_runtime.h>

#include "devutil.hpp"
#include "internal.hpp"

namespace amx {

struct Ray2D {
    float a, c, scale;
    int lo, hi;
};

// Per-ray orientation.  Parallel: per angle (cuda/2d/par_fp.cu:272).  Fan:
// per ray in float32, adding 0.5 in world units as the reference does
// (cuda/2d/fan_fp.cu:79-83); DetS + det * U is one fused multiply-add.
template <bool FAN>
__device__ __forceinline__ bool ray_vertical(const FP2DAngle &G, int det) {
    if (!FAN) return G.vertical != 0;
    const float sx = G.raw[0], sy = G.raw[1], dsx = G.raw[2], dsy = G.raw[3];
    const float ux = G.raw[4], uy = G.raw[5];
    float tx = fmaf((float)det, ux, dsx);
    tx = tx + 0.5f;
    tx = tx - sx;
    float ty = fmaf((float)det, uy, dsy);
    ty = ty + 0.5f;
    ty = ty - sy;
    return fabsf(ty) > fabsf(tx);
}

// FP64 setup of one (sub-)ray through detector position `fdet` (pixel
// units from the detector corner).  t(s) = a s + c is the padded texel
// coordinate along the slice at slice index s.
template <bool FAN>
__device__ __forceinline__ Ray2D ray2d(const FP2DAngle &G, double fdet, bool vertical,
                                      unsigned w, unsigned h) {
    const double P0 = G.p0[0] + (fdet - 0.5) * G.u[0];
    const double P1 = G.p0[1] + (fdet - 0.5) * G.u[1];
    const double rx = FAN ? G.r[0] - P0 : G.r[0];
    const double ry = FAN ? G.r[1] - P1 : G.r[1];
    Ray2D R;
    R.lo = 0;
    double a, c;
    const double len = sqrt(rx * rx + ry * ry);
    if (vertical) {
        // rows are slices (world y = -(r - h/2 + 0.5)); coordinate along columns
        const double k = rx / ry;
        a = -k;
        c = a * (-0.5 * h + 0.5) + P0 - P1 * k + 0.5 * w - 0.5;
        R.hi = (int)h - 1;
        clip_range(a, c, (double)w, (int)h, R.lo, R.hi);
        R.scale = (float)(len / fabs(ry));
    } else {
        // columns are slices (world x = s - w/2 + 0.5); coordinate along rows
        const double k = ry / rx;
        a = -k;
        c = a * (-0.5 * w + 0.5) + 0.5 * h - 0.5 - P1 + P0 * k;
        R.hi = (int)w - 1;
        clip_range(a, c, (double)h, (int)w, R.lo, R.hi);
        R.scale = (float)(len / fabs(rx));
    }
    R.a = (float)a;
    R.c = (float)(c + kPad);
    return R;
}

// Sum of linear samples along a ray over slices [lo, hi] of a padded
// slice-major copy (slice pitch `pitch` texels, coordinate clamp `hi_t`),
// read through a buffer resource over the copy (texel records: one
// v_add3 of per-lane address per sample).  Samples at even offsets from lo
// go to acc0, odd ones to acc1; four loads are issued before the first of
// them is used (the loop is bound by the loads' latency).  The clamped
// coordinate t >= 0.5 truncates to its floor, and frac(t) = t - floor(t).
__device__ __forceinline__ float march2d(__amdgpu_buffer_rsrc_t rs, unsigned pitch, float hi_t,
                                         const Ray2D &R) {
    float acc0 = 0.f, acc1 = 0.f;
    unsigned row = (unsigned)(R.lo > 0 ? R.lo : 0) * pitch;  // first texel of slice s
    int s = R.lo;
    for (; s + 3 <= R.hi; s += 4) {
        float2 q[4];
        float wt[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const float t = clamp_pad(fmaf(R.a, (float)(s + k), R.c), hi_t);
            q[k] = ld2i(rs, row + k * pitch + (unsigned)t);
            wt[k] = frac(t);
        }
        acc0 += lerp(q[0].x, q[0].y, wt[0]);
        acc1 += lerp(q[1].x, q[1].y, wt[1]);
        acc0 += lerp(q[2].x, q[2].y, wt[2]);
        acc1 += lerp(q[3].x, q[3].y, wt[3]);
        row += 4 * pitch;
    }
    if (s + 1 <= R.hi) {
        const float sf = (float)s;
        float t0 = clamp_pad(fmaf(R.a, sf, R.c), hi_t);
        float t1 = clamp_pad(fmaf(R.a, sf + 1.f, R.c), hi_t);
        float2 q0 = ld2i(rs, row + (unsigned)t0), q1 = ld2i(rs, row + pitch + (unsigned)t1);
        acc0 += lerp(q0.x, q0.y, frac(t0));
        acc1 += lerp(q1.x, q1.y, frac(t1));
        row += 2 * pitch;
        s += 2;
    }
    if (s <= R.hi) {
        float t0 = clamp_pad(fmaf(R.a, (float)s, R.c), hi_t);
        float2 q0 = ld2i(rs, row + (unsigned)t0);
        acc0 += lerp(q0.x, q0.y, frac(t0));
    }
    return acc0 + acc1;
}

// Sums of two rays along the same slice axis of one padded copy, over the
// union of their slice ranges: outside its own range a ray's coordinate is
// clamped into the zero border, so the extra samples add exact zeros, and
// one alternation of accumulators over the union splits each ray's
// samples into the same two sums as march2d (possibly with the two roles
// swapped), so each result equals march2d's.  One 16-byte load from the
// lower of the two left texels serves both rays when their left texels
// are at most two apart (the load starts at most pitch - 4, so it stays
// inside the row); otherwise the other ray takes its own 8-byte load.
__device__ __forceinline__ float2 march2d_pair(__amdgpu_buffer_rsrc_t rs, unsigned pitch,
                                               float hi_t, const Ray2D &A, const Ray2D &B) {
    const bool ea = A.lo > A.hi, eb = B.lo > B.hi;
    if (ea && eb) return make_float2(0.f, 0.f);
    const int lo = ea ? B.lo : (eb ? A.lo : min(A.lo, B.lo));
    const int hi = ea ? B.hi : (eb ? A.hi : max(A.hi, B.hi));
    const float gmax = (float)pitch - 4.f;
    float a0 = 0.f, a1 = 0.f, b0 = 0.f, b1 = 0.f;
    unsigned row = (unsigned)(lo > 0 ? lo : 0) * pitch;
    for (int s = lo; s <= hi; ++s, row += pitch) {
        const float sf = (float)s;
        const float ta = clamp_pad(fmaf(A.a, sf, A.c), hi_t);
        const float tb = clamp_pad(fmaf(B.a, sf, B.c), hi_t);
        const float fa = floorf(ta), fb = floorf(tb);
        const float g = fminf(fminf(fa, fb), gmax);
        const float4 x = ld4i(rs, row + (unsigned)g);
        const float da = fa - g, db = fb - g;
        float2 qa = pick2(x, da), qb = pick2(x, db);
        if (da > 2.5f) qa = ld2i(rs, row + (unsigned)fa);
        if (db > 2.5f) qb = ld2i(rs, row + (unsigned)fb);
        const float va = lerp(qa.x, qa.y, ta - fa), vb = lerp(qb.x, qb.y, tb - fb);
        if ((s - lo) & 1) {
            a1 += va;
            b1 += vb;
        } else {
            a0 += va;
            b0 += vb;
        }
    }
    return make_float2(a0 + a1, b0 + b1);
}

// Forward projection value of detector `det` (before the output scale):
// mean over `rays` sub-rays of (ray sum x ray-length weight).
template <bool FAN>
__device__ __forceinline__ float fp2d_value(const FP2DAngle &G, int det, unsigned rays,
                                            unsigned w, unsigned h, const float *rows,
                                            const float *cols) {
    // resources over the two copies, built from their (wave-uniform)
    // bases before the per-ray choice of axis
    const __amdgpu_buffer_rsrc_t rr = texel_rsrc(rows), rc = texel_rsrc(cols);
    const bool vertical = ray_vertical<FAN>(G, det);
    float sum = 0.f;
    for (unsigned k = 0; k < rays; ++k) {
        const double fdet = det + (0.5 + k) / (double)rays;
        Ray2D R = ray2d<FAN>(G, fdet, vertical, w, h);
        float v = vertical ? march2d(rr, w + 2 * kPad, (float)w + 2.5f, R)
                           : march2d(rc, h + 2 * kPad, (float)h + 2.5f, R);
        sum += v * R.scale;
    }
    return sum / (float)rays;
}

// Values of detectors det and det + 1 (one sub-ray each), the two rays
// marched together when they run along the same slice axis; equal to two
// fp2d_value calls.  det + 1 may be past the detector (its value is unused).
template <bool FAN>
__device__ __forceinline__ float2 fp2d_value_pair(const FP2DAngle &G, int det, unsigned w,
                                                  unsigned h, const float *rows,
                                                  const float *cols) {
    const bool va = ray_vertical<FAN>(G, det), vb = ray_vertical<FAN>(G, det + 1);
    if (va != vb)
        return make_float2(fp2d_value<FAN>(G, det, 1, w, h, rows, cols),
                           fp2d_value<FAN>(G, det + 1, 1, w, h, rows, cols));
    const __amdgpu_buffer_rsrc_t rr = texel_rsrc(rows), rc = texel_rsrc(cols);
    const Ray2D A = ray2d<FAN>(G, det + 0.5, va, w, h);
    const Ray2D B = ray2d<FAN>(G, det + 1.5, va, w, h);
    const float2 s = va ? march2d_pair(rr, w + 2 * kPad, (float)w + 2.5f, A, B)
                        : march2d_pair(rc, h + 2 * kPad, (float)h + 2.5f, A, B);
    // fp2d_value: (0 + sum * scale) / 1
    return make_float2(s.x * A.scale, s.y * B.scale);
}

// out[oidx] per mode (OUT_ADD / OUT_SET / OUT_RESID / OUT_ADDMUL)
__device__ __forceinline__ void store_fp(float *out, size_t oidx, float val, int mode,
                                         const float *rb, size_t idx, const float *rw) {
    if (mode == OUT_ADD) {
        out[oidx] += val;
    } else if (mode == OUT_SET) {
        out[oidx] = val;
    } else if (mode == OUT_RESID) {
        float r = rb[idx] + val;
        if (rw) r *= rw[oidx];
        out[oidx] = r;
    } else if (mode == OUT_RATIO) {
        out[oidx] = em_ratio(rb[idx], val);
    } else {
        float r = out[oidx] + val;
        if (rw) r *= rw[oidx];
        out[oidx] = r;
    }
}

// Back projection of PY consecutive rows (Y0 .. Y0+PY-1) of column X over
// all angles from a padded sinogram [na][nd+4].
// KIND: 0 parallel (per-angle weight), 1 fan (fr), 2 fan FBP (fr^2),
// 3 parallel unweighted, 4 fan unweighted (SART's BP, whose per-angle and
// fr weights cancel against its line weights: cuda/2d/par_bp.cu:139-159,
// cuda/2d/fan_bp.cu:167-199).
// PR: rows taken in pairs, one 16-byte load from the lower of the two left
// texels serving both rows when those are at most two apart (the load
// starts at most pitch - 4, inside the row), else an 8-byte load for the
// far one; the same taps and values as PR = false.
template <int KIND, int PY, bool PR = false>
__device__ __forceinline__ void bp2d_column(int X, int Y0, unsigned w, unsigned h, unsigned na,
                                            unsigned nd, const float *__restrict__ sp,
                                            const BP2DAngle *__restrict__ ang, float *acc) {
    const float fx = X - 0.5f * w + 0.5f;
    const float fy0 = -(Y0 - 0.5f * h + 0.5f);  // world y of row Y0
    const unsigned pitch = nd + 2 * kPad;
    const float hi = (float)nd + 2.5f;
#pragma unroll
    for (int i = 0; i < PY; ++i) acc[i] = 0.f;
    const float *row = sp;
    for (unsigned a = 0; a < na; ++a, row += pitch) {
        const BP2DAngle c = ang[a];
        float num = fmaf(fy0, c.num[2], fmaf(fx, c.num[1], c.num[0]));
        float den = fmaf(fy0, c.den[2], fmaf(fx, c.den[1], c.den[0]));
        // every tap load of the PY rows issued before the first use (the
        // loop is bound by the loads' latency)
        float2 q[PY];
        float wt[PY], wg[PY], fl[PY];
#pragma unroll
        for (int i = 0; i < PY; ++i) {
            float fr = (KIND == 0 || KIND == 3) ? 1.f : __builtin_amdgcn_rcpf(den);
            float t = clamp_pad(num * fr, hi);
            // t >= 0.5: truncation is the floor, frac(t) = t - floor(t)
            if (PR) fl[i] = floorf(t);
            if (!PR) q[i] = ld2b(row, (unsigned)t << 2);
            wt[i] = frac(t);
            wg[i] = (KIND == 0) ? c.w : (KIND == 1 ? fr : (KIND == 2 ? fr * fr : 1.f));
            num -= c.num[2];  // next row: world y decreases by 1
            den -= c.den[2];
        }
        if (PR) {
            static_assert(!PR || PY % 2 == 0, "row pairs");
            const float gmax = (float)pitch - 4.f;
#pragma unroll
            for (int i = 0; i < PY; i += 2) {
                const float g = fminf(fminf(fl[i], fl[i + 1]), gmax);
                const float4 x = ld4u(row, (unsigned)g << 2);
                const float d0 = fl[i] - g, d1 = fl[i + 1] - g;
                q[i] = pick2(x, d0);
                q[i + 1] = pick2(x, d1);
                if (d0 > 2.5f) q[i] = ld2b(row, (unsigned)fl[i] << 2);
                if (d1 > 2.5f) q[i + 1] = ld2b(row, (unsigned)fl[i + 1] << 2);
            }
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < PY; ++i) acc[i] = fmaf(wg[i], lerp(q[i].x, q[i].y, wt[i]), acc[i]);
    }
}

// ---- forward projection with slice rows staged in LDS -------------------
// march2d reads the two taps of a sample with one 8-byte gather, which the
// texture-address path serves at 16 clocks per wave and CU.  Here a wave
// takes 64 neighbouring detectors at NA neighbouring angles and marches them
// through the slices together: for a chunk of kFp2SC slices it copies the
// texels that its rays can sample -- one interval, the same for the chunk's
// slices -- to LDS with coalesced dword loads (4 clocks each, shared by the NA
// angles) and takes the taps from there (one read2_b32).  The loads of the
// next chunk are in flight while this one is sampled; a wave uses its own
// part of LDS only, in program order: no barrier.
// At a slice the sample positions of one angle are monotone in the detector
// (a projective map whose denominator keeps its sign: checked), so those of
// its first and last lane bound them; the intervals of 64 slices are computed
// at a time, one per lane.  A chunk whose interval exceeds a staged row takes
// half the slices and rows of twice the length; one that exceeds those samples
// global memory.  A wave takes one slice axis: rays of the other one belong to
// another wave of the launch (both in one wave doubled the longest wave, and
// with it the launch: 356 -> 300 us in the example below).
// Every ray adds the samples of march2d in the same order (the slices before
// and after its own range add exact zeros), so the values equal
// fp2d_value's.
// Bound by issue (VALU 10 per sample) and by the second round of waves that
// does not fill the GPU, no unit saturated; the 128 registers of 4 waves per
// SIMD do not hold the chunk in flight of 2 or 3 angles (spilled: parallel 23
// and 47, fan 8 and 15 registers).  FP of 1024^2 / 720 x 1536, fan: 719 us
// with gathers, 280 to 300 here; of 777 x 641 / 501 x 1013, parallel, 128.
constexpr int kFp2SC = 16;      // slices per staged chunk
constexpr int kFp2Row = 128;    // texels per staged slice row; or half the
                                // slices and twice the texels
constexpr int kFp2Buf = kFp2SC * kFp2Row;  // floats per wave

__device__ __forceinline__ int cvt_floor(float x) {  // floor, exact for |x| < 2^31
    int r;
    asm("v_cvt_flr_i32_f32 %0, %1" : "=v"(r) : "v"(x));
    return r;
}
__device__ __forceinline__ float lane_value(float x, int lane) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), lane));
}

// Samples of SC slices from LDS rows of ROW texels.  CLIP: some sample is
// outside the padded row.
template <int NA, int SC, int ROW, bool CLIP>
__device__ __forceinline__ void fp2d_chunk(const Ray2D (&R)[NA], float sf, float hi_t, unsigned at,
                                           float (&acc)[NA][2]) {
    typedef const __attribute__((address_space(3))) float *lptr;
    constexpr int G = 8;  // samples whose taps are in flight
#pragma unroll
    for (int g = 0; g < SC * NA; g += G) {
        float t0[G], t1[G], wt[G];
#pragma unroll
        for (int e = 0; e < G; ++e) {
            const int i = (g + e) / NA, j = (g + e) % NA;
            float t = fmaf(R[j].a, sf + (float)i, R[j].c);
            if (CLIP) t = clamp_pad(t, hi_t);
            const lptr q = (lptr)(size_t)(((unsigned)t << 2) + (at + i * (ROW * 4)));
            t0[e] = q[0];
            t1[e] = q[1];
            wt[e] = frac(t);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int e = 0; e < G; ++e) {
            const int i = (g + e) / NA, j = (g + e) % NA;
            acc[j][i & 1] += lerp(t0[e], t1[e], wt[e]);
        }
    }
}

// Values of detectors d0 + lane at angles a0 .. a0 + NA - 1 (clamped to the last
// ones), `rays` sub-rays each, of the rays that run along the rows (V) or the
// columns: `mine`; buf: kFp2Buf floats of LDS of this wave.
template <bool FAN, int NA>
__device__ __forceinline__ void fp2d_wave(int d0, int a0, unsigned na, unsigned nd, unsigned rays,
                                          unsigned w, unsigned h, const FP2DAngle *__restrict__ fpa,
                                          const float *__restrict__ rows, const float *__restrict__ cols,
                                          bool V, float (&val)[NA], bool (&mine)[NA], float *buf) {
    const int lane = threadIdx.x & 63;
    const int det = min(d0 + lane, (int)nd - 1);
    const unsigned lds = (unsigned)(size_t)(__attribute__((address_space(3))) float *)buf;
#pragma unroll
    for (int j = 0; j < NA; ++j) val[j] = 0.f;
    bool any = false;
    unsigned long long m[NA];
#pragma unroll
    for (int j = 0; j < NA; ++j) {
        mine[j] = ray_vertical<FAN>(fpa[min(a0 + j, (int)na - 1)], det) == V;
        m[j] = __ballot(mine[j]);
        any = any || m[j];
    }
    if (!any) return;
#pragma unroll 1
    for (unsigned k = 0; k < rays; ++k) {
        const double fdet = det + (0.5 + k) / (double)rays;
        Ray2D R[NA];
        const unsigned pitch = (V ? w : h) + 2 * kPad, nsl = V ? h : w;
        bool simple = (unsigned long long)pitch * nsl < (1ull << 29);  // 32-bit byte offsets
        const float hi_t = (float)(V ? w : h) + 2.5f;
        int glo = 1 << 30, ghi = -1;
#pragma unroll
        for (int j = 0; j < NA; ++j) {
            const FP2DAngle &G = fpa[min(a0 + j, (int)na - 1)];
            R[j] = ray2d<FAN>(G, fdet, V, w, h);
            if (mine[j] && R[j].lo <= R[j].hi) {
                glo = min(glo, R[j].lo);
                ghi = max(ghi, R[j].hi);
            }
            if (FAN && m[j]) {
                const double den = G.r[V] - G.p0[V] - (fdet - 0.5) * G.u[V];
                const unsigned long long neg = __ballot(mine[j] && den < 0.0);
                // farther positions (rays nearly along the slices; NaN where den
                // is 0) round by more than the intervals' margin
                simple = simple && !__ballot(mine[j] && !(fmaf(fabsf(R[j].a), (float)nsl, fabsf(R[j].c)) < 8e4f));
                const int first = __builtin_ctzll(m[j]), last = 63 - __builtin_clzll(m[j]);
                simple = simple && (neg == 0 || neg == m[j]) && __builtin_popcountll(m[j]) == last - first + 1;
                // the other lanes follow the nearest one
                const int near = min(max(lane, first), last);
                R[j].a = __shfl(R[j].a, near, 64);
                R[j].c = __shfl(R[j].c, near, 64);
            }
        }
        if (!simple) {
            const __amdgpu_buffer_rsrc_t rg = texel_rsrc(V ? rows : cols);
#pragma unroll
            for (int j = 0; j < NA; ++j)
                if (mine[j])
                    val[j] += march2d(rg, pitch, hi_t, R[j]) * R[j].scale;
            continue;
        }
        glo = __builtin_amdgcn_readfirstlane(wave_min(glo));
        ghi = __builtin_amdgcn_readfirstlane(wave_max(ghi));
        if (glo > ghi) continue;  // val += 0
        // an angle without rays in this pass follows one that has some
#pragma unroll
        for (int j = 0; j < NA; ++j) {
            if (m[j]) continue;
#pragma unroll
            for (int i = 0; i < NA; ++i)
                if (m[i]) {
                    R[j].a = R[i].a;
                    R[j].c = R[i].c;
                }
        }
        const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
            const_cast<float *>(first_lane_ptr(V ? rows : cols)), (short)0, (int)(nsl * pitch * 4u), 0x00020000);

        int plo = 0, phi = 0, pclip = 0, pbase = 0;
        auto params = [&](int s0) {
            pbase = s0;
            const float sf = (float)(s0 + lane);
            float tmin = INFINITY, tmax = -INFINITY;
#pragma unroll
            for (int j = 0; j < NA; ++j) {
                const float tf = fmaf(lane_value(R[j].a, 0), sf, lane_value(R[j].c, 0));
                const float tl = fmaf(lane_value(R[j].a, 63), sf, lane_value(R[j].c, 63));
                tmin = fminf(tmin, fminf(tf, tl));
                tmax = fmaxf(tmax, fmaxf(tf, tl));
            }
            // 0.01: beyond the rounding of the rays in between (of a and c, 2 x 2^-24 of 8e4)
            pclip = (tmin < 0.51f || tmax > hi_t - 0.01f) ? 1 : 0;
            plo = cvt_floor(clamp_pad(tmin - 0.01f, hi_t));
            phi = cvt_floor(clamp_pad(tmax + 0.01f, hi_t)) + 1;
        };
        // chunk in flight: first texel, texels, slices, clamping
        float g[2 * kFp2SC];
        int zb = 0, len = 0, cs = 0, clip = 0;
        auto issue = [&](int s) {
            if (s + kFp2SC - pbase > 64) params(s);
            const int q = s - pbase;
            // positions are linear in the slice: the ends of the chunk bound it
            const int l0 = __builtin_amdgcn_readlane(plo, q), h0 = __builtin_amdgcn_readlane(phi, q);
            const int c0 = __builtin_amdgcn_readlane(pclip, q);
            cs = kFp2SC;
            zb = min(l0, __builtin_amdgcn_readlane(plo, q + kFp2SC - 1));
            len = max(h0, __builtin_amdgcn_readlane(phi, q + kFp2SC - 1)) - zb + 1;
            clip = c0 | __builtin_amdgcn_readlane(pclip, q + kFp2SC - 1);
            if (len > kFp2Row) {
                cs = kFp2SC / 2;
                zb = min(l0, __builtin_amdgcn_readlane(plo, q + kFp2SC / 2 - 1));
                len = max(h0, __builtin_amdgcn_readlane(phi, q + kFp2SC / 2 - 1)) - zb + 1;
                clip = c0 | __builtin_amdgcn_readlane(pclip, q + kFp2SC / 2 - 1);
                if (len > 2 * kFp2Row) return;
#pragma unroll
                for (int b = 0; b < 4; ++b) {
                    if (b > 1 && len <= 64 * b) break;
                    const int off = (zb + lane + 64 * b) * 4;
#pragma unroll
                    for (int i = 0; i < kFp2SC / 2; ++i)
                        g[b * (kFp2SC / 2) + i] = __int_as_float(__builtin_amdgcn_raw_buffer_load_b32(
                            rs, off, min(s + i, (int)nsl - 1) * (int)(pitch * 4u), 0));
                }
                return;
            }
#pragma unroll
            for (int b = 0; b < 2; ++b) {
                if (b > 0 && len <= 64 * b) break;
                const int off = (zb + lane + 64 * b) * 4;
#pragma unroll
                for (int i = 0; i < kFp2SC; ++i)
                    g[b * kFp2SC + i] = __int_as_float(__builtin_amdgcn_raw_buffer_load_b32(
                        rs, off, min(s + i, (int)nsl - 1) * (int)(pitch * 4u), 0));
            }
        };
        float acc[NA][2];
#pragma unroll
        for (int j = 0; j < NA; ++j) acc[j][0] = acc[j][1] = 0.f;
        params(glo);
        issue(glo);
        for (int s = glo; s <= ghi;) {
            const int cz = zb, cn = len, cc = clip, step = cs;
            const int left = (int)nsl - s;
            if (step == kFp2SC) {
#pragma unroll
                for (int b = 0; b < 2; ++b) {
                    if (b > 0 && cn <= 64 * b) break;
                    if (left >= kFp2SC) {
#pragma unroll
                        for (int i = 0; i < kFp2SC; ++i) buf[i * kFp2Row + 64 * b + lane] = g[b * kFp2SC + i];
                    } else {  // slices past the last one: zeros
#pragma unroll
                        for (int i = 0; i < kFp2SC; ++i)
                            buf[i * kFp2Row + 64 * b + lane] = i < left ? g[b * kFp2SC + i] : 0.f;
                    }
                }
            } else if (cn <= 2 * kFp2Row) {
#pragma unroll
                for (int b = 0; b < 4; ++b) {
                    if (b > 1 && cn <= 64 * b) break;
#pragma unroll
                    for (int i = 0; i < kFp2SC / 2; ++i)
                        buf[i * (2 * kFp2Row) + 64 * b + lane] = i < left ? g[b * (kFp2SC / 2) + i] : 0.f;
                }
            }
            if (s + step <= ghi) issue(s + step);
            const unsigned at = __builtin_amdgcn_readfirstlane(lds - 4u * (unsigned)cz);
            if (step == kFp2SC) {
                if (cc)
                    fp2d_chunk<NA, kFp2SC, kFp2Row, true>(R, (float)s, hi_t, at, acc);
                else
                    fp2d_chunk<NA, kFp2SC, kFp2Row, false>(R, (float)s, hi_t, at, acc);
            } else if (cn <= 2 * kFp2Row) {
                fp2d_chunk<NA, kFp2SC / 2, 2 * kFp2Row, true>(R, (float)s, hi_t, at, acc);
            } else {
                for (int i = 0; i < step && s + i <= ghi; ++i) {
#pragma unroll
                    for (int j = 0; j < NA; ++j) {
                        const float t = clamp_pad(fmaf(R[j].a, (float)(s + i), R[j].c), hi_t);
                        const float2 q = ld2b(V ? rows : cols, ((unsigned)(s + i) * pitch + (unsigned)t) << 2);
                        const float x = lerp(q.x, q.y, frac(t));
                        if (i & 1) acc[j][1] += x;
                        else acc[j][0] += x;
                    }
                }
            }
            s += step;
        }
#pragma unroll
        for (int j = 0; j < NA; ++j)
            if (mine[j]) val[j] += (acc[j][0] + acc[j][1]) * R[j].scale;
    }
#pragma unroll
    for (int j = 0; j < NA; ++j) val[j] /= (float)rays;
}

// ---- back projection with sinogram footprints staged in LDS -------------
// bp2d_column reads the two taps of an update with one 8-byte gather (16
// clocks per wave and CU).  Here a wave covers a tile of LX TX x (64 / LX) TY
// pixels -- lane l its pixels (l % LX + LX i, l / LX + 64 / LX j) -- and
// copies, kBp2KA angles at a time, the texels of each angle's sinogram row
// that the tile's taps can reach to its own part of LDS with coalesced loads;
// the taps are then read from there (one read2_b32).  The loads of the next
// angles are in flight while these are summed, and nothing is shared between
// waves: no barrier.
// The reach is the bounding interval of the tap coordinate at the tile's
// four corner pixels (t is linear-fractional in the pixel position, so its
// extremes over the tile are at the corners, and the clamp is monotone),
// widened by one texel on each side, far beyond the fp32 rounding of the
// taps' incremental coordinates; 64 angles' intervals are computed at a
// time, one per lane.  The corners are the whole tile's, also where the slice's
// edge cuts it: the lanes past the edge store nothing, but read their taps
// from LDS like the others.  If the interval of one of the 64 angles cannot
// be staged (a source just outside the slice), the corners are those of the
// part inside, and every tap is clamped to the staged texels.  An angle whose interval exceeds kBp2Row texels, or
// whose denominator changes sign over the tile, is sampled from global memory.
// Lanes in 8 x 8 squares: the footprint is short for the updates it serves,
// and the taps of neighbouring lanes share LDS words.
// Bound by the VALU (parallel 7, fan 11 instructions per update, the fan's
// reciprocal at a quarter of the rate): BP of 1024^2 / 720 x 1536 359 -> 240
// us (fan, 10.7 clocks per update and CU), of 777 x 641 / 501 x 1013 209 ->
// 82 us (parallel, 5.6).
// With LX = 64 and TX = 1 the taps, weights and the order of the sums are
// those of bp2d_column, so both give the same floats.
constexpr int kBp2KA = 4;     // angles per staged block
constexpr int kBp2Row = 256;  // texels per staged angle row
constexpr int kBp2Buf = kBp2KA * kBp2Row;  // floats per wave

// Interval of an angle packed in an int: first texel | texels << 20 |
// no tap is clamped << 30; texels 0: from global memory.  whole: all of the
// tile's lanes lie within the corners.
template <int KIND>
__device__ __forceinline__ int bp2d_footprint(const BP2DAngle &c, float fx0, float fx1, float fy0,
                                              float fy1, float hi, int pitch, bool whole) {
    float tmin = INFINITY, tmax = -INFINITY, dmin = INFINITY, dmax = -INFINITY;
    for (int j = 0; j < 4; ++j) {
        const float fx = (j & 1) ? fx1 : fx0, fy = (j & 2) ? fy1 : fy0;
        const float num = fmaf(fy, c.num[2], fmaf(fx, c.num[1], c.num[0]));
        const float den = fmaf(fy, c.den[2], fmaf(fx, c.den[1], c.den[0]));
        dmin = fminf(dmin, den);
        dmax = fmaxf(dmax, den);
        const float t = num * ((KIND == 0 || KIND == 3) ? 1.f : 1.f / den);
        tmin = fminf(tmin, t);
        tmax = fmaxf(tmax, t);
    }
    const bool sign_ok = KIND == 0 || KIND == 3 || dmin > 0.f || dmax < 0.f;
    if (!sign_ok || !__builtin_isfinite(tmin) || !__builtin_isfinite(tmax)) return 0;
    const bool inner = whole && tmin >= 1.5f && tmax <= hi - 1.f;
    // taps read texels floor(t) and floor(t) + 1 (t >= 0.5 after the clamp)
    const int t0 = max(0, (int)clamp_pad(tmin, hi) - 1);
    const int t1 = min(pitch - 1, (int)clamp_pad(tmax, hi) + 2);
    const int wd = t1 - t0 + 1;
    return wd <= kBp2Row && t0 < (1 << 20) ? t0 | wd << 20 | (inner ? 1 << 30 : 0) : 0;
}

// One angle's updates of a wave's tile; at: LDS byte address of texel 0 of
// the angle's row (LDS), or the row's byte offset in rs.  CLIP: tap
// coordinates are clamped to [lo, hi].
template <int KIND, int LX, int TX, int TY, bool CLIP, bool LDS>
__device__ __forceinline__ void bp2d_angle(const BP2DAngle &c, float fx, float fy, float lo, float hi, unsigned at,
                                           __amdgpu_buffer_rsrc_t rs, float (&acc)[TY][TX]) {
    typedef const __attribute__((address_space(3))) float *lptr;
    constexpr bool PAR = KIND == 0 || KIND == 3;
    constexpr int N = TX * TY, G = N < 8 ? N : 8;  // updates whose taps are in flight
    constexpr float sx = LX, sy = 64 / LX;
    // steps and weight in vector registers (an operand in a scalar one
    // halves the rate of an addition)
    float nx = sx * c.num[1], ny = sy * c.num[2], dx = sx * c.den[1], dy = sy * c.den[2], cw = c.w;
    asm("" : "+v"(nx), "+v"(ny), "+v"(dx), "+v"(dy), "+v"(cw));
    float nrow = fmaf(fy, c.num[2], fmaf(fx, c.num[1], c.num[0]));
    float drow = fmaf(fy, c.den[2], fmaf(fx, c.den[1], c.den[0]));
    float num = nrow, den = drow;
#pragma unroll
    for (int g = 0; g < N; g += G) {
        float q0[G], q1[G], wt[G], wg[G];
#pragma unroll
        for (int e = 0; e < G; ++e) {
            const float fr = PAR ? 1.f : __builtin_amdgcn_rcpf(den);
            float t = PAR ? num : num * fr;
            if (CLIP) t = __builtin_amdgcn_fmed3f(t, lo, hi);  // (NaN: lo)
            if (LDS) {
                const lptr q = (lptr)(size_t)(((unsigned)t << 2) + at);
                q0[e] = q[0];
                q1[e] = q[1];
            } else {
                const int o = (int)(((unsigned)t << 2) + at);
                q0[e] = __int_as_float(__builtin_amdgcn_raw_buffer_load_b32(rs, o, 0, 0));
                q1[e] = __int_as_float(__builtin_amdgcn_raw_buffer_load_b32(rs, o + 4, 0, 0));
            }
            wt[e] = frac(t);
            wg[e] = KIND == 0 ? cw : KIND == 1 ? fr : KIND == 2 ? fr * fr : 1.f;
            if ((g + e + 1) % TX == 0) {  // next row: world y decreases
                nrow -= ny;
                drow -= dy;
                num = nrow;
                den = drow;
            } else {
                num += nx;
                den += dx;
            }
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int e = 0; e < G; ++e) {
            float &a = acc[(g + e) / TX][(g + e) % TX];
            a = fmaf(wg[e], lerp(q0[e], q1[e], wt[e]), a);
        }
    }
}

// Sums over the angles [alo, ahi) of the pixels of the tile at (X0, Y0), a
// wave's own; buf: kBp2Buf floats of LDS of this wave.  Angle a's padded row
// starts at sp[a * stride]; kBp2KA strides fit in 32-bit byte offsets.
template <int KIND, int LX, int TX, int TY>
__device__ __forceinline__ void bp2d_wave(int X0, int Y0, unsigned w, unsigned h, unsigned alo, unsigned ahi,
                                          unsigned na, unsigned nd, size_t stride,
                                          const float *__restrict__ sp,
                                          const BP2DAngle *__restrict__ ang, float (&acc)[TY][TX],
                                          float *buf) {
    typedef const __attribute__((address_space(4))) float *cptr;  // scalar loads
    const int lane = threadIdx.x & 63;
    const unsigned lds = (unsigned)(size_t)(__attribute__((address_space(3))) float *)buf;
    const float fx = (X0 + lane % LX) - 0.5f * w + 0.5f;
    const float fy = -((Y0 + lane / LX) - 0.5f * h + 0.5f);  // world y
    const unsigned pitch = nd + 2 * kPad;
    const float hi = (float)nd + 2.5f;
    auto interval = [&](const BP2DAngle &c) {
        const float cx0 = X0 - 0.5f * w + 0.5f, cy0 = -(Y0 - 0.5f * h + 0.5f);
        int f = 0, X1 = X0 + LX * TX - 1, Y1 = Y0 + 64 / LX * TY - 1;
#pragma unroll 1
        for (bool all = true;; all = false) {
            f = bp2d_footprint<KIND>(c, cx0, X1 - 0.5f * w + 0.5f, cy0, -(Y1 - 0.5f * h + 0.5f), hi, (int)pitch, all);
            if (!all || __all(f != 0) || (X1 < (int)w && Y1 < (int)h)) return f;
            X1 = min(X1, (int)w - 1);
            Y1 = min(Y1, (int)h - 1);
        }
    };
    const unsigned step = (unsigned)stride * 4u;
    // rows a .. a + kBp2KA - 1, as far as they exist
    auto rows = [&](unsigned a) {
        return __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(first_lane_ptr(sp + a * stride)), (short)0,
                                                 (int)((min((unsigned)kBp2KA, na - a) - 1) * step + pitch * 4u),
                                                 0x00020000);
    };
#pragma unroll
    for (int j = 0; j < TY; ++j)
#pragma unroll
        for (int i = 0; i < TX; ++i) acc[j][i] = 0.f;
    if (alo >= ahi) return;

    int pk = 0;
    int in[kBp2KA];  // intervals of the angles in flight
    float g[kBp2KA][kBp2Row / 64];
    auto issue = [&](unsigned a) {
        const unsigned q = (a - alo) & 63;
        const __amdgpu_buffer_rsrc_t rs = rows(a);
        if (q == 0)
            pk = interval(ang[min(a + lane, na - 1)]);
#pragma unroll
        for (int k = 0; k < kBp2KA; ++k) {
            in[k] = __builtin_amdgcn_readlane(pk, q + k);
            const int off = ((in[k] & 0xfffff) + lane) * 4;
            const int row = (int)(min((unsigned)k, na - 1 - a) * step), wd = (in[k] >> 20) & 0x3ff;
#pragma unroll
            for (int b = 0; b < kBp2Row / 64; ++b) {
                if (b > 0 && wd <= 64 * b) break;
                g[k][b] = __int_as_float(__builtin_amdgcn_raw_buffer_load_b32(rs, off + 256 * b, row, 0));
            }
        }
    };
    issue(alo);
    for (unsigned a = alo; a < ahi; a += kBp2KA) {
        int cur[kBp2KA];
#pragma unroll
        for (int k = 0; k < kBp2KA; ++k) {
            cur[k] = in[k];
            const int wd = (cur[k] >> 20) & 0x3ff;
#pragma unroll
            for (int b = 0; b < kBp2Row / 64; ++b) {
                if (b > 0 && wd <= 64 * b) break;
                buf[k * kBp2Row + 64 * b + lane] = g[k][b];
            }
        }
        if (a + kBp2KA < ahi) issue(a + kBp2KA);
        const __amdgpu_buffer_rsrc_t rs = rows(a);  // unstaged angles
#pragma unroll 1
        for (unsigned k = 0; k < min((unsigned)kBp2KA, ahi - a); ++k) {
            int f = cur[0];
#pragma unroll
            for (int i = 1; i < kBp2KA; ++i) f = k == i ? cur[i] : f;
            const cptr cp = (cptr)(size_t)first_lane_ptr(reinterpret_cast<const float *>(ang + a + k));
            BP2DAngle c;
            for (int i = 0; i < 3; ++i) {
                c.num[i] = cp[i];
                c.den[i] = cp[3 + i];
            }
            c.w = cp[6];
            const unsigned at = __builtin_amdgcn_readfirstlane(lds + k * (kBp2Row * 4) - 4u * (f & 0xfffff));
            if (f >> 30)
                bp2d_angle<KIND, LX, TX, TY, false, true>(c, fx, fy, 0.5f, hi, at, rs, acc);
            else if (f >> 20) {
                // texels [t0, t1]: a pixel within the corners has both its taps at
                // least one texel inside, or is clamped to the row's ends, [0.5, hi]
                const float t0 = (float)(f & 0xfffff), t1 = t0 + (float)((f >> 20) - 1);
                bp2d_angle<KIND, LX, TX, TY, true, true>(c, fx, fy, t0 + 0.5f, t1 - 0.5f, at, rs, acc);
            } else
                bp2d_angle<KIND, LX, TX, TY, true, false>(c, fx, fy, 0.5f, hi, k * step, rs, acc);
        }
    }
}

__device__ __forceinline__ void store_bp(float *vol, size_t idx, float val, int mode,
                                         const float *uw, float lo, float hi) {
    if (mode == OUT_ADD) {
        vol[idx] += val;
    } else if (mode == OUT_SET) {
        vol[idx] = val;
    } else if (mode == OUT_EMUPD) {
        vol[idx] *= val * uw[idx];
    } else {  // OUT_UPDATE: clamp(x + w * val)
        float wv = uw ? uw[idx] : 1.f;
        vol[idx] = fminf(fmaxf(fmaf(wv, val, vol[idx]), lo), hi);
    }
}

// The PY outputs of a thread's pixel column: rows Y0 .. Y0 + nrows - 1
// (nrows <= PY) at vol[idx0 + i * stride], val = acc[i] * scale, stored as
// store_bp does.  Every load (old values, weights) is issued before the
// first store, so the column costs one memory round trip, not one per row
// (the compiler cannot move a load of vol above a store to vol by itself).
template <int PY>
__device__ __forceinline__ void store_bp_rows(float *vol, size_t idx0, size_t stride, int nrows,
                                              const float (&acc)[PY], float scale, int mode,
                                              const float *uw, float lo, float hi) {
    const bool old = mode != OUT_SET;
    const bool wts = (mode == OUT_EMUPD || mode == OUT_UPDATE) && uw;
    float ov[PY], wv[PY];
#pragma unroll
    for (int i = 0; i < PY; ++i) {
        ov[i] = 0.f;
        wv[i] = 1.f;
        if (i < nrows) {
            if (old) ov[i] = vol[idx0 + i * stride];
            if (wts) wv[i] = uw[idx0 + i * stride];
        }
    }
#pragma unroll
    for (int i = 0; i < PY; ++i) {
        if (i < nrows) {
            const float val = acc[i] * scale;
            float out;
            if (mode == OUT_ADD) out = ov[i] + val;
            else if (mode == OUT_SET) out = val;
            else if (mode == OUT_EMUPD) out = ov[i] * (val * wv[i]);
            else out = fminf(fmaxf(fmaf(wv[i], val, ov[i]), lo), hi);  // OUT_UPDATE
            vol[idx0 + i * stride] = out;
        }
    }
}

// One 64 x 64 tile of the padded slice copies of a [h][w] volume: rows copy
// [h][w+4] and columns copy [w][h+4]; tile origin (c0, r0) in padded
// coordinates.  Uses a 64 x 65 LDS tile; 256 threads.
__device__ __forceinline__ void vol2d_copy_tile(const float *__restrict__ vol,
                                                float *__restrict__ rows,
                                                float *__restrict__ cols, unsigned w, unsigned h,
                                                int c0, int r0, float (*tile)[65]) {
    const int pw = w + 2 * kPad, ph = h + 2 * kPad;
    const int tx = threadIdx.x & 63, ty = threadIdx.x >> 6;
    for (int i = ty; i < 64; i += 4) {
        int pr = r0 + i, pc = c0 + tx;
        int r = pr - kPad, c = pc - kPad;
        float v = 0.f;
        if (r >= 0 && r < (int)h && c >= 0 && c < (int)w) v = vol[(size_t)r * w + c];
        tile[i][tx] = v;
        if (r >= 0 && r < (int)h && pc < pw) rows[(size_t)r * pw + pc] = v;
    }
    __syncthreads();
    for (int i = ty; i < 64; i += 4) {
        int pc = c0 + i, pr = r0 + tx;
        int c = pc - kPad;
        if (c >= 0 && c < (int)w && pr < ph) cols[(size_t)c * ph + pr] = tile[tx][i];
    }
}

// 8 TX x 8 TY pixels of a group of NW waves, each wave the sums over its part
// of the angles; store(X, Y, sum): the waves' sums added in their order.
template <int TX, int TY>
constexpr int kBp2TileBuf = kBp2Buf > 64 * TX * TY ? kBp2Buf : 64 * TX * TY;

template <int KIND, int TX, int TY, int NW, class F>
__device__ __forceinline__ void bp2d_tile(int X0, int Y0, unsigned w, unsigned h, unsigned na, unsigned nd,
                                          size_t stride, const float *__restrict__ sp,
                                          const BP2DAngle *__restrict__ ang,
                                          float (&buf)[NW][kBp2TileBuf<TX, TY>], F store) {
    constexpr int N = TX * TY;
    const unsigned wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    float acc[TY][TX];
    bp2d_wave<KIND, 8, TX, TY>(X0, Y0, w, h, (unsigned)((size_t)na * wave / NW),
                               (unsigned)((size_t)na * (wave + 1) / NW), na, nd, stride, sp, ang, acc, buf[wave]);
#pragma unroll
    for (int j = 0; j < TY; ++j)
#pragma unroll
        for (int i = 0; i < TX; ++i) buf[wave][(j * TX + i) * 64 + lane] = acc[j][i];
    __syncthreads();
    for (int p = wave; p < N; p += NW) {
        float sum = buf[0][p * 64 + lane];
#pragma unroll
        for (int k = 1; k < NW; ++k) sum += buf[k][p * 64 + lane];
        const int X = X0 + (int)(lane & 7) + 8 * (p % TX), Y = Y0 + (int)(lane >> 3) + 8 * (p / TX);
        if (X < (int)w && Y < (int)h) store(X, Y, sum);
    }
}

}  // namespace amx
