// BP of a parallel beam with horizontal rays and a vertical detector.
//
// Every tap of the 3D BP then has the same row coordinate at all angles and
// in the whole slice z, so the interpolation between detector rows commutes
// with the sum over the angles: each detector row is back projected once as
// a 2D sinogram (bp2d_tile: two taps an update instead of four, from LDS),
// and a slice is interpolated between the two row images it lies between.
// Bound by the VALU of the 2D BP.  BP of 400 x 397 x 130 / 300 x 513 x 140: 2.5
// ms in staged 3D tiles, 1.26 here (4 waves of 32 x 32 pixels).
#include "proj2d_dev.hpp"
#include "proj3d_dev.hpp"

namespace amx {

namespace {

constexpr int kT = 4, kNW = 4;  // pixels per lane and axis, waves

// part[r][y][x] = 2D BP of detector row v0 + r
__global__ __launch_bounds__(64 * kNW, 4) void flat_rows(BPArgs A, const BP2DAngle *__restrict__ ang, unsigned v0,
                                                         float *__restrict__ part) {
    __shared__ float buf[kNW][kBp2TileBuf<kT, kT>];
    const unsigned pitch = A.nu + 2 * kPad;
    float *out = part + (size_t)blockIdx.z * A.nx * A.ny;
    bp2d_tile<0, kT, kT, kNW>(blockIdx.x * 8 * kT, blockIdx.y * 8 * kT, A.nx, A.ny, A.na, A.nu,
                              (size_t)(A.nv + 2 * kPad) * pitch, A.pp + (size_t)(v0 + blockIdx.z + kPad) * pitch, ang,
                              buf, [&](int X, int Y, float sum) { out[(size_t)Y * A.nx + X] = sum; });
}

// slices z0 + blockIdx.y from the rows [v0, v0 + n); rows off the detector are 0
__global__ __launch_bounds__(256) void flat_slices(BPArgs A, const float *__restrict__ part, int v0, int n, float vz,
                                                   float vc, unsigned z0) {
    const size_t plane = (size_t)A.nx * A.ny, i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= plane) return;
    const unsigned z = z0 + blockIdx.y;
    const float t = clamp_pad(fmaf(z - 0.5f * A.nz + 0.5f, vz, vc), (float)A.nv + 2.5f);
    const int r = (int)t - kPad - v0;
    const float lo = r >= 0 && r < n ? part[r * plane + i] : 0.f;
    const float hi = r + 1 >= 0 && r + 1 < n ? part[(r + 1) * plane + i] : 0.f;
    const float val[1] = {lerp(lo, hi, frac(t))};
    store_bp_rows<1>(A.vol, z * plane + i, 0, 1, val, A.osc, A.mode, A.uw, A.lo, A.hi);
}

size_t flat_cap(const Geom3D &g) {
    // row images: at most 256 MB, and no more than the projections' copy
    const size_t copy = (size_t)g.na * (g.nv + 2 * kPad) * (g.nu + 2 * kPad) * sizeof(float);
    return std::min<size_t>(copy, 256u << 20) / ((size_t)g.nx * g.ny * sizeof(float));
}

}  // namespace

// The staged footprints of 32 x 32 pixels fit (as in the 2D BP), kBp2KA angles
// are within 32-bit offsets, at least 16 rows are done at a time, and the
// groups fill the chip.  The work is a row's, not a slice's: 1.33 rows a slice
// (400 x 397 x 130 / 300 x 513 x 180) 2.5 ms in 3D tiles and 1.65 here, 1.25 rows
// (256 x 253 x 120 / 120 x 300 x 150) 0.45 and 0.31, 0.67 rows (300 x 297 x 290 /
// 200 x 350 x 200) 1.92 and 0.81; both would meet at about two.
bool bp3d_flat_ok(const Geom3D &g) {
    const size_t tiles = (size_t)((g.nx + 31) / 32) * ((g.ny + 31) / 32);
    return g.flat && 31.f * g.flat_reach <= kBp2Row - 6 &&
           (size_t)(g.nv + 2 * kPad) * (g.nu + 2 * kPad) < (1u << 27) && flat_cap(g) >= std::min(16u, g.nv) &&
           tiles * g.nv >= 1024 && g.na >= 16 && std::fabs(g.flat_v[0]) <= 1.5f;
}

void bp3d_flat_launch(const Geom3D &g, const BPArgs &A, const BP2DAngle *ang, hipStream_t s) {
    const int rows = (int)std::min<size_t>(flat_cap(g), g.nv);
    const float hi = (float)g.nv + 2.5f;
    // first of the two detector rows of a slice (may be off the detector)
    auto row = [&](unsigned z) {
        const float t = std::fmaf(z - 0.5f * g.nz + 0.5f, g.flat_v[0], g.flat_v[1]);
        return (int)std::min(std::max(t, 0.5f), hi) - kPad;
    };
    Scratch part((size_t)rows * g.nx * g.ny * sizeof(float), s);
    for (unsigned z = 0; z < g.nz;) {
        int lo = 1 << 30, up = -1;  // rows on the detector of the slices [z, e)
        unsigned e = z;
        for (; e < g.nz && e - z < 65535; ++e) {
            const int r = row(e), a = std::max(r, 0), b = std::min(r + 1, (int)g.nv - 1);
            const int l = a <= b ? std::min(lo, a) : lo, u = a <= b ? std::max(up, b) : up;
            if (u - l + 1 > rows) break;
            lo = l;
            up = u;
        }
        const int n = up >= lo ? up - lo + 1 : 0;
        if (n) {
            flat_rows<<<dim3((g.nx + 31) / 32, (g.ny + 31) / 32, n), 64 * kNW, 0, s>>>(A, ang, (unsigned)lo,
                                                                                      part.as<float>());
            AMX_LAUNCHED();
        }
        const dim3 grid((unsigned)(((size_t)g.nx * g.ny + 255) / 256), e - z);
        flat_slices<<<grid, 256, 0, s>>>(A, part.as<float>(), n ? lo : 0, n, g.flat_v[0], g.flat_v[1], z);
        AMX_LAUNCHED();
        z = e;
    }
}

}  // namespace amx
