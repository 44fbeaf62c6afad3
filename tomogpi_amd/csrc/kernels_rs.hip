// kernels_rs.hip - ray-driven regular-sampling (RS) projector, its exact
// transpose and its sample counter.
//
// Restates K/Projector/projection_ER_kernel_UM.cuh:25-153 (inscribed-cylinder
// FOV, the reference's device-resident kernel) and, with TOMO_FLAG_RS_FOV_CUBE,
// K/Projector/projection_ER_kernel.cuh:56-312 (circumscribed circle clipped
// to the square of voxel centres, the reference's default host-resident
// path).  One thread per detector cell (m,n) of view p:
//   source S = -FOD(cos,sin,0); cell D = (cos(FDD-FOD) - s sin,
//   sin(FDD-FOD) + s cos, t), s = (m-cu)du, t = (n-cv)dv; unit d = (D-S)/|D-S|
//   entry/exit = circle intersections (entry nearer the source); cube mode
//   clips to [0,N-1]^2; a ray whose entry z is outside [0,Nz) ([0,Nz-1] in
//   cube mode) gives 0; an exit beyond z=Nz-1 or z=0 is moved onto that plane;
//   L_r = floor(|exit-entry|) voxels;  g = delta * sum_{n<L_r} trilinear(f, entry + n d)
// The ray setup is FP64 (the reference parametrises by x, which is singular
// for rays parallel to y; the arc-length form here is well conditioned), the
// samples and the sum are FP32.  The output is overwritten.
#include <atomic>
#include <climits>
#include <type_traits>

#include "proj_copy.hpp"
#include "batch.hpp"
#include "stage_box.hpp"

namespace tomo {
namespace {

constexpr int BX = kProjTileU, BY = kProjTileV;

struct RsRay {
    float ex, ey, ez, dx, dy, dz;
    int lr;  // number of samples (0: ray dropped)
};

__device__ __forceinline__ RsRay rs_setup(const DevGeom& g, int cube, int p, int m, int n) {
    RsRay r{0, 0, 0, 0, 0, 0, 0};
    const double* vw = g.view + (size_t)p * kViewStride;
    const double ca = vw[0], sa = vw[1], dl = (double)g.delta;
    const double s = ((double)m - (double)g.cu) * (double)g.du;
    const double t = ((double)n - (double)g.cv) * (double)g.dv;
    const double rx = ca * g.fdd - s * sa, ry = sa * g.fdd + s * ca, rz = t;
    const double L = sqrt((rx * rx + ry * ry) + rz * rz);
    const double d0 = rx / L, d1 = ry / L, d2 = rz / L;
    const double Sx = -g.fod * ca / dl, Sy = -g.fod * sa / dl;
    const double half = 0.5 * (double)g.nx;
    const double R2 = cube ? 2.0 * (half * half) : half * half;
    const double a = d0 * d0 + d1 * d1;
    if (!(a > 0.0)) return r;
    const double b = Sx * d0 + Sy * d1;
    const double c = (Sx * Sx + Sy * Sy) - R2;
    const double disc = b * b - a * c;
    if (!(disc >= 0.0)) return r;
    const double sq = sqrt(disc);
    double l1 = (-b - sq) / a, l2 = (-b + sq) / a;
    const double cx = g.cx, cy = g.cy, cz = g.cz;
    if (cube) {
        // x then y, exactly as the oracle's loop over the two axes.
        {
            const double lo = -cx, hi = (double)(g.nx - 1) - cx;
            if (d0 != 0.0) {
                const double ta = (lo - Sx) / d0, tb = (hi - Sx) / d0;
                l1 = fmax(l1, fmin(ta, tb));
                l2 = fmin(l2, fmax(ta, tb));
            } else if (!(Sx >= lo && Sx <= hi)) {
                return r;
            }
        }
        {
            const double lo = -cy, hi = (double)(g.ny - 1) - cy;
            if (d1 != 0.0) {
                const double ta = (lo - Sy) / d1, tb = (hi - Sy) / d1;
                l1 = fmax(l1, fmin(ta, tb));
                l2 = fmin(l2, fmax(ta, tb));
            } else if (!(Sy >= lo && Sy <= hi)) {
                return r;
            }
        }
        if (!(l1 <= l2)) return r;
    }
    const double ze = l1 * d2 + cz;
    if (cube) {
        if (!(ze >= 0.0 && ze <= (double)(g.nz - 1))) return r;
    } else {
        if (!(ze >= 0.0 && ze < (double)g.nz)) return r;
    }
    const double zx = l2 * d2 + cz;
    if (zx > (double)(g.nz - 1)) l2 = ((double)(g.nz - 1) - cz) / d2;
    else if (zx < 0.0) l2 = -cz / d2;
    const double len = fabs(l2 - l1);
    if (!(len >= 1.0)) return r;
    r.ex = (float)((Sx + l1 * d0) + cx);
    r.ey = (float)((Sy + l1 * d1) + cy);
    r.ez = (float)(l1 * d2 + cz);
    r.dx = (float)d0;
    r.dy = (float)d1;
    r.dz = (float)d2;
    const double lf = floor(len);
    r.lr = lf > 1.0e9 ? 1000000000 : (int)lf;
    return r;
}

__device__ __forceinline__ int wave_min(int v) {
    for (int off = 32; off > 0; off >>= 1) v = min(v, __shfl_xor(v, off, 64));
    return v;
}
__device__ __forceinline__ int wave_max(int v) {
    for (int off = 32; off > 0; off >>= 1) v = max(v, __shfl_xor(v, off, 64));
    return v;
}

// Reads of the RS copy (proj_copy.hpp): 8-byte elements, z fastest; the element of
// the lower corner (floor x, floor y, floor z) and the next one are 16 bytes.
// FP32 elements are x pairs, so the eight taps are two 16-byte loads, at rows y
// and y + 1; 16-bit ones hold the four voxels of a (x, y) cell: one load.
// BUF: by 32-bit byte offset through a buffer resource; an offset past its end
// reads 0 without touching memory.  Otherwise by 64-bit element index, and a
// sample that is not reads element 0, a border element.
constexpr uint32_t kOutside = 0xfffffff0u;

// The corner's taps interpolated along x: c00 at (y, z), c10 at (y+1, z), c01 at
// (y, z+1), c11 at (y+1, z+1).
struct RsRows {
    float c00, c10, c01, c11;
};

template <typename TV, bool BUF> struct RsReader {
    __amdgpu_buffer_rsrc_t r;
    const uint2* p;
    uint32_t sx, sy;  // elements per x and y step; BUF: bytes
    float syf, mz;    // BUF: sy, and 2^23 + the offset of floors (0, 0) from (-1, z0 - 1) in (y, z)
    size_t base;      // index of the element of floors (0, 0, 0)
    using Off = typename std::conditional<BUF, uint32_t, size_t>::type;
    // Offset of the element of the floors, each in [-1, n - 1], z in [z0 - 1, z0 + nz - 1].  BUF: the
    // (y, z) part as exact FP32 integers below 2^24 (sx < 2^23), whose bits
    // hold them above 2^23, and a 24-bit multiply-add for x: fused
    // multiply-adds issue at twice the rate of conversions.
    __device__ __forceinline__ Off at(float xf, float yf, float zf) const {
        if constexpr (BUF) {
            const uint32_t yz = __float_as_uint(fmaf(yf, syf, fmaf(zf, 8.0f, mz)));
            const uint32_t x1 = __float_as_uint(xf + 8388609.0f);
            return __umul24(x1, sx) + yz - 0x4b000000u;
        } else {
            return (size_t)((int64_t)(int)xf * (int64_t)sx + (int64_t)(int)yf * (int64_t)sy + (int)zf) + base;
        }
    }
    // What a sample that is not reads.  BUF: as a mask, since a select of the
    // offset would let the compiler move its arithmetic into a branch, which
    // splits the unrolled samples and serialises their loads.
    __device__ __forceinline__ Off only(bool in, Off o) const {
        if constexpr (BUF) {
            const uint32_t keep = 0u - (uint32_t)in;
            return (o & keep) | (kOutside & ~keep);
        } else {
            return in ? o : 0;
        }
    }
    struct Taps {
        uint32_t d[sizeof(TV) == 4 ? 8 : 4];
    };
    __device__ __forceinline__ Taps load(Off o) const {
        Taps t;
        if constexpr (BUF) {
            const auto v = __builtin_amdgcn_raw_buffer_load_b128(r, (int)o, 0, 0);
            t.d[0] = v[0]; t.d[1] = v[1]; t.d[2] = v[2]; t.d[3] = v[3];
            if constexpr (sizeof(TV) == 4) {
                const auto w = __builtin_amdgcn_raw_buffer_load_b128(r, (int)o, (int)sy, 0);
                t.d[4] = w[0]; t.d[5] = w[1]; t.d[6] = w[2]; t.d[7] = w[3];
            }
        } else {
            __builtin_memcpy(t.d, p + o, 16);
            if constexpr (sizeof(TV) == 4) __builtin_memcpy(t.d + 4, p + o + sy, 16);
        }
        return t;
    }
};

// One x row of a cell from a word of two FP16 voxels, lo + fx (hi - lo): the
// difference and the blend each one v_fma_mix_f32, which takes the halves as
// they are (exact conversions, one rounding: the FP32 operations' results).
// Converted first, the eight taps cost eight conversions more.
__device__ __forceinline__ float mix_lerp(uint32_t w, float fx) {
    float t, c;
    asm("v_fma_mix_f32 %0, 1.0, %1, -%1 op_sel:[0,1,0] op_sel_hi:[0,1,1]" : "=v"(t) : "v"(w));
    asm("v_fma_mix_f32 %0, %1, %2, %3 op_sel_hi:[0,0,1]" : "=v"(c) : "v"(fx), "v"(t), "v"(w));
    return c;
}

template <typename TV, bool BUF>
__device__ __forceinline__ RsRows rs_rows(const typename RsReader<TV, BUF>::Taps& t, float fx) {
    auto lerp = [&](float a, float b) { return fmaf(fx, b - a, a); };
    if constexpr (sizeof(TV) == 4) {
        auto f = [&](int k) { return __uint_as_float(t.d[k]); };
        return RsRows{lerp(f(0), f(1)), lerp(f(4), f(5)), lerp(f(2), f(3)), lerp(f(6), f(7))};
    } else if constexpr (std::is_same<TV, __half>::value) {
        return RsRows{mix_lerp(t.d[0], fx), mix_lerp(t.d[1], fx), mix_lerp(t.d[2], fx), mix_lerp(t.d[3], fx)};
    } else {
        using U = Unpack16<TV>;
        auto row = [&](uint32_t w) { return lerp(U::lo(w), U::hi(w)); };
        return RsRows{row(t.d[0]), row(t.d[1]), row(t.d[2]), row(t.d[3])};
    }
}

template <typename TV, bool BUF>
__device__ __forceinline__ RsReader<TV, BUF> make_rs_reader(const void* copy, int nx, int ny, ProjPlanes zp) {
    RsReader<TV, BUF> q;
    const RsCopyShape c = rs_copy_shape(nx, ny, zp.nz, sizeof(TV));
    q.p = (const uint2*)copy;
    q.sx = c.sx * (BUF ? 8u : 1u);
    q.sy = c.sy * (BUF ? 8u : 1u);
    q.syf = (float)q.sy;
    q.mz = 8388608.0f + ((float)(q.sy + 8u) - 8.0f * (float)zp.z0);
    q.base = (size_t)c.sx + c.sy + 1u - (size_t)zp.z0;
    if constexpr (BUF) q.r = buffer_rsrc(copy, (uint32_t)(c.elems * 8u));
    return q;
}

// Samples of one lane in order: sample s at fma(s, d, entry), s < lr, the
// trilinear blend of its taps (along x, then y, then z, with explicit fmaf),
// taps outside the grid 0.  kRsUnroll samples per iteration, their loads in
// flight together.  INNER: the wave's first and last samples lie in cells with
// a voxel in the grid on every axis; positions are monotone in s, so every
// sample does and none is tested; up to sample kall
// every ray of the wave has one.  A sample that is not (s >= lr, or its cell
// has no voxel in the grid) adds +0, which leaves the sum unchanged (it starts
// at +0 and is never -0).
//
// FP32 is bound by the texture path: two 16-byte gathers a sample, 33 of its
// cycles at best (four lanes a cycle), 512^3 / 512 views in 54.7 ms where
// (B, z) quads of two slab planes along the detector rows took 91.4; with 8 in
// flight 52.6 there, slower at 256^3 and 1024^3.  16-bit volumes take one gather
// and are bound by VALU issue (FP16 37.1 ms, 76.6 before; with 4 in flight 44.6).
template <typename TV> constexpr int kRsUnroll = sizeof(TV) == 4 ? 4 : 2;
template <bool INNER, typename TV, bool BUF>
__device__ __forceinline__ float rs_samples(const RsRay& r, const RsReader<TV, BUF>& q, int nx, int ny, int nz,
                                            int kall, int kend) {
    constexpr int U = kRsUnroll<TV>;
    float acc = 0.0f, sf = 0.0f;
    const float lrf = (float)r.lr;
    auto samples = [&](auto tested) __attribute__((always_inline)) {
        constexpr bool TEST = decltype(tested)::value;
        typename RsReader<TV, BUF>::Taps t[U];
        float fx[U], fy[U], fz[U];
        bool in[U];
#pragma unroll
        for (int j = 0; j < U; ++j) {
            const float s = sf + (float)j;  // below 2^24: exact
            const float x = fmaf(s, r.dx, r.ex), y = fmaf(s, r.dy, r.ey), z = fmaf(s, r.dz, r.ez);
            float xf = floorf(x), yf = floorf(y), zf = floorf(z);
            fx[j] = x - xf;
            fy[j] = y - yf;
            fz[j] = z - zf;
            in[j] = true;
            if constexpr (TEST) in[j] = s < lrf;
            if constexpr (!INNER) {
                const float xc = __builtin_amdgcn_fmed3f(xf, -1.0f, (float)(nx - 1));
                const float yc = __builtin_amdgcn_fmed3f(yf, -1.0f, (float)(ny - 1));
                const float zc = __builtin_amdgcn_fmed3f(zf, -1.0f, (float)(nz - 1));
                in[j] = in[j] & (xc == xf) & (yc == yf) & (zc == zf);
                xf = xc;
                yf = yc;
                zf = zc;
            }
            const auto o = q.at(xf, yf, zf);
            t[j] = q.load(TEST || !INNER ? q.only(in[j], o) : o);
        }
        float v[U];
#pragma unroll
        for (int j = 0; j < U; ++j) {
            const RsRows c = rs_rows<TV, BUF>(t[j], fx[j]);
            const float c0 = fmaf(fy[j], c.c10 - c.c00, c.c00), c1 = fmaf(fy[j], c.c11 - c.c01, c.c01);
            v[j] = fmaf(fz[j], c1 - c0, c0);
            if constexpr (!BUF && (TEST || !INNER)) v[j] = in[j] ? v[j] : 0.0f;
        }
#pragma unroll
        for (int j = 0; j < U; ++j) acc += v[j];
        sf += (float)U;
    };
    int k = 0;
    if constexpr (INNER)
        for (; k + U <= kall; k += U) samples(std::false_type{});
    for (; k < kend; k += U) samples(std::true_type{});
    return acc;
}

// Forward RS projector.  Samples, taps and the order of the sum are those of
// the per-ray loop (sample s at fma(s, d, entry), trilinear interpolation,
// acc += in s order), so results are unchanged; what changes is the schedule
// and the layout.  A wave is `rows` detector rows of 64 / rows columns and takes
// sample s of its rays together.  The rays of a column enter the FOV at the
// same in-plane point and stay close in plane at equal s (their in-plane steps
// differ by the cosine of the cone angle), so the taps of neighbouring rows are
// neighbours along z, the fastest axis of the copy.
template <typename TV, typename TS, bool BUF>
__device__ __forceinline__ void rs_tile(const DevGeom& g, int cube, const void* __restrict__ copy, ProjPlanes zp,
                                        float vol_inv, TS* __restrict__ sino, float sino_scale, int rows, int bx, int pg,
                                        int bz) {
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int per = 64 / rows;  // columns of a wave
    const int p = pg * kProjViews + wv;
    const int m = bx * per + lane / rows;
    const int n = bz * rows + lane % rows;
    const bool inside = p < g.nphi && m < g.nu && n < g.nv;
    // (an entry up to half a voxel above the last slice's centre counts)
    if (proj_rows_miss(g, (cube ? 0.70711 : 0.5) * (double)g.nx * (double)g.delta, (0.5 * g.nz + 0.5) * (double)g.delta,
                       bz * rows, rows)) {
        if (inside) Storage<TS>::store(sino, (size_t)m + (size_t)g.nu * ((size_t)n + (size_t)g.nv * p), 0.0f, sino_scale);
        return;
    }
    RsRay r{0, 0, 0, 0, 0, 0, 0};
    if (inside) r = rs_setup(g, cube, p, m, n);
    const bool ok = r.lr > 0;
    // a lane without a ray samples the first plane's cell (0, 0); its sum is dropped
    if (!ok) r.ez = (float)zp.z0;
    const int nx = g.nx, ny = g.ny, nz = g.nz;
    auto within = [](float a, float b, int n1) {
        const float fa = floorf(a), fb = floorf(b);
        return (fa >= -1.0f) & (fa <= (float)(n1 - 1)) & (fb >= -1.0f) & (fb <= (float)(n1 - 1));
    };
    const float sl = (float)(r.lr - 1);
    const bool inner = within(r.ex, fmaf(sl, r.dx, r.ex), nx) & within(r.ey, fmaf(sl, r.dy, r.ey), ny) &
                       within(r.ez, fmaf(sl, r.dz, r.ez), nz);
    const int kend = __builtin_amdgcn_readfirstlane(wave_max(ok ? r.lr : 0));
    const int kall = __builtin_amdgcn_readfirstlane(min(wave_min(ok ? r.lr : INT_MAX), kend));
    const auto q = make_rs_reader<TV, BUF>(copy, nx, ny, zp);
    float acc = __ballot(ok && !inner) == 0ull ? rs_samples<true>(r, q, nx, ny, nz, kall, kend)
                                               : rs_samples<false>(r, q, nx, ny, nz, kall, kend);
    // 16-bit volumes are read unscaled; the sum is linear in them, so the
    // storage scale applies once to it (FP32 storage has no scale).
    if (sizeof(TV) == 2) acc *= vol_inv;
    if (inside) {
        const size_t o = (size_t)m + (size_t)g.nu * ((size_t)n + (size_t)g.nv * p);
        Storage<TS>::store(sino, o, ok ? acc * g.delta : 0.0f, sino_scale);
    }
}

template <typename TV, typename TS, bool BUF>
__global__ __launch_bounds__(64 * kProjViews) void rs_kernel(DevGeom g, int cube, const void* __restrict__ copy,
                                                             ProjPlanes zp, float vol_inv, TS* __restrict__ sino,
                                                             float sino_scale, int rows) {
    rs_tile<TV, TS, BUF>(g, cube, copy, zp, vol_inv, sino, sino_scale, rows,
                         proj_group(blockIdx.x, gridDim.x, blockIdx.y, gridDim.y, blockIdx.z), blockIdx.y, blockIdx.z);
}

// ---------------------------------------------------------------------------
// LDS-staged RS (FP32 volumes).
//
// A workgroup is 32 x 8 detector cells of one view.  When all its rays share
// the dominant in-plane axis A (|d_A| >= the other two) and its direction,
// it walks A in windows: for the window of samples with floor(A) in
// [wlo, whi] it copies the voxels those samples interpolate (planes
// wlo .. whi + 1, the window's box of z rows and B columns, stage_box.hpp)
// into LDS, and every lane takes its samples of the window with the eight
// taps read from there (four ds_read2_b32 per sample).  The staging is double
// buffered: the copy of window i + 1 is in flight while the workgroup samples
// window i, and one barrier per window separates them.  A window holds up to
// kRsWmax sample planes, fewer (6, 4, 2, then 1) when its box is too large
// for a buffer.  The box is not clipped to the grid: a sample outside the grid (a
// cylinder wider than a y extent smaller than x, or a ray whose clipped exit
// lies behind its entry) reads zero taps there and adds +0, as the range
// test of the per-ray loop makes it.  Samples, taps, arithmetic and the order
// of the sum are those of the per-ray loop, so results equal rs_kernel's bit
// for bit.  A window whose box exceeds a buffer even at one plane, and a
// workgroup whose rays do not share A and its direction, read their taps
// from the volume directly.
constexpr int kRsWmax = 8;  // sample planes per window at most

// The eight taps straight from the volume, 0 off the grid, blended as rs_samples does.
__device__ __forceinline__ float trilinear_direct(const float* __restrict__ f, int nx, int ny, int nz, float x,
                                                  float y, float z) {
    const float xf = floorf(x), yf = floorf(y), zf = floorf(z);
    if (!(xf >= -1.0f && xf <= (float)nx && yf >= -1.0f && yf <= (float)ny && zf >= -1.0f && zf <= (float)nz))
        return 0.0f;
    const int ix = (int)xf, iy = (int)yf, iz = (int)zf;
    const float fx = x - xf, fy = y - yf, fz = z - zf;
    const size_t sy = (size_t)nx, sz = (size_t)nx * ny;
    auto t = [&](int X, int Y, int Z) {
        const bool ok = (unsigned)X < (unsigned)nx && (unsigned)Y < (unsigned)ny && (unsigned)Z < (unsigned)nz;
        return ok ? f[(size_t)X + sy * (size_t)Y + sz * (size_t)Z] : 0.0f;
    };
    const float t000 = t(ix, iy, iz), t100 = t(ix + 1, iy, iz), t010 = t(ix, iy + 1, iz);
    const float t110 = t(ix + 1, iy + 1, iz), t001 = t(ix, iy, iz + 1), t101 = t(ix + 1, iy, iz + 1);
    const float t011 = t(ix, iy + 1, iz + 1), t111 = t(ix + 1, iy + 1, iz + 1);
    const float c00 = fmaf(fx, t100 - t000, t000), c10 = fmaf(fx, t110 - t010, t010);
    const float c01 = fmaf(fx, t101 - t001, t001), c11 = fmaf(fx, t111 - t011, t011);
    const float c0 = fmaf(fy, c10 - c00, c00), c1 = fmaf(fy, c11 - c01, c01);
    return fmaf(fz, c1 - c0, c0);
}

// A window: samples with floor(A) in [wlo, whi], staged planes wlo .. whi + 1
// (s.lo = wlo).  All fields are wave-uniform.
struct RsWindow {
    int wlo, whi;
    StageWin s;
};

// The window that starts at sample plane `from` in the travel direction: the
// largest of kRsWmax, 6, 4, 2, 1 planes whose box fits a buffer.
__device__ __forceinline__ RsWindow rs_plan(const WgCorners& wc, int from, bool inc, int max_nzr) {
    RsWindow w{};
    for (int W = kRsWmax;; W = W > 4 ? W - 2 : W >> 1) {
        const int wlo = inc ? from : from - W + 1, whi = wlo + W - 1;
        const StageBox b = stage_box(wc, (float)wlo, (float)(whi + 1), 0.0f, 0, 1);
        w = RsWindow{wlo, whi, stage_window(b, wlo, W + 1, max_nzr)};
        if (w.s.fits || W == 1) break;
    }
    return w;
}

#ifndef RS_STAGED_UNROLL
#define RS_STAGED_UNROLL 4
#endif

// The window walk of one workgroup along A (0: x, 1: y); inc: A increasing.
// src: rows of nBp floats along B (A = 0: the y-fastest copy, A = 1: the
// volume or its x-padded copy).  first, last: the workgroup's first and last
// sample planes.  wc: the corner rays (every wave plans the same windows).
template <int A>
__device__ __forceinline__ float rs_staged_walk(const DevGeom& g, const RsRay& r, int lr, bool inc, int first, int last,
                                                const float* __restrict__ src, int nBp, const float* __restrict__ vol,
                                                const WgCorners& wc, float* __restrict__ st0,
                                                float* __restrict__ st1, int lane, int wv) {
    const int nx = g.nx, ny = g.ny, nz = g.nz;
    const int nA = A == 0 ? nx : ny;
    const size_t src_elems = (size_t)nBp * (size_t)nA * (size_t)nz;
    float acc = 0.0f;
    int s = 0;
    const int max_nzr = stage_max_rows(nA, nBp);
    RsWindow cur = rs_plan(wc, first, inc, max_nzr);
    if (cur.s.fits) stage_copy(src, src_elems, nA, nBp, nz, cur.s, st0, lane, wv);
    // One window: window `cur` is in `buf`, the next one is copied into
    // `other`; false after the last window.  The windows alternate between
    // the two LDS arrays and each call names them directly, so the compiler
    // knows that the copy in flight does not write what the reads read and
    // does not wait for it before them.
    auto window = [&](const float* __restrict__ buf, float* __restrict__ other) __attribute__((always_inline)) {
        // this wave's copies of window `cur` have landed; every wave is done with the other buffer
        __builtin_amdgcn_s_waitcnt(0);
        __syncthreads();
        const int from = inc ? cur.whi + 1 : cur.wlo - 1;
        const bool more = inc ? from <= last : from >= last;
        RsWindow nxt = cur;
        if (more) {
            nxt = rs_plan(wc, from, inc, max_nzr);
            if (nxt.s.fits) stage_copy(src, src_elems, nA, nBp, nz, nxt.s, other, lane, wv);
        }
        const float wlof = (float)cur.wlo, whif = (float)cur.whi;
        // offset of tap (a, z, b) in the buffer, ((a - wlo) nzr + z - zlo) P + b - blo4 with P = 4 nch
        // floats per row, as one exact FP32 expression of integers below 2^24 (the launcher admits
        // grids with nA kSlotFloats < 2^24)
        const int P = 4 * cur.s.nch;
        const int pstride = cur.s.nzr * P;
        const float ps = (float)pstride, pf = (float)P;
        const float c0 = -((float)cur.wlo * ps + (float)(cur.s.zlo * P + cur.s.blo4));
        for (;;) {
            float px[RS_STAGED_UNROLL], py[RS_STAGED_UNROLL], pz[RS_STAGED_UNROLL];
            bool act[RS_STAGED_UNROLL];
#pragma unroll
            for (int j = 0; j < RS_STAGED_UNROLL; ++j) {
                const float sf = (float)(s + j);
                px[j] = fmaf(sf, r.dx, r.ex);
                py[j] = fmaf(sf, r.dy, r.ey);
                pz[j] = fmaf(sf, r.dz, r.ez);
                const float fa = floorf(A == 0 ? px[j] : py[j]);
                act[j] = (s + j < lr) & (fa >= wlof) & (fa <= whif);
            }
            if (__ballot(act[0]) == 0ull) break;
            float v[RS_STAGED_UNROLL];
            if (cur.s.fits) {
                float fx[RS_STAGED_UNROLL], fy[RS_STAGED_UNROLL], fz[RS_STAGED_UNROLL];
                int off[RS_STAGED_UNROLL];
#pragma unroll
                for (int j = 0; j < RS_STAGED_UNROLL; ++j) {
                    const float xf = floorf(px[j]), yf = floorf(py[j]), zf = floorf(pz[j]);
                    fx[j] = px[j] - xf;
                    fy[j] = py[j] - yf;
                    fz[j] = pz[j] - zf;
                    const float af = A == 0 ? xf : yf, bf = A == 0 ? yf : xf;
                    const int o = (int)fmaf(af, ps, fmaf(zf, pf, bf + c0));
                    off[j] = act[j] ? o : 0;
                }
                float u[RS_STAGED_UNROLL][4], w[RS_STAGED_UNROLL][4];
#pragma unroll
                for (int j = 0; j < RS_STAGED_UNROLL; ++j) {
                    const float* q0 = buf + off[j];
                    const float* q1 = q0 + pstride;
                    // (b, z), (b, z+1), (b+1, z), (b+1, z+1) on planes ia, ia + 1
                    u[j][0] = q0[0];
                    u[j][1] = q0[P];
                    u[j][2] = q0[1];
                    u[j][3] = q0[P + 1];
                    w[j][0] = q1[0];
                    w[j][1] = q1[P];
                    w[j][2] = q1[1];
                    w[j][3] = q1[P + 1];
                }
#pragma unroll
                for (int j = 0; j < RS_STAGED_UNROLL; ++j) {
                    float t000, t100, t010, t110, t001, t101, t011, t111;
                    if (A == 0) {
                        t000 = u[j][0]; t001 = u[j][1]; t010 = u[j][2]; t011 = u[j][3];
                        t100 = w[j][0]; t101 = w[j][1]; t110 = w[j][2]; t111 = w[j][3];
                    } else {
                        t000 = u[j][0]; t001 = u[j][1]; t100 = u[j][2]; t101 = u[j][3];
                        t010 = w[j][0]; t011 = w[j][1]; t110 = w[j][2]; t111 = w[j][3];
                    }
                    const float c00 = fmaf(fx[j], t100 - t000, t000), c10 = fmaf(fx[j], t110 - t010, t010);
                    const float c01 = fmaf(fx[j], t101 - t001, t001), c11 = fmaf(fx[j], t111 - t011, t011);
                    const float e0 = fmaf(fy[j], c10 - c00, c00), e1 = fmaf(fy[j], c11 - c01, c01);
                    const float val = fmaf(fz[j], e1 - e0, e0);
                    v[j] = act[j] ? val : 0.0f;
                }
            } else {
#pragma unroll
                for (int j = 0; j < RS_STAGED_UNROLL; ++j)
                    v[j] = act[j] ? trilinear_direct(vol, nx, ny, nz, px[j], py[j], pz[j]) : 0.0f;
            }
            int adv = 0;
#pragma unroll
            for (int j = 0; j < RS_STAGED_UNROLL; ++j) {
                acc += v[j];
                adv += act[j] ? 1 : 0;
            }
            s += adv;
        }
        cur = nxt;
        return more;
    };
    while (window(st0, st1) && window(st1, st0)) {
    }
    return acc;
}

// Forward RS with LDS-staged taps (FP32 volume `vol`).  volT: its y-fastest
// copy with rows of nyp floats, volP: rows of nxp floats along x (the volume
// itself when nxp = nx); nxp, nyp are nx, ny rounded up to multiples of four.
// Grid: x = column group, y = view, z = row group.
template <typename TS>
__global__ __launch_bounds__(BX* BY, 5) void rs_staged_kernel(DevGeom g, int cube, const float* __restrict__ vol,
                                                             const float* __restrict__ volT,
                                                             const float* __restrict__ volP, int nxp, int nyp,
                                                             TS* __restrict__ sino, float sino_scale) {
    __shared__ float st0[kSlotFloats];
    __shared__ float st1[kSlotFloats];
    __shared__ int wsh[4][3];
    const int tid = threadIdx.y * BX + threadIdx.x;
    const int lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int bx = blockIdx.x, p = blockIdx.y, bz = blockIdx.z;
    const int m = bx * BX + threadIdx.x;
    const int n = bz * BY + threadIdx.y;
    const bool inside = m < g.nu && n < g.nv;
    RsRay r{0, 0, 0, 0, 0, 0, 0};
    if (inside) r = rs_setup(g, cube, p, m, n);
    const bool ok = r.lr > 0;
    int code = -1;
    if (ok) {
        const float ax = fabsf(r.dx), ay = fabsf(r.dy), az = fabsf(r.dz);
        if (ax > 0.0f && ax >= ay && ax >= az) code = r.dx > 0.0f ? 0 : 1;
        else if (ay > 0.0f && ay >= ax && ay >= az) code = r.dy > 0.0f ? 2 : 3;
    }
    // The workgroup's mode: 0..3 (axis x / y, increasing / decreasing), 4: no
    // ray, -1: the rays differ.
    const unsigned long long okmask = __ballot(ok);
    int wmode = 4;
    if (okmask != 0ull) {
        wmode = -1;
#pragma unroll
        for (int c = 0; c < 4; ++c)
            if (__ballot(ok && code == c) == okmask) wmode = c;
    }
    if (lane == 0) wsh[wv][0] = wmode;
    __syncthreads();
    int mode = 4;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const int mk = wsh[k][0];
        if (mk != 4) mode = (mode == 4 || mode == mk) ? mk : -1;
    }
    mode = __builtin_amdgcn_readfirstlane(mode);
    float acc = 0.0f;
    if (mode == -1) {
        for (int s = 0; s < r.lr; ++s) {
            const float sf = (float)s;
            acc += trilinear_direct(vol, g.nx, g.ny, g.nz, fmaf(sf, r.dx, r.ex), fmaf(sf, r.dy, r.ey),
                                    fmaf(sf, r.dz, r.ez));
        }
    } else if (mode != 4) {
        const int A = mode < 2 ? 0 : 1;
        const bool inc = (mode & 1) == 0;
        // the workgroup's first and last sample planes along the travel direction
        int first = inc ? INT_MAX : INT_MIN, last = inc ? INT_MIN : INT_MAX;
        if (ok) {
            const float e = A == 0 ? r.ex : r.ey, d = A == 0 ? r.dx : r.dy;
            first = (int)floorf(e);
            last = (int)floorf(fmaf((float)(r.lr - 1), d, e));
        }
        first = inc ? wave_min(first) : wave_max(first);
        last = inc ? wave_max(last) : wave_min(last);
        __syncthreads();  // every wave has read wsh[*][0]
        if (lane == 0) {
            wsh[wv][1] = first;
            wsh[wv][2] = last;
        }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            first = inc ? min(first, wsh[k][1]) : max(first, wsh[k][1]);
            last = inc ? max(last, wsh[k][2]) : min(last, wsh[k][2]);
        }
        first = __builtin_amdgcn_readfirstlane(first);
        last = __builtin_amdgcn_readfirstlane(last);
        const int mlo = bx * BX, mhi = min(bx * BX + BX - 1, g.nu - 1);
        const int nlo = bz * BY, nhi = min(bz * BY + BY - 1, g.nv - 1);
        const WgCorners wc = wg_corners(g, A, p, mlo, mhi, nlo, nhi);
        if (A == 0)
            acc = rs_staged_walk<0>(g, r, ok ? r.lr : 0, inc, first, last, volT, nyp, vol, wc, st0, st1, lane, wv);
        else
            acc = rs_staged_walk<1>(g, r, ok ? r.lr : 0, inc, first, last, volP, nxp, vol, wc, st0, st1, lane, wv);
    }
    if (inside) {
        const size_t o = (size_t)m + (size_t)g.nu * ((size_t)n + (size_t)g.nv * p);
        Storage<TS>::store(sino, o, r.lr > 0 ? acc * g.delta : 0.0f, sino_scale);
    }
}

// Shared launch (FP32 or BF16 (kItemBF16) RS copies, FP32 sinograms); item
// flags bit 0 selects the cube FOV.  No minimum-waves bound: under one the
// compiler waits for each sample's gathers before it issues the next
// sample's.  Its grid is what the chip holds at once (batch_grids_init), so
// every workgroup is resident from the start.
__global__ __launch_bounds__(64 * kProjViews) void rs_batch_kernel(const BatchTable* __restrict__ t, uint32_t* __restrict__ next) {
    TOMO_BATCH_CLAIMED(t, next) {
        const BatchItem& it = t->item[batch_find(t, tile)];
        const uint32_t local = tile - it.begin;
        const uint32_t rest = local / it.gx;
        const int by = (int)(rest % it.gy), bz = (int)(rest / it.gy), cube = it.flags & 1;
        const int bx = proj_group(local % it.gx, it.gx, (uint32_t)by, it.gy, (uint32_t)bz);
        const bool bf = (it.flags & kItemBF16) != 0;
        const bool buf = rs_copy_shape(it.g.nx, it.g.ny, it.planes.nz, bf ? 2 : 4).buf;
        const int rows = 1 << (it.flags >> kItemRowsShift);
        using BF = __hip_bfloat16;
        if (bf && buf)
            rs_tile<BF, float, true>(it.g, cube, it.in, it.planes, 1.0f, (float*)it.out, 1.0f, rows, bx, by, bz);
        else if (bf)
            rs_tile<BF, float, false>(it.g, cube, it.in, it.planes, 1.0f, (float*)it.out, 1.0f, rows, bx, by, bz);
        else if (buf)
            rs_tile<float, float, true>(it.g, cube, it.in, it.planes, 1.0f, (float*)it.out, 1.0f, rows, bx, by, bz);
        else
            rs_tile<float, float, false>(it.g, cube, it.in, it.planes, 1.0f, (float*)it.out, 1.0f, rows, bx, by, bz);
    }
}

// RS^T: f[tap] += delta * w_tap * g(ray) (FP32 atomics; output zeroed first).
template <typename TS>
__global__ __launch_bounds__(BX* BY) void rs_adjoint_kernel(DevGeom g, int cube, const TS* __restrict__ sino,
                                                          float sino_inv, float* __restrict__ vol) {
    const int m = blockIdx.x * BX + threadIdx.x;
    const int n = blockIdx.y * BY + threadIdx.y;
    const int p = blockIdx.z;
    if (m >= g.nu || n >= g.nv) return;
    const size_t oi = (size_t)m + (size_t)g.nu * ((size_t)n + (size_t)g.nv * p);
    const float gv = Storage<TS>::load(sino, oi, sino_inv);
    if (gv == 0.0f) return;
    const RsRay r = rs_setup(g, cube, p, m, n);
    const float val = g.delta * gv;
    const int nx = g.nx, ny = g.ny, nz = g.nz;
    const int64_t sy = nx, sz = (int64_t)nx * ny;
    for (int s = 0; s < r.lr; ++s) {
        const float sf = (float)s;
        const float x = fmaf(sf, r.dx, r.ex), y = fmaf(sf, r.dy, r.ey), z = fmaf(sf, r.dz, r.ez);
        const float xf = floorf(x), yf = floorf(y), zf = floorf(z);
        if (!(xf >= -1.0f && xf <= (float)nx && yf >= -1.0f && yf <= (float)ny && zf >= -1.0f && zf <= (float)nz))
            continue;
        const int ix = (int)xf, iy = (int)yf, iz = (int)zf;
        const float fx = x - xf, fy = y - yf, fz = z - zf;
#pragma unroll
        for (int c = 0; c < 8; ++c) {
            const int ox = c & 1, oy = (c >> 1) & 1, oz = (c >> 2) & 1;
            const int X = ix + ox, Y = iy + oy, Z = iz + oz;
            if (X < 0 || X >= nx || Y < 0 || Y >= ny || Z < 0 || Z >= nz) continue;
            const float w = (ox ? fx : 1.0f - fx) * (oy ? fy : 1.0f - fy) * (oz ? fz : 1.0f - fz);
            unsafeAtomicAdd(vol + (X + sy * Y + sz * Z), w * val);
        }
    }
}

// ---------------------------------------------------------------------------
// RS^T as a gather: a voxel sums (1-|x-i|)(1-|y-j|)(1-|z-k|) delta g over the
// samples next to it, and is written once.
//
// All rays of a detector column run along one in-plane line, enter the FOV at
// one point of it and differ by their slope: at the in-plane distance t from
// the source (voxels), row n is at z = cz + t (n - cv) qz, its samples at t1 + s c
// with c the cosine of its cone angle.  A wave owns a voxel column (i, j) and 64 K
// of its voxels, lanes along z.  For 64 views at a time each lane finds its
// view's detector columns whose line crosses the square of side 2 around
// (i, j) and that line's terms in FP64; the wave then takes the lines one by one.
// A lane's rows are the two to four that pass its voxel within the square, each
// with one 16-byte read of (delta g, samples, c, its rounding error) from a table
// with rows fastest, and their samples the one to four on the chord.  The terms
// are relative to the point of the line next to the column, so that the weights
// hold no rounding of a large coordinate.
//
// VALU issue bounds it: 8 cycles per sample (6 with its mirror image), 15 per row
// and 20 per line of 64 voxels.  Against the scatter below, 256^3 and 256 views:
// 684 -> 34.0 ms, 26.5 with the mirror images, 25.0 with six waves per SIMD (a few
// registers in memory; 128^3 and 128 views 2.32 ms at four, 2.06 at six, 2.03 at
// seven); 64^3 and 64 views 4.2 -> 0.30 ms; 17^3 and 16 views 78 -> 73 us, so that no
// size goes back to it.
constexpr int kRsTWaves = 4;
__host__ __device__ inline size_t rs_t_rows(int nv) { return (size_t)nv + 2; }  // row -1 and row nv hold no ray

// tab[(q nu + m) rows + n + 1] for the np views from p0 on; 8 x 32 (m, row) per workgroup.
template <typename TS>
__global__ __launch_bounds__(256) void rs_t_prepare_kernel(DevGeom g, int cube, const TS* __restrict__ sino,
                                                           float sino_inv, int p0, float4* __restrict__ tab) {
    const int rows = (int)rs_t_rows(g.nv);
    const uint32_t gx = (uint32_t)(g.nu + 7) / 8, gy = (uint32_t)(rows + 31) / 32;
    const uint32_t bx = blockIdx.x % gx, rest = blockIdx.x / gx, by = rest % gy, q = rest / gy;
    const int m = (int)bx * 8 + (threadIdx.x & 7), n = (int)by * 32 + (threadIdx.x >> 3) - 1;
    if (m >= g.nu || n >= g.nv + 1) return;
    float4 e = make_float4(0.0f, 0.0f, 1.0f, 0.0f);
    if (n >= 0 && n < g.nv) {
        const int p = p0 + (int)q;
        const RsRay r = rs_setup(g, cube, p, m, n);
        const double s = ((double)m - (double)g.cu) * (double)g.du, t = ((double)n - (double)g.cv) * (double)g.dv;
        const double r2 = g.fdd * g.fdd + s * s, c = sqrt(r2 / (r2 + t * t));
        if (r.lr > 0) e.x = g.delta * Storage<TS>::load(sino, (size_t)m + (size_t)g.nu * ((size_t)n + (size_t)g.nv * q), sino_inv);
        e.y = (float)r.lr;
        e.z = (float)c;
        e.w = (float)(c - (double)e.z);
    }
    tab[((size_t)q * g.nu + m) * rows + n + 1] = e;
}

__device__ __forceinline__ float lane_value(float v, int l) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l));
}

// MIRROR: a lane takes its voxel k of the lower half and the mirror image nz - 1 - k,
// whose samples lie on the mirrored rows with the same weights; the rays' values and
// numbers of samples are the mirrored rows' own.
//
// Grid: x, y = (4 voxel columns along x, j), z = z block of 64 K.  Views p0 + [0, np).
template <int K, bool MIRROR>
__global__ __launch_bounds__(64 * kRsTWaves, 6) void rs_t_kernel(DevGeom g, int cube, const float4* __restrict__ tab, int p0,
                                                             int np, int add, float* __restrict__ vol) {
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const uint32_t gx = (uint32_t)(g.nx + kRsTWaves - 1) / kRsTWaves;
    const uint32_t tile = tile_index();
    const int i = (int)(tile % gx) * kRsTWaves + wv, j = (int)(tile / gx);
    if (i >= g.nx || j >= g.ny) return;
    const int kb = (int)blockIdx.z * 64 * K;
    const int rows = (int)rs_t_rows(g.nv);
    const double dl = (double)g.delta, fod = g.fod / dl;
    const double xi = (double)i - (double)g.cx, yj = (double)j - (double)g.cy;
    const double half = 0.5 * (double)g.nx, R2 = cube ? 2.0 * (half * half) : half * half;
    const float cv = g.cv, last = (float)g.nv;
    const float kmax = fmaxf(fabsf((float)kb - g.cz), fabsf((float)min(kb + 64 * K, MIRROR ? (g.nz + 1) / 2 : g.nz) - 1.0f - g.cz));
    constexpr int B = MIRROR ? 2 : 1;
    float kk[K], total[B][K], acc[B][K];
#pragma unroll
    for (int c = 0; c < K; ++c) {
        kk[c] = (float)(kb + 64 * c + lane) - g.cz;
#pragma unroll
        for (int b = 0; b < B; ++b) total[b][c] = 0.0f;
    }
    for (int pb = 0; pb < np; pb += 64) {
        // ---- one view per lane: the detector columns whose lines may cross the square
        const int q = pb + lane;
        const double* vw = g.view + (size_t)(p0 + min(q, np - 1)) * kViewStride;
        const double ca = vw[0], sa = vw[1];
        double u0 = INFINITY, u1 = -INFINITY;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const double x = xi + (e & 1 ? 1.0 : -1.0), y = yj + (e & 2 ? 1.0 : -1.0);
            const double u = (ca * y - sa * x) / (ca * x + sa * y + fod);
            u0 = fmin(u0, u);
            u1 = fmax(u1, u);
        }
        const double ku = g.fdd / (double)g.du;
        const double mlo = ceil(fma(u0, ku, (double)g.cu) - 1e-6), mhi = floor(fma(u1, ku, (double)g.cu) + 1e-6);
        const int m0 = (int)fmax(mlo, 0.0);
        const int cnt = q < np ? max(0, (int)fmin(mhi, (double)(g.nu - 1)) - m0 + 1) : 0;
        const int most = __builtin_amdgcn_readfirstlane(wave_max(cnt));
        for (int h = 0; h < most; ++h) {
            // ---- one line per lane; partial sums of a line, of 64 lines, and of all
#pragma unroll
            for (int c = 0; c < K; ++c)
#pragma unroll
                for (int b = 0; b < B; ++b) acc[b][c] = 0.0f;
            const int m = m0 + h;
            bool on = h < cnt;
            const double sm = ((double)m - (double)g.cu) * (double)g.du;
            const double rx = ca * g.fdd - sm * sa, ry = sa * g.fdd + sm * ca;
            const double ir = 1.0 / sqrt(rx * rx + ry * ry);
            const double ux = rx * ir, uy = ry * ir, Sx = -fod * ca, Sy = -fod * sa;
            const double ta = (xi - Sx) * ux + (yj - Sy) * uy;  // next to the column
            const float lax = (float)((Sx - xi) + ta * ux), lay = (float)((Sy - yj) + ta * uy);
            const float lux = (float)ux, luy = (float)uy;
            // the chord [lo, hi] of the square, from ta
            const float jx = 1.0f / lux, jy = 1.0f / luy;
            const float x0 = (-1.0f - lax) * jx, x1 = (1.0f - lax) * jx;
            const float y0 = (-1.0f - lay) * jy, y1 = (1.0f - lay) * jy;
            const float llo = fmaxf(fminf(x0, x1), fminf(y0, y1)), lhi = fminf(fmaxf(x0, x1), fmaxf(y0, y1));
            // entry, as rs_setup's l1 times the cosine
            const double b = Sx * ux + Sy * uy, disc = b * b - ((Sx * Sx + Sy * Sy) - R2);
            double t1 = -b - sqrt(disc);
            if (cube) {
                const double ex0 = (-(double)g.cx - Sx) / ux, ex1 = ((double)(g.nx - 1) - (double)g.cx - Sx) / ux;
                const double ey0 = (-(double)g.cy - Sy) / uy, ey1 = ((double)(g.ny - 1) - (double)g.cy - Sy) / uy;
                if (ux != 0.0) t1 = fmax(t1, fmin(ex0, ex1));
                if (uy != 0.0) t1 = fmax(t1, fmin(ey0, ey1));
            }
            const double D = ta - t1, qz = (double)g.dv * ir, A = ta * qz;
            const float lD = (float)D, lDl = (float)(D - (double)lD), lA = (float)A, lAl = (float)(A - (double)lA);
            const float lq = (float)qz;
            const float li0 = 1.0f / (float)((ta + (double)llo) * qz), li1 = 1.0f / (float)((ta + (double)lhi) * qz);
            const float steep = fmaxf(cv, last - 1.0f - cv) * lq;
            const float nrows = floorf(2.0f * li0 + kmax * (li0 - li1) + 4e-3f) + 1.0f;
            const float nsamp = floorf((lhi - llo) * sqrtf(fmaf(steep, steep, 1.0f)) + 2e-3f) + 1.0f;
            on = on && disc >= 0.0 && lhi > llo && lD + lhi >= 0.0f;
            const int lnum = (int)fminf(nrows, (float)rows) << 8 | (int)fminf(nsamp, 255.0f);
            const int lbase = q * g.nu + m;
            for (uint64_t todo = __ballot(on); todo != 0ull; todo &= todo - 1) {
                const int l = __builtin_ctzll(todo);
                const float ax = lane_value(lax, l), ay = lane_value(lay, l), uxs = lane_value(lux, l);
                const float uys = lane_value(luy, l), Dh = lane_value(lD, l), Dl = lane_value(lDl, l);
                const float Ah = lane_value(lA, l), Al = lane_value(lAl, l), qs = lane_value(lq, l);
                const float i0 = lane_value(li0, l), i1 = lane_value(li1, l), Dlo = Dh + lane_value(llo, l);
                const int num = __builtin_amdgcn_readlane(lnum, l), R = num >> 8, S = num & 255;
                const float4* line = tab + (size_t)(uint32_t)__builtin_amdgcn_readlane(lbase, l) * rows + 1;
                float row[K], part[B][K];
#pragma unroll
                for (int c = 0; c < K; ++c) {
#pragma unroll
                    for (int b = 0; b < B; ++b) part[b][c] = 0.0f;
                    const float k0 = kk[c] - 1.0f;
                    // first that may reach the voxel; -1 before the detector, whose rows R covers
                    row[c] = fmaxf(ceilf(fminf(k0 * i0, k0 * i1) + (cv - 2e-3f)), -1.0f);
                }
                for (int r = 0; r < R; ++r) {
                    typedef float V4 __attribute__((ext_vector_type(4)));
                    typedef float V2 __attribute__((ext_vector_type(2)));
                    V4 e[K];
                    V2 image[K];  // (delta g, samples) of the mirrored row
#pragma unroll
                    for (int c = 0; c < K; ++c) {
                        e[c] = *(const V4*)(line + (int)__builtin_amdgcn_fmed3f(row[c], -1.0f, last));
                        image[c] = (V2)0.0f;
                        if (MIRROR)
                            image[c] = *(const V2*)(line + (int)__builtin_amdgcn_fmed3f(last - 1.0f - row[c], -1.0f, last));
                    }
                    float sg[K], zb[K], dt[K], rem[B][K], w[B][K];
#pragma unroll
                    for (int c = 0; c < K; ++c) {
                        // whole before the loops on the numbers (empty statement)
                        asm volatile("" : "+v"(e[c]), "+v"(image[c]));
                        const float nr = row[c] - cv;
                        sg[c] = nr * qs;
                        zb[c] = fmaf(nr, Al, fmaf(nr, Ah, -kk[c]));
                        const float s0 = fmaxf(ceilf(fmaf(Dlo, __builtin_amdgcn_rcpf(e[c].z), -1e-3f)), 0.0f);
                        dt[c] = fmaf(s0, e[c].z, -Dh) + fmaf(s0, e[c].w, -Dl);
                        rem[0][c] = e[c].y - s0;
                        w[0][c] = 0.0f;
                        if (MIRROR) {
                            rem[B - 1][c] = image[c].y - s0;
                            w[B - 1][c] = 0.0f;
                        }
                        row[c] += 1.0f;
                    }
                    float ts = 0.0f;
                    for (int t = 0; t < S; ++t) {
#pragma unroll
                        for (int c = 0; c < K; ++c) {
                            const float wx = __builtin_amdgcn_fmed3f(1.0f - fabsf(fmaf(dt[c], uxs, ax)), 0.0f, 1.0f);
                            const float wy = __builtin_amdgcn_fmed3f(1.0f - fabsf(fmaf(dt[c], uys, ay)), 0.0f, 1.0f);
                            const float wz = __builtin_amdgcn_fmed3f(1.0f - fabsf(fmaf(dt[c], sg[c], zb[c])), 0.0f, 1.0f);
                            const float wxy = wx * wy;
#pragma unroll
                            for (int b = 0; b < B; ++b) w[b][c] = fmaf(ts < rem[b][c] ? wxy : 0.0f, wz, w[b][c]);
                            dt[c] += e[c].z;
                        }
                        ts += 1.0f;
                    }
                    // a weight of 0 takes nothing from its ray, whatever it holds
#pragma unroll
                    for (int c = 0; c < K; ++c)
#pragma unroll
                        for (int b = 0; b < B; ++b)
                            part[b][c] = w[b][c] > 0.0f ? fmaf(w[b][c], b ? image[c].x : e[c].x, part[b][c]) : part[b][c];
                }
#pragma unroll
                for (int c = 0; c < K; ++c)
#pragma unroll
                    for (int b = 0; b < B; ++b) acc[b][c] += part[b][c];
            }
#pragma unroll
            for (int c = 0; c < K; ++c)
#pragma unroll
                for (int b = 0; b < B; ++b) total[b][c] += acc[b][c];
        }
    }
    const size_t sxy = (size_t)g.nx * g.ny;
#pragma unroll
    for (int c = 0; c < K; ++c) {
        const int k = kb + 64 * c + lane;
#pragma unroll
        for (int b = 0; b < B; ++b) {
            const int z = b ? g.nz - 1 - k : k;
            // the middle slice of an odd volume belongs to the lower half
            if (!MIRROR ? z < g.nz : b ? 2 * z >= g.nz : 2 * z < g.nz) {
                float* o = vol + ((size_t)i + (size_t)g.nx * j + sxy * z);
                *o = add ? *o + total[b][c] : total[b][c];
            }
        }
    }
}

__global__ __launch_bounds__(BX* BY) void rs_count_kernel(DevGeom g, int cube, unsigned long long* total) {
    const int m = blockIdx.x * BX + threadIdx.x;
    const int n = blockIdx.y * BY + threadIdx.y;
    const int p = blockIdx.z;
    unsigned long long c = 0;
    if (m < g.nu && n < g.nv) c = (unsigned long long)rs_setup(g, cube, p, m, n).lr;
    // wave-level sum, one atomic per wave
    for (int off = 32; off > 0; off >>= 1) c += __shfl_down(c, off, 64);
    if (((threadIdx.y * BX + threadIdx.x) & 63) == 0) atomicAdd(total, c);  // first lane of the wave
}

}  // namespace

int launch_rs(const tomo_geom* g, int cube, Buf vol, MutBuf sino, hipStream_t s, const ProjExtra& x) {
    const DevGeom& d = g->dev;
    const dim3 grid(ceil_div(d.nu, BX), d.nphi, ceil_div(d.nv, BY));
    // LDS-staged taps: FP32 volumes whose tap offsets stay exact in FP32
    // ((max(nx, ny) + 16) kSlotFloats < 2^24)
    if (x.staged && vol.dtype == TOMO_F32 && !x.index_reads && std::max(d.nx, d.ny) <= 4096) {
        StageSources src;
        hipError_t le = src.make((const float*)vol.p, d.nx, d.ny, d.nz, s);
        if (le == hipSuccess) {
            TOMO_DISPATCH_STORAGE(sino.dtype, TS, {
                hipLaunchKernelGGL((rs_staged_kernel<TS>), grid, dim3(BX, BY), 0, s, d, cube, (const float*)vol.p,
                                   (const float*)src.vt, src.rows_x, src.nxp, src.nyp, (TS*)sino.p, sino.scale);
            });
            le = hipGetLastError();
        }
        const hipError_t fe = src.release(s);
        TOMO_HIP(le);
        TOMO_HIP(fe);
        return TOMO_OK;
    }
    const float inv = 1.0f / vol.scale;
    const size_t es = vol.dtype == TOMO_F32 ? 4 : 2;
    const ProjPlanes zp = proj_planes(d, cube);
    const RsCopyShape cs = rs_copy_shape(d.nx, d.ny, zp.nz, es);
    ProjCopy pc;
    hipError_t le = pc.alloc(cs.elems * 8, s, x);
    if (le == hipSuccess) le = launch_rs_copy(vol.p, pc.p, es, d.nx, d.ny, d.nz, zp, s);
    if (le == hipSuccess) {
        const bool buf = cs.buf && !x.index_reads;
        const int rows = rs_wave_rows(d, zp);
        const dim3 cgrid(proj_groups(d.nu, rows), ceil_div(d.nphi, kProjViews), ceil_div(d.nv, rows));
        TOMO_DISPATCH_STORAGE(vol.dtype, TV, {
            TOMO_DISPATCH_STORAGE(sino.dtype, TS, {
                if (buf)
                    hipLaunchKernelGGL((rs_kernel<TV, TS, true>), cgrid, dim3(64 * kProjViews), 0, s, d, cube, pc.p,
                                       zp, inv, (TS*)sino.p, sino.scale, rows);
                else
                    hipLaunchKernelGGL((rs_kernel<TV, TS, false>), cgrid, dim3(64 * kProjViews), 0, s, d, cube, pc.p,
                                       zp, inv, (TS*)sino.p, sino.scale, rows);
            });
        });
        le = hipGetLastError();
    }
    const hipError_t fe = pc.release(s);
    TOMO_HIP(le);
    TOMO_HIP(fe);
    return TOMO_OK;
}

namespace {
std::atomic<int> g_rs_batch_grid{kBatchGrid};
}

int batch_grids_init(int device) {
    int per_cu = 0, cus = 0;
    TOMO_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, rs_batch_kernel, 64 * kProjViews, 0));
    TOMO_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device));
    int grid = per_cu * cus;
    grid -= grid % kBatchXcds;
    g_rs_batch_grid.store(std::min(std::max(grid, kBatchXcds), kBatchGrid));
    return TOMO_OK;
}

hipError_t launch_batch_rs(BatchTable* t, hipStream_t s) {
    hipLaunchKernelGGL(rs_batch_kernel, dim3(g_rs_batch_grid.load()), dim3(64 * kProjViews), 0, s, t, t->next);
    return hipGetLastError();
}

// The gather needs the squares around the voxel columns to be in front of the source
// in every view, and voxel and row coordinates that FP32 holds within 1e-3.  Thin
// problems, whose lanes along z would idle, scatter: the gather costs 60 ps per voxel
// column, view and line that may cross its square (in rounds of 64 views), and per
// line that does 20 and 43 per row that passes a voxel, 1.4 times that for 128 voxels in
// two halves and 2.9 for 256; on a narrow grid (ny < nx / 2), few columns idle the chip, one
// wave's lines, 0.1 us and 0.22 a row.  The scatter costs 262 ps a sample in the grid, 90
// ns per tap of one voxel, or 0.9 us and 0.35 a row (of up to 8) per sample of one ray.
// Scatter and gather in us, 256 x 256 and 256 views: one slice and row 2422 and 9121, 4
// and 4 12900 and 9150, 256 slices by 2 rows 9369 and 21496, by 8 35000 and 21700, one
// slice by 256 rows 2712 and 10667; 64 x 64 x 16, 2 rows and 64 views 179 and 225; 256 x
// 64 x 1, one row and 256 views 920 and 2670.
static bool rs_t_gathers(const DevGeom& d) {
    const double half = 0.5 * (double)std::max(d.nx, d.ny) + 1.0, fod = d.fod / (double)d.delta;
    if (0.5 * (double)d.nv * (double)d.dv > 50.0 * d.fdd) return false;  // at most 255 samples on a chord
    if (!(fod > 1.01 * std::sqrt(2.0) * half && d.nv <= 8192 && d.nz <= 8192 && fod <= 8192.0 &&
          (size_t)d.nu * d.nphi < (1ull << 31)))
        return false;
    const CrossingRows c(d);
    const double mag = (double)d.delta * d.fdd / d.fod, lines = mag / (double)d.du, rows = mag / (double)d.dv;
    const double blocks = d.nz <= 64 ? 1.0 : d.nz <= 128 ? 1.4 : 2.9 * ceil_div(d.nz, 256);
    const double all = d.nx * (double)d.ny * (60.0 * std::ceil(2.83 * lines) * 64.0 * ceil_div(d.nphi, 64) +
                                              2.42 * lines * (20.0 + 43.0 * (2.0 * rows + 1.0)) * blocks * d.nphi);
    const double one = 2 * d.ny < d.nx ? 2.55 * lines * (0.1 + 0.22 * (2.0 * rows + 1.0)) * d.nphi : 0.0;
    const double gather = 50.0 + std::max(1e-6 * all, one);
    const double step = std::max(262e-6, 0.72 / ((double)d.nx * d.ny * d.nz));
    const double row = step * crossing_columns(d, c) * d.nphi * std::min(d.nx, d.ny + 1), enough = (gather - 12.0) / row;
    return gather - 12.0 <= (0.9 + 0.35 * c.count(d, BY)) * d.nx || c.count(d, enough) >= enough;
}

template <int K, bool MIRROR>
static void launch_rs_t(const DevGeom& d, int cube, const float4* tab, int p0, int np, float* vol, hipStream_t s) {
    const dim3 grid = tile_grid((size_t)ceil_div(d.nx, kRsTWaves) * d.ny, 64 * kRsTWaves,
                                ceil_div(MIRROR ? (d.nz + 1) / 2 : d.nz, 64 * K));
    hipLaunchKernelGGL((rs_t_kernel<K, MIRROR>), grid, dim3(64 * kRsTWaves), 0, s, d, cube, tab, p0, np, p0 > 0, vol);
}

int launch_rs_adjoint(const tomo_geom* g, int cube, Buf sino, MutBuf vol, hipStream_t s) {
    if (vol.dtype != TOMO_F32) return fail(TOMO_ERR_UNSUPPORTED, "adjoint output must be F32");
    const DevGeom& d = g->dev;
    const float inv = 1.0f / sino.scale;
    // the rays' table, at most 1 GiB of views at a time; without the memory, or in a
    // stream capture, which is left free of allocations, the samples scatter
    const size_t view = (size_t)d.nu * rs_t_rows(d.nv) * sizeof(float4);
    const int chunk = (int)std::min<size_t>((size_t)d.nphi, std::max<size_t>(1, ((size_t)1 << 30) / view));
    float4* tab = nullptr;
    if (!stream_captures(s) && rs_t_gathers(d) &&
        hipMallocAsync((void**)&tab, view * (size_t)chunk, s) != hipSuccess) {
        (void)hipGetLastError();
        tab = nullptr;
    }
    if (tab) {
        hipError_t e = hipSuccess;
        for (int p0 = 0; p0 < d.nphi && e == hipSuccess; p0 += chunk) {
            const int np = std::min(chunk, d.nphi - p0);
            const size_t skip = (size_t)p0 * d.nu * d.nv;
            const unsigned tiles = ceil_div(d.nu, 8) * ceil_div(rs_t_rows(d.nv), 32) * (unsigned)np;
            TOMO_DISPATCH_STORAGE(sino.dtype, TS, {
                hipLaunchKernelGGL((rs_t_prepare_kernel<TS>), dim3(tiles), dim3(256), 0, s, d, cube,
                                   (const TS*)sino.p + skip, inv, p0, tab);
            });
            // one step of 64 voxels, or one or two of 64 and their mirror images (up to
            // 64 slices these would leave half of the lanes idle)
            if (d.nz <= 64)
                launch_rs_t<1, false>(d, cube, tab, p0, np, (float*)vol.p, s);
            else if (d.nz <= 128)
                launch_rs_t<1, true>(d, cube, tab, p0, np, (float*)vol.p, s);
            else
                launch_rs_t<2, true>(d, cube, tab, p0, np, (float*)vol.p, s);
            e = hipGetLastError();
        }
        const hipError_t f = hipFreeAsync(tab, s);
        TOMO_HIP(e);
        TOMO_HIP(f);
        return TOMO_OK;
    }
    int rc = launch_fill((float*)vol.p, 0.0f, g->nvox(), s);
    if (rc) return rc;
    dim3 grid(ceil_div(d.nu, BX), ceil_div(d.nv, BY), d.nphi);
    TOMO_DISPATCH_STORAGE(sino.dtype, TS, {
        hipLaunchKernelGGL((rs_adjoint_kernel<TS>), grid, dim3(BX, BY), 0, s, d, cube, (const TS*)sino.p, inv,
                           (float*)vol.p);
    });
    TOMO_HIP(hipGetLastError());
    return TOMO_OK;
}

int count_rs_samples(tomo_ctx* ctx, const tomo_geom* g, int cube, uint64_t* out, hipStream_t s) {
    const DevGeom& d = g->dev;
    unsigned long long* dt = nullptr;
    TOMO_HIP(hipMallocAsync((void**)&dt, sizeof(unsigned long long), s));
    TOMO_HIP(hipMemsetAsync(dt, 0, sizeof(unsigned long long), s));
    dim3 grid(ceil_div(d.nu, BX), ceil_div(d.nv, BY), d.nphi);
    hipLaunchKernelGGL(rs_count_kernel, grid, dim3(BX, BY), 0, s, d, cube, dt);
    TOMO_HIP(hipGetLastError());
    unsigned long long h = 0;
    TOMO_HIP(hipMemcpyAsync(&h, dt, sizeof(h), hipMemcpyDeviceToHost, s));
    TOMO_HIP(hipStreamSynchronize(s));
    TOMO_HIP(hipFreeAsync(dt, s));
    *out = h;
    (void)ctx;
    return TOMO_OK;
}

}  // namespace tomo
