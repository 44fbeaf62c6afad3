// kernels_vi.hip - voxel-driven bilinear backprojector (VI) and its exact
// transpose.
//
// Restates K/BackProjector/backprojection3D_kernel_16reg_UM.cuh:23-151 (the
// reference's device-resident VI kernel): for voxel (i,j,k), x'=i-cx,
// y'=j-cy, z'=k-cz and view p,
//   w = delta(cos x' + sin y') + FOD
//   u = (FDD/du) delta (-sin x' + cos y') / w + cu
//   v = A z' + cv,   A = (FDD/dv) delta / w
//   f = delta * sum_p bilinear(g_p, u, v)      (taps outside the detector = 0)
// The output is overwritten.  As in the reference's "16reg" blocking, a
// thread owns a column of voxels that share u and A (16, 8 or 4 of them, for FDK half
// of them at the mirrored heights); the per-(column,view)
// terms w, 1/w, u and A are evaluated in FP64 (the geometry of the FP32 form)
// and the per-voxel v, bilinear weights and sum in FP32.  A BF16 sinogram is
// widened to FP32 (value = stored / scale) before the same kernel; an FP16
// sinogram is read as u-pairs of FP16 taps (vi_pair_kernel) and interpolated
// with v_dot2_f32_f16 (FP16 u-weights in steps of 1/2048, FP32 sums).
#include <algorithm>
#include <climits>
#include <cmath>
#include <type_traits>

#include "device_common.hpp"
#include "fdk_weight.hpp"
#include "batch.hpp"

namespace tomo {
namespace {

constexpr int TX = kViTileX, TY = kViTileY, ZB = kViTileZ;  // VI^T workgroup

struct ColumnView {
    float u, A;
    float num, base;  // FDK weight terms (FDK only)
};

// 1 / w: the hardware's reciprocal (2^-24) and two Newton steps, correctly
// rounded but for a few mantissas next to 2, which come out an ulp off (of
// 1.1e10 values none other); half the instructions of the division.  w = 0 gives
// NaN where the division gives an infinity: a column-view that is dropped either way.
__device__ __forceinline__ double recip64(double w) {
    double r = __builtin_amdgcn_rcp(w);
    r = fma(fma(-w, r, 1.0), r, r);
    return fma(fma(-w, r, 1.0), r, r);
}

// Per (column, view) terms in FP64.  FDK (back_fdk,
// K/BackProjector/FDK3D_kernel_16reg.cuh:71-88; constants C/BackProjector.cu:
// 34-35) adds num = alphaC (FDD/du) / w^2 and base = betaC + u'^2, u' = u - cu
// in pixels, alphaC = (float)(pi FOD FDD / Nphi), betaC = (FDD/du)^2.  A
// column-view with a non-finite u or A contributes 0: it reads off the
// detector (u = -8, A = 0) with a zero weight.
template <bool FDK>
__device__ __forceinline__ ColumnView column_view(const DevGeom& g, const double* c, double xp, double yp) {
    const double w = fma(c[2], xp, fma(c[3], yp, g.fod));
    const double inv = recip64(w);
    const double un = fma(c[4], xp, c[5] * yp);
    ColumnView r;
    r.u = (float)fma(un, inv, (double)g.cu);
    r.A = (float)(c[6] * inv);
    r.num = 0.0f;
    r.base = 1.0f;
    const bool fin = __builtin_isfinite(r.u) && __builtin_isfinite(r.A);
    if (FDK && fin) {
        const double ku = g.fdd / (double)g.du;
        const double alpha_c = (double)(float)(M_PI * g.fod * g.fdd / (double)g.nphi);
        const double up = un * inv;
        // alphaC ku / w^2: a Newton step on 1 / w^2 and a residual step, correctly
        // rounded for each of 1.1e10 random pairs
        const double w2 = w * w, a = alpha_c * ku;
        double i2 = inv * inv;
        i2 = fma(fma(-w2, i2, 1.0), i2, i2);
        const double n = a * i2;
        r.num = (float)fma(fma(-w2, n, a), i2, n);
        r.base = (float)(ku * ku + up * up);
    }
    if (!fin) {
        r.u = -8.0f;
        r.A = 0.0f;
    }
    return r;
}

// ---------------------------------------------------------------------------
// LDS-staged VI for FP32 sinograms.
//
// A workgroup owns SX x SY voxel columns of ZS voxels.  For each view it
// copies the detector taps its voxels read into LDS with coalesced loads
// (taps off the detector as 0), and each voxel-view update reads its four
// taps from there with two ds_read2_b32.  The taps are the box of
// rows [v0, v1 + 1] and columns [u0, u1 + 1] with (u0, u1) the extreme
// clamped cell corners floor(u) of the tile's columns and (v0, v1) the
// extreme floor(v) of its voxels.  A table holds, per (column tile, view),
// u0, u1 and the extreme A of the tile's columns (vi_box_kernel, the same
// FP64 column terms); since v = fmaf(z', A, cv) is monotone in z' and in A,
// the row extremes are the floors at the four (z', A) corners, so the box is
// exact.  A row off the detector holds zeros in the box.  Groups of 1, 2 or 4
// views (ZS 16, 8, 4) alternate between two buffers, so one barrier per group
// separates the copies from the reads.  A group with a box that exceeds its
// buffer reads the taps directly.
//
// Per wave and view, 16 voxels are about 500 VALU cycles of a SIMD, the FP64
// column terms 120 and the copies and plans 40; the LDS reads are 128 cycles of
// the CU, 85% of the time at 512^3 and 512 views, where that binds (and the
// clock falls to 2.05 GHz): 22.0 -> 19.8 ms (20.3 on another card) with the plans made by lane, the
// direct views in a loop of their own, 16-byte copies and the short reciprocal.
// FDK (256^3, 360 views) is bound by VALU: 5.93 -> 3.2 ms (3.5 on another card), most of it from
// fdk_weight and its sharing between mirrored voxels.
constexpr int SX = kViStageX, SY = kViStageY;  // voxel columns per workgroup; a wave is 8 x 8 columns
// Floats per staged row.  A wave's 64 lanes read taps (u, r) at word
// r * pitch + u; lanes spread over about 20 columns and a few rows, so two
// lanes share a bank when their row and column offsets satisfy
// dr * pitch + du = 0 mod 32.  With 8 x 8 waves a pitch of 76 (12 mod 32, and
// whole 16-byte pieces) keeps such pairs rare at 512^3 / 512 views, 2% of the
// LDS cycles; with 32 x 2 waves (40 columns, past the 32 banks) and a pitch of
// 65 (1 mod 32) a ds_read2_b32 took 2.6 extra cycles on bank conflicts.
constexpr int kStagePitch = 76;

// Staging buffers of a workgroup of ZS-voxel columns: `rows` rows of 64 taps for
// each of `views` views, twice, in whole pieces of 256 words (one 16-byte load
// per lane).  16: up to 37 rows (at 512^3 / 512 views about 0.1% of the boxes
// need more and read their taps directly), 22.5 KB of LDS, 7 workgroups per CU.
// Shorter columns stage several views between two barriers: there are few waves
// then to wait for the taps, and the boxes are small.
// 4: 20 rows, what six pieces hold; with 16, 2% of the groups at 64^3 read directly, and
// the slowest workgroup two of twelve (64^3 and 48 views 30.0 us, 27.2 with 20).
// MIRROR: a column is two halves at opposite heights, each with a box of its own.
template <int ZS, bool MIRROR = false>
struct StageShape {
    static_assert(ZS == 16 || ZS == 8 || ZS == 4, "staging buffers sized for 16, 8 and 4 voxels");
    static_assert(SX == 32 && SY == 8, "four 8 x 8 waves per workgroup");
    static_assert(!MIRROR || ZS >= 8, "halves of 8 and 4 voxels");
    static constexpr int boxes = MIRROR ? 2 : 1;                        // per view
    static constexpr int height = ZS / boxes;                           // voxels of a box
    static constexpr int rows = MIRROR ? (ZS == 16 ? 20 : 16) : ZS == 16 ? 37 : ZS == 8 ? 26 : 20;  // rows of a box
    static constexpr int views = ZS == 16 ? 1 : ZS == 8 ? 2 : 4;        // views between two barriers
    static constexpr int pieces = (rows * kStagePitch + 255) / 256;     // of a box
    static constexpr int taps = pieces * 256;                           // floats per box
    static constexpr int words = 2 * views * boxes * taps;
};

__device__ __forceinline__ int wave_min(int v) { return __reduce_min_sync(~0ull, v); }
__device__ __forceinline__ int wave_max(int v) { return __reduce_max_sync(~0ull, v); }

// Order-preserving map of a finite float to int: x < y  <=>  key(x) < key(y).
__device__ __forceinline__ int fkey(float v) {
    const int b = __float_as_int(v);
    return b >= 0 ? b : (int)(0x80000000u - (uint32_t)b);
}
__device__ __forceinline__ float fkey_inv(int k) {
    return __int_as_float(k >= 0 ? k : (int)(0x80000000u - (uint32_t)k));
}

// The ViBox of column tile `tile` (row-major over ntx tiles per row) in view
// p, one workgroup of SX x SY threads (one per column).
__device__ __forceinline__ void vi_box_tile(const DevGeom& g, ViBox* __restrict__ box, int ntx, uint32_t tile,
                                            uint32_t p) {
    const int i = (int)(tile % ntx) * SX + (int)(threadIdx.x % SX);
    const int j = (int)(tile / ntx) * SY + (int)(threadIdx.x / SX);
    int k[4] = {INT_MAX, INT_MIN, INT_MAX, INT_MIN};
    if (i < g.nx && j < g.ny) {
        const double xp = (double)i - (double)g.cx, yp = (double)j - (double)g.cy;
        const ColumnView cvw = column_view<false>(g, g.view + (size_t)p * kViewStride, xp, yp);
        const int uc = (int)__builtin_amdgcn_fmed3f(floorf(cvw.u), -2.0f, (float)g.nu);
        k[0] = k[1] = uc;
        k[2] = k[3] = fkey(cvw.A);
    }
    __shared__ int part[SX * SY / 64][4];
    const int w = threadIdx.x >> 6;
    const int r0 = wave_min(k[0]), r1 = wave_max(k[1]), r2 = wave_min(k[2]), r3 = wave_max(k[3]);
    __syncthreads();  // the previous tile's reads of part are done
    if ((threadIdx.x & 63) == 0) {
        part[w][0] = r0;
        part[w][1] = r1;
        part[w][2] = r2;
        part[w][3] = r3;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        int m[4] = {part[0][0], part[0][1], part[0][2], part[0][3]};
        for (int q = 1; q < SX * SY / 64; ++q) {
            m[0] = min(m[0], part[q][0]);
            m[1] = max(m[1], part[q][1]);
            m[2] = min(m[2], part[q][2]);
            m[3] = max(m[3], part[q][3]);
        }
        ViBox b;
        b.u0 = m[0];
        b.u1 = m[1];
        b.amin = fkey_inv(m[2]);
        b.amax = fkey_inv(m[3]);
        box[(size_t)tile * g.nphi + p] = b;
    }
}

// One workgroup per (column tile, view).
__global__ __launch_bounds__(SX* SY) void vi_box_kernel(DevGeom g, ViBox* __restrict__ box, int ntx) {
    const uint32_t b = tile_index(), tile = b / (uint32_t)g.nphi;
    if (tile < (uint32_t)ntx * (uint32_t)((g.ny + SY - 1) / SY)) vi_box_tile(g, box, ntx, tile, b % (uint32_t)g.nphi);
}

// Per-view staging plan of a workgroup: the box of taps (rows from v0,
// columns from u0), no rows where it does not fit the buffer.  Boxes at the detector's
// ends are copied one column per lane, so a box is at most 64 columns wide.
// Each lane makes the plan of one of 64 views, which the wave then reads lane by
// lane: made by every lane for every view it was an eighth of the instructions.
struct StagePlan {
    int u0, v0, rows;
    bool quads;  // 16-byte loads: no tap of the box is off the detector's left or right end
    bool near;   // 32-bit offsets in the view of the box's rows off the detector do not come round to it
};

// The box rows from the four (z', A) corners; v0 and the number of rows as v0 * 256
// + rows and the flags, 0 where the box does not fit.
template <typename SS>
__device__ __forceinline__ int stage_rows(const ViBox& bb, float zp0, float cv, int rl, int nv) {
    const float zp1 = zp0 + (float)(SS::height - 1);
    const float va = fmaf(zp0, bb.amin, cv), vb = fmaf(zp0, bb.amax, cv);
    const float vc = fmaf(zp1, bb.amin, cv), vd = fmaf(zp1, bb.amax, cv);
    const float vlo = floorf(fminf(fminf(va, vb), fminf(vc, vd)));
    const float vhi = floorf(fmaxf(fmaxf(va, vb), fmaxf(vc, vd)));
    const bool fits = vlo >= -32768.0f && vhi <= 32768.0f && vhi - vlo + 2.0f <= (float)SS::rows &&
                      bb.u1 - bb.u0 + 2 <= 64;
    static_assert(SS::rows < 64, "rows below the flags");
    const bool near = (int)vlo >= -64 && (int)vlo <= nv && (uint64_t)(nv + 128) * (uint32_t)rl < (1u << 29);
    // a lane's four taps start at a tap of the box and end on its row
    const bool quads = near && bb.u0 >= 0 && bb.u1 + 1 + 3 < rl;
    return fits ? (int)vlo * 256 + (quads ? 128 : 0) + (near ? 64 : 0) + (int)(vhi - vlo) + 2 : 0;
}

// FP16 u-weights (1 - w, w) of a column-view, w = fu rounded to a multiple of
// 1/2048: both are exact FP16 values and sum to 1, so a constant row
// interpolates to itself.
__device__ __forceinline__ uint32_t pair_weights(float fu) {
    typedef _Float16 h2 __attribute__((ext_vector_type(2)));
    const float w1 = rintf(fu * 2048.0f) * (1.0f / 2048.0f);
    return __builtin_bit_cast(uint32_t, h2{(_Float16)(1.0f - w1), (_Float16)w1});
}

// Bilinear sample from two u-pair words (rows v and v + 1): r0 = w . P0 and
// the row difference w . P1 - r0, each one v_dot2_f32_f16 (products of FP16
// values are exact in FP32), then r0 + fv (r1 - r0).  The builtins leave the
// wait states a dot2 result needs before its use to the compiler.
__device__ __forceinline__ float pair_sample(uint32_t p0, uint32_t p1, uint32_t w, float fv) {
    typedef _Float16 h2 __attribute__((ext_vector_type(2)));
    const h2 hw = __builtin_bit_cast(h2, w);
    const float r0 = __builtin_amdgcn_fdot2(__builtin_bit_cast(h2, p0), hw, 0.0f, false);
    const float dr = __builtin_amdgcn_fdot2(__builtin_bit_cast(h2, p1), hw, -r0, false);
    return fmaf(fv, dr, r0);
}

// Four bilinear samples at once (the staged path's inner loop): the four
// r0 = w . P0 first, then the four w . P1 - r0, so each dot2 result is read
// three or more instructions after it is written (the wait a VALU read of a
// dot2 result needs), and s_nop 2 before any later read of the last one.
__device__ __forceinline__ void pair_sample4(const uint32_t (&p0)[4], const uint32_t (&p1)[4], uint32_t w,
                                             float (&r0)[4], float (&dr)[4]) {
    asm volatile(
        "v_dot2_f32_f16 %0, %8, %16, 0\n\t"
        "v_dot2_f32_f16 %1, %9, %16, 0\n\t"
        "v_dot2_f32_f16 %2, %10, %16, 0\n\t"
        "v_dot2_f32_f16 %3, %11, %16, 0\n\t"
        "v_dot2_f32_f16 %4, %12, %16, %0 neg_lo:[0,0,1]\n\t"
        "v_dot2_f32_f16 %5, %13, %16, %1 neg_lo:[0,0,1]\n\t"
        "v_dot2_f32_f16 %6, %14, %16, %2 neg_lo:[0,0,1]\n\t"
        "v_dot2_f32_f16 %7, %15, %16, %3 neg_lo:[0,0,1]\n\t"
        "s_nop 2"
        : "=&v"(r0[0]), "=&v"(r0[1]), "=&v"(r0[2]), "=&v"(r0[3]), "=&v"(dr[0]), "=&v"(dr[1]), "=&v"(dr[2]),
          "=&v"(dr[3])
        : "v"(p0[0]), "v"(p0[1]), "v"(p0[2]), "v"(p0[3]), "v"(p1[0]), "v"(p1[1]), "v"(p1[2]), "v"(p1[3]), "v"(w));
}

// PAIR: `sino` holds u-pair words (vi_pair_kernel; nu + 1 per row) instead of
// FP32 taps; the box copy and the tap offsets are the same, one word per row.
// FDK: 0 VI, 1 FDK, 2 FDK whose weights are within fdk_weight's bounds, 3 the same
// on mirrored columns: the weight depends on z'^2, so a voxel at z' and the one at
// -z' share it.  A column is then ZS / 2 voxels from k0 = bz ZS / 2 on and their
// mirror images nz - 1 - k.  256^3 and 360 views: 3.95 ms without, 3.25 with, on one card.
template <typename TV, int FDK, int ZS, bool PAIR = false>
__device__ __forceinline__ void vi_staged_tile(const DevGeom& g, const float* __restrict__ sino,
                                               const ViBox* __restrict__ boxes, TV* __restrict__ vol,
                                               float vol_scale, float post, int bx, int by, int bz,
                                               float* __restrict__ stage) {
    constexpr bool MIRROR = FDK == 3;
    using SS = StageShape<ZS, MIRROR>;
    constexpr int H = SS::height, B = SS::boxes;
    constexpr int NT = SX * SY;
    constexpr int NW = NT / 64;                             // waves per workgroup
    // Waves that copy a box together.  A copy's branches and resources cost each of
    // them the same, so the boxes of short columns, whose waves are alone or two on a
    // SIMD, are dealt out to the waves; all four on each box: 64^3 and 180 views 97 us,
    // dealt out 87; 40^3 and 48 views 28.4 and 25.1; 80^3 and 64 views 43 and 38; at 8
    // voxels 96^3 and 96 views 75 and 73, 128^3 and 180 views 189 and 185.  At 16 the
    // copies are spread over more waves: 512^3 19.8 ms, FDK 256^3 dealt out 1% slower.
    constexpr int CW = ZS == 16 ? NW : NW / (SS::views * B);
    static_assert(CW == NW || CW * SS::views * B == NW, "a wave copies for one box");
    constexpr int kSlots = (SS::rows + CW - 1) / CW;        // box rows per wave at most
    const int tid = threadIdx.x;
    const int lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int cw = wv % CW;
    // wave wv covers columns x in [8 wv, 8 wv + 8), y in [0, 8)
    const int i = bx * SX + wv * 8 + (lane & 7);
    const int j = by * SY + (lane >> 3);
    const int k0 = bz * H;
    // a lane past the volume's edge works on the edge column, and stores nothing
    const double xp = (double)min(i, g.nx - 1) - (double)g.cx, yp = (double)min(j, g.ny - 1) - (double)g.cy;
    const float zp0 = (float)((double)k0 - (double)g.cz);
    const float cv = g.cv;
    const float fnu = (float)g.nu;
    const int nu = g.nu, nv = g.nv;
    const int rl = PAIR ? nu + 1 : nu;  // words per detector row
    const size_t plane = (size_t)rl * nv;
    // The view table is read-only here and indexed by wave-uniform values: read
    // through the constant address space it comes in with scalar loads.
    typedef const __attribute__((address_space(4))) double* ConstView;
    const ViBox* const bt = boxes + (size_t)(by * ((g.nx + SX - 1) / SX) + bx) * g.nphi;
    float acc[ZS];
#pragma unroll
    for (int k = 0; k < ZS; ++k) acc[k] = 0.0f;
    // z' of voxel k; the second half is the first's mirror image, exactly (cz is (nz - 1) / 2)
    auto height = [&](int k) { return k < H ? zp0 + (float)k : -(zp0 + (float)(k - H)); };
    auto weight = [&](const ColumnView& cvw, int k) {
        const float vp = height(k) * cvw.A, q = fmaf(vp, vp, cvw.base);
        return FDK >= 2 ? fdk_weight(cvw.num, q) : cvw.num / sqrtf(q);
    };
    auto add = [&](float wt, int k, float r) { acc[k] += FDK ? wt * r : r; };
    auto bilinear = [&](float fu, float v, float vf, float t00, float t01, float t10, float t11) {
        // t00 = (u, v), t01 = (u, v+1), t10 = (u+1, v), t11 = (u+1, v+1)
        const float fv = v - vf;
        const float a = fmaf(fu, t10 - t00, t00);
        const float b = fmaf(fu, t11 - t01, t01);
        return fmaf(fv, b - a, a);
    };
    const uint32_t view_bytes = (uint32_t)(plane * sizeof(float));
    // Byte offset in the view of a lane's four taps of the wave's q-th piece, from
    // the box's first: word w of the buffer is tap (w / pitch, w mod pitch).
    constexpr int kPieces = (SS::pieces + CW - 1) / CW;
    uint32_t piece[kPieces];
#pragma unroll
    for (int q = 0; q < kPieces; ++q) {
        const int w = 256 * (cw + q * CW) + 4 * lane, row = w / kStagePitch;
        piece[q] = (uint32_t)(row * rl + (w - row * kStagePitch)) * 4u;
    }
    // Copy of a box of view p into buffer b, straight from memory into LDS
    // (buffer_load ... lds); a tap off the detector's upper or lower edge is
    // outside the view's bytes, which writes 0.  Words past the box hold taps
    // that nothing reads.  One 16-byte load per lane brings 3.4 rows; by rows, a
    // 4-byte load each, the copies kept the data return 80% busy at 512^3.
    //
    // Boxes at the detector's left and right ends go by rows: wave cw copies box
    // rows cw + q CW, lane l column l; lanes off the detector read past the view's
    // bytes.  Far from the detector, or on one past 2^29 taps, each row is read
    // through a buffer resource of that detector row (of no bytes for a row off the
    // detector), which takes some 20 instructions a row instead of 5: 64^3 and 180
    // views 90 us, 85 through the view's; 128^3 and 180 views 185 and 182.
    auto copy_box = [&](const StagePlan& s, int p, int b) {
        const float* view = sino + (size_t)p * plane;
        float* dst = stage + b * SS::taps;
        if (s.quads) {
            const __amdgpu_buffer_rsrc_t rr = buffer_rsrc(view, view_bytes);
            const uint32_t at = (uint32_t)(s.v0 * rl + s.u0) * 4u;
            const int words = s.rows * kStagePitch;
#pragma unroll
            for (int q = 0; q < kPieces; ++q)
                if (256 * (cw + q * CW) < words)
                    __builtin_amdgcn_raw_ptr_buffer_load_lds(
                        rr, (__attribute__((address_space(3))) void*)(dst + 256 * (cw + q * CW)), 16,
                        (int)(at + piece[q]), 0, 0, 0);
            return;
        }
        if (s.near) {
            // a lane off the detector's columns starts 2^31 bytes on, past the view's end
            const int u = s.u0 + lane;
            uint32_t off = (unsigned)u < (unsigned)rl ? (uint32_t)(s.v0 * rl + u) * 4u : 0x80000000u;
            off += (uint32_t)(cw * rl) * 4u;
            const __amdgpu_buffer_rsrc_t rr = buffer_rsrc(view, view_bytes);
#pragma unroll
            for (int q = 0; q < kSlots; ++q) {
                if (cw + q * CW < s.rows)
                    __builtin_amdgcn_raw_ptr_buffer_load_lds(
                        rr, (__attribute__((address_space(3))) void*)(dst + (cw + q * CW) * kStagePitch), 4, off, 0, 0, 0);
                off += (uint32_t)(CW * rl) * 4u;
            }
            return;
        }
        // past the row's end unless 0 <= u < nu (FP32) or the pair index u + 1 <= nu
        const uint32_t loff = (uint32_t)(s.u0 + lane) * 4u;
#pragma clang loop unroll(disable)
        for (int q = 0; q < kSlots; ++q) {
            if (cw + q * CW < s.rows) {
                const int v = s.v0 + cw + q * CW;
                const bool vin = (unsigned)v < (unsigned)nv;
                const __amdgpu_buffer_rsrc_t rr =
                    buffer_rsrc(view + (size_t)(vin ? v : 0) * rl, vin ? (uint32_t)rl * 4u : 0u);
                __builtin_amdgcn_raw_ptr_buffer_load_lds(
                    rr, (__attribute__((address_space(3))) void*)(dst + (cw + q * CW) * kStagePitch), 4, loff, 0, 0, 0);
            }
        }
    };
    int plan_u0[B] = {}, plan_v[B] = {};  // of view (p & ~63) + lane
    auto plan_of = [&](int p, int b) {
        const int v = __builtin_amdgcn_readlane(plan_v[b], p & 63);
        return StagePlan{__builtin_amdgcn_readlane(plan_u0[b], p & 63), v >> 8, v & 63, (v & 128) != 0, (v & 64) != 0};
    };
    // Plans and copies of the group of G views from p on; rows is 0 if one of its
    // boxes does not fit, and all of the group's taps are then read directly.
    constexpr int G = SS::views;
    struct Group {
        int u0[G][B], v0[G][B], rows;
    };
    auto stage_group = [&](int p, int half) {
        Group r;
        r.rows = 1;
        if ((p & 63) == 0 && p + lane < g.nphi) {  // G divides 64
            ViBox bb = bt[p + lane];
            bb.u0 += PAIR;  // word index of tap pair (u, u + 1)
            bb.u1 += PAIR;
#pragma unroll
            for (int b = 0; b < B; ++b) {
                plan_v[b] = stage_rows<SS>(bb, b ? -(zp0 + (float)(H - 1)) : zp0, cv, rl, nv);
                plan_u0[b] = (plan_v[b] & 128) ? bb.u0 & ~3 : bb.u0;  // rows of a multiple of 4 taps: aligned loads
            }
        }
#pragma unroll
        for (int t = 0; t < G; ++t)
#pragma unroll
            for (int b = 0; b < B; ++b) {
                const StagePlan s = p + t < g.nphi ? plan_of(p + t, b) : StagePlan{0, 0, 0, false, false};
                r.u0[t][b] = s.u0;
                r.v0[t][b] = s.v0;
                if (p + t < g.nphi) {
                    if (s.rows == 0) r.rows = 0;
                    if (CW == NW) copy_box(s, p + t, (half * G + t) * B + b);
                }
            }
        if (CW < NW) {
            const int box = wv / CW, t = box / B;
            if (p + t < g.nphi) copy_box(box % B ? plan_of(p + t, B - 1) : plan_of(p + t, 0), p + t, half * G * B + box);
        }
        return r;
    };
    auto view_terms = [&](int p) {
        const ConstView vt = (ConstView)(g.view + (size_t)p * kViewStride);
        double c[kViewStride];
#pragma unroll
        for (int e = 0; e < kViewStride; ++e) c[e] = vt[e];
        return column_view<FDK != 0>(g, c, xp, yp);
    };
    Group now, nxt = stage_group(0, 0);
    int p = 0, half = 0;
    // the copies of the group at p have landed (this wave's, then all); every wave is done with the group before
    auto next_group = [&]() {
        __builtin_amdgcn_s_waitcnt(0);
        __syncthreads();
        now = nxt;
        if (p + G < g.nphi) nxt = stage_group(p + G, half ^ 1);
    };
    do {
        // The staged views in a loop of their own: as one branch of two in it, the
        // sums changed registers for every view (16 moves, 6% of the instructions).
        while (p < g.nphi && nxt.rows > 0) {
            next_group();
#pragma unroll
            for (int t = 0; t < G; ++t) {
                if (t > 0 && p + t >= g.nphi) break;
                const ColumnView cvw = view_terms(p + t);
                const float uf = floorf(cvw.u);
                const float fu = cvw.u - uf;
                const float uc = __builtin_amdgcn_fmed3f(uf, -2.0f, fnu);
                // byte offset in the buffer of tap (uc, vf): ((vf - v0) pitch + uc - u0) 4,
                // one exact fma of small integers on top of 2^23, whose low bits are then the
                // offset: an and (0.6 cycles per wave and CU) for a conversion (1.1)
                float colb[B];
#pragma unroll
                for (int b = 0; b < B; ++b)
                    colb[b] = (float)(((int)uc + PAIR - now.u0[t][b] - now.v0[t][b] * kStagePitch +
                                       ((half * G + t) * B + b) * SS::taps) * 4) + 0x1p23f;
                auto taps = [&](float vf, int b) {
                    const uint32_t off = __float_as_uint(fmaf(vf, (float)(kStagePitch * 4), colb[b])) & 0x7fffffu;
                    return (const char*)stage + off;
                };
                if constexpr (PAIR) {
                    static_assert(H % 4 == 0, "u-pair samples go four voxels at a time");
                    const uint32_t pw = pair_weights(fu);
#pragma unroll
                    for (int k4 = 0; k4 < H; k4 += 4) {
                        float wt[4];
#pragma unroll
                        for (int e = 0; e < 4; ++e) wt[e] = FDK ? weight(cvw, k4 + e) : 1.0f;
#pragma unroll
                        for (int b = 0; b < B; ++b) {
                            uint32_t p0[4], p1[4];
                            float fv[4], r0[4], dr[4];
#pragma unroll
                            for (int e = 0; e < 4; ++e) {
                                const float v = fmaf(height(b * H + k4 + e), cvw.A, cv);
                                const float vf = floorf(v);
                                const uint32_t* qw = (const uint32_t*)taps(vf, b);
                                p0[e] = qw[0];
                                p1[e] = qw[kStagePitch];
                                fv[e] = v - vf;
                            }
                            pair_sample4(p0, p1, pw, r0, dr);
#pragma unroll
                            for (int e = 0; e < 4; ++e) add(wt[e], b * H + k4 + e, fmaf(fv[e], dr[e], r0[e]));
                        }
                    }
                } else {
#pragma unroll
                    for (int k = 0; k < H; ++k) {
                        const float wt = FDK ? weight(cvw, k) : 1.0f;
#pragma unroll
                        for (int b = 0; b < B; ++b) {
                            const float v = fmaf(height(b * H + k), cvw.A, cv);
                            const float vf = floorf(v);
                            const float* q = (const float*)taps(vf, b);
                            add(wt, b * H + k, bilinear(fu, v, vf, q[0], q[kStagePitch], q[1], q[kStagePitch + 1]));
                        }
                    }
                }
            }
            p += G;
            half ^= 1;
        }
        if (p >= g.nphi) break;
        // a box larger than the buffer: the four taps straight from the views, one voxel at a time
        next_group();
#pragma clang loop unroll(disable)
        for (int pd = p; pd < min(p + G, g.nphi); ++pd) {
            const ColumnView cvw = view_terms(pd);
            const float uf = floorf(cvw.u);
            const float fu = cvw.u - uf;
            const float uc = __builtin_amdgcn_fmed3f(uf, -2.0f, fnu);
            const uint32_t pw = PAIR ? pair_weights(fu) : 0u;
            const __amdgpu_buffer_rsrc_t rsrc = buffer_rsrc(sino + (size_t)pd * plane, view_bytes);
            const int iu = (int)uc;
            const bool u0ok = (unsigned)iu < (unsigned)nu, u1ok = (unsigned)(iu + 1) < (unsigned)nu;
            const bool pok = (unsigned)(iu + 1) <= (unsigned)nu;  // pair word iu + 1 exists
            auto rd = [&](bool ok, int v, int u) {
                const uint32_t off = ok ? (uint32_t)(v * rl + u) * 4u : 0xfffffff0u;
                return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rsrc, (int)off, 0, 0));
            };
#pragma unroll
            for (int k = 0; k < ZS; ++k) {
                const float v = fmaf(height(k), cvw.A, cv), wt = FDK ? weight(cvw, k) : 1.0f;
                const float vf = floorf(v);
                const int iv = (int)__builtin_amdgcn_fmed3f(vf, -2.0f, (float)nv);
                const bool v0ok = (unsigned)iv < (unsigned)nv, v1ok = (unsigned)(iv + 1) < (unsigned)nv;
                if constexpr (PAIR) {
                    const uint32_t p0 = __builtin_bit_cast(uint32_t, rd(pok && v0ok, iv, iu + 1));
                    const uint32_t p1 = __builtin_bit_cast(uint32_t, rd(pok && v1ok, iv + 1, iu + 1));
                    add(wt, k, pair_sample(p0, p1, pw, v - vf));
                } else {
                    add(wt, k, bilinear(fu, v, vf, rd(u0ok && v0ok, iv, iu), rd(u0ok && v1ok, iv + 1, iu),
                                        rd(u1ok && v0ok, iv, iu + 1), rd(u1ok && v1ok, iv + 1, iu + 1)));
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        p += G;
        half ^= 1;
    } while (p < g.nphi);
    if (i >= g.nx || j >= g.ny) return;
    const size_t sxy = (size_t)g.nx * g.ny;
    const size_t base = (size_t)i + (size_t)g.nx * j;
#pragma unroll
    for (int k = 0; k < ZS; ++k) {
        // mirrored: the middle slice of an odd volume belongs to the first half
        const int zk = k < H ? k0 + k : g.nz - 1 - (k0 + k - H);
        if (MIRROR ? (k < H ? 2 * zk < g.nz : 2 * zk >= g.nz) : zk < g.nz)
            Storage<TV>::store(vol, base + (size_t)zk * sxy, FDK ? acc[k] * post : (acc[k] * g.delta) * post, vol_scale);
    }
}

// Waves per SIMD that a kernel's registers are held to.
constexpr int vi_waves(int fdk, int zs, bool pair) { return fdk == 3 ? 6 : !pair ? 7 : fdk == 1 ? 5 : 6; }

// post: 1 for FP32 taps, 1 / storage scale for FP16 u-pairs.
template <typename TV, int FDK, int ZS, bool PAIR>
__global__ __launch_bounds__(SX* SY, vi_waves(FDK, ZS, PAIR)) void vi_staged_kernel(DevGeom g, const float* __restrict__ sino,
                                                         const ViBox* __restrict__ boxes, TV* __restrict__ vol,
                                                         float vol_scale, float post) {
    __shared__ __align__(16) float stage[StageShape<ZS, FDK == 3>::words];
    vi_staged_tile<TV, FDK, ZS, PAIR>(g, sino, boxes, vol, vol_scale, post, blockIdx.x, blockIdx.y, blockIdx.z,
                                      stage);
}

// u-pair words of an FP16 sinogram, one workgroup per detector row: word j in
// [0, nu] of the row holds taps (j - 1, j) as its low and high halves, a tap
// off the row as 0.
__global__ __launch_bounds__(256) void vi_pair_kernel(const uint16_t* __restrict__ sino,
                                                      uint32_t* __restrict__ pairs, int nu, uint32_t rows) {
    const size_t row = tile_index();
    if (row >= rows) return;
    const uint16_t* src = sino + row * (size_t)nu;
    uint32_t* dst = pairs + row * (size_t)(nu + 1);
    for (int j = threadIdx.x; j <= nu; j += blockDim.x) {
        const uint32_t lo = j >= 1 ? src[j - 1] : 0u;
        const uint32_t hi = j < nu ? src[j] : 0u;
        dst[j] = lo | (hi << 16);
    }
}

// Shared launch (FP32 sinograms and volumes): tile grid (ceil(nx/SX),
// ceil(ny/SY), ceil(nz/16)) on the sinogram `in` with the problem's box table
// `aux` (launch_vi_boxes); the stored value is (delta * sum) * a.
__global__ __launch_bounds__(SX* SY, 7) void vi_batch_kernel(const BatchTable* __restrict__ t, uint32_t* __restrict__ next) {
    __shared__ __align__(16) float stage[StageShape<kViTileZ>::words];
    TOMO_BATCH_CLAIMED(t, next) {
        const BatchItem& it = t->item[batch_find(t, tile)];
        const uint32_t local = tile - it.begin;
        const uint32_t bx = local % it.gx, rest = local / it.gx;
        const int by = (int)(rest % it.gy), bz = (int)(rest / it.gy);
        vi_staged_tile<float, 0, kViTileZ>(it.g, (const float*)it.in, (const ViBox*)it.aux, (float*)it.out, 1.0f,
                                               it.a, (int)bx, by, bz, stage);
    }
}

// VI^T: g_p[tap] += delta * w_tap * f(i,j,k) (FP32 atomics, output zeroed by
// the caller).  The geometry is the backprojector's (column_view), the weights its
// products.
template <typename TV>
__global__ __launch_bounds__(TX* TY) void vi_adjoint_kernel(DevGeom g, const TV* __restrict__ vol, float vol_inv,
                                                          float* __restrict__ sino) {
    const int i = blockIdx.x * TX + (threadIdx.x % TX);
    const int j = blockIdx.y * TY + (threadIdx.x / TX);
    const int k0 = blockIdx.z * ZB;
    if (i >= g.nx || j >= g.ny) return;
    const double xp = (double)i - (double)g.cx, yp = (double)j - (double)g.cy;
    const float zp0 = (float)((double)k0 - (double)g.cz);
    const size_t sxy = (size_t)g.nx * g.ny;
    const size_t base = (size_t)i + (size_t)g.nx * j;
    float fv[ZB];
#pragma unroll
    for (int k = 0; k < ZB; ++k)
        fv[k] = (k0 + k < g.nz) ? Storage<TV>::load(vol, base + (size_t)(k0 + k) * sxy, vol_inv) * g.delta : 0.0f;
    const size_t plane = (size_t)g.nu * g.nv;
    const int nu = g.nu, nv = g.nv;
    for (int p = 0; p < g.nphi; ++p) {
        const ColumnView cvw = column_view<false>(g, g.view + (size_t)p * kViewStride, xp, yp);
        float* gp = sino + (size_t)p * plane;
        const float uf = floorf(cvw.u);
        if (!(uf >= -1.0f && uf <= (float)nu)) continue;
        const int iu = (int)uf;
        const float fu = cvw.u - uf;
        const bool u0 = iu >= 0 && iu < nu, u1 = iu + 1 >= 0 && iu + 1 < nu;
        for (int k = 0; k < ZB; ++k) {
            if (fv[k] == 0.0f) continue;
            const float v = fmaf(zp0 + (float)k, cvw.A, g.cv);
            const float vf = floorf(v);
            if (!(vf >= -1.0f && vf <= (float)nv)) continue;
            const int iv = (int)vf;
            const float fvv = v - vf;
            const bool v0 = iv >= 0 && iv < nv, v1 = iv + 1 >= 0 && iv + 1 < nv;
            const int64_t o = (int64_t)iv * nu + iu;
            const float val = fv[k];
            if (u0 && v0) unsafeAtomicAdd(gp + o, (1.0f - fu) * (1.0f - fvv) * val);
            if (u1 && v0) unsafeAtomicAdd(gp + o + 1, fu * (1.0f - fvv) * val);
            if (u0 && v1) unsafeAtomicAdd(gp + o + nu, (1.0f - fu) * fvv * val);
            if (u1 && v1) unsafeAtomicAdd(gp + o + nu + 1, fu * fvv * val);
        }
    }
}

// ---------------------------------------------------------------------------
// VI^T as a gather: g_p(n, m) = sum over voxels of their bilinear weight at the
// cell times delta f, every cell summed by one lane, written once.
//
// A column (i, j) of voxels projects onto one u for all z, between the detector
// columns floor(u) and floor(u) + 1, and its voxels onto v = fma(z', A, cv).  A
// wave owns M neighbouring detector columns of a view and 64 K rows, a
// lane per row (K of them, 64 apart).  The voxel columns that project between
// its outer neighbours lie in a strip; it is walked along the in-plane axis the
// strip is steeper to, 64 slabs at a time: each lane finds its slab's cells (the
// crossings of the two outer lines) and their FP64 column terms, then the wave
// takes the voxel columns one by one: the column's voxels go through the wave's
// piece of LDS (one 16-byte load per lane, the next column's in flight), and a
// lane sums its two or three with the weights 1 - |v - n|; the sum goes to the
// detector columns on both sides of u.  v - n is one fused operation from the
// exact cv - n, and the fraction of u is taken in FP64: v and u are never
// rounded to the FP32 of a large coordinate.
//
// VALU issue takes about half of its time, waits on the columns most of the rest
// (they come from the memory-side cache: 256^3 and 256 views read 6 GB).  201 x
// 187 x 149, 229 x 173, 131 views: 10.0 -> 1.10 ms against the scatter below, 0.97
// with seven waves per SIMD instead of five; 256^3 and 256 views 71.9 -> 3.27 ms.
constexpr int kViTPad = 4;
constexpr int kViTWords = 512;  // voxels of a column a wave stages, two loads of 64 x 4
__host__ __device__ inline size_t vi_t_pitch(int nz) { return (size_t)(nz + 3) / 4 * 4 + 2 * kViTPad; }

// out[(x ny + y) pitch + pad + z] = delta f(x, y, z), 0 for the pad; one tile of
// 64 x and 64 words of their columns at one y per workgroup.
template <typename TV>
__global__ __launch_bounds__(256) void vi_t_prepare_kernel(DevGeom g, const TV* __restrict__ vol, float vol_inv,
                                                           float* __restrict__ out) {
    __shared__ float tile[64][65];
    const int pitch = (int)vi_t_pitch(g.nz);
    const uint32_t gx = (uint32_t)(g.nx + 63) / 64;
    const uint32_t tile_no = tile_index();
    const uint32_t bx = tile_no % gx, rest = tile_no / gx, y = rest % (uint32_t)g.ny, bz = rest / (uint32_t)g.ny;
    const int tx = threadIdx.x & 63, ty = threadIdx.x >> 6;
    const int x = (int)bx * 64 + tx, r0 = (int)bz * 64;
    for (int r = ty; r < 64; r += 4) {
        const int z = r0 + r - kViTPad;
        float v = 0.0f;
        if (x < g.nx && z >= 0 && z < g.nz)
            v = Storage<TV>::load(vol, (size_t)x + (size_t)g.nx * ((size_t)y + (size_t)g.ny * z), vol_inv) * g.delta;
        tile[r][tx] = v;
    }
    __syncthreads();
    const int row = r0 + tx;
    if (row < pitch)
        for (int r = ty; r < 64; r += 4) {
            const int xo = (int)bx * 64 + r;
            if (xo < g.nx) out[((size_t)xo * g.ny + y) * pitch + row] = tile[tx][r];
        }
}

__device__ __forceinline__ float lane_value(float v, int l) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l));
}

// Grid: x, y = (view, column group), views first; z = block of 64 K of the rows r0 ..
// r1 - 1, which voxels can reach; the others are 0.  One
// wave per workgroup: nothing is shared, and the strips differ in length.
template <int K, int M>
__global__ __launch_bounds__(64, 7) void vi_t_kernel(DevGeom g, const float* __restrict__ vt, float* __restrict__ sino, int r0,
                                                     int r1) {
    typedef float V4 __attribute__((ext_vector_type(4)));
    __shared__ __align__(16) float stage[kViTWords + 8];
    const int lane = threadIdx.x;
    const uint32_t tile = tile_index();
    const int p = (int)(tile % (uint32_t)g.nphi), m0 = (int)(tile / (uint32_t)g.nphi) * M;
    if (m0 >= g.nu) return;
    const int nb = r0 + (int)blockIdx.z * 64 * K;
    typedef const __attribute__((address_space(4))) double* ConstView;
    const ConstView vw = (ConstView)(g.view + (size_t)p * kViewStride);
    double cvt[kViewStride];
#pragma unroll
    for (int e = 0; e < kViewStride; ++e) cvt[e] = vw[e];
    const double ca = cvt[0], sa = cvt[1], dl = (double)g.delta;
    const double Sx = -g.fod * ca, Sy = -g.fod * sa;
    auto line = [&](double col, double& rx, double& ry) {
        const double s = (col - (double)g.cu) * (double)g.du;
        rx = ca * g.fdd - s * sa;
        ry = sa * g.fdd + s * ca;
    };
    double rx, ry, ax, ay, bx, by;
    line((double)m0 + 0.5 * (M - 1), rx, ry);
    line((double)(m0 - 1), ax, ay);
    line((double)(m0 + M), bx, by);
    const bool alongy = fabs(ry) >= fabs(rx);
    const int nA = alongy ? g.ny : g.nx, nB = alongy ? g.nx : g.ny;
    const double cA = alongy ? (double)g.cy : (double)g.cx, cB = alongy ? (double)g.cx : (double)g.cy;
    const double SA = alongy ? Sy : Sx, SB = alongy ? Sx : Sy;
    const double ta = alongy ? ax / ay : ay / ax, tb = alongy ? bx / by : by / bx;  // B per A along the outer lines
    const float row0 = (float)(nb + lane) - g.cv, first = (float)nb - g.cv;  // exact: cv is a multiple of 1/2
    const float czf = g.cz, czs = czf - 2e-3f;
    const int quads = (g.nz + 3) / 4;
    const size_t pitch = vi_t_pitch(g.nz);
    float acc[M][K];
#pragma unroll
    for (int c = 0; c < K; ++c)
#pragma unroll
        for (int e = 0; e < M; ++e) acc[e][c] = 0.0f;
    // first voxel that can reach a row: the rounding of these coordinates is
    // below the 2e-3, whose voxel has a weight of that size at most
    auto first_voxel = [&](float row, float inv) __attribute__((always_inline)) {
        return ceilf(fmaf(row - 1.0f, inv, czs));
    };
    for (int ab = 0; ab < nA; ab += 64) {
        // ---- one slab per lane: its cells between the outer lines
        const int a = ab + lane;
        int b0 = 0, cnt = 0;
        if (a < nA) {
            const double at = ((double)a - cA) * dl - SA;
            const double pa = (SB + at * ta) / dl + cB, pb = (SB + at * tb) / dl + cB;
            const double lo = ceil(fmin(pa, pb) - 1e-6), hi = floor(fmax(pa, pb) + 1e-6);
            b0 = (int)fmax(lo, 0.0);
            cnt = max(0, (int)fmin(hi, (double)(nB - 1)) - b0 + 1);
        }
        const int most = __builtin_amdgcn_readfirstlane(wave_max(cnt));
        for (int q = 0; q < most; ++q) {
            const int b = b0 + q;
            const int i = alongy ? b : a, j = alongy ? a : b;
            const double xp = (double)i - (double)g.cx, yp = (double)j - (double)g.cy;
            const double iw = 1.0 / fma(cvt[2], xp, fma(cvt[3], yp, g.fod));
            const double u = fma(fma(cvt[4], xp, cvt[5] * yp), iw, (double)g.cu), uf = floor(u);
            const double e0 = uf - (double)m0;  // the detector column floor(u), from m0
            const float lwu = (float)(u - uf), lA = (float)(cvt[6] * iw), linv = 1.0f / lA;
            const float lstart = floorf(first_voxel(first, linv) * 0.25f), reach = floorf(2.0f * linv + 4e-3f) + 1.0f;
            // the column's words from lstart on that the rows reach: a second load where they exceed 64 quads
            const float words = first_voxel(first + (float)(64 * K - 1), linv) + reach - 4.0f * lstart;
            const int far = words > 256.0f ? 1 : 0;
            const bool on = q < cnt && e0 >= -1.0 && e0 <= (double)(M - 1) && lA > 0.0f &&
                            lstart < (float)(quads + 1) && words <= (float)kViTWords;
            const int lquad = (int)fmaxf(lstart, -1048576.0f), lcol = i * g.ny + j;
            const int lhow = ((int)e0 + 1) | far << 4 | (int)reach << 8;
            uint64_t todo = __ballot(on);
            if (todo == 0ull) continue;
            V4 f0, f1;
            auto load = [&](int l) __attribute__((always_inline)) {
                const float* zc = vt + (size_t)(uint32_t)__builtin_amdgcn_readlane(lcol, l) * pitch;
                const int at = __builtin_amdgcn_readlane(lquad, l) + lane;
                // quads before and after the column are 0, as its pads are
                f0 = *(const V4*)((const char*)zc + (uint32_t)(min(max(at, -1), quads) + 1) * 16u);
                if (__builtin_amdgcn_readlane(lhow, l) >> 4 & 1)
                    f1 = *(const V4*)((const char*)zc + (uint32_t)(min(max(at + 64, -1), quads) + 1) * 16u);
            };
            f0 = f1 = (V4)0.0f;
            load(__builtin_ctzll(todo));
            do {
                const int l = __builtin_ctzll(todo);
                const int how = __builtin_amdgcn_readlane(lhow, l);
                todo &= todo - 1;
                *(V4*)(stage + 4 * lane) = f0;
                if (how >> 4 & 1) *(V4*)(stage + 256 + 4 * lane) = f1;
                if (todo != 0ull) load(__builtin_ctzll(todo));
                const float A = lane_value(lA, l), inv = lane_value(linv, l), wu = lane_value(lwu, l);
                const float start = 4.0f * lane_value(lstart, l);
                const int voxels = how >> 8;
                const float* at[K];
                float t0[K], part[K];
#pragma unroll
                for (int c = 0; c < K; ++c) {
                    const float row = row0 + (float)(64 * c), k = first_voxel(row, inv);
                    at[c] = stage + (uint32_t)(k - start);
                    t0[c] = fmaf(k - czf, A, -row);
                }
                // The lane's voxels.  A weight of 0 takes nothing from its voxel, whatever it
                // holds: a sum that is not finite is taken again with that test (FINITE off).
                auto sum = [&](auto finite) __attribute__((always_inline)) {
                    float t[K];
                    auto voxel = [&](int c, float fk) __attribute__((always_inline)) {
                        const float w = __builtin_amdgcn_fmed3f(1.0f - fabsf(t[c]), 0.0f, 1.0f);
                        if constexpr (decltype(finite)::value)
                            part[c] = fmaf(w, fk, part[c]);
                        else
                            part[c] = w > 0.0f ? fmaf(w, fk, part[c]) : part[c];
                        t[c] += A;
                    };
#pragma unroll
                    for (int c = 0; c < K; ++c) {
                        t[c] = t0[c];
                        part[c] = 0.0f;
                    }
                    // read in threes, the second and third also where only the first counts
                    for (int k = 0; k < voxels; k += 3) {
                        float f[3][K];
#pragma unroll
                        for (int c = 0; c < K; ++c)
#pragma unroll
                            for (int h = 0; h < 3; ++h) f[h][c] = at[c][k + h];
#pragma unroll
                        for (int c = 0; c < K; ++c) voxel(c, f[0][c]);
                        if (k + 1 < voxels) {
#pragma unroll
                            for (int c = 0; c < K; ++c) voxel(c, f[1][c]);
                        }
                        if (k + 2 < voxels) {
#pragma unroll
                            for (int c = 0; c < K; ++c) voxel(c, f[2][c]);
                        }
                    }
                };
                sum(std::true_type{});
                bool odd = false;
#pragma unroll
                for (int c = 0; c < K; ++c) odd |= !__builtin_isfinite(part[c]);
                if (__ballot(odd) != 0ull) sum(std::false_type{});
                const int e = (how & 15) - 1;
#pragma unroll
                for (int d = -1; d < M; ++d)
                    if (e == d) {
                        // a branch, not selects over all columns (empty statement)
                        asm volatile("" : "+v"(part[0]));
#pragma unroll
                        for (int c = 0; c < K; ++c) {
                            if (d >= 0) acc[d < 0 ? 0 : d][c] = fmaf(1.0f - wu, part[c], acc[d < 0 ? 0 : d][c]);
                            if (d + 1 < M) acc[d + 1 < M ? d + 1 : 0][c] = fmaf(wu, part[c], acc[d + 1 < M ? d + 1 : 0][c]);
                        }
                    }
            } while (todo != 0ull);
        }
    }
#pragma unroll
    for (int c = 0; c < K; ++c) {
        const int n = nb + 64 * c + lane;
        if (n < r1) {
            float* o = sino + ((size_t)m0 + (size_t)g.nu * ((size_t)n + (size_t)g.nv * p));
#pragma unroll
            for (int d = 0; d < M; ++d)
                if (m0 + d < g.nu) o[d] = acc[d][c];
        }
    }
    if (blockIdx.z == 0)
        for (int n = lane; n < g.nv - (r1 - r0); n += 64) {
            const int row = n < r0 ? n : n + (r1 - r0);
            float* o = sino + ((size_t)m0 + (size_t)g.nu * ((size_t)row + (size_t)g.nv * p));
            for (int d = 0; d < M; ++d)
                if (m0 + d < g.nu) o[d] = 0.0f;
        }
}

}  // namespace

// Whether every FDK weight of the geometry is within fdk_weight's bounds: the
// source is outside the volume's square, so that w is within fod +- its half
// diagonal, and the extreme terms of that range are.
static bool fdk_in_bounds(const DevGeom& d) {
    const double half = 0.5 * std::sqrt(2.0) * (double)d.delta * (double)std::max(d.nx, d.ny);
    const double w0 = d.fod - half, w1 = d.fod + half;
    if (!(w0 > 0.01 * d.fod)) return false;
    const double ku = d.fdd / (double)d.du, alpha = M_PI * d.fod * d.fdd / (double)d.nphi;
    const double up = half / w0 * ku, vp = 0.5 * (double)d.nz * (double)d.delta * d.fdd / ((double)d.dv * w0);
    const double num0 = alpha * ku / (w1 * w1), num1 = alpha * ku / (w0 * w0);
    return num0 >= 2.0 * kFdkLeast && num1 <= 0.5 * kFdkMost && ku * ku >= 2.0 * kFdkLeast &&
           ku * ku + up * up + vp * vp <= 0.5 * kFdkMost;
}

template <typename TV, int FDK, int ZS, bool PAIR>
static void launch_vi_tiles(const DevGeom& d, const float* sino, const ViBox* boxes, void* vol, float vol_scale,
                            float post, hipStream_t s) {
    const dim3 grid(ceil_div(d.nx, SX), ceil_div(d.ny, SY),
                    FDK == 3 ? ceil_div((d.nz + 1) / 2, ZS / 2) : ceil_div(d.nz, ZS));
    hipLaunchKernelGGL((vi_staged_kernel<TV, FDK, ZS, PAIR>), grid, dim3(SX * SY), 0, s, d, sino, boxes, (TV*)vol,
                       vol_scale, post);
}

// The staged kernel on an FP32 sinogram, with the geometry's box table
// (`boxes`) or, when null, one made for this call from the stream-ordered
// pool.
template <typename TV, bool PAIR>
static hipError_t launch_vi_staged(const DevGeom& d, int fdk, const float* sino, const void* boxes, void* vol,
                                   float vol_scale, float post, hipStream_t s) {
    const int ntx = ceil_div(d.nx, SX), nty = ceil_div(d.ny, SY);
    void* own = nullptr;
    hipError_t e = hipSuccess;
    if (!boxes) {
        if ((e = hipMallocAsync(&own, vi_box_count(d) * sizeof(ViBox), s)) != hipSuccess) return e;
        hipLaunchKernelGGL(vi_box_kernel, tile_grid(vi_box_count(d), SX * SY), dim3(SX * SY), 0, s, d, (ViBox*)own, ntx);
        e = hipGetLastError();
        boxes = own;
    }
    if (e == hipSuccess) {
        // Columns of 16 voxels share a column-view's terms best; below two or three
        // workgroups per CU the views' latency decides, and shorter columns are more
        // workgroups that wait for several views at once.  VI, us at 4 / 8 / 16
        // voxels by workgroups of 16: 64 (64^3, 64 views) 32 / 48 / 73; 150 (80^3, 64)
        // 39 / 48 / 73; 216 (96^3, 64) 57 / 49 / 73; 512 (128^3, 180 views) 279 / 186 /
        // 214; 765 (136^3, 96) 204 / 155 / 142; 1000 (160^3, 180) 487 / 335 / 281.
        const size_t tiles = (size_t)ntx * nty * ceil_div(d.nz, kViTileZ);
        const int zs = tiles < 192 ? 4 : tiles < 640 ? 8 : 16;
        const ViBox* bt = (const ViBox*)boxes;
        if (fdk && !fdk_in_bounds(d))
            launch_vi_tiles<TV, 1, kViTileZ, PAIR>(d, sino, bt, vol, vol_scale, post, s);
        else if (zs == kViTileZ)
            fdk ? launch_vi_tiles<TV, 3, kViTileZ, PAIR>(d, sino, bt, vol, vol_scale, post, s)
                : launch_vi_tiles<TV, 0, kViTileZ, PAIR>(d, sino, bt, vol, vol_scale, post, s);
        else if (zs == 8)
            fdk ? launch_vi_tiles<TV, 3, 8, PAIR>(d, sino, bt, vol, vol_scale, post, s)
                : launch_vi_tiles<TV, 0, 8, PAIR>(d, sino, bt, vol, vol_scale, post, s);
        else
            fdk ? launch_vi_tiles<TV, 2, 4, PAIR>(d, sino, bt, vol, vol_scale, post, s)
                : launch_vi_tiles<TV, 0, 4, PAIR>(d, sino, bt, vol, vol_scale, post, s);
        e = hipGetLastError();
    }
    if (own) {
        const hipError_t f = hipFreeAsync(own, s);
        if (e == hipSuccess) e = f;
    }
    return e;
}

int launch_vi(const tomo_geom* g, Buf sino, MutBuf vol, hipStream_t s, int fdk) {
    const DevGeom& d = g->dev;
    if (sino.dtype != TOMO_F32 && sino.dtype != TOMO_F16 && sino.dtype != TOMO_BF16)
        return fail(TOMO_ERR_UNSUPPORTED, "unsupported element type");
    if (vol.dtype != TOMO_F32 && vol.dtype != TOMO_F16 && vol.dtype != TOMO_BF16)
        return fail(TOMO_ERR_UNSUPPORTED, "unsupported element type");
    // byte offsets within one view are 32-bit
    if ((size_t)(d.nu + 1) * d.nv >= (1ull << 30))
        return fail(TOMO_ERR_UNSUPPORTED, "VI needs views of fewer than 2^30 cells");
    // An FP16 sinogram becomes u-pair words, a BF16 one is widened (value =
    // stored / scale) to FP32; either copy comes from the stream-ordered pool
    // and is released after the backprojection on the same stream.
    const bool pair = sino.dtype == TOMO_F16;
    const float* taps = (const float*)sino.p;
    void* wide = nullptr;
    if (pair) {
        const size_t rows = (size_t)d.nv * d.nphi;
        if (rows >= (1ull << 31)) return fail(TOMO_ERR_UNSUPPORTED, "VI needs fewer than 2^31 detector rows");
        TOMO_HIP(hipMallocAsync(&wide, rows * (size_t)(d.nu + 1) * sizeof(uint32_t), s));
        if (rows > 0) hipLaunchKernelGGL(vi_pair_kernel, tile_grid(rows, 256), dim3(256), 0, s,
                                         (const uint16_t*)sino.p, (uint32_t*)wide, d.nu, (uint32_t)rows);
        const hipError_t le = hipGetLastError();
        if (le != hipSuccess) {
            (void)hipFreeAsync(wide, s);
            TOMO_HIP(le);
        }
        taps = (const float*)wide;
    } else if (sino.dtype != TOMO_F32) {
        TOMO_HIP(hipMallocAsync(&wide, g->nsino() * sizeof(float), s));
        const int rc = launch_convert(sino, MutBuf{wide, TOMO_F32, 1.0f}, g->nsino(), s);
        if (rc) {
            (void)hipFreeAsync(wide, s);
            return rc;
        }
        taps = (const float*)wide;
    }
    const float post = pair ? 1.0f / sino.scale : 1.0f;
    hipError_t e = hipSuccess;
#define TOMO_VI_LAUNCH(TV)                                                                              \
    e = pair ? launch_vi_staged<TV, true>(d, fdk, taps, g->d_vi_boxes, vol.p, vol.scale, post, s)     \
             : launch_vi_staged<TV, false>(d, fdk, taps, g->d_vi_boxes, vol.p, vol.scale, post, s)
    switch (vol.dtype) {
        case TOMO_F32: TOMO_VI_LAUNCH(float); break;
        case TOMO_F16: TOMO_VI_LAUNCH(__half); break;
        default: TOMO_VI_LAUNCH(__hip_bfloat16); break;
    }
#undef TOMO_VI_LAUNCH
    if (wide) TOMO_HIP(hipFreeAsync(wide, s));
    TOMO_HIP(e);
    return TOMO_OK;
}

int launch_vi_boxes(const DevGeom& d, void* boxes, hipStream_t s) {
    const int ntx = ceil_div(d.nx, SX);
    hipLaunchKernelGGL(vi_box_kernel, tile_grid(vi_box_count(d), SX * SY), dim3(SX * SY), 0, s, d, (ViBox*)boxes, ntx);
    TOMO_HIP(hipGetLastError());
    return TOMO_OK;
}

hipError_t launch_batch_vi(BatchTable* t, hipStream_t s) {
    hipLaunchKernelGGL(vi_batch_kernel, dim3(kBatchGrid), dim3(SX * SY), 0, s, t, t->next);
    return hipGetLastError();
}

// Detector rows that voxels of a geometry with the source outside the volume's square
// project next to, r0 .. r1 - 1 (none: r1 = r0): of a detector taller than the volume's
// shadow only these are walked for (256 x 256 x 1, 256 rows and views 3.06 -> 1.94 ms).
struct ViTRows {
    int r0, r1;
};
static ViTRows vi_t_reach(const DevGeom& d) {
    const double dl = d.delta, nearest = d.fod - dl * std::hypot((double)d.cx, (double)d.cy);
    const double reach = (double)d.cz * dl * d.fdd / ((double)d.dv * nearest) * (1.0 + 1e-6) + 1.0;
    const int r0 = reach < (double)d.cv ? (int)std::ceil((double)d.cv - reach) : 0;
    return ViTRows{r0, std::max(r0, d.nv - r0)};
}

// Row steps per lane of the gather, the fewest row blocks that K <= 4 allows;
// 0 where it does not apply and the voxels scatter: a voxel column behind or
// beside the source, a wave's outer lines too far apart (detector columns as
// wide as a 20th of the distance to them), or 64 rows that reach more than
// kViTWords voxels of a column (7.8 voxels to a row).  There is no lower limit of size:
// 17^3 and 16 views take 33 us here and 108 scattered.  Columns of which hardly a
// voxel is on the detector scatter: 20 ps per column and view and 26 per atomic, two
// a voxel and row, or 2.8 us a view; the gather 80 ps and 31 more per detector column of a
// voxel, and for the strips that are walked past a narrow grid.  256 x 256 and 256 views, scatter and gather in us: one slice and row 1233 and
// 1882, two rows 1849 and 1886, 8 rows 2348 and 1880; 64 x 64 and 64 views 182 and 79; 64
// slices, 4 rows of a quarter voxel, 90 views 541 and 658; 256 x 64 x 1, one row and 256
// views 727 and 838.
static int vi_t_steps(const DevGeom& d) {
    const double half = 0.5 * (double)d.delta * (double)std::max(d.nx, d.ny);
    const double far = d.fod + std::sqrt(2.0) * half;
    const double inv = far * (double)d.dv / ((double)d.delta * d.fdd);  // most voxels to a row
    if (!(d.fod > 1.01 * std::sqrt(2.0) * half && (double)d.du * (4 + 1) < 0.25 * d.fdd)) return 0;
    // FP32 voxel coordinates within 1e-3, 32-bit column numbers
    if (d.nv * inv + d.nz > 8192.0 || (double)d.nx * d.ny > 2147483647.0) return 0;
    const double mag = (double)d.delta * d.fdd / d.fod, views = (double)d.nx * d.ny * d.nphi;
    const double pairs = std::min((double)d.nz * std::min(d.nv, 2), 2.0 * (d.nv + 1) * (double)d.dv / mag);
    const double scatter = std::max(1e-6 * views * (20.0 + 52.0 * pairs), 2.8 * d.nphi);
    const double strips = std::sqrt((double)d.nx * d.ny) * std::max(d.nx, d.ny) * d.nphi;  // walked past narrow grids too
    if (12.0 + scatter < 30.0 + 1e-6 * strips * (80.0 + 31.0 * mag / (double)d.du)) return 0;
    const ViTRows rows = vi_t_reach(d);
    const int steps = std::max(1, (int)ceil_div(rows.r1 - rows.r0, 64)), most = std::min(4, (int)(((kViTWords - 6) / (1.001 * inv) - 1.0) / 64.0));
    return most < 1 ? 0 : (int)ceil_div(steps, ceil_div(steps, most));
}

template <int K>
static void launch_vi_t(const DevGeom& d, const float* vt, float* sino, hipStream_t s) {
    // Columns per wave: wide strips share their voxel columns, M + 1 reads for M
    // columns; narrow ones are more waves (1024 SIMDs).  Waves at M = 4, us at
    // M = 1 / 2 / 4: 1024 (64^3, 64 views) 81 / 103 / 172; 1152 (96^3, 48) 160 /
    // 197 / 311; 4096 (128^3, 128) 484 / 416 / 454; 7598 (201 x 187 x 149, 131)
    // 1253 / 1128 / 1104; 16384 (256^3, 256) 4636 / 3689 / 3445.
    const ViTRows r = vi_t_reach(d);
    const unsigned blocks = std::max(1u, ceil_div(r.r1 - r.r0, 64 * K));
    const size_t waves = (size_t)ceil_div(d.nu, 4) * d.nphi * blocks;
    const int cols = waves < 2048 ? 1 : waves < 6144 ? 2 : 4;
    const dim3 grid = tile_grid((size_t)ceil_div(d.nu, cols) * d.nphi, 64, blocks);
    if (cols == 1)
        hipLaunchKernelGGL((vi_t_kernel<K, 1>), grid, dim3(64), 0, s, d, vt, sino, r.r0, r.r1);
    else if (cols == 2)
        hipLaunchKernelGGL((vi_t_kernel<K, 2>), grid, dim3(64), 0, s, d, vt, sino, r.r0, r.r1);
    else
        hipLaunchKernelGGL((vi_t_kernel<K, 4>), grid, dim3(64), 0, s, d, vt, sino, r.r0, r.r1);
}

int launch_vi_adjoint(const tomo_geom* g, Buf vol, MutBuf sino, hipStream_t s) {
    if (sino.dtype != TOMO_F32) return fail(TOMO_ERR_UNSUPPORTED, "adjoint output must be F32");
    const DevGeom& d = g->dev;
    const float inv = 1.0f / vol.scale;
    float* vt = nullptr;
    // without the copy's memory, or in a stream capture, which is left free of
    // allocations, the voxels scatter
    const int steps = stream_captures(s) ? 0 : vi_t_steps(d);
    if (steps > 0 &&
        hipMallocAsync((void**)&vt, (size_t)d.nx * d.ny * vi_t_pitch(d.nz) * sizeof(float), s) != hipSuccess) {
        (void)hipGetLastError();
        vt = nullptr;
    }
    if (vt) {
        const size_t tiles = (size_t)ceil_div(d.nx, 64) * d.ny * ceil_div(vi_t_pitch(d.nz), 64);
        TOMO_DISPATCH_STORAGE(vol.dtype, TV, {
            hipLaunchKernelGGL((vi_t_prepare_kernel<TV>), tile_grid(tiles, 256), dim3(256), 0, s, d, (const TV*)vol.p, inv, vt);
        });
        switch (steps) {
            case 1: launch_vi_t<1>(d, vt, (float*)sino.p, s); break;
            case 2: launch_vi_t<2>(d, vt, (float*)sino.p, s); break;
            case 3: launch_vi_t<3>(d, vt, (float*)sino.p, s); break;
            default: launch_vi_t<4>(d, vt, (float*)sino.p, s); break;
        }
        const hipError_t e = hipGetLastError();
        const hipError_t f = hipFreeAsync(vt, s);
        TOMO_HIP(e);
        TOMO_HIP(f);
        return TOMO_OK;
    }
    int rc = launch_fill((float*)sino.p, 0.0f, g->nsino(), s);
    if (rc) return rc;
    dim3 grid(ceil_div(d.nx, TX), ceil_div(d.ny, TY), ceil_div(d.nz, ZB));
    TOMO_DISPATCH_STORAGE(vol.dtype, TV, {
        hipLaunchKernelGGL((vi_adjoint_kernel<TV>), grid, dim3(TX * TY), 0, s, d, (const TV*)vol.p, inv,
                           (float*)sino.p);
    });
    TOMO_HIP(hipGetLastError());
    return TOMO_OK;
}

}  // namespace tomo
