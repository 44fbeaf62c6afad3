// tomo_internal.hpp - internal types of libtomogpi_mi355x.so shared by the
// host API (api.cpp, loop.cpp, config.cpp) and the kernel files (*.hip).
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstddef>
#include <string>
#include <vector>

#include "tomogpi.h"

namespace tomo {

// ---------------------------------------------------------------- errors
// Thread-local message of the last failure (tomo_last_error()).
void set_error(const std::string& msg);
int fail(int status, const std::string& msg);
int hip_fail(hipError_t e, const char* what);

#define TOMO_HIP(call)                                         \
    do {                                                       \
        hipError_t e_ = (call);                                \
        if (e_ != hipSuccess) return ::tomo::hip_fail(e_, #call); \
    } while (0)

// -------------------------------------------------------------- geometry
// Scalars every kernel needs, passed by value.  Types follow the reference
// (float detector / voxel sizes and centres, double distances).
struct DevGeom {
    int32_t nx, ny, nz, nu, nv, nphi;
    double fod, fdd;
    float du, dv, cu, cv;
    float delta, cx, cy, cz;
    // Per-view table in device memory, kViewStride doubles per view:
    //   [0] cos phi  [1] sin phi
    //   [2] delta cos  [3] delta sin  [4] -(delta sin) FDD/du
    //   [5] (delta cos) FDD/du  [6] delta FDD/dv  [7] unused
    const double* view;
    // Reference float tables alpha = (float)cos, beta = (float)sin, 2 per view.
    const float* view_f;
};
constexpr int kViewStride = 8;

}  // namespace tomo

struct tomo_ctx {
    int device = 0;
};

struct tomo_geom {
    tomo_ctx* ctx = nullptr;
    tomo_geom_desc desc{};
    tomo_geom_info info{};
    std::vector<double> phi, view;  // host copies
    std::vector<float> view_f;
    double* d_view = nullptr;
    float* d_view_f = nullptr;
    void* d_vi_boxes = nullptr;  // VI box table (tomo_geom_create), or null: made per call
    tomo::DevGeom dev{};
    size_t nvox() const { return (size_t)info.nx * info.ny * info.nz; }
    size_t nsino() const { return (size_t)info.nu * info.nv * info.nphi; }
};

namespace tomo {

// Volumes the Siddon projector takes: its offsets into the z-column copy, and
// their steps, are 32-bit (a copy of up to 2^32 words; this bound is half of it
// and a border).
inline bool sid_volume_fits(int nx, int ny, int nz) {
    const size_t z2 = 2 * ((size_t)nz + 1);
    return (size_t)nx * z2 * ((size_t)ny + 2) < (1ull << 32) && (size_t)ny * z2 * ((size_t)nx + 2) < (1ull << 32);
}
// The planes of the volume that a projector's rays can read, of which its copy is
// made: z0 .. z0 + nz - 1.  The outermost row leaves the field of view farthest
// from the mid plane; 1 1/2 planes more for the neighbours that a sample or a cell
// reads, 1/2 for the rounding of its place.
struct ProjPlanes {
    int z0, nz;
};
inline ProjPlanes proj_planes(const DevGeom& d, int cube) {
    const double fov = 0.5 * (double)d.nx * (double)d.delta * (cube ? 1.4143 : 1.0);
    const double reach = (double)d.cv * (double)d.dv * (d.fod + fov) / (d.fdd * (double)d.delta) + 2.0;
    // below 2^20 planes FP32 places are well within the margin
    if (!(reach < (double)d.cz) || d.nz >= (1 << 20)) return ProjPlanes{0, d.nz};
    const int z0 = (int)((double)d.cz - reach);
    return ProjPlanes{z0, d.nz - 2 * z0};
}
// z-column copy of nz planes of es-byte elements (proj_copy.hpp): 4-byte words per
// (x, y) column, and of the whole copy.
__host__ __device__ inline uint32_t zcol_pitch(int nz, size_t es) { return (uint32_t)nz + (es == 4 ? 2u : 1u); }
__host__ __device__ inline size_t zcol_words(int nx, int ny, int nz, size_t es) {
    return (size_t)nx * ny * zcol_pitch(nz, es);
}
// A projector workgroup: one wave's detector cells in kProjViews consecutive views.
constexpr int kProjViews = 4;
// Column groups (workgroups) of a row band, rounded up to a multiple of the 8
// XCDs.
inline uint32_t proj_groups(int nu, int rows) {
    const uint32_t cols = 64u / (uint32_t)rows;
    return ((uint32_t)nu + 8u * cols - 1u) / (8u * cols) * 8u;
}
// RS copy of nz planes of es-byte elements (proj_copy.hpp): 8-byte elements per x
// and y step and in all, and whether RS reads it through 32-bit byte offsets
// (below 2^32 - 16 bytes, where the offset of a read that returns 0 lies, and
// its steps in signed 24 bits, for 24-bit multiplies).
struct RsCopyShape {
    size_t elems;
    uint32_t sx, sy;
    bool buf;
};
__host__ __device__ inline RsCopyShape rs_copy_shape(int nx, int ny, int nz, size_t es) {
    RsCopyShape c;
    const size_t sy = (size_t)nz + 2, sx = sy * ((size_t)ny + (es == 4 ? 2 : 1));
    c.elems = sx * ((size_t)nx + 1);
    c.sx = (uint32_t)sx;
    c.sy = (uint32_t)sy;
    c.buf = c.elems * 8 < 0xfffffff0ull && sx * 8 < (1ull << 23) && nz < (1 << 23);
    return c;
}
// The detector rows whose rays are in the volume, each by the part of its way through
// the FOV: z leaves the volume at the in-plane distance edge / |n - cv|.  Rows are
// counted from the middle on, until there are `enough`.
struct CrossingRows {
    double fov, nearest, edge;  // radius; of the FOV from the source; mm
    explicit CrossingRows(const DevGeom& d)
        : fov(0.5 * (double)d.nx * (double)d.delta), nearest(d.fod - fov),
          edge(0.5 * (double)d.nz * (double)d.delta * d.fdd / (double)d.dv) {}
    double part(double off) const {
        return off * (nearest + 2.0 * fov) <= edge ? 1.0 : std::max(0.0, (edge / off - nearest) / (2.0 * fov));
    }
    double count(const DevGeom& d, double enough) const {
        double rows = 0.0;
        for (int n = d.nv / 2; n < d.nv && rows < enough; ++n) {
            const double off = (double)n - (double)d.cv, p = part(off);
            if (p == 0.0) break;
            rows += off == 0.0 ? p : 2.0 * p;
        }
        return rows;
    }
};
// Detector columns whose rays cross the FOV.
inline double crossing_columns(const DevGeom& d, const CrossingRows& c) {
    const double reach = c.nearest > 0.0 ? 2.0 * c.fov * d.fdd / std::sqrt(d.fod * d.fod - c.fov * c.fov) / (double)d.du + 1.0 : 1e30;
    return std::min((double)d.nu, reach);
}

// Detector rows of a projector's wave (a power of two up to 64, by 64 / rows columns).
// `tall` where many rows cross the volume, else the rows of the least
//     sum over row groups of max(16 rows, lines) x the longest ray's part of the FOV + 1/2.
// A gather takes 16 cycles of the texture path a wave, 64 / rows columns of it, and the
// L2 lines of the columns' runs of z take more where the runs are short and the columns
// lie far apart; idle rows of a group that holds a ray cost as much as the others.
// lines: 20 + 3 (planes + 2) up to 160 for Siddon, 15 + 4 (planes + 2) up to 120 for RS, and
// up to twice that with few views, whose rays share fewer lines: over 125 and 185 shapes
// of 1 to 48 crossing rows 1% and 2% above the best rows' times.
// Not below `tall` with fewer waves than SIMDs (90 views of 64 x 4 cells, RS: 71 us by 4
// rows, 50 by 16), and one row a wave for one crossing row only (256 x 256 x 1 and 64 rows,
// RS: 171 us by 1 row, 91 by 2).
//
// 512 x 512 and 360 views, us at 64 / 32 / 16 / 8 / 4 / 2 / 1 rows.  Siddon: one slice
// and row 2658 / 1348 / 698 / 380 / 215 / 161 / 155; 8 and 8 2682 / 1371 / 714 / 394 /
// 450 / 820 / 1852; 4 slices, 64 rows 2688 / 2676 / 1395 / 760 / 456 / 408 / 766.  RS: 4152
// / 2149 / 1134 / 632 / 391 / 286 / 210; 4072 / 2064 / 1064 / 564 / 657 / 1180 / 2364; 4228 /
// 4227 / 2207 / 1195 / 687 / 570 / 824.
inline int proj_wave_rows(const DevGeom& d, double lines, int tall) {
    constexpr int kMost = 48;  // rows that cross the volume
    const CrossingRows c(d);
    if (!(c.nearest > 0.0)) return tall;
    const int first = std::max(0, (int)std::ceil((double)d.cv - std::min(c.edge / c.nearest, 1e9)));
    const int crossing = d.nv - 2 * first;  // centred
    if (crossing < 1 || crossing > kMost) return tall;
    const double share = lines * (1.0 + std::min(1.0, 60.0 / d.nphi));
    int best = tall;
    double least = 0.0;
    for (int r = 64; r >= std::min(crossing, 2); r >>= 1) {
        const int g0 = first / r, g1 = (d.nv - 1 - first) / r;
        if (r < tall && (size_t)d.nu * r / 64 * d.nphi * (size_t)(g1 - g0 + 1) < 1024) break;
        double cost = 0.5 * ((d.nv + r - 1) / r - (g1 - g0 + 1));
        for (int g = g0; g <= g1; ++g) {
            // the group's row nearest to the mid plane
            const double n = std::min(std::max((double)d.cv, (double)g * r), std::min((double)g * r + r, (double)d.nv) - 1.0);
            cost += std::max(16.0 * r, share) * c.part(std::fabs(n - (double)d.cv)) + 0.5;
        }
        if (r == 64 || cost <= least) {
            least = cost;
            best = r;
        }
    }
    return best;
}
// Siddon.  tall: the most of 64, 32 and 16 that leave no more than an eighth of the
// row groups' lanes idle.
inline int sid_wave_rows(const DevGeom& d, ProjPlanes zp) {
    int tall = 64;
    while (tall > 16 && ((d.nv + tall - 1) / tall * tall - d.nv) * 8 > d.nv) tall >>= 1;
    return proj_wave_rows(d, std::min(20.0 + 3.0 * (zp.nz + 2), 160.0), tall);
}
// RS.  tall: 32, or 16 where that leaves fewer lanes idle.  At equal sample index the rows
// of a column drift apart in plane with the cosine of the cone angle, so longer waves
// touch more columns at once (512^3 / 512 views: 68.6 ms at 64 rows, 55.3 at 32, 54.6 at
// 16); shorter ones read shorter runs of z (1024^3, 96 views: 82, 87, 101 ms).
inline int rs_wave_rows(const DevGeom& d, ProjPlanes zp) {
    return proj_wave_rows(d, std::min(15.0 + 4.0 * (zp.nz + 2), 120.0),
                          ((d.nv + 31) / 32 * 32 - d.nv) * 8 <= d.nv ? 32 : 16);
}

// Derives the geometry exactly as the reference constructors do.
int derive_geometry(const tomo_geom_desc& d, tomo_geom* g);

// ------------------------------------------------------------- launchers
// All launchers are stream-ordered and check their launch shape against the
// buffers they are given.  Element type codes are TOMO_F32/F16/BF16.
struct Buf {
    const void* p;
    int dtype;
    float scale;
};
struct MutBuf {
    void* p;
    int dtype;
    float scale;
};

// fdk: FDK-weighted form (back_fdk) instead of delta * sum.
int launch_vi(const tomo_geom* g, Buf sino, MutBuf vol, hipStream_t s, int fdk = 0);
int launch_vi_adjoint(const tomo_geom* g, Buf vol, MutBuf sino, hipStream_t s);
// Projector options beyond the FOV / compat mode.  index_reads: read the
// copies through 64-bit element indices even where 32-bit buffer
// offsets apply (the form every copy of 4 GiB or more takes).  copy: memory of
// the caller for the projector's copy of the volume (rs_copy_shape or
// zcol_words, for its planes and the volume's element size); null: the launcher allocates it
// from the stream-ordered pool for the call.
struct ProjExtra {
    bool index_reads = false;
    bool staged = false;  // RS, Siddon (FP32 volumes): LDS-staged taps instead of per-lane gathers
    void* copy = nullptr;
};
int launch_rs(const tomo_geom* g, int cube, Buf vol, MutBuf sino, hipStream_t s, const ProjExtra& x = ProjExtra{});
int launch_rs_adjoint(const tomo_geom* g, int cube, Buf sino, MutBuf vol, hipStream_t s);
int launch_siddon(const tomo_geom* g, int compat, Buf vol, MutBuf sino, hipStream_t s,
                  const ProjExtra& x = ProjExtra{});
int launch_siddon_adjoint(const tomo_geom* g, Buf sino, MutBuf vol, hipStream_t s);
// Work counters (roofline accounting): sum of L_r (RS) and number of
// positive chords (Siddon).  Synchronous.
int count_rs_samples(tomo_ctx* ctx, const tomo_geom* g, int cube, uint64_t* out, hipStream_t s);
int count_siddon_segments(tomo_ctx* ctx, const tomo_geom* g, uint64_t* out, hipStream_t s);

int launch_fill(float* x, float v, size_t n, hipStream_t s);
int launch_diff(const float* a, const float* b, float* out, size_t n, hipStream_t s);
int launch_scale(float* x, float v, size_t n, hipStream_t s);
int launch_axpy(float* y, const float* x, float a, int positive, size_t n, hipStream_t s);
int launch_laplacian(const float* x, float* y, int nx, int ny, int nz, hipStream_t s);

// The loops' steps: fused passes with partial sums (kLoopPartials doubles per
// sum at most, one per block of loop_blocks(n)), and the kernel that ends the
// sums and applies the step rule to the iteration's statistics on the device.
constexpr int kLoopPartials = 2048;
enum LoopSum { kLoopResidual, kLoopReg, kLoopDirReg, kLoopDir, kLoopProj, kLoopSums };
enum LoopRule { kRuleOptimal, kRuleFixed, kRuleBeta, kRuleConjugate, kRuleResidual };
struct LoopStep {
    const double* partial;    // kLoopSums x kLoopPartials
    int blocks[kLoopSums];    // 0: not summed
    tomo_gd_iter_stat* stat;  // of the iteration, device memory (kRuleResidual: its first field only)
    double* state;            // smallest step (gd), last |g|^2 (cg)
    double init;              // state before the first iteration
    double lambda;
    int rule, first, begins;  // first iteration of the run; first call of the iteration
};
unsigned loop_blocks(size_t n);
int launch_loop_sq(const float* x, size_t n, double* partial, hipStream_t s);
int launch_diff_sq(const float* a, const float* b, const float* w, float* o, size_t n, double* partial, hipStream_t s);
int launch_laplacian_sq(const float* x, float* y, int nx, int ny, int nz, double* partial, double* partial_x,
                        hipStream_t s);
int launch_scale_laplacian(const float* x, float* d, float scale, float a, int nx, int ny, int nz, hipStream_t s);
int launch_axpy_scalar(float* y, const float* x, const double* a, int positive, size_t n, hipStream_t s);
int launch_direction(const float* g, float* d, const double* beta, size_t n, double* partial, hipStream_t s);
int launch_loop_step(const LoopStep& a, hipStream_t s);
// SIRT element-wise steps: w = s > 0 ? a / s : 0; x = x + c * b (+clamp).
int launch_recip_weight(const float* s_in, float a, float* w, size_t n, hipStream_t s);
int launch_waxpy(float* x, const float* c, const float* b, int positive, size_t n, hipStream_t s);
int reduce_sq_norm(tomo_ctx* ctx, Buf x, size_t n, double* out, hipStream_t s);
int reduce_dot(tomo_ctx* ctx, const float* a, const float* b, size_t n, double* out, hipStream_t s);
// Allocation-free squared norm: the partial sums live in a device array of
// the library, one per GPU (noalloc_scratch_init looks its address up once per
// device, with that device current; tomo_ctx_create calls it).  Synchronous.
int noalloc_scratch_init(int device);
int reduce_sq_norm_noalloc(int device, Buf x, size_t n, double* out, hipStream_t s);
// max |x| over n FP32 elements.  Synchronous.
int reduce_max_abs(const float* x, size_t n, float* out, hipStream_t s);
int launch_convert(Buf in, MutBuf out, size_t n, hipStream_t s);

// Ellipsoid phantoms.  mode 0: Shepp-Logan form (normalised coordinates,
// rotation then offset, division by squared semi-axes); mode 1: random
// ellipsoids (voxel offsets, offset then rotation, inverse squared axes).
// table: 16 doubles per ellipsoid (9 rotation, 3 centre, 3 axis terms, 1
// density).
int launch_ellipsoids(const tomo_geom* g, int mode, const double* d_table, int count, float* vol,
                      hipStream_t s);

}  // namespace tomo
