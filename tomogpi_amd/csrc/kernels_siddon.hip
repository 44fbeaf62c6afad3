// kernels_siddon.hip - Siddon projector (clean and reference-compatible
// forms), the exact transpose of the clean form, and its segment counter.
//
// Clean form (default).  Exact chord lengths (mm) through the voxels the ray
// crosses inside the FOV = inscribed cylinder of radius N delta/2 (the
// reference Siddon's FOV, SiddonProjector_compute_C_mem_CPU.cpp:99-111) cut by
// the z extent of the volume.  The source sits on the RS/VI side
// (-FOD(cos,sin)), so RS, VI and the clean Siddon share one geometry.  Ray
// setup (FOV entry, first voxel, first plane crossing on each axis, distance
// between crossings) is FP64; the traversal runs in FP32 relative to the FOV
// entry with the n-th crossing of an axis at fma(n, inc, first), so no
// crossing is lost to accumulated rounding; the chord-weighted sum is FP32.
//
// Compat form (TOMO_FLAG_SIDDON_COMPAT).  The reference C path
// (SiddonProjector_compute_C_mem_CPU.cpp:20-276) with its float/double
// evaluation order and quirks: source on the +FOD side (mirror of RS/VI),
// first voxel half a voxel behind the entry, last chord not clipped, indices
// % 256 with unsigned wrap, no z clip.  Defined for 256^3 volumes only.
#include <algorithm>
#include <cmath>

#include "proj_copy.hpp"
#include "batch.hpp"
#include "stage_box.hpp"

namespace tomo {
namespace {

constexpr int BX = kProjTileU, BY = kProjTileV;

struct SidRay {
    int idx[3], step[3];
    float first[3], inc[3], tmax;
    bool ok;
};

// FP64 ray setup (first crossings at +0 or later: "+ 0.0f" turns a -0 into
// +0).  tmax is the FOV chord, shortened to the first crossing
// that takes a voxel index out of the grid (the n-th crossing of axis a is
// at fma(n, inc_a, first_a), the value the traversal computes).  A traversal
// that stops at that crossing takes exactly the segments of one that steps
// out of the grid there and then stops, so no index range test is needed in
// the loops below.
__device__ __forceinline__ SidRay sid_setup(const DevGeom& g, int p, int m, int n) {
    SidRay r{};
    const double* vw = g.view + (size_t)p * kViewStride;
    const double ca = vw[0], sa = vw[1], dl = (double)g.delta;
    const double s = ((double)m - (double)g.cu) * (double)g.du;
    const double t = ((double)n - (double)g.cv) * (double)g.dv;
    const double rx = ca * g.fdd - s * sa, ry = sa * g.fdd + s * ca, rz = t;
    const double L = sqrt((rx * rx + ry * ry) + rz * rz);
    const double d[3] = {rx / L, ry / L, rz / L};
    const double S[3] = {-g.fod * ca, -g.fod * sa, 0.0};
    const double Rm = 0.5 * (double)g.nx * dl;
    const double a = d[0] * d[0] + d[1] * d[1];
    if (!(a > 0.0)) return r;
    const double b = S[0] * d[0] + S[1] * d[1];
    const double c = (S[0] * S[0] + S[1] * S[1]) - Rm * Rm;
    const double disc = b * b - a * c;
    if (!(disc > 0.0)) return r;
    const double sq = sqrt(disc);
    double l0 = (-b - sq) / a, l1 = (-b + sq) / a;
    const double zh = 0.5 * (double)g.nz * dl;
    if (d[2] != 0.0) {
        const double ta = -zh / d[2], tb = zh / d[2];
        l0 = fmax(l0, fmin(ta, tb));
        l1 = fmin(l1, fmax(ta, tb));
    }
    if (!(l1 > l0)) return r;
    const double cen[3] = {(double)g.cx, (double)g.cy, (double)g.cz};
    const int nn[3] = {g.nx, g.ny, g.nz};
    float tmax = (float)(l1 - l0);
#pragma unroll
    for (int ax = 0; ax < 3; ++ax) {
        const double pe = (S[ax] + l0 * d[ax]) / dl + cen[ax];
        double fi = floor(pe + 0.5);
        if (fi < 0.0) fi = 0.0;
        if (fi > (double)(nn[ax] - 1)) fi = (double)(nn[ax] - 1);
        r.idx[ax] = (int)fi;
        if (d[ax] > 0.0) {
            r.step[ax] = 1;
            r.first[ax] = (float)fmax(((fi + 0.5 - cen[ax]) * dl - S[ax]) / d[ax] - l0, 0.0) + 0.0f;
            r.inc[ax] = (float)(dl / d[ax]);
            tmax = fminf(tmax, fmaf((float)(nn[ax] - 1 - r.idx[ax]), r.inc[ax], r.first[ax]));
        } else if (d[ax] < 0.0) {
            r.step[ax] = -1;
            r.first[ax] = (float)fmax(((fi - 0.5 - cen[ax]) * dl - S[ax]) / d[ax] - l0, 0.0) + 0.0f;
            r.inc[ax] = (float)(-dl / d[ax]);
            tmax = fminf(tmax, fmaf((float)r.idx[ax], r.inc[ax], r.first[ax]));
        } else {
            r.step[ax] = 0;
            r.first[ax] = 3.0e38f;
            r.inc[ax] = 0.0f;
        }
    }
    r.tmax = tmax;
    r.ok = true;
    return r;
}

// Per-ray traversal used by the transpose (MODE 1, scatter chord*gval) and
// the segment counter (MODE 2): t from 0 to tmax; the next segment ends at
// the nearest crossing; ties step every tied axis.  The index range test is
// kept as a second guard for the scatter addresses.
template <int MODE>
__device__ __forceinline__ void sid_trace(const DevGeom& g, const SidRay& r, float* __restrict__ scatter, float gval,
                                          unsigned* nseg) {
    float tx = r.first[0], ty = r.first[1], tz = r.first[2];
    float cx = 0.0f, cy = 0.0f, cz = 0.0f;
    int i = r.idx[0], j = r.idx[1], k = r.idx[2];
    const int64_t sy = g.nx, sz = (int64_t)g.nx * g.ny;
    float t = 0.0f;
    int guard = g.nx + g.ny + g.nz + 4;
    unsigned cnt = 0;
    while (t < r.tmax && guard-- > 0) {
        const float tn = fminf(tx, fminf(ty, tz));
        const float te = fminf(tn, r.tmax);
        const float chord = te - t;
        const int64_t o = (int64_t)i + sy * j + sz * k;
        if (MODE == 1) unsafeAtomicAdd(scatter + o, chord * gval);
        if (MODE == 2) cnt += chord > 0.0f ? 1u : 0u;
        t = te;
        if (tx == tn) { i += r.step[0]; cx += 1.0f; tx = fmaf(cx, r.inc[0], r.first[0]); }
        if (ty == tn) { j += r.step[1]; cy += 1.0f; ty = fmaf(cy, r.inc[1], r.first[1]); }
        if (tz == tn) { k += r.step[2]; cz += 1.0f; tz = fmaf(cz, r.inc[2], r.first[2]); }
        if ((unsigned)i >= (unsigned)g.nx || (unsigned)j >= (unsigned)g.ny || (unsigned)k >= (unsigned)g.nz) break;
    }
    if (MODE == 2) *nseg = cnt;
}

// Wave-wide minimum / maximum of an int (wave64 butterfly).
__device__ __forceinline__ int wave_min(int v) {
    for (int off = 32; off > 0; off >>= 1) v = min(v, __shfl_xor(v, off, 64));
    return v;
}
__device__ __forceinline__ int wave_max(int v) {
    for (int off = 32; off > 0; off >>= 1) v = max(v, __shfl_xor(v, off, 64));
    return v;
}

// Volume reads by linear element index.  BUF: a buffer resource with a
// 32-bit byte offset (volumes below 4 GiB); an offset past the end reads 0.
// Otherwise a plain global load.
template <typename TV, bool BUF> struct VolReader;
template <typename TV> struct VolReader<TV, false> {
    const TV* p;
    float inv;
    __device__ __forceinline__ float operator()(unsigned lin) const { return Storage<TV>::load(p, lin, inv); }
};
template <> struct VolReader<float, true> {
    __amdgpu_buffer_rsrc_t r;
    float inv;
    __device__ __forceinline__ float operator()(unsigned lin) const {
        return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, lin * 4u, 0, 0));
    }
};
template <typename TV, bool BUF>
__device__ __forceinline__ VolReader<TV, BUF> make_reader(const TV* p, unsigned bytes, float inv) {
    VolReader<TV, BUF> v;
    if constexpr (BUF) {
        v.r = buffer_rsrc(p, bytes);
    } else {
        v.p = p;
        (void)bytes;
    }
    v.inv = inv;
    return v;
}

// Minimum and maximum of two times of the walk.  Every such time is +0 or
// positive (the first crossings are clamped at +0, increments and tmax are
// positive), and non-negative floats order as their bit patterns do as
// unsigned integers, so one integer min / max gives the exact result without
// the NaN canonicalisation of fminf / fmaxf.
__device__ __forceinline__ float min_nn(float a, float b) {
    return __builtin_bit_cast(float, min(__builtin_bit_cast(uint32_t, a), __builtin_bit_cast(uint32_t, b)));
}
__device__ __forceinline__ float max_nn(float a, float b) {
    return __builtin_bit_cast(float, max(__builtin_bit_cast(uint32_t, a), __builtin_bit_cast(uint32_t, b)));
}

// Per-lane state of the general forward traversal: next crossing and
// crossings taken per axis, the linear index of the current voxel, the
// running sum.
struct SidState {
    float tn[3], cnt[3];
    unsigned lin;
    unsigned dlin[3];
    float t, acc;
    bool live;
};

template <int AX>
__device__ __forceinline__ void sid_advance(SidState& s, const SidRay& r) {
    s.cnt[AX] += 1.0f;
    s.tn[AX] = fmaf(s.cnt[AX], r.inc[AX], r.first[AX]);
    s.lin += s.dlin[AX];
}

// General step (waves without a common slab axis): the next segment ends at
// the nearest crossing; ties step every tied axis.
template <typename RD>
__device__ __forceinline__ void sid_step(SidState& s, const SidRay& r, const RD& rd) {
    const float tn = min_nn(s.tn[0], min_nn(s.tn[1], s.tn[2]));
    const float te = min_nn(tn, r.tmax);
    s.acc = fmaf(te - s.t, rd(s.lin), s.acc);
    s.t = te;
    if (s.tn[0] == tn) sid_advance<0>(s, r);
    if (s.tn[1] == tn) sid_advance<1>(s, r);
    if (s.tn[2] == tn) sid_advance<2>(s, r);
    s.live = s.t < r.tmax;
}

// Column walk on the z-column copy (proj_copy.hpp: z varies fastest).  A lane walks
// the in-plane cells (x, y) its ray crosses, one per iteration; a cell's
// segments are
//   [t, c1] V(z),  [c1, te] V(z + dz)
// with te the nearer of the cell's x and y crossing and tmax and c1 the z
// crossing (te when it comes later).  The wave was admitted only if, for each
// of its rays, consecutive z crossings are spaced more than two ulps of tmax
// beyond the longest stretch in one cell, so a cell holds at most one.  These
// are the segments of the general step in the same order; an absent one has
// zero length and adds exactly 0 (x and y crossed at once are two steps with an
// empty cell between them).
//
// Why columns: all rows of a detector column cross the same in-plane cells
// (the source, the column and the z axis span a vertical plane), so the lanes
// of a wave -- rows of one column, or of a few neighbouring ones -- read one
// contiguous run of z per cell.  A gather of 8 or 16 bytes a lane takes the
// texture path 4 lanes a cycle (16.5 cycles a wave measured), a second pass for
// each four lanes that straddle two rows of the copy, and 2 cycles per 128-byte
// line from L2.  With lanes along the detector rows, four lanes straddle z rows
// often and a wave touches 10-13 lines: 31 cycles per 16-byte gather of a slab's
// (B, z) quad, 46.1 ms at 512^3 / 512 views.  Along the columns a cell's
// 8 bytes take two to four lines, from one copy of the volume (the quads took
// four volumes).
constexpr uint32_t kSidOutside = 0xfffffff0u;

// Reads V(z), V(z + 1) of a column.  BUF: by byte offset through a buffer
// resource; an offset past its end reads 0 without touching memory.
// Otherwise by element index.  FP32 elements are single voxels, 16-bit ones
// (z, z + 1) pairs, one 4-byte word.
template <typename TV, bool BUF> struct ColumnReader {
    static constexpr uint32_t kUnit = BUF ? 4u : 1u;
    static constexpr uint32_t kIdle = BUF ? kSidOutside : 0u;
    static constexpr bool kZeroIdle = BUF;
    __amdgpu_buffer_rsrc_t r;
    const uint32_t* p;
    __device__ __forceinline__ float2 operator()(uint32_t o) const {
        if constexpr (sizeof(TV) == 4) {
            uint32_t w[2];
            if constexpr (BUF) {
                const auto v = __builtin_amdgcn_raw_buffer_load_b64(r, (int)o, 0, 0);
                w[0] = v[0];
                w[1] = v[1];
            } else {
                __builtin_memcpy(w, p + o, 8);
            }
            return make_float2(__uint_as_float(w[0]), __uint_as_float(w[1]));
        } else {
            const uint32_t w = BUF ? __builtin_amdgcn_raw_buffer_load_b32(r, (int)o, 0, 0) : p[o];
            return make_float2(Unpack16<TV>::lo(w), Unpack16<TV>::hi(w));
        }
    }
    // one voxel (the general step)
    __device__ __forceinline__ float one(uint32_t o) const { return (*this)(o).x; }
};

// The ray as its lane walks it; e: offset of V(z), or of V(z - 1) when the ray
// goes down in z (the pair below), dX, dY, dZ its signed steps.
struct ColumnRay {
    float fx, ix, fy, iy, fz, iz, tmax;
    uint32_t e, dX, dY, dZ;
    bool down;
};

// DIR: 0 / 1 when every ray of the wave goes up / down in z, 2 when they differ.
template <int DIR, typename CR>
__device__ __forceinline__ float sid_walk_columns(const ColumnRay& r, const CR& rd, int trips) {
    float tx = r.fx, ty = r.fy, tz = r.fz, k = 0.0f, cx = 0.0f, cz = 0.0f, t = 0.0f, acc = 0.0f;
    uint32_t e = r.e;
    // A lane past its last cell has t = tmax: every later time lies at tmax or
    // beyond, so its segments have no length, and its loads go to kIdle, which
    // reads 0 (by index: a voxel, which is masked).
    struct Cell {
        float d1, d2;
        float2 v;
    };
    auto next = [&]() __attribute__((always_inline)) {
        Cell c;
        const bool live = t < r.tmax;
        c.v = rd(live ? e : CR::kIdle);
        if constexpr (!CR::kZeroIdle) c.v = live ? c.v : make_float2(0.0f, 0.0f);
        const float te = min_nn(min_nn(tx, ty), r.tmax);
        const float c1 = min_nn(tz, te);
        c.d1 = c1 - t;
        c.d2 = te - c1;
        const bool sx = tx <= ty, sz = tz <= te;
        e += (sx ? r.dX : r.dY) + (sz ? r.dZ : 0u);
        t = te;
        k += 1.0f;
        cx += sx ? 1.0f : 0.0f;
        cz += sz ? 1.0f : 0.0f;
        tx = fmaf(cx, r.ix, r.fx);
        ty = fmaf(k - cx, r.iy, r.fy);
        tz = fmaf(cz, r.iz, r.fz);
        return c;
    };
    auto add = [&](const Cell& c) __attribute__((always_inline)) {
        const bool down = DIR == 2 ? r.down : DIR == 1;
        acc = fmaf(c.d1, down ? c.v.y : c.v.x, acc);
        acc = fmaf(c.d2, down ? c.v.x : c.v.y, acc);
    };
    // kAhead cells are loaded before the oldest is summed
    constexpr int kAhead = 3;
    Cell q[kAhead];
#pragma unroll
    for (int j = 0; j < kAhead; ++j) q[j] = next();
    for (int i = 0; i < trips; i += kAhead) {
#pragma unroll
        for (int j = 0; j < kAhead; ++j) {
            add(q[j]);
            q[j] = next();
        }
    }
    return acc;
}

// Forward clean Siddon.  Each lane takes the segments of the per-ray
// traversal (same operations, same order), so results are bit-identical to
// it.  What changes is the schedule and the memory layout (see above).
// A wave is `rows` (sid_wave_rows) detector rows of 64 / rows columns; a
// workgroup is these cells in kProjViews consecutive views, whose rays run
// through nearly the same columns of the volume at the same time (512^3 / 512
// views: 33.1 ms with four neighbouring column groups of one view per
// workgroup, 31.7 ms with four views; 1024^3 / 720 views, bound by the lines
// that miss L2: 238 and 182 ms).  Grid: x = column group, y = view group, z =
// row group: the chip works through every view of one row band before the
// next band, whose rays stay in a z band of the volume.  Workgroups go to the
// XCDs round robin; proj_group gives each XCD neighbouring column groups, so that
// its L2 meets the columns of one view again in the next ones (512^3: 38.1 ms
// without it, at four columns of one view per workgroup).
template <typename TV, typename TS, bool BUF>
__device__ __forceinline__ void siddon_tile(const DevGeom& g, const uint32_t* __restrict__ cols, ProjPlanes zp, float vol_inv,
                                            TS* __restrict__ sino, float sino_scale, int rows, int bx, int pg, int bz) {
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int per = 64 / rows;  // columns of a wave
    const int p = pg * kProjViews + wv;
    const int m = bx * per + lane / rows;
    const int n = bz * rows + lane % rows;
    const bool inside = p < g.nphi && m < g.nu && n < g.nv;
    if (proj_rows_miss(g, 0.5 * (double)g.nx * (double)g.delta, 0.5 * (double)g.nz * (double)g.delta, bz * rows, rows)) {
        if (inside) Storage<TS>::store(sino, (size_t)m + (size_t)g.nu * ((size_t)n + (size_t)g.nv * p), 0.0f, sino_scale);
        return;
    }
    SidRay r{};
    if (inside) r = sid_setup(g, p, m, n);
    const bool ok = r.ok && r.tmax > 0.0f;
    // The z crossings of the ray are spaced farther apart than the longest
    // stretch in one cell, by more than two ulps of tmax; else the wave takes
    // the general step.  The crossings of x (y) are ix (iy) apart, but the first
    // may come later: a FOV entry outside a grid narrower than the FOV is
    // clamped to the border voxel.
    const float big = 3.0e38f;
    const float ix = r.step[0] ? r.inc[0] : big, iy = r.step[1] ? r.inc[1] : big, iz = r.step[2] ? r.inc[2] : big;
    const float cell = fminf(fminf(fmaxf(ix, r.first[0]), fmaxf(iy, r.first[1])), r.tmax);
    const bool walk = __ballot(ok && !(iz > cell + 1.0e-6f * r.tmax)) == 0ull;
    const int ny = g.ny, nz = g.nz;
    const uint32_t pz = zcol_pitch(zp.nz, sizeof(TV)), py = pz * (uint32_t)ny;
    using CR = ColumnReader<TV, BUF>;
    constexpr uint32_t u = CR::kUnit;
    CR rd;
    if constexpr (BUF) rd.r = buffer_rsrc(cols, (uint32_t)(zcol_words(g.nx, ny, zp.nz, sizeof(TV)) * 4u));
    rd.p = cols;
    float acc = 0.0f;
    const uint32_t lin = ok ? (uint32_t)r.idx[0] * py + (uint32_t)r.idx[1] * pz + (uint32_t)(r.idx[2] + 1 - zp.z0) : 0u;
    if (walk) {
        ColumnRay w;
        w.fx = r.first[0];
        w.ix = r.inc[0];
        w.fy = r.first[1];
        w.iy = r.inc[1];
        w.fz = r.first[2];
        w.iz = r.inc[2];
        w.tmax = ok ? r.tmax : 0.0f;
        w.down = r.step[2] < 0;
        w.e = (lin - (w.down ? 1u : 0u)) * u;
        w.dX = (uint32_t)r.step[0] * py * u;
        w.dY = (uint32_t)r.step[1] * pz * u;
        w.dZ = (uint32_t)r.step[2] * u;
        // The wave's iterations, counted once (a scalar loop instead of a vote
        // per cell): the x and y crossings up to tmax, from rounded quotients
        // of two FP32 times that are off by less than one each, with a margin.
        int cells = 0;
        if (ok) {
            const float qx = r.step[0] ? (w.tmax - w.fx) * __builtin_amdgcn_rcpf(w.ix) : 0.0f;
            const float qy = r.step[1] ? (w.tmax - w.fy) * __builtin_amdgcn_rcpf(w.iy) : 0.0f;
            cells = (int)(fminf(fmaxf(qx, 0.0f), 1.0e6f) + fminf(fmaxf(qy, 0.0f), 1.0e6f)) + 6;
        }
        const int trips = __builtin_amdgcn_readfirstlane(min(wave_max(cells), g.nx + ny + 6));
        const bool any_down = __ballot(ok && w.down) != 0ull, any_up = __ballot(ok && !w.down) != 0ull;
        if (!any_down) acc = sid_walk_columns<0>(w, rd, trips);
        else if (!any_up) acc = sid_walk_columns<1>(w, rd, trips);
        else acc = sid_walk_columns<2>(w, rd, trips);
    }
    // A segment of no length takes its voxel times 0, which is not 0 where the voxel
    // is not finite: a sum that is not is taken again by the general step, which
    // reads the voxels on the ray only.
    const bool step = ok && (!walk || !__builtin_isfinite(acc));
    if (__ballot(step) != 0ull) {
        SidState s;
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            s.tn[a] = r.first[a];
            s.cnt[a] = 0.0f;
        }
        // The copy holds fewer than 2^32 elements (checked by the launcher):
        // the index and its signed steps wrap correctly in 32-bit unsigned.
        s.lin = lin * u;
        s.dlin[0] = (uint32_t)r.step[0] * py * u;
        s.dlin[1] = (uint32_t)r.step[1] * pz * u;
        s.dlin[2] = (uint32_t)r.step[2] * u;
        s.t = 0.0f;
        s.acc = 0.0f;
        s.live = step;
        // Every step moves one axis toward the grid exit that bounds tmax;
        // the cap only bounds the loop.
        int guard = g.nx + ny + nz + 4;
        while (s.live && guard-- > 0) sid_step(s, r, [&](unsigned o) { return rd.one(o); });
        if (step) acc = s.acc;
    }
    // 16-bit volumes are read unscaled; the sum is linear in them, so the
    // storage scale applies once here (FP32 storage has no scale).
    if (sizeof(TV) == 2) acc *= vol_inv;
    if (inside) Storage<TS>::store(sino, (size_t)m + (size_t)g.nu * ((size_t)n + (size_t)g.nv * p), acc, sino_scale);
}

// ---------------------------------------------------------------------------
// LDS-staged clean Siddon (FP32 volumes).
//
// The workgroup (32 x 8 detector cells of one view) walks the slabs of A in
// lockstep when all its rays share A and its direction: at iteration k every
// live lane is in slab I + k sA, I the workgroup's first slab.  Iterations go
// in windows of up to kSidWmax slabs [wlo, whi] (fewer when the box is too
// tall for a buffer); for each window the workgroup copies the voxels its
// rays can touch there into LDS (stage_box.hpp: corner rays at the window's
// boundary planes wlo - 1/2 and whi + 1/2, the voxel round(B) and its
// neighbours, likewise in z), and each slab's quad -- the current
// voxel, its B neighbour, its z neighbour and the diagonal one -- is two
// ds_read2_b32 there instead of a gather per lane.  A slab's segments run
// to the nearer and the farther of its B and z crossings and to its end, by
// the crossings of the per-ray traversal in its order: results are
// bit-identical to it.
// A wave whose rays go up and down in z copies its share of rows and keeps
// the barriers, then steps per lane; a window whose box exceeds the buffer
// reads the quads from the volume; a workgroup whose rays do not share A and
// its direction steps per lane on the volume.
constexpr int kSidWmax = 8;  // slabs per window at most

// Per-lane general traversal on the volume (x fastest), as sid_step.
template <typename RD>
__device__ __forceinline__ float sid_general(const SidRay& r, const RD& rd, bool ok, int nx, int ny, int nz) {
    SidState s;
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        s.tn[a] = r.first[a];
        s.cnt[a] = 0.0f;
    }
    const unsigned sy = (unsigned)nx, sz = (unsigned)nx * (unsigned)ny;
    s.lin = ok ? (unsigned)r.idx[0] + sy * (unsigned)r.idx[1] + sz * (unsigned)r.idx[2] : 0u;
    s.dlin[0] = (unsigned)r.step[0];
    s.dlin[1] = (unsigned)r.step[1] * sy;
    s.dlin[2] = (unsigned)r.step[2] * sz;
    s.t = 0.0f;
    s.acc = 0.0f;
    s.live = ok;
    int guard = nx + ny + nz + 4;
    while (s.live && guard-- > 0) sid_step(s, r, rd);
    return s.acc;
}

// The quad of corner (iA, bc, zc) straight from the volume, taps off the
// grid 0: (b, z), (b, z+1), (b+1, z), (b+1, z+1).
template <int A>
__device__ __forceinline__ float4 sid_quad_direct(const float* __restrict__ vol, int nx, int ny, int nz, int iA, int bc,
                                                  int zc) {
    auto at = [&](int b, int z) {
        const int x = A == 0 ? iA : b, y = A == 0 ? b : iA;
        const bool ok = (unsigned)x < (unsigned)nx && (unsigned)y < (unsigned)ny && (unsigned)z < (unsigned)nz;
        return ok ? vol[(size_t)x + (size_t)nx * ((size_t)y + (size_t)ny * (size_t)z)] : 0.0f;
    };
    return make_float4(at(bc, zc), at(bc, zc + 1), at(bc + 1, zc), at(bc + 1, zc + 1));
}

// A window of slabs [wlo, whi] staged as planes wlo .. whi (s.lo = wlo).
// All fields are wave-uniform.
struct SidWindow {
    int wlo, whi;
    StageWin s;
};

// The window that starts at slab `from` in the walk's direction: the largest
// of kSidWmax, 4, 2, 1 slabs whose box fits a buffer.
__device__ __forceinline__ SidWindow sid_plan(const WgCorners& wc, int from, int sAw, int max_nzr) {
    SidWindow w{};
    for (int W = kSidWmax;; W >>= 1) {
        const int wlo = sAw > 0 ? from : from - W + 1, whi = wlo + W - 1;
        const StageBox b = stage_box(wc, (float)wlo - 0.5f, (float)whi + 0.5f, 0.5f, 1, 1);
        w = SidWindow{wlo, whi, stage_window(b, wlo, W, max_nzr)};
        if (w.s.fits || W == 1) break;
    }
    return w;
}

// walks: the wave takes part in the lockstep walk (otherwise it only copies
// its rows and keeps the barriers).  I: the workgroup's first slab, sAw its
// direction along A, trips its iteration count: at iteration k every live
// lane is in slab I + k sAw.  The staging is double buffered: the copy of
// window i + 1 is in flight while the workgroup walks window i, one barrier
// per window.
template <int A, bool ZNEG, int BNEG>
__device__ __forceinline__ float sid_walk_staged(const DevGeom& g, const SidRay& r, bool live, bool walks, int I,
                                                 int sAw, int trips, const float* __restrict__ src, int nBp,
                                                 const float* __restrict__ vol, const WgCorners& wc,
                                                 float* __restrict__ st0, float* __restrict__ st1, int lane, int wv) {
    constexpr int B = 1 - A;
    const int nx = g.nx, ny = g.ny, nz = g.nz;
    const int nA = A == 0 ? nx : ny;
    const size_t src_elems = (size_t)nBp * (size_t)nA * (size_t)nz;
    const int max_nzr = stage_max_rows(nA, nBp);
    const int sB = r.step[B];
    const bool bneg = BNEG == 2 ? sB < 0 : BNEG == 1;
    float tA = r.first[A], tB = r.first[B], tz = r.first[2];
    float cB = 0.0f, cz = 0.0f, cA = 0.0f;
    float t = 0.0f, acc = 0.0f;
    const int lag = live ? abs(r.idx[A] - I) : 0;
    const int b0 = bneg ? r.idx[B] - 1 : r.idx[B], z0 = ZNEG ? r.idx[2] - 1 : r.idx[2];
    // the quad corner's (z, B) part of its offset in the window's buffer, (z - zlo) P + B - blo4
    // with P floats per staged row (set per window); the plane's part is wave-uniform
    int ez = 0;
    const int dB = sB;
    int dZ = 0;
    auto body = [&](const float4 v) {
        // v = (b, z), (b, z+1), (b+1, z), (b+1, z+1) of the block's corner
        const float V0 = bneg ? (ZNEG ? v.w : v.z) : (ZNEG ? v.y : v.x);
        const float Vb = bneg ? (ZNEG ? v.y : v.x) : (ZNEG ? v.w : v.z);
        const float Vz = bneg ? (ZNEG ? v.z : v.w) : (ZNEG ? v.x : v.y);
        const float Vbz = bneg ? (ZNEG ? v.x : v.y) : (ZNEG ? v.z : v.w);
        const bool stepB = tB <= tA, stepZ = tz <= tA;
        const float V1 = tB < tz ? Vb : Vz;
        const float V2 = stepB ? (stepZ ? Vbz : Vb) : (stepZ ? Vz : V0);
        const float c3 = min_nn(tA, r.tmax);
        const float c1 = min_nn(min_nn(tB, tz), c3), c2 = min_nn(max_nn(tB, tz), c3);
        acc = fmaf(c1 - t, V0, acc);
        acc = fmaf(c2 - c1, V1, acc);
        acc = fmaf(c3 - c2, V2, acc);
        t = c3;
        ez += (stepB ? dB : 0) + (stepZ ? dZ : 0);
        cB += stepB ? 1.0f : 0.0f;
        cz += stepZ ? 1.0f : 0.0f;
        tB = fmaf(cB, r.inc[B], r.first[B]);
        tz = fmaf(cz, r.inc[2], r.first[2]);
        cA += 1.0f;
        tA = fmaf(cA, r.inc[A], r.first[A]);
        live = t < r.tmax;
    };
    const int last = I + sAw * (trips - 1);  // the slab of the last iteration
    SidWindow cur = sid_plan(wc, I, sAw, max_nzr);
    if (cur.s.fits) stage_copy(src, src_elems, nA, nBp, nz, cur.s, st0, lane, wv);
    // One window: window `cur` is in `stage`, the next one is copied into
    // `other`; false after the last window.  The windows alternate between
    // the two LDS arrays and each call names them directly, so the compiler
    // knows that the copy in flight does not write what the reads read and
    // does not wait for it before them.
    auto window = [&](const float* __restrict__ stage, float* __restrict__ other) __attribute__((always_inline)) {
        // this wave's copies of window `cur` have landed; every wave is done with the other buffer
        __builtin_amdgcn_s_waitcnt(0);
        __syncthreads();
        const int from = sAw > 0 ? cur.whi + 1 : cur.wlo - 1;
        const bool more = sAw > 0 ? from <= last : from >= last;
        SidWindow nxt = cur;
        if (more) {
            nxt = sid_plan(wc, from, sAw, max_nzr);
            if (nxt.s.fits) stage_copy(src, src_elems, nA, nBp, nz, nxt.s, other, lane, wv);
        }
        if (walks) {
            // iterations of the window's slabs, in the walk's order
            const int k0 = sAw > 0 ? cur.wlo - I : I - cur.whi;
            const int k1 = min(trips, k0 + (cur.whi - cur.wlo + 1));
            if (cur.s.fits) {
                const int P = 4 * cur.s.nch, ps = cur.s.nzr * P;
                dZ = r.step[2] * P;
                // the current quad corner, from the crossings taken so far
                const int bc = b0 + sB * (int)cB, zc = z0 + r.step[2] * (int)cz;
                ez = (zc - cur.s.zlo) * P + (bc - cur.s.blo4);
                for (int outer = k0; outer < k1; ++outer) {
                    if (live && outer >= lag) {
                        const int slab = I + sAw * outer;
                        const float* q = stage + (slab - cur.wlo) * ps + ez;
                        body(make_float4(q[0], q[P], q[1], q[P + 1]));
                    }
                }
            } else {
                for (int outer = k0; outer < k1; ++outer) {
                    if (live && outer >= lag) {
                        const int iA = I + sAw * outer;
                        const int bc = b0 + sB * (int)cB, zc = z0 + r.step[2] * (int)cz;
                        body(sid_quad_direct<A>(vol, nx, ny, nz, iA, bc, zc));
                    }
                }
            }
        }
        cur = nxt;
        return more;
    };
    while (window(st0, st1) && window(st1, st0)) {
    }
    return acc;
}

template <int A, bool ZNEG>
__device__ __forceinline__ float sid_walk_staged_b(const DevGeom& g, const SidRay& r, bool live, bool walks, int I,
                                                   int sAw, int trips, const float* __restrict__ src, int nBp,
                                                   const float* __restrict__ vol, const WgCorners& wc,
                                                   float* __restrict__ st0, float* __restrict__ st1, int lane,
                                                   int wv) {
    const bool pos_all = __ballot(live && r.step[1 - A] < 0) == 0ull;
    const bool neg_all = __ballot(live && r.step[1 - A] >= 0) == 0ull;
    if (pos_all) return sid_walk_staged<A, ZNEG, 0>(g, r, live, walks, I, sAw, trips, src, nBp, vol, wc, st0, st1, lane, wv);
    if (neg_all) return sid_walk_staged<A, ZNEG, 1>(g, r, live, walks, I, sAw, trips, src, nBp, vol, wc, st0, st1, lane, wv);
    return sid_walk_staged<A, ZNEG, 2>(g, r, live, walks, I, sAw, trips, src, nBp, vol, wc, st0, st1, lane, wv);
}

// Forward clean Siddon with LDS-staged quads (FP32 volume `vol`).  volT: its
// y-fastest copy with rows of nyp floats, volP: rows of nxp floats along x
// (the volume itself when nxp = nx); nxp, nyp are nx, ny rounded up to
// multiples of four.  Grid: x = column group, y = view, z = row group.
template <typename TS>
__global__ __launch_bounds__(BX* BY, 5) void siddon_staged_kernel(DevGeom g, const float* __restrict__ vol,
                                                                 const float* __restrict__ volT,
                                                                 const float* __restrict__ volP, int nxp, int nyp,
                                                                 unsigned vol_bytes, TS* __restrict__ sino,
                                                                 float sino_scale) {
    __shared__ float st0[kSlotFloats];
    __shared__ float st1[kSlotFloats];
    __shared__ int wsh[4][3];
    const int tid = threadIdx.y * BX + threadIdx.x;
    const int lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int bx = blockIdx.x, p = blockIdx.y, bz = blockIdx.z;
    const int m = bx * BX + threadIdx.x;
    const int n = bz * BY + threadIdx.y;
    const bool inside = m < g.nu && n < g.nv;
    SidRay r;
    r.ok = false;
    if (inside) r = sid_setup(g, p, m, n);
    const bool ok = r.ok && r.tmax > 0.0f;
    // The ray's slab axis and direction: the crossings of the other axes are spaced
    // farther apart than this one's by more than two ulps of tmax, so a slab holds at
    // most one of each; -1 where neither x nor y is one.  A ray that enters a FOV wider
    // than the grid outside it walks along the border voxels until it gets there, away
    // from its own place, which is what is staged: its first crossing comes late.
    int code = -1;
    if (ok) {
        const float big = 3.0e38f, margin = 1.0e-6f * r.tmax;
        const float ix = r.step[0] ? r.inc[0] : big, iy = r.step[1] ? r.inc[1] : big;
        const float iz = r.step[2] ? r.inc[2] : big;
        const bool late = r.first[0] > ix || r.first[1] > iy;
        if (!late && r.step[0] != 0 && iy > ix + margin && iz > ix + margin)
            code = r.step[0] > 0 ? 0 : 1;
        else if (!late && r.step[1] != 0 && ix > iy + margin && iz > iy + margin)
            code = r.step[1] > 0 ? 2 : 3;
    }
    const unsigned long long okmask = __ballot(ok);
    int wmode = 4;  // 0..3: the wave's common code; -1: codes differ; 4: no ray
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
    const int nx = g.nx, ny = g.ny, nz = g.nz;
    float acc = 0.0f;
    if (mode == -1) {
        if (vol_bytes != 0u)
            acc = sid_general(r, make_reader<float, true>(vol, vol_bytes, 1.0f), ok, nx, ny, nz);
        else
            acc = sid_general(r, make_reader<float, false>(vol, 0u, 1.0f), ok, nx, ny, nz);
    } else if (mode != 4) {
        const int A = mode < 2 ? 0 : 1;
        const int sAw = (mode & 1) ? -1 : 1;
        const int nA = A == 0 ? nx : ny;
        // the workgroup's first slab I, then its iteration count: the crossings of A up to tmax from there
        const int iA = ok ? r.idx[A] : 0;
        int I = sAw > 0 ? wave_min(ok ? iA : 0x7fffffff) : wave_max(ok ? iA : -0x7fffffff);
        __syncthreads();  // every wave has read wsh[*][0]
        if (lane == 0) wsh[wv][1] = I;
        __syncthreads();
#pragma unroll
        for (int k = 0; k < 4; ++k) I = sAw > 0 ? min(I, wsh[k][1]) : max(I, wsh[k][1]);
        I = __builtin_amdgcn_readfirstlane(I);
        int span = 0;
        if (ok) {
            const int lag = abs(iA - I);
            const float kf = ceilf((r.tmax - r.first[A]) * __builtin_amdgcn_rcpf(r.inc[A]));
            span = lag + (int)fminf(fmaxf(kf, 0.0f), 1.0e6f) + 3;
        }
        span = wave_max(span);
        if (lane == 0) wsh[wv][2] = span;
        __syncthreads();
        int trips = 0;
#pragma unroll
        for (int k = 0; k < 4; ++k) trips = max(trips, wsh[k][2]);
        trips = __builtin_amdgcn_readfirstlane(min(trips, nA + 2));
        // one z direction per wave, or none (then the wave steps per lane after the windows)
        const bool zneg_all = __ballot(ok && r.step[2] > 0) == 0ull;
        const bool zpos_all = __ballot(ok && r.step[2] < 0) == 0ull;
        const bool walks = zneg_all || zpos_all;
        const int mlo = bx * BX, mhi = min(bx * BX + BX - 1, g.nu - 1);
        const int nlo = bz * BY, nhi = min(bz * BY + BY - 1, g.nv - 1);
        const WgCorners wc = wg_corners(g, A, p, mlo, mhi, nlo, nhi);
        const float* src = A == 0 ? volT : volP;
        const int nBp = A == 0 ? nyp : nxp;
        const bool zneg = zneg_all && !zpos_all;
        if (A == 0) {
            acc = zneg ? sid_walk_staged_b<0, true>(g, r, ok, walks, I, sAw, trips, src, nBp, vol, wc, st0, st1, lane, wv)
                       : sid_walk_staged_b<0, false>(g, r, ok, walks, I, sAw, trips, src, nBp, vol, wc, st0, st1, lane, wv);
        } else {
            acc = zneg ? sid_walk_staged_b<1, true>(g, r, ok, walks, I, sAw, trips, src, nBp, vol, wc, st0, st1, lane, wv)
                       : sid_walk_staged_b<1, false>(g, r, ok, walks, I, sAw, trips, src, nBp, vol, wc, st0, st1, lane, wv);
        }
        if (!walks) {
            if (vol_bytes != 0u)
                acc = sid_general(r, make_reader<float, true>(vol, vol_bytes, 1.0f), ok, nx, ny, nz);
            else
                acc = sid_general(r, make_reader<float, false>(vol, 0u, 1.0f), ok, nx, ny, nz);
        }
    }
    if (inside) Storage<TS>::store(sino, (size_t)m + (size_t)g.nu * ((size_t)n + (size_t)g.nv * p), acc, sino_scale);
}

template <typename TV, typename TS, bool BUF>
__global__ __launch_bounds__(64 * kProjViews) void siddon_kernel(DevGeom g, const uint32_t* __restrict__ cols, ProjPlanes zp,
                                                     float vol_inv, TS* __restrict__ sino, float sino_scale, int rows) {
    siddon_tile<TV, TS, BUF>(g, cols, zp, vol_inv, sino, sino_scale, rows,
                             proj_group(blockIdx.x, gridDim.x, blockIdx.y, gridDim.y, blockIdx.z), blockIdx.y, blockIdx.z);
}

// Shared launch: tiles are the single-problem grid's workgroups (column
// group fastest, then view, then row group); FP32 or BF16 (kItemBF16) z-column
// copies, FP32 sinograms.
__global__ __launch_bounds__(64 * kProjViews) void siddon_batch_kernel(const BatchTable* __restrict__ t, uint32_t* __restrict__ next) {
    TOMO_BATCH_CLAIMED(t, next) {
        const BatchItem& it = t->item[batch_find(t, tile)];
        const uint32_t local = tile - it.begin;
        const uint32_t rest = local / it.gx;
        const int by = (int)(rest % it.gy), bz = (int)(rest / it.gy);
        const int bx = proj_group(local % it.gx, it.gx, (uint32_t)by, it.gy, (uint32_t)bz);
        const bool bf = (it.flags & kItemBF16) != 0;
        const bool buf = zcol_words(it.g.nx, it.g.ny, it.planes.nz, bf ? 2 : 4) * 4u < kSidOutside;
        const int rows = 1 << (it.flags >> kItemRowsShift);
        const uint32_t* cols = (const uint32_t*)it.in;
        using BF = __hip_bfloat16;
        if (bf && buf)
            siddon_tile<BF, float, true>(it.g, cols, it.planes, 1.0f, (float*)it.out, 1.0f, rows, bx, by, bz);
        else if (bf)
            siddon_tile<BF, float, false>(it.g, cols, it.planes, 1.0f, (float*)it.out, 1.0f, rows, bx, by, bz);
        else if (buf)
            siddon_tile<float, float, true>(it.g, cols, it.planes, 1.0f, (float*)it.out, 1.0f, rows, bx, by, bz);
        else
            siddon_tile<float, float, false>(it.g, cols, it.planes, 1.0f, (float*)it.out, 1.0f, rows, bx, by, bz);
    }
}

// ---------------------------------------------------------------------------
// Transpose of the clean Siddon as a gather: f(i,j,k) = sum over rays of chord
// times g, every voxel summed by one lane, written once.
//
// In terms of tau, the fraction of the way from the source to the detector
// cell, all rows n of a detector column m run over the same in-plane line:
// x(tau) = Sx + tau rx, y(tau) = Sy + tau ry, z(tau) = tau t_n.  So the stretch
// [tau0, tau1] that column m spends over the column (i, j) of voxels is found
// once per (view, m) for all z, and a ray's chord in voxel k is its length from
// source to cell times the part of that stretch in which z(tau) lies between the
// voxel's planes.  A wave owns the voxel column: its lanes first find the
// stretches of 64 views at a time, one view each, in FP64 (the columns m whose
// lines can meet it are those between the projections of its corners), then it
// takes them one by one, a lane per voxel (K of them, 64 apart), over the rows
// that can meet it.  The rows of a lane are read with one 16-byte load from a
// copy of the sinogram with v fastest, already times the ray's length.
//
// VALU issue bounds it: about 13 cycles a row, 2-3 rows a voxel, 1.3 columns a
// view.  256^3 / 256 views: 5.6 ms (6.3 without the bound of 64 registers, which
// spills some of the FP64 part; 11.6 with one 16-byte load in flight a lane),
// rel-L2 8e-8 off 64 bits; scattering the chords with FP32 atomics from one
// lane per ray took 126 ms and was 6e-7 off.  (LDS accumulation is no way
// out: ds_add_f32 took 190 cycles a wave instruction.)
constexpr int kSidTWaves = 8;  // waves per workgroup: voxel columns next to each other in x
constexpr int kSidTPad = 4;    // zero rows at both ends of a column of the sinogram copy

__host__ __device__ inline size_t sid_t_pitch(int nv) { return (size_t)nv + 2 * kSidTPad; }

// out[(p nu + m) pitch + pad + n] = g(p, n, m) |D - S|, 0 for the pad rows; one
// 64 x 64 tile of one view per workgroup, tiles in (u, v, view) order.
template <typename TS>
__global__ __launch_bounds__(256) void siddon_t_prepare_kernel(DevGeom g, const TS* __restrict__ sino, float sino_inv,
                                                               float* __restrict__ out) {
    __shared__ float tile[64][65];
    const int pitch = (int)sid_t_pitch(g.nv);
    const uint32_t gx = (uint32_t)(g.nu + 63) / 64, gy = (uint32_t)(pitch + 63) / 64;
    const uint32_t bx = blockIdx.x % gx, rest = blockIdx.x / gx, by = rest % gy;
    const size_t p = rest / gy;
    const int tx = threadIdx.x & 63, ty = threadIdx.x >> 6;
    const int m = (int)bx * 64 + tx, r0 = (int)by * 64;
    const double s = ((double)m - (double)g.cu) * (double)g.du;
    for (int r = ty; r < 64; r += 4) {
        const int n = r0 + r - kSidTPad;
        float v = 0.0f;
        if (m < g.nu && n >= 0 && n < g.nv) {
            const double t = ((double)n - (double)g.cv) * (double)g.dv;
            const float gv = Storage<TS>::load(sino, (size_t)m + (size_t)g.nu * ((size_t)n + (size_t)g.nv * p), sino_inv);
            v = (float)((double)gv * sqrt((g.fdd * g.fdd + s * s) + t * t));
        }
        tile[r][tx] = v;
    }
    __syncthreads();
    const int row = r0 + tx;
    if (row < pitch)
        for (int r = ty; r < 64; r += 4) {
            const int mo = (int)bx * 64 + r;
            if (mo < g.nu) out[(p * (size_t)g.nu + mo) * pitch + row] = tile[tx][r];
        }
}

// A detector column's line along an axis (its direction's other component r is 0 but
// for the rounding of the view's cosine or sine) has one coordinate there, S + tau
// r at the isocentre.  Where that lies on a plane between two voxels, which of them
// the rays belong to follows from the rounding of the projector's own setup, ray by
// ray: they are left to the per-ray traversal.  kSidBetween: how near, in voxels; more
// than such a line drifts on its way, less than any other lies off a plane.
constexpr double kSidBetween = 1e-5;
__host__ __device__ inline bool sid_line_flat(const DevGeom& g, double r) { return fabs(r) < 1e-9 * g.fdd; }
__host__ __device__ inline double sid_line_at(const DevGeom& g, double S, double r) { return S + g.fod / g.fdd * r; }
// The detector column whose line runs between two rows of voxels in a view, along
// y (x = 0) or x (x = 1), -1 where none does.
__host__ __device__ inline int sid_between_column(const DevGeom& g, const double* vw, int x) {
    const double ca = vw[0], sa = vw[1];
    const double at = rint((x ? -sa / ca : ca / sa) * g.fdd / (double)g.du + (double)g.cu);
    if (!(at >= 0.0 && at < (double)g.nu)) return -1;
    const double s = (at - (double)g.cu) * (double)g.du;
    const double r = x ? sa * g.fdd + s * ca : ca * g.fdd - s * sa;
    if (!sid_line_flat(g, r)) return -1;
    const double pos = sid_line_at(g, x ? -g.fod * sa : -g.fod * ca, r) / (double)g.delta + (double)(x ? g.cy : g.cx) + 0.5;
    const double plane = rint(pos);
    return plane >= 1.0 && plane < (double)(x ? g.ny : g.nx) && fabs(pos - plane) <= kSidBetween ? (int)at : -1;
}

__device__ __forceinline__ double read_lane(double v, int l) {
    const uint64_t b = __builtin_bit_cast(uint64_t, v);
    const uint32_t lo = __builtin_amdgcn_readlane((int)(uint32_t)b, l);
    const uint32_t hi = __builtin_amdgcn_readlane((int)(uint32_t)(b >> 32), l);
    return __builtin_bit_cast(double, (uint64_t)lo | ((uint64_t)hi << 32));
}
__device__ __forceinline__ float read_lane(float v, int l) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l));
}

// views: the np views of `gt`, from view p0; add: to what vol holds.  Grid: x, y =
// (column group, j), z = z block of 64 K voxels.  The rays that enter outside a grid
// narrower than the FOV run along its border rows: those take the views in `parts`, the
// first rows of the grid all but one of them, and add to a cleared volume (256 x 64 x 4,
// 4 rows and 256 views 3.3 ms with one wave a voxel column, 1.5 in parts; 256 x 1 x 1, one
// row and 200 views 5.8 and 0.98).  TIE: an odd number of detector
// rows over an even number of slices: the middle row's rays run along the plane
// between two slices, and belong to the upper one, as the projector's; its height
// is then taken exactly at each row instead of carried on from the first.
template <int K, bool TIE>
__global__ __launch_bounds__(64 * kSidTWaves, 8) void siddon_t_kernel(DevGeom g, const float* __restrict__ gt, int p0,
                                                                   int np, int add, int parts,
                                                                   float* __restrict__ vol) {
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const uint32_t gx = (uint32_t)(g.nx + kSidTWaves - 1) / kSidTWaves;
    const uint32_t tile = tile_index();
    const int ends = min(g.ny, 2), row = (int)(tile / gx) - ends * (parts - 1);
    const int i = (int)(tile % gx) * kSidTWaves + wv, j = row >= 0 ? row : row % ends ? g.ny - 1 : 0;
    if (i >= g.nx || j >= g.ny) return;
    const int kb = (int)blockIdx.z * 64 * K;
    const bool split = parts > 1 && (j == 0 || j == g.ny - 1);
    const int each = split ? (np + parts - 1) / parts : np;
    const int pbegin = row >= 0 ? 0 : ((-1 - row) / ends + 1) * each, pend = min(np, pbegin + each);
    const double dl = (double)g.delta, inf = __builtin_inf();
    // The voxel column's cell in the plane (mm).  The cylinder may be wider than
    // the grid in y (ny < nx): a ray that comes from outside walks along the
    // border row until it reaches the grid, so the border cells reach out to
    // the cylinder for rays that enter on their side.
    const double Rm = 0.5 * (double)g.nx * dl;
    const double xa = ((double)i - 0.5 - (double)g.cx) * dl, xb = ((double)i + 0.5 - (double)g.cx) * dl;
    const double ya = ((double)j - 0.5 - (double)g.cy) * dl, yb = ((double)j + 0.5 - (double)g.cy) * dl;
    const double ylo = j == 0 ? fmin(ya, -Rm) : ya, yhi = j == g.ny - 1 ? fmax(yb, Rm) : yb;
    // a cell inside the cylinder needs no cut by it
    const double fx = fmax(fabs(xa), fabs(xb)), fy = fmax(fabs(ylo), fabs(yhi));
    const bool cut = !(fx * fx + fy * fy < Rm * Rm * (1.0 - 1e-12));
    float acc[K];
#pragma unroll
    for (int c = 0; c < K; ++c) acc[c] = 0.0f;
    // lower plane of the lane's first voxel; the next ones lie zstep apart
    const double zlo = ((double)(kb + lane) - 0.5 - (double)g.cz) * dl, zstep64 = 64.0 * dl;
    const float zl0 = (float)zlo, zstep = (float)zstep64;
    const float zabs =
        (float)(fmax(fabs(((double)kb - 0.5 - (double)g.cz)), fabs((double)min(kb + 64 * K, g.nz) - 0.5 - (double)g.cz)) * dl);
    const int nu = g.nu, nv = g.nv;
    const size_t pitch = sid_t_pitch(nv);
    const float dvf = g.dv, dlf = g.delta, cvf = g.cv;
    for (int pb = pbegin; pb < pend; pb += 64) {
        // ---- one view per lane: the columns m that can meet the cell
        const int pl = pb + lane;
        int m0 = 0, cnt = 0;
        double ca = 1.0, sa = 0.0;
        if (pl < pend) {
            const double* vw = g.view + (size_t)(p0 + pl) * kViewStride;
            ca = vw[0];
            sa = vw[1];
            double u0 = inf, u1 = -inf;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const double X = q & 1 ? xb : xa, Y = q & 2 ? yhi : ylo;
                const double u = (ca * Y - sa * X) * g.fdd / ((ca * X + sa * Y) + g.fod);
                u0 = fmin(u0, u);
                u1 = fmax(u1, u);
            }
            const double eps = 1e-6;
            const double lo = ceil(u0 / (double)g.du + (double)g.cu - eps), hi = floor(u1 / (double)g.du + (double)g.cu + eps);
            m0 = (int)fmax(lo, 0.0);
            cnt = max(0, (int)fmin(hi, (double)(nu - 1)) - m0 + 1);
        }
        const int most = __builtin_amdgcn_readfirstlane(wave_max(cnt));
        for (int q = 0; q < most; ++q) {
            // ---- the stretch of column m0 + q over the cell
            double tau0 = 0.0;
            float span = 0.0f, inv0 = 0.0f, inv1 = 0.0f;
            int rows = 0;
            const int m = m0 + q;
            if (q < cnt) {
                const double s = ((double)m - (double)g.cu) * (double)g.du;
                const double rx = ca * g.fdd - s * sa, ry = sa * g.fdd + s * ca;
                const double Sx = -g.fod * ca, Sy = -g.fod * sa;
                // from the source on; the ray does not end at its detector cell, which may lie
                // inside the volume (fdd < fod + Rm)
                double t0 = 0.0, t1 = inf;
                const double a = rx * rx + ry * ry, b = Sx * rx + Sy * ry, disc = b * b - a * ((Sx * Sx + Sy * Sy) - Rm * Rm);
                bool ok = disc > 0.0;
                if (cut && ok) {
                    const double sq = sqrt(disc);
                    t0 = (-b - sq) / a;
                    t1 = (-b + sq) / a;
                }
                // a line along an axis stays in one row of voxels (kSidBetween)
                if (sid_line_flat(g, rx)) {
                    const double at = sid_line_at(g, Sx, rx);
                    ok = ok && at - xa > kSidBetween * dl && xb - at > kSidBetween * dl;
                } else {
                    const double c0 = (xa - Sx) / rx, c1 = (xb - Sx) / rx;
                    t0 = fmax(t0, fmin(c0, c1));
                    t1 = fmin(t1, fmax(c0, c1));
                }
                if (sid_line_flat(g, ry)) {
                    const double at = sid_line_at(g, Sy, ry);
                    ok = ok && at - ylo > kSidBetween * dl && yhi - at > kSidBetween * dl;
                } else {
                    const double c0 = ((ry > 0.0 ? ylo : ya) - Sy) / ry, c1 = ((ry < 0.0 ? yhi : yb) - Sy) / ry;
                    t0 = fmax(t0, fmin(c0, c1));
                    t1 = fmin(t1, fmax(c0, c1));
                }
                if (ok && t1 > t0) {
                    tau0 = t0;
                    span = (float)(t1 - t0);
                    // rows per mm of height at both ends; the most rows that meet one voxel
                    inv0 = (float)(1.0 / (t0 * (double)g.dv));
                    inv1 = (float)(1.0 / (t1 * (double)g.dv));
                    rows = (int)(dlf * inv0 + zabs * (inv0 - inv1) + 4e-3f) + 1;
                }
            }
            // ---- every voxel of the column, one stretch at a time; the 64 views'
            // parts are summed apart, which keeps the sum's rounding near one
            // of a few dozen terms
            float part[K];
#pragma unroll
            for (int c = 0; c < K; ++c) part[c] = 0.0f;
            for (uint64_t todo = __ballot(rows > 0); todo != 0ull; todo &= todo - 1) {
                const int l = __builtin_ctzll(todo);
                const double step = read_lane(tau0, l) * (double)g.dv;  // z per row at tau0
                const float dt = read_lane(span, l), i0 = read_lane(inv0, l), i1 = read_lane(inv1, l);
                const int most_rows = __builtin_amdgcn_readlane(rows, l), ml = __builtin_amdgcn_readlane(m, l);
                const float* col = gt + ((size_t)(pb + l) * nu + ml) * pitch + kSidTPad;
                const float stepf = (float)step;
                float nf[K];
#pragma unroll
                for (int c = 0; c < K; ++c) {
                    // first row that can reach the voxel
                    const float zl = zl0 + zstep * (float)c;
                    nf[c] = ceilf(fmaf(zl, zl > 0.0f ? i1 : i0, cvf) - 2e-3f);
                }
                for (int left = most_rows; left > 0; left -= 4) {
                    float4 gv[K];
#pragma unroll
                    for (int c = 0; c < K; ++c) {
                        nf[c] = __builtin_amdgcn_fmed3f(nf[c], (float)-kSidTPad, (float)nv);  // within the padded column
                        __builtin_memcpy(&gv[c], col + (int)nf[c], 16);
                    }
#pragma unroll
                    for (int c = 0; c < K; ++c) {
                        // The rows are whole before the branches on their number:
                        // sunk into them, their loads met at a common last one
                        // whose address the compiler (clang 22 of ROCm 7.2) left
                        // undefined for four rows.  An empty statement.
                        asm volatile("" : "+v"(gv[c].x), "+v"(gv[c].y), "+v"(gv[c].z), "+v"(gv[c].w));
                        // height of row nf at tau0 above the voxel's lower plane
                        const double zl = zlo + zstep64 * (double)c;
                        float z0 = (float)fma(step, (double)(nf[c] - cvf), -zl);
                        auto row = [&](float gn, bool first) __attribute__((always_inline)) {
                            if (TIE && !first) z0 = (float)fma(step, (double)(nf[c] - cvf), -zl);
                            const float t = (nf[c] - cvf) * dvf;
                            // The middle row, t = 0, crosses no plane: a height of h ends h 2^100
                            // away.  TIE: a and b are then exact (a power of two), so that the
                            // lower slice's upper plane, at the row's height, ends at 0.
                            const float rt = TIE && t == 0.0f ? 0x1p100f : __builtin_amdgcn_rcpf(t + 1e-30f);
                            // where the row crosses the voxel's planes, from tau0
                            const float a = -z0 * rt, b = fmaf(dlf, rt, a);
                            const float in = fminf(fmaxf(a, b), dt) - fmaxf(fminf(a, b), 0.0f);
                            part[c] = fmaf(in, in > 0.0f ? gn : 0.0f, part[c]);
                            nf[c] += 1.0f;
                            if (!TIE) z0 += stepf;
                        };
                        row(gv[c].x, true);
                        if (left > 1) {
                            row(gv[c].y, false);
                            if (left > 2) {
                                row(gv[c].z, false);
                                if (left > 3) row(gv[c].w, false);
                            }
                        }
                    }
                }
            }
#pragma unroll
            for (int c = 0; c < K; ++c) acc[c] += part[c];
        }
    }
#pragma unroll
    for (int c = 0; c < K; ++c) {
        const int k = kb + 64 * c + lane;
        if (k < g.nz) {
            float* o = vol + ((size_t)i + (size_t)g.nx * ((size_t)j + (size_t)g.ny * k));
            if (split) unsafeAtomicAdd(o, acc[c]);
            else *o = add ? *o + acc[c] : acc[c];
        }
    }
}

// The rays that siddon_t_kernel leaves out, one per thread, added to vol.  Grid: x =
// view, y = row block, z = axis (sid_between_column).
template <typename TS>
__global__ __launch_bounds__(64) void siddon_t_between_kernel(DevGeom g, const TS* __restrict__ sino, float sino_inv,
                                                            float* __restrict__ vol) {
    const int p = blockIdx.x, n = (int)blockIdx.y * 64 + threadIdx.x;
    const int m = sid_between_column(g, g.view + (size_t)p * kViewStride, blockIdx.z);
    if (m < 0 || n >= g.nv) return;
    const float gv = Storage<TS>::load(sino, (size_t)m + (size_t)g.nu * ((size_t)n + (size_t)g.nv * p), sino_inv);
    if (gv == 0.0f) return;
    const SidRay r = sid_setup(g, p, m, n);
    if (r.ok) sid_trace<1>(g, r, vol, gv, nullptr);
}

template <typename TS>
__global__ __launch_bounds__(BX* BY) void siddon_adjoint_kernel(DevGeom g, const TS* __restrict__ sino,
                                                              float sino_inv, float* __restrict__ vol) {
    const int m = blockIdx.x * BX + threadIdx.x;
    const int n = blockIdx.z * BY + threadIdx.y;
    const int p = blockIdx.y;
    if (m >= g.nu || n >= g.nv) return;
    const float gv = Storage<TS>::load(sino, (size_t)m + (size_t)g.nu * ((size_t)n + (size_t)g.nv * p), sino_inv);
    if (gv == 0.0f) return;
    const SidRay r = sid_setup(g, p, m, n);
    if (r.ok) sid_trace<1>(g, r, vol, gv, nullptr);
}

__global__ __launch_bounds__(BX* BY) void siddon_count_kernel(DevGeom g, unsigned long long* total) {
    const int m = blockIdx.x * BX + threadIdx.x;
    const int n = blockIdx.z * BY + threadIdx.y;
    const int p = blockIdx.y;
    unsigned c = 0;
    if (m < g.nu && n < g.nv) {
        const SidRay r = sid_setup(g, p, m, n);
        if (r.ok) sid_trace<2>(g, r, nullptr, 0.0f, &c);
    }
    unsigned long long cc = c;
    for (int off = 32; off > 0; off >>= 1) cc += __shfl_down(cc, off, 64);
    if (((threadIdx.y * BX + threadIdx.x) & 63) == 0) atomicAdd(total, cc);  // first lane of the wave
}

// Reference C path, statement for statement in its arithmetic types.
template <typename TV, typename TS>
__global__ __launch_bounds__(BX* BY) void siddon_compat_kernel(DevGeom g, const TV* __restrict__ vol, float vol_inv,
                                                             TS* __restrict__ sino, float sino_scale) {
    const unsigned long un = blockIdx.x * BX + threadIdx.x;
    const unsigned long vn = blockIdx.z * BY + threadIdx.y;
    const int phi = blockIdx.y;
    const unsigned long nx = g.nx, ny = g.ny, nz = g.nz, nu = g.nu, nv = g.nv;
    if (un >= nu || vn >= nv) return;
    const float fdd = (float)g.fdd, fod = (float)g.fod, dl = g.delta;
    const float xlr = g.cx * dl, ylr = g.cy * dl, zlr = g.cz * dl;
    const float al = g.view_f[2 * phi], be = g.view_f[2 * phi + 1];
    const float xs = xlr + fod * al, ys = ylr + fod * be, zs = zlr;
    const float s = ((float)un - g.cu) * g.du;
    const float t = ((float)vn - g.cv) * g.dv;
    const float xd = (xlr - al * (fdd - fod)) - s * be;
    const float yd = (ylr - be * (fdd - fod)) + s * al;
    const float zd = zlr + t;
    const float L = sqrtf((fdd * fdd + s * s) + t * t);
    const float A = (fdd * fdd + s * s) / (L * L);
    const float B = (-fod * fdd) / L;
    const float C = (float)((double)(fod * fod) - 0.25 * (double)(float)nx * (double)(float)nx * (double)dl * (double)dl);
    const float dlam = B * B - A * C;
    float ray = 0.0f;
    if (dlam > 0.0f) {
        const float lmin = (-B - sqrtf(dlam)) / A;
        const float lmax = (-B + sqrtf(dlam)) / A;
        const float P[3] = {(xs + (lmin * (xd - xs) / L)) / dl, (ys + (lmin * (yd - ys) / L)) / dl,
                            (zs + (lmin * (zd - zs) / L)) / dl};
        const float S[3] = {xs, ys, zs}, D[3] = {xd, yd, zd};
        const unsigned long N[3] = {nx, ny, nz};
        unsigned long idx[3];
        float lam[3], inc[3];
        bool up[3];
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            up[a] = S[a] <= D[a];
            const float pm = up[a] ? (float)((double)P[a] - 0.5) : (float)((double)P[a] + 0.5);
            if (pm < 0.0f) idx[a] = 0;
            else if (pm > (float)(N[a] - 1)) idx[a] = N[a] - 1;
            else idx[a] = up[a] ? (unsigned long)floorf(pm) : (unsigned long)ceilf(pm);
            const float span = D[a] - S[a];
            if (fabsf(span) > dl) {
                const double off = up[a] ? 0.5 : -0.5;
                lam[a] = (float)((double)L * (((double)(float)idx[a] + off) * (double)dl - (double)S[a]) / (double)span);
            } else {
                lam[a] = L;
            }
            inc[a] = (L / fabsf(span)) * dl;
        }
        float lambda = lmin;
        int it = 0;
        const int cap = 4 * (g.nx + g.ny + g.nz) + 16;
        while (lambda <= lmax && it++ < cap) {
            float lk = lam[0];
            if (lam[1] < lk) lk = lam[1];
            if (lam[2] < lk) lk = lam[2];
            const float chord = lk - lambda;
            const unsigned long o = (idx[0] % 256) + (idx[1] % 256) * nx + (idx[2] % 256) * nx * ny;
            const float prod = chord * Storage<TV>::load(vol, o, vol_inv);
            ray = ray + prod;
            lambda = lk;
#pragma unroll
            for (int a = 0; a < 3; ++a) {
                if (lam[a] <= lk) {
                    lam[a] = lam[a] + inc[a];
                    idx[a] = up[a] ? idx[a] + 1 : idx[a] - 1;
                }
            }
        }
    }
    Storage<TS>::store(sino, (un % 256) + (vn % 256) * nu + (unsigned long)phi * nu * nv, ray, sino_scale);
}

}  // namespace

int launch_siddon(const tomo_geom* g, int compat, Buf vol, MutBuf sino, hipStream_t s, const ProjExtra& x) {
    const DevGeom& d = g->dev;
    if (compat && (d.nx != 256 || d.ny != 256 || d.nz != 256 || d.nu > 256 || d.nv > 256))
        return fail(TOMO_ERR_UNSUPPORTED,
                    "compat Siddon is defined for a 256^3 volume and at most 256x256 detector cells "
                    "(the reference indexes modulo 256)");
    // Grid: column group, view, row group (every view of a row band in turn).
    const dim3 grid(ceil_div(d.nu, BX), d.nphi, ceil_div(d.nv, BY));
    const float inv = 1.0f / vol.scale;
    if (compat) {
        TOMO_DISPATCH_STORAGE(vol.dtype, TV, {
            TOMO_DISPATCH_STORAGE(sino.dtype, TS, {
                hipLaunchKernelGGL((siddon_compat_kernel<TV, TS>), grid, dim3(BX, BY), 0, s, d, (const TV*)vol.p, inv,
                                   (TS*)sino.p, sino.scale);
            });
        });
        TOMO_HIP(hipGetLastError());
        return TOMO_OK;
    }
    if (x.staged && vol.dtype == TOMO_F32 && !x.index_reads) {
        // LDS-staged quads, from copies of the volume with rows along y (x
        // slabs) and, when nx is not a multiple of four, along x (y slabs)
        if (g->nvox() >= (1ull << 32))
            return fail(TOMO_ERR_UNSUPPORTED, "volume too large for the 32-bit traversal index of the Siddon projector");
        StageSources src;
        hipError_t le = src.make((const float*)vol.p, d.nx, d.ny, d.nz, s);
        if (le == hipSuccess) {
            const uint64_t vb = (uint64_t)g->nvox() * 4ull;
            const unsigned vol_bytes = vb < (1ull << 32) ? (unsigned)vb : 0u;  // 0: index reads
            TOMO_DISPATCH_STORAGE(sino.dtype, TS, {
                hipLaunchKernelGGL((siddon_staged_kernel<TS>), grid, dim3(BX, BY), 0, s, d, (const float*)vol.p,
                                   (const float*)src.vt, src.rows_x, src.nxp, src.nyp, vol_bytes, (TS*)sino.p,
                                   sino.scale);
            });
            le = hipGetLastError();
        }
        const hipError_t fe = src.release(s);
        TOMO_HIP(le);
        TOMO_HIP(fe);
        return TOMO_OK;
    }
    // z-column copy of the volume (a stream-ordered pool allocation, released
    // after the projection on the same stream)
    const size_t es = vol.dtype == TOMO_F32 ? 4 : 2;
    if (!sid_volume_fits(d.nx, d.ny, d.nz))
        return fail(TOMO_ERR_UNSUPPORTED, "volume too large for the 32-bit traversal index of the Siddon projector");
    ProjCopy zc;
    const ProjPlanes zp = proj_planes(d, 0);
    const size_t words = zcol_words(d.nx, d.ny, zp.nz, es);
    hipError_t le = zc.alloc(words * 4, s, x);
    if (le == hipSuccess) le = launch_zcol(vol.p, (uint32_t*)zc.p, es, d.nx, d.ny, d.nz, zp, s);
    if (le == hipSuccess) {
        const bool buf = words * 4u < kSidOutside && !x.index_reads;
        const int rows = sid_wave_rows(d, zp);
        const dim3 cgrid(proj_groups(d.nu, rows), ceil_div(d.nphi, kProjViews), ceil_div(d.nv, rows));
        TOMO_DISPATCH_STORAGE(vol.dtype, TV, {
            TOMO_DISPATCH_STORAGE(sino.dtype, TS, {
                if (buf)
                    hipLaunchKernelGGL((siddon_kernel<TV, TS, true>), cgrid, dim3(64 * kProjViews), 0, s, d,
                                       (const uint32_t*)zc.p, zp, inv,
                                       (TS*)sino.p, sino.scale, rows);
                else
                    hipLaunchKernelGGL((siddon_kernel<TV, TS, false>), cgrid, dim3(64 * kProjViews), 0, s, d,
                                       (const uint32_t*)zc.p, zp, inv,
                                       (TS*)sino.p, sino.scale, rows);
            });
        });
        le = hipGetLastError();
    }
    const hipError_t fe = zc.release(s);
    TOMO_HIP(le);
    TOMO_HIP(fe);
    return TOMO_OK;
}

hipError_t launch_batch_siddon(BatchTable* t, hipStream_t s) {
    hipLaunchKernelGGL(siddon_batch_kernel, dim3(kBatchGrid), dim3(64 * kProjViews), 0, s, t, t->next);
    return hipGetLastError();
}

// Parts of np views that the border rows of a narrow grid are split into: 64 views
// each, fewer (8 at least) where that leaves fewer than two waves a SIMD.  A border voxel
// has the lines of up to 1 + (nx - ny) / 2 voxels; up to 8 the other rows hide it.
static int sid_t_parts(const DevGeom& d, int np) {
    if (d.nx - d.ny <= 16) return 1;
    int each = 64;
    while (each > 8 && (size_t)std::min(d.ny, 2) * d.nx * ceil_div(d.nz, 256) * ceil_div(np, each) < 2048) each >>= 1;
    return (int)ceil_div(np, each);
}

// The gather needs every voxel column in front of the source in every view (its
// corners project onto the detector plane); a geometry with the source inside
// the cylinder's bounding square scatters.  So do the smallest problems, whose
// few chords cost less than the gather's extra launch and its FP64 chain: 24^3 /
// 16 views 18.8 us against 28.8, 24^3 / 32 views 32.3 and 34.7, 32^3 / 16 views
// 30.0 and 28.6, 32^3 / 32 views 50.0 and 34.6, 64^3 / 64 views 669 and 70; and thin
// ones.  The gather costs 21 ps per voxel column, view and line that may cross it (in
// rounds of 64 views) and 54 ps per line and 64 voxels of it, full or not, and on a narrow
// grid at least the 2.5 us a line and 0.11 more a view of one border wave; the scatter
// 45 ps per ray and slab, or 0.36 us per slab of one, or 65 ns per ray along a border
// voxel.  That picks the faster within 10% at 335 of 344 shapes of 1 to 400 rows and
// slices and ny = nx, and at all but one of 62 narrow ones (128 x 32 x 1, one row and 128
// views: 220 and 282).  Narrow ones scatter from fewer chords, as many fall on a border
// voxel, whose sum in atomics is less exact.  Scatter and gather in us: 256 x
// 256 and 256 views, one slice and row 799 and 1876, 4 and 4 2700 and 1874, 256 slices
// by 4 rows 2983 and 5365, by 12 8700 and 5400, one slice by 256 rows 892 and 1983.
static bool sid_t_gathers(const DevGeom& d) {
    const double half = 0.5 * (double)d.delta * (double)std::max(d.nx, d.ny);
    const double chords = (double)d.nu * d.nv * d.nphi * std::max(d.nx, d.ny);
    if (!(d.fod > 1.01 * std::sqrt(2.0) * half && chords >= 8e5)) return false;
    const CrossingRows c(d);
    const double cols = crossing_columns(d, c);
    const double most = (2 * d.ny < d.nx ? 8e4 : 3e5) / (cols * d.nphi * d.nx);
    if (c.count(d, most) < most) return false;
    const double lines = (double)d.delta * d.fdd / (d.fod * (double)d.du);  // columns per voxel
    const double blocks = ceil_div(d.nz, 64), outside = 0.5 * std::max(0, d.nx - d.ny);  // voxels from the border to the FOV's
    const int parts = sid_t_parts(d, d.nphi);
    const double rounds = 64.0 * ceil_div(d.nphi, 64), each = ceil_div(d.nphi, parts);
    const double grid = d.nx * (double)d.ny * (21.5 * std::ceil(1.41 * lines) * rounds + 54.0 * 1.27 * lines * d.nphi * blocks);
    const double border = 2.0 * d.nx * outside * lines * (21.5 * 1.41 * 64.0 * parts + 54.0 * 1.27 * d.nphi * blocks);
    const double gather = 28.0 + std::max(1e-6 * (grid + border), (2.5 + 0.11 * each) * 1.27 * lines * outside * (d.ny > 1 ? 1.0 : 2.0));
    const double shared = 0.065 * (1.0 - std::min(1.0, (double)d.ny / d.nx)) / (std::min(d.ny, 2) * std::min(d.nz, d.nv));
    const double row = cols * d.nphi * std::max(45e-6 * d.nx, shared), enough = (gather - 16.0) / row;
    return gather - 16.0 <= 0.36 * d.nx || c.count(d, enough) >= enough;
}

template <int K>
static void launch_siddon_t(const DevGeom& d, const float* gt, int p0, int np, int parts, float* vol, hipStream_t s) {
    const size_t rows = (size_t)d.ny + std::min(d.ny, 2) * (parts - 1);
    const dim3 grid = tile_grid(ceil_div(d.nx, kSidTWaves) * rows, 64 * kSidTWaves, ceil_div(d.nz, 64 * K));
    if (d.nv % 2 == 1 && d.nz % 2 == 0)
        hipLaunchKernelGGL((siddon_t_kernel<K, true>), grid, dim3(64 * kSidTWaves), 0, s, d, gt, p0, np, p0 > 0, parts, vol);
    else
        hipLaunchKernelGGL((siddon_t_kernel<K, false>), grid, dim3(64 * kSidTWaves), 0, s, d, gt, p0, np, p0 > 0, parts, vol);
}

int launch_siddon_adjoint(const tomo_geom* g, Buf sino, MutBuf vol, hipStream_t s) {
    if (vol.dtype != TOMO_F32) return fail(TOMO_ERR_UNSUPPORTED, "adjoint output must be F32");
    const DevGeom& d = g->dev;
    const float inv = 1.0f / sino.scale;
    // the sinogram copy, at most 1 GiB of views at a time; without the memory, or in a stream
    // capture, which is left free of allocations, the chords scatter
    const size_t view = (size_t)d.nu * sid_t_pitch(d.nv) * sizeof(float);
    const int chunk = (int)std::min<size_t>((size_t)d.nphi, std::max<size_t>(1, ((size_t)1 << 30) / view));
    float* gt = nullptr;
    if (!stream_captures(s) && sid_t_gathers(d) &&
        hipMallocAsync((void**)&gt, view * (size_t)chunk, s) != hipSuccess) {
        (void)hipGetLastError();
        gt = nullptr;
    }
    if (gt) {
        const int parts = sid_t_parts(d, chunk);
        if (parts > 1) {
            const int rc = launch_fill((float*)vol.p, 0.0f, g->nvox(), s);
            if (rc) {
                (void)hipFreeAsync(gt, s);
                return rc;
            }
        }
        hipError_t e = hipSuccess;
        for (int p0 = 0; p0 < d.nphi && e == hipSuccess; p0 += chunk) {
            const int np = std::min(chunk, d.nphi - p0);
            const size_t skip = (size_t)p0 * d.nu * d.nv;
            const unsigned tiles = ceil_div(d.nu, 64) * ceil_div(sid_t_pitch(d.nv), 64) * (unsigned)np;
            TOMO_DISPATCH_STORAGE(sino.dtype, TS, {
                hipLaunchKernelGGL((siddon_t_prepare_kernel<TS>), dim3(tiles), dim3(256), 0, s, d,
                                   (const TS*)sino.p + skip, inv, gt);
            });
            // K 64-voxel steps per lane: the fewest z blocks that K <= 4 allows
            const int steps = (int)ceil_div(d.nz, 64), blocks = (int)ceil_div(steps, 4);
            switch (ceil_div(steps, blocks)) {
                case 1: launch_siddon_t<1>(d, gt, p0, np, parts, (float*)vol.p, s); break;
                case 2: launch_siddon_t<2>(d, gt, p0, np, parts, (float*)vol.p, s); break;
                case 3: launch_siddon_t<3>(d, gt, p0, np, parts, (float*)vol.p, s); break;
                default: launch_siddon_t<4>(d, gt, p0, np, parts, (float*)vol.p, s); break;
            }
            e = hipGetLastError();
        }
        bool between = false;
        for (int p = 0; p < d.nphi && !between; ++p)
            for (int x = 0; x < 2; ++x) between |= sid_between_column(d, g->view.data() + (size_t)p * kViewStride, x) >= 0;
        if (between && e == hipSuccess) {
            TOMO_DISPATCH_STORAGE(sino.dtype, TS, {
                hipLaunchKernelGGL((siddon_t_between_kernel<TS>), dim3(d.nphi, ceil_div(d.nv, 64), 2), dim3(64), 0, s, d,
                                   (const TS*)sino.p, inv, (float*)vol.p);
            });
            e = hipGetLastError();
        }
        const hipError_t f = hipFreeAsync(gt, s);
        TOMO_HIP(e);
        TOMO_HIP(f);
        return TOMO_OK;
    }
    int rc = launch_fill((float*)vol.p, 0.0f, g->nvox(), s);
    if (rc) return rc;
    const dim3 grid(ceil_div(d.nu, BX), d.nphi, ceil_div(d.nv, BY));
    TOMO_DISPATCH_STORAGE(sino.dtype, TS, {
        hipLaunchKernelGGL((siddon_adjoint_kernel<TS>), grid, dim3(BX, BY), 0, s, d, (const TS*)sino.p, inv,
                           (float*)vol.p);
    });
    TOMO_HIP(hipGetLastError());
    return TOMO_OK;
}

int count_siddon_segments(tomo_ctx* ctx, const tomo_geom* g, uint64_t* out, hipStream_t s) {
    const DevGeom& d = g->dev;
    unsigned long long* dt = nullptr;
    TOMO_HIP(hipMallocAsync((void**)&dt, sizeof(unsigned long long), s));
    TOMO_HIP(hipMemsetAsync(dt, 0, sizeof(unsigned long long), s));
    const dim3 grid(ceil_div(d.nu, BX), d.nphi, ceil_div(d.nv, BY));
    hipLaunchKernelGGL(siddon_count_kernel, grid, dim3(BX, BY), 0, s, d, dt);
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
