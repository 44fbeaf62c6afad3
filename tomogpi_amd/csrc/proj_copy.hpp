// proj_copy.hpp - the copies of a volume that the forward projectors read.
//
// Both have z fastest, then y, then x: the rays of one detector column cross
// the same in-plane cells, so the rows of a wave read runs of z.  They hold the
// planes that rays reach (proj_planes); below, z counts from the first of them and
// nz is their number, and planes -1 and nz are the neighbours, 0 outside the volume.
// Few rows over a tall volume reach few planes: 512 x 512 x 256, four rows and 360
// views, Siddon 892 us from all planes and 711 from 11, RS 1328 and 1074.
//
// The z-column copy (Siddon) holds single voxels.  FP32: word (x, y, zz), zz in
// [0, nz+1], is f(x, y, zz-1); two neighbouring
// words are a voxel and the one above it.  16-bit volumes: word (x, y, zz), zz in
// [0, nz], holds f(x, y, zz-1) in its low half and f(x, y, zz) in its high half,
// so that one aligned word is the two.
//
// The RS copy holds the in-plane taps of a sample side by side, 0 outside the
// grid.  FP32: element (xx, yy, zz), xx in [0, nx], yy in [0, ny+1], zz in
// [0, nz+1], is the pair f(xx-1, yy-1, zz-1), f(xx, yy-1, zz-1); two neighbouring
// elements of two neighbouring rows are the eight taps of the cell with lower
// corner (xx-1, yy-1, zz-1).  16-bit volumes: element (xx, yy, zz), yy in [0, ny],
// is the four voxels (xx-1, yy-1), (xx, yy-1), (xx-1, yy), (xx, yy) of plane zz-1;
// two neighbouring elements are the eight taps.
#pragma once

#include "device_common.hpp"

namespace tomo {

// The column group of the grid's x index `i` (gx of them, a multiple of 8): the
// XCD i mod 8 takes a run of gx / 8 neighbouring groups.  The runs rotate over
// the XCDs with the view group (of `groups`) and the row band, because outer
// columns have shorter rays.
__device__ __forceinline__ int proj_group(uint32_t i, uint32_t gx, uint32_t pg, uint32_t groups, uint32_t bz) {
    const uint32_t run = (i + pg * 8u / groups + bz) & 7u;
    return (int)(run * (gx / 8u) + i / 8u);
}

// Whether none of the rows n0 .. n0 + rows - 1 has a ray in the volume: rays enter the
// FOV (of radius fov, mm) at fod - fov from the source's plane at the nearest, and
// these are above or below `half` there (mm from the mid plane).
__device__ __forceinline__ bool proj_rows_miss(const DevGeom& g, double fov, double half, int n0, int rows) {
    const float off = fmaxf(fmaxf((float)n0 - g.cv, g.cv - (float)(n0 + rows - 1)), 0.0f);
    return (double)off * (double)g.dv * (g.fod - fov) > half * g.fdd * (1.0 + 1e-6);
}

// Fills the z-column copy of planes zp at `out` from an x-fastest volume of es-byte elements.
hipError_t launch_zcol(const void* vol, uint32_t* out, size_t es, int nx, int ny, int nz, ProjPlanes zp, hipStream_t s);

// Fills the RS copy of planes zp at `out` from an x-fastest volume of es-byte elements.
hipError_t launch_rs_copy(const void* vol, void* out, size_t es, int nx, int ny, int nz, ProjPlanes zp, hipStream_t s);

// Memory of a projector's copy for the duration of one operator call: alloc()
// then release() on the same stream.  It comes from the stream-ordered pool, or
// is the caller's (ProjExtra::copy).
struct ProjCopy {
    void* p = nullptr;
    bool owned = false;
    hipError_t alloc(size_t bytes, hipStream_t s, const ProjExtra& x) {
        p = x.copy;
        if (p) return hipSuccess;
        owned = true;
        return hipMallocAsync(&p, bytes, s);
    }
    hipError_t release(hipStream_t s) {
        const hipError_t e = owned && p ? hipFreeAsync(p, s) : hipSuccess;
        p = nullptr;
        owned = false;
        return e;
    }
};

// out[y + nyp (x + nx z)] = vol[x + nx (y + ny z)] for y < ny and 0 for
// ny <= y < nyp (nyp >= ny), FP32: the volume with y fastest and rows padded
// with zeros, read by the LDS-staged projectors for slabs along x.
hipError_t launch_xy_transpose(const float* vol, float* out, int nx, int ny, int nyp, int nz, hipStream_t s);

// out[x + nxp r] = vol[x + nx r] for x < nx and 0 for nx <= x < nxp, r over
// the ny nz rows, FP32: rows along x padded with zeros.
hipError_t launch_row_pad(const float* vol, float* out, int nx, int nxp, size_t rows, hipStream_t s);

// The rows read by the LDS-staged projectors for the duration of one call:
// along y (vt, rows of nyp floats) for slabs along x, along x (the volume
// itself, or vp when nx is not a multiple of four) for slabs along y.  nxp,
// nyp: nx, ny rounded up to multiples of four.  make() then release() on the
// same stream; the copies come from the stream-ordered pool.
struct StageSources {
    float* vt = nullptr;
    float* vp = nullptr;
    const float* rows_x = nullptr;
    int nxp = 0, nyp = 0;
    hipError_t make(const float* vol, int nx, int ny, int nz, hipStream_t s) {
        nxp = (nx + 3) & ~3;
        nyp = (ny + 3) & ~3;
        hipError_t e = hipMallocAsync((void**)&vt, (size_t)nyp * nx * nz * sizeof(float), s);
        if (e == hipSuccess) e = launch_xy_transpose(vol, vt, nx, ny, nyp, nz, s);
        rows_x = vol;
        if (e == hipSuccess && nxp != nx) {
            e = hipMallocAsync((void**)&vp, (size_t)nxp * ny * nz * sizeof(float), s);
            if (e == hipSuccess) e = launch_row_pad(vol, vp, nx, nxp, (size_t)ny * nz, s);
            rows_x = vp;
        }
        return e;
    }
    hipError_t release(hipStream_t s) {
        hipError_t e = hipSuccess, e2 = hipSuccess;
        if (vp) e = hipFreeAsync(vp, s);
        if (vt) e2 = hipFreeAsync(vt, s);
        vp = vt = nullptr;
        return e != hipSuccess ? e : e2;
    }
};

}  // namespace tomo
