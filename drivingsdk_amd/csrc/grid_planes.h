// Grid sampler on planes (NCHW): arguments of its kernels (grid_planes.hip), filled by the entry points in msda_capi.hip.
#pragma once
#include "msda_device.h"

namespace mxd {

constexpr int kGridThreads = 512;           // per workgroup; 1024 where its LDS leaves no room for a second workgroup on the CU
constexpr int kGridStageBytes = 48 * 1024;  // LDS that several planes of a workgroup share: three workgroups fit a CU
constexpr int kGridMaxPx = 9;               // output pixels whose sums a thread of the grid's gradient keeps in registers

struct GridArgs {
    const void* x;         // [n, c, h, w]
    const void* grid;      // [n, outs, 2]
    void* out;             // [n, c, outs]
    const void* grad_out;
    void* grad_x;          // nullptr: not wanted
    void* grad_grid;       // nullptr: not wanted
    float* part;           // [gg_chunks][n, outs, 2]: the gradient of the grid before its sum over the channel chunks
    int32_t n, c, h, w, outs;
    int32_t mode;          // 1 + padding mode (0 zeros, 1 border) + 2 * align_corners
    // forward: planes per workgroup, chunks of them per image, splits of the output pixels
    int32_t planes, chunks, splits, split_px;
    int32_t run_px;  // > 0: a workgroup's planes one after the other, so many output pixels per thread
    // gradient of the maps: planes per workgroup, chunks per image, bands of a large plane and their pixels, workgroups
    int32_t gx_planes, gx_chunks, gx_bands, gx_band_px, gx_wgs;
    // gradient of the grid: channels per workgroup, of which so many planes are staged at a time, chunks per image, ranges of
    // output pixels, output pixels per thread, workgroups
    int32_t gg_channels, gg_planes, gg_chunks, gg_ranges, gg_px, gg_wgs;
    // both gradients by the same workgroups (gb_wgs > 0): channels per workgroup, chunks per image, output pixels per thread
    int32_t gb_channels, gb_chunks, gb_px, gb_wgs;
    int32_t sum_chunks;  // images of sums in `part` that the sum kernel adds up (0, 1: none)
    int32_t block;
    uint32_t lds;
};

// Bytes of a plane's float64 sums in LDS, what lies behind them on a 16-byte boundary.
__host__ __device__ inline uint32_t grid_sums_bytes(int64_t px) { return (uint32_t)((px * 8 + 15) & ~int64_t(15)); }

// Output pixels per thread up to which two workgroups of 1024 threads fit the registers of a CU (forward, planes one after the other).
__host__ __device__ constexpr int grid_run_px(int es) { return es == 4 ? 6 : 3; }

// Elements before a plane in LDS that a corner a row and a pixel before it can reach, in whole 16-byte pieces.
__host__ __device__ inline int grid_margin(int es, int w) { return (w + 16 / es) / (16 / es) * (16 / es); }

hipError_t raise_grid_lds();
hipError_t launch_grid_planes_forward(int dtype, const GridArgs& a, hipStream_t stream);
hipError_t launch_grid_planes_backward(int dtype, const GridArgs& a, hipStream_t stream);

}  // namespace mxd
