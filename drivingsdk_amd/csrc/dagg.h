// Deformable aggregation: arguments of its kernels (dagg.hip), filled by the entry points in msda_capi.hip.
#pragma once
#include "msda_device.h"

namespace mxd {

constexpr int kDaggWaves = 4;        // wavefronts per workgroup of the forward: an anchor each
constexpr int kDaggBackWaves = 8;    // the same for the backward's first kernel, whose sort is the shorter for it (442 anchors: 52 -> 44 us with 8, 43 with
                                     // 16; 6 x 900 anchors lose 5 % with 16)
constexpr int kDaggSortWaves = 16;   // the same for the sort as a launch of its own (6 x 900 anchors: 72 instead of 68 us with 8, before its
                                     // points were compacted)
constexpr int kDaggList = 128;       // locations of an anchor that a wavefront looks through before it samples
constexpr int kDaggSortPx = 4096;    // pixels of a level that a workgroup of the sort counts in LDS
constexpr int kDaggStrip = 8;        // neighbouring pixels whose gradient rows are formed together

struct DaggArgs {
    const void* feat;      // [bs, nf, C]
    const int32_t* shapes; // [cams, scales, 2]
    const int32_t* lsi;    // [cams, scales]
    int32_t meta_i64;
    const void* loc;       // [bs, A, P, cams, 2]
    const void* w;         // [bs, A, P, cams, scales, G]
    void* out;             // [bs, A, C]
    const void* grad_out;
    void* grad_feat;
    void* grad_loc;
    void* grad_w;
    float* image;          // float32 image of grad_feat: grad_feat itself, or in the workspace for 16-bit dtypes
    float* gw_part;        // [G][bs, A][cams, P, scales]: gradients of the weights of one group, locations inside the image only
    float* gl_part;        // [G][bs, A][cams, P][2]: one group's part of the location gradients, summed over the scales
    f32x2* dots;           // [bs, A][P, cams, scales][upper, lower row][G]: dot products of the row's first pixel and of its right
                           //   neighbour, in place of the two above; null: the first kernel forms those
    uint32_t* csr;         // [bs][starts]: per level, first record of every pixel, then their number
    u32x4* rec;            // [bs][nl][2 A P] records sorted by pixel: {anchor << 3 | pixel & 7, row of the sample << 31 | index of the weight of group 0 / G,
                           //   bilinear weight of the pixel, of the pixel to its right}
    int32_t bs, nf, C, G, hd, cams, scales, nl, A, P;
    int32_t nloc;          // P * cams
    uint32_t p_magic;      // ceil(2^20 / P)
    uint32_t sc_magic;     // ceil(2^20 / scales)
    uint32_t pitch_bytes, batch_bytes;
    // a row of the forward and the first backward kernel: the channels of a group, or (forward) 128 bytes of several groups
    int32_t pieces;        // per feature row
    int32_t piece_ch;      // channels
    int32_t piece_heads;   // groups that a piece touches at most; 1 = a piece is a group
    int32_t lpr_log2;      // lanes that share it
    // grad_feat: lanes that share a pixel row, channel blocks per row
    int32_t row_lpr_log2, row_blocks, sort_ranges;
    int64_t starts;        // entries of a batch element's table of record starts (dagg_starts)
    int32_t strip_records; // records per strip aimed at where the strips of a level are split
    mxd_msda_plan map;     // XCD mapping: piece = head, anchor = query
};

hipError_t launch_dagg_forward(int dtype, const DaggArgs& a, hipStream_t stream);
hipError_t launch_dagg_backward(int dtype, const DaggArgs& a, hipStream_t stream);

// Entries of a batch element's table of record starts.  A level takes one per pixel and one more; levels that do not overlap have at
// most the tensor's pixels between them, and 512 entries more per level are room for levels that share rows (cameras that name the
// same map).  What does not fit all the same is added sample by sample (dagg_levels_without_room).
inline int64_t dagg_starts(int64_t nf, int64_t nl) { return nf + nl * (512 + 1); }

// Elements per lane of a row piece of `ch` channels (what the kernels are instantiated for).
inline int dagg_vec(int elem_size, int64_t ch)
{
    int vec = 16 / elem_size;
    while (vec > ch) vec >>= 1;
    return vec;
}

}  // namespace mxd
