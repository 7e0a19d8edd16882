// Geometric kernel attention on maps that fit LDS: arguments of its kernels (gka.hip), filled by the entry points in msda_capi.hip.
#pragma once
#include "msda_device.h"

namespace mxd {

// Samples of a tile of queries that a thread of the scatter keeps in registers while they are sorted, beside the sums of `px` pixels.
constexpr int gka_samples(int px, bool quad) { return quad && px > 8 ? 6 : 8; }
constexpr int kGkaPixels = 16;   // pixels whose sums a lane group of the scatter keeps in registers, at most
constexpr int kGkaLevelBytes = kMaxLevels * 16;

struct GkaArgs {
    const void* value;     // [bs, nk, nh, hd]
    const int32_t* shapes;
    const int32_t* lsi;
    int32_t meta_i64;
    const float* loc;      // [bs, nq, nh, S, 2]
    const void* attn;      // [bs, nq, nh, S]
    void* out;             // [bs, nq, nh, hd]
    const void* grad_out;
    void* grad_value;
    void* grad_attn;
    float* part;           // [splits][bs, nk, nh, hd]: grad_value of one range of the queries
    int32_t bs, nk, nh, hd, nl, np, nq, S;
    uint32_t np_magic;     // ceil(2^20 / np)
    uint32_t s_magic;      // ceil(2^20 / S)
    // maps too large for LDS with whole rows: the channels of a head in parts, each with workgroups of its own
    int32_t parts, part_ch;
    float* dots;           // [parts][bs, nq, nh, S]: the parts' dots, where there are several
    int32_t lpr_log2;      // lanes of 16 bytes that share a part's row
    // forward and dots: workgroups per (batch, head), queries each
    int32_t splits, split_q, block;
    uint32_t lds;
    // grad_value: the same, queries per tile, lanes of 4 channels that share a row, pixels per lane group
    int32_t sc_splits, sc_split_q, sc_block, sc_tile_q, sc_lanes_log2, sc_px;
    uint32_t sc_lds;
    int32_t sc_direct;     // rows of grad_out are 16-byte aligned: they go straight to LDS
    int32_t sc_dots;       // the gradient of the weights is formed there too, else by a kernel of its own
};

hipError_t raise_gka_lds();
hipError_t launch_gka_forward(int dtype, const GkaArgs& a, hipStream_t stream);
hipError_t launch_gka_backward(int dtype, const GkaArgs& a, hipStream_t stream);

}  // namespace mxd
