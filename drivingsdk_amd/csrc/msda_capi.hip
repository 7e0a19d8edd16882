// C ABI entry points (include/mxd_msda.h): argument checks, launch geometry, enqueue.
// Host code only; the kernels live in msda_fwd.hip, msda_fwd_cu.hip, msda_bwd_kernel.h (with msda_bwd*.hip) and msda_bwd_tiles.hip.  Multi-scale
// deformable attention, its fused form, geometric kernel attention and the grid sampler are the same three kernels with
// different sample sources (msda_device.h: sample_ref, source_geometry); deformable aggregation has its own (dagg.hip).
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdarg.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include <atomic>
#include <mutex>

#include "dagg.h"
#include "gka.h"
#include "grid_planes.h"
#include "msda_device.h"

namespace mxd {
hipError_t launch_forward(int dtype, const KArgs& a, hipStream_t stream);
hipError_t launch_forward_cu(int dtype, const KArgs& a, hipStream_t stream);
hipError_t raise_forward_lds();
hipError_t raise_forward_cu_lds();
hipError_t launch_backward(int dtype, const KArgs& a, bool scatter, hipStream_t stream);
hipError_t launch_gradv_tiles(int dtype, const KArgs& a, const TileArgs& t, hipStream_t stream);
hipError_t launch_fill_zero(float* p, size_t n, hipStream_t stream);
hipError_t launch_round(int dtype, const float* src, void* dst, size_t n, hipStream_t stream);
hipError_t launch_round_rows(int dtype, const KArgs& a, hipStream_t stream);
hipError_t launch_sum_heads(int dtype, const float* part, void* dst, size_t n, int nh, hipStream_t stream);
}  // namespace mxd

namespace {

thread_local char g_err[512] = "";

int fail(int code, const char* fmt, ...)
{
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(g_err, sizeof(g_err), fmt, ap);
    va_end(ap);
    return code;
}

// Splits the MXD_META_I64 flag off a dtype argument; returns 1 when it was set.
static int take_meta_flag(int* dtype)
{
    const int f = (*dtype & MXD_META_I64) ? 1 : 0;
    *dtype &= ~MXD_META_I64;
    return f;
}

int elem_size(int dtype)
{
    switch (dtype) {
        case MXD_DTYPE_F32: return 4;
        case MXD_DTYPE_F16:
        case MXD_DTYPE_BF16: return 2;
        default: return 0;
    }
}

int env_int(const char* name, int dflt)
{
    const char* v = getenv(name);
    return (v && *v) ? atoi(v) : dflt;
}

// Tuning knobs, read from the environment once per process (mxd_msda_reload_tuning() reads them again: a hook for
// tests and experiments, not to be called while other threads are inside the library).
struct Tuning {
    int xcd_mode;        // MXD_MSDA_XCD_MODE: 0 = plain workgroup mapping, -1 = by head count
    int bwd_tile_q;      // MXD_MSDA_BWD_TILE_Q: queries per workgroup of the first backward kernel, 0 = chosen here
    int bwd_atomic;      // MXD_MSDA_BWD_ATOMIC: 1 = one-kernel backward with global atomics
    int tile_target;     // MXD_MSDA_TILE_TARGET: pair records per work item of the tile pass, 0 = chosen here
    int fwd_lds;         // MXD_MSDA_FWD_LDS: bytes of the general forward's level cache, -1 = by estimate
    int fwd_iters;       // MXD_MSDA_FWD_ITERS
    int fwd_wgq;         // MXD_MSDA_FWD_WGQ: queries per workgroup of the general forward with a level cache
    int fwd_ahead;       // MXD_MSDA_FWD_AHEAD
    int fwd_cu;          // MXD_MSDA_FWD_CU: 0 = never use the one-workgroup-per-CU forward, 1 = whenever it can run,
                         // -1 = for problems large enough to pay for it
    int fwd_cu_wgs;      // MXD_MSDA_FWD_CU_WGS: its workgroups per (batch, head), 0 = chosen here
    int fwd_cu_cache;    // MXD_MSDA_FWD_CU_CACHE: most bytes of LDS its level cache takes, -1 = all the CU has (a small value
                         // makes every sample come from memory: a hook for measurements)
    int fwd_cu_flip;     // MXD_MSDA_FWD_CU_FLIP: 1 = half of its wavefronts gather from LDS first, the others from memory
                         // first; 0 = all in the same order (sums then formed in the general kernel's order, bit for bit);
                         // -1 = chosen here
    int bwd_fill_kernel; // MXD_MSDA_BWD_FILL_KERNEL: 1 = zero-fill by a kernel of its own
    int tile_order;      // MXD_MSDA_TILE_ORDER: 1 = work items of the tile pass batch-major, 0 = item-major, -1 = chosen here
    int bwd_sparse;      // MXD_MSDA_BWD_SPARSE: 0 = zero-fill (and, for 16-bit dtypes, round) the whole fp32 image of
                         // grad_value, 1 = only the rows that receive atomic additions
    int bwd_unit_split;  // MXD_MSDA_BWD_UNIT_SPLIT: 0 = a unit of the first backward kernel is always a whole query, 1 = queries
                         // of 25 to 32 samples get two units, those of 17 to 24 where it pays, 2 = queries of 17 to 32 samples
    int bwd_lane_bytes;  // MXD_MSDA_BWD_LANE_BYTES: most bytes of a row one lane of the first backward kernel loads
                         // (16, 8, 4), 0 = chosen here
    int tile_px_log2;    // MXD_MSDA_TILE_PX_LOG2: log2 of the pixels per tile of the grad_value pass (9, 8, 7), 0 = chosen here
    int gka_slab;        // MXD_MSDA_GKA_SLAB: geometric kernel attention with value in LDS: 0 = never, 1 = wherever it fits, -1 = chosen here
    int bwd_fixed;       // MXD_MSDA_BWD_FIXED: 0 = the general first backward kernel also where the launch has a geometry that a kernel
                         // (one pass, 4 or 8 lanes per row) or an instantiation (256-byte rows) of its own is built for (default 1)
    int bwd_two_pass;    // MXD_MSDA_BWD_TWO_PASS: 1 = the first backward kernel reads rows of 17 to 32 lanes of 16 bytes with 16
                         // lanes in two passes, 0 = with 32 lanes in one
    int bwd_rec_lds;     // MXD_MSDA_BWD_REC_LDS: 0 = workgroups of the first backward kernel that make several passes store
                         // their records one by one, 1 = they collect their slab in LDS wherever it fits, -1 = chosen here
};
Tuning g_tuning;
std::once_flag g_tuning_once;

void read_tuning()
{
    Tuning t;
    t.xcd_mode = env_int("MXD_MSDA_XCD_MODE", -1);
    t.bwd_tile_q = env_int("MXD_MSDA_BWD_TILE_Q", 0);
    t.bwd_atomic = env_int("MXD_MSDA_BWD_ATOMIC", 0);
    t.tile_target = env_int("MXD_MSDA_TILE_TARGET", 0);
    t.fwd_lds = env_int("MXD_MSDA_FWD_LDS", -1);
    t.fwd_iters = env_int("MXD_MSDA_FWD_ITERS", 1);
    t.fwd_wgq = env_int("MXD_MSDA_FWD_WGQ", 128);
    t.fwd_ahead = env_int("MXD_MSDA_FWD_AHEAD", 1);
    t.fwd_cu = env_int("MXD_MSDA_FWD_CU", -1);
    t.fwd_cu_wgs = env_int("MXD_MSDA_FWD_CU_WGS", 0);
    t.fwd_cu_flip = env_int("MXD_MSDA_FWD_CU_FLIP", -1);
    t.fwd_cu_cache = env_int("MXD_MSDA_FWD_CU_CACHE", -1);
    t.bwd_fill_kernel = env_int("MXD_MSDA_BWD_FILL_KERNEL", 0);
    t.tile_order = env_int("MXD_MSDA_TILE_ORDER", -1);
    t.bwd_lane_bytes = env_int("MXD_MSDA_BWD_LANE_BYTES", 0);
    t.bwd_sparse = env_int("MXD_MSDA_BWD_SPARSE", 1);
    t.bwd_unit_split = env_int("MXD_MSDA_BWD_UNIT_SPLIT", 1);
    t.tile_px_log2 = env_int("MXD_MSDA_TILE_PX_LOG2", 0);
    t.bwd_rec_lds = env_int("MXD_MSDA_BWD_REC_LDS", -1);
    t.gka_slab = env_int("MXD_MSDA_GKA_SLAB", -1);
    t.bwd_fixed = env_int("MXD_MSDA_BWD_FIXED", 1);
    t.bwd_two_pass = env_int("MXD_MSDA_BWD_TWO_PASS", 1);
    g_tuning = t;
}

const Tuning& tuning()
{
    std::call_once(g_tuning_once, read_tuning);
    return g_tuning;
}

// Scratch of mxd_msda_backward_static(): the hand-over between the two backward kernels (and the fp32 image of
// grad_value for 16-bit dtypes) for callers that can neither allocate nor pass a workspace.  Every device that the
// library runs on holds its own copy of the array at its own address until the process ends.  In host code the name
// below is a stand-in, not a device address: g_scratch_ptr[device], resolved once per device, is what is used.
constexpr size_t kStaticScratchBytes = (size_t)MXD_MSDA_STATIC_SCRATCH_BYTES;
static __device__ __align__(256) unsigned char scratch[kStaticScratchBytes];

// Per-device set-up, done once per device on the first call that needs it (or by mxd_msda_init()): the forward
// kernels that use more than 64 KiB of dynamic LDS opt in, and the device address of `scratch` is looked up.
constexpr int kMaxDevices = 64;
std::atomic<int> g_device_ready[kMaxDevices];
void* g_scratch_ptr[kMaxDevices];
std::mutex g_device_mutex;

int ensure_device_ready()
{
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return fail(MXD_E_LAUNCH, "hipGetDevice failed: %s", hipGetErrorString(e));
    if (dev < 0 || dev >= kMaxDevices) return fail(MXD_E_LAUNCH, "device ordinal %d is beyond what this build keeps state for", dev);
    if (g_device_ready[dev].load(std::memory_order_acquire)) return MXD_OK;
    std::lock_guard<std::mutex> lock(g_device_mutex);
    if (g_device_ready[dev].load(std::memory_order_relaxed)) return MXD_OK;
    e = mxd::raise_forward_lds();
    if (e == hipSuccess) e = mxd::raise_forward_cu_lds();
    if (e == hipSuccess) e = mxd::raise_grid_lds();
    if (e == hipSuccess) e = mxd::raise_gka_lds();
    if (e != hipSuccess) return fail(MXD_E_LAUNCH, "raising the dynamic LDS limit failed: %s", hipGetErrorString(e));
    void* ptr = nullptr;
    e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));  // (this device's copy of the array: the device is current)
    if (e != hipSuccess || ptr == nullptr)
        return fail(MXD_E_LAUNCH, "looking up the static scratch array failed: %s", hipGetErrorString(e));
    g_scratch_ptr[dev] = ptr;
    g_device_ready[dev].store(1, std::memory_order_release);
    return MXD_OK;
}

// The current device's copy of `scratch` (after ensure_device_ready()).
void* device_scratch()
{
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return nullptr;
    return g_device_ready[dev].load(std::memory_order_acquire) ? g_scratch_ptr[dev] : nullptr;
}

struct Dims {
    int64_t bs, nk, nh, hd, nl, nl_attn, nq, np;
    int kind = 0;  // which operator the shared kernels run for: 0 the plain one, 1 geometric kernel attention, 2 the fused form
};

size_t round_up(size_t n, size_t to) { return (n + to - 1) / to * to; }

int check_dims(int dtype, const Dims& d)
{
    if (elem_size(dtype) == 0) return fail(MXD_E_DTYPE, "dtype code %d is not float32(0)/float16(1)/bfloat16(2)", dtype);
    if (d.bs <= 0 || d.nk <= 0 || d.nh <= 0 || d.hd <= 0 || d.nl <= 0 || d.nq <= 0 || d.np <= 0)
        return fail(MXD_E_SHAPE, "Input Tensor can not be a empty Tensor (bs=%lld nk=%lld nh=%lld hd=%lld nl=%lld nq=%lld np=%lld)",
                    (long long)d.bs, (long long)d.nk, (long long)d.nh, (long long)d.hd, (long long)d.nl,
                    (long long)d.nq, (long long)d.np);
    if (d.hd > 256) return fail(MXD_E_SHAPE, "The number of embedding dimensions should be less than or equal to 256");
    if (d.nl > mxd::kMaxLevels) return fail(MXD_E_SHAPE, "The number of levels should be less than or equal to %d", mxd::kMaxLevels);
    if (d.nl_attn < d.nl)
        return fail(MXD_E_SHAPE, "attention_weights carries %lld levels but spatial_shapes has %lld", (long long)d.nl_attn,
                    (long long)d.nl);
    if (d.nl * d.np > 4096 || d.nl * d.np * d.np >= (1 << 20))
        return fail(MXD_E_SHAPE, "num_levels*num_points = %lld is beyond what this build indexes", (long long)(d.nl * d.np));
    if (d.nk * d.nh * d.hd * 4 >= (int64_t(1) << 31))
        return fail(MXD_E_SHAPE, "one batch element of value (num_keys*num_heads*embed_dims = %lld elements) must stay below 2 GiB at 4 bytes per element",
                    (long long)(d.nk * d.nh * d.hd));
    if (d.nq >= (int64_t(1) << 31) - 4096 || d.bs >= (1 << 24) || d.nh >= (1 << 16) ||
        d.nl_attn * d.np >= (int64_t(1) << 24))
        return fail(MXD_E_SHAPE, "a dimension is beyond what this build indexes");
    return MXD_OK;
}

// Fills the XCD mapping fields of a plan for `ntiles` work items per (batch, head); returns the grid.
//
// row_bytes: length of the rows that are gathered (0: of no matter).  Rows of up to 64 bytes of neighbouring heads share the lines of
// 128 bytes that move between memory, L2 and L1: pinned to an XCD each, such heads fetch every line twice and fill twice the L2 for the
// same rows.  Heads that share a line then share an XCD, and where that leaves XCDs without a head of their own, several XCDs share
// the heads' (batch element, tile) pairs, each taking a contiguous part of them (mode 3).  A head per XCD / this: 6 x 9675 queries of 32
// samples over 30 825 keys in float16, forward 231 / 203 us, first backward kernel 379 / 356; two batch elements of the encoder in
// bfloat16, fused forward 79.6 / 74.6 (one round of workgroups: the slices of two heads side by side fill no more of an L2 than one
// did); 43 problems of 16 to 32 channels, one to five levels, 300 to 20 000 queries: forward 0.71 to 1.03 of the time, 0.90 on average,
// backward 0.94 to 1.03, 0.98.  The tile pass gains nothing by it (408 / 409 us at the first of these) and keeps a head per XCD.
int64_t fill_xcd_map(mxd_msda_plan* p, int64_t bs, int64_t nh, int64_t ntiles, int64_t row_bytes = 0)
{
    p->ntiles = (int32_t)ntiles;
    const int mode_override = tuning().xcd_mode;
    int64_t share = 1;  // heads that share a line
    while (row_bytes > 0 && 2 * share * row_bytes <= 128 && nh % (2 * share) == 0) share *= 2;
    const int64_t groups = nh / share;
    if (mode_override != 0 && share > 1 && groups < mxd::kNumXcd && mxd::kNumXcd % groups == 0) {
        p->xcd_mode = 3;
        p->heads_per_xcd = (int32_t)share;
        p->xcds_per_head = (int32_t)(mxd::kNumXcd / groups);
        const int64_t each = (bs * ntiles * share + p->xcds_per_head - 1) / p->xcds_per_head;
        p->tiles_per_part = (int32_t)each;  // (the callers refuse grids beyond 2^31)
        return (int64_t)mxd::kNumXcd * each;
    }
    if (mode_override != 0 && nh % mxd::kNumXcd == 0) {
        p->xcd_mode = 1;
        p->heads_per_xcd = (int32_t)(nh / mxd::kNumXcd);
        p->xcds_per_head = 1;
        p->tiles_per_part = (int32_t)ntiles;
        return (int64_t)mxd::kNumXcd * p->heads_per_xcd * ntiles * bs;
    }
    if (mode_override != 0 && mxd::kNumXcd % nh == 0) {
        p->xcd_mode = 2;
        p->heads_per_xcd = 1;
        p->xcds_per_head = (int32_t)(mxd::kNumXcd / nh);
        p->tiles_per_part = (int32_t)((ntiles + p->xcds_per_head - 1) / p->xcds_per_head);
        return (int64_t)mxd::kNumXcd * p->tiles_per_part * bs;
    }
    p->xcd_mode = 0;
    p->heads_per_xcd = 1;
    p->xcds_per_head = 1;
    p->tiles_per_part = (int32_t)ntiles;
    return bs * nh * ntiles;
}

// Bytes of dynamic LDS of the first backward kernel for a plan (tile mode: with the per-tile counters).
size_t backward_lds_bytes(int units_per_wave, int waves, bool tiles, int64_t tbl_stride)
{
    const size_t per_unit = mxd::kChunkStride * sizeof(mxd::Entry) + mxd::kChunk * sizeof(mxd::f32x4);
    size_t n = mxd::kMaxLevels * sizeof(mxd::i32x4) + (size_t)waves * units_per_wave * per_unit;
    if (tiles) n += (size_t)(mxd::kMaxLevels + tbl_stride) * sizeof(int32_t);
    return n;
}

// Row geometry of a problem: elements per lane, lanes per row, row passes.
// two_pass_rows: rows of 17 to 32 lanes of 16 bytes are read by 16 lanes in two passes instead (four units per
// wavefront rather than two: the first backward kernel then fills its geometry lanes and sums its dots over 16 lanes
// with DPP alone; backward at 8 heads x 128 channels in float32 587 -> 572 us, 545 with the slab collected in LDS).
// whole_pieces: only pieces that divide the row and that `align_bytes` allows; otherwise a row that is no multiple of the
// piece is read in pieces of which the last one overlaps the one before it (piece_start, msda_device.h), wherever it
// starts: pieces that divide the 37 channels of a head are single elements, 37 of 64 lanes at work and a unit per
// wavefront (6 x 9680 queries of 4 heads x 37 channels, five levels with 3 points, float32: forward 226 -> 144 us, the backward's
// first kernel 582 -> 212, its tile pass, which then reads the records once for up to 64 channels, 331 -> 219).
void row_geometry(int es, int64_t hd, int lane_bytes, int* vec_out, int* lpr_out, int* npass_out, bool two_pass_rows = false,
                  bool whole_pieces = false)
{
    if (lane_bytes < es) lane_bytes = es;
    int vec = lane_bytes / es < 16 / es ? lane_bytes / es : 16 / es;
    while (vec > 1 && (whole_pieces ? hd % vec != 0 : hd < vec)) vec >>= 1;
    const int lanes_needed = (int)((hd + vec - 1) / vec);
    int lpr = 4;
    while (lpr < lanes_needed && lpr < mxd::kWave) lpr <<= 1;
    if (two_pass_rows && vec * es == 16 && lpr == 32) lpr = 16;
    int npass = (lanes_needed + lpr - 1) / lpr;
    if (npass == 3) npass = 4;
    *vec_out = vec;
    *lpr_out = lpr;
    *npass_out = npass;
}

// Most bytes of a row that one lane of the first backward kernel loads.
int backward_lane_bytes(int dtype, const Dims& d)
{
    const int v = tuning().bwd_lane_bytes;
    if (v == 4 || v == 8 || v == 16) return v;
    // Rows of 33 to 64 bytes: 8 lanes of 8 bytes per row rather than 4 lanes of 16 in the general kernel, whose staging strips of 16
    // units per wavefront take 51 KiB of LDS (encoder shape in float16 / bfloat16: backward 322 -> 300 us; with rows of 256 bytes
    // halving the lane width costs 10 %).  The kernel of one-pass workgroups takes 4 lanes by itself where it has the workgroups.
    // Rows of up to 32 bytes: 8 lanes of 4 for units that fill a chunk of 16 samples (16 channels in float16, 2 x 13253 queries of 18
    // samples: backward 289 -> 251 us; 3 samples 53 -> 55), with half as many queries per workgroup.
    const int64_t row = d.hd * elem_size(dtype);
    if (row > 16 && row <= 32) return d.nl * d.np > 12 ? 4 : 16;
    return (row > 32 && row <= 64) ? 8 : 16;
}

// How the backward pass is laid out for a problem size: whether grad_value goes through the
// tile-ownership pass (and then the hand-over buffers between its two kernels) or through
// global atomics, and where things live in the caller's workspace.
//   workspace = [run table][pair records][fp32 image of grad_value, 16-bit dtypes only]
// Queries per workgroup of the first backward kernel (tile pass).  Larger workgroups give the tile pass
// longer runs; with few queries they leave the chip short of workgroups, so the size steps down until the
// launch has about six workgroups per CU.  64 is the least for rows of up to 64 bytes (16 units per
// wavefront, 4 wavefronts), 32 otherwise.  MXD_MSDA_BWD_TILE_Q overrides (32/64/128/256).
static int64_t bwd_tile_q(int dtype, const Dims& d, bool early_split)
{
    // (units with very many samples measured 1 to 2 % better with 64)
    int vec, lpr, npass;
    row_geometry(elem_size(dtype), d.hd, backward_lane_bytes(dtype, d), &vec, &lpr, &npass, tuning().bwd_two_pass != 0);
    const int64_t least = (mxd::kWave / lpr > 8 || d.nl * d.np >= 256) ? 64 : 32;
    const int v = tuning().bwd_tile_q;
    if (v == 32 || v == 64 || v == 128 || v == 256) return v < least ? least : v;
    // about 512 samples per workgroup for rows of up to 128 bytes, 1024 for longer ones (measured: 32 queries of 16
    // or of 32 samples are the optima of the encoder and the BEVFormer shapes -- with 16 samples per query all of a
    // workgroup's samples are then staged while its records are counted --, 64 queries of 16 samples that of 512-byte
    // rows; 128 queries cost 3 to 7 %)
    const int64_t samples = d.hd * elem_size(dtype) <= 128 ? 512 : 1024;
    int64_t first = 128;
    while (first > least && first * d.nl * d.np > samples) first >>= 1;
    for (int64_t tq = first; tq > least; tq >>= 1)
        if (d.bs * d.nh * ((d.nq + tq - 1) / tq) >= 6 * 256) return tq;
    // Queries of 17 to 32 samples in a workgroup that makes one pass: two neighbouring units share a query, each taking
    // 16 of its samples, so that the workgroup -- half as many queries -- stages all its samples while it counts its
    // records (their geometry is derived once) and collects its records in LDS to write its slab in whole lines, as
    // with up to 16 samples per query.
    // From 25 samples on the second unit has work for most of its lanes (encoder levels, float32, 32 samples: one unit / two 566 /
    // 486 us, BEVFormer 1044 / 967).  With 17 to 24 samples, most of whose second units idle, it depends on what the shorter
    // slabs cost the tile pass: it pays from 16 000 keys on (18, 22, 21 and 24 samples, three types, 40 000 to 58 000 queries: 19 000
    // keys 0.85 to 1.01 of the time with one unit, 32 000 keys 0.79 to 0.98; 12 000 keys 0.93 to 1.06, 5 000 keys 0.96 to 1.10),
    // for rows of more than 64 bytes in float32 (5 000 keys 0.96 to 1.03, 12 000 keys 0.93 to 1.03) and where queries are
    // few (5 000 queries x 8 heads: 5 000 keys 0.89 to 1.04, 12 000 keys 0.83 to 0.98).  The plain operator's only, whose workgroups
    // collect their slab in LDS by it: the fused form takes 0.96 to 1.22, geometric kernel attention 0.99 to 1.14 of the
    // time with one unit.  MXD_MSDA_BWD_UNIT_SPLIT=2 splits from 17 on.
    const int units = mxd::kWave / lpr * 4;
    const bool early = tuning().bwd_unit_split >= 2 ||
                       (early_split && d.kind == 0 && (d.nk >= 16384 || (elem_size(dtype) == 4 && d.hd > 16) || d.bs * d.nh * d.nq <= 65536));
    const int64_t split_from = early ? mxd::kChunk + 1 : mxd::kChunk + mxd::kChunk / 2 + 1;
    if (tuning().bwd_unit_split && least == units && units >= 8 && d.nl * d.np >= split_from && d.nl * d.np <= 2 * mxd::kChunk)
        return least / 2;
    return least;
}
struct BwdLayout {
    bool tiles;          // false: one kernel with global atomics
    int tile_px_log2;    // log2 of the pixels per tile of the grad_value pass
    int64_t tile_q;      // queries per workgroup of the first kernel
    int64_t nwg;         // workgroups of the first kernel per (batch, head)
    int64_t rec_cap;     // pair records per workgroup slab: 2 per sample
    int64_t tbl_stride;  // tiles per (batch, head) at most, plus one
    size_t tbl_bytes, rec_bytes, image_bytes, total;
};

// Pixels per tile of the grad_value pass, as a power of two: every thread of its workgroups keeps 32 sums, so 512 pixels
// of up to 32 channels, 256 of up to 64, 128 of more (msda_plan.h).
int preferred_tile_px_log2(int dtype, const Dims& d)
{
    // (16-bit rows of fewer than 4 channels, which no lane can read four of, have the tile pass for 512 pixels alone)
    if (elem_size(dtype) == 2 && d.hd < 4) return mxd::kTilePxLog2Max;
    const int v = tuning().tile_px_log2;
    if (v >= 7 && v <= mxd::kTilePxLog2Max) return v;
    if (d.hd <= 32) return mxd::kTilePxLog2Max;
    // Geometric kernel attention clamps its samples to the map, which piles many of them on the border's pixels.  Those get extra
    // lists in the slots of a workgroup that its tile leaves free; a map cut in tiles of 256 or 128 pixels has none to speak of.
    // With enough samples that is worth two to four passes over the records.  15 x 25 pixels, 24 x 7156 queries x 15, backward,
    // tiles by head size -> one tile of 512: float32 48 channels 692 -> 584 us, 96 channels 1076 -> 918, 160 channels
    // 2417 -> 1791; float16 646 -> 576, 812 -> 758, 1546 -> 1232.  From 3.6 million samples on 18 of 24 sizes of 280 to 360
    // pixels gain 10 to 30 %, the others are within 5 % of even (but for one at +15 %: 96 channels in float16, 280 pixels, 20.6
    // million).  Not with fewer samples (half a million 1.3 to 1.7 times as long), not on maps that one smaller tile holds (6 x 10:
    // 1.04 to 1.5), not where the free slots are fewer than the pixels that want them (420 pixels, 48 channels: 1.13 to
    // 1.3) and not for several levels (15 x 25 and 8 x 13, 48 channels, 11 million: 1.13 and 1.21).
    if (d.kind == 1 && d.nl == 1 && d.nk > 256 && d.nk <= 384 && d.bs * d.nh * d.nq * d.np >= (int64_t(3) << 20)) return mxd::kTilePxLog2Max;
    // (measured at 8 heads x 128 channels, encoder levels: float16 backward 588 us with tiles of 512 pixels, 431 with 256,
    //  383 with 128; float32 722, 590, 586)
    return d.hd <= 64 ? 8 : 7;
}

BwdLayout bwd_layout_for(int dtype, const Dims& d, int tile_px_log2, bool early_split)
{
    BwdLayout L;
    memset(&L, 0, sizeof(L));
    L.tile_px_log2 = tile_px_log2;
    L.tile_q = bwd_tile_q(dtype, d, early_split);
    L.nwg = (d.nq + L.tile_q - 1) / L.tile_q;
    L.rec_cap = 2 * L.tile_q * d.nl * d.np;
    // tiles per (batch, head) when the levels do not overlap: sum of ceil(pixels / tile) <= nk / tile + nl
    // (levels that would not fit, which can only happen for overlapping ones, leave no records: add_levels_without_tiles)
    L.tbl_stride = (d.nk >> tile_px_log2) + d.nl + 1;
    const int64_t tbl = d.bs * d.nh * L.nwg * L.tbl_stride * 4;
    // dynamic LDS of the first kernel with the most units per wavefront the row can have (16-byte aligned pointers)
    int vec, lpr, npass;
    row_geometry(elem_size(dtype), d.hd, backward_lane_bytes(dtype, d), &vec, &lpr, &npass, tuning().bwd_two_pass != 0);
    const size_t lds = backward_lds_bytes(mxd::kWave / lpr, 4, true, L.tbl_stride);
    L.tiles = tuning().bwd_atomic == 0 &&
              L.tbl_stride <= 4096 &&                      // counters of the first kernel live in LDS ...
              lds <= 64 * 1024 &&                          // ... and its strips and counters fit the default limit
              tbl <= (int64_t(1) << 28) &&                 // run table of at most 256 MiB
              L.nwg * L.rec_cap * (mxd::kRecDwords * 4) < (int64_t(1) << 32) &&  // 32-bit byte offsets of the records of a (batch, head)
              d.nq < (int64_t(1) << (32 - mxd::kTilePxLog2Max)) &&  // a record holds the query above the pixel of its tile
              d.nq * d.nh * d.hd * 4 < (int64_t(1) << 31); // grad_output rows addressed with 32-bit byte offsets
    if (L.tiles) {
        L.tbl_bytes = ((size_t)tbl + 255) & ~(size_t)255;
        L.rec_bytes = ((size_t)d.bs * d.nh * L.nwg * L.rec_cap * (mxd::kRecDwords * 4) + 255) & ~(size_t)255;
    }
    if (elem_size(dtype) == 2) L.image_bytes = (size_t)d.bs * d.nk * d.nh * d.hd * 4;
    L.total = L.tbl_bytes + L.rec_bytes + L.image_bytes;
    return L;
}

// The layout a launch uses: the tile size preferred for the rows, or 512-pixel tiles where the finer run table would
// not fit the first kernel's bookkeeping.  Queries of 17 to 24 samples keep one unit where the longer run table of two would not
// fit, or would take the workspace beyond the static array that the one of whole queries fits.
BwdLayout bwd_layout(int dtype, const Dims& d)
{
    const int pref = preferred_tile_px_log2(dtype, d);
    BwdLayout L = bwd_layout_for(dtype, d, pref, true);
    if (!L.tiles || L.total > kStaticScratchBytes) {
        const BwdLayout whole = bwd_layout_for(dtype, d, pref, false);
        if (whole.tiles && (!L.tiles || whole.total <= kStaticScratchBytes)) L = whole;
    }
    if (!L.tiles && pref != mxd::kTilePxLog2Max) L = bwd_layout_for(dtype, d, mxd::kTilePxLog2Max, false);
    return L;
}

// Step through the slabs of a (batch, head) in the tile pass: near the golden section of their number, which spreads any
// stretch of steps evenly over the query range, and without a common divisor with it, so that every slab is met once.
uint32_t run_step(int64_t nwg)
{
    if (nwg < 4 || nwg > 65535) return 1;  // (index times step stays below 2^32)
    auto gcd = [](uint32_t x, uint32_t y) {
        while (y != 0) {
            const uint32_t r = x % y;
            x = y;
            y = r;
        }
        return x;
    };
    uint32_t step = (uint32_t)(0.6180339887 * (double)nwg);
    while (step > 1 && gcd((uint32_t)nwg, step) != 1) --step;
    return step;
}

// LDS for the slab of a workgroup of the first backward kernel that makes several passes (msda_bwd_kernel.h): 12 bytes per
// record behind the counters, when the slab is small enough to leave four workgroups to a CU and the kernel stays
// inside the default limit of dynamic LDS.  A workgroup that makes one pass of one chunk (the plain operator and the
// fused form) collects its records in its staging strips instead.  Adds the bytes to the plan.
int plan_record_buffer(mxd_msda_plan* p, const BwdLayout& L, const Dims& d, int dtype, bool plain_or_fused, int unit_split_log2)
{
    if (!L.tiles || !plain_or_fused) return 0;  // (the kernel is built with the buffer for these two sources only)
    // By default for the plain operator and its fused form, for slabs of up to 12 KiB and, with at most four units per
    // wavefront (rows of 16 lanes and more, whose staging strips are small), of up to 24 KiB (MXD_MSDA_BWD_REC_LDS=1:
    // wherever it fits).  Measured, backward: encoder levels with 2 points, float32 (12 KiB) 231 -> 216 us; 8 heads x 128
    // channels, tiles of 128 pixels (24 KiB, four units): float16 414 -> 383 us, float32 572 -> 545 us (with two units of
    // 32 lanes: 586 -> 596); geometric kernel attention (64 channels, float32, 23 KiB) 0.80 -> 0.86 ms per step -- where
    // it loses, the buffer costs the kernel a workgroup per CU, which weighs more than the partial lines.
    (void)dtype;
    const int64_t slab = L.rec_cap * (mxd::kRecDwords * 4);
    if (tuning().bwd_rec_lds < 0 && !(slab <= 12 * 1024 || p->units_per_wave <= 4)) return 0;
    const bool one_pass = plain_or_fused && p->iters == 1 && d.nl * d.np <= ((int64_t)mxd::kChunk << unit_split_log2);
    const int64_t bytes = L.rec_cap * (mxd::kRecDwords * 4);
    const int64_t total = (((int64_t)p->lds_bytes + 15) & ~(int64_t)15) + bytes;
    if (one_pass || bytes > 24 * 1024 || total > 40 * 1024 || tuning().bwd_rec_lds == 0) return 0;
    p->lds_bytes = (uint32_t)total;
    return (int)bytes;
}

// Geometry of the tile-ownership grad_value kernel (msda_bwd_tiles.hip).
int make_tile_args(const Dims& d, const BwdLayout& L, int accumulate, mxd::TileArgs* t, bool plain_operator = false)
{
    memset(t, 0, sizeof(*t));
    // pair records (counted before merging) per work item when a hot tile is split: enough items to fill the 512
    // workgroup slots of the chip about twice (measured optimum on MI355X; fewer, longer items lose to imbalance,
    // more, shorter ones to the atomics of their write-out).  Below 8192 records the write-out starts to
    // weigh more and the measured optimum falls more slowly than the problem size: geometric mean of the two
    // (0.17 M samples: 2 100, 0.5 M: 3 600, 1.3 M: 5 700 records per item).
    int64_t target = 2 * d.bs * d.nh * d.nq * d.nl * d.np / 512;
    if (target < 8192) target = (int64_t)sqrt(8192.0 * (double)(target > 32 ? target : 32));
    // (capped: 32 768 measured 0.6 to 1.7 % behind 49 152 on problems of 10 to 40 M samples, 65 536 up to 4 % behind it and
    //  100 000 up to 20 %: the launch then has too few items to fill the chip evenly)
    if (target > 49152) target = 49152;
    if (d.nl == 1) {
        // One level: its tiles all collect about the same number of records, so the launch is a whole number of
        // equal work items per tile.  Up to 512 of them run side by side in the chip's workgroup slots; a few more
        // than that make the launch last two items (measured, geometric kernel attention: 672 items 0.92 ms per
        // step, 480 items 0.81 ms, 384 items 0.87 ms).  Pick the chunk count with the least estimated duration:
        // items in flight one after another x (records per item + about 8192 records' worth of start, statistics
        // round and write-out per item).
        const int64_t nt = (d.nk + (int64_t(1) << L.tile_px_log2) - 1) >> L.tile_px_log2;
        const int64_t per_tile = 2 * d.nq * d.np / nt;
        int64_t best_c = 1;
        double best_cost = -1.0;
        for (int64_t c = 1; c <= 64 && c <= L.nwg; ++c) {
            const double items = (double)(d.bs * d.nh * nt * c);
            const double cost = (items <= 512.0 ? 1.0 : items / 512.0 + 0.5) * ((double)per_tile / (double)c + 8192.0);
            if (best_cost < 0.0 || cost < best_cost) {
                best_cost = cost;
                best_c = c;
            }
        }
        // (few records: a tile split in two pays zeros, atomic additions and, in 16 bits, a rounding pass for its rows, which weighs
        //  more than an item that lasts longer -- 28 x 57 pixels, 1596 queries x 2, 128 channels, bfloat16: 57 -> 37 us)
        const int64_t equal = (per_tile + best_c - 1) / best_c;
        if (target >= 8192 || equal > target) target = equal;
    }
    t->target = tuning().tile_target > 0 ? tuning().tile_target : (int)target;
    if (t->target < 128) t->target = 128;
    t->max_chunks = 64;
    // work items per (batch, head): sum over levels of tiles*chunks <= 2*nl*nq*np/target + nl + sum of tiles
    const int64_t items = d.nl * ((2 * d.nq * d.np + t->target - 1) / t->target + 1) + L.tbl_stride;
    if (items >= (int64_t(1) << 24)) return fail(MXD_E_SHAPE, "backward needs %lld work items per (batch, head)", (long long)items);
    t->items_per_bh = (int32_t)items;  // (the callers add TileArgs::extra)
    t->accumulate = accumulate;
    t->batch_major = tuning().tile_order > 0 ? 1 : 0;
    t->map.tile_q = 1;
    t->extra = plain_operator ? 8 : 0;
    t->items_per_bh += t->extra;
    const int64_t grid = fill_xcd_map(&t->map, d.bs, d.nh, t->items_per_bh);
    if (grid >= (int64_t(1) << 31)) return fail(MXD_E_SHAPE, "backward needs %lld workgroups, beyond the launch limit", (long long)grid);
    t->grid = (uint32_t)grid;
    t->block = mxd::kTileThreads;
    return MXD_OK;
}

// Tile mode: how the fp32 image of grad_value gets its zeros and how its rows reach the caller's tensor.  Tiles that
// one workgroup of the tile pass owns store their rows once; when the rows can be written in 16-byte pieces only the
// other rows (those that receive atomic additions) are zero-filled, and for 16-bit dtypes the owner stores rounded rows
// straight into the caller's tensor, so that only those other rows go through the fp32 image and the rounding pass.
void plan_image(mxd::KArgs* a, mxd::TileArgs* t, bool half, bool accumulate, float* image, void* grad_value, int64_t hd)
{
    a->tile_target = t->target;
    a->tile_max_chunks = t->max_chunks;
    t->store_vec = (hd % 4 == 0 && (reinterpret_cast<uintptr_t>(image) & 15u) == 0) ? 4 : 1;
    a->sparse = tuning().bwd_sparse != 0 && tuning().bwd_fill_kernel == 0 && t->store_vec == 4 && !accumulate &&
                (!half || (reinterpret_cast<uintptr_t>(grad_value) & 7u) == 0);
    a->grad_value_t = (a->sparse && half) ? grad_value : nullptr;
}

// Bytes of LDS the plain forward sets aside for the rows of the last levels (0: none).  Needs 16-byte lanes.
// LDS for the forward's level cache, 0 = run without.  The cache pays when the coarsest level fits in it
// (a quarter of the samples of a 4-level pyramid then are gathered from LDS) and costs otherwise: its
// workgroups are larger and hold more LDS, which leaves fewer wavefronts per CU.  The level shapes live in
// device memory, so the decision here rests on an estimate: in a pyramid that halves from level to level
// the last one has nk*3/(4^nl - 1) pixels.  With more than 8 units per wavefront (rows of 64 bytes) the
// staging strips alone limit the wavefronts per CU, and the cache is left out.
// MXD_MSDA_FWD_LDS set in the environment overrides the estimate (0 = off, bytes = on).
int forward_cache_bytes(int vec, int es, const Dims& d, int units_per_wave)
{
    const bool forced = tuning().fwd_lds >= 0;
    const int v = forced ? tuning().fwd_lds : 40960;
    if (!(vec * es == 16 && v >= 1024 && v <= 65536)) return 0;
    if (!forced) {
        if (units_per_wave > 8) return 0;
        // Small problems lose more to the cache fill of every workgroup than the gather gains (float32, with / without:
        // 2 x 300 queries 11.3 / 6.1 us, 8 x 900 queries 37 / 34; five levels with 4 points and 6.4 M samples 120 / 139).  Over 300
        // problems whose last level fits, with / without: float32 rows of up to 256 bytes at 1 to 2 M samples 0.77 to 1.31 (median 1.00), at
        // 2 to 4 M 0.80 to 1.13 (0.95), at 4 to 8 M 0.69 to 1.17 (0.91); 16-bit rows, whose conversions take the wavefronts that
        // hide the memory's latency, at 2 to 4 M 0.87 to 1.39 (1.04), at 4 to 8 M 0.85 to 1.11 (1.00), beyond 0.88 to 1.11 (0.95).
        const bool words = es == 4 && d.hd * es <= 256;
        if (d.bs * d.nh * d.nq * d.nl * d.np < (int64_t(1) << (words ? 21 : 23))) return 0;
        double last = (double)d.nk;
        if (d.nl > 1) last = (double)d.nk * 3.0 / ((double)(int64_t(1) << (2 * (d.nl < 16 ? d.nl : 16))) - 1.0);
        if (last * 1.1 * (double)(d.hd * es) > (double)v) return 0;
    }
    return v & ~15;
}

// Rows of the last levels that an LDS cache of `cap_rows` rows would hold, estimated for a pyramid that halves
// from level to level (the level shapes live in device memory): the last level has nk*3/(4^nl - 1) pixels.
int64_t estimated_cached_rows(const Dims& d, int64_t cap_rows)
{
    double last = (double)d.nk;
    if (d.nl > 1) last = (double)d.nk * 3.0 / ((double)(int64_t(1) << (2 * (d.nl < 16 ? d.nl : 16))) - 1.0);
    double r = last * 1.1, total = 0.0;
    for (int l = 0; l < d.nl && total + r <= (double)cap_rows; ++l) {
        total += r;
        r *= 4.0;
    }
    return (int64_t)total;
}

// Time of the forward's one-workgroup-per-CU form over that of the general kernel, estimated.  What the form gains: a row takes fewer
// instructions, and rows of cached levels come from LDS beside the others.  What it loses: its units work through whole chunks of 16
// samples, the general kernel's through as many as there are and three samples' worth of a unit's start; rows from memory cost more
// where the slices that run side by side on an XCD overflow its L2 (`spill`: by how many L2s, beyond 1.4 of them), because four
// wavefronts per SIMD hide less of it; every workgroup pays its launch and cache fill (`start`, in rows of its share) before its share
// of the rows.  Conversions weigh more here, most with 16 lanes per row (and in bfloat16, which has no mixed multiply-add).  The
// fused form's general kernel computes its softmax in a pass of its own over the samples.
// Weights fitted to 3 339 pairs of timings: one to six levels of 20 x 20 to 300 x 400 pixels, 1 to 8 points, 4, 8 and 16 heads of 16
// to 128 channels, 500 to 60 000 queries or every pixel, from a million samples on, all three types, plain and fused, uniformly
// random locations: the form chosen takes 1.6 % longer than the better of the two on average (104 of them more than 15 % longer),
// always the general kernel 7.8 %.  On 408 problems drawn afterwards: plain 1.9 % (3.9 % with separate lines for samples, cached
// levels, slices and types before it; always the general kernel 8.3 %), fused 1.5 % (1.7, 7.5).
double cu_over_general(int dtype, bool fused, int lpr, int64_t samples, double from_memory, double spill, double start)
{
    double row = 0.64;
    if (dtype != MXD_DTYPE_F32) row = lpr <= 4 ? 0.64 : lpr <= 8 ? 0.72 : dtype == MXD_DTYPE_F16 ? 0.82 : 0.9;
    if (fused) row *= 0.8;
    return row * (1.0 + 1.5 * from_memory * spill) * (double)round_up((size_t)samples, mxd::kChunk) / (double)(samples + 3) + start;
}

// The forward's one-workgroup-per-CU form (msda_fwd_cu.hip): whether a problem takes it, and its launch geometry.
// It needs 16-byte lanes, rows of at most 16 lanes and the plain operator or its fused form; it pays when at least the last level fits
// the CU's LDS and the problem is large enough to keep 256 such workgroups busy well beyond their cache fill (cu_over_general).
bool plan_forward_cu(int dtype, const Dims& d, bool fused, int vec, int lpr, int npass, mxd_msda_plan* p, int* cache_bytes)
{
    const int mode = tuning().fwd_cu;
    const int es = elem_size(dtype);
    if (mode == 0 || vec * es != 16 || npass != 1 || lpr > 16) return false;
    // What the kernel's index arithmetic assumes, whatever the environment asks for: pixel indices and the distance
    // between neighbouring pixels are multiplied as 24-bit integers, and the locations, weights, results (and the
    // fused form's reference points) of one batch element are addressed with 32-bit byte offsets inside a buffer
    // descriptor.  Anything larger goes to the general kernel, which indexes with 64-bit offsets.
    const int64_t kMul24 = int64_t(1) << 23, kOff32 = int64_t(1) << 31;
    if (d.nk >= kMul24 || d.nh * d.hd * es >= kMul24 || d.nq * d.nh * d.nl_attn * d.np * 2 * es >= kOff32 ||
        d.nq * d.nh * d.hd * es >= kOff32 || d.nq * d.nl * 2 * es >= kOff32)
        return false;
    const int cap = mxd::kCuLdsBytes - mxd::kCuTableBytes;  // (two level tables come first)
    const int64_t cap_rows = cap / (d.hd * es) - 1;
    const int64_t cached = estimated_cached_rows(d, cap_rows);
    // Levels whose rows come from LDS, estimated as above.
    double last = (double)d.nk, rows = 0.0;
    if (d.nl > 1) last = (double)d.nk * 3.0 / ((double)(int64_t(1) << (2 * (d.nl < 16 ? d.nl : 16))) - 1.0);
    int levels_cached = 0;
    for (double r = last; levels_cached < d.nl && rows + r <= (double)cap_rows; r *= 4.0) {
        rows += r;
        ++levels_cached;
    }
    // (nothing cached is nothing gained; 8 x 900 queries, under a million samples: 59 against 37 us)
    const double from_memory = (double)(d.nl - levels_cached) / (double)d.nl;
    if (mode < 0 && (levels_cached == 0 || d.bs * d.nh * d.nq * d.nl * d.np < (int64_t(1) << 20) ||
                     cu_over_general(dtype, fused, lpr, d.nl * d.np, from_memory, 0.0, 0.0) >= 1.0))
        return false;
    const int U = mxd::kWave / lpr;
    const int64_t groups = (d.nq + U - 1) / U;
    // Workgroups per (batch, head): every XCD has 32 CUs, each of which runs one workgroup at a time; the launch
    // lasts (rounds of 32 workgroups per XCD) x (cache fill + the workgroup's share of the gathers).  The rows that
    // are not cached come from the XCD's 4 MiB L2: the workgroups that run side by side on an XCD should work on as
    // few (batch, head) slices as possible (workgroups of an XCD are numbered head, query range, batch element).
    int64_t best_p = 1;
    double best_cost = -1.0, best_spill = 0.0, best_rows = 1.0;
    const int64_t max_p = groups < 512 ? groups : 512;
    const double slice_bytes = (double)(d.nk - cached) * (double)(d.hd * es);
    const double launch = 3000.0, fill = (double)cached + 1000.0;   // in units of one gathered row
    for (int64_t P = 1; P <= max_p; ++P) {
        if (tuning().fwd_cu_wgs > 0 && P != tuning().fwd_cu_wgs && tuning().fwd_cu_wgs <= max_p) continue;
        const int64_t tq = U * (((d.nq + P - 1) / P + U - 1) / U);
        const int64_t nt = (d.nq + tq - 1) / tq;
        mxd_msda_plan trial;
        memset(&trial, 0, sizeof(trial));
        const int64_t grid = fill_xcd_map(&trial, d.bs, d.nh, nt, d.hd * es);
        const double per_xcd = (double)grid / mxd::kNumXcd;
        const double rounds = ceil(per_xcd / 32.0);
        double slices = 32.0 / (double)(trial.xcd_mode == 2 ? trial.tiles_per_part : nt);  // side by side on an XCD
        if (trial.xcd_mode == 3) slices /= (double)trial.heads_per_xcd;  // (heads that share their lines fill the L2 as one)
        if (trial.xcd_mode == 1 && slices < (double)trial.heads_per_xcd) slices = (double)trial.heads_per_xcd;
        if (trial.xcd_mode == 0) slices = slices * 8.0 < (double)d.nh ? (double)d.nh : slices * 8.0;
        if (slices < 1.0) slices = 1.0;
        // (measured at the encoder shape: two slices side by side cost 10 to 15 % also where both fit the L2 --
        //  float16, 2 x 1.2 MB -- and 15 to 25 % where they do not -- float32, 2 x 2.4 MB)
        // By default only where whole heads are pinned to an XCD, at most two of them: a head that several XCDs share
        // needs so many workgroups per (batch, head) to keep the slices side by side on an XCD few that the cache fills
        // outweigh the gain.  Measured at the encoder shape with the 16 (batch, head) pairs split as bs x heads --
        // this form against the general kernel: 2 x 8: 91 / 102 us, 1 x 16: 96 / 123, 4 x 4: 102 / 102, 8 x 2: 120 / 105
        // (152 with one round of workgroups), 16 x 1: 133 / 112 (175), 2 x 6 heads, no pinning: 106 / 94.
        // (four heads, each shared by two XCDs: with the encoder's queries and two batch elements 44.8 against 50.2 us)
        if (mode < 0 && !((trial.xcd_mode == 1 && trial.heads_per_xcd <= 2) || (trial.xcd_mode == 2 && trial.xcds_per_head <= 2) ||
                           (trial.xcd_mode == 3 && trial.xcds_per_head <= 2 * trial.heads_per_xcd)))
            continue;
        double over = ceil(slices) * slice_bytes / (4.0 * 1024 * 1024) - 0.4;
        const double spill = over < 1.0 ? 0.0 : (over > 3.0 ? 2.0 : over - 1.0);
        over = over < 0.0 ? 0.0 : (over > 1.0 ? 1.0 : over);
        const double gather = (1.0 + 0.5 * over) * (double)tq * (double)(d.nl * d.np) * 4.0;
        const double cost = rounds * (launch + fill + gather);
        if (best_cost < 0.0 || cost < best_cost) {
            best_cost = cost;
            best_p = P;
            best_spill = spill;
            best_rows = (double)tq * (double)(d.nl * d.np) * 4.0;
        }
    }
    if (best_cost < 0.0) return false;  // (not a shape for this form)
    if (mode < 0 && cu_over_general(dtype, fused, lpr, d.nl * d.np, from_memory, best_spill, (launch + 3000.0 + (double)cached) / best_rows) >= 1.0)
        return false;
    const int64_t tq = U * (((d.nq + best_p - 1) / best_p + U - 1) / U);
    const int64_t nt = (d.nq + tq - 1) / tq;
    memset(p, 0, sizeof(*p));
    p->vec = vec;
    p->lanes_per_row = lpr;
    p->npass = 1;
    p->units_per_wave = U;
    p->waves_per_block = mxd::kCuWaves;
    p->iters = (int32_t)((tq / U + mxd::kCuWaves - 1) / mxd::kCuWaves);
    p->tile_q = (int32_t)tq;
    const int64_t grid = fill_xcd_map(p, d.bs, d.nh, nt, d.hd * es);
    if (grid >= (int64_t(1) << 31)) return false;
    p->grid = (uint32_t)grid;
    p->block = (uint32_t)(mxd::kCuWaves * mxd::kWave);
    p->lds_bytes = (uint32_t)mxd::kCuLdsBytes;
    *cache_bytes = cap & ~15;
    if (tuning().fwd_cu_cache >= 0 && tuning().fwd_cu_cache < *cache_bytes) {
        // (at least the row of zeros that stands for corners outside the image)
        const int least = (int)(d.hd * es + 15) & ~15;
        *cache_bytes = tuning().fwd_cu_cache < least ? least : (tuning().fwd_cu_cache & ~15);
    }
    return true;
}

// Whether half of the wavefronts of the forward's one-workgroup-per-CU form work through their chunks from the LDS
// groups on, so that memory gathers and LDS gathers of a CU's wavefronts run side by side.  Measured at the encoder
// shape (alternating launches, one box): float16 70.9 -> 69.0 us -- 16 rows of 64 bytes per load instruction keep the
// vector-memory pipeline twice as long as 8 rows of 128 bytes --, float32 78.9 -> 79.8 us: by default for 16-bit rows.
int forward_cu_flip(int dtype)
{
    const int v = tuning().fwd_cu_flip;
    return v >= 0 ? (v != 0) : (elem_size(dtype) == 2);
}

// level_cache: in/out, bytes of LDS for the forward's level cache (asked for -> granted)
// cu_form: in/out, whether the forward may take (2: in its fused form) / takes the one-workgroup-per-CU form
// align_bytes: alignment of the rows' buffers; whole_pieces: see row_geometry (launches read rows in overlapping pieces where
// no whole ones fit; the plan that mxd_msda_make_plan reports describes whole pieces)
int make_plan(int backward, int dtype, const Dims& d, int align_bytes, mxd_msda_plan* p, int* level_cache = nullptr,
              int* cu_form = nullptr, bool whole_pieces = false)
{
    const int rc = check_dims(dtype, d);
    if (rc != MXD_OK) return rc;
    const int es = elem_size(dtype);
    int vec, lpr, npass;
    // (rows in LDS -- the one-workgroup-per-CU form, the level cache -- are copied and read in aligned pieces of 16 bytes)
    const bool rows_of_16 = align_bytes >= 16 && d.hd * es % 16 == 0;
    int lane_bytes = whole_pieces ? align_bytes : 16;
    if (backward && lane_bytes > backward_lane_bytes(dtype, d)) lane_bytes = backward_lane_bytes(dtype, d);
    // (the forward keeps 32 lanes in one pass: at 8 heads x 128 channels in float32 two passes take 248 against 237 us)
    row_geometry(es, d.hd, lane_bytes, &vec, &lpr, &npass, backward && tuning().bwd_two_pass != 0, whole_pieces);
    if (!backward && rows_of_16 && cu_form && *cu_form && level_cache) {
        if (plan_forward_cu(dtype, d, *cu_form == 2, vec, lpr, npass, p, level_cache)) return MXD_OK;
    }
    if (cu_form) *cu_form = 0;
    // (a row is shared by four lanes at least: 8 bytes each for rows of 32 -- 16 channels in float16, 2 x 13253 queries of 18
    //  samples: forward 75 -> 63 us)
    if (!backward && d.hd * es <= 32 && lane_bytes > 8) row_geometry(es, d.hd, 8, &vec, &lpr, &npass, false, whole_pieces);
    memset(p, 0, sizeof(*p));
    p->vec = vec;
    p->lanes_per_row = lpr;
    p->npass = npass;
    p->units_per_wave = mxd::kWave / lpr;
    // The forward's wavefronts share nothing but the level table: in workgroups of one they start as soon as there is room for one,
    // and no wavefront waits for the others' table (300 queries 6.0 -> 5.3 us, 3 x 12824 queries of 6 samples 52.5 -> 48.9;
    // beyond some 40 000 of them the dispatch of so many workgroups costs 1 %).
    const int64_t wavefronts = d.bs * d.nh * ((d.nq + mxd::kWave / lpr - 1) / (mxd::kWave / lpr));
    p->waves_per_block = backward || wavefronts > 40000 ? 4 : 1;
    int iters = tuning().fwd_iters;
    if (iters < 1) iters = 1;
    const BwdLayout L = bwd_layout(dtype, d);
    // the tile pass wants L.tile_q queries per workgroup of the first backward kernel
    int split = 1;  // units of the backward's first kernel that share a query
    if (backward) {
        iters = L.tiles ? (int)(L.tile_q / (p->units_per_wave * p->waves_per_block)) : 1;
        if (iters < 1) {
            iters = 1;
            split = (int)(p->units_per_wave * p->waves_per_block / L.tile_q);
        }
    }
    int cache = (level_cache && *level_cache && !backward && rows_of_16) ? forward_cache_bytes(vec, es, d, p->units_per_wave) : 0;
    if (cache > 0) {
        // 8 wavefronts share one copy of the cached rows and work through 128 queries (MXD_MSDA_FWD_WGQ; 256 and
        // 64 measure within 2 % of it); two such workgroups
        // must fit a CU (80 KiB each), else fewer wavefronts, else no cache
        int waves = 8;
        while (waves > 2 && mxd::kMaxLevels * sizeof(mxd::i32x4) + (size_t)waves * p->units_per_wave *
                                    (mxd::kChunkStride * sizeof(mxd::Entry) + 2 * sizeof(float)) + cache > 80 * 1024)
            waves >>= 1;
        if (waves > 2) {
            p->waves_per_block = waves;
            iters = tuning().fwd_wgq / (p->units_per_wave * p->waves_per_block);
            if (iters < 1) iters = 1;
        } else {
            cache = 0;
        }
    }
    p->iters = iters;
    p->tile_q = p->units_per_wave * p->waves_per_block * p->iters / split;
    const int64_t ntiles = (d.nq + p->tile_q - 1) / p->tile_q;
    p->ntiles = (int32_t)ntiles;
    const int64_t grid = fill_xcd_map(p, d.bs, d.nh, ntiles, d.hd * es);
    if (grid >= (int64_t(1) << 31)) return fail(MXD_E_SHAPE, "problem needs %lld workgroups, beyond the launch limit", (long long)grid);
    p->grid = (uint32_t)grid;
    p->block = (uint32_t)(p->waves_per_block * mxd::kWave);
    if (backward) {
        p->lds_bytes = (uint32_t)backward_lds_bytes(p->units_per_wave, p->waves_per_block, L.tiles, L.tbl_stride);
    } else {
        p->lds_bytes = (uint32_t)(mxd::kMaxLevels * sizeof(mxd::i32x4) +
                                  (size_t)p->waves_per_block * p->units_per_wave * mxd::kChunkStride * sizeof(mxd::Entry));
        p->lds_bytes += (uint32_t)(p->waves_per_block * p->units_per_wave * 2 * sizeof(float));  // softmax statistics (fused form)
    }
    if (cache > 0) p->lds_bytes += (uint32_t)cache;
    if (level_cache) *level_cache = cache;
    return MXD_OK;
}

int ptr_align(const void* p)
{
    const uintptr_t v = reinterpret_cast<uintptr_t>(p);
    int a = 16;
    while (a > 1 && (v & (uintptr_t)(a - 1))) a >>= 1;
    return a;
}

// Units of the backward's first kernel that share a query, as a power of two (see bwd_tile_q).
int unit_split_log2(const mxd_msda_plan& p)
{
    const int units = p.units_per_wave * p.waves_per_block * p.iters;
    int s = 0;
    while (p.tile_q > 0 && (p.tile_q << (s + 1)) <= units) ++s;
    return s;
}

void fill_args(mxd::KArgs* a, int dtype, const Dims& d)
{
    const int es = elem_size(dtype);
    a->bs = (int32_t)d.bs;
    a->nk = (int32_t)d.nk;
    a->nh = (int32_t)d.nh;
    a->hd = (int32_t)d.hd;
    a->nl = (int32_t)d.nl;
    a->np = (int32_t)d.np;
    a->nq = (int32_t)d.nq;
    a->S = (int32_t)(d.nl * d.np);
    a->S_full = (int32_t)(d.nl_attn * d.np);
    const int64_t S = d.nl * d.np, n0 = S < mxd::kChunk ? S : mxd::kChunk, n1 = S % mxd::kChunk ? S % mxd::kChunk : mxd::kChunk;
    a->chunk_magic = (uint32_t)(((1 << 16) + n0 - 1) / n0);
    a->tail_magic = (uint32_t)(((1 << 16) + n1 - 1) / n1);
    a->np_magic = (uint32_t)(((1u << 20) + d.np - 1) / d.np);
    a->pitch_bytes = (uint32_t)(d.nh * d.hd * es);
    a->batch_bytes = (uint32_t)(d.nk * d.nh * d.hd * es);
    a->gbatch_bytes = (uint32_t)(d.nk * d.nh * d.hd * 4);
}

int log2_lanes(int64_t lanes)
{
    int s = 0;
    while ((int64_t(1) << s) < lanes && s < 6) ++s;
    return s;
}

// Checks the sizes of a deformable aggregation and fills in what follows from them.
int dagg_args(int dtype, int64_t bs, int64_t nf, int64_t C, int64_t cams, int64_t scales, int64_t A, int64_t P, int64_t G,
              mxd::DaggArgs* a)
{
    if (G <= 0 || cams <= 0 || scales <= 0 || C <= 0)
        return fail(MXD_E_SHAPE, "Input Tensor can not be a empty Tensor (C=%lld cams=%lld scales=%lld groups=%lld)",
                    (long long)C, (long long)cams, (long long)scales, (long long)G);
    if (C % G != 0) return fail(MXD_E_SHAPE, "num_embeds (%lld) must be a multiple of num_groups (%lld)", (long long)C, (long long)G);
    const Dims d{bs, nf, G, C / G, cams * scales, cams * scales, A, P};  // (a group is a head, a (camera, scale) pair a level)
    const int rc = check_dims(dtype, d);
    if (rc != MXD_OK) return rc;
    if (A >= (int64_t(1) << 29) || A * P * d.nl >= (int64_t(1) << 31) || bs * A >= (int64_t(1) << 30))
        return fail(MXD_E_SHAPE, "num_anchors*num_pts*num_cams*num_scale = %lld is beyond what this build indexes", (long long)(A * P * d.nl));
    memset(a, 0, sizeof(*a));
    const int es = elem_size(dtype);
    a->bs = (int32_t)bs;
    a->nf = (int32_t)nf;
    a->C = (int32_t)C;
    a->G = (int32_t)G;
    a->hd = (int32_t)d.hd;
    a->cams = (int32_t)cams;
    a->scales = (int32_t)scales;
    a->nl = (int32_t)d.nl;
    a->A = (int32_t)A;
    a->P = (int32_t)P;
    a->nloc = (int32_t)(P * cams);
    a->p_magic = (uint32_t)(((1u << 20) + P - 1) / P);
    a->sc_magic = (uint32_t)(((1u << 20) + scales - 1) / scales);
    a->pitch_bytes = (uint32_t)(C * es);
    a->batch_bytes = (uint32_t)(nf * C * es);
    const int vec = mxd::dagg_vec(es, C);
    a->row_lpr_log2 = log2_lanes((C + vec - 1) / vec);
    a->row_blocks = (int32_t)(((C + vec - 1) / vec + mxd::kWave - 1) / mxd::kWave);
    a->sort_ranges = (int32_t)((nf + mxd::kDaggSortPx - 1) / mxd::kDaggSortPx);
    a->starts = mxd::dagg_starts(nf, d.nl);
    // A unit of lanes goes through a strip's records one batch after the other, a trip to memory each.  Where the strips alone leave
    // the chip short of units they are split down to 96 records (829 anchors x 9 points, 4 levels from 58 x 28, 64 channels: 90 us
    // with parts of 1024 records, 27 with 96, 31 with 64); a split costs zeros and atomic additions, so that strips enough for two
    // thirds of 16 wavefronts per CU are split only where samples pile up.
    const int64_t strips = bs * (nf / mxd::kDaggStrip + d.nl) * a->row_blocks, units = 16 * 256 * (mxd::kWave >> a->row_lpr_log2);
    a->strip_records = 3 * strips >= 2 * units ? 1024 : 96;
    return MXD_OK;
}

// Launch geometry of the forward (or of the backward's first kernel): an anchor per wavefront and row piece.
int dagg_plan(mxd::DaggArgs* a, int es, bool backward)
{
    // A piece is a group's channels.  In the forward several groups share one where a group's row is short of the 128
    // bytes of a cache line (float16, groups of 32 channels: a line that two XCDs fetch for half of it each), if the lanes'
    // channels do not straddle groups; the backward's dot products belong to one group each.
    int vec = mxd::dagg_vec(es, a->hd);
    a->piece_ch = a->hd;
    a->piece_heads = 1;
    if (!backward && a->hd % vec == 0 && a->hd * es < 128 && a->G > 1) {
        a->piece_ch = 128 / es < a->C ? 128 / es : a->C;
        // (at most 32 of them: a wavefront keeps the weights of 64 samples per group in LDS, and those of 64 groups would take the
        //  workgroup to 80 KiB, beyond what a kernel is promised without opting in; 128 groups of one channel, 900 anchors x 13 points in six
        //  cameras, float16: 64 / 32 groups a piece 114 / 85 us)
        if (a->piece_ch > 32 * a->hd) a->piece_ch = 32 * a->hd;
        a->piece_heads = a->piece_ch % a->hd == 0 ? a->piece_ch / a->hd : (a->piece_ch - 1) / a->hd + 2;
    }
    a->pieces = (a->C + a->piece_ch - 1) / a->piece_ch;
    a->lpr_log2 = log2_lanes((a->piece_ch + vec - 1) / vec);
    const int waves = backward ? mxd::kDaggBackWaves : mxd::kDaggWaves;
    a->map.tile_q = waves;
    const int64_t grid = fill_xcd_map(&a->map, a->bs, a->pieces, (a->A + waves - 1) / waves);
    if (grid >= (int64_t(1) << 31)) return fail(MXD_E_SHAPE, "problem needs %lld workgroups, beyond the launch limit", (long long)grid);
    if ((int64_t)a->bs * a->nl * a->sort_ranges >= (int64_t(1) << 31)) return fail(MXD_E_SHAPE, "problem needs too many workgroups");
    a->map.grid = (uint32_t)grid;
    return MXD_OK;
}

// Whether the kernel that forms the rows of grad_feat forms the dot products as well: it has a sample's grad_out row at hand, in the
// order of the pixels, so that every value row is read once, in order, in place of a gather of four rows per sample and group that
// misses the L2 in two fifths of them.  In return the sort is no longer hidden behind that gather (43 us), and rows that few samples
// touch are read whole.  6 x 900 anchors x 13 points, six cameras of four scales (538k pixels), 256 channels of float32: 320 + 224 +
// 42 us for the three kernels, 43 + 351 + 50 with this.  Which is faster is a matter of that gather: a
// wavefront of it per anchor and group costs as much as 40 locations and the locations that it looks at, times the 128-byte lines of
// a group's row; where the maps fit the caches it takes half of that.  The backward's time that way over this way (256 channels in
// groups of 32, two fifths of the locations inside):
//   900 anchors x 13 points, maps of 92 MB: 1 / 2 / 3 / 4 / 6 batch elements (0.85 M each by that count) 0.82 / 0.91 / 1.18 / 1.27 / 1.36; groups
//   of 8 channels (3.4 M) 1.01 / 1.38 / 1.56 / 1.69 / 1.81; 512 channels (1.7 M) 0.97 / 1.21 / 1.32 / 1.37 / 1.39; maps of 23 MB 0.77 / 1.01 / 0.98 /
//   0.95 / 1.13; 600 anchors (0.57 M): 2 / 3 / 4 / 6 / 8 0.80 / 0.87 / 1.06 / 1.21 / 1.27; 300 (0.28 M): 4 / 6 / 8 / 12 0.85 / 0.95 / 1.02 / 1.02.
// Over 473 problems of all sizes this line is 1.7 % from the faster way on average (never this way: 11 %, always: 7 %).
// Rows of 128 channels, which units of less than a wavefront share, were at 0.87 .. 1.02, 16-bit rows at 0.71 .. 1.05: not for them.
bool dagg_dots_with_rows(const mxd::DaggArgs& a, int es)
{
    const int lanes = a.hd / 4;
    if (es != 4 || a.C % 256 != 0 || a.hd % 4 != 0 || lanes > mxd::kWave || (lanes & (lanes - 1)) != 0) return false;
    if (a.G > mxd::kWave || (a.G & (a.G - 1)) != 0) return false;
    const int64_t samples = (int64_t)a.A * a.P * a.nl;
    const int64_t gather = a.bs * (int64_t)a.A * a.G * (a.nloc + 40) * (a.hd > 32 ? a.hd / 32 : 1);
    return samples >= a.nf && gather >= ((int64_t)a.bs * a.nf * a.C * 4 >= (int64_t(64) << 20) ? 2400000 : 4800000);
}

// Workspace of the backward: {weights' gradients per group, location gradients per group (or the samples' dot products), record starts, records, float32
// image of grad_mc_ms_feat for 16-bit dtypes}.
struct DaggSpace {
    size_t gl, csr, rec, image, total;
    DaggSpace(const mxd::DaggArgs& a, int es)
    {
        const size_t locs = (size_t)a.bs * a.A * a.nloc;
        gl = round_up((size_t)a.G * locs * a.scales * 4, 256);
        csr = gl + round_up((size_t)a.G * locs * 8, 256);
        if (dagg_dots_with_rows(a, es)) {
            const size_t dots = round_up((size_t)a.G * locs * a.scales * 16, 256);
            if (csr < dots) csr = dots;
        }
        rec = csr + round_up((size_t)a.bs * (size_t)a.starts * 4, 256);
        image = rec + (size_t)a.bs * a.nl * 2 * a.A * a.P * 16;
        total = image + (es == 2 ? (size_t)a.bs * a.nf * a.C * 4 : 0);
    }
};

int64_t ceil_div(int64_t x, int64_t y) { return (x + y - 1) / y; }

// Workgroups per (batch, head) such that `slots` of them run side by side: as many rounds of whole launches as cost least, each
// paying `fixed` (in units of one query's work) before its queries.
int64_t gka_splits(int64_t slabs, int64_t nq, int64_t slots, double fixed, int64_t least)
{
    int64_t best = 1;
    double best_cost = -1.0;
    for (int64_t s = 1; s <= 64 && (s == 1 || nq / s >= least); ++s) {
        const double cost = (double)ceil_div(slabs * s, slots) * ((double)ceil_div(nq, s) + fixed);
        if (best_cost < 0.0 || cost < best_cost) {
            best_cost = cost;
            best = s;
        }
    }
    return best;
}

// Geometric kernel attention with the (batch, head)'s slab of value in LDS (gka.hip), `parts` of its channels at a time: whether the
// part's slab, in the dtype for the gather and as float32 sums in registers for grad_value, fits, and the launch geometry.  Without
// `gather` the slab in LDS is not asked for where the scatter forms the dots, which then is the backward's only kernel over the samples.
bool gka_plan_parts(int dtype, const Dims& d, int64_t parts, bool gather, mxd::GkaArgs* a)
{
    memset(a, 0, sizeof(*a));
    const int es = elem_size(dtype);
    const int64_t ch = d.hd / parts, row = ch * es, lanes = row / 16, sc_lanes = ch / 4, S = d.nl * d.np;
    if (d.hd % parts != 0 || row % 16 != 0 || (lanes & (lanes - 1)) != 0 || lanes < 2 || lanes > 32 || sc_lanes > 64) return false;
    a->bs = (int32_t)d.bs;
    a->nk = (int32_t)d.nk;
    a->nh = (int32_t)d.nh;
    a->hd = (int32_t)d.hd;
    a->nl = (int32_t)d.nl;
    a->np = (int32_t)d.np;
    a->nq = (int32_t)d.nq;
    a->S = (int32_t)S;
    a->np_magic = (uint32_t)(((1u << 20) + d.np - 1) / d.np);
    a->s_magic = (uint32_t)(((1u << 20) + S - 1) / S);
    a->parts = (int32_t)parts;
    a->part_ch = (int32_t)ch;
    a->lpr_log2 = log2_lanes((int)lanes);
    // gather: two workgroups of 8 wavefronts per CU, or one of 16
    const int64_t slab = (d.nk + 1) * row, strip = (64 / lanes) * mxd::kChunkStride * 8, lim = mxd::kCuLdsBytes - 256;
    const int64_t lds2 = mxd::kGkaLevelBytes + slab + 8 * strip, lds1 = mxd::kGkaLevelBytes + slab + 16 * strip;
    const bool two = 2 * lds2 <= lim || lds1 > lim;
    a->block = two ? 512 : 1024;
    a->lds = (uint32_t)(two ? lds2 : lds1);
    if ((two ? lds2 : lds1) > lim && (gather || sc_lanes < 4)) return false;
    const int64_t slabs = d.bs * d.nh * parts;
    int64_t s = gka_splits(slabs, d.nq, 2 * (int64_t)a->lds <= lim ? 512 : 256, (double)d.nk / 2, 64 / lanes * (a->block / 64));
    a->split_q = (int32_t)ceil_div(d.nq, s);
    a->splits = (int32_t)ceil_div(d.nq, a->split_q);
    // grad_value: tiles of queries that let two workgroups share a CU's LDS
    a->sc_lanes_log2 = log2_lanes((int)sc_lanes);
    a->sc_block = ceil_div(d.nk, 512 / sc_lanes) <= mxd::kGkaPixels ? 512 : 1024;
    a->sc_px = (int32_t)ceil_div(d.nk, a->sc_block / sc_lanes);
    if (a->sc_px > mxd::kGkaPixels) return false;
    // (places for pixels in the lane groups: as many as the kernel is built for)
    const int64_t places = sc_lanes < 4 ? 0 : ceil_div(a->sc_px, 4) * 4 * (a->sc_block / sc_lanes);
    const int64_t tables = row + (2 * d.nk + 1 + mxd::kWave) * 4 + places * 2;
    const int64_t room = (a->sc_block == 512 ? lim / 2 : lim) - mxd::kGkaLevelBytes - tables - 32;
    int64_t tile = room / (row + S * 8);
    if (tile > mxd::gka_samples(a->sc_px, sc_lanes >= 4) * a->sc_block / S) tile = mxd::gka_samples(a->sc_px, sc_lanes >= 4) * a->sc_block / S;
    if (tile * S * S >= (1 << 20)) tile = (1 << 20) / (S * S) - 1;
    if (tile > 4088) tile = 4088;  // (32-bit products of the division by S)
    const int64_t reach = (int64_t(1) << 31) / (d.nh * (S * 8 > d.hd * es ? S * 8 : d.hd * es));  // (32-bit offsets of locations and rows)
    if (tile > reach) tile = reach;
    if (tile > d.nq) tile = d.nq;
    if (tile >= 8) tile &= ~(int64_t)7;
    if (tile < 8 && tile < d.nq) return false;
    a->sc_tile_q = (int32_t)tile;
    s = gka_splits(slabs, d.nq, a->sc_block == 512 ? 512 : 256, (double)tile, tile);
    a->sc_split_q = (int32_t)ceil_div(d.nq, s);
    a->sc_splits = (int32_t)ceil_div(d.nq, a->sc_split_q);
    // The scatter forms the dots from the rows that it reads anyway; lane pairs (8 channels in float32) cannot.
    a->sc_dots = sc_lanes >= 4;
    a->sc_lds = (uint32_t)(mxd::kGkaLevelBytes + ((tile * S * 8 + 15) & ~15) + tile * row + tables);
    return true;
}

// Whether these kernels take a problem.  Forward: whole rows only (with the channels in two parts, which read the locations twice, it
// takes 36 us where the general kernel takes 29), and from as many samples on as pay for the slabs' way into LDS, general kernel / this
// one at 64 channels, 375 pixels, 15 points, 2 batch elements x 4 heads: float32 0.52 million samples 8.7 / 6.6 us, 1.0 million 14.4 /
// 8.8, 3 million 39 / 20; float16, whose rows cost the general kernel half as many lines, 0.52 million 6.7 / 7.4, 0.7 million 7.5 /
// 7.6, 1.0 million 11.0 / 9.3, 3 million 27.6 / 19.4 (of five maps of 160 to 2400 pixels two are even or better at 0.7 million and
// three at 1.0 million; in float32 three of four at half a million).  16-bit units of fewer than 4 samples stay with the general
// kernel (1 to 3 samples: 0.9 to 1.2 of its time), with fewer than 8 slabs those of fewer than 12 (four slabs: 1 sample 1.5, 4 samples 1.1
// to 1.3, 8 samples 1.0 to 1.2, 12 samples 0.9 to 1.0).  Backward: wherever the slab fits, whole or in two parts (48 x 24 pixels, 64 channels, float32,
// two parts: 180 -> 112 us; in four parts 64 x 46 pixels of 32 channels went from 80 to 107 us).  Maps whose slab does not fit, float32, go to
// the scatter whole where it takes them (its rows of value stay in registers) if two parts would leave rows of 8 channels to lane pairs, whose dots
// are a gather of their own -- 60 x 43 and 45 x 60 pixels of 16 channels, 26 sizes: 1.2 to 2.0 times as fast as in parts -- and from 1.5 million
// samples on, 16 to 128 channels: 1.06 to 2.7 times as fast as in two parts, which sort the samples twice, or as the general kernels.  Fewer fill the chip
// better in two parts: 1.3 million samples 0.95 to 1.4, 0.6 0.89 to 1.4, 0.3 0.7 to 0.9.
bool gka_plan(int dtype, const Dims& d, bool backward, mxd::GkaArgs* a)
{
    const int mode = tuning().gka_slab;
    if (mode == 0 || tuning().bwd_atomic || d.nk >= 32768 || d.nl * d.np > 256 || d.nl != d.nl_attn || d.bs * d.nh > 65536) return false;
    if (!backward) {
        const bool half = elem_size(dtype) == 2, pays = d.bs * d.nh * d.nq * d.nl * d.np >= (half ? int64_t(7) << 17 : int64_t(1) << 19) &&
                                                        (!half || d.nl * d.np >= (d.bs * d.nh < 8 ? 12 : 4));
        return (mode > 0 || pays) && gka_plan_parts(dtype, d, 1, true, a);
    }
    if (gka_plan_parts(dtype, d, 1, true, a)) return true;
    mxd::GkaArgs two;
    const bool parts = gka_plan_parts(dtype, d, 2, true, &two), many = mode > 0 || d.bs * d.nh * d.nq * d.nl * d.np >= int64_t(3) << 19;
    if ((many || (parts && !two.sc_dots)) && gka_plan_parts(dtype, d, 1, false, a)) return true;
    if (parts) *a = two;
    return parts;
}

// Workspace of its backward: images of grad_value, dots of the channel parts.
size_t gka_image_bytes(const mxd::GkaArgs& a) { return round_up((size_t)a.sc_splits * a.bs * a.nk * a.nh * a.hd * sizeof(float), 256); }
size_t gka_part_bytes(const mxd::GkaArgs& a)
{
    return gka_image_bytes(a) + (a.parts > 1 ? (size_t)a.parts * a.bs * a.nq * a.nh * a.S * sizeof(float) : 0);
}

// Grid sampler on planes: whether a plane fits the LDS of a CU (as float32, whatever the dtype) and every index its type.
bool grid_planes_fit(int64_t n, int64_t c, int64_t h, int64_t w, int64_t h_out, int64_t w_out)
{
    const int64_t lim = int64_t(1) << 28;
    if (n <= 0 || c <= 0 || h <= 0 || w <= 0 || h_out <= 0 || w_out <= 0 || c > 256 || n >= (1 << 20)) return false;
    if (h >= lim || w >= lim || h_out >= lim || w_out >= lim || h_out * w_out >= lim) return false;
    return h * w * 4 <= mxd::kCuLdsBytes;
}

// Sizes, and the work split: how many planes a workgroup takes and, where there are few, how the output pixels are shared out.
// Small planes share a workgroup (one geometry for all of them) as long as two workgroups per CU are left; large ones (one
// workgroup per CU) get more threads.
int grid_planes_args(int dtype, int64_t n, int64_t c, int64_t h, int64_t w, int64_t h_out, int64_t w_out, int mode, mxd::GridArgs* a)
{
    const int es = elem_size(dtype);
    if (es == 0) return fail(MXD_E_DTYPE, "dtype code %d is not float32(0)/float16(1)/bfloat16(2)", dtype);
    if (!grid_planes_fit(n, c, h, w, h_out, w_out))
        return fail(MXD_E_SHAPE, "grid_sampler2d: [%lld, %lld, %lld, %lld] is beyond what the kernels for planes take", (long long)n,
                    (long long)c, (long long)h, (long long)w);
    memset(a, 0, sizeof(*a));
    a->n = (int32_t)n;
    a->c = (int32_t)c;
    a->h = (int32_t)h;
    a->w = (int32_t)w;
    a->outs = (int32_t)(h_out * w_out);
    a->mode = mode;
    return MXD_OK;
}

constexpr int64_t kGridFill = 512;  // workgroups aimed at: two per CU

// Planes of `bytes` that a workgroup takes when `items` of them have to be shared out.
int64_t grid_planes_together(int64_t bytes, int64_t c, int64_t n)
{
    int64_t k = mxd::kGridStageBytes / bytes;
    if (k > ceil_div(n * c, kGridFill)) k = ceil_div(n * c, kGridFill);
    if (k > c) k = c;
    return k < 1 ? 1 : k;
}

int grid_block(int64_t lds) { return 2 * lds > mxd::kCuLdsBytes ? 2 * mxd::kGridThreads : mxd::kGridThreads; }

// Planes one after the other, the geometry kept: for planes of 20 KB and more (below, several share a workgroup and its geometry already:
// 60 x 128 of 40 x 100, float32, 62 -> 53 us for 60 x 70 samples but 29 -> 33 for 20 x 30; 24 x 128 of 64 x 88, float16, 26 -> 30) and for runs
// at least twice as long as what would share (24 x 64 of 64 x 88 in float32, three a run: 14.0 -> 14.5; 24 x 128 of them 23 -> 21).
// 24 x 128 planes of 64 x 176 and 24 x 176 samples: 51 -> 39 us, float16 29.0 -> 26.2; 24 x 80 of 80 x 160 and 90 x 100 samples 58 -> 42.
// The run's length: the least of rounds of workgroups times planes, and one more for a run's start.
bool grid_planes_run_plan(int es, mxd::GridArgs* a)
{
    const int64_t px = (int64_t)a->h * a->w, block = 2 * mxd::kGridThreads, each = ceil_div(a->outs, block);
    const int64_t lds = ((mxd::grid_margin(es, a->w) + px + a->w + 1) * es + 15) & ~int64_t(15);
    const int64_t slots = 2 * lds <= mxd::kCuLdsBytes && each <= mxd::grid_run_px(es) ? kGridFill : kGridFill / 2;
    if (px * es < 20 * 1024 || lds > mxd::kCuLdsBytes || each > mxd::kGridMaxPx || (int64_t)a->n * a->c < 2 * slots) return false;
    int64_t best = INT64_MAX, run = 0;
    for (int64_t planes = a->c; planes >= 2; --planes) {
        const int64_t cost = ceil_div(a->n * ceil_div(a->c, planes), slots) * (planes + 1);
        if (cost < best || (cost == best && ceil_div(a->c, planes) == ceil_div(a->c, run))) {
            best = cost;
            run = planes;
        }
    }
    if (run <= 2 * (mxd::kGridStageBytes / (px * es))) return false;
    // How much of their rounds the runs must fill, and how long they may be, by the output pixels per thread, whose geometry is what a run saves.  (A
    // workgroup per plane leaves no round empty and has more planes on their way at a time.)  That form / this one over 590 sizes:
    // from 1.8 pixels per thread on 0.97 to 1.51 with two workgroups per CU, whatever the fill, with one 1.00 to 1.66 from 0.6 full on (0.81 to 1.11
    // at 0.5), but planes of 20 to 23 KB from 0.9 on (0.89 to 1.05 below).  Fewer pixels: 0.67 to 1.14 at 0.5 to 0.68; from 0.7 on, above one
    // pixel, 0.98 to 1.28 in runs of up to ten planes, 0.83 to 1.16 in longer ones, up to one pixel 0.97 to 1.21 in runs of up to five, 0.83 to 1.12 in longer ones.
    const bool two = slots == kGridFill, few = 5 * (int64_t)a->outs < 9 * block;
    const double fill = (double)((int64_t)a->n * a->c) / (double)(slots * run * ceil_div(a->n * ceil_div(a->c, run), slots));
    if (fill < (few ? 0.7 : two ? 0.0 : px * es < 24 * 1024 ? 0.9 : 0.6)) return false;
    if (few && run > (each > 1 && two ? 10 : 5)) return false;
    a->planes = (int32_t)run;
    a->chunks = (int32_t)ceil_div(a->c, run);
    a->run_px = (int32_t)each;
    a->splits = 1;
    a->block = (int32_t)block;
    a->lds = (uint32_t)lds;
    return true;
}

int grid_planes_forward_plan(int es, mxd::GridArgs* a)
{
    if (grid_planes_run_plan(es, a)) return MXD_OK;
    const int64_t bytes = (int64_t)a->h * a->w * es;
    a->planes = (int32_t)grid_planes_together(bytes, a->c, a->n);
    a->chunks = (int32_t)ceil_div(a->c, a->planes);
    a->lds = (uint32_t)((a->planes * bytes + 15) & ~15);
    a->block = grid_block(a->lds);
    // few planes: each is read by several workgroups, of at least one pass of their threads
    int64_t splits = ceil_div(kGridFill, (int64_t)a->n * a->chunks);
    if (splits > ceil_div(a->outs, a->block)) splits = ceil_div(a->outs, a->block);
    a->split_px = (int32_t)ceil_div(a->outs, splits);
    a->splits = (int32_t)ceil_div(a->outs, a->split_px);
    if ((int64_t)a->n * a->chunks * a->splits >= (int64_t(1) << 31)) return fail(MXD_E_SHAPE, "problem needs too many workgroups");
    return MXD_OK;
}

// Both gradients by the same workgroups, each a chunk of an image's channels, plane by plane: for planes whose float64 sums take
// more than half of a CU's LDS, so that the two kinds of workgroups get one at a time onto a CU, and which fit it together with the
// plane; at least one plane per CU, and no more output pixels than the registers of a workgroup hold.  24 x 128 planes of 64 x 176:
// 122 -> 82 us, 2 x 128 of 70 x 150 12.7 -> 11.2, 300 x 8 of 80 x 160 in float16 with the sum over chunks 88 -> 73.  Below the line it
// gains or loses: 23 x 128 planes of 70 x 110 104 -> 95, 10 x 64 of them 28.6 -> 29.2, 300 x 8 of 75 x 95 52 -> 61, 24 x 64 of 32 x 88 30 -> 33.
//
// Chunks per image: what costs least of rounds of workgroups times planes, a plane and a half more for a workgroup's start and, from two
// chunks on, the sum over them (some 4.5 us, and 4 more for 128 images of 24 x 176 output pixels; a plane takes some 6).  From one round of workgroups
// to four; never more chunks than the two kinds would make, whose sums size the workspace.  (One round alone leaves half of the chip idle
// where the images are not many fewer than the CUs: 130 x 64 planes of 64 x 176 388 us in one chunk, 274 + 12 in three, two kinds of
// workgroups 322 + 12; 300 x 64 767, in two 590 + 24, two kinds 710 + 25.)
bool grid_planes_both_plan(int es, mxd::GridArgs* a)
{
    const int64_t px = (int64_t)a->h * a->w, block = 2 * mxd::kGridThreads, cus = kGridFill / 2, n = a->n;
    const int64_t lds = mxd::grid_sums_bytes(px) + (((px + a->w + 1) * es + 15) & ~int64_t(15)) + mxd::kWave * 8;
    if (2 * px * 8 <= mxd::kCuLdsBytes || lds > mxd::kCuLdsBytes || a->outs > block * mxd::kGridMaxPx || n * a->c < cus) return false;
    int64_t chunks = 1;
    double best = 0.0;
    auto consider = [&](int64_t k) {
        const int64_t planes = ceil_div(a->c, k), wgs = n * ceil_div(a->c, planes);
        const double cost = (double)ceil_div(wgs, cus) * ((double)planes + 1.5) + (k > 1 ? 0.75 + (double)n / 128.0 : 0.0);
        if (best == 0.0 || cost < best) {
            best = cost;
            chunks = k;
        }
    };
    consider(1);
    for (int64_t k = cus / n < 2 ? 2 : cus / n; k <= a->gg_chunks && n * k <= 4 * cus + n; ++k) consider(k);
    // Where the two kinds make one chunk too (one channel, or two images per CU and more) nothing is summed either way, and an image count just
    // beyond a whole number of rounds leaves theirs the faster ones (their time in planes, fitted to these): 300 x 1 planes 21.9 / 23.4 us,
    // 400 x 1 27.2 / 25.0, 513 x 3 68.6 / 73.9, 520 x 16 328 / 310; 300 x 1 of 70 x 150 with 96 x 96 output pixels 38 / 43, 400 x 1 48 / 46.  With one output
    // pixel per thread the step between planes is most of it: 257 x 1 of 75 x 160, 12 x 20, float16, 9.2 / 7.9.
    const double rounds = (double)ceil_div(n, cus);
    if (a->gg_chunks == 1 && a->outs > block && rounds * ((double)a->c + 1.0) > (double)n * ((double)a->c + 0.5) / 168.0 + 0.95) return false;
    a->gb_channels = (int32_t)ceil_div(a->c, chunks);
    a->gb_chunks = (int32_t)ceil_div(a->c, a->gb_channels);
    a->gb_px = (int32_t)ceil_div(a->outs, block);
    a->gb_wgs = a->n * a->gb_chunks;
    a->sum_chunks = a->gb_chunks;
    a->block = (int32_t)block;
    a->lds = (uint32_t)lds;
    return true;
}

int grid_planes_backward_plan(int es, bool maps, bool points, mxd::GridArgs* a)
{
    const int64_t px = (int64_t)a->h * a->w, images = a->n;
    int64_t lds = 0, wgs = 0;
    a->gx_planes = (int32_t)grid_planes_together(px * 8, a->c, images);
    a->gx_chunks = (int32_t)ceil_div(a->c, a->gx_planes);
    a->gx_bands = (int32_t)ceil_div(px * 8, mxd::kCuLdsBytes);  // (a plane whole where it fits: two bands of 45 KB took 85 us, one plane 77)
    a->gx_band_px = (int32_t)ceil_div(px, a->gx_bands);
    a->gx_bands = (int32_t)ceil_div(px, a->gx_band_px);
    if (maps) {
        wgs = images * a->gx_chunks * a->gx_bands;
        lds = (int64_t)a->gx_planes * a->gx_band_px * 8;
    }
    a->gx_wgs = (int32_t)wgs;
    a->block = grid_block((int64_t)a->gx_planes * a->gx_band_px * 8);
    a->gg_ranges = (int32_t)ceil_div(a->outs, (int64_t)a->block * mxd::kGridMaxPx);
    a->gg_px = (int32_t)ceil_div(a->outs, (int64_t)a->block * a->gg_ranges);
    a->gg_ranges = (int32_t)ceil_div(a->outs, (int64_t)a->block * a->gg_px);
    // as many channels per workgroup as leave the chip full: every chunk more is one more image of sums to write and to read
    int64_t channels = images * a->gg_ranges * a->c / kGridFill;
    if (channels > a->c) channels = a->c;
    if (channels < 1) channels = 1;
    a->gg_chunks = (int32_t)ceil_div(a->c, channels);
    a->gg_channels = (int32_t)ceil_div(a->c, a->gg_chunks);
    a->gg_chunks = (int32_t)ceil_div(a->c, a->gg_channels);
    int64_t staged = (lds > mxd::kGridStageBytes ? lds : mxd::kGridStageBytes) / (px * es);
    if (staged > a->gg_channels) staged = a->gg_channels;
    a->gg_planes = (int32_t)(staged < 1 ? 1 : staged);
    if (maps && points && grid_planes_both_plan(es, a)) return MXD_OK;
    if (points) {
        const int64_t gg = images * a->gg_chunks * a->gg_ranges;
        if (a->gg_planes * px * es > lds) lds = a->gg_planes * px * es;
        wgs += gg;
        a->gg_wgs = (int32_t)gg;
        a->sum_chunks = a->gg_chunks;
    }
    if (wgs >= (int64_t(1) << 31)) return fail(MXD_E_SHAPE, "problem needs too many workgroups");
    a->lds = (uint32_t)((lds + 15) & ~15);
    return MXD_OK;
}

size_t grid_part_bytes(const mxd::GridArgs& a)
{
    return a.gg_chunks > 1 ? (size_t)a.gg_chunks * a.n * a.outs * 2 * sizeof(float) : 0;
}

}  // namespace

extern "C" {

int mxd_msda_version(void) { return MXD_MSDA_VERSION; }

const char* mxd_msda_last_error(void) { return g_err; }

int mxd_msda_make_plan(int backward, int dtype, int64_t bs, int64_t nk, int64_t nh, int64_t hd, int64_t nl, int64_t nl_attn,
                  int64_t nq, int64_t np, int align_bytes, mxd_msda_plan* plan)
{
    take_meta_flag(&dtype);
    if (!plan) return fail(MXD_E_NULL, "plan is NULL");
    const Dims d{bs, nk, nh, hd, nl, nl_attn, nq, np};
    int cache = 1, cu = 1;
    return make_plan(backward != 0, dtype, d, align_bytes, plan, &cache, &cu, true);
}

int mxd_msda_init(void)
{
    tuning();
    return ensure_device_ready();
}

void mxd_msda_reload_tuning(void) { tuning(); read_tuning(); }

int mxd_msda_decode_block(const mxd_msda_plan* plan, uint32_t block_index, int64_t bs, int64_t nh, int64_t nq,
                          int32_t work[4])
{
    if (!plan || !work) return 0;
    mxd::Work w;
    if (!mxd::decode_block(*plan, block_index, (int32_t)bs, (int32_t)nh, (int32_t)nq, &w)) return 0;
    work[0] = w.b;
    work[1] = w.h;
    work[2] = w.q_begin;
    work[3] = w.q_end;
    return 1;
}

// kind: 0 multi-scale deformable attention, 1 geometric kernel attention, >= 2: grid sampler with mode kind - 1
static int forward_common(int kind, const void* value, const int32_t* spatial_shapes, const int32_t* level_start_index,
                          const void* sampling_loc, const void* attn_weight, void* output, int dtype, int64_t bs,
                          int64_t nk, int64_t nh, int64_t hd, int64_t nl, int64_t nl_attn, int64_t nq, int64_t np,
                          void* hip_stream, int64_t grid_h = 0, int64_t grid_w = 0)
{
    const int meta64 = take_meta_flag(&dtype);
    const Dims d{bs, nk, nh, hd, nl, nl_attn, nq, np};
    const int gka = kind == 1, grid = kind >= 2 ? kind - 1 : 0;
    const char* who = grid ? "mxd_grid_sampler2d_forward" : gka ? "mxd_gka_forward" : "mxd_msda_forward";
    int rc = check_dims(dtype, d);
    if (rc != MXD_OK) return rc;
    if (!value || !sampling_loc || !output || (!grid && (!spatial_shapes || !level_start_index || !attn_weight)))
        return fail(MXD_E_NULL, "%s: NULL data pointer", who);
    int align = ptr_align(value);
    if (ptr_align(output) < align) align = ptr_align(output);
    mxd::KArgs a;
    memset(&a, 0, sizeof(a));
    rc = ensure_device_ready();
    if (rc != MXD_OK) return rc;
    int cache = kind == 0;
    // (the one-workgroup-per-CU form reads a location pair with one load)
    int cu = kind == 0 && ptr_align(sampling_loc) >= 2 * elem_size(dtype);
    rc = make_plan(0, dtype, d, align, &a.plan, &cache, &cu);
    if (rc != MXD_OK) return rc;
    fill_args(&a, dtype, d);
    a.meta_i64 = meta64;
    a.value = value;
    a.shapes = spatial_shapes;
    a.lsi = level_start_index;
    a.loc = sampling_loc;
    a.attn = attn_weight;
    a.out = output;
    a.gka = gka;
    a.grid = grid;
    a.grid_h = (int32_t)grid_h;
    a.grid_w = (int32_t)grid_w;
    a.lds_cache_bytes = cache;
    a.fwd_ahead = tuning().fwd_ahead;
    a.fwd_cu_flip = forward_cu_flip(dtype);
    const hipError_t e = cu ? mxd::launch_forward_cu(dtype, a, static_cast<hipStream_t>(hip_stream))
                            : mxd::launch_forward(dtype, a, static_cast<hipStream_t>(hip_stream));
    if (e != hipSuccess) return fail(MXD_E_LAUNCH, "%s: launch failed: %s", who, hipGetErrorString(e));
    return MXD_OK;
}

int mxd_msda_forward(const void* value, const int32_t* spatial_shapes, const int32_t* level_start_index,
                     const void* sampling_loc, const void* attn_weight, void* output, int dtype, int64_t bs, int64_t nk,
                     int64_t nh, int64_t hd, int64_t nl, int64_t nl_attn, int64_t nq, int64_t np, void* hip_stream)
{
    return forward_common(0, value, spatial_shapes, level_start_index, sampling_loc, attn_weight, output, dtype, bs, nk,
                          nh, hd, nl, nl_attn, nq, np, hip_stream);
}

int mxd_gka_forward(const void* value, const int32_t* spatial_shapes, const int32_t* level_start_index,
                    const void* sampling_locations, const void* attn_weights, void* output, int dtype, int64_t bs,
                    int64_t nk, int64_t nh, int64_t hd, int64_t nl, int64_t nq, int64_t np, void* hip_stream)
{
    int code = dtype;
    const int meta64 = take_meta_flag(&code);
    const Dims d{bs, nk, nh, hd, nl, nl, nq, np};
    mxd::GkaArgs a;
    if (check_dims(code, d) != MXD_OK || !gka_plan(code, d, false, &a))
        return forward_common(1, value, spatial_shapes, level_start_index, sampling_locations, attn_weights, output, dtype,
                              bs, nk, nh, hd, nl, nl, nq, np, hip_stream);
    if (!value || !spatial_shapes || !level_start_index || !sampling_locations || !attn_weights || !output)
        return fail(MXD_E_NULL, "mxd_gka_forward: NULL data pointer");
    const int rc = ensure_device_ready();
    if (rc != MXD_OK) return rc;
    a.meta_i64 = meta64;
    a.value = value;
    a.shapes = spatial_shapes;
    a.lsi = level_start_index;
    a.loc = static_cast<const float*>(sampling_locations);
    a.attn = attn_weights;
    a.out = output;
    const hipError_t e = mxd::launch_gka_forward(code, a, static_cast<hipStream_t>(hip_stream));
    if (e != hipSuccess) return fail(MXD_E_LAUNCH, "mxd_gka_forward: launch failed: %s", hipGetErrorString(e));
    return MXD_OK;
}

static int grid_mode(int interpolation_mode, int padding_mode, int align_corners)
{
    if (interpolation_mode != 0) return fail(MXD_E_SHAPE, "grid_sampler2d: only bilinear interpolation (0) is built, got %d", interpolation_mode);
    if (padding_mode != 0 && padding_mode != 1)
        return fail(MXD_E_SHAPE, "grid_sampler2d: padding_mode must be 0 (zeros) or 1 (border), got %d", padding_mode);
    return 1 + padding_mode + (align_corners ? 2 : 0);
}

int mxd_grid_sampler2d_forward(const void* input_nhwc, const void* grid, void* output_nhwc, int dtype, int64_t n,
                               int64_t c, int64_t h_in, int64_t w_in, int64_t h_out, int64_t w_out,
                               int interpolation_mode, int padding_mode, int align_corners, void* hip_stream)
{
    const int mode = grid_mode(interpolation_mode, padding_mode, align_corners);
    if (mode < 0) return mode;
    if (h_in <= 0 || w_in <= 0 || h_in * w_in >= (int64_t(1) << 31))
        return fail(MXD_E_SHAPE, "grid_sampler2d: input of %lld x %lld pixels is beyond what this build indexes", (long long)h_in, (long long)w_in);
    return forward_common(1 + mode, input_nhwc, nullptr, nullptr, grid, nullptr, output_nhwc, dtype, n, h_in * w_in, 1, c, 1,
                          1, h_out * w_out, 1, hip_stream, h_in, w_in);
}

int mxd_msda_fused_forward(const void* value, const int32_t* spatial_shapes, const int32_t* level_start_index,
                           const void* reference_points, int ref_dim, const void* sampling_offsets,
                           const void* attn_logits, void* output, int dtype, int64_t bs, int64_t nk, int64_t nh,
                           int64_t hd, int64_t nl, int64_t nq, int64_t np, void* hip_stream)
{
    const int meta64 = take_meta_flag(&dtype);
    const Dims d{bs, nk, nh, hd, nl, nl, nq, np};
    int rc = check_dims(dtype, d);
    if (rc != MXD_OK) return rc;
    if (!value || !spatial_shapes || !level_start_index || !reference_points || !sampling_offsets || !attn_logits || !output)
        return fail(MXD_E_NULL, "mxd_msda_fused_forward: NULL data pointer");
    if (ref_dim != 2 && ref_dim != 4)
        return fail(MXD_E_SHAPE, "Last dim of reference_points must be 2 or 4, but get %d instead.", ref_dim);
    int align = ptr_align(value);
    if (ptr_align(output) < align) align = ptr_align(output);
    mxd::KArgs a;
    memset(&a, 0, sizeof(a));
    rc = ensure_device_ready();
    if (rc != MXD_OK) return rc;
    // The one-workgroup-per-CU form takes reference points (x, y) and units of one chunk (the softmax is formed by the
    // unit's lanes from the logits they hold); it reads offset pairs and reference points with one load each.
    int cache = 0, cu = ref_dim == 2 && nl * np <= mxd::kChunk && ptr_align(sampling_offsets) >= 2 * elem_size(dtype) &&
                        ptr_align(reference_points) >= 2 * elem_size(dtype);
    if (cu) {
        cache = 1;
        cu = 2;
        rc = make_plan(0, dtype, d, align, &a.plan, &cache, &cu);
        if (rc != MXD_OK) return rc;
    }
    if (!cu) {
        cache = 0;
        rc = make_plan(0, dtype, d, align, &a.plan);
        if (rc != MXD_OK) return rc;
    }
    fill_args(&a, dtype, d);
    a.meta_i64 = meta64;
    a.value = value;
    a.shapes = spatial_shapes;
    a.lsi = level_start_index;
    a.loc = sampling_offsets;
    a.attn = attn_logits;
    a.ref = reference_points;
    a.ref_dim = ref_dim;
    a.out = output;
    a.lds_cache_bytes = cache;
    a.fwd_cu_flip = forward_cu_flip(dtype);
    const hipError_t e = cu ? mxd::launch_forward_cu(dtype, a, static_cast<hipStream_t>(hip_stream))
                            : mxd::launch_forward(dtype, a, static_cast<hipStream_t>(hip_stream));
    if (e != hipSuccess) return fail(MXD_E_LAUNCH, "mxd_msda_fused_forward: launch failed: %s", hipGetErrorString(e));
    return MXD_OK;
}

size_t mxd_msda_backward_workspace_bytes(int dtype, int64_t bs, int64_t nk, int64_t nh, int64_t hd, int64_t nl,
                                         int64_t nl_attn, int64_t nq, int64_t np)
{
    take_meta_flag(&dtype);
    const Dims d{bs, nk, nh, hd, nl, nl_attn, nq, np};
    if (check_dims(dtype, d) != MXD_OK) return 0;
    return bwd_layout(dtype, d).total;
}

// What the fused form adds to a backward call.
struct FusedBackward {
    const void* ref;
    int ref_dim;
    const void* out;   // forward result
    void* grad_ref;    // may be nullptr
};

static size_t fused_part_bytes(const Dims& d, int ref_dim)
{
    return (((size_t)d.nh * d.bs * d.nq * d.nl * ref_dim * sizeof(float)) + 15) & ~(size_t)15;
}

static int backward_common(int kind, const void* value, const int32_t* spatial_shapes, const int32_t* level_start_index,
                           const void* sampling_loc, const void* attn_weight, const void* grad_output, void* grad_value,
                           void* grad_loc, void* grad_attn, void* workspace, size_t workspace_bytes, int dtype,
                           int64_t bs, int64_t nk, int64_t nh, int64_t hd, int64_t nl, int64_t nl_attn, int64_t nq,
                           int64_t np, int flags, void* hip_stream, int64_t grid_h = 0, int64_t grid_w = 0,
                           const FusedBackward* fused = nullptr)
{
    const int meta64 = take_meta_flag(&dtype);
    const int gka = kind == 1, grid = kind >= 2 ? kind - 1 : 0;
    const Dims d{bs, nk, nh, hd, nl, nl_attn, nq, np, fused ? 2 : gka};
    const char* who = fused  ? "mxd_msda_fused_backward"
                      : grid ? "mxd_grid_sampler2d_backward"
                      : gka  ? "mxd_gka_backward"
                             : "mxd_msda_backward";
    int rc = check_dims(dtype, d);
    if (rc != MXD_OK) return rc;
    if (!value || !sampling_loc || !grad_output || !grad_value || (!grad_loc && !gka) || (!grad_attn && !grid) ||
        (!grid && (!spatial_shapes || !level_start_index || !attn_weight)))
        return fail(MXD_E_NULL, "%s: NULL data pointer", who);
    if (fused && (!fused->ref || !fused->out)) return fail(MXD_E_NULL, "%s: NULL data pointer", who);
    if (fused && fused->ref_dim != 2 && fused->ref_dim != 4)
        return fail(MXD_E_SHAPE, "Last dim of reference_points must be 2 or 4, but get %d instead.", fused->ref_dim);
    int align = ptr_align(value);
    if (ptr_align(grad_output) < align) align = ptr_align(grad_output);
    mxd::KArgs a;
    memset(&a, 0, sizeof(a));
    rc = make_plan(1, dtype, d, align, &a.plan);
    if (rc != MXD_OK) return rc;
    const BwdLayout L = bwd_layout(dtype, d);  // (as make_plan laid the first kernel's LDS out)
    const size_t part_bytes = (fused && fused->grad_ref) ? fused_part_bytes(d, fused->ref_dim) : 0;
    const size_t need = L.total + part_bytes;
    if (need > 0 && (!workspace || workspace_bytes < need))
        return fail(MXD_E_WORKSPACE, "%s: workspace of %zu bytes required, %zu given", who, need,
                    workspace ? workspace_bytes : (size_t)0);
    if (need > 0 && (reinterpret_cast<uintptr_t>(workspace) & 15u))
        return fail(MXD_E_WORKSPACE, "%s: workspace must be 16-byte aligned", who);
    const bool half = elem_size(dtype) == 2;
    if ((flags & MXD_BWD_ACCUMULATE) && half)
        return fail(MXD_E_DTYPE, "%s: MXD_BWD_ACCUMULATE is only available for float32", who);
    char* ws = static_cast<char*>(workspace);
    float* image = half ? reinterpret_cast<float*>(ws + L.tbl_bytes + L.rec_bytes) : static_cast<float*>(grad_value);
    if (reinterpret_cast<uintptr_t>(image) & 3u) return fail(MXD_E_SHAPE, "%s: grad_value is not 4-byte aligned", who);
    fill_args(&a, dtype, d);
    a.tile_px_log2 = L.tile_px_log2;
    a.unit_split_log2 = unit_split_log2(a.plan);
    a.rec_lds_bytes = plan_record_buffer(&a.plan, L, d, dtype, !gka && !grid, a.unit_split_log2);
    a.bwd_fixed = (tuning().bwd_fixed != 0 && (!fused || a.unit_split_log2 == 0) && !gka && !grid && L.tiles && a.plan.lanes_per_row == 8 &&
                   a.plan.units_per_wave == 8 && a.plan.npass == 1 && a.plan.iters == 1 && a.unit_split_log2 <= 1 &&
                   d.nl * d.np <= ((int64_t)mxd::kChunk << a.unit_split_log2) && a.rec_lds_bytes == 0 &&
                   d.nh * d.nl_attn * d.np < (int64_t(1) << 24))  // (32-bit offsets of a wavefront's samples)
                      ? 1 + a.unit_split_log2 : 0;
    if (tuning().bwd_fixed != 0 && !fused && !gka && !grid && L.tiles && a.plan.lanes_per_row == 16 && a.plan.units_per_wave == 4 &&
        a.plan.npass == 1 && a.plan.vec * (int)elem_size(dtype) == 16 && a.unit_split_log2 == 0)
        a.bwd_fixed = 3;
    a.meta_i64 = meta64;
    a.value = value;
    a.shapes = spatial_shapes;
    a.lsi = level_start_index;
    a.loc = sampling_loc;
    a.attn = attn_weight;
    a.grad_out = grad_output;
    a.grad_value = image;
    a.tbl = reinterpret_cast<uint32_t*>(ws);
    a.rec = reinterpret_cast<uint32_t*>(ws + L.tbl_bytes);
    a.nwg = (int32_t)L.nwg;
    a.run_step = run_step(L.nwg);
    a.rec_cap = (int32_t)L.rec_cap;
    a.tbl_stride = (int32_t)L.tbl_stride;
    a.grad_loc = grad_loc;
    a.grad_attn = grad_attn;
    a.gka = gka;
    a.grid = grid;
    a.grid_h = (int32_t)grid_h;
    a.grid_w = (int32_t)grid_w;
    float* part = nullptr;
    if (fused) {
        a.ref = fused->ref;
        a.ref_dim = fused->ref_dim;
        a.out = const_cast<void*>(fused->out);
        a.np_pow2 = (np & (np - 1)) == 0 && np <= 16;
        if (part_bytes > 0) part = reinterpret_cast<float*>(ws + L.total);
        a.grad_ref = part;
    }
    hipStream_t stream = static_cast<hipStream_t>(hip_stream);
    const size_t n = (size_t)bs * nk * nh * hd;
    // every step that can fail for the sizes given comes before the first launch
    // (MXD_BWD_ANY_LAYOUT: the one-kernel form with global atomics, which takes level_start_index as it comes)
    const bool atomic_mode = !L.tiles || (flags & MXD_BWD_ANY_LAYOUT) != 0;
    mxd::TileArgs t;
    if (!atomic_mode) {
        rc = make_tile_args(d, L, (flags & MXD_BWD_ACCUMULATE) ? 1 : 0, &t, !fused && !gka && !grid);
        if (rc != MXD_OK) return rc;
        plan_image(&a, &t, half, (flags & MXD_BWD_ACCUMULATE) != 0, image, grad_value, hd);
    }
    hipError_t e = hipSuccess;
    // zero-fill of the image: by the first kernel's workgroups when the tile pass is the first to touch it and it
    // can be written in 16-byte pieces, by a kernel of its own otherwise
    const bool fill_inside = !atomic_mode && n % 4 == 0 && (reinterpret_cast<uintptr_t>(image) & 15u) == 0 &&
                             tuning().bwd_fill_kernel == 0;
    if (!(flags & MXD_BWD_ACCUMULATE)) {
        if (fill_inside) a.fill_n4 = n / 4;
        else e = mxd::launch_fill_zero(image, n, stream);
    }
    // (a level whose points lie in two chunks is added up in memory: not where a query is one chunk)
    if (e == hipSuccess && part && !a.np_pow2 && nl * np > mxd::kChunk) e = mxd::launch_fill_zero(part, part_bytes / sizeof(float), stream);
    if (e != hipSuccess) return fail(MXD_E_LAUNCH, "%s: zero-fill launch failed: %s", who, hipGetErrorString(e));
    e = mxd::launch_backward(dtype, a, atomic_mode, stream);
    if (e != hipSuccess) return fail(MXD_E_LAUNCH, "%s: launch failed: %s", who, hipGetErrorString(e));
    if (!atomic_mode) {
        e = mxd::launch_gradv_tiles(dtype, a, t, stream);
        if (e != hipSuccess) return fail(MXD_E_LAUNCH, "%s: tile kernel launch failed: %s", who, hipGetErrorString(e));
    }
    if (half) {
        e = a.sparse ? mxd::launch_round_rows(dtype, a, stream) : mxd::launch_round(dtype, image, grad_value, n, stream);
        if (e != hipSuccess) return fail(MXD_E_LAUNCH, "%s: rounding launch failed: %s", who, hipGetErrorString(e));
    }
    if (part) {
        e = mxd::launch_sum_heads(dtype, part, fused->grad_ref, (size_t)bs * nq * nl * fused->ref_dim, (int)nh, stream);
        if (e != hipSuccess) return fail(MXD_E_LAUNCH, "%s: head sum launch failed: %s", who, hipGetErrorString(e));
    }
    return MXD_OK;
}

size_t mxd_msda_fused_backward_workspace_bytes(int dtype, int64_t bs, int64_t nk, int64_t nh, int64_t hd,
                                               int64_t nl, int64_t nq, int64_t np, int ref_dim, int want_grad_ref)
{
    take_meta_flag(&dtype);
    const Dims d{bs, nk, nh, hd, nl, nl, nq, np, 2};
    if (check_dims(dtype, d) != MXD_OK || (ref_dim != 2 && ref_dim != 4)) return 0;
    return bwd_layout(dtype, d).total + (want_grad_ref ? fused_part_bytes(d, ref_dim) : 0);
}

int mxd_msda_fused_backward(const void* value, const int32_t* spatial_shapes, const int32_t* level_start_index,
                            const void* reference_points, int ref_dim, const void* sampling_offsets,
                            const void* attn_logits, const void* output, const void* grad_output, void* grad_value,
                            void* grad_reference_points, void* grad_sampling_offsets, void* grad_attn_logits,
                            void* workspace, size_t workspace_bytes, int dtype, int64_t bs, int64_t nk, int64_t nh,
                            int64_t hd, int64_t nl, int64_t nq, int64_t np, int flags, void* hip_stream)
{
    const FusedBackward f{reference_points, ref_dim, output, grad_reference_points};
    return backward_common(0, value, spatial_shapes, level_start_index, sampling_offsets, attn_logits, grad_output,
                           grad_value, grad_sampling_offsets, grad_attn_logits, workspace, workspace_bytes, dtype, bs,
                           nk, nh, hd, nl, nl, nq, np, flags, hip_stream, 0, 0, &f);
}

int mxd_msda_backward(const void* value, const int32_t* spatial_shapes, const int32_t* level_start_index,
                      const void* sampling_loc, const void* attn_weight, const void* grad_output, void* grad_value,
                      void* grad_loc, void* grad_attn, void* workspace, size_t workspace_bytes, int dtype, int64_t bs,
                      int64_t nk, int64_t nh, int64_t hd, int64_t nl, int64_t nl_attn, int64_t nq, int64_t np,
                      int flags, void* hip_stream)
{
    return backward_common(0, value, spatial_shapes, level_start_index, sampling_loc, attn_weight, grad_output,
                           grad_value, grad_loc, grad_attn, workspace, workspace_bytes, dtype, bs, nk, nh, hd, nl,
                           nl_attn, nq, np, flags, hip_stream);
}

size_t mxd_msda_backward_static_limit(void) { return kStaticScratchBytes; }

int mxd_msda_backward_static(const void* value, const int32_t* spatial_shapes, const int32_t* level_start_index,
                             const void* sampling_loc, const void* attn_weight, const void* grad_output,
                             void* grad_value, void* grad_loc, void* grad_attn, int dtype, int64_t bs, int64_t nk,
                             int64_t nh, int64_t hd, int64_t nl, int64_t nl_attn, int64_t nq, int64_t np, int flags,
                             void* hip_stream)
{
    // (allocates nothing: the scratch is the library's own static device array; sizes beyond it are refused)
    const size_t need = mxd_msda_backward_workspace_bytes(dtype, bs, nk, nh, hd, nl, nl_attn, nq, np);
    if (need > kStaticScratchBytes)
        return fail(MXD_E_WORKSPACE,
                    "mxd_msda_backward_static: this problem needs %zu bytes of scratch, the static array holds %zu; "
                    "use mxd_msda_backward with a workspace",
                    need, kStaticScratchBytes);
    int rc = ensure_device_ready();
    if (rc != MXD_OK) return rc;
    void* ws = device_scratch();
    if (!ws) return fail(MXD_E_LAUNCH, "mxd_msda_backward_static: the static scratch array is not set up on this device");
    return backward_common(0, value, spatial_shapes, level_start_index, sampling_loc, attn_weight, grad_output,
                           grad_value, grad_loc, grad_attn, ws, kStaticScratchBytes, dtype, bs, nk, nh, hd, nl, nl_attn,
                           nq, np, flags, hip_stream);
}

size_t mxd_gka_backward_workspace_bytes(int dtype, int64_t bs, int64_t nk, int64_t nh, int64_t hd, int64_t nl,
                                        int64_t nq, int64_t np)
{
    take_meta_flag(&dtype);
    const Dims d{bs, nk, nh, hd, nl, nl, nq, np, 1};
    if (check_dims(dtype, d) != MXD_OK) return 0;
    mxd::GkaArgs a;
    return gka_plan(dtype, d, true, &a) ? gka_part_bytes(a) : bwd_layout(dtype, d).total;
}

int mxd_gka_backward(const void* value, const int32_t* spatial_shapes, const int32_t* level_start_index,
                     const void* sampling_locations, const void* attn_weights, const void* grad_output,
                     void* grad_value, void* grad_attn_weights, void* workspace, size_t workspace_bytes, int dtype,
                     int64_t bs, int64_t nk, int64_t nh, int64_t hd, int64_t nl, int64_t nq, int64_t np,
                     void* hip_stream)
{
    int code = dtype;
    const int meta64 = take_meta_flag(&code);
    const Dims d{bs, nk, nh, hd, nl, nl, nq, np};
    mxd::GkaArgs a;
    if (check_dims(code, d) != MXD_OK || !gka_plan(code, d, true, &a))
        return backward_common(1, value, spatial_shapes, level_start_index, sampling_locations, attn_weights, grad_output,
                               grad_value, nullptr, grad_attn_weights, workspace, workspace_bytes, dtype, bs, nk, nh, hd, nl,
                               nl, nq, np, 0, hip_stream);
    if (!value || !spatial_shapes || !level_start_index || !sampling_locations || !attn_weights || !grad_output || !grad_value ||
        !grad_attn_weights)
        return fail(MXD_E_NULL, "mxd_gka_backward: NULL data pointer");
    const size_t need = gka_part_bytes(a);
    if (!workspace || workspace_bytes < need)
        return fail(MXD_E_WORKSPACE, "mxd_gka_backward: workspace of %zu bytes required, %zu given", need,
                    workspace ? workspace_bytes : (size_t)0);
    if (reinterpret_cast<uintptr_t>(workspace) & 15u) return fail(MXD_E_WORKSPACE, "mxd_gka_backward: workspace must be 16-byte aligned");
    const int rc = ensure_device_ready();
    if (rc != MXD_OK) return rc;
    a.meta_i64 = meta64;
    a.value = value;
    a.shapes = spatial_shapes;
    a.lsi = level_start_index;
    a.loc = static_cast<const float*>(sampling_locations);
    a.attn = attn_weights;
    a.grad_out = grad_output;
    a.grad_value = grad_value;
    a.grad_attn = grad_attn_weights;
    a.part = static_cast<float*>(workspace);
    a.dots = reinterpret_cast<float*>(static_cast<char*>(workspace) + gka_image_bytes(a));
    a.sc_direct = (reinterpret_cast<uintptr_t>(grad_output) & 15u) == 0;
    const hipError_t e = mxd::launch_gka_backward(code, a, static_cast<hipStream_t>(hip_stream));
    if (e != hipSuccess) return fail(MXD_E_LAUNCH, "mxd_gka_backward: launch failed: %s", hipGetErrorString(e));
    return MXD_OK;
}

size_t mxd_grid_sampler2d_backward_workspace_bytes(int dtype, int64_t n, int64_t c, int64_t h_in, int64_t w_in,
                                                   int64_t h_out, int64_t w_out)
{
    if (h_in <= 0 || w_in <= 0 || h_in * w_in >= (int64_t(1) << 31)) return 0;
    return mxd_msda_backward_workspace_bytes(dtype, n, h_in * w_in, 1, c, 1, 1, h_out * w_out, 1);
}

int mxd_grid_sampler2d_backward(const void* grad_output_nhwc, const void* input_nhwc, const void* grid,
                                void* grad_input_nhwc, void* grad_grid, void* workspace, size_t workspace_bytes,
                                int dtype, int64_t n, int64_t c, int64_t h_in, int64_t w_in, int64_t h_out,
                                int64_t w_out, int interpolation_mode, int padding_mode, int align_corners,
                                void* hip_stream)
{
    const int mode = grid_mode(interpolation_mode, padding_mode, align_corners);
    if (mode < 0) return mode;
    if (h_in <= 0 || w_in <= 0 || h_in * w_in >= (int64_t(1) << 31))
        return fail(MXD_E_SHAPE, "grid_sampler2d: input of %lld x %lld pixels is beyond what this build indexes", (long long)h_in, (long long)w_in);
    return backward_common(1 + mode, input_nhwc, nullptr, nullptr, grid, nullptr, grad_output_nhwc, grad_input_nhwc,
                           grad_grid, nullptr, workspace, workspace_bytes, dtype, n, h_in * w_in, 1, c, 1, 1,
                           h_out * w_out, 1, 0, hip_stream, h_in, w_in);
}

int mxd_dagg_forward(const void* mc_ms_feat, const int32_t* spatial_shape, const int32_t* scale_start_index,
                     const void* sampling_location, const void* weights, void* output, int dtype, int64_t bs,
                     int64_t num_feat, int64_t num_embeds, int64_t num_cams, int64_t num_scale, int64_t num_anchors,
                     int64_t num_pts, int64_t num_groups, void* hip_stream)
{
    const int meta64 = take_meta_flag(&dtype);
    mxd::DaggArgs a;
    int rc = dagg_args(dtype, bs, num_feat, num_embeds, num_cams, num_scale, num_anchors, num_pts, num_groups, &a);
    if (rc == MXD_OK && (!mc_ms_feat || !spatial_shape || !scale_start_index || !sampling_location || !weights || !output))
        rc = fail(MXD_E_NULL, "mxd_dagg_forward: NULL data pointer");
    if (rc == MXD_OK) rc = dagg_plan(&a, elem_size(dtype), false);
    if (rc != MXD_OK) return rc;
    a.meta_i64 = meta64;
    a.feat = mc_ms_feat;
    a.shapes = spatial_shape;
    a.lsi = scale_start_index;
    a.loc = sampling_location;
    a.w = weights;
    a.out = output;
    const hipError_t e = mxd::launch_dagg_forward(dtype, a, static_cast<hipStream_t>(hip_stream));
    if (e != hipSuccess) return fail(MXD_E_LAUNCH, "mxd_dagg_forward: launch failed: %s", hipGetErrorString(e));
    return MXD_OK;
}

size_t mxd_dagg_backward_workspace_bytes(int dtype, int64_t bs, int64_t num_feat, int64_t num_embeds, int64_t num_cams,
                                         int64_t num_scale, int64_t num_anchors, int64_t num_pts, int64_t num_groups)
{
    take_meta_flag(&dtype);
    mxd::DaggArgs a;
    if (dagg_args(dtype, bs, num_feat, num_embeds, num_cams, num_scale, num_anchors, num_pts, num_groups, &a) != MXD_OK) return 0;
    return DaggSpace(a, elem_size(dtype)).total;
}

int mxd_dagg_backward(const void* mc_ms_feat, const int32_t* spatial_shape, const int32_t* scale_start_index,
                      const void* sampling_location, const void* weights, const void* grad_output,
                      void* grad_mc_ms_feat, void* grad_sampling_location, void* grad_weights, void* workspace,
                      size_t workspace_bytes, int dtype, int64_t bs, int64_t num_feat, int64_t num_embeds,
                      int64_t num_cams, int64_t num_scale, int64_t num_anchors, int64_t num_pts, int64_t num_groups,
                      void* hip_stream)
{
    const int meta64 = take_meta_flag(&dtype);
    mxd::DaggArgs a;
    int rc = dagg_args(dtype, bs, num_feat, num_embeds, num_cams, num_scale, num_anchors, num_pts, num_groups, &a);
    if (rc != MXD_OK) return rc;
    if (!mc_ms_feat || !spatial_shape || !scale_start_index || !sampling_location || !weights || !grad_output ||
        !grad_mc_ms_feat || !grad_sampling_location || !grad_weights)
        return fail(MXD_E_NULL, "mxd_dagg_backward: NULL data pointer");
    const int es = elem_size(dtype);
    rc = dagg_plan(&a, es, true);
    if (rc != MXD_OK) return rc;
    const DaggSpace space(a, es);
    if (!workspace || workspace_bytes < space.total)
        return fail(MXD_E_WORKSPACE, "mxd_dagg_backward: workspace of %zu bytes required, %zu given", space.total,
                    workspace ? workspace_bytes : (size_t)0);
    if (reinterpret_cast<uintptr_t>(workspace) & 15u)
        return fail(MXD_E_WORKSPACE, "mxd_dagg_backward: workspace must be 16-byte aligned");
    char* ws = static_cast<char*>(workspace);
    a.meta_i64 = meta64;
    a.feat = mc_ms_feat;
    a.shapes = spatial_shape;
    a.lsi = scale_start_index;
    a.loc = sampling_location;
    a.w = weights;
    a.grad_out = grad_output;
    a.grad_feat = grad_mc_ms_feat;
    a.grad_loc = grad_sampling_location;
    a.grad_w = grad_weights;
    a.image = es == 2 ? reinterpret_cast<float*>(ws + space.image) : static_cast<float*>(grad_mc_ms_feat);
    if (reinterpret_cast<uintptr_t>(a.image) & 3u) return fail(MXD_E_SHAPE, "mxd_dagg_backward: grad_mc_ms_feat is not 4-byte aligned");
    a.gw_part = reinterpret_cast<float*>(ws);
    a.gl_part = reinterpret_cast<float*>(ws + space.gl);
    // (the value rows are copied to LDS 16 bytes a lane)
    if (dagg_dots_with_rows(a, es) && (reinterpret_cast<uintptr_t>(mc_ms_feat) & 15u) == 0) a.dots = reinterpret_cast<mxd::f32x2*>(ws);
    a.csr = reinterpret_cast<uint32_t*>(ws + space.csr);
    a.rec = reinterpret_cast<mxd::u32x4*>(ws + space.rec);
    const hipError_t e = mxd::launch_dagg_backward(dtype, a, static_cast<hipStream_t>(hip_stream));
    if (e != hipSuccess) return fail(MXD_E_LAUNCH, "mxd_dagg_backward: launch failed: %s", hipGetErrorString(e));
    return MXD_OK;
}

int mxd_grid_sampler2d_planes_fit(int64_t n, int64_t c, int64_t h_in, int64_t w_in, int64_t h_out, int64_t w_out)
{
    return grid_planes_fit(n, c, h_in, w_in, h_out, w_out) ? 1 : 0;
}

int mxd_grid_sampler2d_planes_forward(const void* input, const void* grid, void* output, int dtype, int64_t n, int64_t c,
                                      int64_t h_in, int64_t w_in, int64_t h_out, int64_t w_out, int interpolation_mode,
                                      int padding_mode, int align_corners, void* hip_stream)
{
    const int mode = grid_mode(interpolation_mode, padding_mode, align_corners);
    if (mode < 0) return mode;
    mxd::GridArgs a;
    int rc = grid_planes_args(dtype, n, c, h_in, w_in, h_out, w_out, mode, &a);
    if (rc == MXD_OK && (!input || !grid || !output)) rc = fail(MXD_E_NULL, "mxd_grid_sampler2d_planes_forward: NULL data pointer");
    if (rc == MXD_OK) rc = grid_planes_forward_plan(elem_size(dtype), &a);
    if (rc == MXD_OK) rc = ensure_device_ready();
    if (rc != MXD_OK) return rc;
    a.x = input;
    a.grid = grid;
    a.out = output;
    const hipError_t e = mxd::launch_grid_planes_forward(dtype, a, static_cast<hipStream_t>(hip_stream));
    if (e != hipSuccess) return fail(MXD_E_LAUNCH, "mxd_grid_sampler2d_planes_forward: launch failed: %s", hipGetErrorString(e));
    return MXD_OK;
}

size_t mxd_grid_sampler2d_planes_backward_workspace_bytes(int dtype, int64_t n, int64_t c, int64_t h_in, int64_t w_in,
                                                          int64_t h_out, int64_t w_out)
{
    mxd::GridArgs a;
    if (grid_planes_args(dtype, n, c, h_in, w_in, h_out, w_out, 1, &a) != MXD_OK) return 0;
    if (grid_planes_backward_plan(elem_size(dtype), true, true, &a) != MXD_OK) return 0;
    return grid_part_bytes(a);
}

int mxd_grid_sampler2d_planes_backward(const void* grad_output, const void* input, const void* grid, void* grad_input,
                                       void* grad_grid, void* workspace, size_t workspace_bytes, int dtype, int64_t n,
                                       int64_t c, int64_t h_in, int64_t w_in, int64_t h_out, int64_t w_out,
                                       int interpolation_mode, int padding_mode, int align_corners, void* hip_stream)
{
    const int mode = grid_mode(interpolation_mode, padding_mode, align_corners);
    if (mode < 0) return mode;
    mxd::GridArgs a;
    int rc = grid_planes_args(dtype, n, c, h_in, w_in, h_out, w_out, mode, &a);
    if (rc == MXD_OK && (!grad_output || !input || !grid || (!grad_input && !grad_grid)))
        rc = fail(MXD_E_NULL, "mxd_grid_sampler2d_planes_backward: NULL data pointer");
    if (rc == MXD_OK) rc = grid_planes_backward_plan(elem_size(dtype), grad_input != nullptr, grad_grid != nullptr, &a);
    if (rc == MXD_OK) rc = ensure_device_ready();
    if (rc != MXD_OK) return rc;
    const size_t need = grad_grid ? grid_part_bytes(a) : 0;
    if (need > 0 && (!workspace || workspace_bytes < need))
        return fail(MXD_E_WORKSPACE, "mxd_grid_sampler2d_planes_backward: workspace of %zu bytes required, %zu given", need,
                    workspace ? workspace_bytes : (size_t)0);
    if (need > 0 && (reinterpret_cast<uintptr_t>(workspace) & 15u))
        return fail(MXD_E_WORKSPACE, "mxd_grid_sampler2d_planes_backward: workspace must be 16-byte aligned");
    a.x = input;
    a.grid = grid;
    a.grad_out = grad_output;
    a.grad_x = grad_input;
    a.grad_grid = grad_grid;
    a.part = static_cast<float*>(workspace);
    const hipError_t e = mxd::launch_grid_planes_backward(dtype, a, static_cast<hipStream_t>(hip_stream));
    if (e != hipSuccess) return fail(MXD_E_LAUNCH, "mxd_grid_sampler2d_planes_backward: launch failed: %s", hipGetErrorString(e));
    return MXD_OK;
}

}  // extern "C"
