// Geometric kernel attention on small maps for gfx950 (MI355X), wave64: forward and backward.
//
//   out[b,q,h,:] = sum over samples s of w[b,q,h,s] * value[b, pixel(b,q,h,s), h, :]        (one pixel per sample, clamped)
//
// (reference: mx_driving/ops/geometric_kernel_attention.py:29-57.)  The maps of this operator are small -- 15 x 25 pixels of 64
// channels, 96 KB per (batch, head) in float32 -- and every pixel is sampled hundreds of times, 2.6 GB of rows per pass at
// [24, 7156 queries, 4 heads, 15 points].  From L1 and L2 they come at 18 TB/s (the general kernels: forward 147 us, dots of the
// backward 279 us with their records); LDS gives 128 bytes per clock and CU, 78 TB/s.  So
//
//   * forward and the dots of the backward (gradient of the weights) put the (batch, head)'s slab of value into LDS once per
//     workgroup and gather there.  What bounds them: reading locations and weights and writing the result (300 MB), and LDS.
//   * grad_value is summed by pixel: a workgroup takes tiles of queries, puts their grad_out rows into LDS, sorts the tile's
//     samples by pixel (integer LDS counters) and lets lane groups that own pixels add the rows of their samples to registers.
//     Clamping piles samples on the border pixels (16 times the average on the corners): pixels are dealt to the groups in turn.
//     The query ranges of a slab leave float32 images of it, which a last kernel adds up and rounds.
//     What bounds it: LDS again, and half of what it reads there is for groups whose lists have ended (a tile of 192 queries has 7
//     samples per pixel).  Smaller tiles lose (64 queries: 356 against 286 us for the backward), so do larger ones that a CU holds one
//     workgroup of (307), and so does sharing long lists among the groups of a wavefront (327).
//
// Measured at that size, float32: forward 147 -> 82 us, dots 279 -> 112, grad_value 370 -> 183 + 9; float16 forward and backward
// 65 and 220 us.
#include "gka.h"

namespace mxd {

namespace {

// Work items in the order of their numbers on every XCD (workgroups are dealt to the XCDs in turn): the heads of a range of
// queries, whose locations share cache lines, follow each other in one L2.
__device__ inline uint32_t xcd_order(uint32_t wg, uint32_t total)
{
    const uint32_t x = wg % kNumXcd, each = total / kNumXcd, more = total % kNumXcd;
    return x * each + (x < more ? x : more) + wg / kNumXcd;
}

__device__ inline void load_levels(const GkaArgs& a, i32x4* lvl)
{
    const int sh = a.meta_i64, l = (int)threadIdx.x;
    if (l < a.nl) lvl[l] = i32x4{a.shapes[(2 * l) << sh], a.shapes[(2 * l + 1) << sh], a.lsi[l << sh], 0};
}

__device__ inline f32x2 load_xy(const float* loc, int64_t i)
{
    typedef f32x2 mem_t __attribute__((aligned(4)));
    return *reinterpret_cast<const mem_t*>(loc + 2 * i);
}

// Pixel of sample s of a query, -1 if it has none.
__device__ inline int32_t sample_pixel(const GkaArgs& a, const i32x4* lvl, int s, f32x2 xy)
{
    const Sample sm = gka_geometry(xy.x, xy.y, lvl[((uint32_t)s * a.np_magic) >> 20], a.nk, true);
    return sm.cvalid[0] ? sm.pix[0] : -1;
}

// Forward (DOTS = false) or gradient of the weights (DOTS = true); LPR lanes of 16 bytes share a row.
template <typename T, int LPR_LOG2, bool DOTS>
__global__ __launch_bounds__(1024) void gka_slab_kernel(const GkaArgs a)
{
    constexpr int LPR = 1 << LPR_LOG2, U = kWave / LPR, VEC = 16 / (int)sizeof(T);
    constexpr int K = LPR < kChunk ? kChunk / LPR : 1;  // staged samples (and dots) per lane
    typedef RowIO<T, VEC> Row;
    struct Staged {
        uint32_t row, w;
    };
    extern __shared__ __align__(16) unsigned char smem[];
    i32x4* lvl = reinterpret_cast<i32x4*>(smem);
    const int lane = (int)threadIdx.x & (kWave - 1), wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int nw = (int)blockDim.x >> 6;
    Staged* stage = reinterpret_cast<Staged*>(smem + kGkaLevelBytes) + wave * (U * kChunkStride);
    unsigned char* slab = smem + kGkaLevelBytes + (size_t)nw * (U * kChunkStride) * sizeof(Staged);
    uint32_t wg = xcd_order(blockIdx.x, gridDim.x);
    const int h = (int)(wg % (uint32_t)a.nh);
    wg /= (uint32_t)a.nh;
    const int part = (int)(wg % (uint32_t)a.parts), ch = h * a.hd + part * a.part_ch;  // first channel of the rows
    wg /= (uint32_t)a.parts;
    const int b = (int)(wg / (uint32_t)a.splits), q_begin = (int)(wg % (uint32_t)a.splits) * a.split_q;
    const int q_end = q_begin + a.split_q < a.nq ? q_begin + a.split_q : a.nq;
    const int g = lane >> LPR_LOG2, c = lane & (LPR - 1);
    const uint32_t row_bytes = LPR * 16u, zero_row = (uint32_t)a.nk * row_bytes;

    load_levels(a, lvl);
    {
        const T* src = static_cast<const T*>(a.value) + (int64_t)b * a.nk * a.nh * a.hd + ch;
        const int64_t pitch = (int64_t)a.nh * a.hd;
        const int total = a.nk << LPR_LOG2, step = (int)blockDim.x;
        for (int i0 = (int)threadIdx.x; i0 < total; i0 += 4 * step) {
            typename Row::vec_t v[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int i = i0 + j * step;
                if (i < total) v[j] = *reinterpret_cast<const typename Row::mem_t*>(src + (i >> LPR_LOG2) * pitch + (i & (LPR - 1)) * VEC);
            }
#pragma unroll
            for (int j = 0; j < 4; ++j)
                if (i0 + j * step < total) reinterpret_cast<typename Row::vec_t*>(slab)[i0 + j * step] = v[j];
        }
        if ((int)threadIdx.x < LPR) reinterpret_cast<u32x4*>(slab + zero_row)[threadIdx.x] = u32x4{0u, 0u, 0u, 0u};
    }
    __syncthreads();

    const T* attn = static_cast<const T*>(a.attn);
    const T* gout = static_cast<const T*>(a.grad_out);
    struct Raw {
        f32x2 xy;
        T w;
    };
    auto index = [&](int q, int s) { return (((int64_t)b * a.nq + q) * a.nh + h) * a.S + s; };
    auto fetch = [&](int q0, int c0, Raw (&r)[K]) {
#pragma unroll
        for (int k = 0; k < K; ++k) {
            const int i = lane + k * kWave, q = q0 + (i >> 4), s = c0 + (i & (kChunk - 1));
            r[k].xy = f32x2{__builtin_nanf(""), 0.0f};
            r[k].w = (T)0.0f;
            if (i < U * kChunk && q < q_end && s < a.S) {
                r[k].xy = load_xy(a.loc, index(q, s));
                if constexpr (!DOTS) r[k].w = attn[index(q, s)];
            }
        }
    };
    auto fetch_row = [&](int q0) {
        const int q = q0 + g < q_end ? q0 + g : q_begin;
        return Row::load_held(gout + ((int64_t)b * a.nq + q) * a.nh * a.hd + ch + c * VEC);
    };
    // (the samples, and grad_out rows, of the next pass are on their way while this one's are gathered)
    int q0 = q_begin + wave * U;
    if (q0 >= q_end) return;  // wavefront-uniform; no workgroup barrier follows
    Raw next[K];
    fetch(q0, 0, next);
    typename Row::held_t next_row;
    if constexpr (DOTS) next_row = fetch_row(q0);
    const Staged* mine = stage + g * kChunkStride;
    for (; q0 < q_end; q0 += nw * U) {
        float acc[VEC], gv[VEC];
        uint32_t gp[VEC / 2];
        typedef T t2 __attribute__((ext_vector_type(2)));
#pragma unroll
        for (int e = 0; e < VEC; ++e) acc[e] = 0.0f;
        if constexpr (DOTS) {
            Row::unpack_held(next_row, gv);
            if constexpr (sizeof(T) == 2) {
#pragma unroll
                for (int e = 0; e < VEC / 2; ++e) gp[e] = __builtin_bit_cast(uint32_t, t2{next_row[2 * e], next_row[2 * e + 1]});
            }
            next_row = fetch_row(q0 + nw * U);
        }
        for (int c0 = 0; c0 < a.S; c0 += kChunk) {
#pragma unroll
            for (int k = 0; k < K; ++k) {
                const int i = lane + k * kWave, s = c0 + (i & (kChunk - 1));
                if (i < U * kChunk) {
                    const int32_t px = s < a.S ? sample_pixel(a, lvl, s, next[k].xy) : -1;
                    const float w = px >= 0 ? to_f32(next[k].w) : 0.0f;
                    stage[(i >> 4) * kChunkStride + (i & (kChunk - 1))] =
                        Staged{px >= 0 ? (uint32_t)px * row_bytes : zero_row, __builtin_bit_cast(uint32_t, w)};
                }
            }
            wave_lds_sync();
            if (c0 + kChunk < a.S) fetch(q0, c0 + kChunk, next);
            else fetch(q0 + nw * U, 0, next);
            const int ns = a.S - c0 < kChunk ? a.S - c0 : kChunk;
            if constexpr (!DOTS) {
#pragma unroll 4
                for (int s = 0; s < ((ns + 3) & ~3); ++s) {  // (what is staged behind the last one is the row of zeros)
                    const Staged en = mine[s];
                    float v[VEC];
                    Row::unpack(*reinterpret_cast<const typename Row::raw_t*>(slab + en.row + c * 16), v);
                    const float w = __builtin_bit_cast(float, en.w);
#pragma unroll
                    for (int e = 0; e < VEC; ++e) acc[e] = __builtin_fmaf(w, v[e], acc[e]);
                }
            } else {
                float dot[K];
#pragma unroll
                for (int s4 = 0; s4 < kChunk; s4 += 4) {
                    if (s4 >= ns) break;
                    // (four samples side by side; what is staged behind the last one is the row of zeros)
#pragma unroll
                    for (int s = s4; s < s4 + 4; ++s) {
                        const u32x4 raw = *reinterpret_cast<const u32x4*>(slab + mine[s].row + c * 16);
                        float p = 0.0f;
                        if constexpr (sizeof(T) == 2) {
#pragma unroll
                            for (int e = 0; e < VEC / 2; ++e) {
                                const uint32_t pair = raw[e];
                                p = dot2_acc<T>(pair, gp[e], p);
                            }
                        } else {
                            float v[VEC];
                            Row::unpack(raw, v);
#pragma unroll
                            for (int e = 0; e < VEC; ++e) p = __builtin_fmaf(v[e], gv[e], p);
                        }
                        p = group_sum<LPR_LOG2>(p);
                        if (c == (s & (LPR - 1))) dot[s >> LPR_LOG2 < K ? s >> LPR_LOG2 : 0] = p;
                    }
                }
                T* dst = static_cast<T*>(a.grad_attn);
                float* dots = a.dots + (int64_t)part * a.bs * a.nq * a.nh * a.S;
#pragma unroll
                for (int k = 0; k < K; ++k) {
                    const int s = c + k * LPR;
                    if (s < ns && q0 + g < q_end) {
                        const float d = mine[s].row == zero_row ? 0.0f : dot[k];
                        if (a.parts == 1) dst[index(q0 + g, c0 + s)] = from_f32<T>(d);
                        else dots[index(q0 + g, c0 + s)] = d;
                    }
                }
            }
            wave_lds_sync();
        }
        if constexpr (!DOTS) {
            if (q0 + g < q_end) Row::store_global(static_cast<T*>(a.out) + ((int64_t)b * a.nq + q0 + g) * a.nh * a.hd + ch + c * VEC, acc);
        }
    }
}

// grad_value, or one query range's part of it: PX pixels per lane group.
template <typename T, int PX>
__global__ __launch_bounds__(1024) void gka_scatter_kernel(const GkaArgs a)
{
    typedef RowIO<T, 4> Row;
    extern __shared__ __align__(16) unsigned char smem[];
    __shared__ uint32_t wave_sum[16];
    const int tid = (int)threadIdx.x, block = (int)blockDim.x, lane = tid & (kWave - 1);
    const int row_bytes = a.part_ch * (int)sizeof(T);
    i32x4* lvl = reinterpret_cast<i32x4*>(smem);
    u32x2* ent = reinterpret_cast<u32x2*>(smem + kGkaLevelBytes);                    // sorted samples: {row in `rows`, weight}
    unsigned char* rows = reinterpret_cast<unsigned char*>(ent) + (((size_t)a.sc_tile_q * a.S * 8 + 15) & ~(size_t)15);
    uint32_t* count = reinterpret_cast<uint32_t*>(rows + (size_t)a.sc_tile_q * row_bytes);  // [nk]
    uint32_t* start = count + a.nk;                                                  // [nk + 1]
    uint32_t wg = xcd_order(blockIdx.x, gridDim.x);
    const int h = (int)(wg % (uint32_t)a.nh);
    wg /= (uint32_t)a.nh;
    const int ch = h * a.hd + (int)(wg % (uint32_t)a.parts) * a.part_ch;  // first channel of the rows
    wg /= (uint32_t)a.parts;
    const int split = (int)(wg % (uint32_t)a.sc_splits), b = (int)(wg / (uint32_t)a.sc_splits);
    const int q_begin = split * a.sc_split_q, q_end = q_begin + a.sc_split_q < a.nq ? q_begin + a.sc_split_q : a.nq;
    const T* attn = static_cast<const T*>(a.attn);
    const T* gout = static_cast<const T*>(a.grad_out) + (int64_t)b * a.nq * a.nh * a.hd + ch;
    const int64_t pitch = (int64_t)a.nh * a.hd;
    load_levels(a, lvl);
    for (int i = tid; i < a.nk; i += block) count[i] = 0;
    float acc[PX][4];
#pragma unroll
    for (int i = 0; i < PX; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[i][e] = 0.0f;
    const int groups = block >> a.sc_lanes_log2, grp = tid >> a.sc_lanes_log2, j = tid & ((1 << a.sc_lanes_log2) - 1);
    constexpr int kTogether = 4;                       // rows of a pixel that are read side by side
    const int per = (a.nk + block - 1) / block;        // counters of a thread in the prefix sum
    const int piece_log2 = a.lpr_log2;                 // 16-byte pieces of a row
    __syncthreads();
    for (int q0 = q_begin; q0 < q_end; q0 += a.sc_tile_q) {
        const int nq = q0 + a.sc_tile_q < q_end ? a.sc_tile_q : q_end - q0, n = nq * a.S;
        // ---- samples of the tile: pixel, weight, place among the samples of the pixel; rows of the tile into LDS ----------
        uint32_t place[kGkaSamples];  // pixel | place << 16, ~0: none
        T w[kGkaSamples];
        int t0 = tid;
        asm volatile("" : "+v"(t0));  // (what follows from it is not to be kept across the tiles)
#pragma unroll
        for (int half = 0; half < kGkaSamples; half += 4) {
            f32x2 xy[4];
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const int i = t0 + (half + k) * block;
                if (i < n) {
                    const int q = (int)(((uint32_t)i * a.s_magic) >> 20), s = i - q * a.S;
                    const int64_t at = (((int64_t)b * a.nq + q0 + q) * a.nh + h) * a.S + s;
                    xy[k] = load_xy(a.loc, at);
                    w[half + k] = attn[at];
                }
            }
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const int i = t0 + (half + k) * block;
                place[half + k] = ~0u;
                if (i < n) {
                    const int q = (int)(((uint32_t)i * a.s_magic) >> 20), s = i - q * a.S;
                    const int32_t px = sample_pixel(a, lvl, s, xy[k]);
                    if (px >= 0) place[half + k] = (uint32_t)px | atomicAdd(&count[px], 1u) << 16;
                }
            }
        }
        typedef RowIO<T, 16 / (int)sizeof(T)> Wide;
        for (int i0 = t0; i0 < nq << piece_log2; i0 += 4 * block) {
            typename Wide::vec_t v[4];
#pragma unroll
            for (int m = 0; m < 4; ++m) {
                const int i = i0 + m * block, q = i >> piece_log2, p = i & ((1 << piece_log2) - 1);
                if (q < nq) v[m] = *reinterpret_cast<const typename Wide::mem_t*>(gout + (q0 + q) * pitch + p * (16 / (int)sizeof(T)));
            }
#pragma unroll
            for (int m = 0; m < 4; ++m)
                if ((i0 + m * block) >> piece_log2 < nq) reinterpret_cast<typename Wide::vec_t*>(rows)[i0 + m * block] = v[m];
        }
        __syncthreads();
        // ---- first sample of every pixel ------------------------------------------------------------------------------------
        uint32_t sum = 0;
        const int c0 = tid * per;
        for (int i = c0; i < c0 + per && i < a.nk; ++i) sum += count[i];
        uint32_t inc = sum;
#pragma unroll
        for (int d = 1; d < kWave; d <<= 1) {
            const uint32_t o = __shfl_up(inc, d, kWave);
            if (lane >= d) inc += o;
        }
        if (lane == kWave - 1) wave_sum[tid >> 6] = inc;
        __syncthreads();
        uint32_t at = inc - sum;
        for (int v = 0; v < tid >> 6; ++v) at += wave_sum[v];
        for (int i = c0; i < c0 + per && i < a.nk; ++i) {
            start[i] = at;
            at += count[i];
            count[i] = 0;
            if (i == a.nk - 1) start[a.nk] = at;
        }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < kGkaSamples; ++k) {
            if (place[k] != ~0u) {
                const uint32_t q = ((uint32_t)(t0 + k * block) * a.s_magic) >> 20;
                ent[start[place[k] & 0xFFFFu] + (place[k] >> 16)] = u32x2{q * (uint32_t)row_bytes, __builtin_bit_cast(uint32_t, to_f32(w[k]))};
            }
        }
        __syncthreads();
        // ---- the groups add the rows of their pixels' samples ---------------------------------------------------------------
        int g0 = grp;
#pragma unroll
        for (int i = 0; i < PX; ++i) {
            asm volatile("" : "+v"(g0));
            const int p = i * groups + g0;
            uint32_t k = 0, end = 0;
            if (p < a.nk) {
                k = start[p];
                end = start[p + 1];
            }
            while (k < end) {
                typename Row::held_t row[kTogether];
                float wt[kTogether];
#pragma unroll
                for (int m = 0; m < kTogether; ++m) {
                    const u32x2 en = ent[k + m < end ? k + m : end - 1];
                    const uint32_t ow = en.y;
                    wt[m] = __builtin_bit_cast(float, ow);
                    row[m] = *reinterpret_cast<const typename Row::vec_t*>(rows + en.x + j * 4 * (int)sizeof(T));
                }
#pragma unroll
                for (int m = 0; m < kTogether; ++m) {
                    float v[4];
                    Row::unpack_held(row[m], v);
                    if (k + m < end) {
#pragma unroll
                        for (int e = 0; e < 4; ++e) acc[i][e] = __builtin_fmaf(wt[m], v[e], acc[i][e]);
                    }
                }
                k += kTogether;
            }
        }
        __syncthreads();
    }
    float* part = a.part + ((int64_t)split * a.bs + b) * a.nk * a.nh * a.hd + ch + j * 4;
    int g0 = grp;
#pragma unroll
    for (int i = 0; i < PX; ++i) {
        asm volatile("" : "+v"(g0));
        const int p = i * groups + g0;
        if (p < a.nk) *reinterpret_cast<f32x4*>(part + p * pitch) = f32x4{acc[i][0], acc[i][1], acc[i][2], acc[i][3]};
    }
}

// Adds up the query ranges' images of grad_value and, behind those workgroups, the channel parts' dots.
template <typename T>
__global__ __launch_bounds__(256) void gka_sum_kernel(const GkaArgs a, uint32_t image_wgs)
{
    if (blockIdx.x >= image_wgs) {
        const int64_t n = (int64_t)a.bs * a.nq * a.nh * a.S, i = (int64_t)(blockIdx.x - image_wgs) * 256 + threadIdx.x;
        if (i >= n) return;
        float sum = a.dots[i];
        for (int p = 1; p < a.parts; ++p) sum += a.dots[p * n + i];
        static_cast<T*>(a.grad_attn)[i] = from_f32<T>(sum);
        return;
    }
    const int64_t n4 = (int64_t)a.bs * a.nk * a.nh * a.hd / 4, i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= n4) return;
    const f32x4* part = reinterpret_cast<const f32x4*>(a.part) + i;
    f32x4 sum = part[0];
#pragma unroll 4
    for (int s = 1; s < a.sc_splits; ++s) sum += part[s * n4];
    const float v[4] = {sum[0], sum[1], sum[2], sum[3]};
    RowIO<T, 4>::store_global(static_cast<T*>(a.grad_value) + 4 * i, v);
}

template <typename T, bool DOTS, typename F>
hipError_t by_lanes(int lpr_log2, F f)
{
    switch (lpr_log2) {
        case 1: return f(&gka_slab_kernel<T, 1, DOTS>);
        case 2: return f(&gka_slab_kernel<T, 2, DOTS>);
        case 3: return f(&gka_slab_kernel<T, 3, DOTS>);
        case 4: return f(&gka_slab_kernel<T, 4, DOTS>);
        case 5: return f(&gka_slab_kernel<T, 5, DOTS>);
        default: return hipErrorInvalidConfiguration;
    }
}

template <typename T, typename F>
hipError_t by_pixels(int px, F f)
{
    if (px <= 4) return f(&gka_scatter_kernel<T, 4>);
    if (px <= 8) return f(&gka_scatter_kernel<T, 8>);
    if (px <= 12) return f(&gka_scatter_kernel<T, 12>);
    if (px <= kGkaPixels) return f(&gka_scatter_kernel<T, kGkaPixels>);
    return hipErrorInvalidConfiguration;
}

template <typename T>
hipError_t raise_t()
{
    auto raise = [](auto* kernel) {
        return hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, kCuLdsBytes - 256);
    };
    hipError_t e = hipSuccess;
    for (int l = 1; l <= 5; ++l) {
        if (e == hipSuccess) e = by_lanes<T, false>(l, raise);
        if (e == hipSuccess) e = by_lanes<T, true>(l, raise);
    }
    for (int px = 4; px <= kGkaPixels; px += 4)
        if (e == hipSuccess) e = by_pixels<T>(px, raise);
    return e;
}

template <typename T, bool DOTS>
hipError_t slab_t(const GkaArgs& a, hipStream_t stream)
{
    return by_lanes<T, DOTS>(a.lpr_log2, [&](auto* kernel) {
        hipLaunchKernelGGL(kernel, dim3((unsigned)(a.bs * a.nh * a.parts * a.splits)), dim3(a.block), a.lds, stream, a);
        return hipGetLastError();
    });
}

template <typename T>
hipError_t backward_t(const GkaArgs& a, hipStream_t stream)
{
    hipError_t e = slab_t<T, true>(a, stream);
    if (e != hipSuccess) return e;
    e = by_pixels<T>(a.sc_px, [&](auto* kernel) {
        hipLaunchKernelGGL(kernel, dim3((unsigned)(a.bs * a.nh * a.parts * a.sc_splits)), dim3(a.sc_block), a.sc_lds, stream, a);
        return hipGetLastError();
    });
    if (e != hipSuccess) return e;
    const int64_t n4 = (int64_t)a.bs * a.nk * a.nh * a.hd / 4;
    const uint32_t image_wgs = (uint32_t)((n4 + 255) / 256);
    const int64_t dot_wgs = a.parts > 1 ? ((int64_t)a.bs * a.nq * a.nh * a.S + 255) / 256 : 0;
    hipLaunchKernelGGL(gka_sum_kernel<T>, dim3(image_wgs + (uint32_t)dot_wgs), dim3(256), 0, stream, a, image_wgs);
    return hipGetLastError();
}

}  // namespace

hipError_t raise_gka_lds()
{
    hipError_t e = raise_t<float>();
    if (e == hipSuccess) e = raise_t<f16_t>();
    if (e == hipSuccess) e = raise_t<bf16_t>();
    return e;
}

hipError_t launch_gka_forward(int dtype, const GkaArgs& a, hipStream_t stream)
{
    switch (dtype) {
        case MXD_DTYPE_F32: return slab_t<float, false>(a, stream);
        case MXD_DTYPE_F16: return slab_t<f16_t, false>(a, stream);
        case MXD_DTYPE_BF16: return slab_t<bf16_t, false>(a, stream);
        default: return hipErrorInvalidValue;
    }
}

hipError_t launch_gka_backward(int dtype, const GkaArgs& a, hipStream_t stream)
{
    switch (dtype) {
        case MXD_DTYPE_F32: return backward_t<float>(a, stream);
        case MXD_DTYPE_F16: return backward_t<f16_t>(a, stream);
        case MXD_DTYPE_BF16: return backward_t<bf16_t>(a, stream);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace mxd
