// Geometric kernel attention on small maps for gfx950 (MI355X), wave64: forward and backward.
//
//   out[b,q,h,:] = sum over samples s of w[b,q,h,s] * value[b, pixel(b,q,h,s), h, :]        (one pixel per sample, clamped)
//
// (reference: mx_driving/ops/geometric_kernel_attention.py:29-57.)  The maps of this operator are small -- 15 x 25 pixels of 64
// channels, 96 KB per (batch, head) in float32 -- and every pixel is sampled hundreds of times, 2.6 GB of rows per pass at
// [24, 7156 queries, 4 heads, 15 points].  From L1 and L2 they come at 18 TB/s (the general kernels: forward 147 us, dots of the
// backward 279 us with their records); LDS gives 128 bytes per clock and CU, 78 TB/s.  So
//
//   * the forward (and the dots of the backward where lane pairs share a row) puts the (batch, head)'s slab of value into LDS once per
//     workgroup and gathers there.  What bounds them: reading locations and weights and writing the result (300 MB), and LDS.
//   * grad_value is summed by pixel: a workgroup takes tiles of queries, puts their grad_out rows into LDS, sorts the tile's
//     samples by pixel (integer LDS counters) and lets lane groups that own pixels add the rows of their samples to registers.
//     The query ranges of a slab leave float32 images of it, which a last kernel adds up and rounds.
//   * The dots of the backward (gradient of the weights) are formed on the way, with the pixel's row of value in registers: a sample's
//     grad_out row is read once for both.  (As a kernel of their own, gathering rows of value from the slab: 112 us at the size above.)
//     What bounds it: the vector ALU of the walk (60 instructions for four samples of each of a wavefront's groups) and, with clamping that
//     piles samples on the border pixels (16 times the average on the corners), groups whose lists have ended: a tile of 192 queries has 7
//     samples per pixel.  Smaller tiles lose (64 queries: 356 against 286 us for the backward), so do larger ones that a CU holds one
//     workgroup of (307), and so does sharing long lists among the groups of a wavefront (327; hot pixels in two to four parts: 226 against 207).  (The weights go round a quad by moves: folded into the multiply-adds by inline
//     assembly, whose operands' wait states the compiler does not see, they were read too early.)
//
// Measured at that size, float32: forward 147 -> 82 us, dots and grad_value 649 -> 295 (112 + 183) -> 207, sum of the images 9; float16
// forward and backward 65 and 220 -> 190 us.
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

// Forward (DOTS = false) or, of rows of 8 channels in float32, gradient of the weights (DOTS = true); LPR lanes of 16 bytes share a row.
template <typename T, int LPR_LOG2, bool DOTS>
__global__ __launch_bounds__(1024) void gka_slab_kernel(const GkaArgs a)
{
    constexpr int LPR = 1 << LPR_LOG2, U = kWave / LPR, VEC = 16 / (int)sizeof(T);
    static_assert(!DOTS || sizeof(T) == 4);
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
#pragma unroll
        for (int e = 0; e < VEC; ++e) acc[e] = 0.0f;
        if constexpr (DOTS) {
            Row::unpack_held(next_row, gv);
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
                        float v[VEC], p = 0.0f;
                        Row::unpack(*reinterpret_cast<const typename Row::raw_t*>(slab + mine[s].row + c * 16), v);
#pragma unroll
                        for (int e = 0; e < VEC; ++e) p = __builtin_fmaf(v[e], gv[e], p);
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

// grad_value, or one query range's part of it, and the gradient of the weights: PX pixels per lane group.
// QUAD: four lanes and more share a row (GkaArgs::sc_dots); without, the gradient of the weights is left to gka_slab_kernel.
template <typename T, int PX, bool QUAD>
__global__ __launch_bounds__(1024) void gka_scatter_kernel(const GkaArgs a)
{
    typedef RowIO<T, 4> Row;
    constexpr bool kLeaveOut = !(QUAD && sizeof(T) == 4 && PX > 12);
    constexpr int NS = gka_samples(PX, QUAD), HS = PX > 12 ? 2 : NS / 2;  // samples of a tile per thread, and those requested together
    extern __shared__ __align__(16) unsigned char smem[];
    __shared__ uint32_t wave_sum[16];
    const int tid = (int)threadIdx.x, block = (int)blockDim.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    auto add = [](uint32_t x, uint32_t y) { return x + y; };
    const int row_bytes = a.part_ch * (int)sizeof(T);
    i32x4* lvl = reinterpret_cast<i32x4*>(smem);
    u32x2* ent = reinterpret_cast<u32x2*>(smem + kGkaLevelBytes);                    // sorted samples: {row in `rows`, weight}
    unsigned char* rows = reinterpret_cast<unsigned char*>(ent) + (((size_t)a.sc_tile_q * a.S * 8 + 15) & ~(size_t)15);
    const uint32_t zero_row = (uint32_t)a.sc_tile_q * (uint32_t)row_bytes;           // (behind the tile's rows, one of zeros)
    uint32_t* count = reinterpret_cast<uint32_t*>(rows + zero_row + row_bytes);      // [nk]
    uint32_t* start = count + a.nk;                                                  // [nk + 1]
    uint32_t* ranks = start + a.nk + 1;                                              // [kWave]
    uint16_t* pixel_of = reinterpret_cast<uint16_t*>(ranks + kWave);                 // QUAD: [PX][groups] the groups' pixels, nk: none
    uint32_t wg = xcd_order(blockIdx.x, gridDim.x);
    const int h = (int)(wg % (uint32_t)a.nh);
    wg /= (uint32_t)a.nh;
    const int cpart = (int)(wg % (uint32_t)a.parts), ch = h * a.hd + cpart * a.part_ch;  // first channel of the rows
    wg /= (uint32_t)a.parts;
    const int split = (int)(wg % (uint32_t)a.sc_splits), b = (int)(wg / (uint32_t)a.sc_splits);
    const int q_begin = split * a.sc_split_q, q_end = q_begin + a.sc_split_q < a.nq ? q_begin + a.sc_split_q : a.nq;
    const T* attn = static_cast<const T*>(a.attn);
    const T* gout = static_cast<const T*>(a.grad_out) + (int64_t)b * a.nq * a.nh * a.hd + ch;
    const int pitch = a.nh * a.hd;
    const int groups_log2 = __builtin_ctz(block) - a.sc_lanes_log2, groups = 1 << groups_log2;
    load_levels(a, lvl);
    for (int i = tid; i < a.nk; i += block) count[i] = 0;
    if constexpr (QUAD)
        for (int i = tid; i < PX << groups_log2; i += block) pixel_of[i] = (uint16_t)(i < a.nk ? i : a.nk);
    if (tid < kWave) ranks[tid] = 0;
    for (int i = tid; i < row_bytes / 4; i += block) reinterpret_cast<uint32_t*>(rows + zero_row)[i] = 0;
    float acc[PX][4];
#pragma unroll
    for (int i = 0; i < PX; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[i][e] = 0.0f;
    const uint32_t spare = min((uint32_t)(tid & (kWave - 1)), (uint32_t)a.nk);  // (of the words from count[nk] on, start[0] to start[nk])
    const int per = (a.nk + block - 1) / block;        // counters of a thread in the prefix sum
    const int piece_log2 = a.lpr_log2;                 // 16-byte pieces of a row
    __syncthreads();
    for (int q0 = q_begin; q0 < q_end; q0 += a.sc_tile_q) {
        const int nq = q0 + a.sc_tile_q < q_end ? a.sc_tile_q : q_end - q0, n = nq * a.S;
        // ---- samples of the tile: pixel, weight, place among the samples of the pixel; rows of the tile into LDS ----------
        uint32_t place[NS];  // pixel (nk: none) | place << 16
        T w[NS];
        int t0 = tid;
        asm volatile("" : "+v"(t0));  // (what follows from it is not to be kept across the tiles)
        typedef RowIO<T, 16 / (int)sizeof(T)> Wide;
        const int pieces = nq << piece_log2;
        // (the tile's parts of the tensors, from where 32-bit offsets reach: gka_plan_parts)
        const int64_t first = (((int64_t)b * a.nq + q0) * a.nh + h) * a.S;
        const float* tile_loc = a.loc + 2 * first;
        const T *tile_attn = attn + first, *tile_rows = gout + (int64_t)q0 * pitch;
        const uint32_t per_q = (uint32_t)(a.nh * a.S);
        if (a.sc_direct) {
            // (straight into LDS, while the samples are on their way too)
            for (int i0 = wave * kWave; i0 < pieces; i0 += block) {
                const int i = i0 + (t0 & (kWave - 1)), q = i >> piece_log2, p = i & ((1 << piece_log2) - 1);
                if (i < pieces)
                    __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(tile_rows + (uint32_t)(q * pitch + p * (16 / (int)sizeof(T)))),
                                                     (__attribute__((address_space(3))) void*)(rows + i0 * 16), 16, 0, 0);
            }
        }
#pragma unroll
        for (int half = 0; half < NS; half += HS) {
            // (A wavefront beyond the tile's samples, whose lanes would all count on the same word, one addition after the other: 6 x 900 queries x 4
            //  heads x 4 points on 15 x 25 pixels, backward in float32 8 channels 33.5 -> 29.8 us, 64 channels 30.9 -> 27.6, on 60 x 66 in float16 16
            //  channels 41.6 -> 33.7.  Not where the branch costs 34 spilled registers more: 24 x 7156 x 4 x 15 on 30 x 30 pixels 0.88 of the speed.
            //  There, and in float32's other forms, the lanes without a sample count on words of their own: 30 x 30 pixels, 6 x 900 x 4 x 4, 1.07.)
            if (kLeaveOut && half * block + wave * kWave >= n) {
#pragma unroll
                for (int k = 0; k < HS; ++k) place[half + k] = (uint32_t)a.nk;
                continue;
            }
            f32x2 xy[HS];
#pragma unroll
            for (int k = 0; k < HS; ++k) {
                const uint32_t i = t0 + (half + k) * block < n ? t0 + (half + k) * block : 0, q = (i * a.s_magic) >> 20, at = q * per_q + (i - q * (uint32_t)a.S);
                xy[k] = load_xy(tile_loc, at);
                w[half + k] = tile_attn[at];
            }
            asm volatile("" ::: "memory");
            __builtin_amdgcn_sched_barrier(0);  // (requested together)
#pragma unroll
            for (int k = 0; k < HS; ++k) {
                const int i = t0 + (half + k) * block, q = (int)(((uint32_t)i * a.s_magic) >> 20);
                const int32_t px = sample_pixel(a, lvl, i < n ? i - q * a.S : 0, xy[k]);
                place[half + k] = (uint32_t)(i < n && px >= 0 ? px : a.nk);
            }
            uint32_t before[HS];
#pragma unroll
            for (int k = 0; k < HS; ++k) {  // (samples without a pixel: `start`, not yet in use)
                uint32_t at = place[half + k];
                if (QUAD && sizeof(T) == 4 && at == (uint32_t)a.nk) at += spare;
                before[k] = atomicAdd(&count[at], 1u);
            }
#pragma unroll
            for (int k = 0; k < HS; ++k) place[half + k] |= before[k] << 16;
        }
        if (a.sc_direct) {
            __builtin_amdgcn_s_waitcnt(0x0F70);  // (vmcnt(0))
        } else for (int i0 = t0; i0 < pieces; i0 += 4 * block) {
            typename Wide::vec_t v[4];
#pragma unroll
            for (int m = 0; m < 4; ++m) {
                const int i = i0 + m * block, q = i >> piece_log2, p = i & ((1 << piece_log2) - 1);
                if (q < nq) v[m] = *reinterpret_cast<const typename Wide::mem_t*>(tile_rows + (uint32_t)(q * pitch + p * (16 / (int)sizeof(T))));
            }
#pragma unroll
            for (int m = 0; m < 4; ++m)
                if ((i0 + m * block) >> piece_log2 < nq) reinterpret_cast<typename Wide::vec_t*>(rows)[i0 + m * block] = v[m];
        }
        __syncthreads();
        if (QUAD && q0 == q_begin && q_end - q_begin > a.sc_tile_q) {
            // Pixels are dealt to the groups by the samples they have in the first tile, most first: the groups of a wavefront walk
            // pixels of about the same number of samples side by side.  The wavefront that has the most of the first row -- the corners
            // -- and the one beside it on its SIMD have the least of the other rows.  (Four buckets per power of two of the number over
            // the average.  Workgroups of one tile have nothing to learn from it, and where lane pairs walk a pixel it gains nothing.)
            auto bucket = [&](uint32_t c) {
                const uint32_t v = __builtin_bit_cast(uint32_t, (float)c * (float)a.nk / (float)n) >> 21;
                const uint32_t k = v < ((127u - 4u) << 2) ? 0u : v - ((127u - 4u) << 2);
                return kWave - 1 - (k < kWave ? k : kWave - 1);
            };
            int t = tid;
            asm volatile("" : "+v"(t));
#pragma unroll 1
            for (int i = t; i < a.nk; i += block) atomicAdd(&ranks[bucket(count[i])], 1u);
            __syncthreads();
            if (tid < kWave) {
                const uint32_t v = ranks[tid];
                ranks[tid] = wave_scan(v, add) - v;
            }
            __syncthreads();
            const int per_wave_log2 = 6 - a.sc_lanes_log2, waves = block / kWave;
#pragma unroll 1
            for (int i = t; i < PX << groups_log2; i += block) {
                const int rank = i < a.nk ? (int)atomicAdd(&ranks[bucket(count[i])], 1u) : i, row = rank >> groups_log2;
                int at = rank & (groups - 1);
                if (row > 0) {
                    const int v = at >> per_wave_log2, to = v < waves - 2 ? (v < 3 ? v + 1 : v + 2) : v == waves - 2 ? 4 : 0;
                    at = (at & ((1 << per_wave_log2) - 1)) | to << per_wave_log2;
                }
                pixel_of[(row << groups_log2) + at] = (uint16_t)(i < a.nk ? i : a.nk);
            }
        }
        // ---- first sample of every pixel ------------------------------------------------------------------------------------
        uint32_t sum = 0;
        int t2 = tid;
        asm volatile("" : "+v"(t2));
        const int c0 = t2 * per;
        for (int i = c0; i < c0 + per && i < a.nk; ++i) sum += count[i];
        const uint32_t inc = wave_scan(sum, add);
        if ((t2 & (kWave - 1)) == kWave - 1) wave_sum[wave] = inc;
        __syncthreads();
        uint32_t at = inc - sum;
        for (int v = 0; v < wave; ++v) at += wave_sum[v];
        for (int i = c0; i < c0 + per && i < a.nk; ++i) {
            start[i] = at;
            at += count[i];
            count[i] = 0;
            if (i == a.nk - 1) start[a.nk] = at;
        }
        __syncthreads();
        uint32_t at2[NS / 2];  // entries of the samples, two per word, 0xFFFF: none
#pragma unroll
        for (int k = 0; k < NS; ++k) {
            uint32_t e = 0xFFFFu;
            if ((place[k] & 0xFFFFu) < (uint32_t)a.nk) {
                const uint32_t q = ((uint32_t)(t0 + k * block) * a.s_magic) >> 20;
                e = start[place[k] & 0xFFFFu] + (place[k] >> 16);
                ent[e] = u32x2{q * (uint32_t)row_bytes, __builtin_bit_cast(uint32_t, to_f32(w[k]))};
            }
            at2[k / 2] = k % 2 == 0 ? e : at2[k / 2] | e << 16;
        }
        __syncthreads();
        // ---- the groups add the rows of their pixels' samples ---------------------------------------------------------------
        int t3 = tid;
        asm volatile("" : "+v"(t3));
        int g0 = t3 >> a.sc_lanes_log2;
        const int j = t3 & ((1 << a.sc_lanes_log2) - 1);
        auto samples_of = [&](int p, uint32_t& k, uint32_t& end) {
            if (p < a.nk) {
                k = start[p];
                end = start[p + 1];
            }
        };
        if constexpr (QUAD) {
            // A lane looks up one entry of four, and a quad hands them round: what the walk reads from LDS, which binds it, is rows.
            // An entry's weight gives way to its dot product with the pixel's row of value.
            const T* value = static_cast<const T*>(a.value) + (int64_t)b * a.nk * a.nh * a.hd + ch + j * 4;
            const uint32_t mine = (uint32_t)(j & 3), turned = mine ^ ((j >> 2) & 1 ? 3u : 0u);  // (the mirrors below turn a quad round)
            const bool odd = (turned & 1u) != 0, upper = (turned & 2u) != 0;
            const unsigned char* my_rows = rows + j * 4 * (int)sizeof(T);
            auto fetch = [&](int p) { return Row::load_held(value + (uint32_t)((p < a.nk ? p : 0) * pitch)); };
            int p = pixel_of[g0];
            typename Row::held_t vnext = fetch(p);
#pragma unroll
            for (int i = 0; i < PX; ++i) {
                asm volatile("" : "+v"(g0));
                uint32_t k = 0, end = 0;
                samples_of(p, k, end);
                const typename Row::held_t vrow = vnext;
                if (i + 1 < PX) {
                    p = pixel_of[((i + 1) << groups_log2) + g0];
                    vnext = fetch(p);
                }
                while (k < end) {
                    const bool ok = k + mine < end;
                    const u32x2 en = ent[ok ? k + mine : k];
                    const uint32_t ox = en.x, oy = en.y;
                    const int off = (int)(ok ? ox : zero_row);
                    const float wt = ok ? __builtin_bit_cast(float, oy) : 0.0f;
                    typename Row::held_t row[4];
                    row[0] = *reinterpret_cast<const typename Row::vec_t*>(my_rows + (uint32_t)__builtin_amdgcn_update_dpp(0, off, 0x00, 0xF, 0xF, true));
                    row[1] = *reinterpret_cast<const typename Row::vec_t*>(my_rows + (uint32_t)__builtin_amdgcn_update_dpp(0, off, 0x55, 0xF, 0xF, true));
                    row[2] = *reinterpret_cast<const typename Row::vec_t*>(my_rows + (uint32_t)__builtin_amdgcn_update_dpp(0, off, 0xAA, 0xF, 0xF, true));
                    row[3] = *reinterpret_cast<const typename Row::vec_t*>(my_rows + (uint32_t)__builtin_amdgcn_update_dpp(0, off, 0xFF, 0xF, 0xF, true));
                    float d[4];
                    auto use = [&](auto lane_of_quad) {
                        constexpr int m = decltype(lane_of_quad)::value;
                        if constexpr (sizeof(T) == 2) {
                            typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));
                            const u32x2_t vv = __builtin_bit_cast(u32x2_t, vrow), gg = __builtin_bit_cast(u32x2_t, row[m]);
                            const uint32_t v0 = vv.x, v1 = vv.y, g0 = gg.x, g1 = gg.y;
                            d[m] = dot2_acc<T>(v1, g1, dot2_acc<T>(v0, g0, 0.0f));
                        } else {
                            d[m] = vrow[0] * row[m][0];
#pragma unroll
                            for (int e = 1; e < 4; ++e) d[m] = __builtin_fmaf(vrow[e], row[m][e], d[m]);
                        }
                        float g[4];
                        Row::unpack_held(row[m], g);
                        const float w1 = dpp_xchg<m * 0x55>(wt);
#pragma unroll
                        for (int e = 0; e < 4; ++e) acc[i][e] = __builtin_fmaf(w1, g[e], acc[i][e]);
                    };
                    use(std::integral_constant<int, 0>{});
                    use(std::integral_constant<int, 1>{});
                    use(std::integral_constant<int, 2>{});
                    use(std::integral_constant<int, 3>{});
                    // over the lanes of the group, four sums at a time: every step halves what a lane keeps
                    const float d01 = (odd ? d[1] : d[0]) + dpp_xchg<0xB1>(odd ? d[0] : d[1]);
                    const float d23 = (odd ? d[3] : d[2]) + dpp_xchg<0xB1>(odd ? d[2] : d[3]);
                    float dot = (upper ? d23 : d01) + dpp_xchg<0x4E>(upper ? d01 : d23);
                    if (a.sc_lanes_log2 >= 3) dot += dpp_xchg<0x141>(dot);
                    if (a.sc_lanes_log2 >= 4) dot += dpp_xchg<0x140>(dot);
                    if (a.sc_lanes_log2 >= 5) dot += __shfl_xor(dot, 16, 64);
                    if (a.sc_lanes_log2 >= 6) dot += __shfl_xor(dot, 32, 64);
                    if (ok && j < 4) reinterpret_cast<float*>(ent)[2 * (k + mine) + 1] = dot;
                    k += 4;
                }
            }
        } else {
#pragma unroll
            for (int i = 0; i < PX; ++i) {
                asm volatile("" : "+v"(g0));
                uint32_t k = 0, end = 0;
                samples_of((i << groups_log2) + g0, k, end);
                for (; k < end; k += 4) {
                    typename Row::held_t row[4];
                    float wt[4];
#pragma unroll
                    for (int m = 0; m < 4; ++m) {
                        const u32x2 en = ent[k + m < end ? k + m : end - 1];
                        const uint32_t ow = en.y;
                        wt[m] = __builtin_bit_cast(float, ow);
                        row[m] = *reinterpret_cast<const typename Row::vec_t*>(rows + en.x + j * 4 * (int)sizeof(T));
                    }
#pragma unroll
                    for (int m = 0; m < 4; ++m) {
                        float v[4];
                        Row::unpack_held(row[m], v);
                        if (k + m < end) {
#pragma unroll
                            for (int e = 0; e < 4; ++e) acc[i][e] = __builtin_fmaf(wt[m], v[e], acc[i][e]);
                        }
                    }
                }
            }
        }
        __syncthreads();
        if constexpr (QUAD) {
            T* dst = static_cast<T*>(a.grad_attn) + first;
            float* dots = a.dots + (int64_t)cpart * a.bs * a.nq * a.nh * a.S + first;
            int t1 = tid;
            asm volatile("" : "+v"(t1));
#pragma unroll
            for (int k = 0; k < NS; ++k) {
                const int i = t1 + k * block;
                if (i >= n) break;
                const uint32_t e = at2[k / 2] >> (k % 2 * 16) & 0xFFFFu;
                const float d = e != 0xFFFFu ? reinterpret_cast<const float*>(ent)[2 * e + 1] : 0.0f;
                const uint32_t q = ((uint32_t)i * a.s_magic) >> 20, at = q * per_q + ((uint32_t)i - q * (uint32_t)a.S);
                if (a.parts == 1) dst[at] = from_f32<T>(d);
                else dots[at] = d;
            }
        }
    }
    int g0 = tid >> a.sc_lanes_log2;
    float* part = a.part + ((int64_t)split * a.bs + b) * a.nk * a.nh * a.hd + ch + (tid & ((1 << a.sc_lanes_log2) - 1)) * 4;
#pragma unroll
    for (int i = 0; i < PX; ++i) {
        asm volatile("" : "+v"(g0));
        const int p = QUAD ? pixel_of[(i << groups_log2) + g0] : (i << groups_log2) + g0;
        if (p < a.nk) *reinterpret_cast<f32x4*>(part + (int64_t)p * pitch) = f32x4{acc[i][0], acc[i][1], acc[i][2], acc[i][3]};
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

template <typename T, typename F>
hipError_t by_lanes(int lpr_log2, F f)
{
    switch (lpr_log2) {
        case 1: return f(&gka_slab_kernel<T, 1, false>);
        case 2: return f(&gka_slab_kernel<T, 2, false>);
        case 3: return f(&gka_slab_kernel<T, 3, false>);
        case 4: return f(&gka_slab_kernel<T, 4, false>);
        case 5: return f(&gka_slab_kernel<T, 5, false>);
        default: return hipErrorInvalidConfiguration;
    }
}

template <typename T, typename F>
hipError_t by_pixels(int px, int lanes_log2, F f)
{
    if constexpr (sizeof(T) == 4)  // (16-bit rows are shared by four lanes at least)
        if (lanes_log2 < 2) {
            if (px <= 4) return f(&gka_scatter_kernel<T, 4, false>);
            if (px <= 8) return f(&gka_scatter_kernel<T, 8, false>);
            if (px <= 12) return f(&gka_scatter_kernel<T, 12, false>);
            return px <= kGkaPixels ? f(&gka_scatter_kernel<T, kGkaPixels, false>) : hipErrorInvalidConfiguration;
        }
    if (px <= 4) return f(&gka_scatter_kernel<T, 4, true>);
    if (px <= 8) return f(&gka_scatter_kernel<T, 8, true>);
    if (px <= 12) return f(&gka_scatter_kernel<T, 12, true>);
    if (px <= kGkaPixels) return f(&gka_scatter_kernel<T, kGkaPixels, true>);
    return hipErrorInvalidConfiguration;
}

template <typename T>
hipError_t raise_t()
{
    auto raise = [](auto* kernel) {
        return hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, kCuLdsBytes - 256);
    };
    hipError_t e = hipSuccess;
    for (int l = 1; l <= 5; ++l)
        if (e == hipSuccess) e = by_lanes<T>(l, raise);
    if constexpr (sizeof(T) == 4)
        if (e == hipSuccess) e = raise(&gka_slab_kernel<T, 1, true>);
    for (int px = 4; px <= kGkaPixels; px += 4)
        for (int lanes_log2 : {1, 2})
            if (e == hipSuccess) e = by_pixels<T>(px, lanes_log2, raise);
    return e;
}

hipError_t launch_slab(void (*kernel)(const GkaArgs), const GkaArgs& a, hipStream_t stream)
{
    hipLaunchKernelGGL(kernel, dim3((unsigned)(a.bs * a.nh * a.parts * a.splits)), dim3(a.block), a.lds, stream, a);
    return hipGetLastError();
}

template <typename T>
hipError_t backward_t(const GkaArgs& a, hipStream_t stream)
{
    hipError_t e = hipSuccess;
    if (!a.sc_dots) {  // (lane pairs share a row: 8 channels in float32)
        if constexpr (sizeof(T) == 4) e = a.lpr_log2 == 1 ? launch_slab(&gka_slab_kernel<T, 1, true>, a, stream) : hipErrorInvalidConfiguration;
        else e = hipErrorInvalidConfiguration;
    }
    if (e != hipSuccess) return e;
    e = by_pixels<T>(a.sc_px, a.sc_lanes_log2, [&](auto* kernel) {
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
        case MXD_DTYPE_F32: return by_lanes<float>(a.lpr_log2, [&](auto* kernel) { return launch_slab(kernel, a, stream); });
        case MXD_DTYPE_F16: return by_lanes<f16_t>(a.lpr_log2, [&](auto* kernel) { return launch_slab(kernel, a, stream); });
        case MXD_DTYPE_BF16: return by_lanes<bf16_t>(a.lpr_log2, [&](auto* kernel) { return launch_slab(kernel, a, stream); });
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
