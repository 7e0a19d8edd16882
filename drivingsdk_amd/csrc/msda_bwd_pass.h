// First backward kernel of multi-scale deformable attention for gfx950 (MI355X), wave64, in its common form: rows of up to 128 bytes
// whose workgroups make one pass -- 32 units, with one unit per query (up to 16 samples) or two (up to 32).  Plain operator and its
// fused form, tile pass behind it.  What it computes and what it hands over: msda_bwd_kernel.h, which has the general form.
//
// What bounds it: the way of the rows from L2 into the registers and, behind it, the vector ALU, so whatever is neither a row nor
// a product of one is kept small:
//   * a sample's geometry (and the fused form's softmax weight) is derived once.  Its pair records are merged with their weights and
//     counted, their place in the run is what the counter returns, and they are written before the gather, which covers their way
//     to memory;
//   * run starts are a scan that every wavefront makes for itself (up to 64 tiles): three barriers per slab;
//   * the dots replace the row offsets that they were gathered by, in place;
//   * rows of 33 to 64 bytes are read by 4 lanes of 16 bytes (where there are enough of them: launch_pass): a row of 64 bytes costs the
//     L1 a line of 128 however it is read, but half of the instructions of 8 lanes of 8 bytes (181 -> 117 million at the last shape
//     below).
// Measured, this kernel against the instantiations of the general one that it replaces (two batch elements of the encoder in float32 /
// the same in bfloat16, fused / 6 x 9675 queries of 32 samples over 30 825 keys in float16): 142 -> 132, 185 -> 132, 399 -> 379 us.
// A workgroup goes through one slab: with a loop over several, shared out evenly, the last case took 430 to 490 us (values kept across
// the loop cost a wavefront per SIMD, and a share of slow slabs nobody helps with), and 28 bytes of scratch memory per lane, for spilled
// values, cost a sixth of the time by themselves: every wavefront waits for it before it starts.
#pragma once
#include <type_traits>

#include "msda_bwd_parts.h"

namespace mxd {

constexpr int kPassUnits = 32;                          // units per workgroup, whatever the lanes per unit
constexpr int kPassRecWords = 2 * kChunk * kRecDwords;  // words of a unit's records, at most
constexpr int kPassGradWords = 4;                       // words of a lane's piece of a row of grad_out

// LDS: levels, softmax terms of the fused form, strips (a unit's row offsets, then its dots), records, counters.  With 4 lanes per
// unit a workgroup is two wavefronts, and the strips take the records' place once the slab is written: 12.8 KB instead of 21.
inline __host__ __device__ size_t pass_lds_bytes(int nl, int tbl_stride, int lpr, bool fused)
{
    const size_t strips = kPassUnits * kChunkStride * sizeof(u32x4), recs = kPassUnits * kPassRecWords * 4;
    return (size_t)nl * sizeof(i32x4) + (fused ? kPassUnits * sizeof(f32x4) : 0) + (lpr == 4 ? recs : strips + recs) + (size_t)tbl_stride * 4;
}

template <typename T, int VEC, int LPR, int SRC, int UPQ>
__global__ __launch_bounds__(kPassUnits* LPR, LPR == 8 ? 6 : 4) void msda_bwd_pass_kernel(const KArgs a)
{
    static_assert(SRC == kSrcPlain || SRC == kSrcFused, "the plain operator and its fused form");
    static_assert(UPQ == 1 || UPQ == 2, "units per query");
    constexpr bool FUSED = SRC == kSrcFused;
    static_assert(LPR == 4 || LPR == 8, "lanes per unit");
    constexpr int LG = LPR == 4 ? 2 : 3, U = kWave / LPR, SP = UPQ - 1;  // ..., units per wavefront, log2 of the units per query
    constexpr int KS = kChunk / LPR;                                     // samples per lane
    constexpr int kThreads = kPassUnits * LPR;
    constexpr bool OVER = LPR == 4;  // strips in the records' place
    static_assert(kChunkStride * 4 <= kPassRecWords, "strips fit the records' place");
    typedef typename RowIO<T, VEC>::raw_t raw_t;
    static_assert(VEC * (sizeof(T) == 2 && VEC % 2 == 0 ? 2 : 4) <= kPassGradWords * 4);

    extern __shared__ __align__(16) unsigned char smem[];
    {
        const LevelLanes lv(a, (int)threadIdx.x & (kWave - 1));
        if ((int)threadIdx.x < a.nl) reinterpret_cast<i32x4*>(smem)[threadIdx.x] = i32x4{lv.geo.x, lv.geo.y, lv.geo.z, lv.first};
        zero_fill(a, lv);
    }
    // (the arithmetic phases run at a raised priority, the gather at the default one: BEVFormer shape 988.6 -> 964.8 us, encoder
    //  shape unchanged; the other way round the encoder shape loses 7 us)
    __builtin_amdgcn_s_setprio(2);

    const int tid = (int)threadIdx.x;
    const int lane = tid & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    i32x4* lvl = reinterpret_cast<i32x4*>(smem);  // {H, W, first key, first tile (-1: none in the run table)}
    float* stats = reinterpret_cast<float*>(smem + (size_t)a.nl * sizeof(i32x4));  // fused form: per unit {max logit, sum of exponentials, D}
    u32x4* strips = reinterpret_cast<u32x4*>(stats + (FUSED ? 4 * kPassUnits : 0));
    u32_alias* recs = reinterpret_cast<u32_alias*>(strips + (OVER ? 0 : kPassUnits * kChunkStride));
    int32_t* cursor = reinterpret_cast<int32_t*>(recs + kPassUnits * kPassRecWords);  // [tbl_stride] records per tile
    // where eight points of a unit are gathered side by side, this wavefront's rows of grad_out: in the records' place, behind the strips
    // if those are there
    u32_alias* grads = recs + (OVER ? kPassUnits * kChunkStride * 4 : 0) + wave * kWave * kPassGradWords;
    static_assert((OVER ? kPassUnits * kChunkStride * 4 : 0) + kThreads * kPassGradWords <= kPassUnits * kPassRecWords, "rows fit behind the strips");
    const bool eight = a.np >= 8 && (UPQ == 2 || (LPR == 4 && a.S % 8 == 0));

    const int g = lane / LPR, c = lane % LPR;
    u32x4* strip = strips + wave * U * kChunkStride;  // this wavefront's
    u32x4* mine = strip + g * kChunkStride;           // this lane's unit's
    if constexpr (FUSED) stats += wave * U * 4;
    const T* attn = static_cast<const T*>(a.attn);
    const T* ref = static_cast<const T*>(a.ref);
    T* gloc = static_cast<T*>(a.grad_loc);
    T* gattn = static_cast<T*>(a.grad_attn);
    const int ch = c * VEC, start = ch < a.hd ? piece_start<VEC>(ch, a.hd) : 0;
    // lanes of a pass per unit: 16, or 8 or 4 for queries of so few samples (aligned groups of 4 lanes belong to one query either way)
    const int pk = a.S <= 4 ? 2 : a.S <= 8 ? 3 : 4, pk_mask = (1 << pk) - 1, entries = U << pk;
    constexpr bool kDot2 = sizeof(T) == 2 && VEC % 2 == 0;
    constexpr int kPairs = kDot2 ? VEC / 2 : 1;

    Work wk;
    if (!decode_block(a.plan, blockIdx.x, a.bs, a.nh, a.nq, &wk)) return;  // (uniform)
    const int q0 = wk.q_begin + ((wave * U) >> SP);
    const int64_t bq = (int64_t)wk.b * a.nq;
    for (int i = tid; i < a.tbl_stride; i += kThreads) cursor[i] = 0;

    // ---- everything that comes from memory but the rows of value -------------------------------------------------------
    // (sample k of a lane: number sn of the query that its unit u has a part of; e: index of the location pair and of the weight,
    //  from the wavefront's first query on)
    struct Place {
        int u, sn, q;
        uint32_t e;
        bool active;
    };
    // (derived from the lane again wherever it is needed: kept, it takes ten registers through the whole trip)
    auto place = [&](int k) {
        Place p;
        int i = lane + k * kWave;
        asm volatile("" : "+v"(i));
        p.u = i >> pk;
        p.sn = ((p.u & SP) << 4) + (i & pk_mask);
        p.q = q0 + (p.u >> SP);
        p.e = (uint32_t)((p.u >> SP) * a.nh * a.S_full + p.sn);
        p.active = i < entries && p.q < wk.q_end && p.sn < a.S;
        return p;
    };
    auto level_of = [&](const Place& p) { return p.active ? (int)(((uint32_t)p.sn * a.np_magic) >> 20) : 0; };
    const int64_t e0 = ((bq + q0) * a.nh + wk.h) * a.S_full;
    float x[KS], y[KS], aw[KS];
#pragma unroll
    for (int k = 0; k < KS; ++k) {
        const Place p = place(k);
        x[k] = y[k] = aw[k] = 0.0f;
        if (p.active) {
            x[k] = to_f32((static_cast<const T*>(a.loc) + 2 * e0)[2 * p.e]);
            y[k] = to_f32((static_cast<const T*>(a.loc) + 2 * e0)[2 * p.e + 1]);
            aw[k] = to_f32((attn + e0)[p.e]);
        }
    }
    const int qg = q0 + (g >> SP);
    const bool row_ok = qg < wk.q_end && ch < a.hd;
    const int64_t row = ((bq + (qg < wk.q_end ? qg : wk.q_begin)) * a.nh + wk.h) * a.hd + start;
    typename RowIO<T, VEC>::held_t grow = RowIO<T, VEC>::load_held(static_cast<const T*>(a.grad_out) + row);
    float gv[VEC];
    uint32_t gpk[kPairs];
    auto unpack_grad = [&]() {
        RowIO<T, VEC>::unpack_held(grow, gv);
        // (channels that the piece before it has as well count there)
#pragma unroll
        for (int e = 0; e < VEC; ++e)
            if (!row_ok || start + e < ch) gv[e] = 0.0f;
        if constexpr (kDot2) {
            typedef T t2 __attribute__((ext_vector_type(2)));
#pragma unroll
            for (int e = 0; e < kPairs; ++e)
                gpk[e] = __builtin_bit_cast(uint32_t, t2{from_f32<T>(gv[2 * e]), from_f32<T>(gv[2 * e + 1])});
        }
    };
    __syncthreads();  // counters are zero (and, the first time, the levels are there)
    if constexpr (FUSED) {
        // softmax backward: grad_logit_s = w_s * (grad_w_s - sum_t w_t * grad_w_t), and the sum over the
        // unit's samples equals the dot product of the forward row with the grad_out row
        float orow[VEC], dsum = 0.0f;
        RowIO<T, VEC>::load_global(static_cast<const T*>(a.out) + row, orow);
        unpack_grad();
#pragma unroll
        for (int e = 0; e < VEC; ++e) dsum = __builtin_fmaf(orow[e], gv[e], dsum);
        dsum = group_sum<LG>(dsum);
        if (c == 0) stats[4 * g + 2] = dsum;
        // lanes 16u .. 16u + 15 share unit u
#pragma unroll
        for (int k = 0; k < KS; ++k) {
            const int i = lane + k * kWave, u = i >> 4, sn = i & (kChunk - 1), q = q0 + u;
            const bool act = q < wk.q_end && sn < a.S;
            const float lg = act ? to_f32(attn[((bq + q) * a.nh + wk.h) * a.S_full + sn]) : -__builtin_inff();
            const float m = group_max<4>(lg), sum = group_sum<4>(act ? expf(lg - m) : 0.0f);
            if (sn == 0) {
                stats[4 * u + 0] = m;
                stats[4 * u + 1] = sum;
            }
        }
        wave_lds_sync();
    }

    // ---- geometry, records ---------------------------------------------------------------------------------------------
    float lw[KS], lh[KS];
    bool valid[KS];
    int32_t held[KS];  // with the strips in the records' place: {first pixel, which corners exist}
    struct {
        int32_t tile, at;  // its tile (-1: no record) and its place in the tile's run
        uint32_t x;        // {pixel within the tile | query}
        float wa, wb;
    } rec[KS][2];
#pragma unroll
    for (int k = 0; k < KS; ++k) {
        const Place p = place(k);
        const int l = level_of(p);
        const i32x4 L = lvl[l];
        float xk = x[k], yk = y[k];
        if constexpr (FUSED) {
            if (p.active) {
                fused_location(a, ref + ((bq + p.q) * a.nl + l) * a.ref_dim, L, xk, yk);
                aw[k] = expf(aw[k] - stats[4 * p.u + 0]) / stats[4 * p.u + 1];
            }
        }
        const Sample sm = sample_geometry(xk, yk, L, a.nk, p.active);
        lw[k] = sm.lw;
        lh[k] = sm.lh;
        valid[k] = sm.valid;
        if constexpr (OVER) {
            // (fewer than 2^27 rows: the slice is below 2 GiB and its rows are longer than 16 bytes)
            held[k] = (sm.pix[0] << 4) | (sm.cvalid[0] ? 1 : 0) | (sm.cvalid[1] ? 2 : 0) | (sm.cvalid[2] ? 4 : 0) | (sm.cvalid[3] ? 8 : 0);
        } else if (lane + k * kWave < entries) {
            u32x4 off;
#pragma unroll
            for (int j = 0; j < 4; ++j) off[j] = sm.cvalid[j] ? (uint32_t)sm.pix[j] * a.pitch_bytes : kInvalidCorner;
            strip[p.u * kChunkStride + (p.sn & (kChunk - 1))] = off;
        }
        // the sample's pair records (upper and lower corners)
        bool have[2], keep[2];
        int32_t key[2];
        float wa[2], wb[2];
        pair_records(sm, aw[k], p.active && L.w >= 0, have, key, wa, wb);
        merge_pair_records_in_quad<true>(have, key, wa, wb, keep);
#pragma unroll
        for (int r = 0; r < 2; ++r) {
            const uint32_t in_level = (uint32_t)(key[r] - L.z);
            rec[k][r].tile = keep[r] ? L.w + (int32_t)(in_level >> a.tile_px_log2) : -1;
            rec[k][r].x = (in_level & ((1u << a.tile_px_log2) - 1u)) | ((uint32_t)p.q << a.tile_px_log2);
            rec[k][r].wa = wa[r];
            rec[k][r].wb = wb[r];
            // (formed here: their two dozen terms would otherwise be kept until they are stored)
            asm volatile("" : "+v"(rec[k][r].tile), "+v"(rec[k][r].x), "+v"(rec[k][r].wa), "+v"(rec[k][r].wb));
            if (keep[r]) rec[k][r].at = atomicAdd(&cursor[rec[k][r].tile], 1);
        }
        // (one sample after the other: side by side they take twice the registers)
        __builtin_amdgcn_sched_barrier(0);
    }
    __syncthreads();  // the counts are whole
    const int64_t wg_row = ((int64_t)wk.b * a.nh + wk.h) * a.nwg + wk.q_begin / a.plan.tile_q;
    uint32_t* tbl = a.tbl + wg_row * a.tbl_stride;
    int32_t starts = 0, total;
    if (a.tbl_stride <= kWave) {
        const int32_t v = lane < a.tbl_stride ? cursor[lane] : 0;
        int32_t inc = v;
        for (int d = 1; d < a.tbl_stride; d <<= 1) {
            const int32_t o = __shfl_up(inc, d, kWave);
            if (lane >= d) inc += o;
        }
        starts = inc - v;
        total = __builtin_amdgcn_readlane(inc, a.tbl_stride - 1);  // (the entry behind the last tile counts nothing)
        if (wave == 0 && lane < a.tbl_stride) tbl[lane] = (uint32_t)starts;
    } else {
        if (wave == 0)
            scan_counters(cursor, a.tbl_stride, lane, [&](int i, int32_t start) {
                cursor[i] = start;
                tbl[i] = (uint32_t)start;
            });
        __syncthreads();
        total = cursor[a.tbl_stride - 1];  // (no record has this number: the entry behind the last tile holds the sum)
    }
#pragma unroll
    for (int k = 0; k < KS; ++k)
#pragma unroll
        for (int r = 0; r < 2; ++r) {
            const int32_t tile = rec[k][r].tile;
            const int32_t first = a.tbl_stride <= kWave ? __builtin_amdgcn_ds_bpermute(tile * 4, starts) : tile >= 0 ? cursor[tile] : 0;
            if (tile >= 0) {
                u32_alias* d = recs + (first + rec[k][r].at) * kRecDwords;
                d[0] = rec[k][r].x;
                d[1] = __builtin_bit_cast(uint32_t, rec[k][r].wa);
                d[2] = __builtin_bit_cast(uint32_t, rec[k][r].wb);
            }
        }
    __syncthreads();  // the records are whole (and nobody reads the counters any more)
    {
        const __amdgpu_buffer_rsrc_t sres = make_rsrc(a.rec + wg_row * a.rec_cap * kRecDwords, (uint32_t)a.rec_cap * (kRecDwords * 4u));
        store_slab(recs, kRecDwords * total, sres, tid, kThreads);
    }
    if (OVER || eight) __syncthreads();  // the slab is on its way
    if constexpr (OVER) {
#pragma unroll
        for (int k = 0; k < KS; ++k) {
            const Place p = place(k);
            if (lane + k * kWave >= entries) break;
            const uint32_t o = (uint32_t)(held[k] >> 4) * a.pitch_bytes, down = (uint32_t)lvl[level_of(p)].y * a.pitch_bytes;
            strip[p.u * kChunkStride + (p.sn & (kChunk - 1))] =
                u32x4{held[k] & 1 ? o : kInvalidCorner, held[k] & 2 ? o + a.pitch_bytes : kInvalidCorner, held[k] & 4 ? o + down : kInvalidCorner,
                      held[k] & 8 ? o + down + a.pitch_bytes : kInvalidCorner};
        }
    }
    if (q0 >= wk.q_end) return;  // (a wavefront without queries)

    // ---- gather and dots: the rows of the next sample are requested before the dots of the one at hand are formed ------------
    if constexpr (!FUSED) unpack_grad();
    {
        const __amdgpu_buffer_rsrc_t vres =
            make_rsrc(static_cast<const char*>(a.value) + (size_t)wk.b * a.batch_bytes, a.batch_bytes);
        const uint32_t choff = (uint32_t)(wk.h * a.hd + start) * (uint32_t)sizeof(T);
        auto request = [&](const u32x4* at, raw_t (&raw)[4]) {
            const u32x4 off = *at;
#pragma unroll
            for (int k = 0; k < 4; ++k) raw[k] = RowIO<T, VEC>::load_raw(vres, off[k] + choff);
        };
        auto consume = [&](u32x4* at, const raw_t (&raw)[4]) {
            float d[4];
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                float dk = 0.0f;
                if constexpr (kDot2) {
                    uint32_t words[kPairs];
                    __builtin_memcpy(words, &raw[k], sizeof(words));
                    // (4 lanes: the sums of 8 lanes of 8 bytes, in their order, where pieces of 16 bytes divide the row)
                    constexpr int kPart = LPR == 4 ? kPairs / 2 : kPairs;
#pragma unroll
                    for (int e = 0; e < kPart; ++e) dk = dot2_acc<T>(words[e], gpk[e], dk);
                    if constexpr (LPR == 4) {
                        float more = 0.0f;
#pragma unroll
                        for (int e = kPart; e < kPairs; ++e) more = dot2_acc<T>(words[e], gpk[e], more);
                        dk += more;
                    }
                } else {
                    float v[VEC];
                    RowIO<T, VEC>::unpack(raw[k], v);
                    constexpr int kPart = LPR == 4 ? VEC / 2 : VEC;
#pragma unroll
                    for (int e = 0; e < kPart; ++e) dk = __builtin_fmaf(v[e], gv[e], dk);
                    if constexpr (LPR == 4) {
                        float more = 0.0f;
#pragma unroll
                        for (int e = kPart; e < VEC; ++e) more = __builtin_fmaf(v[e], gv[e], more);
                        dk += more;
                    }
                }
                d[k] = group_sum<LG>(dk);
                asm volatile("" : "+v"(d[k]));  // (the last addition would otherwise become two instructions under the condition below)
            }
            if (c == 0) *at = __builtin_bit_cast(u32x4, f32x4{d[0], d[1], d[2], d[3]});
        };
        raw_t ra[4], rb[4];
        // Eight points and more per level: a trip takes eight of a unit side by side (rows of 4 lanes: of two units, and unit after unit before
        // the next eight; rows of 8 lanes: a unit's other eight next).  They touch the same rows on the coarse levels, which have left
        // the L1 when a sample of every unit at a time comes to the unit's next point.  This kernel at 2 x 12000 queries in no order, 8
        // heads of 32 channels, 4 levels x 8 points: float16 128 -> 104 us, float32 168 -> 148; at 2 x 19947 in the raster order of the maps, where
        // neighbouring queries' points are close to each other: 191 -> 190 and 284 -> 268; 6 x 9675 queries over four levels, float16,
        // 360 -> 317.  Fewer points per level gain where there is no order and mostly lose in raster order (of the
        // time before, in no order / in raster order): seven 0.87 / 1.03 in float16, 0.92 / 0.98 in float32, six 0.92 / 1.02 and 0.94 / 0.99, five
        // 0.95 / 1.02 and 0.96 / 1.03, four in float16 0.90 / 1.05: they stay as they were.  So do rows of 8 lanes with one unit per query
        // (four points in float32, raster order: 150 -> 158 us).
        if (eight) {
            // Units of 16 samples (or of 8): the trip's part of their rows of grad_out comes from LDS.
            constexpr int kWords = kDot2 ? kPairs : VEC;
#pragma unroll
            for (int e = 0; e < kWords; ++e) {
                if constexpr (kDot2) grads[lane * kWords + e] = gpk[e];
                else grads[lane * kWords + e] = __builtin_bit_cast(uint32_t, gv[e]);
            }
            wave_lds_sync();
            __builtin_amdgcn_s_setprio(0);
            const int ns = UPQ == 2 ? kChunk : a.S;  // trips
            u32x4* at = strip + (g >> 3) * kChunkStride + (g & 7);
            const u32_alias* my_grads = grads + ((g >> 3) * LPR + c) * kWords;
            auto unit_of = [&](int t) { return LPR == 8 ? t >> 1 : (t & 7) * 2; };  // (the first one)
            auto place_of = [&](int t) { return at + unit_of(t) * kChunkStride + (LPR == 8 ? t & 1 : t >> 3) * 8; };
            auto take_grad = [&](int t) {
                const u32_alias* from = my_grads + unit_of(t) * LPR * kWords;
#pragma unroll
                for (int e = 0; e < kWords; ++e) {
                    if constexpr (kDot2) gpk[e] = from[e];
                    else gv[e] = __builtin_bit_cast(float, (uint32_t)from[e]);
                }
            };
            request(place_of(0), ra);
            request(place_of(1), rb);
            for (int t = 0; t < ns - 2; t += 2) {
                take_grad(t);
                consume(place_of(t), ra);
                request(place_of(t + 2), ra);
                take_grad(t + 1);
                consume(place_of(t + 1), rb);
                request(place_of(t + 3), rb);
            }
            take_grad(ns - 2);
            consume(place_of(ns - 2), ra);
            take_grad(ns - 1);
            consume(place_of(ns - 1), rb);
        } else {
            wave_lds_sync();
            __builtin_amdgcn_s_setprio(0);
            // Nothing in the loop is conditional: behind a branch around a request the compiler can only wait for every request there
            // is, also for those of the samples ahead.  (An odd number of samples is made even: places without a sample hold offsets
            // that read as zeros.)
            const int ns = a.S < kChunk ? (a.S + 1) & ~1 : kChunk;
            request(mine, ra);
            request(mine + 1, rb);
            for (int t = 0; t < ns - 2; t += 2) {
                consume(mine + t, ra);
                request(mine + t + 2, ra);
                consume(mine + t + 1, rb);
                request(mine + t + 3, rb);
            }
            consume(mine + ns - 2, ra);
            consume(mine + ns - 1, rb);
        }
        __builtin_amdgcn_s_setprio(2);
        wave_lds_sync();
    }

    // ---- grad_attn / grad_loc from the reduced dots, one sample per lane -----------------------------------------------------
#pragma unroll
    for (int k = 0; k < KS; ++k) {
        const Place p = place(k);
        if (!p.active) continue;
        const f32x4 dd = __builtin_bit_cast(f32x4, strip[p.u * kChunkStride + (p.sn & (kChunk - 1))]);
        const int l = level_of(p);
        const i32x4 L = lvl[l];
        const float Wf = (float)L.y, Hf = (float)L.x;
        float ga = 0.f, gx = 0.f, gy = 0.f;
        if (valid[k]) sample_gradients(lw[k], lh[k], Wf, Hf, aw[k], dd, ga, gx, gy);
        T* la = gattn + e0;
        T* ll = gloc + 2 * e0;
        if constexpr (FUSED) {
            const T* off = static_cast<const T*>(a.loc) + 2 * e0;
            la[p.e] = from_f32<T>(aw[k] * (ga - stats[4 * p.u + 2]));
            const f32x4 gr = offset_gradient(a, ref + ((bq + p.q) * a.nl + l) * a.ref_dim, Wf, Hf, gx, gy, ll + 2 * p.e,
                                             [&](int j) { return to_f32(off[2 * p.e + j]); });
            if (a.grad_ref != nullptr) {
                if (a.np_pow2) store_reference_sum(a, reference_part(a, wk.b, wk.h, p.q, l), p.sn, gr);
                else strip[p.u * kChunkStride + p.sn] = __builtin_bit_cast(u32x4, gr);  // (any other number of points: summed below, from the place of the dots)
            }
        } else {
            // (streamed out like the records)
            __builtin_nontemporal_store(from_f32<T>(ga), la + p.e);
            __builtin_nontemporal_store(from_f32<T>(gx), ll + 2 * p.e);
            __builtin_nontemporal_store(from_f32<T>(gy), ll + 2 * p.e + 1);
        }
    }

    if constexpr (FUSED) {
        if (a.grad_ref != nullptr && !a.np_pow2) {
            wave_lds_sync();
            for (int i = lane; i < U * a.nl; i += kWave) {
                const int u = i / a.nl, l = i - u * a.nl, q = q0 + u;
                if (q >= wk.q_end) continue;
                f32x4 sum = {0.f, 0.f, 0.f, 0.f};
                for (int t = 0; t < a.np; ++t) sum += __builtin_bit_cast(f32x4, strip[u * kChunkStride + l * a.np + t]);
                float* part = reference_part(a, wk.b, wk.h, q, l);
                part[0] = sum[0];
                part[1] = sum[1];
                if (a.ref_dim == 4) {
                    part[2] = sum[2];
                    part[3] = sum[3];
                }
            }
        }
    }

    zero_extra_slots<T>(a, wk.b, wk.h, q0, wk.q_end, U >> SP, lane, gattn, gloc);
}

}  // namespace mxd
