// Deformable aggregation for gfx950 (MI355X), wave64: forward and backward.
//
//   out[b,a,c] = sum over (point p, camera, scale) of w[b,a,p,camera,scale,group(c)] * bilinear(feat of (camera, scale), loc[b,a,p,camera])
//
// (reference: mx_driving/ops/npu_deformable_aggregation.py:10-88, kernels/deformable_aggregation/.)  A location counts only
// strictly inside (0, 1) x (0, 1), and an anchor projects into one or two of the cameras: most samples of the sum do not exist.
//
// What bounds it: the feature maps of a training step (552 MB for 6 x 6 cameras of 256 x 704 pixels, 256 channels) fit no
// cache, every row that is touched has to come from HBM once and should not come twice, and an anchor's few hundred samples
// are one long chain when a unit of lanes works through them alone (one unit per anchor and group: forward 395 us at that
// size, 140 us for one frame in float16, which leaves half of the CUs without a workgroup).  Here
//
//   * a WAVEFRONT owns an (anchor, group): its lanes look at 64 locations at a time, keep those inside the image (ballot),
//     compute one sample per lane and then gather, 64 / lanes-per-row samples side by side, so that the chain is an eighth as
//     long, absent samples cost a lane of one test, and 256 CUs are filled from 900 anchors on;
//   * groups are pinned to XCDs (msda_plan.h) and the locations are taken camera by camera: the wavefronts of an XCD, which
//     run side by side through the anchors of one batch element, then share the (camera, group) slice of the maps they are
//     in -- 1.9 MB, of 4 MB of L2;
//   * the gradient of the maps is gathered, not scattered: a sort by pixel of the samples' upper and lower corner pairs (LDS
//     counters, one workgroup per (batch, level)), then every pixel row is formed once, by lanes that own its channels, from
//     the grad_out rows of its records -- those of a batch element stay in L2 -- and stored once, whole.
//
// Measured (6 x 900 anchors x 13 points, 6 cameras x 4 scales, 256 channels in 8 groups, float32), one unit of lanes per anchor and
// group and the tile pass -> these: forward 395 -> 237 us (float16, one batch element 140 -> 25), forward and backward 1969 -> 820
// with the dots formed by the anchors' wavefronts -- 318 us with the sort beside them, the gradient of the maps 221, the caller's
// layouts 40 -- and 670 with the dots formed beside the maps' gradient: sort 43, rows and dots 351, layouts 51 (kernel times one at
// a time; rows that the L2 does not hold bound all but the sort and the layouts: with six cameras that name the same maps the forward
// takes 131 us).
#include "dagg.h"

namespace mxd {

namespace {

__device__ inline i32x4 dagg_level(const DaggArgs& a, int l)
{
    const int sh = a.meta_i64;
    return i32x4{a.shapes[(2 * l) << sh], a.shapes[(2 * l + 1) << sh], a.lsi[l << sh], 0};
}

__device__ inline bool inside(float x, float y) { return x > 0.0f && x < 1.0f && y > 0.0f && y < 1.0f; }  // (false for NaN)

template <typename T>
__device__ inline f32x2 load_xy(const void* loc, int64_t i)
{
    const T* p = static_cast<const T*>(loc) + 2 * i;
    return f32x2{to_f32(p[0]), to_f32(p[1])};
}

// A location inside the image: {x, y, position in camera-major order << 16 | position in memory order, camera}.
typedef u32x4 Found;

// Per-wavefront LDS of the sampling kernels, in this order: found locations, the staged samples' row offsets, and then the
// forward's corner weights and group weights or the backward's dots and location gradients.
constexpr int kFoundBytes = kDaggList * 16, kOffBytes = kWave * 16;

// Keeps the locations of anchor (b, q) from number `first` on, in camera-major order, that lie inside the image; returns
// how many (at most kDaggList looked at).
template <typename T>
__device__ inline int find_locations(const DaggArgs& a, int64_t anchor, int first, Found* found, int lane)
{
    int n = 0;
#pragma unroll
    for (int k = 0; k < kDaggList / kWave; ++k) {
        const int j = first + k * kWave + lane;
        bool ok = j < a.nloc;
        uint32_t cam = 0;
        int li = 0;
        f32x2 xy = {0.f, 0.f};
        if (ok) {
            cam = ((uint32_t)j * a.p_magic) >> 20;
            li = (j - (int)cam * a.P) * a.cams + (int)cam;
            xy = load_xy<T>(a.loc, anchor * a.nloc + li);
            ok = inside(xy.x, xy.y);
        }
        const uint64_t mask = __ballot(ok);
        if (ok) {
            const int pos = n + (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0));
            const float fx = xy.x, fy = xy.y;
            found[pos] = Found{__builtin_bit_cast(uint32_t, fx), __builtin_bit_cast(uint32_t, fy), ((uint32_t)j << 16) | (uint32_t)li, cam};
        }
        n += __builtin_popcountll(mask);
    }
    return n;
}

// A group of samples is staged location by location (lane t: scale t % scales of its location t / scales, so that the weights of a
// location's scales are read side by side) and gathered scale by scale: the place in LDS of the sample that a lane stages.
// (Neighbouring lane groups then gather from the same map at a time, where an anchor's points are close to each other: 6 x 900 anchors in
// float32, forward, 272 us with the scales of a location side by side, 235 like this.  With lanes standing for the samples in the
// order of the gather small calls lose 2 to 5 %: 6 x 296 anchors, 8 groups of 4 channels in float16 11.1 -> 11.6.)
__device__ inline int sample_place(int lane, bool act, int locs, int scale, int loc) { return act ? scale * locs + loc : lane; }

// ---- forward -------------------------------------------------------------------------------------------------------------
// ONE: a row piece is the channels of one group (its weight is multiplied into the corner weights once); otherwise 128
// bytes of several groups' channels, whose weights wait in LDS.
template <typename T, int VEC, bool ONE>
__global__ __launch_bounds__(kDaggWaves * kWave) void dagg_fwd_kernel(const DaggArgs a)
{
    extern __shared__ __align__(16) unsigned char smem[];
    __shared__ i32x4 lvl[kMaxLevels];
    Work wk;
    if (!decode_block(a.map, blockIdx.x, a.bs, a.pieces, a.A, &wk)) return;
    if ((int)threadIdx.x < a.nl) lvl[threadIdx.x] = dagg_level(a, threadIdx.x);
    __syncthreads();
    const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x >> 6;
    const int q = wk.q_begin + wave;
    if (q >= wk.q_end) return;
    const int64_t anchor = (int64_t)wk.b * a.A + q;

    const int per_wave = kFoundBytes + kOffBytes + kWave * 16 + (ONE ? 0 : kWave * a.piece_heads * 4);
    unsigned char* mine = smem + wave * per_wave;
    Found* found = reinterpret_cast<Found*>(mine);
    u32x4* off = reinterpret_cast<u32x4*>(mine + kFoundBytes);
    f32x4* wts = reinterpret_cast<f32x4*>(mine + kFoundBytes + kOffBytes);
    float* gws = reinterpret_cast<float*>(mine + kFoundBytes + kOffBytes + kWave * 16);

    const int U = kWave >> a.lpr_log2, u = lane >> a.lpr_log2, c = lane & ((1 << a.lpr_log2) - 1);
    const int ch0 = wk.h * a.piece_ch, nch = a.C - ch0 < a.piece_ch ? a.C - ch0 : a.piece_ch;
    const bool chan_ok = c * VEC < nch;
    const int ch = ch0 + (chan_ok ? piece_start<VEC>(c * VEC, nch) : 0);
    const uint32_t choff = (uint32_t)ch * (uint32_t)sizeof(T);
    const int h0 = ch0 / a.hd, heads = ONE ? 1 : (ch0 + nch - 1) / a.hd - h0 + 1, my_head = ONE ? 0 : ch / a.hd - h0;
    const T* w = static_cast<const T*>(a.w) + anchor * a.nloc * a.scales * a.G + h0;
    const __amdgpu_buffer_rsrc_t vres =
        make_rsrc(static_cast<const char*>(a.feat) + (size_t)wk.b * a.batch_bytes, a.batch_bytes);

    const int step = (int)(((uint32_t)kWave * a.sc_magic) >> 20);  // locations per group of samples
    const int tl = (int)(((uint32_t)lane * a.sc_magic) >> 20), ts = lane - tl * a.scales;

    float acc[VEC];
#pragma unroll
    for (int e = 0; e < VEC; ++e) acc[e] = 0.0f;
    for (int first = 0; first < a.nloc; first += kDaggList) {
        const int n = find_locations<T>(a, anchor, first, found, lane);
        wave_lds_sync();
        for (int v0 = 0; v0 < n; v0 += step) {
            const int locs = n - v0 < step ? n - v0 : step;
            const bool act = tl < locs;
            const int place = sample_place(lane, act, locs, ts, tl);
            const Found f = found[act ? v0 + tl : 0];
            const uint32_t fx = f.x, fy = f.y, fj = f.z, fc = f.w;
            const Sample sm = sample_geometry(__builtin_bit_cast(float, fx), __builtin_bit_cast(float, fy), lvl[act ? (int)fc * a.scales + ts : 0],
                                              a.nf, act);
            u32x4 o;
            f32x4 cw;
            const T* gw = w + (int64_t)((int)(fj & 0xFFFFu) * a.scales + ts) * a.G;
            float aw = 1.0f;
            if constexpr (ONE) aw = act ? to_f32(*gw) : 0.0f;
            else
                for (int k = 0; k < heads; ++k) gws[place * a.piece_heads + k] = act ? to_f32(gw[k]) : 0.0f;
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                o[k] = sm.cvalid[k] ? (uint32_t)sm.pix[k] * a.pitch_bytes : kInvalidCorner;
                cw[k] = sm.valid ? sm.w[k] * aw : 0.0f;
            }
            off[place] = o;
            wts[place] = cw;
            wave_lds_sync();
            const int trips = (locs * a.scales + U - 1) >> (6 - a.lpr_log2);  // (uniform; samples that do not exist read zeros)
#pragma unroll 2
            for (int t = 0; t < trips; ++t) {
                const int s = t * U + u;
                const u32x4 ro = off[s];
                const f32x4 rw = wts[s];
                typename RowIO<T, VEC>::raw_t raw[4];
#pragma unroll
                for (int k = 0; k < 4; ++k) raw[k] = RowIO<T, VEC>::load_raw(vres, ro[k] + choff);
                const float g = ONE ? 1.0f : gws[s * a.piece_heads + my_head];
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    float v[VEC];
                    RowIO<T, VEC>::unpack(raw[k], v);
                    const float wk4 = ONE ? rw[k] : rw[k] * g;
#pragma unroll
                    for (int e = 0; e < VEC; ++e) acc[e] = __builtin_fmaf(wk4, v[e], acc[e]);
                }
            }
            wave_lds_sync();
        }
    }
    // the samples were dealt to U groups of lanes: add them up, the first group stores
    for (int d = 1 << a.lpr_log2; d < kWave; d <<= 1)
#pragma unroll
        for (int e = 0; e < VEC; ++e) acc[e] += __shfl_xor(acc[e], d, kWave);
    if (u == 0 && chan_ok) RowIO<T, VEC>::store_global(static_cast<T*>(a.out) + anchor * a.C + ch, acc);
}

// ---- backward, first kernel: gradients of the weights and locations, per group ---------------------------------------------
// LDS per wavefront: found locations, row offsets, dots, location gradients
constexpr int kDotsLds = kFoundBytes + kOffBytes + kWave * 16 + kWave * 8;

template <typename T, int VEC>
__device__ inline void dagg_dots(const DaggArgs& a, uint32_t block, unsigned char* smem, i32x4* lvl)
{
    Work wk;
    if (!decode_block(a.map, block, a.bs, a.pieces, a.A, &wk)) return;
    if ((int)threadIdx.x < a.nl) lvl[threadIdx.x] = dagg_level(a, threadIdx.x);
    __syncthreads();
    const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x >> 6;
    const int q = wk.q_begin + wave;
    if (q >= wk.q_end) return;
    const int64_t anchor = (int64_t)wk.b * a.A + q;

    unsigned char* mine = smem + wave * kDotsLds;
    Found* found = reinterpret_cast<Found*>(mine);
    u32x4* off = reinterpret_cast<u32x4*>(mine + kFoundBytes);
    f32x4* dots = reinterpret_cast<f32x4*>(mine + kFoundBytes + kOffBytes);
    f32x2* gxy = reinterpret_cast<f32x2*>(mine + kFoundBytes + kOffBytes + kWave * 16);

    const int U = kWave >> a.lpr_log2, u = lane >> a.lpr_log2, c = lane & ((1 << a.lpr_log2) - 1);
    const bool chan_ok = c * VEC < a.hd;
    const int start = chan_ok ? piece_start<VEC>(c * VEC, a.hd) : 0;
    const uint32_t choff = (uint32_t)(wk.h * a.hd + start) * (uint32_t)sizeof(T);
    const __amdgpu_buffer_rsrc_t vres =
        make_rsrc(static_cast<const char*>(a.feat) + (size_t)wk.b * a.batch_bytes, a.batch_bytes);
    const T* w = static_cast<const T*>(a.w) + anchor * a.nloc * a.scales * a.G + wk.h;
    const int64_t part = (int64_t)wk.h * a.bs * a.A + anchor;
    float* gw = a.gw_part + part * a.nloc * a.scales;
    f32x2* gl = reinterpret_cast<f32x2*>(a.gl_part) + part * a.nloc;

    // the anchor's grad_out row, in every group of lanes (16-bit rows as pairs for v_dot2)
    constexpr bool kDot2 = sizeof(T) == 2 && VEC % 2 == 0;
    constexpr int kPairs = kDot2 ? VEC / 2 : 1;
    float gv[VEC];
    uint32_t gpk[kPairs];
#pragma unroll
    for (int e = 0; e < VEC; ++e) gv[e] = 0.0f;
    if (chan_ok) {
        RowIO<T, VEC>::load_global(static_cast<const T*>(a.grad_out) + anchor * a.C + wk.h * a.hd + start, gv);
#pragma unroll
        for (int e = 0; e < VEC - 1; ++e)
            if (start + e < c * VEC) gv[e] = 0.0f;  // (counted by the piece before it)
    }
    if constexpr (kDot2) {
        typedef T t2 __attribute__((ext_vector_type(2)));
#pragma unroll
        for (int e = 0; e < kPairs; ++e) gpk[e] = __builtin_bit_cast(uint32_t, t2{from_f32<T>(gv[2 * e]), from_f32<T>(gv[2 * e + 1])});
    }

    const int step = (int)(((uint32_t)kWave * a.sc_magic) >> 20);
    const int tl = (int)(((uint32_t)lane * a.sc_magic) >> 20), ts = lane - tl * a.scales;
    for (int first = 0; first < a.nloc; first += kDaggList) {
        const int n = find_locations<T>(a, anchor, first, found, lane);
        wave_lds_sync();
        for (int v0 = 0; v0 < n; v0 += step) {
            const int locs = n - v0 < step ? n - v0 : step;
            const bool act = tl < locs;
            const int place = sample_place(lane, act, locs, ts, tl);
            const Found f = found[act ? v0 + tl : 0];
            const uint32_t fx = f.x, fy = f.y, fj = f.z, fc = f.w;
            const Sample sm = sample_geometry(__builtin_bit_cast(float, fx), __builtin_bit_cast(float, fy), lvl[act ? (int)fc * a.scales + ts : 0],
                                              a.nf, act);
            const float aw = act ? to_f32(w[(int64_t)((int)(fj & 0xFFFFu) * a.scales + ts) * a.G]) : 0.0f;
            u32x4 o;
#pragma unroll
            for (int k = 0; k < 4; ++k) o[k] = sm.cvalid[k] ? (uint32_t)sm.pix[k] * a.pitch_bytes : kInvalidCorner;
            off[place] = o;
            wave_lds_sync();
            const int trips = (locs * a.scales + U - 1) >> (6 - a.lpr_log2);
            auto gather = [&](auto lg) {
                constexpr int LG = decltype(lg)::value;
#pragma unroll 2
                for (int t = 0; t < trips; ++t) {
                    const int s = t * (kWave >> LG) + u;
                    const u32x4 ro = off[s];
                    typename RowIO<T, VEC>::raw_t raw[4];
#pragma unroll
                    for (int k = 0; k < 4; ++k) raw[k] = RowIO<T, VEC>::load_raw(vres, ro[k] + choff);
                    f32x4 d;
#pragma unroll
                    for (int k = 0; k < 4; ++k) {
                        float dk = 0.0f;
                        if constexpr (kDot2) {
                            uint32_t words[kPairs];
                            __builtin_memcpy(words, &raw[k], sizeof(words));
#pragma unroll
                            for (int e = 0; e < kPairs; ++e) dk = dot2_acc<T>(words[e], gpk[e], dk);
                        } else {
                            float v[VEC];
                            RowIO<T, VEC>::unpack(raw[k], v);
#pragma unroll
                            for (int e = 0; e < VEC; ++e) dk = __builtin_fmaf(v[e], gv[e], dk);
                        }
                        d[k] = group_sum<LG>(dk);
                    }
                    if (c == 0) dots[s] = d;
                }
            };
            switch (a.lpr_log2) {
                case 0: gather(std::integral_constant<int, 0>{}); break;
                case 1: gather(std::integral_constant<int, 1>{}); break;
                case 2: gather(std::integral_constant<int, 2>{}); break;
                case 3: gather(std::integral_constant<int, 3>{}); break;
                case 4: gather(std::integral_constant<int, 4>{}); break;
                case 5: gather(std::integral_constant<int, 5>{}); break;
                default: gather(std::integral_constant<int, 6>{}); break;
            }
            wave_lds_sync();
            f32x2 g = {0.f, 0.f};
            if (act) {
                float ga = 0.f;
                if (sm.valid) {
                    float gx, gy;
                    sample_gradients(sm.lw, sm.lh, sm.Wf, sm.Hf, aw, dots[place], ga, gx, gy);
                    g = f32x2{gx, gy};
                }
                gw[(int)(fj >> 16) * a.scales + ts] = ga;
            }
            gxy[lane] = g;
            wave_lds_sync();
            if (act && ts == 0) {
                // the scales of a location share it
                for (int k = 1; k < a.scales; ++k) g += gxy[lane + k];
                gl[fj >> 16] = g;
            }
            wave_lds_sync();
        }
    }
}

// ---- the levels as the kernels behind it see them ---------------------------------------------------------------------------
struct DaggLevels {
    int32_t H[kMaxLevels], W[kMaxLevels], base[kMaxLevels];
    int32_t px[kMaxLevels];      // pixels that the sort has records of, inside the feature tensor; 0: none (no rows, or one of `lost`)
    int32_t csr[kMaxLevels];     // its first entry of DaggArgs::csr
    int32_t chunks[kMaxLevels];  // parts its strips' records are split into
    int32_t first[kMaxLevels + 1];  // work items of the levels before it
    int32_t tiled;               // the levels tile the keys in order: a pixel row belongs to one level
    uint64_t lost;               // levels, by bit, with rows that no record stands for: dagg_levels_without_room

    // (a level per lane of the first wavefront: one after the other, 24 levels were 5 us in front of every workgroup)
    __device__ void fill(const DaggArgs& a)
    {
        static_assert(kMaxLevels <= kWave, "a lane per level");
        if (threadIdx.x < kWave) {
            const int lane = (int)threadIdx.x;
            const i32x4 L = lane < a.nl ? dagg_level(a, lane) : i32x4{0, 0, 0, 0};
            int32_t P;
            level_tile_count(L.x, L.y, L.z, a.nf, 0, &P);
            auto prefix = [&](int64_t v) {
                for (int d = 1; d < a.nl; d <<= 1) {
                    const int64_t o = __shfl_up(v, d, kWave);
                    if (lane >= d) v += o;
                }
                return v;
            };
            const int64_t p = (int64_t)L.x * L.y;
            const bool whole = L.x > 0 && L.y > 0 && p == P;
            const int32_t end = L.z + P, before = __shfl_up(end, 1, kWave);
            const bool follows = whole && L.z == (lane == 0 ? 0 : before);
            tiled = __ballot(lane < a.nl && !follows) == 0 && __builtin_amdgcn_readlane(end, a.nl - 1) == a.nf;
            // (levels without records: the ones that find no room in the table of record starts, where levels overlap far, and one
            //  that starts before the tensor and reaches into it, whose pixels are not numbered from its first row on)
            int64_t used = P > 0 ? P + 1 : 0, at = prefix(used) - used;
            bool fits = !(L.x > 0 && L.y > 0 && L.z < 0 && L.z + p > 0);
            if (__ballot(at + used > a.starts) != 0) {
                int64_t room = 0;
                for (int l = 0; l < a.nl; ++l) {
                    const int32_t u = __builtin_amdgcn_readlane((int32_t)used, l);
                    const bool room_left = room + u <= a.starts;
                    if (lane == l) {
                        at = room;
                        fits = fits && room_left;
                    }
                    if (room_left) room += u;
                }
                if (!fits) P = 0;
            }
            lost = __ballot(!fits);
            // records of a strip if every location were inside and spread evenly
            const float expect = P > 0 ? 2.0f * (float)a.A * (float)a.P * (float)(kDaggStrip + 1) / (float)P : 0.0f;
            int32_t n = (int32_t)__builtin_ceilf(expect / (float)a.strip_records);
            n = n < 1 ? 1 : n > 64 ? 64 : n;
            const int32_t items = (P + kDaggStrip - 1) / kDaggStrip * n, upto = (int32_t)prefix(items);
            if (lane < a.nl) {
                H[lane] = L.x;
                W[lane] = L.y;
                base[lane] = L.z;
                px[lane] = P;
                csr[lane] = (int32_t)at;
                chunks[lane] = n;
                first[lane] = upto - items;
                if (lane == a.nl - 1) first[a.nl] = upto;
            }
        }
        __syncthreads();
    }
    __device__ bool direct(int l) const { return tiled && chunks[l] == 1; }
};

// ---- sort of the corner pairs by pixel -------------------------------------------------------------------------------------
// One workgroup per (batch, level, range of kDaggSortPx pixels): counts the records of every pixel in LDS, turns the counts
// into starts, and drops every record at its place.
struct alignas(16) DaggSort {
    DaggLevels lv;
    uint32_t wsum[kDaggSortWaves];
    uint32_t before_s;
    uint32_t cnt[kDaggSortPx];
};
// What a wavefront keeps of the points that it has requested: those inside the image.
struct DaggInside {
    static constexpr int kRounds = 4;
    f32x2 xy[kRounds * kWave];
    uint16_t at[kRounds * kWave];  // request << 6 | lane
};
// COMPACT: the points inside the image side by side before their geometry is derived, or else a wavefront derives it for all 64
// wherever one is inside (6 x 900 anchors, a third of the points inside: 50 -> 43 us; the sort beside the dots, which cover it, does
// without the LDS for it).
template <typename T, int WAVES, bool COMPACT>
__device__ inline void dagg_sort(const DaggArgs& a, uint32_t block, unsigned char* smem)
{
    constexpr int kThreads = WAVES * kWave;
    DaggSort& sh = *reinterpret_cast<DaggSort*>(smem);
    DaggLevels& lv = sh.lv;
    uint32_t *cnt = sh.cnt, *wsum = sh.wsum, &before_s = sh.before_s;
    // first ranges first, scale by scale: the workgroups that have pixels are neighbours, and so spread over the XCDs (range by range of a
    // level, 22 apart, they met on four of them: the launch took 68 us with 6 x 900 anchors, 50 like this)
    const uint32_t maps = (uint32_t)a.bs * (uint32_t)a.cams, i = block % (maps * a.scales);
    const int range = (int)(block / (maps * a.scales)), b = (int)(i % a.bs), l = (int)(i % maps) / a.bs * a.scales + (int)(i / maps);
    const i32x4 own = dagg_level(a, l);
    if ((int64_t)own.x * own.y <= (int64_t)range * kDaggSortPx) return;  // (uniform)
    lv.fill(a);
    const int tid = threadIdx.x;
    const int r0 = range * kDaggSortPx, P = lv.px[l], r1 = P - r0 < kDaggSortPx ? P : r0 + kDaggSortPx;
    if (range >= a.sort_ranges || r0 >= P) return;  // (uniform; the launch has a multiple of 8 sort workgroups)
    for (int i = tid; i < kDaggSortPx; i += kThreads) cnt[i] = 0;
    if (tid == 0) before_s = 0;
    __syncthreads();

    const int cam = l / a.scales, sc = l - cam * a.scales;
    const i32x4 level = {lv.H[l], lv.W[l], lv.base[l], 0};
    const uint32_t points = (uint32_t)a.A * (uint32_t)a.P;
    // the records of a location on this level: (key, weights) of up to two
    auto each_record = [&](const f32x2 xy, auto take) {
        if (!inside(xy.x, xy.y)) return;
        const Sample sm = sample_geometry(xy.x, xy.y, level, a.nf, true);
#pragma unroll
        for (int r = 0; r < 2; ++r) {
            const bool vl = sm.cvalid[2 * r], vr = sm.cvalid[2 * r + 1];
            if (vl || vr)
                take(r, (vl ? sm.pix[2 * r] : sm.pix[2 * r + 1]) - level.z, vl ? sm.w[2 * r] : sm.w[2 * r + 1], vl && vr ? sm.w[2 * r + 1] : 0.0f);
        }
    };
    // eight points' locations are requested together: one at a time, the two passes are a chain of trips to memory
    constexpr int kTogether = 8;
    auto each_point = [&](auto take) {
        for (uint32_t i0 = tid; COMPACT ? (i0 & ~(uint32_t)(kWave - 1)) < points : i0 < points; i0 += kTogether * kThreads) {
            f32x2 xy[kTogether];
#pragma unroll
            for (int k = 0; k < kTogether; ++k) {
                const uint32_t i = i0 + k * kThreads;
                xy[k] = i < points ? load_xy<T>(a.loc, ((int64_t)b * points + i) * a.cams + cam) : f32x2{0.f, 0.f};
            }
            if constexpr (COMPACT) {
                DaggInside& list = reinterpret_cast<DaggInside*>(smem + sizeof(DaggSort))[tid >> 6];
                for (int half = 0; half < kTogether; half += DaggInside::kRounds) {
                    uint32_t n = 0;
#pragma unroll
                    for (int k = 0; k < DaggInside::kRounds; ++k) {
                        const f32x2 p = xy[k];
                        const bool in = inside(p.x, p.y);
                        const uint64_t mask = __ballot(in);
                        if (in) {
                            const uint32_t pos = n + __builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0));
                            list.xy[pos] = p;
                            list.at[pos] = (uint16_t)((half + k) << 6 | (tid & (kWave - 1)));
                        }
                        n += (uint32_t)__builtin_popcountll(mask);
                    }
#pragma unroll
                    for (int k = 0; k < DaggInside::kRounds; ++k) xy[k] = xy[k + DaggInside::kRounds];
                    wave_lds_sync();
                    for (uint32_t e = tid & (kWave - 1); e < n; e += kWave) {
                        const uint32_t at = list.at[e], i = i0 - (tid & (kWave - 1)) + (at >> 6) * kThreads + (at & (kWave - 1));
                        each_record(list.xy[e], [&](uint32_t r, int key, float wa, float wb) { take(i, r, key, wa, wb); });
                    }
                    wave_lds_sync();
                }
                continue;
            }
            for (int k = 0; k < kTogether; ++k) {
                each_record(xy[0], [&](uint32_t r, int key, float wa, float wb) { take(i0 + k * kThreads, r, key, wa, wb); });
#pragma unroll
                for (int m = 0; m + 1 < kTogether; ++m) xy[m] = xy[m + 1];
            }
        }
    };
    uint32_t before = 0;  // records of the ranges before this one
    each_point([&](uint32_t, uint32_t, int key, float, float) {
        if (key < r0) ++before;
        else if (key < r1) atomicAdd(&cnt[key - r0], 1u);
    });
    if (r0 > 0 && before != 0) atomicAdd(&before_s, before);
    __syncthreads();

    // exclusive prefix: neighbouring counters per thread, then over the threads
    constexpr int kPer = kDaggSortPx / kThreads;
    uint32_t sum = 0;
    for (int k = 0; k < kPer; ++k) sum += cnt[tid * kPer + k];
    uint32_t inc = sum;
    const int lane = tid & (kWave - 1), wave = tid >> 6;
#pragma unroll
    for (int d = 1; d < kWave; d <<= 1) {
        const uint32_t o = __shfl_up(inc, d, kWave);
        if (lane >= d) inc += o;
    }
    if (lane == kWave - 1) wsum[wave] = inc;
    __syncthreads();
    uint32_t at = before_s + inc - sum;
    for (int k = 0; k < wave; ++k) at += wsum[k];
    uint32_t* csr = a.csr + (size_t)b * (size_t)a.starts + lv.csr[l];
    for (int k = 0; k < kPer; ++k) {
        const int p = tid * kPer + k;
        const uint32_t v = cnt[p];
        cnt[p] = at;
        if (r0 + p < P) csr[r0 + p] = at;
        at += v;
        if (r0 + p == P - 1) csr[P] = at;
    }
    __syncthreads();

    u32x4* rec = a.rec + ((size_t)b * a.nl + l) * 2 * points;
    each_point([&](uint32_t i, uint32_t r, int key, float wa, float wb) {
        if (key < r0 || key >= r1) return;
        const uint32_t pos = atomicAdd(&cnt[key - r0], 1u);
        rec[pos] = u32x4{(i / (uint32_t)a.P) << 3 | ((uint32_t)key & 7u), r << 31 | ((i * (uint32_t)a.cams + (uint32_t)cam) * (uint32_t)a.scales + (uint32_t)sc),
                         __builtin_bit_cast(uint32_t, wa), __builtin_bit_cast(uint32_t, wb)};
    });
}

// Zeros for the rows of grad_feat's float32 image that the kernel behind it adds to: those of levels whose strips are split, or,
// where the levels do not tile the features (rows that several levels share or none has), all.  (By workgroups of their own: a level's
// rows zeroed by the workgroup that sorts it kept the launch 100 us longer with 512 channels.)
constexpr uint32_t kDaggZeroWgs = 128;
__device__ inline void dagg_zero(const DaggArgs& a, uint32_t block, unsigned char* smem)
{
    DaggLevels& lv = reinterpret_cast<DaggSort*>(smem)->lv;
    lv.fill(a);
    const uint32_t step = kDaggZeroWgs * blockDim.x;
    auto zero = [&](uint64_t lo, uint64_t hi) {
        if (((lo | hi) & 3) == 0 && (reinterpret_cast<uintptr_t>(a.image) & 15) == 0)
            for (uint64_t i = lo / 4 + block * blockDim.x + threadIdx.x; i < hi / 4; i += step) reinterpret_cast<f32x4*>(a.image)[i] = f32x4{0.f, 0.f, 0.f, 0.f};
        else
            for (uint64_t i = lo + block * blockDim.x + threadIdx.x; i < hi; i += step) a.image[i] = 0.0f;
    };
    if (!lv.tiled) {
        zero(0, (uint64_t)a.bs * a.nf * a.C);
        return;
    }
    for (int l = 0; l < a.nl; ++l)
        if (lv.chunks[l] > 1)
            for (int b = 0; b < a.bs; ++b) {
                const uint64_t lo = ((uint64_t)b * a.nf + lv.base[l]) * a.C;
                zero(lo, lo + (uint64_t)lv.px[l] * a.C);
            }
}

// The kernels side by side in one launch: the sort has work for a few workgroups, whose time the others' gathers cover
// (43 us as a launch of its own for 6 x 900 anchors).
template <typename T, int VEC>
__global__ __launch_bounds__(kDaggBackWaves * kWave) void dagg_dots_and_sort_kernel(const DaggArgs a, uint32_t sorts)
{
    extern __shared__ __align__(16) unsigned char smem[];
    __shared__ i32x4 lvl[kMaxLevels];
    if (blockIdx.x < sorts) dagg_sort<T, kDaggBackWaves, false>(a, blockIdx.x, smem);
    else if (blockIdx.x < sorts + kDaggZeroWgs) dagg_zero(a, blockIdx.x - sorts, smem);
    else dagg_dots<T, VEC>(a, blockIdx.x - sorts - kDaggZeroWgs, smem, lvl);
}

static_assert(sizeof(DaggSort) % 16 == 0 && sizeof(DaggInside) % 8 == 0);
constexpr size_t kDaggSortLds = sizeof(DaggSort) + kDaggSortWaves * sizeof(DaggInside);
static_assert(kDaggSortLds <= 64 * 1024, "what a launch may take without opting in");

// The same without dot products, where the kernel behind it forms them.
template <typename T>
__global__ __launch_bounds__(kDaggSortWaves * kWave) void dagg_sort_kernel(const DaggArgs a, uint32_t sorts)
{
    extern __shared__ __align__(16) unsigned char smem[];
    if (blockIdx.x < sorts) dagg_sort<T, kDaggSortWaves, true>(a, blockIdx.x, smem);
    else dagg_zero(a, blockIdx.x - sorts, smem);
}

// ---- gradient of the feature maps --------------------------------------------------------------------------------------------
// The samples of levels without records (DaggLevels::lost), added to grad_feat's float32 image by atomics, and their dots where the
// finish kernel takes those from DaggArgs::dots: a sample per wavefront, a channel per lane.  Only levels that overlap or start before
// the tensor come here, and then every row has been zeroed and every other level adds with atomics as well.  Slow, and there so that
// scale_start_index is honoured however it comes.
template <typename T>
__device__ inline void dagg_levels_without_room(const DaggArgs& a, const DaggLevels& lv)
{
    const T* gout = static_cast<const T*>(a.grad_out);
    const uint32_t lane = threadIdx.x & (kWave - 1), waves = gridDim.x * (blockDim.x / kWave);
    const uint64_t points = (uint64_t)a.A * (uint64_t)a.P, total = points * a.bs;
    for (uint64_t i = blockIdx.x * (blockDim.x / kWave) + threadIdx.x / kWave; i < total; i += waves) {
        const uint64_t b = i / points, anchor = i / (uint64_t)a.P;  // (anchor of all batch elements)
        for (uint64_t m = lv.lost; m != 0; m &= m - 1) {
            const int l = __builtin_ctzll(m), cam = l / a.scales;
            const uint64_t li = i * a.cams + cam;
            const f32x2 xy = load_xy<T>(a.loc, (int64_t)li);
            if (!inside(xy.x, xy.y)) continue;
            const Sample sm = sample_geometry(xy.x, xy.y, i32x4{lv.H[l], lv.W[l], lv.base[l], 0}, a.nf, true);
            const T* w = static_cast<const T*>(a.w) + (li * a.scales + (l - cam * a.scales)) * a.G;
            float* image = a.image + b * a.nf * a.C;
            if (a.dots != nullptr)
                for (int g = 0; g < a.G; ++g) {
                    float d[4] = {0.f, 0.f, 0.f, 0.f};
                    for (int ch = g * a.hd + (int)lane; ch < (g + 1) * a.hd; ch += kWave)
                        for (int k = 0; k < 4; ++k)
                            if (sm.cvalid[k]) d[k] += to_f32(static_cast<const T*>(a.feat)[(b * a.nf + sm.pix[k]) * a.C + ch]) * to_f32(gout[anchor * a.C + ch]);
                    for (int k = 0; k < 4; ++k) d[k] = group_sum<6>(d[k]);
                    if (lane == 0)
                        for (int r = 0; r < 2; ++r)
                            a.dots[((li * a.scales + (l - cam * a.scales)) * 2 + r) * a.G + g] = f32x2{sm.cvalid[2 * r] ? d[2 * r] : d[2 * r + 1], d[2 * r + 1]};
                }
            for (int ch = (int)lane; ch < a.C; ch += kWave) {
                const float g = to_f32(gout[anchor * a.C + ch]) * to_f32(w[ch / a.hd]);
                for (int k = 0; k < 4; ++k)
                    if (sm.cvalid[k]) unsafeAtomicAdd(image + (size_t)sm.pix[k] * a.C + ch, sm.w[k] * g);
            }
        }
    }
}

// A unit of 2^row_lpr_log2 lanes forms the rows of a strip of 8 neighbouring pixels, or of one block of their channels, from
// the strip's records in pixel order: one row of sums for the pixel at hand and one for the pixel to its right; the records
// of the pixel before the strip are met for their right halves.  Every row is stored once, whole (strips split by record
// number -- levels with few pixels -- add theirs with atomics to rows that the sort has zeroed).
// MIXED: a lane's channels may belong to several groups.
// WAVE: a unit is a wavefront -- what it reads of records and starts is the same for all lanes and comes through the scalar
// cache.
// DOTS: forms the samples' dot products with the value rows too.  A record stands for two neighbouring pixels, whose value rows are in
// registers while the strip is at the first of them; a strip's rows and the one behind them go to LDS with the first records'
// requests, so that no trip to memory is added, and a record's dots are stored by one lane per group, each taking another record of
// the batch.  Bound by memory (6 x 900 anchors, 256 channels: 348 us for 972 MB read and 635 written, 4.6 TB/s, nine tenths of a copy's rate,
// with 16 wavefronts per CU for their LDS and registers; 1.1 GB are rows in and out that it cannot do without).  Samples that are
// shared between strips have their dots from the strip of the first pixel.
template <typename T, int VEC, bool MIXED, bool WAVE, bool DOTS>
__global__ __launch_bounds__(256, DOTS ? 4 : 1) void dagg_gradf_kernel(const DaggArgs a)
{
    // (memory that this kernel does not write, as far as the compiler is concerned: uniform loads become scalar ones)
    typedef const __attribute__((address_space(4))) u32x4* rec_ptr;
    typedef const __attribute__((address_space(4))) uint32_t* csr_ptr;
    __shared__ DaggLevels lv;
    __shared__ float turn_all[WAVE && !DOTS ? 256 * VEC : 1];
    // per wavefront, the strip's value rows and the one behind them
    static_assert(!DOTS || (WAVE && !MIXED && VEC * sizeof(T) == 16 && sizeof(T) == 4));
    typedef typename RowIO<T, VEC>::held_t held_t;
    constexpr int kRows = kDaggStrip + 1;
    __shared__ __align__(16) held_t values_all[DOTS ? 256 * kRows : 1];
    lv.fill(a);
    [[maybe_unused]] float* turn = turn_all + (WAVE && !DOTS ? (threadIdx.x & ~63u) * VEC : 0u);
    [[maybe_unused]] held_t* values = values_all + (DOTS ? __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)) * kWave * kRows : 0);
    [[maybe_unused]] const int lane = threadIdx.x & (kWave - 1);
    auto scalar = [](int v) { return WAVE ? __builtin_amdgcn_readfirstlane(v) : v; };
    const int lpr = 1 << a.row_lpr_log2, units = 256 >> a.row_lpr_log2;
    const int c = threadIdx.x & (lpr - 1);
    const uint32_t per_b = (uint32_t)lv.first[a.nl] * (uint32_t)a.row_blocks;
    const uint64_t total = (uint64_t)per_b * a.bs;
    const T* gout = static_cast<const T*>(a.grad_out);
    const uint32_t points = (uint32_t)a.A * (uint32_t)a.P;
    const uint32_t per_anchor = (uint32_t)a.nloc * (uint32_t)a.scales;
    const uint32_t unit = threadIdx.x >> a.row_lpr_log2;
    for (uint64_t item = (uint64_t)blockIdx.x * units + (WAVE ? (uint32_t)__builtin_amdgcn_readfirstlane((int)unit) : unit); item < total; item += (uint64_t)gridDim.x * units) {
        const int b = (int)(item / per_b);
        const uint32_t r = (uint32_t)(item - (uint64_t)b * per_b);
        const int blk = (int)(r % (uint32_t)a.row_blocks);
        // (the coarse levels, whose strips have the most records, are numbered last and start first)
        const int it = lv.first[a.nl] - 1 - (int)(r / (uint32_t)a.row_blocks);
        int l = 0;
        for (int s = 32; s > 0; s >>= 1)
            if (l + s < a.nl && lv.first[l + s] <= it) l += s;
        l = scalar(l);
        const int k = scalar(it - lv.first[l]), chunks = scalar(lv.chunks[l]), strip = k / chunks, chunk = k - strip * chunks;
        const int p0 = strip * kDaggStrip, px_l = scalar(lv.px[l]), p1 = p0 + kDaggStrip < px_l ? p0 + kDaggStrip : px_l;
        const bool direct = lv.direct(l);
        const csr_ptr csr = (csr_ptr)(a.csr + (size_t)b * (size_t)a.starts + scalar(lv.csr[l]));
        const uint32_t s1 = csr[p0];
        uint32_t lo = p0 > 0 ? csr[p0 - 1] : s1, hi = csr[p1];
        if (chunks > 1) {
            const uint32_t s0 = lo, n = hi - lo;
            lo = s0 + (uint32_t)((uint64_t)n * chunk / chunks);
            hi = s0 + (uint32_t)((uint64_t)n * (chunk + 1) / chunks);
        }
        const int chn = (blk * lpr + c) * VEC;
        const bool chan_ok = chn < a.C;
        const int ch = chan_ok ? piece_start<VEC>(chn, a.C) : 0;
        const T* grow = gout + (size_t)b * a.A * a.C + ch;
        const T* w = static_cast<const T*>(a.w) + (size_t)b * a.A * per_anchor * a.G + ch / a.hd;
        const rec_ptr rec = (rec_ptr)(a.rec + ((size_t)b * a.nl + l) * 2 * points);

        float acc[VEC], nxt[VEC];
#pragma unroll
        for (int e = 0; e < VEC; ++e) acc[e] = nxt[e] = 0.0f;
        int cur = 0;         // pixel of the strip whose sums are in acc
        [[maybe_unused]] held_t here = {}, right = {};  // its value row, and its right neighbour's
        uint32_t nan_px = 0; // pixels of the strip whose sums hold NaN
        auto flush = [&]() { // its row is complete
            bool bad = false;
#pragma unroll
            for (int e = 0; e < VEC; ++e) bad |= acc[e] != acc[e];
            if (__ballot(bad) != 0) {
                if (bad) nan_px |= 1u << cur;
                // (added below; a row that is stored whole is stored again)
#pragma unroll
                for (int e = 0; e < VEC; ++e) acc[e] = bad ? 0.0f : acc[e];
            }
            const size_t row = ((size_t)b * a.nf + lv.base[l] + p0 + cur) * a.C + ch;
            if constexpr (DOTS) {
                // to where its value row was, and from there with the strip's others: stores between the records' loads would be
                // waited for with those, and the registers of their addresses kept (372 -> 344 us)
                __builtin_memcpy(&values[cur * kWave + lane], acc, sizeof(acc));
            } else if (direct) {
                if (chan_ok) RowIO<T, VEC>::store_global(static_cast<T*>(a.grad_feat) + row, acc);
            } else if constexpr (WAVE) {
                // through LDS, so that neighbouring lanes add to neighbouring channels: an addition is carried out per 64 bytes that
                // an instruction touches, and a lane's own channels are 4 VEC bytes from the next lane's (6 x 900 anchors,
                // 256 channels in float32: backward 628 -> 585 us; shorter rows, whose units diverge, lose by it)
                if (chan_ok) {
#pragma unroll
                    for (int e = 0; e < VEC; ++e)
                        if (ch + e >= chn) turn[ch + e - blk * kWave * VEC] = acc[e];
                }
                wave_lds_sync();
#pragma unroll
                for (int e = 0; e < VEC; ++e) {
                    const int i = blk * kWave * VEC + e * kWave + c;
                    const float v = i < a.C ? turn[e * kWave + c] : 0.0f;
                    if (v != 0.0f) unsafeAtomicAdd(a.image + row - ch + i, v);
                }
                wave_lds_sync();
            } else if (chan_ok) {
#pragma unroll
                for (int e = 0; e < VEC; ++e)
                    if (ch + e >= chn && acc[e] != 0.0f) unsafeAtomicAdd(a.image + row + e, acc[e]);
            }
#pragma unroll
            for (int e = 0; e < VEC; ++e) acc[e] = nxt[e], nxt[e] = 0.0f;
            ++cur;
            if constexpr (DOTS) {
                here = right;
                right = values[(cur + 1 < kRows ? cur + 1 : cur) * kWave + lane];
            }
        };
        // (records whose rows are in flight together; the records after them are requested with those rows, or else every
        //  batch would be two trips to memory one after the other)
        constexpr int kAhead = WAVE ? 6 : 4;  // (4, 6, 8, 12 with a wavefront per row: 250, 236, 237, 279 us)
        u32x4 next[kAhead];
        auto request = [&](uint32_t e0) {
#pragma unroll
            for (int j = 0; j < kAhead; ++j) next[j] = rec[e0 + j < hi ? e0 + j : hi - 1];
        };
        if constexpr (DOTS)
            if (lo < hi) {
                wave_lds_sync();
                __builtin_amdgcn_s_waitcnt(0xC07F);  // (lgkmcnt(0): the strip before has read its rows)
                const int32_t row0 = lv.base[l] + p0;
#pragma unroll
                for (int i = 0; i < kRows; ++i) {
                    // (a row behind the tensor's last is nobody's right half)
                    const int32_t row = row0 + i < a.nf ? row0 + i : a.nf - 1;
                    const T* from = static_cast<const T*>(a.feat) + ((size_t)b * a.nf + row) * a.C + ch;
                    __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)from,
                                                     (__attribute__((address_space(3))) void*)(values + i * kWave), 16, 0, 0);
                }
            }
        if (lo < hi) request(lo);
        for (uint32_t e0 = lo; e0 < hi; e0 += kAhead) {
            u32x4 rc[kAhead];
            typename RowIO<T, VEC>::held_t row[kAhead];
            float aw[kAhead][MIXED ? VEC : 1];
#pragma unroll
            for (int j = 0; j < kAhead; ++j) rc[j] = next[j];
#pragma unroll
            for (int j = 0; j < kAhead; ++j) {
                row[j] = RowIO<T, VEC>::load_held(grow + (size_t)(rc[j].x >> 3) * a.C);
                const T* wj = w + (size_t)(rc[j].y & 0x7FFFFFFFu) * a.G;
                if constexpr (MIXED) {
#pragma unroll
                    for (int e = 0; e < VEC; ++e) aw[j][e] = to_f32(wj[(ch + e) / a.hd - ch / a.hd]);
                } else {
                    aw[j][0] = to_f32(*wj);
                }
            }
            if (e0 + kAhead < hi) request(e0 + kAhead);
            [[maybe_unused]] float d0[kAhead], d1[kAhead];
            if constexpr (DOTS) {
                if (e0 == lo) {
                    __builtin_amdgcn_s_waitcnt(0x0F70);  // (vmcnt(0): the value rows are there)
                    wave_lds_sync();
                    here = values[lane];
                    right = values[kWave + lane];
                }
#pragma unroll
                for (int j = 0; j < kAhead; ++j) d0[j] = d1[j] = 0.0f;
            }
#pragma unroll
            for (int j = 0; j < kAhead; ++j) {
                if (e0 + j >= hi) break;
                const uint32_t za = rc[j].z, zb = rc[j].w;
                float wa = __builtin_bit_cast(float, za), wb = __builtin_bit_cast(float, zb);
                if (e0 + j < s1) {  // a pair that starts on the pixel before the strip
                    wa = wb;
                    wb = 0.0f;
                } else {
                    const int px = (int)(rc[j].x & 7u);
                    while (cur < px) flush();
                }
                float g[VEC];
                RowIO<T, VEC>::unpack_held(row[j], g);
#pragma unroll
                for (int e = 0; e < VEC; ++e) {
                    const float gw = g[e] * aw[j][MIXED ? e : 0];
                    acc[e] = __builtin_fmaf(wa, gw, acc[e]);
                    nxt[e] = __builtin_fmaf(wb, gw, nxt[e]);
                }
                if constexpr (DOTS) {
#pragma unroll
                    for (int e = 0; e < VEC; ++e) {
                        d0[j] = __builtin_fmaf(here[e], g[e], d0[j]);
                        d1[j] = __builtin_fmaf(right[e], g[e], d1[j]);
                    }
                }
            }
            if constexpr (DOTS) {
                // over the lanes of a group, which then store a record's each (with the sample's other group's and row's: 64 bytes of 8 groups)
                auto over = [&](auto lanes, auto sum) {
                    if (a.lpr_log2 >= decltype(lanes)::value) {
#pragma unroll
                        for (int j = 0; j < kAhead; ++j) d0[j] += sum(d0[j]), d1[j] += sum(d1[j]);
                    }
                };
                over(std::integral_constant<int, 1>{}, [](float v) { return dpp_xchg<0xB1>(v); });
                over(std::integral_constant<int, 2>{}, [](float v) { return dpp_xchg<0x4E>(v); });
                over(std::integral_constant<int, 3>{}, [](float v) { return dpp_xchg<0x141>(v); });
                over(std::integral_constant<int, 4>{}, [](float v) { return dpp_xchg<0x140>(v); });
                over(std::integral_constant<int, 5>{}, [](float v) { return __shfl_xor(v, 16, 64); });
                over(std::integral_constant<int, 6>{}, [](float v) { return __shfl_xor(v, 32, 64); });
                f32x2* dots = a.dots + (size_t)b * a.A * per_anchor * 2 * a.G + ((blk * kWave + c) >> a.lpr_log2);
                const int lanes = 1 << a.lpr_log2;
                for (int j0 = 0; j0 < kAhead; j0 += lanes) {
                    const int mine = j0 + (c & (lanes - 1));
                    uint32_t y = 0;
                    f32x2 d = {0.f, 0.f};
#pragma unroll
                    for (int j = 0; j < kAhead; ++j) {
                        y = mine == j ? rc[j].y : y;
                        d.x = mine == j ? d0[j] : d.x;
                        d.y = mine == j ? d1[j] : d.y;
                    }
                    if (mine < kAhead && e0 + mine < hi && e0 + mine >= s1) dots[((size_t)(y & 0x7FFFFFFFu) * 2 + (y >> 31)) * a.G] = d;
                }
            }
        }
        while (cur < p1 - p0) flush();
        // A record's row is multiplied by both weights, also where there is no pixel to the right (or, for the records of the pixel
        // before the strip, none to the left): an infinite row of grad_out leaves NaN there.  Sums that hold NaN are formed again from
        // what there is, record by record.  (This costs the form with dots 346 -> 351 us at the size above; tests among the
        // products, as branches or as selections, 364 to 390.)
        if (__ballot(nan_px != 0) != 0) {
            for (int i = 0; i < p1 - p0; ++i) {
                if (((nan_px >> i) & 1u) == 0) continue;
                float sum[VEC];
#pragma unroll
                for (int e = 0; e < VEC; ++e) sum[e] = 0.0f;
                for (uint32_t k = lo; k < hi; ++k) {
                    const u32x4 rc = rec[k];
                    const int px = k < s1 ? -1 : (int)(rc.x & 7u);
                    const uint32_t z = px == i ? rc.z : rc.w;
                    if (px != i && (px + 1 != i || z << 1 == 0)) continue;
                    float g[VEC];
                    RowIO<T, VEC>::load_global(grow + (size_t)(rc.x >> 3) * a.C, g);
                    const T* wk = w + (size_t)(rc.y & 0x7FFFFFFFu) * a.G;
#pragma unroll
                    for (int e = 0; e < VEC; ++e)
                        sum[e] = __builtin_fmaf(__builtin_bit_cast(float, z), g[e] * to_f32(wk[MIXED ? (ch + e) / a.hd - ch / a.hd : 0]), sum[e]);
                }
                const size_t row = ((size_t)b * a.nf + lv.base[l] + p0 + i) * a.C + ch;
                if constexpr (DOTS) {
                    __builtin_memcpy(&values[i * kWave + lane], sum, sizeof(sum));
                } else if (chan_ok && direct) {
                    RowIO<T, VEC>::store_global(static_cast<T*>(a.grad_feat) + row, sum);
                } else if (chan_ok) {
#pragma unroll
                    for (int e = 0; e < VEC; ++e)
                        if (ch + e >= chn) unsafeAtomicAdd(a.image + row + e, sum[e]);
                }
            }
        }
        if constexpr (DOTS) {
            const size_t row0 = ((size_t)b * a.nf + lv.base[l] + p0) * a.C;
            if (direct) {
#pragma unroll
                for (int i = 0; i < kDaggStrip; ++i)
                    if (i < cur) __builtin_nontemporal_store(values[i * kWave + lane], reinterpret_cast<typename RowIO<T, VEC>::mem_t*>(static_cast<T*>(a.grad_feat) + row0 + (size_t)i * a.C + ch));
            } else {
                wave_lds_sync();
                const float* sums = reinterpret_cast<const float*>(values);
                for (int i = 0; i < cur; ++i)
#pragma unroll
                    for (int e = 0; e < VEC; ++e) {  // (neighbouring lanes add to neighbouring channels, as above)
                        const float v = sums[(i * VEC + e) * kWave + lane];
                        if (v != 0.0f) unsafeAtomicAdd(a.image + row0 + (size_t)i * a.C + (blk * VEC + e) * kWave + lane, v);
                    }
            }
        }
    }
    if (lv.lost != 0) dagg_levels_without_room<T>(a, lv);
}

// ---- the rest: weights' and locations' gradients in the caller's layout, rounding ---------------------------------------------
// A workgroup per anchor turns the per-group images into the caller's tensors (zeros for locations outside the image); for
// 16-bit dtypes further ones round the rows of grad_feat that were added to in the float32 image.
template <typename T>
__global__ __launch_bounds__(256) void dagg_finish_kernel(const DaggArgs a)
{
    extern __shared__ __align__(16) unsigned char smem[];
    const int anchors = a.bs * a.A;
    if ((int)blockIdx.x >= anchors) {
        __shared__ DaggLevels lv;
        lv.fill(a);
        const uint64_t part = blockIdx.x - anchors, parts = gridDim.x - anchors;
        auto round = [&](uint64_t lo, uint64_t n) {
            for (uint64_t i = part * 256 + threadIdx.x; i < n; i += parts * 256) static_cast<T*>(a.grad_feat)[lo + i] = from_f32<T>(a.image[lo + i]);
        };
        if (!lv.tiled) {
            round(0, (uint64_t)a.bs * a.nf * a.C);
        } else {
            for (int b = 0; b < a.bs; ++b)
                for (int l = 0; l < a.nl; ++l)
                    if (lv.chunks[l] > 1) round(((uint64_t)b * a.nf + lv.base[l]) * a.C, (uint64_t)lv.px[l] * a.C);
        }
        return;
    }
    // position of a location in the images, or 0xFFFF outside the image
    uint16_t* pos = reinterpret_cast<uint16_t*>(smem);
    const int64_t anchor = blockIdx.x;
    const int64_t stride = (int64_t)anchors * a.nloc;  // locations per group
    const f32x2* gl = reinterpret_cast<const f32x2*>(a.gl_part) + anchor * a.nloc;
    T* out_l = static_cast<T*>(a.grad_loc) + anchor * a.nloc * 2;
    for (int li = threadIdx.x; li < a.nloc; li += 256) {
        const int p = li / a.cams, j = (li - p * a.cams) * a.P + p;
        const f32x2 xy = load_xy<T>(a.loc, anchor * a.nloc + li);
        const bool in = inside(xy.x, xy.y);
        pos[li] = in ? (uint16_t)j : (uint16_t)0xFFFFu;
        f32x2 s = {0.f, 0.f};
        if (in)
            for (int g = 0; g < a.G; ++g) s += gl[g * stride + j];
        out_l[2 * li] = from_f32<T>(s.x);
        out_l[2 * li + 1] = from_f32<T>(s.y);
    }
    __syncthreads();
    const int gs = a.G < 256 ? a.G : 256, rows = 256 / gs;  // groups and (location, scale) pairs side by side
    const int g0 = threadIdx.x % gs, r0 = threadIdx.x / gs, n = a.nloc * a.scales;
    const float* gw = a.gw_part + anchor * n;
    T* out_w = static_cast<T*>(a.grad_w) + anchor * n * a.G;
    if (r0 < rows)
        for (int r = r0; r < n; r += rows) {
            const int li = (int)(((uint32_t)r * a.sc_magic) >> 20), sc = r - li * a.scales;
            const uint32_t j = pos[li];
            for (int g = g0; g < a.G; g += gs)
                out_w[(int64_t)r * a.G + g] =
                    from_f32<T>(j != 0xFFFFu ? gw[(int64_t)g * stride * a.scales + (int)j * a.scales + sc] : 0.0f);
        }
}

// The same from the dot products of whole samples: a lane per (location, group), scale after scale.
__global__ __launch_bounds__(256) void dagg_finish_dots_kernel(const DaggArgs a)
{
    __shared__ i32x4 lvl[kMaxLevels];
    if ((int)threadIdx.x < a.nl) lvl[threadIdx.x] = dagg_level(a, threadIdx.x);
    __syncthreads();
    const int64_t anchor = blockIdx.x, loc0 = anchor * a.nloc;
    const int g_log2 = 31 - __builtin_clz(a.G);
    for (int i = threadIdx.x; i < a.nloc << g_log2; i += 256) {
        const int li = i >> g_log2, g = i & (a.G - 1), cam = li % a.cams;
        const f32x2 xy = load_xy<float>(a.loc, loc0 + li);
        const bool in = inside(xy.x, xy.y);
        float sx = 0.f, sy = 0.f;
        for (int sc = 0; sc < a.scales; ++sc) {
            const int64_t sample = (loc0 + li) * a.scales + sc;
            float ga = 0.f, gx = 0.f, gy = 0.f;
            if (in) {
                const Sample sm = sample_geometry(xy.x, xy.y, lvl[cam * a.scales + sc], a.nf, true);
                if (sm.valid) {
                    // (a row's dots are those of its first pixel inside and of that one's right neighbour)
                    const f32x2 up = a.dots[sample * 2 * a.G + g], lo = a.dots[(sample * 2 + 1) * a.G + g];
                    f32x4 d;
                    d.x = sm.cvalid[0] ? up.x : 0.0f;
                    d.y = sm.cvalid[1] ? (sm.cvalid[0] ? up.y : up.x) : 0.0f;
                    d.z = sm.cvalid[2] ? lo.x : 0.0f;
                    d.w = sm.cvalid[3] ? (sm.cvalid[2] ? lo.y : lo.x) : 0.0f;
                    sample_gradients(sm.lw, sm.lh, sm.Wf, sm.Hf, static_cast<const float*>(a.w)[sample * a.G + g], d, ga, gx, gy);
                }
            }
            static_cast<float*>(a.grad_w)[sample * a.G + g] = ga;
            sx += gx;
            sy += gy;
        }
        for (int d = 1; d < a.G; d <<= 1) {
            sx += __shfl_xor(sx, d, kWave);
            sy += __shfl_xor(sy, d, kWave);
        }
        if (g == 0) {
            static_cast<float*>(a.grad_loc)[(loc0 + li) * 2] = sx;
            static_cast<float*>(a.grad_loc)[(loc0 + li) * 2 + 1] = sy;
        }
    }
}

template <typename F>
hipError_t by_vec(int es, int vec, F f)
{
    switch (vec) {
        case 8: if (es == 2) return f(std::integral_constant<int, 8>{}); break;
        case 4: return f(std::integral_constant<int, 4>{});
        case 2: return f(std::integral_constant<int, 2>{});
        case 1: return f(std::integral_constant<int, 1>{});
    }
    return hipErrorInvalidConfiguration;
}

template <typename T>
hipError_t forward_t(const DaggArgs& a, hipStream_t stream)
{
    const dim3 grid(a.map.grid), block(kDaggWaves * kWave);
    return by_vec(sizeof(T), dagg_vec(sizeof(T), a.piece_heads == 1 ? a.piece_ch : a.hd), [&](auto v) {
        constexpr int VEC = decltype(v)::value;
        if constexpr (VEC * sizeof(T) <= 16) {
            const size_t lds = kDaggWaves * (kFoundBytes + kOffBytes + kWave * 16 + (a.piece_heads == 1 ? 0 : kWave * a.piece_heads * 4));
            if (a.piece_heads == 1) hipLaunchKernelGGL((dagg_fwd_kernel<T, VEC, true>), grid, block, lds, stream, a);
            else hipLaunchKernelGGL((dagg_fwd_kernel<T, VEC, false>), grid, block, lds, stream, a);
            return hipGetLastError();
        } else {
            return hipErrorInvalidConfiguration;
        }
    });
}

template <typename T>
hipError_t backward_t(const DaggArgs& a, hipStream_t stream)
{
    // (a multiple of 8 sort workgroups: the others keep their places in the XCD mapping)
    const uint32_t sorts = ((uint32_t)(a.bs * a.nl * a.sort_ranges) + kNumXcd - 1) / kNumXcd * kNumXcd;
    hipError_t e = hipSuccess;
    if (a.dots != nullptr) {
        hipLaunchKernelGGL(dagg_sort_kernel<T>, dim3(sorts + kDaggZeroWgs), dim3(kDaggSortWaves * kWave), kDaggSortLds, stream, a, sorts);
        e = hipGetLastError();
    } else e = by_vec(sizeof(T), dagg_vec(sizeof(T), a.hd), [&](auto v) {
        constexpr int VEC = decltype(v)::value;
        if constexpr (VEC * sizeof(T) <= 16) {
            size_t lds = kDaggBackWaves * kDotsLds;
            if (lds < sizeof(DaggSort)) lds = sizeof(DaggSort);
            hipLaunchKernelGGL((dagg_dots_and_sort_kernel<T, VEC>), dim3(sorts + kDaggZeroWgs + a.map.grid), dim3(kDaggBackWaves * kWave), lds, stream, a, sorts);
            return hipGetLastError();
        } else {
            return hipErrorInvalidConfiguration;
        }
    });
    if (e != hipSuccess) return e;
    e = by_vec(sizeof(T), dagg_vec(sizeof(T), a.C), [&](auto v) {
        constexpr int VEC = decltype(v)::value;
        if constexpr (VEC * sizeof(T) <= 16) {
            // enough workgroups to fill the chip eight times over, or a strip per unit
            const int units = 256 >> a.row_lpr_log2;
            // (strips, and the parts of those that are split: at most one per strip_records records)
            int64_t items = (a.nf + kDaggStrip - 1) / kDaggStrip + 2 * (int64_t)a.nl;
            items += 2 * (int64_t)a.nl * a.A * a.P * (kDaggStrip + 1) / kDaggStrip / a.strip_records;
            int64_t blocks = (a.bs * items * a.row_blocks + units - 1) / units;
            if (blocks > 256 * 32) blocks = 256 * 32;
            const dim3 grid((unsigned)blocks), block(256);
            if constexpr (VEC == 4 && sizeof(T) == 4)
                if (a.dots != nullptr) {
                    hipLaunchKernelGGL((dagg_gradf_kernel<T, VEC, false, true, true>), grid, block, 0, stream, a);
                    return hipGetLastError();
                }
            if (a.hd % VEC != 0) hipLaunchKernelGGL((dagg_gradf_kernel<T, VEC, true, false, false>), grid, block, 0, stream, a);
            else if (a.row_lpr_log2 == 6) hipLaunchKernelGGL((dagg_gradf_kernel<T, VEC, false, true, false>), grid, block, 0, stream, a);
            else hipLaunchKernelGGL((dagg_gradf_kernel<T, VEC, false, false, false>), grid, block, 0, stream, a);
            return hipGetLastError();
        } else {
            return hipErrorInvalidConfiguration;
        }
    });
    if (e != hipSuccess) return e;
    const unsigned rounding = sizeof(T) == 2 ? 512u : 0u;
    if (a.dots != nullptr) hipLaunchKernelGGL(dagg_finish_dots_kernel, dim3((unsigned)(a.bs * a.A)), dim3(256), 0, stream, a);
    else hipLaunchKernelGGL(dagg_finish_kernel<T>, dim3((unsigned)(a.bs * a.A) + rounding), dim3(256), (size_t)((a.nloc + 1) & ~1) * 2, stream, a);
    return hipGetLastError();
}

}  // namespace

hipError_t launch_dagg_forward(int dtype, const DaggArgs& a, hipStream_t stream)
{
    switch (dtype) {
        case MXD_DTYPE_F32: return forward_t<float>(a, stream);
        case MXD_DTYPE_F16: return forward_t<f16_t>(a, stream);
        case MXD_DTYPE_BF16: return forward_t<bf16_t>(a, stream);
        default: return hipErrorInvalidValue;
    }
}

hipError_t launch_dagg_backward(int dtype, const DaggArgs& a, hipStream_t stream)
{
    switch (dtype) {
        case MXD_DTYPE_F32: return backward_t<float>(a, stream);
        case MXD_DTYPE_F16: return backward_t<f16_t>(a, stream);
        case MXD_DTYPE_BF16: return backward_t<bf16_t>(a, stream);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace mxd
