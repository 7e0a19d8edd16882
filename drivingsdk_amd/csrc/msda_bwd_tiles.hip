// grad_value by tile ownership (gfx950, wave64) -- the scatter half of the backward pass.
//
//   grad_value[b, pix_c, h, :] += w_c * attn * grad_out[b, q, h, :]     for the 4 corners c
//
// (reference: kernels/multi_scale_deformable_attn/op_kernel/multi_scale_deformable_attn_grad.cpp:52-126,181-186,
//  where the same sums are issued as atomic-add DMAs.)
//
// Measured on MI355X: a global fp32 atomic is carried out at the memory side at ~20 G
// 64-byte requests/s, and an LDS fp32 atomic add retires ~0.3 lanes per clock per CU.  Either
// makes a per-sample scatter cost milliseconds.  Integer LDS atomics, plain LDS traffic and
// registers are fast, so the scatter is turned inside out:
//
//   * The pixels of every level are cut into tiles.  A workgroup (512 threads) owns one tile of
//     one (batch, head); every thread keeps 32 sums in registers for the whole kernel: a group
//     of 4 to 16 lanes owns 2 to 8 consecutive pixels of up to 32 channels (tiles of 512 pixels),
//     up to 64 (256) or up to 128 (128) -- so that the records are streamed and the lists built
//     and walked once whatever head_dim is (heads of more than 128 channels take two passes
//     over 128-pixel tiles).
//   * The backward's first kernel leaves its samples as pair records {pixel, query, weight,
//     weight of the pixel to the right}, sorted by tile inside the slab of each of its
//     workgroups, with a table of run starts.  The owner of a tile streams the runs of its
//     tile (dense batches of 64 records, fetched two batches ahead) and appends an entry per
//     record to the PIXEL's linked list in LDS (one integer exchange on the list head; entry
//     storage is private to the wavefront, so no allocation atomics are needed).
//   * When the entry storage fills up (or the input ends) the workgroup meets at a barrier and
//     every lane group walks the lists of its own pixels: one coalesced load of the grad_out
//     row of the entry's query per group, fma into the registers.  No atomics, no
//     read-modify-write of shared accumulators.  The walk is pipelined by hand: the entries and
//     rows of the next trip are requested before the rows of the current trip are used.
//   * At the end plain 16-byte stores for tiles a single workgroup owns; tiles of hot (coarse)
//     levels are split over several workgroups by query range, which add their rows with atomics.
//     Tiles much smaller than the workgroup are held in several copies, which are added up in LDS.
//   * Slots of the workgroup that stand for no pixel take extra lists of pixels that collect
//     far more entries than the others (decided from the counts of a work item's first round),
//     so that a hot pixel's entries are walked by several lane groups side by side.
//
// Which (level, tile, query chunk) a workgroup works on is derived on the device from
// spatial_shapes / level_start_index, which never leave device memory; the host only needs
// an upper bound of the number of work items, which follows from nk, nq, nl and np.
#include <type_traits>

#include "msda_device.h"

namespace mxd {

// A work item: a tile, or the share of a hot one that a range of the slabs holds.
struct TileItem {
    int32_t p0, p1;              // pixel range of the tile, relative to the batch element
    int32_t c0, cstep;           // the item takes slabs c0, c0 + cstep, c0 + 2 cstep, ... in the order of KArgs::run_step
    int32_t tile;                // index of the tile within the (batch, head): column of the run table
    int32_t exclusive;           // 1: no other workgroup touches this tile (the item is not split by query range and the
                                 // levels tile the keys, so that no tile of another level holds the same rows)
};

// Work item number `item` of a (batch, head).  Items are numbered from the last level to the first: the coarse levels, whose
// tiles are split into many long-running items, start first and the short items of the fine levels fill the end of the launch.
// (by whole wavefronts)
__device__ inline bool decode_tile_item(const KArgs& a, int32_t item, int lane, TileItem* out)
{
    const LevelLanes lv(a, lane);
    const int32_t n = lv.nt * lv.chunks, inc = LevelLanes::prefix(a, n, lane);
    const int32_t start = __builtin_amdgcn_readlane(inc, a.nl - 1) - inc;
    const uint64_t owner = __ballot(item >= start && item < start + n);
    if (owner == 0) return false;
    const int l = __builtin_ctzll(owner);
    const int32_t chunks = __builtin_amdgcn_readlane(lv.chunks, l), at = item - __builtin_amdgcn_readlane(start, l);
    const int32_t ti = (int32_t)((uint32_t)at / (uint32_t)chunks), tile_px = 1 << a.tile_px_log2;
    const int32_t end = lv.base(l) + __builtin_amdgcn_readlane(lv.px, l);
    out->p0 = lv.base(l) + ti * tile_px;
    out->p1 = (out->p0 + tile_px) < end ? (out->p0 + tile_px) : end;
    out->c0 = at - ti * chunks;
    out->cstep = chunks;
    out->tile = __builtin_amdgcn_readlane(lv.first, l) + ti;
    out->exclusive = chunks == 1 && lv.canonical;
    return true;
}

// The samples of levels whose tiles found no room in the run table, and of levels that start before the tensor and reach
// into it (they have no tiles: LevelLanes), added to grad_value one sample per thread with atomics: share `part` of
// `parts` of the samples of (batch b, head h).  Only levels that overlap can have more tiles between them than the
// table holds; for such layouts the whole image was zero-filled and every tile adds with atomics as well.  Slow, and
// there so that level_start_index is honoured however it comes.  Plain operator only.
// unfit: kMaxLevels flags in LDS, filled here.
template <typename T>
__device__ inline void add_levels_without_tiles(const KArgs& a, int b, int h, int part, int parts, int32_t* unfit)
{
    __shared__ int any_unfit;
    if (threadIdx.x == 0) {
        int32_t first = 0, any = 0;
        for (int l = 0; l < a.nl; ++l) {
            const i32x4 L = load_level(a, l);
            int32_t P;
            const int32_t nt = level_tile_count(L.x, L.y, L.z, a.nk, a.tile_px_log2, &P);
            const bool before = L.x > 0 && L.y > 0 && L.z < 0 && L.z + (int64_t)L.x * L.y > 0;
            const bool fits = !before && first + nt <= a.tbl_stride - 1;
            unfit[l] = fits ? 0 : 1;
            if (fits) first += nt;
            else if (before || nt > 0) any = 1;
        }
        any_unfit = any;
    }
    __syncthreads();
    if (!any_unfit) return;
    const T* loc = static_cast<const T*>(a.loc);
    const T* attn = static_cast<const T*>(a.attn);
    const T* gout = static_cast<const T*>(a.grad_out);
    float* img = a.grad_value + (size_t)b * (a.gbatch_bytes / 4) + (size_t)h * a.hd;
    const int64_t n = (int64_t)a.nq * a.S;
    for (int64_t i = (int64_t)part * blockDim.x + threadIdx.x; i < n; i += (int64_t)parts * blockDim.x) {
        const int q = (int)(i / a.S), s = (int)(i - (int64_t)q * a.S);
        const int l = (int)(((uint32_t)s * a.np_magic) >> 20);
        if (!unfit[l]) continue;
        const int64_t e = (((int64_t)b * a.nq + q) * a.nh + h) * a.S_full + s;
        const Sample sm = sample_geometry(to_f32(loc[2 * e]), to_f32(loc[2 * e + 1]), load_level(a, l), a.nk, true);
        if (!sm.valid) continue;
        const float aw = to_f32(attn[e]);
        const T* grow = gout + (((int64_t)b * a.nq + q) * a.nh + h) * a.hd;
        for (int ch = 0; ch < a.hd; ++ch) {
            const float gch = to_f32(grow[ch]) * aw;
#pragma unroll
            for (int k = 0; k < 4; ++k)
                if (sm.cvalid[k]) unsafeAtomicAdd(img + (size_t)sm.pix[k] * ((size_t)a.nh * a.hd) + ch, sm.w[k] * gch);
        }
    }
}

// LPG lanes (a lane group) read a grad_out row together, VEC elements per load.  A lane accumulates CHL channels per pass: PIECE =
// max(VEC, 4) consecutive ones of every block of LPG * PIECE channels, of 32 / CHL pixels (32 sums per lane) and of the pixel behind
// them.  That makes tiles of 512 pixels (LPG 8 and CHL 4, LPG 4 and CHL 8), 256 (8, 8) or 128 (8, 16 and 16, 8); heads with more than
// LPG * CHL channels are done in several passes over the same records.
// What a load costs the memory pipeline is its 64 addresses, whatever each of them brings (17 clocks per load of 4, 8 or 16 bytes a lane
// with every row in L1, and as many when half of the lanes have no row), so 16-bit rows are read 16 bytes a lane like float32 ones
// (two batch elements of the encoder in bfloat16 168 -> 141 us; 6 x 9675 queries of 32 samples in float16 408 -> 376; 128 channels
// in bfloat16 182 -> 153).  The pixel behind the group's last one, whose sums the narrowest form alone kept before: 128
// channels in bfloat16 153 -> 134 us, 37 in float32 228 -> 204 (with one list per trip instead of two, which pays for the registers),
// whole backward of 72 to 128 channels in float32 0.86 to 1.01 of the time (16 lanes of 8 channels instead of 8 of 16; in the
// 16-bit types 8 of 16 are up to 5 % faster).
template <typename T, int LPG, int CHL, int VEC>
__global__ __launch_bounds__(kTileThreads, 4) void msda_gradv_tiles_kernel(const KArgs a, const TileArgs t)
{
    constexpr int PIECE = VEC < 4 ? 4 : VEC;            // consecutive channels of a lane
    static_assert((LPG == 4 || LPG == 8 || LPG == 16) && (CHL == 4 || CHL == 8 || CHL == 16) && CHL % PIECE == 0 && PIECE % VEC == 0, "a lane owns whole pieces");
    constexpr int CH = LPG * CHL;                       // channels per pass
    constexpr int NB = CHL / PIECE;                     // pieces per lane and pass, CB channels apart
    constexpr int NV = PIECE / VEC;                     // loads per piece
    constexpr int CB = LPG * PIECE;
    constexpr int PPG = 32 / CHL;                       // pixels per lane group
    constexpr int GPW = kWave / LPG;                    // lane groups per wavefront
    constexpr int kTilePx = (kTileThreads / LPG) * PPG;  // pixels per tile = pixel slots of the workgroup
    constexpr int kTilePxLog2 = kTilePx == 512 ? 9 : kTilePx == 256 ? 8 : 7;
    static_assert((1 << kTilePxLog2) == kTilePx, "tile size");
    // lists a lane group walks together, one entry of each per trip, two trips in flight (tiles of 512 pixels with one list per trip:
    // encoder float32 165 -> 184 us, bfloat16 142 -> 148, the float16 shape above 376 -> 397; 128 channels with two 153 -> 161)
    constexpr int kWalk = LPG * CHL >= 64 ? 1 : 2;
    // A lane group also keeps the sums its pairs leave for the pixel behind its last one (the first pixel of the next group) and
    // hands them over when the rounds are done: a pair is then one list entry wherever it lies in the tile, instead of two for
    // the one pair in PPG that straddles two groups.
    constexpr int kAccPx = PPG + 1;
    constexpr int kCarryAt = kTileEntCap - 1 - LPG * CHL / 4;  // entries of a wavefront's storage through which its last group hands over
    constexpr int NW = kTileThreads / kWave;            // wavefronts per workgroup
    constexpr uint32_t kDummyOfWave = kTileEntCap - 1;  // last entry slot of every wavefront
    __shared__ uint32_t heads[kTileThreads];            // list head per pixel slot (byte offset of the entry in `ent`)
    // entry: {byte offset of the grad_out row, weight for the list's pixel, weight for the
    // next pixel, next entry of the same list}
    __shared__ u32x4 ent[NW * kTileEntCap];
    static_assert(kTilePx * CH * sizeof(float) <= sizeof(ent), "a tile's sums fit the entry storage");
    // up to 64 runs of records per wavefront at a time: where the run's records lie less the records before it, records before the run
    // (and behind the last one), and the run of every record of the window at hand
    __shared__ uint32_t run_at_all[NW * kWave];
    __shared__ uint32_t run_pre_all[NW * (kWave + 1)];
    __shared__ uint32_t run_of_all[NW * kWave];
    __shared__ int32_t lv_unfit[kMaxLevels];
    __shared__ int done_count, nan_seen;
    // Pixels that collect far more entries than the others (inputs that pile samples on a few pixels) get extra
    // lists in the slots of the workgroup that no pixel of the tile uses -- when there are such slots.  The first
    // round counts entries per slot (two 16-bit counters per word); after it the same array holds, per slot,
    // {first extra slot, number of extra slots (2^k - 1)} as 9 + 4 bits.
    __shared__ uint32_t slot_info[kTileThreads / 2];
    __shared__ uint32_t spare_next, round1_total;

    if (a.tile_px_log2 != kTilePxLog2) return;  // (uniform; the launcher derives both from head_dim)
    Work wk;
    if (!decode_block(t.map, blockIdx.x, a.bs, a.nh, t.items_per_bh, &wk)) return;
    if (t.batch_major == 0) {
        // item-major, batch-minor: the long-running items (coarse levels, numbered first) of every
        // batch element start at the beginning of the launch
        const int64_t r = (int64_t)wk.b * t.items_per_bh + wk.q_begin;
        wk.b = (int32_t)(r % a.bs);
        wk.q_begin = (int32_t)(r / a.bs);
    }
    if (wk.q_begin >= t.items_per_bh - t.extra) {  // (uniform: one of the workgroups behind the work items)
        add_levels_without_tiles<T>(a, wk.b, wk.h, wk.q_begin - (t.items_per_bh - t.extra), t.extra, lv_unfit);
        return;
    }
    if (threadIdx.x < kTileThreads / 2) slot_info[threadIdx.x] = 0;
    // an empty list points at the dummy entry of the wavefront that owns the pixel slot (slot s belongs to lane group
    // s / PPG, i.e. to wavefront s / (GPW PPG); slots past the tile size are never used)
    heads[threadIdx.x] = ((threadIdx.x / (GPW * PPG)) % NW * kTileEntCap + kDummyOfWave) * 16u;
    if (threadIdx.x == 0) {
        done_count = 0;
        nan_seen = 0;
        spare_next = 0;
        round1_total = 0;
    }
    TileItem it;
    if (!decode_tile_item(a, wk.q_begin, (int)threadIdx.x & (kWave - 1), &it)) return;  // uniform
    __syncthreads();

    const int hd = a.hd;
    const int tid = threadIdx.x;
    const int lane = tid & (kWave - 1);
    // (read as a scalar -- the compiler cannot know that tid >> 6 is the same in every lane of a wavefront, and whatever
    //  depends on it, the wavefront's runs and its entry storage, is otherwise a per-lane value steered by exec masks)
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int npx = it.p1 - it.p0;
    // A tile much smaller than the workgroup is held in several copies (lists and registers),
    // each taking the samples of some queries; the copies are added up at the end.
    const int npx_pad = (npx + PPG - 1) / PPG * PPG;
    int copies = 1;
    while (copies < 8 && 2 * copies * npx_pad <= kTilePx) copies *= 2;
    const bool owned = it.exclusive != 0;            // plain stores are enough (this is what tile_stored_directly() says of the tile)
    const int copies_log2 = __builtin_ctz(copies);
    const int nused = copies * npx_pad;              // slots that stand for a pixel of the tile
    const int nspare = kTilePx - nused;              // slots free for extra lists
    const bool can_split = nspare >= tile_group_px(kTilePxLog2);
    const bool direct_t = a.sparse != 0 && a.grad_value_t != nullptr && owned;
    typedef uint16_t __attribute__((may_alias)) u16_alias;  // halves of LDS words that are also accessed whole
    u16_alias* slot_info16 = reinterpret_cast<u16_alias*>(slot_info);
    bool first_round = true;                         // (of the first channel pass)
    const uint32_t seg = wave * kTileEntCap;  // this wavefront's entry storage
    uint32_t* run_at = run_at_all + wave * kWave;
    uint32_t* run_pre = run_pre_all + wave * (kWave + 1);
    typedef uint32_t __attribute__((may_alias)) u32_bytes;
    u32_bytes* run_of4 = run_of_all + wave * kWave;
    const uint8_t* run_of = reinterpret_cast<const uint8_t*>(run_of_all + wave * kWave);

    const T* gout = static_cast<const T*>(a.grad_out);
    const int64_t bh = (int64_t)wk.b * a.nh + wk.h;
    const uint32_t* tbl = a.tbl + bh * a.nwg * a.tbl_stride + it.tile;
    // the records of this (batch, head) as a bound buffer (the layout keeps them below 4 GiB)
    typedef uint32_t u32x3 __attribute__((ext_vector_type(3)));
    const __amdgpu_buffer_rsrc_t rres = make_rsrc(a.rec + bh * a.nwg * a.rec_cap * kRecDwords,
                                                  (uint32_t)a.nwg * (uint32_t)a.rec_cap * (kRecDwords * 4u));
    // Runs of this wavefront: number wave, + NW, + 2 NW, ... of the item's.  Every item, and every stretch of an item's
    // stream, takes slabs from all over the query range: with queries in the raster order of a feature map a stretch of
    // neighbouring slabs puts its records on a few rows of pixels, and the few lane groups that own those walk long
    // lists while the others wait.
    const int item_runs = (a.nwg - it.c0 + it.cstep - 1) / it.cstep;
    const int nruns = (item_runs - wave + NW - 1) / NW;  // <= 0: none

    float* gimg = a.grad_value + (size_t)wk.b * (a.gbatch_bytes / 4);
    const int64_t row_pitch = (int64_t)a.nh * hd;  // floats between neighbouring pixels
    const uint32_t row_bytes = (uint32_t)(a.nh * hd * (int)sizeof(T));  // between the grad_out rows of two queries
    // grad_out of this batch element as a bound buffer: offsets >= 2^31 read as zeros
    const uint32_t gout_batch_bytes = (uint32_t)a.nq * row_bytes;
    const __amdgpu_buffer_rsrc_t gres =
        make_rsrc(reinterpret_cast<const char*>(gout) + (size_t)wk.b * gout_batch_bytes, gout_batch_bytes);
    const uint32_t ghead_off = (uint32_t)wk.h * hd * (uint32_t)sizeof(T);
    // the dummy entry ends every list of this wavefront's pixels: weight 0, a row offset the
    // buffer range check answers with zeros (at no cost in the memory pipeline), next = itself
    // (lists are linked by byte offsets into `ent`: the walk then needs no shift per entry)
    const uint32_t dummy = (seg + kDummyOfWave) * 16u;
    auto ent_at = [&](uint32_t off) -> u32x4& { return *reinterpret_cast<u32x4*>(reinterpret_cast<unsigned char*>(ent) + off); };
    if (lane == 0) ent_at(dummy) = u32x4{kInvalidCorner, 0u, 0u, dummy};

    // lane j of a group keeps its channels of the pixels grp * PPG .. grp * PPG + PPG - 1
    const int grp = tid / LPG, j = tid % LPG;

    // First channel of the four that a lane loads for channels ch .. ch + 3: its own -- what lies behind a float32 row's
    // end is read and never written, and the range check at the end of the buffer zeroes single dwords.  A dword holds
    // two 16-bit elements, so there the last lane of a row whose length is no multiple of 4 reads the row's last four
    // and moves its sums to their places when the rounds are done.
    auto first_channel = [&](int ch) { return sizeof(T) == 2 && VEC == 4 ? piece_start<4>(ch, hd) : ch; };

    // the next channel pass starts from a clean state (the dummy entry may have been overwritten by the transposition)
    auto clean_state = [&]() {
        __syncthreads();
        if (threadIdx.x == 0) {
            done_count = 0;
            nan_seen = 0;
        }
        // (opaque: the entry would otherwise be kept through the whole pass, in registers that some forms do not have -- and
        //  memory for spilled ones costs every wavefront time before it starts)
        uint32_t none = 0u;
        asm volatile("" : "+v"(none));
        if (lane == 0) ent_at(dummy) = u32x4{none | kInvalidCorner, none, none, none + dummy};
        __syncthreads();
    };

    for (int cb = 0; cb < hd; cb += CH) {
        float acc[kAccPx][CHL];
#pragma unroll
        for (int i = 0; i < kAccPx; ++i)
#pragma unroll
            for (int c = 0; c < CHL; ++c) acc[i][c] = 0.0f;
        // channels past head_dim re-read channel 0; their sums are never written out
        const int my_ch = cb + j * PIECE;  // (first channel of this lane in block 0; block k: + CB k)
        uint32_t lane_off[NB];
#pragma unroll
        for (int k = 0; k < NB; ++k)
            lane_off[k] = ghead_off + (uint32_t)(my_ch + CB * k < hd ? first_channel(my_ch + CB * k) : 0) * (uint32_t)sizeof(T);
        const int nch = (hd - cb) < CH ? (hd - cb) : CH;

        // input state of this wavefront (uniform): next group of runs, records of the current
        // group, next unread record, window of records whose runs are known, and the two batches fetched ahead
        int rg = 0, N = 0, i0 = 0, window = -1;
        u32x3 ahead[2] = {};
        // The runs of kWindow records from record w0 of the group on: a run's lane marks its first record there, and a running maximum
        // over the window, four records per lane, spreads the marks.  (A search among the run starts took every batch of 64 records
        // eight trips to LDS one after the other; a window of four batches takes three, and a batch two.  With the batches requested two
        // ahead instead of one -- a batch took the time of a trip to memory -- and eight of them per round instead of seven: 6 x 9675
        // queries of 32 samples in float16 363 -> 340 us, two batch elements of the encoder in bfloat16 138 -> 129, in float32
        // 158 -> 153, 37 channels in float32 191 -> 184.)
        constexpr int kWindow = 4 * kWave;
        auto open_window = [&](uint32_t w0) {
            run_of4[lane] = 0u;
            const uint32_t pre = run_pre[lane], end = run_pre[lane + 1], at = pre > w0 ? pre : w0;
            wave_lds_sync();
            if (at < end && at < w0 + kWindow) reinterpret_cast<uint8_t*>(run_of_all + wave * kWave)[at - w0] = (uint8_t)lane;
            wave_lds_sync();
            const uint32_t m = run_of4[lane];
            auto larger = [](uint32_t x, uint32_t y) { return x > y ? x : y; };
            const uint32_t m0 = m & 255u, m1 = larger(m0, (m >> 8) & 255u), m2 = larger(m1, (m >> 16) & 255u), m3 = larger(m2, m >> 24);
            const uint32_t up = wave_scan(m3, larger);  // largest mark so far
            const uint32_t before = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)up, 0x138, 0xF, 0xF, false);  // wave_shr 1
            run_of4[lane] = larger(m0, before) | larger(m1, before) << 8 | larger(m2, before) << 16 | larger(m3, before) << 24;
            wave_lds_sync();
        };
        auto request = [&](int first, u32x3& to) {
            if (first < N && (first & ~(kWindow - 1)) != window) {
                window = first & ~(kWindow - 1);
                open_window((uint32_t)window);
            }
            // (one 12-byte load, non-temporal: a record is read once, but for the two batches ahead that a walk drops and the next round asks for
            //  again, up to 128 of some 500 records: 3 to 17 % more bytes than with one batch ahead where items have many rounds.
            //  Unconditional, beyond the buffer where there is no record: behind a branch around a load the compiler can only wait for
            //  every load there is)
            const int i = first + lane;
            const uint32_t at = i < N ? (run_at[run_of[i & (kWindow - 1)]] + (uint32_t)i) * (kRecDwords * 4u) : ~0u;
            to = __builtin_bit_cast(u32x3, __builtin_amdgcn_raw_buffer_load_b96(rres, at, 0, 2));
        };
        bool counted = false;    // this wavefront has reported the end of its work
        while (true) {
            // ---- stream records, append list entries ------------------------------------------
            int count = 0;  // entries of this wavefront in this round (uniform)
            request(i0, ahead[0]);  // (again after a walk: the batches fetched ahead are not kept across it)
            request(i0 + kWave, ahead[1]);
            // (room for a batch of records, which leave two entries each where extra lists take some)
            auto full = [&]() { return count + (can_split ? 2 : 1) * kWave > (int)kDummyOfWave; };
            auto next_group = [&]() {
                // up to 64 runs: one run per lane
                const int r = rg + lane;
                uint32_t len = 0, src = 0;
                if (r < nruns) {
                    const uint32_t i = (uint32_t)(it.c0 + it.cstep * (wave + NW * r));
                    const uint32_t w = i * a.run_step % (uint32_t)a.nwg;  // (below 2^32: the launcher's choice of the step)
                    const uint32_t* row = tbl + (size_t)w * a.tbl_stride;
                    const uint32_t s = row[0];
                    len = row[1] - s;
                    src = w * (uint32_t)a.rec_cap + s;
                }
                uint32_t inc = len;
#pragma unroll
                for (int d = 1; d < kWave; d <<= 1) {
                    const uint32_t o = __shfl_up(inc, d, kWave);
                    if (lane >= d) inc += o;
                }
                wave_lds_sync();
                run_at[lane] = src - (inc - len);
                run_pre[lane + 1] = inc;
                if (lane == 0) run_pre[0] = 0u;
                wave_lds_sync();
                // (read as a scalar: the loop that N bounds is then steered by scalar branches; a lane shuffle would make
                //  N, and with it the whole input state of the wavefront, a per-lane value)
                N = (int)__builtin_amdgcn_readlane(inc, kWave - 1);
                rg += kWave;
                i0 = 0;
                window = -1;
                request(0, ahead[0]);
                request(kWave, ahead[1]);
            };
            auto batch = [&](u32x3& mine) {
                const bool have = i0 + lane < N;
                const u32x3 rc = mine;
                i0 += kWave;
                request(i0 + kWave, mine);
                // A record is the pair (pixel, pixel + 1) and becomes ONE entry in the list of the left pixel (the grad_out row
                // is fetched once for both).  The right pixel of the last pixel of the tile belongs to the next tile: added
                // with atomics.
                int lst[2] = {-1, -1};
                float w0[2] = {0.f, 0.f}, w1[2] = {0.f, 0.f};
                uint32_t q = 0;
                bool spill = false;
                float wb = 0.f;
                // (a record that does not belong to this tile or names no query of the batch element is dropped:
                // the run table and the records are only as good as the workspace the caller hands over)
                const uint32_t rkey = rc.x;
                if (have && (rkey & (uint32_t)(kTilePx - 1)) < (uint32_t)npx && (rkey >> kTilePxLog2) < (uint32_t)a.nq) {
                    const uint32_t ya = rc.y, za = rc.z;
                    q = rkey >> kTilePxLog2;
                    const int pl = (int)(rkey & (uint32_t)(kTilePx - 1));
                    const float wa = __builtin_bit_cast(float, ya);
                    wb = __builtin_bit_cast(float, za);
                    const int copy_off = (int)(q & (uint32_t)(copies - 1)) * npx_pad;
                    const bool in_r = pl + 1 < npx;
                    lst[0] = pl + copy_off;
                    w0[0] = wa;
                    w1[0] = in_r ? wb : 0.0f;
                    spill = !in_r && wb != 0.0f;
                }
                if (can_split && !first_round) {
                    // entries of a pixel with extra lists are dealt to them by query; a pair entry that moves
                    // to an extra list leaves its right half to the right pixel's own lists
#pragma unroll
                    for (int k = 0; k < 2; ++k) {
                        if (lst[k] >= 0) {
                            const uint32_t o = slot_info16[lst[k]];
                            const uint32_t r = (q >> copies_log2) & (o >> 9);
                            if (r != 0) {
                                if (k == 0 && w1[0] != 0.0f) {
                                    lst[1] = lst[0] + 1;
                                    w0[1] = w1[0];
                                    w1[0] = 0.0f;
                                }
                                lst[k] = nused + (int)(o & 511u) + (int)r - 1;
                            }
                        }
                    }
                }
                const bool count_slots = can_split && first_round;
#pragma unroll
                for (int k = 0; k < 2; ++k) {
                    if (k == 1 && (!can_split || first_round)) break;  // (only a pair that moved to an extra list leaves a second entry)
                    const bool push = lst[k] >= 0;
                    const uint64_t mask = __ballot(push);
                    if (mask) {
                        if (push) {
                            const uint32_t pos = seg + count +
                                                 __builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32),
                                                                           __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0));
                            const uint32_t next = atomicExch(&heads[lst[k]], pos * 16u);
                            ent[pos] = u32x4{q * row_bytes, __builtin_bit_cast(uint32_t, w0[k]),
                                             __builtin_bit_cast(uint32_t, w1[k]), next};
                            if (count_slots) atomicAdd(&slot_info[lst[k] >> 1], (lst[k] & 1) ? 0x10000u : 1u);
                        }
                        count += __builtin_popcountll(mask);
                    }
                }
                // pairs that reach into the next tile: one at a time, the wavefront adds the row
                uint64_t smask = __ballot(spill);
                while (smask) {
                    const int src_lane = __builtin_ctzll(smask);
                    smask &= smask - 1;
                    const uint32_t sq = __builtin_amdgcn_readlane(q, src_lane);
                    const float sw = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(uint32_t, wb), src_lane));
                    for (int ch = lane; ch < nch; ch += kWave) {
                        const float g = to_f32(gout[((int64_t)wk.b * a.nq + sq) * row_pitch + (int64_t)wk.h * hd + cb + ch]);
                        unsafeAtomicAdd(gimg + (int64_t)it.p1 * row_pitch + (int64_t)wk.h * hd + cb + ch, sw * g);
                    }
                }
            };
            while (true) {
                if (i0 >= N) {
                    if (rg >= nruns) break;  // input exhausted
                    next_group();
                    continue;
                }
                if (full()) break;
                batch(ahead[0]);
                if (i0 >= N) continue;
                if (full()) break;
                batch(ahead[1]);
            }
            if (rg >= nruns && i0 >= N && !counted) {
                counted = true;
                if (lane == 0) atomicAdd(&done_count, 1);
            }
            if (can_split && first_round && lane == 0) atomicAdd(&round1_total, (uint32_t)count);
            __syncthreads();
            const bool all_done = done_count == NW;
            if (can_split && first_round) {
                // a slot with more than 1.5 times the average gets extra lists for the rounds to come
                // (every thread replaces the counter of its own slot; neighbours share a word, not a half)
                uint32_t o = 0;
                if (!all_done && tid < nused) {
                    const uint32_t c = slot_info16[tid];
                    const float limit = __builtin_fmaxf(1.5f * (float)round1_total / (float)nused, 4.0f);
                    const uint32_t m = (uint32_t)__builtin_ceilf((float)c / limit);
                    uint32_t extra = m <= 1 ? 0u : m <= 2 ? 1u : m <= 4 ? 3u : m <= 8 ? 7u : 15u;
                    if (extra != 0) {
                        const uint32_t base = atomicAdd(&spare_next, extra);
                        while (extra != 0 && base + extra > (uint32_t)nspare) extra >>= 1;
                        if (extra != 0) o = base | (extra << 9);
                    }
                }
                slot_info16[tid] = (uint16_t)o;
                first_round = false;
            }

            // ---- every group of LPG lanes walks the lists of its PPG pixels --------------------
            // The lanes of a group read a block of a grad_out row with ONE coalesced load.
            // The loop body is branch-free: a list that has ended keeps "reading" the dummy entry.
            // kWalk lists are walked together, one entry of each per trip, and two trips are in flight.
            {
                // (a row stays as it was loaded until it is used: what is in flight takes half the registers in the 16-bit
                //  types, and no conversion waits for its row where the row is requested)
                typedef typename RowIO<T, VEC>::raw_t raw_t;
                auto fetch = [&](uint32_t& e, raw_t (&g)[NB][NV], float& wa, float& wb) {
                    const u32x4 en = ent_at(e);
                    // (a bit cast applied directly to a vector element picks up element 0: copy first)
                    const uint32_t ya = en.y, za = en.z;
                    wa = __builtin_bit_cast(float, ya);
                    wb = __builtin_bit_cast(float, za);
#pragma unroll
                    for (int k = 0; k < NB; ++k)
#pragma unroll
                        for (int v = 0; v < NV; ++v)
                            g[k][v] = RowIO<T, VEC>::load_raw(gres, en.x + lane_off[k] + (uint32_t)(v * VEC * sizeof(T)));
                    e = en.w;
                };
#pragma unroll
                for (int i = 0; i < PPG; i += kWalk) {
                    const int px = grp * PPG + i;
                    uint32_t e[kWalk];
#pragma unroll
                    for (int m = 0; m < kWalk; ++m) e[m] = heads[px + m];
                    if (j == 0) {  // same wavefront: ordered after the reads above
#pragma unroll
                        for (int m = 0; m < kWalk; ++m) heads[px + m] = dummy;
                    }
                    // two sets of rows in flight: the entries and rows of the next trip are requested before the
                    // rows of this trip are used, so that a long list costs its entries' LDS latency per trip
                    // and not the latency of a row load (reads past a list's end land on the dummy entry)
                    raw_t gA[kWalk][NB][NV], gB[kWalk][NB][NV];
                    float uA[kWalk], vA[kWalk], uB[kWalk], vB[kWalk];
                    auto use = [&](raw_t (&g)[kWalk][NB][NV], float (&u)[kWalk], float (&v)[kWalk]) {
#pragma unroll
                        for (int m = 0; m < kWalk; ++m) {
#pragma unroll
                            for (int k = 0; k < NB * NV; ++k) {
                                float row[VEC];
                                RowIO<T, VEC>::unpack(g[m][k / NV][k % NV], row);
#pragma unroll
                                for (int e = 0; e < VEC; ++e) {
                                    const int c = k * VEC + e;
                                    acc[i + m][c] = __builtin_fmaf(u[m], row[e], acc[i + m][c]);
                                    acc[i + m + 1][c] = __builtin_fmaf(v[m], row[e], acc[i + m + 1][c]);
                                }
                            }
                        }
                    };
                    // Neither the scheduler nor the optimiser may move the requests behind the use of the other set (left to
                    // itself the compiler sinks one of the two past the loop's exit test, in some instantiations both).
                    auto keep_order = []() {
                        asm volatile("" ::: "memory");
                        __builtin_amdgcn_sched_barrier(0);
                    };
                    auto any_left = [&]() {
                        bool t = false;
#pragma unroll
                        for (int m = 0; m < kWalk; ++m) t |= e[m] != dummy;
                        return __ballot(t) != 0;
                    };
                    if (any_left()) {
#pragma unroll
                        for (int m = 0; m < kWalk; ++m) fetch(e[m], gA[m], uA[m], vA[m]);
                        while (true) {
                            // A holds a trip that has not been used; is there anything after it?
                            bool pending = any_left();
#pragma unroll
                            for (int m = 0; m < kWalk; ++m) fetch(e[m], gB[m], uB[m], vB[m]);
                            keep_order();
                            use(gA, uA, vA);
                            if (!pending) break;  // (B holds dummy entries only)
                            pending = any_left();
#pragma unroll
                            for (int m = 0; m < kWalk; ++m) fetch(e[m], gA[m], uA[m], vA[m]);
                            keep_order();
                            use(gB, uB, vB);
                            if (!pending) break;  // (A holds dummy entries only)
                        }
                    }
                }
            }
            __syncthreads();
            if (all_done) break;
        }

        {
            bool bad = false;
#pragma unroll
            for (int i = 0; i < kAccPx; ++i)
#pragma unroll
                for (int c = 0; c < CHL; ++c) bad |= acc[i][c] != acc[i][c];
            if (bad) nan_seen = 1;
            // what a group collected for the first pixel of the next group: inside a wavefront from lane to lane, from
            // the last group of a wavefront to the first of the next through the entry storage (free now; the last
            // group of the workgroup has nothing to hand over: a pair never starts on the last pixel of a tile)
            const int gw = lane / LPG;
            if (gw == GPW - 1) {
#pragma unroll
                for (int k = 0; k < CHL / 4; ++k)
                    ent[seg + kCarryAt + k * LPG + j] =
                        u32x4{__builtin_bit_cast(uint32_t, acc[PPG][4 * k]), __builtin_bit_cast(uint32_t, acc[PPG][4 * k + 1]),
                              __builtin_bit_cast(uint32_t, acc[PPG][4 * k + 2]), __builtin_bit_cast(uint32_t, acc[PPG][4 * k + 3])};
            }
            __syncthreads();
            if (__builtin_amdgcn_readfirstlane(nan_seen) != 0) {
                // The walk adds a row of grad_out to the pixel of an entry and, times the entry's other weight, to the pixel behind it,
                // also where that weight is zero because there is no such pixel: an infinite row leaves NaN there.  Sums that hold
                // NaN are formed again here, by a wavefront for an eighth of the pixels, in LDS, from what is there only: record by
                // record, ten times as long, and only for tiles that have such rows.  (With a mask in the walk the forms of two
                // lists per trip take 3 to 4 % longer: two batch elements of the encoder in float32 166 -> 171 us, 6 x 9675 queries
                // of 32 samples in float16 378 -> 394.)
                typedef float __attribute__((may_alias)) f32_alias;
                f32_alias* sums = reinterpret_cast<f32_alias*>(ent);
                constexpr int kOwn = kTilePx / NW;
                const int own0 = wave * kOwn, own1 = own0 + kOwn < npx ? own0 + kOwn : npx;
                __syncthreads();  // (the handed-over sums are not needed)
                for (int k = lane; k < kOwn * CH; k += kWave) sums[own0 * CH + k] = 0.0f;
                wave_lds_sync();
                for (int r = 0; r < item_runs && own0 < npx; ++r) {
                    const uint32_t w = (uint32_t)(it.c0 + it.cstep * r) * a.run_step % (uint32_t)a.nwg;
                    const uint32_t* row = tbl + (size_t)w * a.tbl_stride;
                    const uint32_t first = row[0], n = row[1] - first;
                    for (uint32_t i0 = 0; i0 < n; i0 += kWave) {
                        const uint32_t i = i0 + lane;
                        u32x3 rc = {0u, 0u, 0u};
                        if (i < n) rc = __builtin_bit_cast(u32x3, __builtin_amdgcn_raw_buffer_load_b96(rres, (w * (uint32_t)a.rec_cap + first + i) * (kRecDwords * 4u), 0, 0));
                        const uint32_t key = rc.x, ya = rc.y, za = rc.z;
                        const int pl = (int)(key & (uint32_t)(kTilePx - 1));
                        uint64_t mask = __ballot(i < n && pl < npx && (key >> kTilePxLog2) < (uint32_t)a.nq && pl + 1 >= own0 && pl < own1);
                        while (mask) {
                            const int from = __builtin_ctzll(mask);
                            mask &= mask - 1;
                            const uint32_t k = __builtin_amdgcn_readlane(key, from);
                            const float wa = __builtin_bit_cast(float, __builtin_amdgcn_readlane(ya, from));
                            const float wb = __builtin_bit_cast(float, __builtin_amdgcn_readlane(za, from));
                            const int p = (int)(k & (uint32_t)(kTilePx - 1));
                            const T* grow = gout + ((int64_t)wk.b * a.nq + (k >> kTilePxLog2)) * row_pitch + (int64_t)wk.h * hd + cb;
                            for (int c = lane; c < nch; c += kWave) {
                                const float g = to_f32(grow[c]);
                                if (p >= own0) sums[p * CH + c] = __builtin_fmaf(wa, g, sums[p * CH + c]);
                                if (p + 1 < own1 && wb != 0.0f) sums[(p + 1) * CH + c] = __builtin_fmaf(wb, g, sums[(p + 1) * CH + c]);
                            }
                        }
                    }
                }
                wave_lds_sync();
                for (int k = lane; k < (own1 - own0) * CH; k += kWave) {
                    const int px = own0 + k / CH, c = k % CH;
                    if (c >= nch) continue;
                    const int64_t at = (int64_t)(it.p0 + px) * row_pitch + (int64_t)wk.h * hd + cb + c;
                    const float v = sums[px * CH + c];
                    if (!owned || px == 0) unsafeAtomicAdd(gimg + at, v);
                    else if (sizeof(T) == 2 && direct_t) static_cast<T*>(a.grad_value_t)[(size_t)wk.b * (a.gbatch_bytes / 4) + at] = from_f32<T>(v);
                    else gimg[at] = t.accumulate ? gimg[at] + v : v;
                }
                clean_state();
                continue;
            }
            float cin[CHL];
#pragma unroll
            for (int c = 0; c < CHL; ++c) cin[c] = __shfl_up(acc[PPG][c], LPG, kWave);
            if (gw == 0) {
#pragma unroll
                for (int k = 0; k < CHL / 4; ++k) {
                    const u32x4 o = wave > 0 ? ent[seg - kTileEntCap + kCarryAt + k * LPG + j] : u32x4{0u, 0u, 0u, 0u};
                    const uint32_t o0 = o.x, o1 = o.y, o2 = o.z, o3 = o.w;
                    cin[4 * k] = __builtin_bit_cast(float, o0);
                    cin[4 * k + 1] = __builtin_bit_cast(float, o1);
                    cin[4 * k + 2] = __builtin_bit_cast(float, o2);
                    cin[4 * k + 3] = __builtin_bit_cast(float, o3);
                }
            }
#pragma unroll
            for (int c = 0; c < CHL; ++c) acc[0][c] += cin[c];
        }
        if constexpr (sizeof(T) == 2 && VEC == 4) {
            if ((hd & 3) != 0) {  // (uniform)
#pragma unroll
                for (int kb = 0; kb < NB; ++kb) {
                    const int ch = my_ch + CB * kb;
                    const int sh = ch < hd ? ch - first_channel(ch) : 0;
#pragma unroll
                    for (int i = 0; i < PPG; ++i) {
                        const float v1 = acc[i][4 * kb + 1], v2 = acc[i][4 * kb + 2], v3 = acc[i][4 * kb + 3];
                        if (sh == 1) acc[i][4 * kb] = v1, acc[i][4 * kb + 1] = v2, acc[i][4 * kb + 2] = v3;
                        if (sh == 2) acc[i][4 * kb] = v2, acc[i][4 * kb + 1] = v3;
                        if (sh == 3) acc[i][4 * kb] = v3;
                    }
                }
            }
        }
        // ---- write the CH channels of this tile -------------------------------------------
        // (address arithmetic derived from these opaque copies stays inside this section instead of
        // occupying registers during the rounds)
        int grp_w = grp, lane_w = lane;
        asm volatile("" : "+v"(grp_w), "+v"(lane_w));
        const bool split = __builtin_amdgcn_readfirstlane((int)spare_next) != 0;  // extra lists were handed out
        // A row of the image, in four-byte steps of the caller's channel, and what becomes of four sums of it.
        auto put = [&](int px, int ch, f32x4 v) {
            float* dst = gimg + (int64_t)(it.p0 + px) * row_pitch + (int64_t)wk.h * hd + ch;
            if (px == 0) {
                // the first pixel of a tile also receives, through atomics, the right
                // halves of pairs that start on the last pixel of the previous tile
#pragma unroll
                for (int c = 0; c < 4; ++c)
                    if (ch + c < hd) unsafeAtomicAdd(dst + c, v[c]);
            } else if (sizeof(T) == 2 && direct_t) {
                // 16-bit dtypes: nobody else adds to this row, so it goes to the caller's tensor at once
                // (the fp32 image keeps only the rows that receive atomic additions)
                typedef T t4 __attribute__((ext_vector_type(4)));
                const t4 r = {from_f32<T>(v[0]), from_f32<T>(v[1]), from_f32<T>(v[2]), from_f32<T>(v[3])};
                __builtin_nontemporal_store(r, reinterpret_cast<t4*>(static_cast<T*>(a.grad_value_t) + (size_t)wk.b * (a.gbatch_bytes / 4) +
                                                                     (dst - gimg)));
            } else if (t.store_vec == 4) {
                if (t.accumulate) v += *reinterpret_cast<f32x4*>(dst);
                // (non-temporal: nothing reads these rows again before the kernel ends; backward 283.8 ->
                //  281.3 us at the encoder shape)
                __builtin_nontemporal_store(v, reinterpret_cast<f32x4*>(dst));
            } else {
                typedef f32x4 __attribute__((aligned(4))) any4;  // (rows start anywhere)
                if (t.accumulate) {
                    for (int c = 0; c < 4 && ch + c < hd; ++c) dst[c] += v[c];
                } else if (ch + 4 <= hd) {
                    *reinterpret_cast<any4*>(dst) = v;
                } else {
                    for (int c = 0; c < 4 && ch + c < hd; ++c) dst[c] = v[c];
                }
            }
        };
        if (owned && copies == 1 && !split && t.store_vec == 4) {
            // the lanes of a group hold a whole row of each of their pixels: 16-byte stores
#pragma unroll
            for (int c4 = 0; c4 < CHL; c4 += 4) {
                const int ch_w = my_ch + CB * (c4 / PIECE) + c4 % PIECE;
                if (ch_w >= hd) continue;
#pragma unroll
                for (int i = 0; i < PPG; ++i) {
                    const int px = grp_w * PPG + i;
                    if (px < npx) put(px, ch_w, f32x4{acc[i][c4], acc[i][c4 + 1], acc[i][c4 + 2], acc[i][c4 + 3]});
                }
            }
        } else {
            // Through LDS (the entry storage, free after the last round): the copies of a small tile and the extra lists of
            // hot pixels are added up there, so that a tile that no other workgroup touches is stored like any other and one
            // that several share costs one atomic addition per row and not one per copy.  (Atomics are what the write-out waits for, 64
            // bytes in some 22 clocks of a CU: with one per copy a tile of 152 pixels in two took 9.5 of its item's 19 us, the last of the
            // launch -- 2 x 900 queries of 16 samples in float32 31.6 -> 25.8 us.)  They are carried out per 64-byte request, so
            // consecutive lanes hold consecutive floats there.
            typedef f32x4 __attribute__((may_alias)) f32x4_alias;
            typedef float __attribute__((may_alias)) f32_alias;
            f32x4_alias* sums4 = reinterpret_cast<f32x4_alias*>(ent);
            const f32_alias* sums1 = reinterpret_cast<const f32_alias*>(ent);
            constexpr int QR = CH / 4;  // quads of a row
            __syncthreads();            // (the sums handed over have been read)
#pragma unroll
            for (int i = 0; i < PPG; ++i)
#pragma unroll
                for (int c4 = 0; c4 < CHL; c4 += 4)
                    sums4[(grp_w * PPG + i) * QR + (CB * (c4 / PIECE) + c4 % PIECE + PIECE * j) / 4] =
                        f32x4{acc[i][c4], acc[i][c4 + 1], acc[i][c4 + 2], acc[i][c4 + 3]};
            __syncthreads();
            const int tid_w = wave * kWave + lane_w;
            // every slot that stands for pixel px of the tile
            auto each_slot = [&](int px, auto take) {
                for (int c = 0, slot = px; c < copies; ++c, slot += npx_pad) {
                    take(slot);
                    if (split) {
                        const uint32_t o = slot_info16[slot];
                        for (uint32_t r = 0; r < (o >> 9); ++r)
                            if ((o & 511u) + r < (uint32_t)nspare) take(nused + (int)((o & 511u) + r));
                    }
                }
            };
            if (owned) {
                for (int i = tid_w; i < npx * QR; i += kTileThreads) {
                    const int px = i / QR, q4 = i % QR;
                    if (4 * q4 >= nch) continue;
                    f32x4 v = {0.f, 0.f, 0.f, 0.f};
                    each_slot(px, [&](int slot) { v += sums4[slot * QR + q4]; });
                    put(px, cb + 4 * q4, v);
                }
            } else {
#pragma unroll 2
                for (int i = tid_w; i < npx * CH; i += kTileThreads) {
                    const int px = i / CH, c = i % CH;
                    if (c >= nch) continue;
                    float v = 0.0f;
                    each_slot(px, [&](int slot) { v += sums1[slot * CH + c]; });
                    unsafeAtomicAdd(gimg + (int64_t)(it.p0 + px) * row_pitch + (int64_t)wk.h * hd + cb + c, v);
                }
            }
            __syncthreads();
        }
        if (cb + CH < hd) clean_state();
    }
}

template <typename T>
static hipError_t launch_t(const KArgs& a, const TileArgs& t, hipStream_t stream)
{
    // A load brings 16 bytes per lane, or 8 of 16-bit rows that pieces of 16 do not divide; one load per lane and piece whatever the
    // row's length and alignment (but for 16-bit rows of fewer than 4 channels).
    const dim3 grid(t.grid), block(t.block);
    constexpr bool kHalf = sizeof(T) == 2;
    auto launch = [&](auto lpg, auto chl, auto vec) {
        hipLaunchKernelGGL((msda_gradv_tiles_kernel<T, decltype(lpg)::value, decltype(chl)::value, decltype(vec)::value>), grid, block, 0, stream, a, t);
    };
    constexpr std::integral_constant<int, 1> one;
    constexpr std::integral_constant<int, 4> four;
    constexpr std::integral_constant<int, 8> eight;
    constexpr std::integral_constant<int, 16> sixteen;
    if constexpr (kHalf) {
        if (a.hd < 4) {
            if (a.tile_px_log2 != kTilePxLog2Max) return hipErrorInvalidConfiguration;
            launch(eight, four, one);
            return hipGetLastError();
        }
        if (a.hd % 8 == 0) {
            if (a.tile_px_log2 == 8) launch(eight, eight, eight);
            else if (a.tile_px_log2 == 7) launch(eight, sixteen, eight);
            else launch(four, eight, eight);
            return hipGetLastError();
        }
    }
    if (a.tile_px_log2 == 8) launch(eight, eight, four);
    else if (a.tile_px_log2 == 7) launch(sixteen, eight, four);
    else launch(eight, four, four);
    return hipGetLastError();
}

hipError_t launch_gradv_tiles(int dtype, const KArgs& a, const TileArgs& t, hipStream_t stream)
{
    switch (dtype) {
        case MXD_DTYPE_F32: return launch_t<float>(a, t, stream);
        case MXD_DTYPE_F16: return launch_t<f16_t>(a, t, stream);
        case MXD_DTYPE_BF16: return launch_t<bf16_t>(a, t, stream);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace mxd
