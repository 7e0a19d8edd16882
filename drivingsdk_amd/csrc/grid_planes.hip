// 2-D grid sampler on planes for gfx950 (MI355X), wave64: forward and backward of NCHW tensors.
//
// The channel-last kernels (msda_fwd.hip, msda_bwd_kernel.h, msda_bwd_tiles.hip with kSrcGrid) gather rows of channels; an NCHW
// caller had to transpose the input, the result and, for the backward, grad_out and the gradient: 480 of the 668 us that forward
// and backward of [24, 128, 64, 176] -> [24, 128, 24, 176], float32, took.
//
// What bounds it: memory.  Every plane is read once (138 MB of maps at that size) and every result written once.  A plane is
// small (45 KB), so a workgroup puts one, or several small ones, into LDS with coalesced loads, and what the sampling scatters is
// LDS addresses: four 4-byte reads per output pixel and channel in the forward and in the gradient of the grid, four LDS
// additions in the gradient of the maps.  Planes of one image share their sampling points: a thread computes the geometry of an
// output pixel once for all the planes at hand.
//
// The gradient of the grid is a sum over the channels: a workgroup takes a range of output pixels and a chunk of the channels,
// stages the planes one after another (several at a time where they are small) and keeps the sums of its pixels in registers;
// chunks are added up by a kernel of its own.  The gradient of the maps needs all output pixels of a plane and the gradient of the
// grid many channels of a pixel: two kinds of workgroups of one launch, which read grad_out twice (a fifth of what moves) -- or, where
// a plane with its sums leaves a CU room for one workgroup anyway, one kind that does both plane by plane.
//
// Measured at that size: forward 39 us (190 MB, 4.9 TB/s: the rate of a copy), both gradients by two kinds of workgroups 122 us (400 MB,
// 3.3 TB/s), by one 82; in float16 109 and 70 us.  Small calls ([24, 128, 16, 20] -> 12 x 20) take 5 and 9 us.
#include "grid_planes.h"

namespace mxd {

namespace {

template <typename T>
struct Piece {
    static constexpr int kElems = 16 / (int)sizeof(T);
    typedef T vec_t __attribute__((ext_vector_type(16 / sizeof(T))));
    typedef vec_t mem_t __attribute__((aligned(sizeof(T))));  // a plane of odd size starts anywhere
};

// Consecutive elements on their way to LDS: request() asks for a thread's first four (kAhead) 16-byte pieces, place() stores them,
// and the rest of a stretch that is longer than that (kWhole: there is none).
template <typename T, int kAhead = 4, bool kWhole = false>
struct Stage {
    typedef typename Piece<T>::vec_t vec_t;
    typedef typename Piece<T>::mem_t mem_t;
    static constexpr int kE = Piece<T>::kElems;
    vec_t v[kAhead];

    __device__ inline void request(const T* src, int elems, int i0)
    {
        const int pieces = elems / kE, step = (int)blockDim.x;
#pragma unroll
        for (int j = 0; j < kAhead; ++j)
            if (i0 + j * step < pieces) v[j] = *reinterpret_cast<const mem_t*>(src + (int64_t)(i0 + j * step) * kE);
    }
    __device__ inline void request(const T* src, int elems) { request(src, elems, (int)threadIdx.x); }
    __device__ inline void place(const T* src, T* lds, int elems)
    {
        const int pieces = elems / kE, step = (int)blockDim.x;
        for (int i0 = (int)threadIdx.x;;) {
#pragma unroll
            for (int j = 0; j < kAhead; ++j)
                if (i0 + j * step < pieces) *reinterpret_cast<vec_t*>(lds + (i0 + j * step) * kE) = v[j];
            i0 += kAhead * step;
            if (kWhole || i0 >= pieces) break;
            request(src, elems, i0);
        }
        if constexpr (kWhole) {
            // (fewer than a piece is left: no loop, which the compiler unrolls for lengths that do not occur)
            const int i = pieces * kE + (int)threadIdx.x;
            if (i < elems) lds[i] = src[i];
        } else {
            for (int i = pieces * kE + (int)threadIdx.x; i < elems; i += step) lds[i] = src[i];
        }
    }
};

template <typename T>
__device__ inline f32x2 load_xy(const T* grid, int64_t i)
{
    typedef T pair_t __attribute__((ext_vector_type(2)));
    typedef pair_t mem_t __attribute__((aligned(sizeof(T))));
    const pair_t p = *reinterpret_cast<const mem_t*>(grid + 2 * i);
    return f32x2{to_f32<T>(p.x), to_f32<T>(p.y)};
}

__device__ inline Sample grid_sample(const GridArgs& a, f32x2 xy)
{
    return grid_geometry(xy.x, xy.y, i32x4{a.h, a.w, 0, 0}, a.h * a.w, true, a.mode);
}

// What the planes of an image share of an output pixel: {upper left corner + w + 1, which corners exist << 28} (the corner may lie a
// row and a pixel before the plane) and its place in the cell; zeros for one without a corner, and where there is no pixel (`there`).
template <typename T>
__device__ inline void pixel_geometry(const GridArgs& a, const T* grid, int at, bool there, uint32_t& corner, float& lw, float& lh)
{
    corner = 0;
    lw = lh = 0.0f;
    if (there) {
        const Sample s = grid_sample(a, load_xy(grid, at));
        uint32_t mask = 0;
#pragma unroll
        for (int j = 0; j < 4; ++j) mask |= s.cvalid[j] ? 1u << j : 0u;
        if (mask) {
            corner = (uint32_t)(s.pix[0] + a.w + 1) | mask << 28;
            lw = s.lw;
            lh = s.lh;
        }
    }
}

// Work items in the order of their numbers on every XCD (workgroups are dealt to the XCDs in turn): the splits and ranges that read
// the same planes follow each other in one L2.
__device__ inline uint32_t xcd_order(uint32_t wg, uint32_t total)
{
    const uint32_t x = wg % kNumXcd, each = total / kNumXcd, more = total % kNumXcd;
    return x * each + (x < more ? x : more) + wg / kNumXcd;
}

template <typename T>
__global__ __launch_bounds__(1024) void grid_planes_fwd_kernel(const GridArgs a)
{
    extern __shared__ __align__(16) unsigned char smem[];
    T* planes = reinterpret_cast<T*>(smem);
    const uint32_t wg = xcd_order(blockIdx.x, gridDim.x), split = wg % (uint32_t)a.splits, rest = wg / (uint32_t)a.splits;
    const int img = (int)(rest / (uint32_t)a.chunks), c0 = (int)(rest % (uint32_t)a.chunks) * a.planes;
    const int cn = c0 + a.planes <= a.c ? a.planes : a.c - c0;
    const int px = a.h * a.w, step = (int)blockDim.x;
    const int end = (int)(split + 1) * a.split_px < a.outs ? (int)(split + 1) * a.split_px : a.outs;
    const T* grid = static_cast<const T*>(a.grid) + (int64_t)img * a.outs * 2;
    T* out = static_cast<T*>(a.out) + ((int64_t)img * a.c + c0) * a.outs;
    int p = (int)split * a.split_px + (int)threadIdx.x;
    f32x2 xy = {0.f, 0.f};
    if (p < end) xy = load_xy(grid, p);
    {
        const T* src = static_cast<const T*>(a.x) + ((int64_t)img * a.c + c0) * px;
        Stage<T> st;
        st.request(src, cn * px);
        st.place(src, planes, cn * px);
    }
    __syncthreads();
    for (; p < end; p += step) {
        const Sample s = grid_sample(a, xy);
        if (p + step < end) xy = load_xy(grid, p + step);
        int at[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) at[k] = s.cvalid[k] ? s.pix[k] : 0;
        const T* plane = planes;
        T* o = out + p;
#pragma unroll 4
        for (int c = 0; c < cn; ++c, plane += px, o += a.outs) {
            // (corners outside are left out by selecting zero, whatever the pixel that is read in their place holds; the order
            //  of the sum is the channel-last kernel's, bit for bit)
            float acc = 0.0f;
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const float v = to_f32(plane[at[k]]);
                acc = __builtin_fmaf(s.w[k], s.cvalid[k] ? v : 0.0f, acc);
            }
            *o = from_f32<T>(acc);
        }
    }
}

// Forward of many planes of an image, one after the other: the geometry of the workgroup's output pixels stays in registers, and the next
// plane travels while the one at hand is sampled.  Bound by memory: 24 x 128 planes of 64 x 176, 24 x 176 samples, float32, 39 us (190 MB,
// 4.9 TB/s, a copy's rate) where a workgroup per plane took 51, half of its time in geometry.
template <typename T, int PX>
__global__ __launch_bounds__(1024, PX <= grid_run_px((int)sizeof(T)) ? 8 : 4) void grid_planes_fwd_run_kernel(const GridArgs a)
{
    extern __shared__ __align__(16) unsigned char smem[];
    constexpr int step = 2 * kGridThreads;
    const int px = a.h * a.w, first = (int)threadIdx.x;
    // (a corner outside the plane is read where it would lie, in the room left before and behind the plane)
    T* plane = reinterpret_cast<T*>(smem) + grid_margin((int)sizeof(T), a.w);
    const uint32_t wg = xcd_order(blockIdx.x, gridDim.x);
    const int img = (int)(wg / (uint32_t)a.chunks), c_begin = (int)(wg % (uint32_t)a.chunks) * a.planes;
    const int c_end = c_begin + a.planes < a.c ? c_begin + a.planes : a.c;
    const T* grid = static_cast<const T*>(a.grid) + (int64_t)img * a.outs * 2;
    const T* src = static_cast<const T*>(a.x) + ((int64_t)img * a.c + c_begin) * px;
    T* out = static_cast<T*>(a.out) + ((int64_t)img * a.c + c_begin) * a.outs;
    int wave_first = __builtin_amdgcn_readfirstlane(first & ~(kWave - 1));
    Stage<T, (int)sizeof(T) == 4 ? 3 : 2> st;
    st.request(src, px);
    uint32_t corner[PX];
    float lw[PX], lh[PX];
#pragma unroll
    for (int k = 0; k < PX; ++k) pixel_geometry(a, grid, first + k * step, first + k * step < a.outs, corner[k], lw[k], lh[k]);
    st.place(src, plane, px);
    __syncthreads();
    for (int c = c_begin + 1;; ++c, out += a.outs) {
        if (c < c_end) {
            src += px;
            st.request(src, px);
        }
        asm volatile("" : "+s"(wave_first));  // (opaque: one comparison per pixel, not nine kept)
#pragma unroll
        for (int k = 0; k < PX; ++k) {
            if (k * step + wave_first >= a.outs) break;
            asm volatile("" : "+v"(corner[k]), "+v"(lw[k]), "+v"(lh[k]));
            const int m = (int)corner[k];
            const T *r0 = plane + ((m & 0x0FFFFFFF) - a.w - 1), *r1 = r0 + a.w;
            const T r[4] = {r0[0], r0[1], r1[0], r1[1]};
            float wt[4], acc = 0.0f;
            bilinear_weights(lw[k], lh[k], wt);
#pragma unroll
            for (int j = 0; j < 4; ++j) acc = __builtin_fmaf(wt[j], m & (int)(1u << (28 + j)) ? to_f32(r[j]) : 0.0f, acc);
            if (k * step + first < a.outs) (out + k * step)[(uint32_t)first] = from_f32<T>(acc);
        }
        if (c >= c_end) break;
        __syncthreads();  // (the plane has been read)
        st.place(src, plane, px);
        __syncthreads();
    }
}

// (The float32 value is made opaque: the compiler otherwise rounds to 16 bits from float64 in some 60 instructions.)
template <typename T>
__device__ inline T from_f64(double v)
{
    float f = (float)v;
    asm("" : "+v"(f));
    return from_f32<T>(f);
}

// Gradient of the maps: a plane, a band of one, or several small ones as float64 sums in LDS.  (On gfx950 ds_add_f32 takes 190
// cycles per wavefront wherever its lanes point, ds_add_f64 9 to 26: the same additions in float32 took 242 us at the size above.)
template <typename T>
__device__ inline void grad_maps(const GridArgs& a, uint32_t wg, unsigned char* smem)
{
    double* acc = reinterpret_cast<double*>(smem);
    const int band = (int)(wg % (uint32_t)a.gx_bands);
    wg /= (uint32_t)a.gx_bands;
    const int img = (int)(wg / (uint32_t)a.gx_chunks), c0 = (int)(wg % (uint32_t)a.gx_chunks) * a.gx_planes;
    const int cn = c0 + a.gx_planes <= a.c ? a.gx_planes : a.c - c0;
    const int px = a.h * a.w, step = (int)blockDim.x;
    const int b0 = band * a.gx_band_px, bn = b0 + a.gx_band_px <= px ? a.gx_band_px : px - b0, elems = cn * bn;
    const T* grid = static_cast<const T*>(a.grid) + (int64_t)img * a.outs * 2;
    const T* grad = static_cast<const T*>(a.grad_out) + ((int64_t)img * a.c + c0) * a.outs;
    int p = (int)threadIdx.x;
    f32x2 xy = {0.f, 0.f};
    T g0 = (T)0.0f;
    if (p < a.outs) {
        xy = load_xy(grid, p);
        g0 = grad[p];
    }
    for (int i = (int)threadIdx.x; i < (elems + 1) / 2; i += step) reinterpret_cast<u32x4*>(acc)[i] = u32x4{0u, 0u, 0u, 0u};
    __syncthreads();
    for (; p < a.outs; p += step) {
        const Sample s = grid_sample(a, xy);
        T g = g0;
        const T* gp = grad + p;
        if (p + step < a.outs) {
            xy = load_xy(grid, p + step);
            g0 = gp[step];
        }
        int at[4];
        bool in[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            at[k] = s.pix[k] - b0;
            in[k] = s.cvalid[k] && (uint32_t)at[k] < (uint32_t)bn;
        }
        double* plane = acc;
        for (int c = 0;;) {
            const float gc = to_f32(g);
            if (c + 1 < cn) g = gp[(int64_t)(c + 1) * a.outs];
#pragma unroll
            for (int k = 0; k < 4; ++k)
                if (in[k]) __hip_atomic_fetch_add(plane + at[k], (double)(s.w[k] * gc), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
            if (++c == cn) break;
            plane += bn;
        }
    }
    __syncthreads();
    // (several planes are whole ones: one stretch of memory either way.  Two sums per lane: LDS gives those without bank conflicts.)
    typedef T pair_t __attribute__((ext_vector_type(2)));
    typedef pair_t mem_t __attribute__((aligned(sizeof(T))));
    typedef double f64x2 __attribute__((ext_vector_type(2)));
    T* dst = static_cast<T*>(a.grad_x) + ((int64_t)img * a.c + c0) * px + b0;
    for (int i = (int)threadIdx.x; i < elems / 2; i += step) {
        const f64x2 v = reinterpret_cast<const f64x2*>(acc)[i];
        *reinterpret_cast<mem_t*>(dst + 2 * (int64_t)i) = pair_t{from_f64<T>(v.x), from_f64<T>(v.y)};
    }
    if ((elems & 1) && threadIdx.x == 0) dst[elems - 1] = from_f64<T>(acc[elems - 1]);
}

// A pixel's sums over the channels of a chunk: into the chunk's image of sums, or, where there is one chunk, to grad_grid.
template <typename T>
__device__ inline void store_points(const GridArgs& a, int chunks, int chunk, int img, int p, float sx, float sy)
{
    const int64_t at = (int64_t)img * a.outs + p;
    if (chunks > 1) {
        reinterpret_cast<f32x2*>(a.part)[(int64_t)chunk * a.n * a.outs + at] = f32x2{sx, sy};
        return;
    }
    const Sample s = grid_sample(a, load_xy(static_cast<const T*>(a.grid), at));  // for d(pixel)/d(grid)
    T* dst = static_cast<T*>(a.grad_grid) + 2 * at;
    dst[0] = from_f32<T>(sx * s.Wf);
    dst[1] = from_f32<T>(sy * s.Hf);
}

// Gradient of the grid: PX output pixels per thread, their sums over the channels of a chunk in registers.
template <typename T, int PX>
__device__ inline void grad_points(const GridArgs& a, uint32_t wg, unsigned char* smem)
{
    T* planes = reinterpret_cast<T*>(smem);
    const int range = (int)(wg % (uint32_t)a.gg_ranges);
    const uint32_t rest = wg / (uint32_t)a.gg_ranges;
    const int chunk = (int)(rest % (uint32_t)a.gg_chunks), img = (int)(rest / (uint32_t)a.gg_chunks);
    const int c_begin = chunk * a.gg_channels, c_end = c_begin + a.gg_channels < a.c ? c_begin + a.gg_channels : a.c;
    const int px = a.h * a.w, step = (int)blockDim.x, first = range * a.gg_px * step + (int)threadIdx.x;
    const T* grid = static_cast<const T*>(a.grid) + (int64_t)img * a.outs * 2;
    const T* grad = static_cast<const T*>(a.grad_out) + (int64_t)img * a.c * a.outs;

    uint32_t corner[PX];
    float lw[PX], lh[PX], sx[PX], sy[PX];
    T g[PX];
    auto load_grad = [&](int c) {
        const T* row = grad + (int64_t)c * a.outs;
#pragma unroll
        for (int k = 0; k < PX; ++k) {
            g[k] = (T)0.0f;
            if (k < a.gg_px && k * step + first < a.outs) g[k] = (row + k * step)[(uint32_t)first];
        }
    };
#pragma unroll
    for (int k = 0; k < PX; ++k) {
        sx[k] = sy[k] = 0.0f;
        pixel_geometry(a, grid, first + k * step, k < a.gg_px && first + k * step < a.outs, corner[k], lw[k], lh[k]);
    }
    // (the next planes are requested before the ones at hand are used)
    const T* src = static_cast<const T*>(a.x) + ((int64_t)img * a.c + c_begin) * px;
    auto together = [&](int c0) { return c0 + a.gg_planes < c_end ? a.gg_planes : c_end - c0; };
    Stage<T> st;
    st.request(src, together(c_begin) * px);
    for (int c0 = c_begin; c0 < c_end; c0 += a.gg_planes) {
        const int cn = together(c0);
        load_grad(c0);
        __syncthreads();  // (the planes before these have been read)
        st.place(src, planes, cn * px);
        src += cn * px;
        __syncthreads();
        if (c0 + cn < c_end) st.request(src, together(c0 + cn) * px);
        const T* plane = planes;
        for (int c = 0; c < cn; ++c, plane += px) {
            float gc[PX];
#pragma unroll
            for (int k = 0; k < PX; ++k) gc[k] = to_f32(g[k]);
            if (c + 1 < cn) load_grad(c0 + c + 1);
#pragma unroll
            for (int k = 0; k < PX; ++k) {
                // (opaque: what follows from it would otherwise be kept for all pixels across the channels, which does not fit)
                asm volatile("" : "+v"(corner[k]));
                const uint32_t m = corner[k] >> 28;
                const int p = (int)(corner[k] & 0x0FFFFFFFu) - a.w - 1;
                float v00 = to_f32(plane[m & 1 ? p : 0]), v01 = to_f32(plane[m & 2 ? p + 1 : 0]);
                float v10 = to_f32(plane[m & 4 ? p + a.w : 0]), v11 = to_f32(plane[m & 8 ? p + a.w + 1 : 0]);
                v00 = m & 1 ? v00 : 0.0f;
                v01 = m & 2 ? v01 : 0.0f;
                v10 = m & 4 ? v10 : 0.0f;
                v11 = m & 8 ? v11 : 0.0f;
                const float dx = __builtin_fmaf(lh[k], v11 - v10, (1.0f - lh[k]) * (v01 - v00));
                const float dy = __builtin_fmaf(lw[k], v11 - v01, (1.0f - lw[k]) * (v10 - v00));
                sx[k] = __builtin_fmaf(gc[k], dx, sx[k]);
                sy[k] = __builtin_fmaf(gc[k], dy, sy[k]);
            }
        }
    }
#pragma unroll
    for (int k = 0; k < PX; ++k) {
        const int p = first + k * step;
        if (k < a.gg_px && p < a.outs) store_points<T>(a, a.gg_chunks, chunk, img, p, sx[k], sy[k]);
    }
}

template <typename T, int PX>
__global__ __launch_bounds__(1024) void grid_planes_bwd_kernel(const GridArgs a)
{
    extern __shared__ __align__(16) unsigned char smem[];
    // (the workgroups that read much come first: the others fill up behind them)
    if ((int)blockIdx.x < a.gg_wgs) grad_points<T, PX>(a, xcd_order(blockIdx.x, (uint32_t)a.gg_wgs), smem);
    else grad_maps<T>(a, xcd_order(blockIdx.x - (uint32_t)a.gg_wgs, (uint32_t)a.gx_wgs), smem);
}

// Both gradients, of planes whose sums leave a CU room for one workgroup: a workgroup takes a chunk of an image's channels, a plane
// at a time, whose pixels and float64 sums lie in LDS side by side.  The geometry of its output pixels and the sums of the grid's
// gradient stay in registers from plane to plane; the next plane and its grad_out travel while the one at hand is worked on, and
// its sums go out, and are cleared, in the step that puts the next plane in place: two barriers per plane, grad_out read once.
// What bounds it is LDS, at work for 3.9 of some 6 us per plane of 64 x 176 and 24 x 176 output pixels; 1.2 us are the step between.
// (No VGPR may spill here, nor in the forward's runs: the build checks it.  A build of this kernel that spilled 28, in float32 with nine pixels per
//  thread, gave wrong sums; its listing had a store to the stack inside the masked end of place(), where lanes that are masked off leave theirs
//  unsaved.  Most of the registers went to place(): the loop over what does not occur here -- pieces beyond the first ones, elements behind
//  the last piece, eight at a time -- took 8 to 20 of them.  Without it: 24 x 128 planes of 64 x 176 in float32 87 -> 82 us.  grad_out is
//  kept once, and reloaded pixel by pixel.)
template <typename T, int PX>
__global__ __launch_bounds__(1024) void grid_planes_both_kernel(const GridArgs a)
{
    extern __shared__ __align__(16) unsigned char smem[];
    double* sums = reinterpret_cast<double*>(smem);
    const int px = a.h * a.w, first = (int)threadIdx.x;
    constexpr int step = 2 * kGridThreads;
    // (a corner outside the plane is read where it would lie, up to w + 1 elements before or behind: in the sums or in the room left
    //  behind the plane; it is added to a word that nobody reads, one per lane)
    T* plane = reinterpret_cast<T*>(smem + grid_sums_bytes(px));
    double* nowhere = reinterpret_cast<double*>(smem + a.lds - kWave * sizeof(double)) + (first & (kWave - 1));
    int wave_first = __builtin_amdgcn_readfirstlane(first & ~(kWave - 1));
    const uint32_t wg = xcd_order(blockIdx.x, gridDim.x);
    const int img = (int)(wg / (uint32_t)a.gb_chunks), chunk = (int)(wg % (uint32_t)a.gb_chunks);
    const int c_begin = chunk * a.gb_channels, c_end = c_begin + a.gb_channels < a.c ? c_begin + a.gb_channels : a.c;
    const T* grid = static_cast<const T*>(a.grid) + (int64_t)img * a.outs * 2;
    const T* grad = static_cast<const T*>(a.grad_out) + ((int64_t)img * a.c + c_begin) * a.outs;
    const T* src = static_cast<const T*>(a.x) + ((int64_t)img * a.c + c_begin) * px;
    T* dst = static_cast<T*>(a.grad_x) + ((int64_t)img * a.c + c_begin) * px;

    // (past the last output pixel: zero, from the buffer's bounds check)
    T g[PX];
    auto load_grad = [&](int k) {
        const int left = a.outs - k * step;
        const __amdgpu_buffer_rsrc_t row = make_rsrc(grad + k * step, left > 0 ? (uint32_t)left * (uint32_t)sizeof(T) : 0u);
        const int at = first * (int)sizeof(T);
        if constexpr (sizeof(T) == 4) g[k] = __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b32(row, at, 0, 0));
        else g[k] = __builtin_bit_cast(T, (uint16_t)__builtin_amdgcn_raw_buffer_load_b16(row, at, 0, 0));
    };
    Stage<T, (int)sizeof(T), true> st;  // (the largest plane that fits, in one go)
    static_assert(kCuLdsBytes / (8 + (int)sizeof(T)) <= (int)sizeof(T) * step * Piece<T>::kElems);
    st.request(src, px);
#pragma unroll
    for (int k = 0; k < PX; ++k) load_grad(k);
    uint32_t corner[PX];
    float lw[PX], lh[PX], sx[PX], sy[PX];
#pragma unroll
    for (int k = 0; k < PX; ++k) {
        sx[k] = sy[k] = 0.0f;
        pixel_geometry(a, grid, first + k * step, first + k * step < a.outs, corner[k], lw[k], lh[k]);
    }
    for (int i = first; i < (px + 1) / 2; i += step) reinterpret_cast<u32x4*>(sums)[i] = u32x4{0u, 0u, 0u, 0u};
    st.place(src, plane, px);
    __syncthreads();
    for (int c = c_begin + 1;; ++c) {
        if (c < c_end) {
            src += px;
            grad += a.outs;
            st.request(src, px);
        }
        T r[2][4];
        int at[2];
        auto read = [&](int k) {
            // (opaque: what follows from it would otherwise be kept for all pixels across the channels, which does not fit)
            asm volatile("" : "+v"(corner[k]), "+v"(lw[k]), "+v"(lh[k]));
            at[k & 1] = (int)(corner[k] & 0x0FFFFFFFu) - a.w - 1;
            const T *r0 = plane + at[k & 1], *r1 = r0 + a.w;
            r[k & 1][0] = r0[0];
            r[k & 1][1] = r0[1];
            r[k & 1][2] = r1[0];
            r[k & 1][3] = r1[1];
        };
        asm volatile("" : "+s"(wave_first));  // (opaque: one comparison per pixel, not nine kept)
        read(0);
#pragma unroll
        for (int k = 0; k < PX; ++k) {
            if (k + 1 < PX) read(k + 1);
            if (k * step + wave_first >= a.outs) break;
            const int m = (int)corner[k], p = at[k & 1];
            const float gc = to_f32(g[k]);
            bool in[4];
            float v[4], wt[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                in[j] = (m & (int)(1u << (28 + j))) != 0;
                v[j] = in[j] ? to_f32(r[k & 1][j]) : 0.0f;
            }
            const float dx = __builtin_fmaf(lh[k], v[3] - v[2], (1.0f - lh[k]) * (v[1] - v[0]));
            const float dy = __builtin_fmaf(lw[k], v[3] - v[1], (1.0f - lw[k]) * (v[2] - v[0]));
            sx[k] = __builtin_fmaf(gc, dx, sx[k]);
            sy[k] = __builtin_fmaf(gc, dy, sy[k]);
            // (opaque: the sums would otherwise be formed behind the last pixel, from the rows of all pixels kept in registers)
            asm volatile("" : "+v"(sx[k]), "+v"(sy[k]));
            bilinear_weights(lw[k], lh[k], wt);
            const int to[4] = {p, p + 1, p + a.w, p + a.w + 1};
            // (no branches: behind one, the wait for a pixel's four values is one for the additions of the pixel before it as well,
            //  110 us instead of 93 at the size above before the registers were trimmed)
#pragma unroll
            for (int j = 0; j < 4; ++j)
                __hip_atomic_fetch_add(in[j] ? sums + to[j] : nowhere, (double)(wt[j] * gc), __ATOMIC_RELAXED,
                                       __HIP_MEMORY_SCOPE_WORKGROUP);
            if (c < c_end) load_grad(k);  // (of the next channel)
            __builtin_amdgcn_sched_barrier(0);  // (one pixel ahead, no more: the registers are full)
        }
        __syncthreads();
        if (c < c_end) {
            // (waited for here, and not behind the stores that come next: loads and stores return in order)
#pragma unroll
            for (int k = 0; k < PX; ++k) asm volatile("" ::"v"(g[k]));
            st.place(src, plane, px);
        }
        // (two sums per lane: LDS gives those without bank conflicts)
        typedef T pair_t __attribute__((ext_vector_type(2)));
        typedef pair_t mem_t __attribute__((aligned(sizeof(T))));
        typedef double f64x2 __attribute__((ext_vector_type(2)));
        for (int i = first; i < px / 2; i += step) {
            const f64x2 v = reinterpret_cast<const f64x2*>(sums)[i];
            reinterpret_cast<f64x2*>(sums)[i] = f64x2{0.0, 0.0};
            *reinterpret_cast<mem_t*>(dst + 2 * (int64_t)i) = pair_t{from_f64<T>(v.x), from_f64<T>(v.y)};
        }
        if ((px & 1) && first == 0) {
            dst[px - 1] = from_f64<T>(sums[px - 1]);
            sums[px - 1] = 0.0;
        }
        if (c >= c_end) break;
        dst += px;
        __syncthreads();
    }
    int mine = first;
    asm volatile("" : "+v"(mine));  // (opaque: as above)
#pragma unroll
    for (int k = 0; k < PX; ++k) {
        const int p = mine + k * step;
        if (p < a.outs) store_points<T>(a, a.gb_chunks, chunk, img, p, sx[k], sy[k]);
    }
}

// Sum over the channel chunks: 32 output pixels per workgroup, 8 threads that share the chunks of each.
template <typename T>
__global__ __launch_bounds__(256) void grid_planes_sum_kernel(const GridArgs a)
{
    __shared__ f32x2 sums[8][32];
    const int64_t total = (int64_t)a.n * a.outs, i = (int64_t)blockIdx.x * 32 + (threadIdx.x & 31);
    const int row = (int)threadIdx.x >> 5;
    f32x2 sum = {0.f, 0.f};
    if (i < total) {
        const f32x2* part = reinterpret_cast<const f32x2*>(a.part) + i;
#pragma unroll 4
        for (int c = row; c < a.sum_chunks; c += 8) sum += part[c * total];
    }
    sums[row][threadIdx.x & 31] = sum;
    __syncthreads();
    if (row != 0 || i >= total) return;
#pragma unroll
    for (int r = 1; r < 8; ++r) sum += sums[r][threadIdx.x];
    const Sample s = grid_sample(a, load_xy(static_cast<const T*>(a.grid), i));
    T* dst = static_cast<T*>(a.grad_grid) + 2 * i;
    dst[0] = from_f32<T>(sum.x * s.Wf);
    dst[1] = from_f32<T>(sum.y * s.Hf);
}

template <typename F>
hipError_t by_pixels(int px, F f)
{
    if (px <= 1) return f(std::integral_constant<int, 1>{});
    if (px <= 3) return f(std::integral_constant<int, 3>{});
    if (px <= 6) return f(std::integral_constant<int, 6>{});
    if (px <= kGridMaxPx) return f(std::integral_constant<int, kGridMaxPx>{});
    return hipErrorInvalidConfiguration;
}

template <typename T>
hipError_t raise_t()
{
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&grid_planes_fwd_kernel<T>), hipFuncAttributeMaxDynamicSharedMemorySize,
                                       kCuLdsBytes);
    for (int px : {1, 3, 6, kGridMaxPx})
        if (e == hipSuccess)
            e = by_pixels(px, [](auto p) {
                hipError_t r = hipFuncSetAttribute(reinterpret_cast<const void*>(&grid_planes_bwd_kernel<T, decltype(p)::value>),
                                                   hipFuncAttributeMaxDynamicSharedMemorySize, kCuLdsBytes);
                if (r == hipSuccess)
                    r = hipFuncSetAttribute(reinterpret_cast<const void*>(&grid_planes_both_kernel<T, decltype(p)::value>),
                                            hipFuncAttributeMaxDynamicSharedMemorySize, kCuLdsBytes);
                if (r == hipSuccess)
                    r = hipFuncSetAttribute(reinterpret_cast<const void*>(&grid_planes_fwd_run_kernel<T, decltype(p)::value>),
                                            hipFuncAttributeMaxDynamicSharedMemorySize, kCuLdsBytes);
                return r;
            });
    return e;
}

template <typename T>
hipError_t forward_t(const GridArgs& a, hipStream_t stream)
{
    if (a.run_px)
        return by_pixels(a.run_px, [&](auto p) {
            hipLaunchKernelGGL((grid_planes_fwd_run_kernel<T, decltype(p)::value>), dim3((unsigned)a.n * a.chunks), dim3(a.block), a.lds,
                               stream, a);
            return hipGetLastError();
        });
    hipLaunchKernelGGL(grid_planes_fwd_kernel<T>, dim3((unsigned)a.n * a.chunks * a.splits), dim3(a.block), a.lds, stream, a);
    return hipGetLastError();
}

template <typename T>
hipError_t backward_t(const GridArgs& a, hipStream_t stream)
{
    hipError_t e;
    if (a.gb_wgs) {
        e = by_pixels(a.gb_px, [&](auto p) {
            hipLaunchKernelGGL((grid_planes_both_kernel<T, decltype(p)::value>), dim3((unsigned)a.gb_wgs), dim3(a.block), a.lds, stream, a);
            return hipGetLastError();
        });
    } else {
        e = by_pixels(a.gg_px, [&](auto p) {
            hipLaunchKernelGGL((grid_planes_bwd_kernel<T, decltype(p)::value>), dim3((unsigned)(a.gx_wgs + a.gg_wgs)), dim3(a.block), a.lds,
                               stream, a);
            return hipGetLastError();
        });
    }
    if (e != hipSuccess || a.sum_chunks <= 1) return e;
    const int64_t total = (int64_t)a.n * a.outs;
    hipLaunchKernelGGL(grid_planes_sum_kernel<T>, dim3((unsigned)((total + 31) / 32)), dim3(256), 0, stream, a);
    return hipGetLastError();
}

}  // namespace

hipError_t raise_grid_lds()
{
    hipError_t e = raise_t<float>();
    if (e == hipSuccess) e = raise_t<f16_t>();
    if (e == hipSuccess) e = raise_t<bf16_t>();
    return e;
}

hipError_t launch_grid_planes_forward(int dtype, const GridArgs& a, hipStream_t stream)
{
    switch (dtype) {
        case MXD_DTYPE_F32: return forward_t<float>(a, stream);
        case MXD_DTYPE_F16: return forward_t<f16_t>(a, stream);
        case MXD_DTYPE_BF16: return forward_t<bf16_t>(a, stream);
        default: return hipErrorInvalidValue;
    }
}

hipError_t launch_grid_planes_backward(int dtype, const GridArgs& a, hipStream_t stream)
{
    switch (dtype) {
        case MXD_DTYPE_F32: return backward_t<float>(a, stream);
        case MXD_DTYPE_F16: return backward_t<f16_t>(a, stream);
        case MXD_DTYPE_BF16: return backward_t<bf16_t>(a, stream);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace mxd
