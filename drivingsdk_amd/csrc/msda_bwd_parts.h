// What the two first backward kernels of multi-scale deformable attention (msda_bwd_kernel.h, msda_bwd_pass.h) have in common, sample by
// sample and at the ends of a workgroup's work.
#pragma once
#include "msda_device.h"

namespace mxd {

// The pair records of a sample for the tile pass: [0] of its upper corners, [1] of its lower ones.  ok: the sample counts and its
// level has tiles.
__device__ inline void pair_records(const Sample& sm, float aw, bool ok, bool (&have)[2], int32_t (&key)[2], float (&wa)[2], float (&wb)[2])
{
#pragma unroll
    for (int r = 0; r < 2; ++r) {
        const bool vl = sm.cvalid[2 * r], vr = sm.cvalid[2 * r + 1];
        have[r] = ok && (vl || vr);
        key[r] = vl ? sm.pix[2 * r] : sm.pix[2 * r + 1];
        wa[r] = (vl ? sm.w[2 * r] : sm.w[2 * r + 1]) * aw;
        wb[r] = (vl && vr) ? sm.w[2 * r + 1] * aw : 0.0f;
    }
}

// Exclusive prefix over a workgroup's counters of records per tile, 64 at a time by one wavefront; put(i, start) for each.
template <typename F>
__device__ inline void scan_counters(const int32_t* counters, int32_t n, int lane, F put)
{
    int32_t carry = 0;
    for (int base = 0; base < n; base += kWave) {
        const int i = base + lane;
        const int32_t v = i < n ? counters[i] : 0;
        int32_t inc = v;
#pragma unroll
        for (int d = 1; d < kWave; d <<= 1) {
            const int32_t o = __shfl_up(inc, d, kWave);
            if (lane >= d) inc += o;
        }
        if (i < n) put(i, carry + inc - v);
        carry += __builtin_amdgcn_readlane(inc, kWave - 1);
    }
}

// A slab as it lies in LDS: 16 bytes per lane, then the odd words.  (Non-temporal: the records are read by the next kernel and should not
// push value rows out of L2)
typedef uint32_t __attribute__((may_alias)) u32_alias;
__device__ inline void store_slab(const u32_alias* words, int n, __amdgpu_buffer_rsrc_t slab, int tid, int threads)
{
    const int quads = n >> 2;
    for (int i = tid; i < quads; i += threads)
        __builtin_amdgcn_raw_buffer_store_b128(u32x4{words[4 * i], words[4 * i + 1], words[4 * i + 2], words[4 * i + 3]}, slab, (uint32_t)i * 16u, 0, 2);
    for (int i = 4 * quads + tid; i < n; i += threads) __builtin_amdgcn_raw_buffer_store_b32(words[i], slab, (uint32_t)i * 4u, 0, 2);
}

// Fused form: chain rule through location = reference + offset * scale.  Stores the gradient of the offset pair and returns that of the
// reference point, (x, y) or a box's (x, y, w, h).  offset(k): the raw offset's element k.
template <typename T, typename F>
__device__ inline f32x4 offset_gradient(const KArgs& a, const T* rp, float Wf, float Hf, float gx, float gy, T* goff, F offset)
{
    if (a.ref_dim == 2) {
        goff[0] = from_f32<T>(gx / Wf);
        goff[1] = from_f32<T>(gy / Hf);
        return f32x4{gx, gy, 0.0f, 0.0f};
    }
    goff[0] = from_f32<T>(gx / (float)a.np * to_f32(rp[2]) * 0.5f);
    goff[1] = from_f32<T>(gy / (float)a.np * to_f32(rp[3]) * 0.5f);
    return f32x4{gx, gy, gx * (offset(0) / (float)a.np * 0.5f), gy * (offset(1) / (float)a.np * 0.5f)};
}

// Where a head's part of the gradient of the reference point of (query q, level l) is kept: the points of a level share it and are summed
// by the first kernel, into a float32 image per head that a small kernel adds up over the heads.
__device__ inline float* reference_part(const KArgs& a, int b, int h, int q, int l)
{
    return a.grad_ref + (((int64_t)h * a.bs + b) * a.nq + q) * (a.nl * a.ref_dim) + l * a.ref_dim;
}

// Sum over the points of a level across lanes, for numbers of points that are powers of two (KArgs::np_pow2); point 0 stores it.
__device__ inline void store_reference_sum(const KArgs& a, float* part, int s, f32x4 r)
{
    float gx = r.x, gy = r.y, r2 = r.z, r3 = r.w;
    for (int d = 1; d < a.np; d <<= 1) {
        gx += __shfl_xor(gx, d, kWave);
        gy += __shfl_xor(gy, d, kWave);
        r2 += __shfl_xor(r2, d, kWave);
        r3 += __shfl_xor(r3, d, kWave);
    }
    if ((s & (a.np - 1)) == 0) {
        part[0] = gx;
        part[1] = gy;
        if (a.ref_dim == 4) {
            part[2] = r2;
            part[3] = r3;
        }
    }
}

// Slots of levels that attention_weights carries beyond spatial_shapes: zero gradients for the `queries` from q0 on.
template <typename T>
__device__ inline void zero_extra_slots(const KArgs& a, int b, int h, int q0, int q_end, int queries, int lane, T* gattn, T* gloc)
{
    const int extra = a.S_full - a.S;
    if (extra > 0) {
        for (int i = lane; i < queries * extra; i += kWave) {
            const int u = i / extra, s = a.S + i % extra, q = q0 + u;
            if (q < q_end) {
                const int64_t e = (((int64_t)b * a.nq + q) * a.nh + h) * a.S_full + s;
                gattn[e] = from_f32<T>(0.f);
                gloc[2 * e] = from_f32<T>(0.f);
                gloc[2 * e + 1] = from_f32<T>(0.f);
            }
        }
    }
}

}  // namespace mxd
