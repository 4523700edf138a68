// mh_sample.h -- sample_token's sampling branch (reference csrc/src/sampler.cpp:30-78) on one
// 256-thread workgroup, shared by the sampler kernels and the fused local half (gfx950).
//
// What bounds it is a chain, not work: 1024 values have to be ordered, and the reference's sums
// over the ordered candidates are serial fp32 chains whose order is part of the result.
//  * Ordering in registers: lanes exchange keys by DPP / permlane swaps, so a compare-exchange
//    step has no LDS round trip and no barrier.  Up to 64 candidates (every top_k in use) only
//    the 64 smallest keys are kept: each wave sorts its four 64-key runs and merges them by
//    min of an ascending and a descending run, then every wave merges the four waves' runs --
//    one barrier.  Beyond 64 the 1024 keys are sorted whole (three exchange rounds in LDS).
//  * A serial chain x_i = x_(i-1) + e_i over the lanes of a wave: n rounds of "add the left
//    neighbour's x" (one DPP add each).  Round i makes lane i final, later rounds leave it
//    unchanged, so every lane ends with exactly the serial prefix.
#pragma once
#include "mh_device.h"

namespace mh {

struct SampleLds {
    uint64_t keys[kCodebook];  // sort keys: value descending, index ascending
    float ex[kCodebook];       // more than 64 candidates: exp(v - max) in sorted order,
    float pre[kCodebook];      //   and its serial prefix sums
    int pick;
};

// Order-preserving map of a float to uint32 (larger float -> larger key), and back.
__device__ __forceinline__ uint32_t float_order(float f) {
    const uint32_t u = __float_as_uint(f);
    return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}
__device__ __forceinline__ float float_unorder(uint32_t o) {
    return __uint_as_float((o & 0x80000000u) ? (o & 0x7fffffffu) : ~o);
}
__device__ __forceinline__ float key_value(uint64_t k) { return float_unorder(~(uint32_t)(k >> 32)); }

template <int M>
__device__ __forceinline__ uint64_t xshfl64(uint64_t v) {
    const uint32_t lo = (uint32_t)xshfl<M>((int)(uint32_t)v), hi = (uint32_t)xshfl<M>((int)(uint32_t)(v >> 32));
    return ((uint64_t)hi << 32) | lo;
}

// One compare-exchange with lane ^ M (the keys are all different).
template <int M>
__device__ __forceinline__ void key_cx(uint64_t &k, bool keep_min) {
    const uint64_t o = xshfl64<M>(k);
    k = ((k < o) == keep_min) ? k : o;
}

// A bitonic run of 64 keys, one per lane, into ascending (or descending) order: the last M .. 1.
template <int M, int R>
__device__ __forceinline__ void key_merge(uint64_t (&k)[R], int lane, const bool (&desc)[R]) {
#pragma unroll
    for (int r = 0; r < R; ++r) key_cx<M>(k[r], ((lane & M) == 0) != desc[r]);
    if constexpr (M > 1) key_merge<M / 2, R>(k, lane, desc);
}
// R independent bitonic sorts of 64 keys each.
template <int S, int R>
__device__ __forceinline__ void key_sort(uint64_t (&k)[R], int lane, const bool (&desc)[R]) {
    if constexpr (S > 2) key_sort<S / 2, R>(k, lane, desc);
    bool d[R];
#pragma unroll
    for (int r = 0; r < R; ++r) d[r] = ((lane & S) != 0) != desc[r];  // S == 64: bit never set
    key_merge<S / 2, R>(k, lane, d);
}
__device__ __forceinline__ uint64_t key_min(uint64_t a, uint64_t b) { return a < b ? a : b; }
__device__ __forceinline__ void key_cx_own(uint64_t &a, uint64_t &b, bool up) {
    const bool swap = (b < a) == up;
    const uint64_t x = a;
    a = swap ? b : a;
    b = swap ? x : b;
}

// Lane i < n ends with ((e_0 + e_1) + ...) + e_i, summed serially (n rounds, rounded up to 8).
__device__ __forceinline__ float serial_prefix(float e, int n) {
#pragma clang fp contract(off)
    float x = 0.0f;
    for (int i = 0; i < n; i += 8)
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            // wave_shr:1, the first lane reads 0
            const float left = __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x138, 0xF, 0xF, true));
            x = left + e;
        }
    return x;
}
__device__ __forceinline__ float lane_value(float v, int lane) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane));
}

// Softmax over the n sorted candidates (lane i holds candidate i's key), the top-p cut and the
// draw u walked down them (sampler.cpp:43-78), by one wave; n <= 64.
__device__ __forceinline__ int sample_walk64(uint64_t key, int n, const SampleCfg &c, float u) {
#pragma clang fp contract(off)
    const int lane = threadIdx.x & 63;
    const float v = key_value(key);
    const float ex = lane < n ? expf(v - lane_value(v, 0)) : 0.0f;
    const float pre = serial_prefix(ex, n);
    float sum = lane_value(pre, n - 1);
    int cnt = n;
    if (c.top_p < 1.0f) {
        const float cum = serial_prefix(ex / sum, n);
        const uint64_t over = __ballot(lane < n && cum >= c.top_p);
        if (over) cnt = __builtin_ctzll(over) + 1;
        sum = lane_value(pre, cnt - 1);
    }
    const float r0 = u * sum;
    const float r = serial_prefix(lane == 0 ? r0 - ex : -ex, cnt);
    const uint64_t done = __ballot(lane < cnt && r <= 0.0f);
    return __builtin_amdgcn_readlane((int)(uint32_t)key, done ? __builtin_ctzll(done) : cnt - 1);
}

// The same for any n, 64 candidates at a time with the serial chains carried over, by one wave
// from the sorted keys in LDS.
__device__ __forceinline__ int sample_walk(SampleLds &L, int n, const SampleCfg &c, float u) {
#pragma clang fp contract(off)
    const int lane = threadIdx.x & 63;
    const float maxv = key_value(L.keys[0]);
    float carry = 0.0f;
    for (int b = 0; b < n; b += 64) {
        const float ex = b + lane < n ? expf(key_value(L.keys[b + lane]) - maxv) : 0.0f;
        const float pre = serial_prefix(lane == 0 ? carry + ex : ex, 64);
        L.ex[b + lane] = ex;
        L.pre[b + lane] = pre;
        carry = lane_value(pre, min(n - b, 64) - 1);
    }
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
    float sum = carry;
    int cnt = n;
    if (c.top_p < 1.0f) {
        carry = 0.0f;
        for (int b = 0; b < n; b += 64) {
            const float p = L.ex[b + lane] / sum;
            const float cum = serial_prefix(lane == 0 ? carry + p : p, 64);
            const uint64_t over = __ballot(b + lane < n && cum >= c.top_p);
            if (over) {
                cnt = b + __builtin_ctzll(over) + 1;
                break;
            }
            carry = lane_value(cum, 63);
        }
        sum = L.pre[cnt - 1];
    }
    carry = u * sum;
    for (int b = 0; b < cnt; b += 64) {
        const float ex = L.ex[b + lane];
        const float r = serial_prefix(lane == 0 ? carry - ex : -ex, 64);
        const uint64_t done = __ballot(b + lane < cnt && r <= 0.0f);
        if (done) return (int)(uint32_t)L.keys[b + __builtin_ctzll(done)];
        carry = lane_value(r, 63);
    }
    return (int)(uint32_t)L.keys[cnt - 1];
}

// One draw from 1024 penalised logits: temperature, top-k, softmax, top-p, the walk.  Thread t
// holds the values of indices t + 256 k; the pick returns in every thread.  `u` is the draw
// (rng_uniform), made by the caller.  Calls on the same L are separated by a barrier.
__device__ __forceinline__ int pick_sampled(const float (&vals)[kCodebook / 256], const SampleCfg &c, float u,
                                            SampleLds &L) {
#pragma clang fp contract(off)
    static_assert(kCodebook == 1024, "four keys per thread");
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const bool scale = c.temperature > 0.0f && c.temperature != 1.0f;
    const float inv = scale ? 1.0f / c.temperature : 1.0f;
    uint64_t k[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const float v = scale ? vals[r] * inv : vals[r];
        k[r] = ((uint64_t)(~float_order(v)) << 32) | (uint32_t)(t + 256 * r);
    }
    const int n = c.top_k > 0 ? (c.top_k < kCodebook ? c.top_k : kCodebook) : kCodebook;
    if (n <= 64) {  // (uniform)
        const bool alt[4] = {false, true, false, true};
        key_sort<64, 4>(k, lane, alt);
        uint64_t m2[2] = {key_min(k[0], k[1]), key_min(k[2], k[3])};
        const bool alt2[2] = {false, true};
        key_merge<32, 2>(m2, lane, alt2);
        uint64_t m1[1] = {key_min(m2[0], m2[1])};
        const bool odd[1] = {(wave & 1) != 0};
        key_merge<32, 1>(m1, lane, odd);
        L.keys[64 * wave + lane] = m1[0];
        __syncthreads();
        m2[0] = key_min(L.keys[lane], L.keys[64 + lane]);
        m2[1] = key_min(L.keys[128 + lane], L.keys[192 + lane]);
        key_merge<32, 2>(m2, lane, alt2);
        m1[0] = key_min(m2[0], m2[1]);
        const bool up[1] = {false};
        key_merge<32, 1>(m1, lane, up);
        return sample_walk64(m1[0], n, c, u);  // every wave for itself
    }
    // all 1024: position p = 4 t + r
    for (int s = 2; s <= kCodebook; s <<= 1)
        for (int j = s >> 1; j > 0; j >>= 1) {
            if (j >= 256) {  // another wave's keys
#pragma unroll
                for (int r = 0; r < 4; ++r) L.keys[4 * t + r] = k[r];
                __syncthreads();
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int p = 4 * t + r;
                    const uint64_t o = L.keys[p ^ j];
                    k[r] = ((k[r] < o) == (((p & j) == 0) == ((p & s) == 0))) ? k[r] : o;
                }
                __syncthreads();
            } else if (j >= 4) {
                const bool mn = (((4 * t) & j) == 0) == (((4 * t) & s) == 0);
#pragma unroll
                for (int r = 0; r < 4; ++r) switch (j) {
                        case 4: key_cx<1>(k[r], mn); break;
                        case 8: key_cx<2>(k[r], mn); break;
                        case 16: key_cx<4>(k[r], mn); break;
                        case 32: key_cx<8>(k[r], mn); break;
                        case 64: key_cx<16>(k[r], mn); break;
                        default: key_cx<32>(k[r], mn); break;
                    }
            } else if (j == 2) {  // this thread's own keys
                key_cx_own(k[0], k[2], ((4 * t) & s) == 0);
                key_cx_own(k[1], k[3], ((4 * t + 1) & s) == 0);
            } else {
                key_cx_own(k[0], k[1], ((4 * t) & s) == 0);
                key_cx_own(k[2], k[3], ((4 * t + 2) & s) == 0);
            }
        }
#pragma unroll
    for (int r = 0; r < 4; ++r) L.keys[4 * t + r] = k[r];
    __syncthreads();
    if (wave == 0) {
        const int pick = sample_walk(L, n, c, u);
        if (lane == 0) L.pick = pick;
    }
    __syncthreads();
    return L.pick;
}

// The same from raw logits and their counts (in.cnt 0 where the penalty is 1).
__device__ __forceinline__ int pick_penalised(const PickIn &in, float pen, const SampleCfg &c, float u, SampleLds &L) {
    float v[kCodebook / 256];
#pragma unroll
    for (int k = 0; k < kCodebook / 256; ++k) v[k] = penalised(in.vals[k], in.cnt[k], pen);
    return pick_sampled(v, c, u, L);
}

}  // namespace mh
