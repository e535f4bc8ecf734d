// zs_sampler.h -- state and helpers shared by the sampler kernels
// (zs_sample.hip: the GPU-wide big-row kernels and the output kernel;
// zs_row.hip: the one-workgroup-per-row step).
#pragma once
#include <hip/hip_runtime.h>
#include "zs_internal.h"
#include "zs_dev.h"
#include "zs_seq.h"
#include "zs_terms.h"
struct zs_sargs {
    zs_batch b;
    uint32_t* p_cnt;
    uint32_t* p_id;
    uint32_t* p_flags;
    float* p_y;
    zs_row_state* rst;
    uint32_t* pairs;
    uint32_t* pv;
    uint32_t nch;
    uint32_t max_vocab;   // stride of the scratch rows: the context's max_vocab rounded up to 4
    uint32_t* p_sub;
    uint32_t max_subs;
    double* k_ap;
    zs_sub_sum* k_sum;
    zs_sub_sum* k_xsum;  // crossing records beside k_sum (same indexing)
    zs_tp_bucket* tp_bk;
    uint32_t* tp_cl;
    uint32_t* tp_pre;
    uint32_t* kcnt;
    uint32_t* tp_task;   // buckets zs_k_tp_sort presorts: count, then (row << 8 | candidate)
    zs_sub_sum* s_rec;
    zs_sub_sum* s_xrec;  // crossing records beside s_rec (same indexing)
    float* s_apx;
    float* gath;
    float* s_hterm;
    uint32_t pstride;   // entries per row of the merged patch list (p_id, p_flags, p_y): the same stride
    uint32_t gshift;    // zs_k_scan: log2 of the ids per group (0: no scan)
    uint32_t ncu;       // CUs of the device
    uint32_t gstride;   // groups per row of gmax
    uint32_t* gmax;     // [rows][gstride] keys of the group maxima
};

#define ZS_ST_FALLBACK 0x200u

// zs_row.hip: the per-row front of the step (patches, row statistics,
// candidates, greedy and small rows)
extern "C" int zs_row_launch(const zs_sargs& a, hipStream_t stream);
// log2 of the ids per group of zs_k_scan for rows of V ids (0: no scan)
uint32_t zs_scan_gshift(uint32_t V);
// zs_sums.hip: the row sums (the big rows' sampler S; S_obs, then the
// entropy) spread over the GPU (one kernel per call, `which` 0..7)
extern "C" int zs_sums_launch(const zs_sargs& a, uint32_t which, hipStream_t stream);

__device__ __forceinline__ bool zs_penalty_active(const zs_row_params& P) {
    return P.repeat != 1.0f || P.presence != 0.0f || P.frequency != 0.0f;
}
__device__ __forceinline__ float zs_temper(float y, float T) {
    // sampler.rs:47-51: divide only when T != 1 (T > 0 here)
    return (T > 0.0f && T != 1.0f) ? y / T : y;
}
__device__ __forceinline__ bool zs_allowed_bit(const zs_batch& b, uint32_t r, uint32_t idx) {
    uint32_t w = b.d_allow_bits[(size_t)r * b.allow_words + (idx >> 5)];
    return (w >> (idx & 31)) & 1u;
}

// Small survivor sets (n <= ZS_SMALL_CAP, all other logits are -inf after
// top-k / mask) are sampled exactly in the row kernel, up to 64 by one wave
// (small_path_wave), more by the workgroup: zero terms of the reference's
// full-vocabulary loops do not change a running sum.
#define ZS_SMALL_CAP 512

// Ascending bitonic sort of 64*E u64 keys by one wave, element i = lane*E + e
// in register e of lane i / E: strides below E inside the lane, the others by
// lane exchanges.
template <int E>
__device__ __forceinline__ void wave_sort_u64_e(unsigned long long (&v)[E]) {
    const uint32_t lane = (uint32_t)zs_lane();
#pragma unroll
    for (uint32_t k = 2; k <= 64u * E; k <<= 1) {
#pragma unroll
        for (uint32_t j = k >> 1; j > 0; j >>= 1) {
            if (j < (uint32_t)E) {
#pragma unroll
                for (uint32_t e = 0; e < (uint32_t)E; e++) {
                    const uint32_t pe = e ^ j;
                    if (pe > e) {
                        const bool asc = ((lane * E + e) & k) == 0u;
                        const unsigned long long x = v[e], y = v[pe];
                        if ((x > y) == asc) { v[e] = y; v[pe] = x; }
                    }
                }
            } else {
#pragma unroll
                for (uint32_t e = 0; e < (uint32_t)E; e++) {
                    const unsigned long long o = zs_lane_xor_by(v[e], j / E);
                    const uint32_t i = lane * E + e;
                    const bool asc = (i & k) == 0u, lower = (i & j) == 0u;
                    v[e] = (lower == asc) ? (o < v[e] ? o : v[e]) : (o > v[e] ? o : v[e]);
                }
            }
        }
    }
}

#ifndef ZS_SP_T
#define ZS_SP_T(i) do { } while (0)
#endif

// The wave's values (one per lane, the first n) written to LDS scratch, for a
// serial pass.
__device__ __forceinline__ void wave_stage_f(float* buf, float v, uint32_t n) {
    const uint32_t lane = (uint32_t)zs_lane();
    if (lane < n) buf[lane] = v;
    __builtin_amdgcn_s_waitcnt(0);   // the wave's own LDS writes before its reads
    __builtin_amdgcn_wave_barrier();
}
// Index of the first element after which s0 + buf[0] + ... + buf[i] (f32,
// one addition at a time in order) reaches thresh (never for NaN); n if none.
// *s gets the sum up to and including that element (all n when none). Every
// lane runs it on the same LDS values (broadcast reads) and ends with the same
// result.
__device__ __forceinline__ uint32_t serial_scan_f(const float* buf, uint32_t n, float s0, float thresh, float* s) {
    float acc = s0;
    uint32_t i = 0;
    // 32 terms per batch of reads, their latency off the chain of additions
    // (the terms are probabilities, never negative: a running sum below
    // thresh after the batch was below it inside); the batch that reaches
    // thresh is added again below to find the element. 512 terms: 8.6 us one
    // test and one read of 4 at a time, 3 us so.
    for (; i + 32 <= n; i += 32) {
        float4 q8[8];
#pragma unroll
        for (int u = 0; u < 8; u++) q8[u] = *reinterpret_cast<const float4*>(buf + i + 4 * u);
        float c = acc;
#pragma unroll
        for (int u = 0; u < 8; u++) c = (((c + q8[u].x) + q8[u].y) + q8[u].z) + q8[u].w;
        if (c >= thresh) break;
        acc = c;
    }
    for (; i + 4 <= n; i += 4) {
        const float4 q = *reinterpret_cast<const float4*>(buf + i);
        acc = acc + q.x;
        if (acc >= thresh) { *s = acc; return i; }
        acc = acc + q.y;
        if (acc >= thresh) { *s = acc; return i + 1; }
        acc = acc + q.z;
        if (acc >= thresh) { *s = acc; return i + 2; }
        acc = acc + q.w;
        if (acc >= thresh) { *s = acc; return i + 3; }
    }
    for (; i < n; i++) {
        acc = acc + buf[i];
        if (acc >= thresh) { *s = acc; return i; }
    }
    *s = acc;
    return n;
}

// Exact sampler over a small survivor set (n <= 64, every other element below
// the top-k threshold, masked or -inf), by one wave: the reference's
// sequential f32 sums are done literally, one addition at a time in the
// reference's order, with no workgroup synchronisation (sampler.rs:46-127).
// The additions run over LDS copies of the values (sval, sidx: the survivors
// on entry, then scratch; 16-byte aligned). Called by the 64 lanes of one
// wave; returns the token on every lane.
__device__ __forceinline__ uint32_t small_path_wave(uint64_t seed, uint64_t counter, uint32_t V, const zs_row_params& P,
                                                    uint32_t n, float m, float* sval, uint32_t* sidx) {
    const uint32_t lane = (uint32_t)zs_lane();
    const bool live = lane < n;
#ifdef ZS_WALK_DEBUG
    unsigned long long sp_t0 = wall_clock64();
#endif
    // survivors by index, one per lane
    const unsigned long long key = wave_sort_u64(live ? (((unsigned long long)sidx[lane] << 32) | zs_f2u(sval[lane])) : ~0ull);
    ZS_SP_T(0);
    const uint32_t id = (uint32_t)(key >> 32);
    float p = live ? zs_expf(zs_u2f((uint32_t)key) - m) : 0.0f;
    // s0 + v of lane 0 + v of lane 1 + ... (sampler.rs:68, 80, 107)
    auto seq_sum = [&](float v, float s0) {
        wave_stage_f(sval, v, n);
        float s;
        serial_scan_f(sval, n, s0, NAN, &s);
        __builtin_amdgcn_wave_barrier();
        return s;
    };
    // softmax (sampler.rs:67-69)
    ZS_SP_T(1);
    p = p / seq_sum(p, -0.0f);
    ZS_SP_T(2);
    // min-p (sampler.rs:72-88)
    if (P.min_p > 0.0f) {
        const float cut = P.min_p * wave_max_f(live ? p : 0.0f);
        if (p < cut) p = 0.0f;
        const float kept = seq_sum(p, 0.0f);
        if (kept > 0.0f) p = p / kept;
    }
    // top-p (sampler.rs:91-115): cumsum in (p desc, idx asc) order
    if (P.top_p < 1.0f) {
        uint32_t vstar = 0, istar = 0xffffffffu;
        const bool none = !(P.top_p > 0.0f);  // cumsum 0 >= top_p: nothing kept
        if (!none) {
            const unsigned long long k2 = wave_sort_u64(live ? (((unsigned long long)(~zs_f2u(p)) << 32) | id) : ~0ull);
            ZS_SP_T(3);
            if (live) sidx[lane] = (uint32_t)k2;
            wave_stage_f(sval, zs_u2f(~(uint32_t)(k2 >> 32)), n);
            float cum;
            const uint32_t i = serial_scan_f(sval, n, 0.0f, P.top_p, &cum);
            if (i < n) {
                vstar = zs_f2u(sval[i]);
                istar = sidx[i];
            }
            __builtin_amdgcn_wave_barrier();
            ZS_SP_T(4);
        }
        const uint32_t pb = zs_f2u(p);
        const bool keep = !none && (pb > vstar || (pb == vstar && id <= istar));
        const float f = keep ? p : 0.0f;
        const float sum = seq_sum(f, -0.0f);
        if (sum > 0.0f) p = f / sum;
        ZS_SP_T(5);
    }
    // draw (sampler.rs:118-127); r == 0 stops at index 0 whatever its p
    const float rr = zs_philox_uniform(seed, counter, 0u);
    if (rr <= 0.0f) return 0;
    if (live) sidx[lane] = id;
    wave_stage_f(sval, p, n);
    float cum;
    const uint32_t i = serial_scan_f(sval, n, 0.0f, rr, &cum);
    ZS_SP_T(6);
    return i < n ? sidx[i] : V - 1;
}

