// zs_lane.hip -- the batched GPU lane of the reference (continuous batching,
// gpu/batch.rs:176-192): batched argmax, Gumbel-max temperature sampling,
// top-K extraction and the top-K nucleus draw, with the reference semantics of
// shaders.rs:758-937 and gpu/sampling.rs:9-56, on-device (no readback).
//
// The WGSL kernels reduce with a 256-thread workgroup: thread t scans ids
// t, t+256, ... keeping the first strict maximum, then a stride-128..1 tree
// keeps the lower slot unless the upper one is strictly greater. The winner
// among equal maxima is therefore the slot with the smallest bit-reversed
// 8-bit slot number, then the smallest id within that slot; candidates must be
// strictly greater than the initial -1e30 (NaN never wins). These kernels
// reduce a composite key that encodes exactly that order, which lets any
// workgroup shape reproduce the WGSL result.
#include <hip/hip_runtime.h>
#include "zs_internal.h"
#include "zs_dev.h"

#define LN_NT 1024

__device__ __forceinline__ uint32_t zs_bitrev8(uint32_t x) { return __brev(x) >> 24; }

// composite for the WGSL argmax order: larger value, then preferred slot, then lower id
__device__ __forceinline__ unsigned long long wg_key(float v, uint32_t idx) {
    if (!(v > -1e30f)) return 0ull;  // not a candidate (also NaN)
    float vv = (v == 0.0f) ? 0.0f : v;
    uint32_t slot = idx & 255u, hi = idx >> 8;
    return ((unsigned long long)zs_total_key(vv) << 32) | ((unsigned long long)(255u - zs_bitrev8(slot)) << 24) |
           (unsigned long long)(0xffffffu - (hi & 0xffffffu));
}
__device__ __forceinline__ uint32_t wg_key_idx(unsigned long long k) {
    uint32_t slot = zs_bitrev8(255u - (uint32_t)((k >> 24) & 255u));
    uint32_t hi = 0xffffffu - (uint32_t)(k & 0xffffffu);
    return (hi << 8) | slot;
}

__device__ __forceinline__ unsigned long long block_max_u64(unsigned long long v, unsigned long long* sh) {
    v = zs_wave_reduce(v, [](unsigned long long x, unsigned long long y) { return x > y ? x : y; });
    if (zs_lane() == 0) sh[zs_wid()] = v;
    __syncthreads();
    unsigned long long r = 0;
    for (int i = 0; i < LN_NT / 64; i++) r = sh[i] > r ? sh[i] : r;
    __syncthreads();
    return r;
}

// shaders.rs:805-815
__device__ __forceinline__ uint32_t zs_hash_u32(uint32_t x) {
    uint32_t h = x;
    h ^= h >> 16; h *= 0x7feb352du;
    h ^= h >> 15; h *= 0x846ca68bu;
    h ^= h >> 16;
    return h;
}
// rand01 from the id's half of the hash, hi = zs_hash_u32(i)
__device__ __forceinline__ float zs_rand01_h(uint32_t s, uint32_t hi) {
    uint32_t r = zs_hash_u32(s ^ hi);
    return ((float)(r >> 8) + 0.5f) / 16777216.0f;
}
__device__ __forceinline__ float zs_rand01(uint32_t s, uint32_t i) { return zs_rand01_h(s, zs_hash_u32(i)); }

// ih[i] = zs_hash_u32(i): the id half of every row's uniforms, computed once
// per context (BSAMPLE reads it instead of hashing each id again)
__global__ void zs_k_lane_hash_fill(uint32_t* ih, uint32_t n) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) ih[i] = zs_hash_u32(i);
}
extern "C" int zs_lane_hash_fill(uint32_t* ih, uint32_t n, hipStream_t stream) {
    hipLaunchKernelGGL(zs_k_lane_hash_fill, dim3((n + 255) / 256), dim3(256), 0, stream, ih, n);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}
// WGSL `log` has no precision contract; this build fixes it as the f32
// rounding of the double log. Fast path: ln x in double from the atanh series
// of m in [sqrt(1/2), sqrt(2)) (x = m 2^e), relative error below 2^-44.7
// over every positive normal float up to 18 (the arguments here: u in (0, 1)
// and -ln u <= 17.33); its f32 rounding is certain unless the value lies
// within 2^-40 (relative) of a midpoint between floats (about 2e-5 of the
// inputs), where the double log is evaluated as the reference does; so are
// arguments outside that range.
__device__ __forceinline__ double zs_log_series(float x) {
    const uint32_t ix = __float_as_uint(x);
    int e = (int)(ix >> 23) - 127;
    float m = __uint_as_float((ix & 0x7fffffu) | 0x3f800000u);
    if (m > 1.41421356f) { m *= 0.5f; e += 1; }
    const double md = (double)m, num = md - 1.0, den = md + 1.0;
    double r = __builtin_amdgcn_rcp(den);
    r = fma(fma(-den, r, 1.0), r, r);
    r = fma(fma(-den, r, 1.0), r, r);
    const double f = num * r, f2 = f * f;
    double p = 1.0 / 15;
    p = fma(p, f2, 1.0 / 13);
    p = fma(p, f2, 1.0 / 11);
    p = fma(p, f2, 1.0 / 9);
    p = fma(p, f2, 1.0 / 7);
    p = fma(p, f2, 1.0 / 5);
    p = fma(p, f2, 1.0 / 3);
    p = fma(p, f2, 1.0);
    return fma((double)e, 0.6931471805599453, 2.0 * f * p);
}
__device__ __forceinline__ float zs_log_cr(float x) {
    // zeros (u = 1 gives -ln u = -0, whose log is -inf), infinities, NaN and
    // subnormals take the double log
    if (!(x >= 0x1p-126f && x <= 18.0f)) return (float)log((double)x);   // rare
    const double a = zs_log_series(x);
    const float r = (float)a;
    const double rd = (double)r, err = fabs(a) * 0x1p-40;
    const double up = (double)__uint_as_float(__float_as_uint(r) + (r >= 0.0f ? 1u : 0xffffffffu));
    const double dn = (double)__uint_as_float(__float_as_uint(r) + (r >= 0.0f ? 0xffffffffu : 1u));
    if (fabs(a - 0.5 * (rd + up)) <= err || fabs(a - 0.5 * (rd + dn)) <= err) return (float)log((double)x);  // rare
    return r;
}

// Gumbel term -ln(-ln u) with v_log_f32: within ZS_GUMBEL_EPS of the exact
// term for every u the hash can give (2^24 values, checked by
// tests/c/calib_gumbel.hip: the largest difference is 2^-19).
#define ZS_GUMBEL_EPS 0x1p-16f
__device__ __forceinline__ float zs_gumbel_fast(float u) {
    const float w = -(__builtin_amdgcn_logf(u) * 0.693147180559945309f);
    return -(__builtin_amdgcn_logf(w) * 0.693147180559945309f);
}
// Largest distance between an approximate Gumbel value a = RN(x/T) + g~ and
// its exact b (both rounded sums): the term's error plus an ulp each way.
__device__ __forceinline__ float zs_gumbel_band(float a) { return ZS_GUMBEL_EPS + fabsf(a) * 0x1p-22f; }
__device__ __forceinline__ float zs_gumbel_exact(float x, float inv_t, uint32_t sd, uint32_t i) {
    const float u = zs_rand01(sd, i);
    const float g = -zs_log_cr(-zs_log_cr(u));
    float v = x * inv_t;
    return v + g;
}

// BARGMAX (shaders.rs:761-789): one workgroup per row.
__global__ __launch_bounds__(LN_NT) void zs_k_bargmax(const float* logits, uint32_t V, uint64_t ld, uint32_t* out) {
    __shared__ unsigned long long sh[LN_NT / 64];
    const uint32_t r = blockIdx.x;
    const float* row = logits + (size_t)r * ld;
    unsigned long long best = 0;
    for (uint32_t i0 = threadIdx.x * 4; i0 < V; i0 += LN_NT * 4) {
        float4 v4 = *reinterpret_cast<const float4*>(row + i0);
        float vv[4] = {v4.x, v4.y, v4.z, v4.w};
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const uint32_t i = i0 + q;
            if (i >= V) continue;
            const unsigned long long k = wg_key(vv[q], i);
            best = k > best ? k : best;
        }
    }
    best = block_max_u64(best, sh);
    if (threadIdx.x == 0) out[r] = best ? wg_key_idx(best) : 0u;
}

// BSAMPLE (shaders.rs:796-850; rows with temperature <= 0 take the argmax)
// over segments of BS_SEG ids, one workgroup each (rows x segments fill the
// GPU). Two steps: every id's value with the fast Gumbel term, then the exact
// values (correctly rounded logs) only for the ids whose fast value lies
// within two bands of the segment's fast maximum -- the row's exact winner is
// among them, any other id being strictly below it. The segment's best exact
// key is merged into keys[row] with a 64-bit atomic max; zs_k_bsample_fin
// turns the keys into ids and clears them for the next call.
#define BS_NT 256
#define BS_SEG (BS_NT * 32)
__global__ __launch_bounds__(BS_NT) void zs_k_bsample(const float* logits, uint32_t V, uint64_t ld, const float* temp,
                                                      const uint32_t* seed, const uint32_t* ih,
                                                      unsigned long long* keys) {
    __shared__ unsigned long long shk[BS_NT / 64];
    __shared__ float shf[BS_NT / 64];
    const uint32_t r = blockIdx.y;
    const uint32_t s0 = blockIdx.x * BS_SEG, s1 = min(s0 + BS_SEG, V);
    const float* row = logits + (size_t)r * ld;
    const float ts = temp[r];
    const bool greedy = ts <= 0.0f;
    const float inv_t = greedy ? 1.0f : 1.0f / ts;
    const uint32_t sd = seed[r];
    const uint32_t last4 = (V - 1) & ~3u;
    unsigned long long best = 0;
    // exact keys of the thread's ids of the segment (greedy rows; threads
    // whose fast values cannot decide)
    auto exact_all = [&]() {
        for (uint32_t i0 = s0 + threadIdx.x * 4; i0 < s1; i0 += BS_NT * 4) {
            const float4 v4 = *reinterpret_cast<const float4*>(row + min(i0, last4));
            const float vv[4] = {v4.x, v4.y, v4.z, v4.w};
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const uint32_t i = i0 + q;
                if (i >= s1) continue;
                const float v = greedy ? vv[q] : zs_gumbel_exact(vv[q], inv_t, sd, i);
                const unsigned long long k = wg_key(v, i);
                best = k > best ? k : best;
            }
        }
    };
    if (greedy) {
        exact_all();
    } else {
        float ba = -INFINITY, bb = -INFINITY, bx = 0.0f;
        uint32_t bi = 0;
        bool exact = false;
        for (uint32_t i0 = s0 + threadIdx.x * 4; i0 < s1; i0 += BS_NT * 16) {
            float4 v4[4];
            uint4 h4[4];
#pragma unroll
            for (int u = 0; u < 4; u++) {
                const uint32_t j = min(i0 + (uint32_t)u * BS_NT * 4, last4);
                v4[u] = *reinterpret_cast<const float4*>(row + j);
                h4[u] = *reinterpret_cast<const uint4*>(ih + j);
            }
            float va[16], xs[16];
#pragma unroll
            for (int u = 0; u < 4; u++) {
                const float vv[4] = {v4[u].x, v4[u].y, v4[u].z, v4[u].w};
                const uint32_t hh[4] = {h4[u].x, h4[u].y, h4[u].z, h4[u].w};
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    const uint32_t i = i0 + (uint32_t)u * BS_NT * 4 + q;
                    xs[4 * u + q] = i < s1 ? vv[q] : -INFINITY;
                    const float v = xs[4 * u + q] * inv_t;
                    va[4 * u + q] = v + zs_gumbel_fast(zs_rand01_h(sd, hh[q]));
                }
            }
#pragma unroll
            for (int e = 0; e < 16; e++) {
                const float a = va[e];
                const bool fin = fabsf(a) < 1e29f;
                exact = exact | ((!fin) & (a == a) & (a != -INFINITY));   // -inf and NaN never win
                const float vf = fin ? a : -INFINITY;
                const bool gt = vf > ba;
                bb = fmaxf(bb, fminf(vf, ba));
                bx = gt ? xs[e] : bx;
                bi = gt ? i0 + (uint32_t)(e >> 2) * BS_NT * 4 + (uint32_t)(e & 3) : bi;
                ba = fmaxf(ba, vf);
            }
        }
        const bool near = bb > -INFINITY && ba - bb <= 2.0f * zs_gumbel_band(fmaxf(fabsf(ba), fabsf(bb)));
        float m = ba;
        m = wave_max_f(m);
        if (zs_lane() == 0) shf[zs_wid()] = m;
        __syncthreads();
        m = -INFINITY;
#pragma unroll
        for (int w = 0; w < BS_NT / 64; w++) m = fmaxf(m, shf[w]);
        const bool cand = exact || (ba > -INFINITY && ba >= m - 2.0f * zs_gumbel_band(fmaxf(fabsf(m), fabsf(ba))));
        if (cand) {
            if (exact || near) exact_all();   // rare
            else best = wg_key(zs_gumbel_exact(bx, inv_t, sd, bi), bi);
        }
    }
    best = zs_wave_reduce(best, [](unsigned long long x, unsigned long long y) { return x > y ? x : y; });
    if (zs_lane() == 0) shk[zs_wid()] = best;
    __syncthreads();
    if (threadIdx.x == 0) {
        unsigned long long b = 0;
#pragma unroll
        for (int w = 0; w < BS_NT / 64; w++) b = shk[w] > b ? shk[w] : b;
        if (b) atomicMax(&keys[r], b);
    }
}
__global__ void zs_k_bsample_fin(unsigned long long* keys, uint32_t B, uint32_t* out) {
    const uint32_t r = blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= B) return;
    const unsigned long long k = keys[r];
    out[r] = k ? wg_key_idx(k) : 0u;
    keys[r] = 0ull;
}

// BTOPK (shaders.rs:859-905): the K largest (value desc, id asc) among values in
// [-3e38, 3e38) (NaN and values outside never qualify: they are never "below"
// the previous winner or "better" than the -3e38 seed); sentinel (-3e38,
// 0xffffffff) pads rows with fewer candidates. Keys merge -0.0 and +0.0 (they
// compare equal in WGSL); the output keeps each element's own value.
#define TK_MAX 1024
__device__ __forceinline__ bool tk_cand(float v) { return v >= -3.0e38f && v < 3.0e38f; }
__device__ __forceinline__ uint32_t tk_key(float v) { return zs_total_key(v == 0.0f ? 0.0f : v); }

__global__ __launch_bounds__(LN_NT) void zs_k_btopk(const float* logits, uint32_t V, uint64_t ld, uint32_t K,
                                                     float* vals, uint32_t* idxs) {
    __shared__ uint32_t hist[256];
    __shared__ uint32_t u[4];
    __shared__ unsigned long long buf[TK_MAX];
    __shared__ uint32_t scan_sh[LN_NT / 64];
    const uint32_t r = blockIdx.x;
    const int t = threadIdx.x;
    const float* row = logits + (size_t)r * ld;
    // radix select of the K-th largest candidate key
    uint32_t ncand = 0;
    for (uint32_t i = t; i < V; i += LN_NT) ncand += tk_cand(row[i]) ? 1u : 0u;
    ncand = block_sum_u<LN_NT>(ncand, scan_sh);
    const uint32_t KK = ncand < K ? ncand : K;
    uint32_t prefix = 0, mask = 0, need = KK;
    if (KK > 0) {
        for (int shift = 24; shift >= 0; shift -= 8) {
            if (t < 256) hist[t] = 0;
            __syncthreads();
            for (uint32_t i = t; i < V; i += LN_NT) {
                float v = row[i];
                if (!tk_cand(v)) continue;
                uint32_t k = tk_key(v);
                if ((k & mask) == prefix) atomicAdd(&hist[(k >> shift) & 255u], 1u);
            }
            __syncthreads();
            if (t < 64) {
                uint32_t c[4], loc = 0;
                for (int q = 0; q < 4; q++) { c[q] = hist[255 - 4 * t - q]; loc += c[q]; }
                uint32_t inc = wave_incl_scan_u(loc);
                uint32_t before = inc - loc;
                for (int q = 0; q < 4; q++) {
                    if (before < need && need <= before + c[q]) { u[0] = 255 - 4 * t - q; u[1] = need - before; }
                    before += c[q];
                }
            }
            __syncthreads();
            prefix |= u[0] << shift;
            mask |= 0xffu << shift;
            need = u[1];
            __syncthreads();
        }
    }
    // gather: keys above the K-th, then the lowest-id `need` equal ones (ids in order)
    if (t == 0) u[2] = 0;
    __syncthreads();
    uint32_t carry = 0;
    for (uint32_t base = 0; base < V && KK > 0; base += LN_NT) {
        uint32_t i = base + t;
        float v = i < V ? row[i] : NAN;
        bool c = i < V && tk_cand(v);
        uint32_t k = c ? tk_key(v) : 0;
        bool gt = c && k > prefix, eq = c && k == prefix;
        uint32_t tot;
        uint32_t ex = block_excl_scan_u<LN_NT>(eq ? 1u : 0u, scan_sh, &tot);
        if (gt || (eq && carry + ex < need)) {
            uint32_t pos = atomicAdd(&u[2], 1u);
            if (pos < TK_MAX) buf[pos] = ((unsigned long long)(~k) << 32) | i;
        }
        carry += tot;
    }
    __syncthreads();
    uint32_t n = KK;
    uint32_t np2 = 1;
    while (np2 < n) np2 <<= 1;
    for (uint32_t i = n + t; i < np2; i += LN_NT) buf[i] = ~0ull;
    __syncthreads();
    if (np2 > 1) block_sort_u64<LN_NT>(buf, np2);
    for (uint32_t j = t; j < K; j += LN_NT) {
        if (j < n) {
            uint32_t id = (uint32_t)(buf[j] & 0xffffffffull);
            vals[(size_t)r * K + j] = row[id];
            idxs[(size_t)r * K + j] = id;
        } else {
            vals[(size_t)r * K + j] = -3.0e38f;
            idxs[(size_t)r * K + j] = 0xffffffffu;
        }
    }
}

// BTOPK for K <= 64 from group maxima. zs_k_lane_scan reads the logits once
// over the whole GPU and leaves the largest candidate key of every group of
// 2^gshift consecutive ids; zs_k_btopk_pick (one workgroup per row) takes a
// key that at least K groups reach: the row's first K by (key desc, id asc)
// lie in the groups whose maximum reaches it, a few more than K, whose ids are
// read again, listed and sorted. With the draw of zs_lane_step's top-K path
// in the same kernel. 256 rows of 151936 ids: the scan 24 us (6.5 TB/s), the
// pick 20 us; chunks of 16384 ids with a top-K each and a merge took 54 + 20.
// Rows with many groups or ids at the key (sorted rows, equal values) are cut
// level by level instead (8 rows of 128256: equal values 18 us a call, sorted
// 28, of whole numbers 26, rows in no order 13; 256 rows 37, 47, 44 and 34).
#define LS_NT 256
#define LS_IDS (16 * LS_NT)   // ids per workgroup of the scan
#define LP_NT 256
#define LP_GPT 20             // groups per thread of the pick at most
#define LP_GL 192             // listed groups at most (rows in no order list K + 20 to K + 80)
#define LP_LIST LP_NT         // listed keys at most: one per thread
#define TC_K 64
template <int GS>
__global__ __launch_bounds__(LS_NT) void zs_k_lane_scan(const float* logits, uint32_t V, uint64_t ld, uint32_t* gmax,
                                                        uint32_t gstride) {
    typedef float ls_f4 __attribute__((ext_vector_type(4)));
    const uint32_t r = blockIdx.y, lane = (uint32_t)zs_lane();
    const float* row = logits + (size_t)r * ld;
    const uint32_t base = blockIdx.x * LS_IDS + 4u * threadIdx.x;
    const uint32_t last4 = (V - 1u) & ~3u;   // (rows are whole multiples of 4 in memory)
    ls_f4 v[4];
#pragma unroll
    for (int u = 0; u < 4; u++) v[u] = *reinterpret_cast<const ls_f4*>(row + min(base + (uint32_t)u * (4u * LS_NT), last4));
    uint32_t k[4];
#pragma unroll
    for (int u = 0; u < 4; u++) {
        const uint32_t id = base + (uint32_t)u * (4u * LS_NT);
        const float x[4] = {v[u].x, v[u].y, v[u].z, v[u].w};
        // (non-candidates, NaN among them, count as no value)
        float m = -INFINITY;
#pragma unroll
        for (int q = 0; q < 4; q++) m = fmaxf(m, id + (uint32_t)q < V && tk_cand(x[q]) ? x[q] : -INFINITY);
        k[u] = tk_cand(m) ? tk_key(m) : 0u;
        k[u] = max(k[u], (uint32_t)__builtin_amdgcn_update_dpp(0, (int)k[u], 0xB1, 0xf, 0xf, false));    // quad_perm [1,0,3,2]
        k[u] = max(k[u], (uint32_t)__builtin_amdgcn_update_dpp(0, (int)k[u], 0x4E, 0xf, 0xf, false));    // quad_perm [2,3,0,1]
        if (GS >= 5) k[u] = max(k[u], (uint32_t)__builtin_amdgcn_update_dpp(0, (int)k[u], 0x141, 0xf, 0xf, false));   // row_half_mirror
        if (GS >= 6) k[u] = max(k[u], (uint32_t)__builtin_amdgcn_update_dpp(0, (int)k[u], 0x140, 0xf, 0xf, false));   // row_mirror
    }
    // lane q of a quad stores load q's group (one store for all four)
    constexpr uint32_t LG = 1u << (GS - 2);   // lanes per group
    const uint32_t q = lane & 3u;
    const uint32_t kq = q == 0 ? k[0] : q == 1 ? k[1] : q == 2 ? k[2] : k[3];
    const uint32_t g = (blockIdx.x * LS_IDS + q * (4u * LS_NT) + 4u * threadIdx.x) >> GS;
    if ((lane & (LG - 1u)) < 4u && g < (V + (1u << GS) - 1u) >> GS) gmax[(size_t)r * gstride + g] = kq;
}

struct tm_draw {   // the nucleus draw after the pick (zs_lane_step's top-K path)
    const float* temp;
    const uint32_t *top_k;
    const float* top_p;
    const uint32_t* seed;
    uint32_t* out;
};
__device__ __forceinline__ uint32_t lane_draw64(float v, uint32_t id, uint32_t K, float T, uint32_t top_k, float tp,
                                                uint32_t seed);
// Of the workgroup's E * LP_NT places (t, t + LP_NT, ...: bit e), the first K
// by (key desc, place asc); places of key 0 are none. Radix selection of the
// K-th key over the digits in which the keys differ, then the places at it in
// order. Called by every thread; hist: 256 words, u: 4 words.
template <int E>
__device__ __forceinline__ uint32_t tk_first(const uint32_t (&k)[E], uint32_t K, uint32_t* hist, uint32_t* u) {
    constexpr uint32_t NW = LP_NT / 64;
    static_assert(3 * NW <= 256 && E * NW <= 256 && LP_NT == 256, "one histogram holds the counts");
    const uint32_t t = threadIdx.x, lane = (uint32_t)zs_lane(), wid = (uint32_t)zs_wid();
    uint32_t lo = ~0u, hi = 0, n = 0, all = 0;
#pragma unroll
    for (int e = 0; e < E; e++) {
        if (!k[e]) continue;
        lo = min(lo, k[e]);
        hi = max(hi, k[e]);
        n++;
        all |= 1u << e;
    }
    lo = zs_wave_reduce(lo, [](uint32_t x, uint32_t y) { return min(x, y); });
    hi = zs_wave_reduce(hi, [](uint32_t x, uint32_t y) { return max(x, y); });
    n = wave_sum_u(n);
    if (lane == 0) { hist[wid] = lo; hist[NW + wid] = hi; hist[2 * NW + wid] = n; }
    __syncthreads();
    n = 0;
#pragma unroll
    for (uint32_t w = 0; w < NW; w++) {
        lo = min(lo, hist[w]);
        hi = max(hi, hist[NW + w]);
        n += hist[2 * NW + w];
    }
    __syncthreads();
    if (n <= K) return all;
    // key: the K-th once its digits are known; those above the first in which
    // the keys differ are hi's
    int shift = lo != hi ? (31 - __clz((int)(lo ^ hi))) & ~7 : -8;
    uint32_t mask = shift < 0 ? ~0u : shift == 24 ? 0u : ~0u << (shift + 8);
    uint32_t key = hi & mask, need = K;
    for (; shift >= 0; shift -= 8) {
        hist[t] = 0;
        __syncthreads();
#pragma unroll
        for (int e = 0; e < E; e++)
            if (k[e] && (k[e] & mask) == key) atomicAdd(&hist[(k[e] >> shift) & 255u], 1u);
        __syncthreads();
        if (t < 64) {
            uint32_t c[4], loc = 0;
#pragma unroll
            for (int q = 0; q < 4; q++) { c[q] = hist[255u - 4u * t - (uint32_t)q]; loc += c[q]; }
            const uint32_t inc = wave_incl_scan_u(loc);
            uint32_t before = inc - loc;
#pragma unroll
            for (int q = 0; q < 4; q++) {
                if (before < need && need <= before + c[q]) { u[0] = 255u - 4u * t - (uint32_t)q; u[1] = need - before; }
                before += c[q];
            }
        }
        __syncthreads();
        key |= u[0] << shift;
        mask |= 0xffu << shift;
        need = u[1];
    }
#pragma unroll
    for (int e = 0; e < E; e++) {
        const uint32_t c = (uint32_t)__popcll(__ballot(k[e] == key));
        if (lane == 0) hist[(uint32_t)e * NW + wid] = c;
    }
    __syncthreads();
    uint32_t run = 0, first = 0;
#pragma unroll
    for (int e = 0; e < E; e++) {
        const unsigned long long m = __ballot(k[e] == key);
        uint32_t before = run;
#pragma unroll
        for (uint32_t w = 0; w < NW; w++) {
            const uint32_t c = hist[(uint32_t)e * NW + w];
            before += w < wid ? c : 0u;
            run += c;
        }
        before = __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, before));
        if (k[e] > key || (k[e] == key && before < need)) first |= 1u << e;
    }
    __syncthreads();
    return first;
}
// The chosen places in ascending order to gl (K <= 64 of them; the return is
// their number). Called by every thread; u: 4 words, u[2] is 0 before and after.
__device__ __forceinline__ uint32_t tk_places(uint32_t first, uint16_t* gl, uint32_t* u) {
    const uint32_t t = threadIdx.x;
    while (first) {
        const uint32_t e = (uint32_t)__builtin_ctz(first);
        first &= first - 1u;
        gl[atomicAdd(&u[2], 1u)] = (uint16_t)(t + e * LP_NT);
    }
    __syncthreads();
    const uint32_t n = u[2];
    __syncthreads();
    if (t < 64) {
        const uint32_t g = wave_sort_u32(t < n ? (uint32_t)gl[t] : ~0u);
        if (t < n) gl[t] = (uint16_t)g;
        if (t == 0) u[2] = 0;
    }
    __syncthreads();
    return n;
}

template <bool DRAW>
__global__ __launch_bounds__(LP_NT) void zs_k_btopk_pick(const float* logits, uint32_t V, uint64_t ld, uint32_t K,
                                                         const uint32_t* gmax, uint32_t gstride, uint32_t gs, float* vals,
                                                         uint32_t* idxs, tm_draw d) {
    constexpr uint32_t NW = LP_NT / 64;
    typedef float ls_f4 __attribute__((ext_vector_type(4)));
    __shared__ unsigned long long list[LP_LIST];
    __shared__ alignas(16) uint16_t gl[LP_GL];
    __shared__ uint32_t hist[256], u[4], wthr[NW];
    const uint32_t r = blockIdx.x, t = threadIdx.x, lane = (uint32_t)zs_lane(), wid = (uint32_t)zs_wid();
    const float* row = logits + (size_t)r * ld;
    const uint32_t ng = (V + (1u << gs) - 1u) >> gs, last4 = (V - 1u) & ~3u;
    const uint32_t* gm = gmax + (size_t)r * gstride;
    uint32_t k[LP_GPT], tm = 0;
    auto load_groups = [&]() {
#pragma unroll
        for (int e = 0; e < LP_GPT; e++) k[e] = zs_gload(gm + min(t + (uint32_t)e * LP_NT, ng - 1u));
#pragma unroll
        for (int e = 0; e < LP_GPT; e++)
            if (t + (uint32_t)e * LP_NT >= ng) k[e] = 0u;
    };
    load_groups();
#pragma unroll
    for (int e = 0; e < LP_GPT; e++) tm = max(tm, k[e]);
    if (t < 4) u[t] = 0;
    // theta: in every wave the ceil(K / waves)-th largest thread maximum; the
    // smallest of them is reached by K groups (0: too few hold a candidate;
    // every candidate is listed then)
    const uint32_t srt = wave_sort_u32(tm);
    const uint32_t wt = (uint32_t)__builtin_amdgcn_readlane((int)srt, 64 - (int)((K + NW - 1u) / NW));
    if (lane == 0) wthr[wid] = wt;
    __syncthreads();
    uint32_t theta = wthr[0];
#pragma unroll
    for (uint32_t w = 1; w < NW; w++) theta = min(theta, wthr[w]);
    theta = max(theta, 1u);
    uint32_t ngt = 0;
#pragma unroll
    for (int e = 0; e < LP_GPT; e++) ngt += k[e] >= theta ? 1u : 0u;
    // (a thread's places at once: an atomic per group is served lane by lane)
    uint32_t p = ngt ? atomicAdd(&u[0], ngt) : 0u;
#pragma unroll
    for (int e = 0; e < LP_GPT; e++) {
        if (k[e] < theta) continue;
        if (p < LP_GL) gl[p] = (uint16_t)(t + (uint32_t)e * LP_NT);
        p++;
    }
    __syncthreads();
    const uint32_t n_gl = u[0], qs = gs - 2u, qm = (1u << qs) - 1u;
    // keys of the ids x.x .. x.w from id on, 0 for no candidate
    auto keys4 = [&](const ls_f4& x, uint32_t id, uint32_t (&kq)[4]) {
        const float xs[4] = {x.x, x.y, x.z, x.w};
#pragma unroll
        for (int q = 0; q < 4; q++) kq[q] = id + (uint32_t)q < V && tk_cand(xs[q]) ? tk_key(xs[q]) : 0u;
    };
    if (n_gl <= LP_GL) {
        const uint32_t nit = n_gl << qs;
        constexpr int NU = 4;
        for (uint32_t i0 = 0; i0 < nit; i0 += NU * LP_NT) {
            ls_f4 v[NU];
            uint32_t id[NU];
#pragma unroll
            for (int w = 0; w < NU; w++) {
                const uint32_t i = i0 + t + (uint32_t)w * LP_NT, ic = min(i, nit - 1u);
                id[w] = ((uint32_t)gl[ic >> qs] << gs) + 4u * (ic & qm);
                v[w] = zs_gload(reinterpret_cast<const ls_f4*>(row + min(id[w], last4)));
                if (i >= nit) id[w] = V;
            }
#pragma unroll
            for (int w = 0; w < NU; w++) {
                // (one atomic per wave: one per lane is served lane by lane)
                uint32_t kq[4], p = 0, n = 0;
                keys4(v[w], id[w], kq);
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    const unsigned long long m = __ballot(kq[q] >= theta);
                    p = __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, p));
                    n += (uint32_t)__popcll(m);
                }
                if (!n) continue;
                uint32_t p0 = 0;
                if (lane == 0) p0 = atomicAdd(&u[1], n);
                p += (uint32_t)__builtin_amdgcn_readfirstlane((int)p0);
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    if (kq[q] < theta) continue;
                    if (p < LP_LIST) list[p] = ((unsigned long long)(~kq[q]) << 32) | (id[w] + (uint32_t)q);
                    p++;
                }
            }
        }
    }
    __syncthreads();
    uint32_t n = u[1];
    if (n_gl > LP_GL || n > LP_LIST) {
        // Many groups or ids reach theta. The first K ids lie in the first K
        // groups by (maximum desc, group asc) -- K groups in front of another
        // hold K ids in front of any of its -- and in the first K quads of
        // those by the same order, 4 K ids.
        constexpr int NQ = TC_K * 16 / LP_NT;   // quads per thread at most (K groups of 64 ids)
        uint32_t ngl = n_gl;
        if (n_gl <= LP_GL && (n_gl << qs) <= NQ * LP_NT) {
            // the listed groups' quads fit as they are: in ascending order
            static_assert(LP_GL <= LP_NT, "one listed group per thread");
            static_assert(LP_GL % 8 == 0, "eight to a read");
            if (t >= n_gl && t < LP_GL) gl[t] = 0xffffu;
            __syncthreads();
            const uint32_t g = t < n_gl ? gl[t] : 0xffffu;
            uint32_t before = 0;
#pragma unroll 4
            for (uint32_t j = 0; j < LP_GL / 8; j++) {
                const uint4 o = reinterpret_cast<const uint4*>(gl)[j];
                const uint32_t ow[4] = {o.x, o.y, o.z, o.w};
#pragma unroll
                for (int q = 0; q < 4; q++) before += ((ow[q] & 0xffffu) < g ? 1u : 0u) + ((ow[q] >> 16) < g ? 1u : 0u);
            }
            __syncthreads();
            if (t < n_gl) gl[before] = (uint16_t)g;
            __syncthreads();
        } else {
            __syncthreads();
            load_groups();
#pragma unroll
            for (int e = 0; e < LP_GPT; e++)
                if (k[e] < theta) k[e] = 0u;
            ngl = tk_places(tk_first<LP_GPT>(k, K, hist, u), gl, u);
        }
        const uint32_t nit = ngl << qs;
        uint32_t qk[NQ], qid[NQ];
        ls_f4 v[NQ];
#pragma unroll
        for (int w = 0; w < NQ; w++) {
            const uint32_t i = t + (uint32_t)w * LP_NT, ic = min(i, nit - 1u);
            qid[w] = ((uint32_t)gl[ic >> qs] << gs) + 4u * (ic & qm);
            v[w] = zs_gload(reinterpret_cast<const ls_f4*>(row + min(qid[w], last4)));
            if (i >= nit) qid[w] = V;
        }
#pragma unroll
        for (int w = 0; w < NQ; w++) {
            uint32_t kq[4];
            keys4(v[w], qid[w], kq);
            qk[w] = max(max(kq[0], kq[1]), max(kq[2], kq[3]));
        }
        uint32_t first = tk_first<NQ>(qk, K, hist, u);
        if (t == 0) u[1] = 0;
        __syncthreads();
#pragma unroll
        for (int w = 0; w < NQ; w++) {
            if (!(first >> w & 1u)) continue;
            uint32_t kq[4];
            keys4(v[w], qid[w], kq);
            uint32_t p = atomicAdd(&u[1], 4u);   // at most 4 K <= LP_LIST
#pragma unroll
            for (int q = 0; q < 4; q++) list[p + (uint32_t)q] = kq[q] ? ((unsigned long long)(~kq[q]) << 32) | (qid[w] + (uint32_t)q) : ~0ull;
        }
        __syncthreads();
        n = u[1];
    }
    static_assert(4 * TC_K <= LP_LIST, "the quads' ids fit the list");
    uint32_t np2 = 64;
    while (np2 < n) np2 <<= 1;
    if (t >= n && t < np2) list[t] = ~0ull;
    __syncthreads();
    block_sort_reg_u64<LP_NT, 1>(list, np2);
    if (t >= 64) return;
    float v = -3.0e38f;
    uint32_t id = 0xffffffffu;
    const unsigned long long e = lane < min(K, n) ? list[lane] : ~0ull;
    if (e != ~0ull) {
        id = (uint32_t)e;
        v = row[id];
    }
    if (lane < K) {
        vals[(size_t)r * K + lane] = v;
        idxs[(size_t)r * K + lane] = id;
    }
    if (DRAW) {
        // the pool as zs_k_sample_topk64 reads it back
        const uint32_t res = lane_draw64(lane < K ? v : -INFINITY, lane < K ? id : 0u, K, d.temp[r], d.top_k[r],
                                         d.top_p[r], d.seed[r]);
        if (lane == 0) d.out[r] = res;
    }
}
// Launches the scan and the pick; gmax: B rows of gstride >= ceil(V / 16) keys.
template <bool DRAW>
static void lane_topk_groups(const float* logits, uint32_t B, uint32_t V, uint64_t ld, uint32_t K, float* vals,
                             uint32_t* idxs, uint32_t* gmax, uint32_t gstride, const tm_draw& d, hipStream_t stream) {
    uint32_t gs = 4;
    while (((V + (1u << gs) - 1u) >> gs) > LP_GPT * LP_NT) gs++;
    const dim3 grid((V + LS_IDS - 1) / LS_IDS, B);
    if (gs == 4) hipLaunchKernelGGL(zs_k_lane_scan<4>, grid, dim3(LS_NT), 0, stream, logits, V, ld, gmax, gstride);
    else if (gs == 5) hipLaunchKernelGGL(zs_k_lane_scan<5>, grid, dim3(LS_NT), 0, stream, logits, V, ld, gmax, gstride);
    else hipLaunchKernelGGL(zs_k_lane_scan<6>, grid, dim3(LS_NT), 0, stream, logits, V, ld, gmax, gstride);
    hipLaunchKernelGGL(zs_k_btopk_pick<DRAW>, dim3(B), dim3(LP_NT), 0, stream, logits, V, ld, K, gmax, gstride, gs, vals,
                       idxs, d);
}

// gpu/sampling.rs:24-31
__device__ __forceinline__ float zs_rng01(uint32_t seed) {
    uint64_t z = (uint64_t)seed * 0x9E3779B97F4A7C15ull + 0x9E3779B97F4A7C15ull;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    z ^= z >> 31;
    return ((float)(z >> 40) + 0.5f) / 16777216.0f;
}

// gpu/sampling.rs:35-56, one thread per row over its descending pool.
__global__ void zs_k_sample_topk(const float* vals, const uint32_t* idxs, uint32_t B, uint32_t K,
                                 const float* temp, const uint32_t* top_k, const float* top_p,
                                 const uint32_t* seed, uint32_t* out) {
    uint32_t r = blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= B) return;
    const float* v = vals + (size_t)r * K;
    const uint32_t* id = idxs + (size_t)r * K;
    uint32_t n = 0;
    while (n < K && v[n] > -3.0e37f) n++;
    if (n == 0 || temp[r] <= 0.0f) { out[r] = id[0]; return; }
    const float T = temp[r];
    uint32_t kk = top_k[r] == 0 ? n : (top_k[r] < n ? top_k[r] : n);
    const float maxv = v[0];
    float z = -0.0f;
    for (uint32_t i = 0; i < kk; i++) z = z + zs_expf((v[i] - maxv) / T);
    uint32_t cut = kk;
    const float tp = top_p[r];
    if (tp > 0.0f && tp < 1.0f) {
        float cum = 0.0f;
        for (uint32_t i = 0; i < kk; i++) {
            cum = cum + zs_expf((v[i] - maxv) / T) / z;
            if (cum >= tp) { cut = i + 1; break; }
        }
    }
    float zc = -0.0f;
    for (uint32_t i = 0; i < cut; i++) zc = zc + zs_expf((v[i] - maxv) / T) / z;
    const float target = zs_rng01(seed[r]) * zc;
    float acc = 0.0f;
    uint32_t res = id[cut - 1];
    for (uint32_t i = 0; i < cut; i++) {
        acc = acc + zs_expf((v[i] - maxv) / T) / z;
        if (acc >= target) { res = id[i]; break; }
    }
    out[r] = res;
}

// The same draw by one wave for a pool of at most 64 (lane i holds entry i:
// value v, id; lanes >= K hold -inf): the exponentials in parallel, the
// sequential sums (sampler order, f32) as chains of lane reads (the index is
// uniform: v_readlane, no LDS permute). Returns the id (uniform).
__device__ __forceinline__ uint32_t lane_draw64(float v, uint32_t id, uint32_t K, float T, uint32_t top_k, float tp,
                                                uint32_t seed) {
    const int lane = zs_lane();
    const uint32_t id0 = __shfl(id, 0, 64);
    // n: length of the leading run of values above the sentinel
    const unsigned long long fail = __ballot(!((uint32_t)lane < K && v > -3.0e37f));
    const uint32_t n = fail ? (uint32_t)__ffsll((long long)fail) - 1u : 64u;
    if (n == 0 || T <= 0.0f) return id0;
    const uint32_t kk = top_k == 0 ? n : (top_k < n ? top_k : n);
    const float maxv = __shfl(v, 0, 64);
    const float e = (uint32_t)lane < kk ? zs_expf((v - maxv) / T) : 0.0f;
    float z = -0.0f;
    for (uint32_t i = 0; i < kk; i++) z = z + zs_readlane_f(e, i);
    const float p = e / z;
    uint32_t cut = kk;
    if (tp > 0.0f && tp < 1.0f) {
        float cum = 0.0f;
        for (uint32_t i = 0; i < kk; i++) {
            cum = cum + zs_readlane_f(p, i);
            if (cum >= tp) { cut = i + 1; break; }
        }
    }
    float zc = -0.0f;
    for (uint32_t i = 0; i < cut; i++) zc = zc + zs_readlane_f(p, i);
    const float target = zs_rng01(seed) * zc;
    float acc = 0.0f;
    uint32_t pick = cut - 1;
    for (uint32_t i = 0; i < cut; i++) {
        acc = acc + zs_readlane_f(p, i);
        if (acc >= target) { pick = i; break; }
    }
    return __shfl(id, (int)pick, 64);
}

#define TM_ROWS 4
__global__ __launch_bounds__(64 * TM_ROWS) void zs_k_sample_topk64(const float* vals, const uint32_t* idxs,
                                                                    uint32_t B, uint32_t K, const float* temp,
                                                                    const uint32_t* top_k, const float* top_p,
                                                                    const uint32_t* seed, uint32_t* out) {
    const uint32_t r = blockIdx.x * TM_ROWS + zs_wid();
    if (r >= B) return;
    const int lane = zs_lane();
    const float v = (uint32_t)lane < K ? vals[(size_t)r * K + lane] : -INFINITY;
    const uint32_t id = (uint32_t)lane < K ? idxs[(size_t)r * K + lane] : 0u;
    const uint32_t res = lane_draw64(v, id, K, temp[r], top_k[r], top_p[r], seed[r]);
    if (lane == 0) out[r] = res;
}

// ih: zs_lane_hash_fill of at least round_up(V, 4) ids; keys: B zeroed u64
// (left zeroed) -- both used when temp is set
extern "C" int zs_lane_argmax_launch(const float* logits, uint32_t B, uint32_t V, uint64_t ld, const float* temp,
                                     const uint32_t* seed, const uint32_t* ih, unsigned long long* keys,
                                     uint32_t* out, hipStream_t stream) {
    if (temp) {
        hipLaunchKernelGGL(zs_k_bsample, dim3((V + BS_SEG - 1) / BS_SEG, B), dim3(BS_NT), 0, stream, logits, V, ld,
                           temp, seed, ih, keys);
        hipLaunchKernelGGL(zs_k_bsample_fin, dim3((B + 255) / 256), dim3(256), 0, stream, keys, B, out);
        return hipGetLastError() == hipSuccess ? 0 : -1;
    }
    hipLaunchKernelGGL(zs_k_bargmax, dim3(B), dim3(LN_NT), 0, stream, logits, V, ld, out);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}
// gmax: scratch of B rows of gstride >= ceil(V / 16) keys (the path from group
// maxima, K <= 64, V <= ZS_MAX_VOCAB); nullptr forces the passes by one workgroup
extern "C" int zs_lane_topk_launch(const float* logits, uint32_t B, uint32_t V, uint64_t ld, uint32_t K,
                                   float* vals, uint32_t* idxs, uint32_t* gmax, uint32_t gstride,
                                   hipStream_t stream) {
    if (gmax && K <= TC_K && V <= ZS_MAX_VOCAB) {
        lane_topk_groups<false>(logits, B, V, ld, K, vals, idxs, gmax, gstride, tm_draw{}, stream);
    } else {
        hipLaunchKernelGGL(zs_k_btopk, dim3(B), dim3(LN_NT), 0, stream, logits, V, ld, K, vals, idxs);
    }
    return hipGetLastError() == hipSuccess ? 0 : -1;
}
// The top-K pool and its nucleus draw: on the group path the pick kernel
// draws too (one launch and no read-back of the pool), else the two launches.
extern "C" int zs_lane_sample_topk_launch(const float* vals, const uint32_t* idxs, uint32_t B, uint32_t K,
                                          const float* temp, const uint32_t* top_k, const float* top_p,
                                          const uint32_t* seed, uint32_t* out, hipStream_t stream);
extern "C" int zs_lane_topk_draw_launch(const float* logits, uint32_t B, uint32_t V, uint64_t ld, uint32_t K,
                                        float* vals, uint32_t* idxs, uint32_t* gmax, uint32_t gstride,
                                        const float* temp, const uint32_t* top_k, const float* top_p,
                                        const uint32_t* seed, uint32_t* out, hipStream_t stream) {
    if (gmax && K <= TC_K && V <= ZS_MAX_VOCAB) {
        lane_topk_groups<true>(logits, B, V, ld, K, vals, idxs, gmax, gstride, tm_draw{temp, top_k, top_p, seed, out}, stream);
        return hipGetLastError() == hipSuccess ? 0 : -1;
    }
    if (zs_lane_topk_launch(logits, B, V, ld, K, vals, idxs, gmax, gstride, stream)) return -1;
    return zs_lane_sample_topk_launch(vals, idxs, B, K, temp, top_k, top_p, seed, out, stream);
}
extern "C" int zs_lane_sample_topk_launch(const float* vals, const uint32_t* idxs, uint32_t B, uint32_t K,
                                          const float* temp, const uint32_t* top_k, const float* top_p,
                                          const uint32_t* seed, uint32_t* out, hipStream_t stream) {
    if (K <= 64)
        hipLaunchKernelGGL(zs_k_sample_topk64, dim3((B + TM_ROWS - 1) / TM_ROWS), dim3(64 * TM_ROWS), 0, stream, vals,
                           idxs, B, K, temp, top_k, top_p, seed, out);
    else
        hipLaunchKernelGGL(zs_k_sample_topk, dim3((B + 63) / 64), dim3(64), 0, stream, vals, idxs, B, K, temp, top_k,
                           top_p, seed, out);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}
