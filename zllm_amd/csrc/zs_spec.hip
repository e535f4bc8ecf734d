// zs_spec.hip -- speculative-decode verification over k draft positions.
//
// temperature <= 0: greedy verification exactly as spec_decode.rs:241-279
// (accept drafts while argmax(target_i) == draft_i, first-max argmax with
// strict >, bonus = argmax of the first mismatching row or of row k).
//
// temperature > 0: rejection sampling (Leviathan et al. 2023; Chen et al.
// 2023), which the reference does not implement (rest.rs:2639). To make it
// reproducible bit-for-bit on any reduction order, probabilities are integer
// quantised: with m = max x (NaN ignored) and c = log2(e) / T (one f32
// division per row), the weight of id v is
//   P_v = rint(2^24 * 2^t),  t = (x_v - m) * c   (target),   Q_v likewise (draft),
// from a fixed sequence of f32 operations (sp_weight), 0 below t = -25 (where
// the formula itself rounds to 0). No per-element division by T is needed.
// Draft i (token d) is accepted iff U_i * Q_d * sum(P) <= P_d * sum(Q) * 2^32,
// U_i the 32-bit Philox word of (seed, counter, tag 1+i). At the first
// rejection i the replacement token is drawn from R_v = max(0, P_v sum(Q) -
// Q_v sum(P)) (from P when sum(R) == 0) with tag 1+k+i; when all k drafts are
// accepted the bonus token is drawn from the target row k with tag 1+2k. A draw
// with weights W and word U returns the first id whose inclusive prefix of W
// exceeds floor(U * sum(W) / 2^32). Draft ids >= V are rejected. A row whose
// target or draft logits contain NaN / +inf or are all -inf is verified
// greedily.
#include <hip/hip_runtime.h>
#include "zs_internal.h"
#include "zs_dev.h"
#include <algorithm>
#include <mutex>

#define SP_NT 256
#define SP_CH 8192
#define SP_EPT (SP_CH / SP_NT)   // 32 elements per thread, as 8 float4
#define SP_BIG_NT 1024
// weights are 0 below this log-ratio
#define SP_ZERO_T (-25.0f)

typedef unsigned __int128 u128;

__device__ __forceinline__ const float* sp_row(const zs_spec_args& a, uint32_t r, uint32_t pos) {
    if (pos <= a.k) return a.target + ((size_t)r * (a.k + 1) + pos) * a.ld;
    return a.draft + ((size_t)r * a.k + (pos - a.k - 1)) * a.ld;
}
// c = log2(e) / T, the factor of the exponent (T > 0)
__device__ __forceinline__ float sp_c(float T) { return __fdiv_rn(1.44269502f, T); }
// Integer weight rint(2^24 * 2^t), t = (x - m) * c, through a fixed sequence of
// correctly rounded f32 operations (t = n + f with n = floor(t), 2^f by a
// degree-7 Taylor polynomial in fmaf Horner form, exact scaling by 2^(24+n),
// rint), so the CPU restatement reproduces every weight bit for bit. t < -25
// gives 2^f * 2^(24+n) < 0.5, i.e. 0. For x <= m the weight is below 2^25, so
// 32 of them add up in 32 bits.
__device__ __forceinline__ uint32_t sp_weight(float x, float m, float c) {
    const float t = __fmul_rn(__fsub_rn(x, m), c);
    const float n = floorf(t);
    const float f = __fsub_rn(t, n);
    float p = 1.52527338e-05f;
    p = fmaf(p, f, 1.54035304e-04f);
    p = fmaf(p, f, 1.33335581e-03f);
    p = fmaf(p, f, 9.61812911e-03f);
    p = fmaf(p, f, 5.55041087e-02f);
    p = fmaf(p, f, 2.40226507e-01f);
    p = fmaf(p, f, 6.93147182e-01f);
    p = fmaf(p, f, 1.0f);
    const uint32_t w = (uint32_t)rintf(ldexpf(p, 24 + (int)n));
    return t >= SP_ZERO_T ? w : 0u;
}
// whether any x <= xc can have a positive weight
__device__ __forceinline__ bool sp_live(float xc, float m, float c) {
    return __fmul_rn(__fsub_rn(xc, m), c) >= SP_ZERO_T;
}
// the chunk's elements of thread t: float4 j covers ids base + (j*SP_NT + t)*4
// .. +3. Non-temporal: a verification reads each of its rows once (the residual
// pass one pair a row again), and its gigabytes would push the sampler's rows,
// which the kernels beside it read several times, out of the caches (256 rows
// of 9 positions of 151936 ids beside the sampler: 697 -> 682 us). Alone, plain
// / non-temporal loads in both passes: 5 positions greedily 128 x 151936 71 /
// 64 us, 9 positions 256 x 151936 300 / 295, 64 x 128256 85.0 / 84.5; calls
// below 25 us lose 1.
typedef float sp_f4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ void sp_load(const float* row, uint32_t base, uint32_t V, float (&x)[SP_EPT]) {
#pragma unroll
    for (int j = 0; j < SP_EPT / 4; j++) {
        const uint32_t id = base + (j * SP_NT + threadIdx.x) * 4;
        sp_f4 v = {-INFINITY, -INFINITY, -INFINITY, -INFINITY};
        if (id < V) v = __builtin_nontemporal_load(reinterpret_cast<const sp_f4*>(row + id));
        x[4 * j] = v.x; x[4 * j + 1] = v.y; x[4 * j + 2] = v.z; x[4 * j + 3] = v.w;
    }
    if (base + SP_CH > V) {  // ids past V read as -inf (neutral in every pass)
#pragma unroll
        for (int e = 0; e < SP_EPT; e++)
            if (base + ((e >> 2) * SP_NT + threadIdx.x) * 4 + (e & 3) >= V) x[e] = -INFINITY;
    }
}
__device__ __forceinline__ uint32_t sp_id(uint32_t base, int e) {
    return base + ((e >> 2) * SP_NT + threadIdx.x) * 4 + (e & 3);
}

// One pass per chunk: the chunk maximum, flags, the first strict maximum of x
// (greedy verification) and, once the chunk maximum is known, the chunk sum of
// the weights w_v = W((x_v - m_c) c). The rows from r0 on.
//
// Bound by HBM. A workgroup is small and needs few registers, so a launch of
// many holds every slot that one of its own gives up, and a kernel beside it on
// another stream that needs much of a CU (zs_k_row: 168 registers of 8 waves
// and 149 KB of LDS at 151936 ids) waits for its end: 190 us instead of 47 beside
// 43776 workgroups. So where a sampler may run beside it (zs_spec_args.beside)
// the rows go in equal launches of at most SP_PART workgroups: between two of
// them the CUs come free. Full step of 256 rows (9 positions of 151936 ids
// beside the sampler; one batch of logits): one launch 677 us, two 638, three
// 645, five 651, ten 658; other batches, one and two: 680 and 656. Alone each
// further launch adds about 10 us (302 and 316), so it is one launch there.
#define SP_PART 24576u
__global__ __launch_bounds__(SP_NT) void zs_k_spec_chunk(zs_spec_args a, uint32_t r0) {
    const uint32_t c = blockIdx.x, pos = blockIdx.y, r = r0 + blockIdx.z;
    const uint32_t npos = a.draft ? 2 * a.k + 1 : a.k + 1;
    if (pos >= npos) return;
    const uint32_t base = c * SP_CH;
    if (base >= a.V) return;
    __shared__ float fsh[SP_NT / 64];
    __shared__ uint32_t ush[SP_NT / 64];
    __shared__ unsigned long long gsh[SP_NT / 64], wsh[SP_NT / 64];
    float x[SP_EPT];
    sp_load(sp_row(a, r, pos), base, a.V, x);
    // first strict maximum (init -inf, NaN never wins) in index order: the
    // elements of a thread ascend with e; it is also the NaN-ignoring max
    float bv = -INFINITY;
    int be = -1;
    bool nan = false;
#pragma unroll
    for (int e = 0; e < SP_EPT; e++) {
        const float xv = x[e];
        nan |= xv != xv;
        if (xv > bv) { bv = xv; be = e; }
    }
    uint32_t fl = nan ? 1u : 0u;
    if (bv == INFINITY) fl |= 2u;
    // (value key, ~idx): larger value first, then the lower id; -0 == +0
    unsigned long long best = be < 0 ? 0ull
        : ((unsigned long long)zs_total_key(bv == 0.0f ? 0.0f : bv) << 32) | (0xffffffffu - sp_id(base, be));
    const float xmax = block_max_f<SP_NT>(bv, fsh);
    fl = block_or_u<SP_NT>(fl, ush);
    best = zs_wave_reduce(best, [](unsigned long long x, unsigned long long y) { return x > y ? x : y; });
    // chunk sum of the weights relative to the chunk maximum (at most 32
    // weights below 2^25 each per thread)
    const float T = a.temperature[r];
    unsigned long long wsum = 0;
    if (T > 0.0f && a.draft && xmax > -INFINITY && xmax < INFINITY) {
        const float cT = sp_c(T);
        uint32_t s32 = 0;
#pragma unroll
        for (int e = 0; e < SP_EPT; e++) s32 += sp_weight(x[e], xmax, cT);
        wsum = s32;
        wsum = zs_wave_reduce(wsum, [](unsigned long long x, unsigned long long y) { return x + y; });
    }
    if (zs_lane() == 0) { gsh[zs_wid()] = best; wsh[zs_wid()] = wsum; }
    __syncthreads();
    if (threadIdx.x == 0) {
        unsigned long long ws = 0;
        for (int i = 0; i < SP_NT / 64; i++) { best = gsh[i] > best ? gsh[i] : best; ws += wsh[i]; }
        zs_spec_chunk& o = a.cst[((size_t)r * a.npos_max + pos) * a.nch + c];
        o.xmax = xmax;
        o.flags = fl;
        o.amax_val = best ? zs_key_to_float((uint32_t)(best >> 32)) : -INFINITY;
        o.amax_idx = best ? 0xffffffffu - (uint32_t)(best & 0xffffffffull) : 0xffffffffu;
        o.wsum = ws;
    }
}

// The same per (row, position) by one workgroup walking the row's chunks once,
// two at a time. One workgroup per CU (its LDS request keeps a second one out):
// the verification then leaves most of each CU to the sampler's kernels when
// the two run side by side.
#define SR_NT 1024
#define SR_NW (SR_NT / 64)
#define SR_EPT (SP_CH / SR_NT)  // 8 elements per thread, as 2 float4
#define SR_PAIR 2               // chunks loaded together
#define SR_LDS_HOLD 90000       // bytes of LDS requested to keep occupancy at one workgroup per CU
__device__ __forceinline__ void sr_load(const float* row, uint32_t base, uint32_t V, float* x) {
#pragma unroll
    for (int j = 0; j < SR_EPT / 4; j++) {
        const uint32_t id = base + (j * SR_NT + threadIdx.x) * 4;
        float4 v = make_float4(-INFINITY, -INFINITY, -INFINITY, -INFINITY);
        if (id < V) v = *reinterpret_cast<const float4*>(row + id);
        x[4 * j] = v.x; x[4 * j + 1] = v.y; x[4 * j + 2] = v.z; x[4 * j + 3] = v.w;
    }
    if (base + SP_CH > V) {  // ids past V read as -inf
#pragma unroll
        for (int e = 0; e < SR_EPT; e++)
            if (base + ((e >> 2) * SR_NT + threadIdx.x) * 4 + (e & 3) >= V) x[e] = -INFINITY;
    }
}
__device__ __forceinline__ uint32_t sr_id(uint32_t base, int e) {
    return base + ((e >> 2) * SR_NT + threadIdx.x) * 4 + (e & 3);
}

__global__ __launch_bounds__(SR_NT) void zs_k_spec_row(zs_spec_args a) {
    extern __shared__ uint32_t hold[];  // occupancy limiter only
    const uint32_t pos = blockIdx.x, r = blockIdx.y;
    const uint32_t V = a.V;
    const uint32_t nch = (V + SP_CH - 1) / SP_CH;
    __shared__ float wz[SR_PAIR][SR_NW];
    __shared__ uint32_t wf[ZS_MAX_CHUNKS][SR_NW];
    __shared__ unsigned long long wb[ZS_MAX_CHUNKS][SR_NW];
    __shared__ unsigned long long ws[ZS_MAX_CHUNKS][SR_NW];
    __shared__ float cz[ZS_MAX_CHUNKS];
    if (threadIdx.x == 0) hold[0] = 0;  // the request is used, so it is kept
    const float T = a.temperature[r];
    const bool weights = T > 0.0f && a.draft;
    const float cT = weights ? sp_c(T) : 1.0f;
    const float* row = sp_row(a, r, pos);
    const int lane = zs_lane(), wid = zs_wid();
    zs_spec_chunk* cs = a.cst + ((size_t)r * a.npos_max + pos) * a.nch;
    for (uint32_t c0 = 0; c0 < nch; c0 += SR_PAIR) {
        float x[SR_PAIR][SR_EPT];
#pragma unroll
        for (int h = 0; h < SR_PAIR; h++) sr_load(row, (c0 + h) * SP_CH, V, x[h]);
#pragma unroll
        for (int h = 0; h < SR_PAIR; h++) {
            const uint32_t c = c0 + h;
            if (c >= nch) break;
            const uint32_t base = c * SP_CH;
            float bv = -INFINITY;
            int be = -1;
            bool nan = false;
#pragma unroll
            for (int e = 0; e < SR_EPT; e++) {
                const float xv = x[h][e];
                nan |= xv != xv;
                if (xv > bv) { bv = xv; be = e; }
            }
            uint32_t fl = nan ? 1u : 0u;
            unsigned long long best = be < 0 ? 0ull
                : ((unsigned long long)zs_total_key(bv == 0.0f ? 0.0f : bv) << 32) | (0xffffffffu - sr_id(base, be));
            const float xmax = wave_max_f(bv);
            fl = wave_or_u(fl);
            best = zs_wave_reduce(best, [](unsigned long long x, unsigned long long y) { return x > y ? x : y; });
            if (lane == 0) { wz[h][wid] = xmax; wf[c][wid] = fl; wb[c][wid] = best; }
        }
        __syncthreads();
        // chunk maxima, then the chunk weight sums from the registers
#pragma unroll
        for (int h = 0; h < SR_PAIR; h++) {
            const uint32_t c = c0 + h;
            if (c >= nch) break;
            float m = -INFINITY;
            for (int w = 0; w < SR_NW; w++) m = fmaxf(m, wz[h][w]);
            if (threadIdx.x == 0) cz[c] = m;
            unsigned long long s = 0;
            if (weights && m > -INFINITY && m < INFINITY) {
                uint32_t s32 = 0;  // at most 8 weights below 2^25 each
#pragma unroll
                for (int e = 0; e < SR_EPT; e++) s32 += sp_weight(x[h][e], m, cT);
                s = s32;
                s = zs_wave_reduce(s, [](unsigned long long x, unsigned long long y) { return x + y; });
            }
            if (lane == 0) ws[c][wid] = s;
        }
        __syncthreads();
    }
    if (threadIdx.x < nch) {
        const uint32_t c = threadIdx.x;
        uint32_t fl = 0;
        unsigned long long best = 0, s = 0;
        for (int w = 0; w < SR_NW; w++) {
            fl |= wf[c][w];
            best = wb[c][w] > best ? wb[c][w] : best;
            s += ws[c][w];
        }
        if (cz[c] == INFINITY) fl |= 2u;
        zs_spec_chunk& o = cs[c];
        o.xmax = cz[c];
        o.flags = fl;
        o.amax_val = best ? zs_key_to_float((uint32_t)(best >> 32)) : -INFINITY;
        o.amax_idx = best ? 0xffffffffu - (uint32_t)(best & 0xffffffffull) : 0xffffffffu;
        o.wsum = s;
    }
}

// bit length of a u128
__device__ __forceinline__ int sp_bitlen(u128 v) {
    const unsigned long long hi = (unsigned long long)(v >> 64), lo = (unsigned long long)v;
    return hi ? 128 - __clzll((long long)hi) : (lo ? 64 - __clzll((long long)lo) : 0);
}
// u128 helpers
struct u128p { unsigned long long lo, hi; };
__device__ __forceinline__ u128 u128_of(u128p v) { return ((u128)v.hi << 64) | v.lo; }
__device__ __forceinline__ u128p u128p_of(u128 v) { return {(unsigned long long)v, (unsigned long long)(v >> 64)}; }
__device__ __forceinline__ u128 shfl_up_u128(u128 v, int d) {
    u128p p = u128p_of(v);
    p.lo = __shfl_up(p.lo, d, 64);
    p.hi = __shfl_up(p.hi, d, 64);
    return u128_of(p);
}
template <int J>
__device__ __forceinline__ u128 xor_add_u128(u128 v) {
    u128p p = u128p_of(v);
    p.lo = zs_lane_xor<J>(p.lo);
    p.hi = zs_lane_xor<J>(p.hi);
    return v + u128_of(p);
}
__device__ __forceinline__ u128 wave_sum_u128(u128 v) {
    return xor_add_u128<1>(xor_add_u128<2>(xor_add_u128<4>(xor_add_u128<8>(xor_add_u128<16>(xor_add_u128<32>(v))))));
}

// pass 2: accept / reject decisions of a row and the sums of its draw, by an
// SP_NT-thread workgroup: the waves take the positions in turn (maximum, first
// argmax, weight sum and the draft id's weight of a position in one visit to
// its chunk records), then one lane per draft makes its accept test and the
// first rejection decides (one wave per row visiting the positions one after
// the other, and the drafts' tests one after the other, took a launch of 18 us
// on 64 rows of 9 positions). In a launch of its own (zs_k_spec_decide), or, of
// at most SP_DECIDE_WGS workgroups, by every workgroup of the residual pass for
// itself: that saves the launch but repeats the work once a chunk.
#define SP_NPOS (2 * ZS_SPEC_KMAX + 1)
struct sp_decision {
    zs_spec_row row;
    uint32_t accepted, next;   // next: greedy rows (row.mode 0) only
    unsigned long long slo[SP_NPOS], shi[SP_NPOS];   // weight sums
    unsigned long long wt[SP_NPOS];                  // weight of the draft id at its target / draft position
    float m[SP_NPOS];
    uint32_t am[SP_NPOS], fl[SP_NPOS];
};
__device__ __forceinline__ void sp_decide(const zs_spec_args& a, uint32_t r, sp_decision& S) {
    const uint32_t k = a.k, V = a.V, lane = (uint32_t)zs_lane(), wid = (uint32_t)zs_wid();
    const uint32_t nch = (V + SP_CH - 1) / SP_CH;
    const uint32_t npos = a.draft ? 2 * k + 1 : k + 1;
    const float T = a.temperature[r];
    const bool weights = T > 0.0f && a.draft;
    const float cT = weights ? sp_c(T) : 0.0f;
    const uint32_t* drafts = a.draft_ids + (size_t)r * k;
    constexpr uint32_t PU = 3;   // positions of a wave with their first loads in flight
    for (uint32_t p0 = wid; p0 < npos; p0 += PU * (SP_NT / 64)) {
        zs_spec_chunk q[PU];
        uint32_t d[PU];
        float xd[PU], xm[PU];   // the draft id's logit and its chunk's maximum
#pragma unroll
        for (uint32_t u = 0; u < PU; u++) {
            const uint32_t p = p0 + u * (SP_NT / 64);
            q[u].xmax = -INFINITY; q[u].flags = 0; q[u].amax_val = -INFINITY; q[u].amax_idx = 0xffffffffu; q[u].wsum = 0;
            d[u] = 0xffffffffu;
            if (p >= npos) continue;
            if (lane < nch) q[u] = a.cst[((size_t)r * a.npos_max + p) * a.nch + lane];
            if (weights && p != k) d[u] = drafts[p < k ? p : p - k - 1];
        }
#pragma unroll
        for (uint32_t u = 0; u < PU; u++) {
            const uint32_t p = p0 + u * (SP_NT / 64);
            xd[u] = xm[u] = 0.0f;
            if (p < npos && d[u] < V) {
                xd[u] = sp_row(a, r, p)[d[u]];
                xm[u] = a.cst[((size_t)r * a.npos_max + p) * a.nch + d[u] / SP_CH].xmax;
            }
        }
#pragma unroll
        for (uint32_t u = 0; u < PU; u++) {
            const uint32_t p = p0 + u * (SP_NT / 64);
            if (p >= npos) continue;
            const zs_spec_chunk* cs = a.cst + ((size_t)r * a.npos_max + p) * a.nch;
            auto key = [](const zs_spec_chunk& c) -> unsigned long long {   // (value key, ~id) of the first maximum
                return c.amax_idx == 0xffffffffu ? 0ull : ((unsigned long long)zs_total_key(c.amax_val) << 32) | (0xffffffffu - c.amax_idx);
            };
            float m = q[u].xmax;
            uint32_t fl = q[u].flags;
            unsigned long long best = key(q[u]);
            for (uint32_t c = lane + 64; c < nch; c += 64) {
                const zs_spec_chunk w = cs[c];
                m = fmaxf(m, w.xmax);
                fl |= w.flags;
                const unsigned long long kw = key(w);
                best = kw > best ? kw : best;
            }
            m = wave_max_f(m);
            fl = wave_or_u(fl);
            best = zs_wave_reduce(best, [](unsigned long long x, unsigned long long y) { return x > y ? x : y; });
            u128 s = 0;
            unsigned long long wt = 0;
            if (weights && !fl && m > -INFINITY) {
                // sum_c F_c * S_c, and P_d = w_d * F_c of the chunk holding d
                if (lane < nch) s = (u128)((unsigned long long)sp_weight(q[u].xmax, m, cT) * q[u].wsum);
                for (uint32_t c = lane + 64; c < nch; c += 64) s += (u128)((unsigned long long)sp_weight(cs[c].xmax, m, cT) * cs[c].wsum);
                s = wave_sum_u128(s);
                if (d[u] < V) wt = (unsigned long long)sp_weight(xd[u], xm[u], cT) * sp_weight(xm[u], m, cT);
            }
            if (lane == 0) {
                S.m[p] = m;
                S.fl[p] = (fl || m == -INFINITY) ? 1u : 0u;
                S.am[p] = best ? 0xffffffffu - (uint32_t)best : 0u;
                S.slo[p] = (unsigned long long)s;
                S.shi[p] = (unsigned long long)(s >> 64);
                S.wt[p] = wt;
            }
        }
    }
    __syncthreads();
    if (wid == 0) {
        bool bad = !weights;
        for (uint32_t p = lane; p < npos; p += 64) bad |= S.fl[p] != 0u;
        const bool degenerate = __ballot(bad) != 0ull;
        const uint32_t dr = lane < k ? drafts[lane] : 0u;
        // lane i: whether draft i is turned away
        bool rej = false;
        u128 sp = 0, sq = 0;
        int sh = 0;
        if (lane < k) {
            if (degenerate) {
                rej = S.am[lane] != dr;
            } else {
                sp = ((u128)S.shi[lane] << 64) | S.slo[lane];
                sq = ((u128)S.shi[k + 1 + lane] << 64) | S.slo[k + 1 + lane];
                sh = max(0, sp_bitlen(sp | sq) - 40);
                const unsigned long long Ps = (unsigned long long)(sp >> sh), Qs = (unsigned long long)(sq >> sh);
                const uint32_t U = zs_philox_u32(a.seed[r], a.counter[r], 1u + lane);
                const u128 lhs = ((u128)U * S.wt[k + 1 + lane]) * Ps;  // < 2^122
                const u128 rhs = ((u128)S.wt[lane] * Qs) << 32;       // < 2^122
                rej = dr >= V || !(lhs <= rhs);
            }
        }
        const unsigned long long rm = __ballot(rej);
        const uint32_t i = rm ? (uint32_t)__ffsll((long long)rm) - 1u : k;
        if (degenerate) {
            if (lane == 0) {
                S.accepted = i;
                S.next = S.am[i];
                S.row.mode = 0;
            }
        } else if (lane == (i < k ? i : 0u)) {
            zs_spec_row o;
            o.mode = 1;
            o.pos = i;
            o.m_t = S.m[i];
            o.m_d = 0.f;
            o.ps = o.qs = 0;
            if (i == k) {
                o.residual = 0;
                o.sum_lo = S.slo[k];
                o.sum_hi = S.shi[k];
                o.word = zs_philox_u32(a.seed[r], a.counter[r], 1u + 2 * k);
            } else {
                o.residual = 1;
                o.m_d = S.m[k + 1 + i];
                o.ps = (unsigned long long)(sp >> sh);
                o.qs = (unsigned long long)(sq >> sh);
                o.sum_lo = S.slo[i];  // the target's sum: the draw when R is all 0
                o.sum_hi = S.shi[i];
                o.word = zs_philox_u32(a.seed[r], a.counter[r], 1u + k + i);
            }
            S.accepted = i;
            S.row = o;
        }
    }
    __syncthreads();
}

// Draw weight of id v (given its target / draft logits and its chunk's maxima
// and scales): P, or the residual max(0, P Qs - Q Ps) (below 2^90).
struct sp_chunk_w {
    float mt, md;
    unsigned long long ft, fd;
};
// tpos: the target position the draw's P comes from (pos after a rejection,
// k after k acceptances)
__device__ __forceinline__ sp_chunk_w sp_chunk_scales(const zs_spec_args& a, uint32_t r, const zs_spec_row& s, uint32_t c,
                                                      float cT, uint32_t tpos) {
    sp_chunk_w w;
    w.mt = a.cst[((size_t)r * a.npos_max + tpos) * a.nch + c].xmax;
    w.ft = sp_weight(w.mt, s.m_t, cT);
    w.md = 0.0f;
    w.fd = 0;
    if (s.residual) {
        w.md = a.cst[((size_t)r * a.npos_max + a.k + 1 + s.pos) * a.nch + c].xmax;
        w.fd = sp_weight(w.md, s.m_d, cT);
    }
    return w;
}
__device__ __forceinline__ u128 spd_weight2(const zs_spec_row& s, const sp_chunk_w& cw, float cT, float xt, float xd) {
    const unsigned long long P = (unsigned long long)sp_weight(xt, cw.mt, cT) * cw.ft;
    if (!s.residual) return P;
    const unsigned long long Q = (unsigned long long)sp_weight(xd, cw.md, cT) * cw.fd;
    const u128 pp = (u128)P * s.qs, qq = (u128)Q * s.ps;
    return pp > qq ? pp - qq : 0;
}

__device__ __forceinline__ void sp_store(const zs_spec_args& a, uint32_t r, const sp_decision& S) {
    if (threadIdx.x != 0) return;
    a.accepted[r] = S.accepted;
    if (S.row.mode == 0) a.next[r] = S.next;
    a.rs[r] = S.row;
}
__global__ __launch_bounds__(SP_NT) void zs_k_spec_decide(zs_spec_args a) {
    __shared__ sp_decision S;
    sp_decide(a, blockIdx.x, S);
    sp_store(a, blockIdx.x, S);
}

// pass 3: chunk sums of the residual weights (rows that rejected a draft);
// DECIDE: the decision in front, stored by chunk 0's workgroup, as long as all
// workgroups are resident at once (4 a CU): past that a second round repeats
// it. Rejection sampling alone, in a launch of its own / in front (us a call; 3,
// 9 and 17 positions): 32 x 151936 (608 workgroups, 9 positions) 68 / 67,
// 64 x 128256 (1024) 91 / 90; 60 x 151936 (1140) 54 / 57, 94 / 100, 144 / 149;
// 80 x 128256 (1280) 53 / 56, 96 / 102, 157 / 166; 128 x 128256 (2048) 68 / 71,
// 138 / 145, 237 / 253; 256 x 151936 (4864, 9 positions) 302 / 323.
#define SP_DECIDE_WGS 1024u
template <bool DECIDE>
__global__ __launch_bounds__(SP_NT) void zs_k_spec_rsum(zs_spec_args a) {
    const uint32_t c = blockIdx.x, r = blockIdx.y;
    const uint32_t base = c * SP_CH;
    if (base >= a.V) return;
    zs_spec_row s;
    if constexpr (DECIDE) {
        __shared__ sp_decision S;
        sp_decide(a, r, S);
        s = S.row;
        if (c == 0) sp_store(a, r, S);
    } else {
        s = a.rs[r];
    }
    if (s.mode != 1 || !s.residual) return;
    __shared__ unsigned long long lo[SP_NT / 64], hi[SP_NT / 64];
    const float cT = sp_c(a.temperature[r]);
    const sp_chunk_w cw = sp_chunk_scales(a, r, s, c, cT, s.pos);
    float xt[SP_EPT], xd[SP_EPT];
    sp_load(sp_row(a, r, s.pos), base, a.V, xt);
    sp_load(sp_row(a, r, a.k + 1 + s.pos), base, a.V, xd);
    u128 acc = 0;
#pragma unroll
    for (int e = 0; e < SP_EPT; e++)
        acc += spd_weight2(s, cw, cT, xt[e], xd[e]);
    acc = wave_sum_u128(acc);
    if (zs_lane() == 0) { lo[zs_wid()] = (unsigned long long)acc; hi[zs_wid()] = (unsigned long long)(acc >> 64); }
    __syncthreads();
    if (threadIdx.x == 0) {
        u128 t = 0;
        for (int i = 0; i < SP_NT / 64; i++) t += ((u128)hi[i] << 64) | lo[i];
        zs_spec_chunk& o = a.cst[((size_t)r * a.npos_max + 0) * a.nch + c];
        o.rlo = (unsigned long long)t;
        o.rhi = (unsigned long long)(t >> 64);
    }
}

// pass 4: one workgroup per row -- the replacement / bonus draw: the chunk
// holding the target from the chunk sums, then the first id of that chunk whose
// inclusive prefix exceeds the target
__global__ __launch_bounds__(SP_BIG_NT) void zs_k_spec_draw(zs_spec_args a) {
    const uint32_t r = blockIdx.x;
    __shared__ unsigned long long lo[SP_BIG_NT / 64], hi[SP_BIG_NT / 64];
    __shared__ int imin[SP_BIG_NT / 64];
    __shared__ uint32_t csel;
    __shared__ unsigned long long clo, chi, rzero;
    zs_spec_row s = a.rs[r];
    if (s.mode != 1) return;
    const float cT = sp_c(a.temperature[r]);
    const int t = threadIdx.x;
    const uint32_t V = a.V;
    const uint32_t nch = (V + SP_CH - 1) / SP_CH;
    const zs_spec_chunk* c0 = a.cst + ((size_t)r * a.npos_max + 0) * a.nch;                   // residual sums
    const zs_spec_chunk* cp = a.cst + ((size_t)r * a.npos_max + (s.residual ? s.pos : a.k)) * a.nch;  // P sums
    if (t < 64) {
        // residual total; p == q exactly leaves no residual: draw from the target
        u128 rt = 0;
        if (s.residual)
            for (uint32_t c = t; c < nch; c += 64) rt += ((u128)c0[c].rhi << 64) | c0[c].rlo;
        rt = wave_sum_u128(rt);
        const bool resid = s.residual && rt != 0;
        const u128 total = resid ? rt : (((u128)s.sum_hi << 64) | s.sum_lo);
        // floor(word * total / 2^32) without overflow: total < 2^108
        const u128 target = (((u128)s.word * (unsigned long long)(total >> 64)) << 32) +
                            (((u128)s.word * (unsigned long long)total) >> 32);
        // chunk prefix over the lanes (nch <= 64 for the vocab limit)
        u128 w = 0;
        if ((uint32_t)t < nch)
            w = resid ? (((u128)c0[t].rhi << 64) | c0[t].rlo)
                      : (u128)((unsigned long long)sp_weight(cp[t].xmax, s.m_t, cT) * cp[t].wsum);
        u128 inc = w;
        for (int d = 1; d < 64; d <<= 1) {
            u128 y = shfl_up_u128(inc, d);
            if (t >= d) inc += y;
        }
        const bool hit = w > 0 && inc > target;
        const unsigned long long bal = __ballot(hit);
        const int first = bal ? __ffsll((long long)bal) - 1 : -1;
        const u128 before = __shfl(first >= 0 ? (unsigned long long)(inc - w) : 0ull, first >= 0 ? first : 0, 64);
        const u128 beforeh = __shfl(first >= 0 ? (unsigned long long)((inc - w) >> 64) : 0ull, first >= 0 ? first : 0, 64);
        if (t == 0) {
            csel = first >= 0 ? (uint32_t)first : 0xffffffffu;
            const u128 rem = target - ((beforeh << 64) | (unsigned long long)before);
            clo = (unsigned long long)rem;
            chi = (unsigned long long)(rem >> 64);
            rzero = resid ? 1ull : 0ull;
        }
    }
    __syncthreads();
    const uint32_t c = csel;
    if (c == 0xffffffffu) {
        if (t == 0) a.next[r] = V - 1;
        return;
    }
    const uint32_t tpos = s.residual ? s.pos : a.k;
    if (!rzero) s.residual = 0;
    const u128 rem = ((u128)chi << 64) | clo;  // target minus the weight of the chunks before
    const uint32_t base = c * SP_CH;
    const sp_chunk_w cw = sp_chunk_scales(a, r, s, c, cT, tpos);
    // 8192 ids, 8 per thread in two float4 of each row
    const float* rt = sp_row(a, r, s.pos);
    const float* rd = s.residual ? sp_row(a, r, a.k + 1 + s.pos) : rt;
    u128 w[8], loc = 0;
#pragma unroll
    for (int h = 0; h < 2; h++) {
        const uint32_t id = base + (h * SP_BIG_NT + t) * 4;
        float4 vt = make_float4(-INFINITY, -INFINITY, -INFINITY, -INFINITY), vd = vt;
        if (id < V) {
            vt = *reinterpret_cast<const float4*>(rt + id);
            vd = *reinterpret_cast<const float4*>(rd + id);
        }
        const float xt[4] = {vt.x, vt.y, vt.z, vt.w}, xd[4] = {vd.x, vd.y, vd.z, vd.w};
#pragma unroll
        for (int q = 0; q < 4; q++) {
            w[4 * h + q] = id + q < V ? spd_weight2(s, cw, cT, xt[q], xd[q]) : 0;
        }
    }
    // inclusive prefix in id order: ids of thread t are base + 4t..4t+3 (h=0)
    // and base + 4096 + 4t..+3 (h=1); scan the two halves one after the other
    int found = ZS_BIGI;
    u128 carry = 0;
#pragma unroll
    for (int h = 0; h < 2; h++) {
        u128 l = w[4 * h] + w[4 * h + 1] + w[4 * h + 2] + w[4 * h + 3];
        u128 inc = l;
        for (int d = 1; d < 64; d <<= 1) {
            u128 y = shfl_up_u128(inc, d);
            if (zs_lane() >= d) inc += y;
        }
        if (zs_lane() == 63) { lo[zs_wid()] = (unsigned long long)inc; hi[zs_wid()] = (unsigned long long)(inc >> 64); }
        __syncthreads();
        u128 pre = 0, tot = 0;
        for (int i = 0; i < SP_BIG_NT / 64; i++) {
            u128 wv = ((u128)hi[i] << 64) | lo[i];
            if (i < zs_wid()) pre += wv;
            tot += wv;
        }
        __syncthreads();
        u128 run = carry + pre + inc - l;
        int my = ZS_BIGI;
#pragma unroll
        for (int q = 0; q < 4; q++) {
            run += w[4 * h + q];
            if (my == ZS_BIGI && w[4 * h + q] > 0 && run > rem) my = h * 4 * SP_BIG_NT + 4 * t + q;
        }
        const int f = block_min_i<SP_BIG_NT>(my, imin);
        if (found == ZS_BIGI) found = f;
        carry += tot;
    }
    if (t == 0) a.next[r] = found == ZS_BIGI ? V - 1 : base + (uint32_t)found;
}

extern "C" int zs_spec_launch(const zs_spec_args& a, const zs_prof& prof, hipStream_t stream) {
    const uint32_t npos = a.draft ? 2 * a.k + 1 : a.k + 1;
    const uint32_t nch = (a.V + SP_CH - 1) / SP_CH;
    int ev = 0;
    auto mark = [&](const char* name) {
        if (!prof.on) return;
        prof.names[ev] = name;
        (void)hipEventRecord((hipEvent_t)prof.events[ev], stream);
        ev++;
    };
    mark(nullptr);
    if (a.background) {
        hipLaunchKernelGGL(zs_k_spec_row, dim3(npos, a.B), dim3(SR_NT), SR_LDS_HOLD, stream, a);
        mark("zs_k_spec_row");
    } else {
        const uint64_t parts = a.beside ? ((uint64_t)nch * npos * a.B + SP_PART - 1) / SP_PART : 1;
        const uint32_t per = (uint32_t)((a.B + parts - 1) / parts);
        for (uint32_t r0 = 0; r0 < a.B; r0 += per)
            hipLaunchKernelGGL(zs_k_spec_chunk, dim3(nch, npos, std::min(per, a.B - r0)), dim3(SP_NT), 0, stream, a, r0);
        mark("zs_k_spec_chunk");
    }
    // (without draft logits every row is verified greedily: the decision is all)
    if (a.draft && (uint64_t)nch * a.B <= SP_DECIDE_WGS) {
        hipLaunchKernelGGL(zs_k_spec_rsum<true>, dim3(nch, a.B), dim3(SP_NT), 0, stream, a);
    } else {
        hipLaunchKernelGGL(zs_k_spec_decide, dim3(a.B), dim3(SP_NT), 0, stream, a);
        if (a.draft) hipLaunchKernelGGL(zs_k_spec_rsum<false>, dim3(nch, a.B), dim3(SP_NT), 0, stream, a);
    }
    if (a.draft) hipLaunchKernelGGL(zs_k_spec_draw, dim3(a.B), dim3(SP_BIG_NT), 0, stream, a);
    mark("zs_k_spec_draw");
    if (prof.on) *prof.n = ev - 1;
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

// ---------------------------------------------------------------------------
// zs_spec_verify_static: the same verification without a context, for callers
// that cannot allocate (HIP graph capture, serving loops that forbid
// hipMalloc). The chunk records and per-row state live in `scratch`, one copy
// per GPU for the life of the process. The host never passes the array's own
// name to a kernel (in host code it is only a stand-in for the symbol): the
// device address of each GPU's copy is looked up once with
// hipGetSymbolAddress, with that GPU current, and kept per device.
// Every kernel writes the records it later reads, so nothing needs clearing.
// Calls that overlap on one GPU share the array and race.
// ---------------------------------------------------------------------------
struct zs_spec_static_area {
    zs_spec_chunk cst[ZS_SPEC_STATIC_MAX_RECORDS];
    zs_spec_row rs[ZS_SPEC_STATIC_MAX_ROWS];
};
static __device__ __align__(256) zs_spec_static_area scratch;

#define ZS_STATIC_MAX_DEVICES 64
static zs_spec_static_area* g_static_area[ZS_STATIC_MAX_DEVICES];
static std::mutex g_static_mu;

// Device address of the current GPU's copy of `scratch` (looked up once per
// device), or null when the lookup fails.
static zs_spec_static_area* zs_spec_static_area_of(int dev) {
    if (dev < 0 || dev >= ZS_STATIC_MAX_DEVICES) return nullptr;
    std::lock_guard<std::mutex> lk(g_static_mu);
    if (!g_static_area[dev]) {
        void* p = nullptr;
        if (hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) != hipSuccess || !p) return nullptr;
        g_static_area[dev] = static_cast<zs_spec_static_area*>(p);
    }
    return g_static_area[dev];
}

extern "C" int zs_spec_verify_static(const zs_spec_batch* b, void* stream) {
    if (!b) return ZS_EINVAL;
    if (b->B == 0) return ZS_OK;
    if (b->V == 0 || b->k > ZS_SPEC_KMAX || b->B > ZS_SPEC_STATIC_MAX_ROWS) return ZS_ELIMIT;
    if (!b->d_target || (b->k && !b->d_draft_ids) || !b->d_temperature || !b->d_seed || !b->d_counter ||
        !b->d_accepted || !b->d_next)
        return ZS_EINVAL;
    if (b->ld < b->V || (b->ld & 3u) || ((uintptr_t)b->d_target & 15u) || ((uintptr_t)b->d_draft & 15u))
        return ZS_EINVAL;
    if (b->flags & ~(uint32_t)ZS_SPEC_BACKGROUND) return ZS_EINVAL;
    const uint32_t k = b->k;
    const bool draft = k && b->d_draft;
    const uint64_t npos = draft ? 2ull * k + 1 : (uint64_t)k + 1;
    const uint64_t nch = (b->V + SP_CH - 1) / SP_CH;
    if ((uint64_t)b->B * npos * nch > ZS_SPEC_STATIC_MAX_RECORDS) return ZS_ELIMIT;
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return ZS_EHIP;
    zs_spec_static_area* area = zs_spec_static_area_of(dev);
    if (!area) return ZS_EHIP;
    zs_spec_args a{};
    a.B = b->B; a.V = b->V; a.k = k; a.ld = b->ld;
    a.target = b->d_target; a.draft = k ? b->d_draft : nullptr; a.draft_ids = b->d_draft_ids;
    a.temperature = b->d_temperature; a.seed = b->d_seed; a.counter = b->d_counter;
    a.accepted = b->d_accepted; a.next = b->d_next;
    a.cst = area->cst;        // device address of this GPU's copy
    a.rs = area->rs;
    a.nch = (uint32_t)nch;
    a.npos_max = (uint32_t)npos;
    a.background = (b->flags & ZS_SPEC_BACKGROUND) ? 1u : 0u;
    zs_prof prof{0, nullptr, nullptr, nullptr};
    return zs_spec_launch(a, prof, (hipStream_t)stream) ? ZS_EHIP : ZS_OK;
}
