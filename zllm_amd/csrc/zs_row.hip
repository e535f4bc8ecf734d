// zs_row.hip -- the front of the sampler step, one 512-thread workgroup per
// row: everything of a row that needs the whole row, with no other workgroup
// involved and therefore no device-scope synchronisation and no launch
// boundary between the phases.
//
// Reference semantics (per row, in the order of rest.rs:2594-2624):
//   x~ = apply_mask(x)                    logit_fsm.rs:247-270 (bans, allow bits)
//   y  = adjust_logits(x~)                decode_ctrl.rs:107-126
//   token = sample_with_rng(y, cfg, r)    sampler.rs:31-128
//   logprobs / token_uncertainty on x~    logprobs.rs:34-54, hallucination.rs:129-154
//
// Phases of zs_k_row:
//   P0  patches: the row's ban / bias / count-map entries merged into one list
//       sorted by id with the exact patched y of every listed id
//       (decode_ctrl.rs:107-126 operation order; lists of any length: the
//       first ZS_PATCH_LDS entries in LDS, the rest in row scratch), ranked by
//       a bitmap of the patched ids with per-word prefix counts, and stored
//       for the later kernels;
//   P1  the row's maxima and candidate lists (the observers' top entries by
//       (x~ desc, id asc) for top_logprobs / margin; the sampler's top-k by
//       (z desc, id asc), sampler.rs:53-64: its k-th key is the threshold; or
//       every finite z when no top-k applies and at most ZS_SMALL_CAP are
//       finite) from the group maxima that zs_k_scan took over the whole GPU
//       (rw_groups), or from a masked row's gathered ids. Rows these cannot
//       serve (narrow rows, long patch lists, lists that would overflow) read
//       their logits here, keeping the lists in LDS behind a rising
//       threshold (greedy argmax: the last maximal element, a NaN restarts
//       the fold, sampler.rs:35-43);
//   decisions: greedy / non-finite rows get their token; rows whose survivors
//       fit ZS_SMALL_CAP are sampled exactly, up to 64 by one wave
//       (small_path_wave), more by the workgroup (rw_small_wg); other rows are
//       "big" and continue in zs_sample.hip;
//   state: which exact sums the row needs (zs_sums.hip: the observers' S and
//       entropy, a big row's sampler S), over the whole row or over the
//       allowed ids a masked row gathered to row scratch.
#include <hip/hip_runtime.h>
#ifdef ZS_WALK_DEBUG
// Debug builds: wall-clock time of zs_k_row's phases (0-5, row count in 7; of
// rw_groups the corrected maxima in 6, the thresholds in 15, both within 2)
// and of the small path's (8-14), summed over rows (zs_dbg_row_stats).
__device__ unsigned long long rw_dbg[16];
#define ZS_SP_T(i)                                               \
    do {                                                         \
        if (zs_lane() == 0) {                                    \
            const unsigned long long c_ = wall_clock64();        \
            atomicAdd(&rw_dbg[8 + (i)], c_ - sp_t0);             \
            sp_t0 = c_;                                          \
        }                                                        \
    } while (0)
#endif
#include "zs_sampler.h"

#define RW_NT 512
#define RW_NW (RW_NT / 64)
#define RW_G 2048          // ids per tile: one float4 per thread
#define RW_BUF 2048        // candidate buffer entries (per list)
#define RW_KEEP 1024       // a list above this is compacted to its top K

struct rw_shared {
    uint32_t pid[4096];             // the patch list's head (ZS_PATCH_LDS): ids (sorted) | flags << 30
    float py[4096];                 // their y
    union {
        struct {
            unsigned long long o[RW_BUF];         // P1: observer candidates
            unsigned long long s[RW_BUF];         // P1: sampler candidates
        } b;
    } u;
    alignas(16) float sval[ZS_SMALL_CAP];   // also the small path's scratch
    uint32_t sidx[ZS_SMALL_CAP];
    uint32_t cand_id[ZS_OBS_CAND];
    float cand_x[ZS_OBS_CAND];
    uint32_t ru[6][RW_NW];
    float rf[3][RW_NW];
    float fthr[2];                  // candidate thresholds as values
    float fcut[2];                  // largest values cut from the lists
    unsigned long long rl[RW_NW];
    unsigned long long n_os;        // rw_groups: entries of the observers' list | of the sampler's << 32
    uint32_t n_surv, tok;
    uint32_t n_gl;                  // groups listed by rw_groups
    uint32_t ovf[3];                // first tile that lost a list entry, per group slot
    float fsh;
    uint32_t sel_hist[2][256];      // list selection: digit histogram (double buffered)
    uint32_t sel_mm[3][RW_NW];      // list selection: per-wave member count, key min / max
    uint32_t sel_n;                 // list selection: places taken by the gather
    uint32_t inf_lim;               // observers: largest id whose -inf can enter the list
    uint32_t g_n, g_done;           // masked rows: allowed ids gathered to row scratch, gather done
    uint32_t sel_st[2];             // rw_kth_key: chosen digit, rank inside it
};
// The workgroup's LDS (one object, so that functions outside the kernel
// address it directly).
__shared__ rw_shared rw_sh;
// Bitmap of the row's patched ids, ceil(V / 32) words, followed by the number
// of patched ids before each word (dynamic LDS); behind them rw_patches' two
// bias bitmaps, then rw_groups' maxima in the same place.
extern __shared__ uint32_t rw_pbits[];
// Words of dynamic LDS: a CU's 160 KB less rw_shared and what the kernel's
// other functions declare (below 1 KB).
#define RW_DYN_WORDS ((163840u - (uint32_t)sizeof(rw_shared) - 1024u) / 4u)
// Words of each bias bitmap: the whole row up to about 180000 ids; the bias
// lists of wider rows are taken in windows of as many ids as fit.
__host__ __device__ __forceinline__ uint32_t rw_bias_words(uint32_t words) {
    const uint32_t fit = (RW_DYN_WORDS - 2u * words) / 2u;
    return words < fit ? words : fit;
}
static_assert(2u * (ZS_MAX_VOCAB / 32u) + 2048u <= RW_DYN_WORDS, "the widest row's bitmap, counts and bias windows fit");

#define RW_PF_SHIFT 30u

#ifdef ZS_WALK_DEBUG
#define RW_T(i)                                                  \
    do {                                                         \
        if (threadIdx.x == 0) {                                  \
            const unsigned long long c_ = wall_clock64();        \
            atomicAdd(&rw_dbg[i], c_ - rw_t0);                   \
            rw_t0 = c_;                                          \
        }                                                        \
    } while (0)
#else
#define RW_T(i) do { } while (0)
#endif

// A value every lane holds equally (read from LDS after a barrier), moved to
// a scalar register so that the compiler branches on it without exec masks.
__device__ __forceinline__ uint32_t rw_uni(uint32_t v) { return __builtin_amdgcn_readfirstlane(v); }
__device__ __forceinline__ float rw_unif(float v) { return __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(v))); }
// Sum of a u32 over the wave (no overflow check), uniform: pairs, quads,
// eights and rows of 16 by DPP permutations, then the rows by broadcasts;
// lane 63 ends with the total.
__device__ __forceinline__ uint32_t rw_wave_sum(uint32_t v) {
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0xB1, 0xf, 0xf, false);    // quad_perm [1,0,3,2]
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x4E, 0xf, 0xf, false);    // quad_perm [2,3,0,1]
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x141, 0xf, 0xf, false);   // row_half_mirror
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x140, 0xf, 0xf, false);   // row_mirror
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x142, 0xa, 0xf, false);   // row_bcast:15
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x143, 0xc, 0xf, false);   // row_bcast:31
    return (uint32_t)__builtin_amdgcn_readlane((int)v, 63);
}

// Inclusive scan of a u32 over the wave (no overflow check): shifts inside
// each row of 16 lanes, then the rows by broadcasts.
__device__ __forceinline__ uint32_t rw_wave_scan(uint32_t v) {
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x111, 0xf, 0xf, true);    // row_shr:1
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x112, 0xf, 0xf, true);    // row_shr:2
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x114, 0xf, 0xf, true);    // row_shr:4
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x118, 0xf, 0xf, true);    // row_shr:8
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x142, 0xa, 0xf, false);   // row_bcast:15
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x143, 0xc, 0xf, false);   // row_bcast:31
    return v;
}

// Workgroup barrier that orders LDS accesses only. __syncthreads() also waits
// for every outstanding global load of the calling wave, which would drain the
// loads the tile loops keep in flight ahead of the tile being processed.
__device__ __forceinline__ void rw_bar() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// Ascending sort of the m <= 256 entries at buf by one wave (called by the 64
// lanes of one wave; no barrier).
template <int E>
__device__ __forceinline__ void rw_wave_sort_e(unsigned long long* buf, uint32_t m) {
    const uint32_t lane = (uint32_t)zs_lane();
    unsigned long long k[E];
#pragma unroll
    for (int e = 0; e < E; e++) k[e] = lane * E + e < m ? buf[lane * E + e] : ~0ull;
    wave_sort_u64_e<E>(k);
#pragma unroll
    for (int e = 0; e < E; e++) if (lane * E + e < m) buf[lane * E + e] = k[e];
}
__device__ __forceinline__ void rw_wave_sort(unsigned long long* buf, uint32_t m) {
    if (m <= 64) rw_wave_sort_e<1>(buf, m);
    else if (m <= 128) rw_wave_sort_e<2>(buf, m);
    else rw_wave_sort_e<4>(buf, m);
}

// ---------------------------------------------------------------------------
// P0: merged patch list. The row's ban / bias / count entries (any number)
// are merged into one entry per patched id, in id order, with the exact
// patched y of the reference's per-token operation sequence: bans first
// (logit_fsm.rs:248-252), then the logit_bias entries in list order, then the
// penalty of the count map (decode_ctrl.rs:107-126). The ids' bitmap and its
// per-word prefix counts (dynamic LDS) give every patched id its rank in the
// list; the list itself is in row scratch (a.pstride entries per row), its
// first ZS_PATCH_LDS entries also in LDS for the row kernel's phases.
// Returns the number of patched ids.
// ---------------------------------------------------------------------------
#define ZS_PATCH_LDS 4096
__device__ __forceinline__ uint32_t rw_rank(uint32_t id, uint32_t words) {
    const uint32_t wd = rw_pbits[id >> 5];
    return rw_pbits[words + (id >> 5)] + __popc(wd & ((1u << (id & 31)) - 1u));
}

#define RW_PE 2   // list entries a thread keeps in registers
__device__ __forceinline__ int rw_patches(const zs_sargs& a, uint32_t r, const zs_row_params& P, rw_shared& sh) {
    const zs_batch& b = a.b;
    const uint32_t t = threadIdx.x, V = b.V;
    const uint32_t words = (V + 31) / 32;
    const uint32_t bw = rw_bias_words(words);
    uint32_t* seen = rw_pbits + 2 * words;   // bias ids met once, and more than once
    uint32_t* dup = seen + bw;
    const uint32_t ban0 = b.d_ban_off ? b.d_ban_off[r] : 0, ban1 = b.d_ban_off ? b.d_ban_off[r + 1] : 0;
    const uint32_t bi0 = b.d_bias_off ? b.d_bias_off[r] : 0, bi1 = b.d_bias_off ? b.d_bias_off[r + 1] : 0;
    uint32_t c0 = b.d_cnt_off ? b.d_cnt_off[r] : 0, c1 = b.d_cnt_off ? b.d_cnt_off[r + 1] : 0;
    if (!zs_penalty_active(P)) c1 = c0;  // counts only matter when penalties are active
    const uint32_t nb = ban1 - ban0, nbi = bi1 - bi0, nc = c1 - c0, ne = nb + nbi + nc;
    const uint32_t nsub = (V + ZS_SUB - 1) / ZS_SUB;
    uint32_t* psub = a.p_sub + (size_t)r * (a.max_subs + 1);
    uint32_t* out_id = a.p_id + (size_t)r * a.pstride;
    uint32_t* out_fl = a.p_flags + (size_t)r * a.pstride;
    float* out_y = a.p_y + (size_t)r * a.pstride;
    if (ne == 0) {
        // (the bitmap is read only for rows with patches)
        if (t == 0) a.p_cnt[r] = 0;
        for (uint32_t j = t; j <= nsub; j += RW_NT) psub[j] = 0;
        __syncthreads();
        return 0;
    }
    // Entry i of the row's three lists (bans, biases, counts in this order):
    // its id and its value (bias or count, as bits). The first RW_PE entries
    // of a thread stay in registers with their logit, so that every list
    // element of a row of up to 1024 is loaded once, all loads at once: the
    // lists re-read per step and the logits gathered word by word took
    // 10.5 us on 256 counts, 5.5 now.
    const bool masked = (P.flags & ZS_ROW_MASKED) && b.d_allow_bits;
    auto id_of = [&](uint32_t i) -> uint32_t {
        return i < nb ? b.d_ban_ids[ban0 + i] : i < nb + nbi ? b.d_bias_ids[bi0 + i - nb] : b.d_cnt_ids[c0 + i - nb - nbi];
    };
    auto val_of = [&](uint32_t i) -> uint32_t {
        return i < nb ? 0u : i < nb + nbi ? zs_f2u(b.d_bias_vals[bi0 + i - nb]) : b.d_cnt_vals[c0 + i - nb - nbi];
    };
    auto x_of = [&](uint32_t id) -> float {
        const float x = b.d_logits[(size_t)r * b.ld + id];
        return masked && !zs_allowed_bit(b, r, id) ? -INFINITY : x;
    };
    uint32_t eid[RW_PE], ev[RW_PE];
    float ex[RW_PE];
#pragma unroll
    for (int u = 0; u < RW_PE; u++) {
        const uint32_t i = t + (uint32_t)u * RW_NT;
        eid[u] = i < ne ? id_of(i) : 0xffffffffu;
        ev[u] = i < ne ? val_of(i) : 0u;
    }
    for (uint32_t i = t; i < words; i += RW_NT) rw_pbits[i] = 0u;
#pragma unroll
    for (int u = 0; u < RW_PE; u++) ex[u] = eid[u] < V ? x_of(eid[u]) : 0.0f;
    // calls f(i, id, value, x) for this thread's entries of [i0, i1) with an id
    // in the row
    auto each = [&](uint32_t i0, uint32_t i1, auto&& f) {
#pragma unroll
        for (int u = 0; u < RW_PE; u++) {
            const uint32_t i = t + (uint32_t)u * RW_NT;
            if (i >= i0 && i < i1 && eid[u] < V) f(i, eid[u], ev[u], [&] { return ex[u]; });
        }
        for (uint32_t i = t + RW_PE * RW_NT; i < i1; i += RW_NT) {
            if (i < i0) continue;
            const uint32_t id = id_of(i);
            if (id < V) f(i, id, val_of(i), [&] { return x_of(id); });
        }
    };
    // entry k: in LDS (ids and flags in sh.pid, y in sh.py) for the list's
    // head, in row scratch past it; the head is copied out at the end
    auto FL = [&](uint32_t k) -> uint32_t { return k < ZS_PATCH_LDS ? sh.pid[k] >> RW_PF_SHIFT : out_fl[k]; };
    auto SET_FL = [&](uint32_t k, uint32_t f) {
        if (k < ZS_PATCH_LDS) sh.pid[k] = (sh.pid[k] & ((1u << RW_PF_SHIFT) - 1u)) | (f << RW_PF_SHIFT);
        else out_fl[k] = f;
    };
    auto Y = [&](uint32_t k) -> float { return k < ZS_PATCH_LDS ? sh.py[k] : out_y[k]; };
    auto SET_Y = [&](uint32_t k, float y) {
        if (k < ZS_PATCH_LDS) sh.py[k] = y;
        else out_y[k] = y;
    };
    rw_bar();
    // the patched ids
    each(0, ne, [&](uint32_t, uint32_t id, uint32_t, auto&&) { atomicOr(&rw_pbits[id >> 5], 1u << (id & 31)); });
    rw_bar();
    // per-word prefix counts of the bitmap: each wave its own stretch of
    // words, 64 at a time
    uint32_t np;
    {
        const uint32_t lane = (uint32_t)zs_lane(), wid = (uint32_t)zs_wid();
        const uint32_t per = ((words + RW_NT - 1) / RW_NT) * 64u, w0 = wid * per, w1 = min(w0 + per, words);
        uint32_t c = 0;
        for (uint32_t w = w0 + lane; w < w1; w += 64) c += __popc(rw_pbits[w]);
        c = rw_wave_sum(c);
        if (lane == 0) sh.ru[2][wid] = c;
        rw_bar();
        uint32_t run = 0;
        np = 0;
#pragma unroll
        for (int w = 0; w < RW_NW; w++) {
            const uint32_t k = sh.ru[2][w];
            run += (uint32_t)w < wid ? k : 0u;
            np += k;
        }
        for (uint32_t wb = w0; wb < w1; wb += 64) {
            const uint32_t w = wb + lane;
            const uint32_t k = w < w1 ? __popc(rw_pbits[w]) : 0u;
            const uint32_t inc = rw_wave_scan(k);
            if (w < w1) rw_pbits[words + w] = run + inc - k;
            run += (uint32_t)__builtin_amdgcn_readlane((int)inc, 63);
        }
    }
    np = rw_uni(np);
    rw_bar();
    // the list in id order: every patched id with its masked logit
    each(0, ne, [&](uint32_t, uint32_t id, uint32_t, auto&& x) {
        const uint32_t k = rw_rank(id, words);
        if (k < ZS_PATCH_LDS) {
            sh.pid[k] = id;
            sh.py[k] = x();
        } else {
            out_id[k] = id;
            out_fl[k] = 0u;
            out_y[k] = x();
        }
    });
    __syncthreads();
    // bans (a banned x~ and y are -inf)
    if (nb) {
        each(0, nb, [&](uint32_t, uint32_t id, uint32_t, auto&&) {
            const uint32_t k = rw_rank(id, words);
            SET_FL(k, ZS_PF_BAN);
            SET_Y(k, -INFINITY);
        });
        __syncthreads();
    }
    // logit_bias (decode_ctrl.rs:108-112): an id met once takes its bias in
    // parallel; the entries of an id met more than once are added by one
    // thread in list order. By windows of the ids (one window up to about
    // 180000 ids): word w of the row is word w - b0 of a window.
    for (uint32_t b0 = 0; nbi && b0 < words; b0 += bw) {
        for (uint32_t i = t; i < 2 * bw; i += RW_NT) seen[i] = 0u;   // (dup follows seen)
        rw_bar();
        each(nb, nb + nbi, [&](uint32_t, uint32_t id, uint32_t, auto&&) {
            const uint32_t w = (id >> 5) - b0, bit = 1u << (id & 31);
            if (w < bw && (atomicOr(&seen[w], bit) & bit)) atomicOr(&dup[w], bit);
        });
        rw_bar();
        each(nb, nb + nbi, [&](uint32_t, uint32_t id, uint32_t v, auto&&) {
            const uint32_t w = (id >> 5) - b0;
            if (w >= bw || ((dup[w] >> (id & 31)) & 1u)) return;
            const uint32_t k = rw_rank(id, words);
            SET_Y(k, Y(k) + zs_u2f(v));
            SET_FL(k, FL(k) | ZS_PF_Y);
        });
        if (t == 0) {
            for (uint32_t i = 0; i < nbi; i++) {
                const uint32_t id = b.d_bias_ids[bi0 + i], w = (id >> 5) - b0;
                if (id >= V || w >= bw || !((dup[w] >> (id & 31)) & 1u)) continue;
                const uint32_t k = rw_rank(id, words);
                SET_Y(k, Y(k) + b.d_bias_vals[bi0 + i]);
                SET_FL(k, FL(k) | ZS_PF_Y);
            }
        }
        __syncthreads();
    }
    // penalty (decode_ctrl.rs:113-125): repeat, then frequency * count + presence
    // (the count map holds each id once)
    each(nb + nbi, ne, [&](uint32_t, uint32_t id, uint32_t cnt, auto&&) {
        const uint32_t k = rw_rank(id, words);
        float y = Y(k);
        if (P.repeat != 1.0f) {
            if (y > 0.0f) y = y / P.repeat;
            else y = y * P.repeat;
        }
        float pen_v = __fmul_rn(P.frequency, (float)cnt);
        pen_v = __fadd_rn(pen_v, P.presence);
        y = __fsub_rn(y, pen_v);
        SET_Y(k, y);
        SET_FL(k, FL(k) | ZS_PF_Y);
    });
    __syncthreads();
    // the list's head out to row scratch (the later kernels read it there)
    for (uint32_t k = t; k < min(np, (uint32_t)ZS_PATCH_LDS); k += RW_NT) {
        out_id[k] = sh.pid[k] & ((1u << RW_PF_SHIFT) - 1u);
        out_fl[k] = sh.pid[k] >> RW_PF_SHIFT;
        out_y[k] = sh.py[k];
    }
    if (t == 0) a.p_cnt[r] = np;
    // first patch of every 1024-id sub-chunk (read by the sum, big-row and
    // output kernels): the bitmap's prefix count at the sub-chunk start
    for (uint32_t j = t; j <= nsub; j += RW_NT) psub[j] = j * (ZS_SUB / 32) < words ? rw_pbits[words + j * (ZS_SUB / 32)] : np;
    return (int)np;
}

// ---------------------------------------------------------------------------
// Element access: x~ (observers: mask and bans) and z (sampler: patched y,
// divided by T) of the 4 ids g*RW_G + 4t .. +3.
// ---------------------------------------------------------------------------
struct rw_row {
    const uint32_t* gfl;            // the patch list in row scratch (entries past its LDS head)
    const float* gy;
    const float* row;
    const uint32_t* allow;
    const uint32_t* allow_or_row;   // allow bits, or any readable words when unmasked
    uint32_t V, np, words;
    uint32_t ldm4, wmax;            // last float4 of the row, last readable word
    uint32_t amask;                 // 15 for an unmasked row, else 0
    uint32_t tiles;                 // tiles of the row
};
struct rw_raw {
    float4 v;
    uint32_t w;   // the allow word holding the 4 ids
    uint32_t pw;  // the patch bitmap word holding them (rows with patches)
};
// Loads of tile g for this thread, as global-memory loads (a generic pointer
// would be loaded with flat instructions, whose completion every LDS wait
// also waits for). Unconditional, from addresses clamped into the row (rows
// are ld >= V floats, ld a multiple of 4) and into the allow bitset, so that
// nothing waits for them before their data is used.
__device__ __forceinline__ rw_raw rw_fetch(const rw_row& R, uint32_t g) {
    const uint32_t idx0 = min(g * RW_G + 4 * threadIdx.x, R.ldm4);
    rw_raw o;
    typedef float rw_f4 __attribute__((ext_vector_type(4)));
    const rw_f4 v = zs_gload(reinterpret_cast<const rw_f4*>(R.row + idx0));
    o.v = make_float4(v.x, v.y, v.z, v.w);
    o.w = zs_gload(R.allow_or_row + min(idx0 >> 5, R.wmax));
    // read with the loads, long before its use
    o.pw = R.np ? rw_pbits[min((g * RW_G + 4 * threadIdx.x) >> 5, R.words - 1)] : 0u;
    return o;
}
// The patched ids among the 4 ids from idx0 (bits of pb): bans set x~ and
// y to -inf, biased or counted ids take their y from the patch list. Their
// rank in the sorted list is the number of bitmap bits before them (per-word
// prefix counts follow the bitmap). GP: the list is longer than its LDS head,
// and ranks past it read the row's copy in global memory (a load that the
// streaming loops must not contain otherwise: the compiler then waits for
// every load in flight after each tile).
template <bool GP>
__device__ __forceinline__ void rw_patch4(const rw_row& R, uint32_t idx0, uint32_t pb, uint32_t wd, float (&x)[4],
                                          float (&y)[4], const rw_shared& sh) {
    uint32_t rank = rw_pbits[R.words + (idx0 >> 5)] + __popc(wd & ((1u << (idx0 & 31)) - 1u));
#pragma unroll
    for (int q = 0; q < 4; q++) {
        if (!((pb >> q) & 1u)) continue;
        uint32_t fl;
        float py;
        if (!GP || rank < ZS_PATCH_LDS) { fl = sh.pid[rank] >> RW_PF_SHIFT; py = sh.py[rank]; }
        else { fl = R.gfl[rank]; py = R.gy[rank]; }
        if (fl & ZS_PF_BAN) { x[q] = -INFINITY; y[q] = -INFINITY; }
        if (fl & ZS_PF_Y) y[q] = py;
        rank++;
    }
}
// x~ (observers: mask and bans) and y (sampler: patched, before the
// temperature) of the 4 ids g*RW_G + 4t .. +3; ids >= V read -inf. Branch
// free but for two uniform tests (the row's last tile, patches in the row)
// and the rare threads holding a patched id.
template <bool GP>
__device__ __forceinline__ void rw_elems(const rw_row& R, uint32_t g, const rw_raw& raw, float (&x)[4], float (&y)[4],
                                         const rw_shared& sh) {
    const uint32_t idx0 = g * RW_G + 4 * threadIdx.x;
    const uint32_t aw = (raw.w >> (idx0 & 31)) | R.amask;   // amask: 15 when unmasked
    x[0] = (aw & 1u) ? raw.v.x : -INFINITY;
    x[1] = (aw & 2u) ? raw.v.y : -INFINITY;
    x[2] = (aw & 4u) ? raw.v.z : -INFINITY;
    x[3] = (aw & 8u) ? raw.v.w : -INFINITY;
    const bool last = g >= R.tiles - 1u;   // uniform
    if (last) {
#pragma unroll
        for (int q = 0; q < 4; q++) x[q] = idx0 + q < R.V ? x[q] : -INFINITY;
    }
#pragma unroll
    for (int q = 0; q < 4; q++) y[q] = x[q];
    if (R.np) {
        const uint32_t wd = raw.pw;
        uint32_t pb = (wd >> (idx0 & 31)) & 15u;
        if (last) pb = idx0 < R.V ? pb : 0u;
        if (pb) rw_patch4<GP>(R, idx0, pb, wd, x, y, sh);
    }
}

// Calls f(g, u, x, y) for the tiles from g_begin on in order, in
// groups of four (u = 0..3, a constant in each unrolled copy: per-tile state
// of a group can live in registers indexed by u), with four tiles of loads in
// flight: unrolled by four so that each load stays in its own registers until
// used (copying a register whose load is outstanding waits for every load). f
// returns true (uniformly) to stop; rw_stream then returns that tile's index,
// else R.tiles. The last group is padded with tiles past the row (ids >= R.V,
// read as -inf), which f must treat as neutral. f must not call functions: a call inside the
// loop saves the registers of the loads in flight, which waits for them.
template <bool GP, class F>
__device__ __forceinline__ uint32_t rw_stream(const rw_row& R, const rw_shared& sh, uint32_t g_begin, const F& f) {
    const uint32_t ng = R.tiles;
    rw_raw raw[4];
#pragma unroll
    for (int u = 0; u < 4; u++) {
        raw[u] = rw_fetch(R, min(g_begin + (uint32_t)u, ng - 1));
        // issued in slot order, as in the loop: the wait before a slot's use
        // then covers only that slot's loads
        __asm__ volatile("" ::: "memory");
    }
    for (uint32_t g0 = g_begin; g0 < ng; g0 += 4) {
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const uint32_t g = g0 + u;
            float x[4], y[4];
            rw_elems<GP>(R, g, raw[u], x, y, sh);
            raw[u] = rw_fetch(R, min(g + 4, ng - 1));
            __asm__ volatile("" ::: "memory");   // keep the loads issued here, ahead of their use
            if (rw_uni(f(g, u, x, y) ? 1u : 0u)) return g;
        }
    }
    return ng;
}

// The elements of one tile (the tile a stream stopped at).
__device__ __forceinline__ void rw_tile(const rw_row& R, const rw_shared& sh, uint32_t g, float (&x)[4], float (&y)[4]) {
    const rw_raw raw = rw_fetch(R, g);
    rw_elems<true>(R, g, raw, x, y, sh);
}

// ---------------------------------------------------------------------------
// Candidate lists (P1). Entries are ((~key) << 32) | id: ascending order is
// key descending, id ascending (Rust's stable descending sort on total_cmp).
// A list admits the elements whose key exceeds its threshold (the key of its
// K-th entry once known); when it holds more than RW_KEEP entries it is
// sorted and cut to its first K, raising the threshold. Elements equal to the
// threshold that arrive later have larger ids than the K entries at or above
// it, so they can never enter the first K.
// ---------------------------------------------------------------------------
struct rw_list {
    unsigned long long* buf;
    uint32_t* cnt;      // [3] per-tile reservation counters (rotating)
    long long* thr;     // admission threshold: keys > thr enter
};

// Selection on a list (list 0: observers, 1: sampler): of its first n
// entries, those of ids < idlim are the list's members; the K1 smallest
// members (all of them when fewer) are brought to the front of the buffer in
// ascending order. Returns the number of members. Called by every thread.
//
// An MSB radix selection on the 64-bit entries, 8-bit digits: the digits
// above the first bit where the members' keys differ are skipped; each pass
// histograms one digit of the members that share the bits above it with the
// K1-th smallest, and one wave picks the digit where the count reaches K1. It
// stops once the members up to and including the chosen digit number at most the cap (always by the last digit: entries are distinct;
// K1 <= RW_SEL_MAX); those are gathered to the front and sorted, by one wave
// up to RW_SEL_CAP, else by the workgroup.
#define RW_SEL_CAP 256
#define RW_SEL_MAX 512
#define RW_SEL_E (RW_BUF / RW_NT)   // list entries per thread
static_assert(RW_BUF % RW_NT == 0, "the list is spread evenly over the threads");

__device__ __noinline__ uint32_t rw_select(int which, uint32_t n, uint32_t K1, uint32_t idlim) {
    rw_shared& sh = rw_sh;
    unsigned long long* buf = which ? sh.u.b.s : sh.u.b.o;
    const uint32_t t = threadIdx.x, lane = (uint32_t)zs_lane(), wid = (uint32_t)zs_wid();
    const unsigned long long NONE = ~0ull;   // no member: ids are below 2^32 - 1
    unsigned long long v[RW_SEL_E];
    uint32_t lo = 0xffffffffu, hi = 0;       // keys (high words) of the members
    uint32_t c = 0;
#pragma unroll
    for (int e = 0; e < RW_SEL_E; e++) {
        const uint32_t i = t + (uint32_t)e * RW_NT;
        v[e] = NONE;
        if (i < n) {
            const unsigned long long w = buf[i];
            if ((uint32_t)w < idlim) v[e] = w;
        }
        const bool mem = v[e] != NONE;
        c += (uint32_t)__popcll(__ballot(mem));
        if (mem) {
            lo = min(lo, (uint32_t)(v[e] >> 32));
            hi = max(hi, (uint32_t)(v[e] >> 32));
        }
    }
    lo = zs_wave_reduce(lo, [](uint32_t x, uint32_t y) { return min(x, y); });
    hi = zs_wave_reduce(hi, [](uint32_t x, uint32_t y) { return max(x, y); });
    if (lane == 0) { sh.sel_mm[0][wid] = c; sh.sel_mm[1][wid] = lo; sh.sel_mm[2][wid] = hi; }
    __syncthreads();
    c = 0; lo = 0xffffffffu; hi = 0;
#pragma unroll
    for (int w = 0; w < RW_NW; w++) {
        c += sh.sel_mm[0][w];
        lo = min(lo, sh.sel_mm[1][w]);
        hi = max(hi, sh.sel_mm[2][w]);
    }
    c = rw_uni(c);
    if (c == 0) return 0;   // every thread read buf before the barrier above
    const uint32_t need = min(c, K1);
    const uint32_t cap = K1 <= RW_SEL_CAP ? RW_SEL_CAP : RW_SEL_MAX;
    // the selected members: (v >> shift) <= (pre >> shift)
    int shift = 0;
    unsigned long long pre = NONE - 1ull;   // every member (ids < 2^32 - 1)
    if (c > cap) {
        lo = rw_uni(lo); hi = rw_uni(hi);
        shift = lo != hi ? 32 + ((31 - __clz(lo ^ hi)) & ~7) : 24;
        pre = ((unsigned long long)lo << 32) & ~((2ull << (shift + 7)) - 1ull);   // the bits above the digit
        uint32_t below = 0;   // members with a smaller prefix
        if (t < 256) sh.sel_hist[0][t] = 0;
        for (int pass = 0;; pass ^= 1) {
            // histogram pass-parity buffer; the other one is cleared for the
            // next pass (its last reader finished before this pass's first barrier)
            if (t < 256) sh.sel_hist[pass ^ 1][t] = 0;
            __syncthreads();
            const int up = shift + 8;
#pragma unroll
            for (int e = 0; e < RW_SEL_E; e++) {
                const bool in = v[e] != NONE && (up >= 64 || (v[e] >> up) == (pre >> up));
                const uint32_t dg = (uint32_t)(v[e] >> shift) & 255u;
                if (in) atomicAdd(&sh.sel_hist[pass][dg], 1u);
            }
            __syncthreads();
            if (wid == 0) {
                // the digit where the running count reaches need
                uint32_t h[4], s4 = 0;
#pragma unroll
                for (int q = 0; q < 4; q++) { h[q] = sh.sel_hist[pass][lane * 4 + q]; s4 += h[q]; }
                const uint32_t inc = wave_incl_scan_u(s4);
                const unsigned long long hit = __ballot(below + inc >= need);
                const uint32_t L = (uint32_t)__ffsll((long long)hit) - 1u;   // one exists
                if (lane == L) {
                    uint32_t run = below + inc - s4;
#pragma unroll
                    for (int q = 0; q < 4; q++) {
                        if (run + h[q] >= need) {
                            sh.sel_mm[0][0] = lane * 4 + q;
                            sh.sel_mm[1][0] = run;
                            sh.sel_mm[2][0] = h[q];
                            break;
                        }
                        run += h[q];
                    }
                }
            }
            __syncthreads();
            const uint32_t dg = rw_uni(sh.sel_mm[0][0]), cb = rw_uni(sh.sel_mm[2][0]);
            below = rw_uni(sh.sel_mm[1][0]);
            pre |= (unsigned long long)dg << shift;
            if (below + cb <= cap || shift == 0) break;
            shift -= 8;
        }
    }
    // gather the selected members to the front (every read of buf is done)
    if (t == 0) sh.sel_n = 0;
    __syncthreads();
#pragma unroll
    for (int e = 0; e < RW_SEL_E; e++) {
        if (v[e] == NONE || (v[e] >> shift) > (pre >> shift)) continue;
        buf[atomicAdd(&sh.sel_n, 1u)] = v[e];
    }
    __syncthreads();
    const uint32_t m = rw_uni(sh.sel_n);
    if (m <= RW_SEL_CAP) {
        if (wid == 0) rw_wave_sort(buf, m);
        __syncthreads();
    } else {
        static_assert(RW_SEL_MAX == RW_NT, "one entry per thread");
        if (t >= m) buf[t] = NONE;
        __syncthreads();
        block_sort_reg_u64<RW_NT, 1>(buf, RW_SEL_MAX);
    }
    return c;
}

// Cuts a list to its K smallest members (rw_select); the K-th key becomes the
// threshold (below K members: every id is admitted). Also records the value
// of the threshold and the largest value cut (into *cutmax).
// Returns the new entry count. Called by every thread.
__device__ uint32_t rw_compact(int which, const rw_list& L, uint32_t n, uint32_t K, uint32_t idlim, float* fthr,
                               float* cutmax) {
    const uint32_t c = rw_select(which, n, K + 1, idlim);
    const uint32_t keep = min(c, K);
    if (threadIdx.x == 0) {
        if (c >= K) {
            const uint32_t kk = ~(uint32_t)(L.buf[K - 1] >> 32);
            *L.thr = (long long)kk;
            *fthr = zs_key_to_float(kk);
            if (c > K) *cutmax = fmaxf(*cutmax, zs_key_to_float(~(uint32_t)(L.buf[K] >> 32)));
        } else {
            *L.thr = -1;
            *fthr = -INFINITY;
        }
    }
    __syncthreads();
    return keep;
}

// Writes the admitted elements (bit q of m = element q: key kk[q], id idx0 +
// q) at base + their reservation on counter ctr; an element whose place is
// past the buffer is not written and its tile is reported in *ovf (the lowest
// such tile is streamed again after a compaction).
__device__ __forceinline__ void rw_admit(const rw_list& L, uint32_t* ctr, uint32_t base, uint32_t m,
                                         const uint32_t (&kk)[4], uint32_t idx0, uint32_t g, uint32_t* ovf) {
    const uint32_t n = __popc(m);
    uint32_t p = base + atomicAdd(ctr, n);
#pragma unroll
    for (int q = 0; q < 4; q++) {
        if (!((m >> q) & 1u)) continue;
        if (p < RW_BUF) L.buf[p] = ((unsigned long long)(~kk[q]) << 32) | (idx0 + q);
        else atomicMin(ovf, g);
        p++;
    }
}

// Row scratch of a masked row's gathered values, 16-byte aligned.
__device__ __forceinline__ float* rw_scratch(const zs_sargs& a, uint32_t r) {
    float* cx = a.gath + (size_t)r * (2 * (size_t)a.max_vocab + 16);
    return cx + ((4u - (uint32_t)((reinterpret_cast<uintptr_t>(cx) >> 2) & 3u)) & 3u);
}

// A masked row's allowed ids in index order, with their x~ (cx) and y (cy)
// written to row scratch: the sums then run over these values only (a
// masked id's term is zero, which leaves a running sum unchanged). cx, cy
// hold round_up(n, 4) values each (the tail padded with -inf); cy = cx +
// round_up(n, 4); the ids follow at cy + round_up(n, 4). Returns n, or 0
// when no id, more than RW_BUF ids or more than a quarter of the row is
// allowed (then the sums run over the whole row with its allow bits: each
// thread's loop over its allowed ids, with a dependent load per id, took 29 us
// on rows with tens of thousands of them, more than P1's whole stream saves).
// Uniform.
__device__ __noinline__ uint32_t rw_gather_allowed(const float* row, const uint32_t* allow, uint32_t V, uint32_t np,
                                                   float* cx, const uint32_t* gfl, const float* gy) {
    rw_shared& sh = rw_sh;
    const uint32_t t = threadIdx.x, words = (V + 31) / 32;
    const uint32_t lane = (uint32_t)zs_lane(), wid = (uint32_t)zs_wid();
    // each wave its own stretch of words, 64 at a time: the counts of the
    // waves, then every allowed id to its place in an LDS list, then their
    // values, all of a thread's loads at once (a loop per thread over its
    // words with a load per id took 10 us on JSON masks)
    const uint32_t per = ((words + RW_NT - 1) / RW_NT) * 64u, w0 = wid * per, w1 = min(w0 + per, words);
    auto word = [&](uint32_t w) {
        uint32_t a = w < w1 ? zs_gload(allow + w) : 0u;
        if (w == words - 1 && (V & 31)) a &= (1u << (V & 31)) - 1u;
        return a;
    };
    constexpr uint32_t NWD = 10;   // words a thread keeps in registers
    uint32_t aw[NWD], c = 0;
#pragma unroll
    for (uint32_t i = 0; i < NWD; i++) aw[i] = word(w0 + lane + 64u * i);
#pragma unroll
    for (uint32_t i = 0; i < NWD; i++) c += __popc(aw[i]);
    for (uint32_t wb = w0 + 64u * NWD; wb < w1; wb += 64) c += __popc(word(wb + lane));
    c = rw_wave_sum(c);
    if (lane == 0) sh.ru[4][wid] = c;
    rw_bar();
    uint32_t n = 0, pos = 0;
#pragma unroll
    for (int w = 0; w < RW_NW; w++) {
        const uint32_t k = sh.ru[4][w];
        pos += (uint32_t)w < wid ? k : 0u;
        n += k;
    }
    n = rw_uni(n);
    rw_bar();
    if (n == 0 || n > RW_BUF || n > V / 4 || V < 16) return 0;   // V >= 16: 3 round_up(n, 4) + 3 values fit 2 V
    const uint32_t n4 = (n + 3) & ~3u;
    float* cy = cx + n4;
    uint32_t* lid = reinterpret_cast<uint32_t*>(sh.u.b.o);   // RW_BUF ids (the list is built after)
    auto place = [&](uint32_t a, uint32_t wb) {
        const uint32_t k = __popc(a), inc = rw_wave_scan(k);
        uint32_t p = pos + inc - k;
        while (a) {
            lid[p++] = (wb + lane) * 32 + (uint32_t)__builtin_ctz(a);
            a &= a - 1u;
        }
        pos += (uint32_t)__builtin_amdgcn_readlane((int)inc, 63);
    };
    for (uint32_t i = 0; i < NWD; i++) {
        if (w0 + 64u * i >= w1) break;   // (uniform)
        uint32_t a = 0;
#pragma unroll
        for (uint32_t j = 0; j < NWD; j++) a = j == i ? aw[j] : a;
        place(a, w0 + 64u * i);
    }
    for (uint32_t wb = w0 + 64u * NWD; wb < w1; wb += 64) place(word(wb + lane), wb);
    rw_bar();
    constexpr uint32_t NE = RW_BUF / RW_NT;
    uint32_t id[NE];
    float xv[NE];
#pragma unroll
    for (uint32_t e = 0; e < NE; e++) {
        id[e] = lid[min(t + e * RW_NT, n - 1u)];
        xv[e] = zs_gload(row + id[e]);
    }
#pragma unroll
    for (uint32_t e = 0; e < NE; e++) {
        const uint32_t i = t + e * RW_NT;
        if (i >= n) continue;
        float x = xv[e], y = x;
        if (np) {
            const uint32_t wd = rw_pbits[id[e] >> 5];
            if ((wd >> (id[e] & 31)) & 1u) {
                const uint32_t rank = rw_pbits[words + (id[e] >> 5)] + __popc(wd & ((1u << (id[e] & 31)) - 1u));
                const uint32_t fl = rank < ZS_PATCH_LDS ? sh.pid[rank] >> RW_PF_SHIFT : gfl[rank];
                if (fl & ZS_PF_BAN) { x = -INFINITY; y = -INFINITY; }
                if (fl & ZS_PF_Y) y = rank < ZS_PATCH_LDS ? sh.py[rank] : gy[rank];
            }
        }
        cx[i] = x;
        cy[i] = y;
        reinterpret_cast<uint32_t*>(cy + n4)[i] = id[e];
    }
    if (t < n4 - n) { cx[n + t] = -INFINITY; cy[n + t] = -INFINITY; }
    __syncthreads();
    return n;
}

// Exact sampling of 65 to ZS_SMALL_CAP survivors by the whole workgroup, one
// survivor per thread: the steps of small_path_wave with the two sorts spread
// over the waves (the sequential sums stay with wave 0, over LDS copies).
// One wave with 8 survivors per lane spent 6.4 us on each sort and 35 us in
// all on 512 survivors, this 18 us. Called by every thread (token to sh.tok).
__device__ __noinline__ void rw_small_wg(uint64_t seed, uint64_t counter, uint32_t V, float top_p, float min_p, uint32_t n,
                                         float m) {
    rw_shared& sh = rw_sh;
    const uint32_t t = threadIdx.x;
    unsigned long long* kb = sh.u.b.s;   // (the lists are no longer needed)
    const bool live = t < n;
    static_assert(ZS_SMALL_CAP == RW_NT, "one survivor per thread");
    uint32_t np2 = 128;
    while (np2 < n) np2 <<= 1;
    // survivors by index
    if (t < np2) kb[t] = live ? (((unsigned long long)sh.sidx[t] << 32) | zs_f2u(sh.sval[t])) : ~0ull;
    __syncthreads();
    block_sort_reg_u64<RW_NT, 1>(kb, np2);
    const unsigned long long e0 = live ? kb[t] : 0ull;
    const uint32_t id = (uint32_t)(e0 >> 32);
    float p = live ? zs_expf(zs_u2f((uint32_t)e0) - m) : 0.0f;
    // s0 + v of thread 0 + v of thread 1 + ... (sampler.rs:68, 80, 107), or
    // the first thread where the sum reaches thresh (to sh.n_surv)
    auto scan = [&](float v, float s0, float thresh) {
        if (live) sh.sval[t] = v;
        __syncthreads();
        if (t < 64) {
            float s;
            const uint32_t i = serial_scan_f(sh.sval, n, s0, thresh, &s);
            if (t == 0) { sh.fsh = s; sh.n_surv = i; }
        }
        __syncthreads();
    };
    // softmax (sampler.rs:67-69)
    scan(p, -0.0f, NAN);
    p = p / sh.fsh;
    // min-p (sampler.rs:72-88)
    if (min_p > 0.0f) {
        const float pm = block_max_f<RW_NT>(live ? p : 0.0f, sh.rf[0]);
        if (p < min_p * pm) p = 0.0f;
        scan(p, 0.0f, NAN);
        const float kept = sh.fsh;
        if (kept > 0.0f) p = p / kept;
    }
    // top-p (sampler.rs:91-115): cumsum in (p desc, idx asc) order
    if (top_p < 1.0f) {
        uint32_t vstar = 0, istar = 0xffffffffu;
        const bool none = !(top_p > 0.0f);  // cumsum 0 >= top_p: nothing kept
        if (!none) {
            if (t < np2) kb[t] = live ? (((unsigned long long)(~zs_f2u(p)) << 32) | id) : ~0ull;
            __syncthreads();
            block_sort_reg_u64<RW_NT, 1>(kb, np2);
            scan(live ? zs_u2f(~(uint32_t)(kb[t] >> 32)) : 0.0f, 0.0f, top_p);
            const uint32_t i = sh.n_surv;
            if (i < n) {
                vstar = ~(uint32_t)(kb[i] >> 32);
                istar = (uint32_t)kb[i];
            }
        }
        const uint32_t pb = zs_f2u(p);
        const bool keep = live && !none && (pb > vstar || (pb == vstar && id <= istar));
        const float f = keep ? p : 0.0f;
        scan(f, -0.0f, NAN);
        const float sum = sh.fsh;
        if (sum > 0.0f) p = f / sum;
    }
    // draw (sampler.rs:118-127); r == 0 stops at index 0 whatever its p
    const float rr = zs_philox_uniform(seed, counter, 0u);
    scan(p, 0.0f, rr);
    if (live && t == sh.n_surv) sh.tok = id;
    if (t == 0) {
        if (rr <= 0.0f) sh.tok = 0;
        else if (sh.n_surv >= n) sh.tok = V - 1;
    }
}

// Exact sampling of a small survivor set (token to sh.tok): up to 64 by wave
// 0, more by the workgroup. Called by every thread.
__device__ __forceinline__ void rw_small(uint64_t seed, uint64_t counter, uint32_t V, const zs_row_params& P, uint32_t nsv,
                                         float zmax, rw_shared& sh) {
    if (nsv > 64) {
        rw_small_wg(seed, counter, V, P.top_p, P.min_p, nsv, zmax);
    } else if (threadIdx.x < 64) {
        const uint32_t tk = small_path_wave(seed, counter, V, P, nsv, zmax, sh.sval, sh.sidx);
        if (threadIdx.x == 0) sh.tok = tk;
    }
}

// The row of the j-th row workgroup: the unmasked rows in index order, then
// the masked ones, when there are more rows than CUs (a CU holds one of these
// workgroups; with a CU for each the order changes nothing). Uniform.
__device__ __forceinline__ uint32_t rw_block_row(const zs_batch& b, uint32_t j, uint32_t ncu) {
    if (!b.d_allow_bits || b.B <= ncu || b.B > 4 * RW_NT) return j;
    rw_shared& sh = rw_sh;
    const uint32_t t = threadIdx.x, lane = (uint32_t)zs_lane(), wid = (uint32_t)zs_wid();
    const uint32_t nchunk = (b.B + RW_NT - 1) / RW_NT;
    uint32_t rank[4], um = 0;      // rank among the rows of its kind; bit c: unmasked
    uint32_t carry = 0;            // unmasked rows in the chunks before
#pragma unroll
    for (uint32_t c = 0; c < 4; c++) {
        rank[c] = 0;
        if (c >= nchunk) continue;
        const uint32_t i = c * RW_NT + t;
        const bool in = i < b.B;
        const bool u = in && !(b.d_params[i].flags & ZS_ROW_MASKED);
        const unsigned long long m = __ballot(u);
        if (lane == 0) sh.sel_mm[0][wid] = (uint32_t)__popcll(m);
        __syncthreads();
        uint32_t before = carry, tot = 0;
#pragma unroll
        for (int w = 0; w < RW_NW; w++) {
            const uint32_t k = sh.sel_mm[0][w];
            before += (uint32_t)w < wid ? k : 0u;
            tot += k;
        }
        __syncthreads();
        before += (uint32_t)__popcll(m & ((1ull << lane) - 1ull));
        rank[c] = u ? before : i - before;   // masked: rows before it minus unmasked before it
        um |= u ? (1u << c) : 0u;
        carry += tot;
    }
    const uint32_t nu = carry;
    if (t == 0) sh.sel_n = j;   // fallback (not reached: every j < B has a row)
    __syncthreads();
#pragma unroll
    for (uint32_t c = 0; c < 4; c++) {
        const uint32_t i = c * RW_NT + t;
        if (c >= nchunk || i >= b.B) continue;
        const uint32_t pos = ((um >> c) & 1u) ? rank[c] : nu + rank[c];
        if (pos == j) sh.sel_n = i;
    }
    __syncthreads();
    const uint32_t r = rw_uni(sh.sel_n);
    __syncthreads();
    return r;
}


// ---------------------------------------------------------------------------
// P1 from group maxima. zs_k_scan (below) reads the row's logits once over the
// whole GPU and leaves the key of the largest x~ of every group of 2^gshift
// consecutive ids (mask applied, bans and biases not). Here the groups holding
// a patched id are read again and the maxima of x~ and y corrected; then
//   - with t0 a key that at least K groups reach, the first K entries of the
//     row by (value desc, id asc) all have keys >= t0, and they lie in the
//     groups whose maximum reaches t0: a few more than K of them;
//   - only the ids of those groups are read again and listed.
// A chain of dependent loads and LDS steps bounds it, not V. The streaming
// loop with its admissions spent 50 us on half a row of 128256 ids; measured,
// scan + row kernel against the streaming row kernel (us):
//   1 x 32000 3 + 19 / 43, 64 x 128256 8 + 30 / 92, 256 x 151936 (half the rows
//   masked) 20 + 46 / 139, 128 x 151936 masked 11 + 46 / 87.
// Longest are the rows of a wide top-k (8 x 100003; k = 40 20 us): k = 500 64,
// its survivors sampled here, k = 2000 57 (two radix selections, of up to 4096
// keys).
// Returns false (uniformly) for rows whose lists would overflow: they take
// the streaming loop of zs_k_row.
// ---------------------------------------------------------------------------
#define RW_WIDE (2 * RW_BUF)   // keys in the sampler list's place
#define RW_GOBS (RW_BUF / 2)   // observers listed at most; the listed groups (u16) follow them in LDS
#define RW_GL (RW_BUF * 2)     // listed groups at most
#define RW_GF 14u              // a listed group: group | list flags << RW_GF
#define RW_GTIES 1024          // groups listed beyond k at most without a cut of the ties among them
#define RW_GPT 10          // groups per thread at most (zs_scan_gshift)
struct rw_gst {
    float omax, ymax, rejf;
    unsigned long long gbest;
    uint32_t n_o, n_s, fl;
    bool s_over;
    bool s_drop;   // the sampler's list did not fit and is not kept (k > ZS_KS)
};
// Whether the groups give a threshold close to the k-th of k > ZS_KS: at most
// three quarters of them reach it, and the ids expected at or above it fit
// their list. With ids in no order a group holds Poisson(m) of them, m = -ln(1
// - k / groups), which is ng * m in all (of 128256 ids, k = 2594 lists 4176 and
// k = 3000 5540); a list that overflows costs a sixth of what one
// that fits saves, so the line lies 2% past its length (1.6% are one standard
// deviation). zs_k_big selects the threshold of the others. 8 rows, us a call,
// by lists / by zs_k_big: k = 2250 of 100003 ids 214 / 573, k = 2550 of 128256
// 222 / 682.
__device__ __forceinline__ bool rw_wide_fits(uint32_t k, uint32_t ng) {
    if (4u * k > 3u * ng) return false;
    const float n = (float)ng;
    return -n * __logf(1.0f - (float)k / n) <= 1.02f * (float)RW_WIDE;
}
__device__ __forceinline__ uint32_t rw_wave_umax(uint32_t v) {
    v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0xB1, 0xf, 0xf, false));    // quad_perm [1,0,3,2]
    v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x4E, 0xf, 0xf, false));    // quad_perm [2,3,0,1]
    v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x141, 0xf, 0xf, false));   // row_half_mirror
    v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x140, 0xf, 0xf, false));   // row_mirror
    v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x142, 0xa, 0xf, false));   // row_bcast:15
    v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x143, 0xc, 0xf, false));   // row_bcast:31
    return (uint32_t)__builtin_amdgcn_readlane((int)v, 63);
}
// Maximum over the 4, 8 or 16 adjacent lanes of a group (qs = 2, 3, 4; uniform).
__device__ __forceinline__ uint32_t rw_lanes_umax(uint32_t v, uint32_t qs) {
    v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0xB1, 0xf, 0xf, false));    // quad_perm [1,0,3,2]
    v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x4E, 0xf, 0xf, false));    // quad_perm [2,3,0,1]
    if (qs >= 3) v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x141, 0xf, 0xf, false));   // row_half_mirror
    if (qs >= 4) v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x140, 0xf, 0xf, false));   // row_mirror
    return v;
}
// Key of a group maximum: -0 and +0 alike, a NaN above everything.
#define RW_KNAN 0xffffffffu
__device__ __forceinline__ uint32_t rw_gkey(float m, bool nan) { return nan ? RW_KNAN : zs_total_key(m + 0.0f); }

// Places behind a counter for n entries of each lane, one atomic per wave (one
// per lane is served lane by lane: a row of equal values spent 350 us on 64 K
// of them). Called by whole waves.
__device__ __forceinline__ uint32_t rw_wave_reserve(uint32_t* ctr, uint32_t n) {
    const uint32_t inc = rw_wave_scan(n);
    uint32_t p = 0;
    if (zs_lane() == 63) p = atomicAdd(ctr, inc);
    return (uint32_t)__builtin_amdgcn_readlane((int)p, 63) + inc - n;
}
// The same behind both halves of a counter, for at most 64 K entries of a wave each.
__device__ __forceinline__ void rw_wave_reserve2(unsigned long long* ctr, uint32_t n0, uint32_t n1, uint32_t& p0, uint32_t& p1) {
    const uint32_t n = n0 | (n1 << 16), inc = rw_wave_scan(n);
    unsigned long long p = 0;
    if (zs_lane() == 63) p = atomicAdd(ctr, (unsigned long long)(inc & 0xffffu) | ((unsigned long long)(inc >> 16) << 32));
    p0 = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)p, 63) + (inc & 0xffffu) - n0;
    p1 = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(p >> 32), 63) + (inc >> 16) - n1;
}

// x~ and y of the 4 ids from idx0 (a multiple of 4; ids >= V read -inf).
__device__ __forceinline__ void rw_load4(const rw_row& R, uint32_t idx0, const float4& v, uint32_t w, float (&x)[4],
                                         float (&y)[4], const rw_shared& sh) {
    const uint32_t aw = (w >> (idx0 & 31)) | R.amask;
    x[0] = (aw & 1u) ? v.x : -INFINITY;
    x[1] = (aw & 2u) ? v.y : -INFINITY;
    x[2] = (aw & 4u) ? v.z : -INFINITY;
    x[3] = (aw & 8u) ? v.w : -INFINITY;
#pragma unroll
    for (int q = 0; q < 4; q++) {
        if (idx0 + q >= R.V) x[q] = -INFINITY;
        y[q] = x[q];
    }
    if (R.np) {
        const uint32_t wd = rw_pbits[min(idx0 >> 5, R.words - 1)];
        const uint32_t pb = idx0 < R.V ? (wd >> (idx0 & 31)) & 15u : 0u;
        if (pb) rw_patch4<false>(R, idx0, pb, wd, x, y, sh);
    }
}
__device__ __forceinline__ float4 rw_fetch4(const rw_row& R, uint32_t idx0, uint32_t& w) {
    typedef float rw_f4 __attribute__((ext_vector_type(4)));
    const uint32_t ia = min(idx0, R.ldm4);
    const rw_f4 v = zs_gload(reinterpret_cast<const rw_f4*>(R.row + ia));
    w = zs_gload(R.allow_or_row + min(ia >> 5, R.wmax));
    return make_float4(v.x, v.y, v.z, v.w);
}

// The K-th largest of n >= K keys in LDS (radix selection, 8-bit digits): the
// words from offset `off` of the dynamic LDS (the group maxima), or
// (off = ~0) of the sampler list's place. Called by every thread; uniform.
__device__ __noinline__ uint32_t rw_kth_key(uint32_t off, uint32_t n, uint32_t K) {
    rw_shared& sh = rw_sh;
    const bool list = off == 0xffffffffu;
    const uint32_t t = threadIdx.x, lane = (uint32_t)zs_lane(), wid = (uint32_t)zs_wid();
    uint32_t pre = 0, need = K;
    for (int shift = 24; shift >= 0; shift -= 8) {
        if (t < 256) sh.sel_hist[0][t] = 0;
        __syncthreads();
        for (uint32_t i = t; i < n; i += RW_NT) {
            const uint32_t k = list ? reinterpret_cast<uint32_t*>(sh.u.b.s)[i] : rw_pbits[off + i];
            if (shift == 24 || (k >> (shift + 8)) == (pre >> (shift + 8))) atomicAdd(&sh.sel_hist[0][(k >> shift) & 255u], 1u);
        }
        __syncthreads();
        if (wid == 0) {
            // digits in descending order: lane l holds 255 - 4l .. 252 - 4l
            uint32_t h[4], s4 = 0;
#pragma unroll
            for (int q = 0; q < 4; q++) { h[q] = sh.sel_hist[0][255u - 4u * lane - (uint32_t)q]; s4 += h[q]; }
            const uint32_t inc = wave_incl_scan_u(s4);
            const unsigned long long hit = __ballot(inc >= need);
            const uint32_t L = (uint32_t)__ffsll((long long)hit) - 1u;   // one exists: n >= K
            if (lane == L) {
                uint32_t run = inc - s4;
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    if (run + h[q] >= need) {
                        sh.sel_st[0] = 255u - 4u * lane - (uint32_t)q;
                        sh.sel_st[1] = need - run;
                        break;
                    }
                    run += h[q];
                }
            }
        }
        __syncthreads();
        pre |= rw_uni(sh.sel_st[0]) << shift;
        need = rw_uni(sh.sel_st[1]);
        __syncthreads();
    }
    return pre;
}

// Of the n group maxima at offset `off` of the dynamic LDS, this thread's
// (t, t + RW_NT, ...: bit e) that are not `key` or among the first K equal to
// it. Called by every thread.
__device__ __noinline__ uint32_t rw_first_ties(uint32_t off, uint32_t n, uint32_t key, uint32_t K) {
    rw_shared& sh = rw_sh;
    const uint32_t t = threadIdx.x, wid = (uint32_t)zs_wid();
    auto tied = [&](uint32_t e) {
        const uint32_t i = t + e * RW_NT;
        return __ballot(i < n && rw_pbits[off + min(i, n - 1u)] == key);
    };
    for (uint32_t e = 0; e < RW_GPT; e++) {
        const uint32_t c = (uint32_t)__popcll(tied(e));
        if (zs_lane() == 0) sh.sel_hist[0][e * RW_NW + wid] = c;
    }
    rw_bar();
    uint32_t run = 0, keep = ~0u;
    for (uint32_t e = 0; e < RW_GPT; e++) {
        const unsigned long long m = tied(e);
        uint32_t before = run;
        for (uint32_t w = 0; w < RW_NW; w++) {
            const uint32_t c = sh.sel_hist[0][e * RW_NW + w];
            before += w < wid ? c : 0u;
            run += c;
        }
        before = __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, before));
        if ((m >> zs_lane() & 1ull) && before >= K) keep &= ~(1u << e);
    }
    rw_bar();
    return keep;
}

__device__ __forceinline__ bool rw_groups(const zs_sargs& a, uint32_t r, const rw_row& R, bool greedy, bool tinf,
                                          uint32_t smode, uint32_t Ks, uint32_t Ko, rw_gst& G) {
    rw_shared& sh = rw_sh;
    const uint32_t t = threadIdx.x, wid = (uint32_t)zs_wid();
    const uint32_t gs = a.gshift, ng = (R.V + (1u << gs) - 1u) >> gs;
    uint32_t* gx = rw_pbits + 2 * R.words;   // (the bias bitmaps of rw_patches are no longer needed)
    uint32_t* gy = gx + ng;
    const uint32_t* gm = a.gmax + (size_t)r * a.gstride;
    const uint32_t kinf = zs_total_key(-INFINITY);
#ifdef ZS_WALK_DEBUG
    unsigned long long rw_t0 = wall_clock64();
#endif
    {
        uint32_t k[RW_GPT];
#pragma unroll
        for (int e = 0; e < RW_GPT; e++) k[e] = zs_gload(gm + min(t + (uint32_t)e * RW_NT, ng - 1u));
#pragma unroll
        for (int e = 0; e < RW_GPT; e++) {
            const uint32_t i = t + (uint32_t)e * RW_NT;
            if (i < ng) { gx[i] = k[e]; gy[i] = k[e]; }
        }
    }
    if (t == 0) { sh.n_gl = 0; sh.n_os = 0; }
    __syncthreads();
    // groups with patched ids are read again: the first patch of a group lists
    // it, then one lane per 4 ids (the lanes of a group adjacent)
    uint16_t* gl = reinterpret_cast<uint16_t*>(sh.u.b.o + RW_GOBS);
    static_assert(RW_GL * sizeof(uint16_t) <= (RW_BUF - RW_GOBS) * sizeof(unsigned long long) &&
                  RW_GPT * RW_NT <= 1u << RW_GF && ZS_PATCH_LDS <= RW_GL, "the listed groups fit");
    const uint32_t qs = gs - 2u, qm = (1u << qs) - 1u;   // log2 of the lanes per group
    if (R.np) {
        for (uint32_t p = t; p < R.np; p += RW_NT) {
            const uint32_t gp = (sh.pid[p] & ((1u << RW_PF_SHIFT) - 1u)) >> gs;
            const uint32_t gq = p ? (sh.pid[p - 1] & ((1u << RW_PF_SHIFT) - 1u)) >> gs : 0xffffffffu;
            if (gp != gq) gl[atomicAdd(&sh.n_gl, 1u)] = (uint16_t)gp;
        }
        rw_bar();
        const uint32_t nit = rw_uni(sh.n_gl) << qs;
        constexpr int NU = 4;
        for (uint32_t i0 = 0; i0 < nit; i0 += NU * RW_NT) {
            float4 v[NU];
            uint32_t w[NU], idx0[NU];
#pragma unroll
            for (int u = 0; u < NU; u++) {
                const uint32_t i = min(i0 + t + (uint32_t)u * RW_NT, nit - 1u);
                idx0[u] = ((uint32_t)gl[i >> qs] << gs) + 4u * (i & qm);
                v[u] = rw_fetch4(R, idx0[u], w[u]);
            }
#pragma unroll
            for (int u = 0; u < NU; u++) {
                if (i0 + (uint32_t)u * RW_NT >= nit) break;
                float x[4], y[4];
                rw_load4(R, idx0[u], v[u], w[u], x, y, sh);
                uint32_t mx = rw_gkey(fmaxf(fmaxf(x[0], x[1]), fmaxf(x[2], x[3])),
                                      __builtin_isunordered(x[0], x[1]) || __builtin_isunordered(x[2], x[3]));
                uint32_t my = rw_gkey(fmaxf(fmaxf(y[0], y[1]), fmaxf(y[2], y[3])),
                                      __builtin_isunordered(y[0], y[1]) || __builtin_isunordered(y[2], y[3]));
                mx = rw_lanes_umax(mx, qs);
                my = rw_lanes_umax(my, qs);
                // (the clamped lanes past the last item lie in its group: the same maxima)
                if ((t & qm) == 0u && i0 + t + (uint32_t)u * RW_NT < nit) {
                    gx[idx0[u] >> gs] = mx;
                    gy[idx0[u] >> gs] = my;
                }
            }
        }
    }
    rw_bar();
    if (t == 0) sh.n_gl = 0;
    RW_T(6);
    // this thread's groups t, t + RW_NT, ...
    uint32_t kx[RW_GPT], ky[RW_GPT], mo = 0, ms = 0, fin = 0;
    auto load_groups = [&]() {
#pragma unroll
        for (int e = 0; e < RW_GPT; e++) {
            const uint32_t i = t + (uint32_t)e * RW_NT, ic = min(i, ng - 1u);
            kx[e] = gx[ic];
            ky[e] = gy[ic];
            if (i >= ng) kx[e] = ky[e] = 0u;
        }
    };
    load_groups();
#pragma unroll
    for (int e = 0; e < RW_GPT; e++) {
        mo = max(mo, kx[e]);
        ms = max(ms, ky[e]);
        fin += ky[e] > kinf ? 1u : 0u;
    }
    // t0: in every wave the c-th largest thread maximum, c = ceil(K / waves),
    // is reached by c groups of that wave, so the smallest of the waves' is
    // reached by K groups (k past a wave's width: the K-th largest group
    // maximum itself)
    const bool wide = Ks > ZS_KS;   // (a quarter of the threads)
    const uint32_t so = wave_sort_u32(mo), ss = wave_sort_u32(ms);
    const int co = max((int)((Ko + RW_NW - 1) / RW_NW), 1), cs = wide ? 1 : max((int)((Ks + RW_NW - 1) / RW_NW), 1);
    const uint32_t wo = (uint32_t)__builtin_amdgcn_readlane((int)so, 64 - co);
    const uint32_t ws = (uint32_t)__builtin_amdgcn_readlane((int)ss, 64 - cs);
    const uint32_t wf = rw_wave_sum(fin);
    if (zs_lane() == 63) {
        sh.ru[0][wid] = wo; sh.ru[1][wid] = ws; sh.ru[2][wid] = wf;
        sh.ru[3][wid] = so; sh.ru[4][wid] = ss;
    }
    __syncthreads();
    uint32_t to = 0xffffffffu, ts = 0xffffffffu, nfin = 0, kmo = 0, kms = 0;
#pragma unroll
    for (int w = 0; w < RW_NW; w++) {
        to = min(to, sh.ru[0][w]); ts = min(ts, sh.ru[1][w]); nfin += sh.ru[2][w];
        kmo = max(kmo, sh.ru[3][w]); kms = max(kms, sh.ru[4][w]);
    }
    to = rw_uni(to); ts = rw_uni(ts); nfin = rw_uni(nfin); kmo = rw_uni(kmo); kms = rw_uni(kms);
    // (a NaN in x~ or in y: the observers' or the sampler's list is not needed)
    const bool xnan = kmo == RW_KNAN, ynan = kms == RW_KNAN;
    G.fl = (xnan ? ZS_CF_OBS_NAN : 0u) | (ynan ? ZS_CF_Z_NAN : 0u);
    const bool ol = Ko && !xnan;
    // (too many of a wave's groups at -inf, as under a mask: exactly)
    if (ol && to <= kinf) to = rw_kth_key(2 * R.words, ng, Ko);
    if ((smode & 1u) && !ynan) {
        if (wide || ts <= kinf) ts = rw_kth_key(2 * R.words + ng, ng, Ks);
    } else if (smode == 2) {
        // every y above -inf, when few enough groups hold one
        G.s_over = nfin > ZS_SMALL_CAP;
        ts = kinf + 1u;
    }
    const bool sl = !ynan && ((smode & 1u) || (smode == 2 && !G.s_over));   // a sampler list is kept
    // (-inf is no member of either list here: the observers' -inf entries are
    // added below, the sampler's survivors are above -inf)
    to = max(to, kinf + 1u);
    ts = max(ts, kinf + 1u);
    RW_T(15);
    uint32_t* wk = reinterpret_cast<uint32_t*>(sh.u.b.s);
    const uint32_t scap = smode == 3 ? (uint32_t)RW_WIDE : smode == 2 ? (uint32_t)ZS_SMALL_CAP : (uint32_t)RW_BUF;
    constexpr int NU = 4;
    uint32_t rej, n_gl, n_o, n_s, keep = ~0u, pad = 0u;   // keep: bit e, the observers of group e are listed
    for (bool cut = false;; cut = true) {
        // the groups that reach a threshold
        uint32_t fl2 = 0, n = 0;
        rej = 0;
        static_assert(2 * RW_GPT <= 32, "two bits per group of a thread");
#pragma unroll
        for (int e = 0; e < RW_GPT; e++) {
            const uint32_t f = (ol && kx[e] >= to && (keep >> e & 1u) ? 1u : 0u) | (sl && ky[e] >= ts ? 2u : 0u);
            if (!(f & 2u)) rej = max(rej, ky[e]);
            fl2 |= f << (2 * e);
            n += f ? 1u : 0u;
        }
        uint32_t p = rw_wave_reserve(&sh.n_gl, n);
        for (; fl2; p++) {
            const uint32_t e = (uint32_t)__builtin_ctz(fl2) >> 1, f = fl2 >> (2 * e) & 3u;
            fl2 &= ~(3u << (2 * e));
            if (p < RW_GL) gl[p] = (uint16_t)((t + e * RW_NT) | (f << RW_GF));
        }
        __syncthreads();
        n_gl = rw_uni(sh.n_gl);
        const uint32_t nit = cut || n_gl <= RW_GTIES + Ks ? min(n_gl, (uint32_t)RW_GL) << qs : 0u;
        for (uint32_t i0 = 0; i0 < nit; i0 += NU * RW_NT) {
            float4 v[NU];
            uint32_t w[NU], ge[NU];
#pragma unroll
            for (int u = 0; u < NU; u++) {
                const uint32_t i = i0 + t + (uint32_t)u * RW_NT;
                ge[u] = gl[min(i, nit - 1u) >> qs];
                if (i >= nit) ge[u] &= (1u << RW_GF) - 1u;
                v[u] = rw_fetch4(R, ((ge[u] & ((1u << RW_GF) - 1u)) << gs) + 4u * (i & qm), w[u]);
            }
#pragma unroll
            for (int u = 0; u < NU; u++) {
                const uint32_t f = ge[u] >> RW_GF;
                if (!__ballot(f != 0u)) continue;   // (past the last item)
                const uint32_t idx0 = ((ge[u] & ((1u << RW_GF) - 1u)) << gs) + 4u * ((i0 + t + (uint32_t)u * RW_NT) & qm);
                float x[4], y[4];
                rw_load4(R, idx0, v[u], w[u], x, y, sh);
                // (thresholds are keys of group maxima: compared with -0 as +0, the
                // sampler's entries themselves in total order as Rust sorts them)
                uint32_t kxq[4], kyq[4], mo4 = 0, ms4 = 0;
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    kxq[q] = zs_total_key(x[q] + 0.0f);
                    kyq[q] = zs_total_key(y[q] + 0.0f);
                    mo4 |= (f & 1u) && kxq[q] >= to ? 1u << q : 0u;
                    const bool in = (f & 2u) && kyq[q] >= ts;
                    ms4 |= in ? 1u << q : 0u;
                    if (f && !in) rej = max(rej, kyq[q]);
                }
                if (!__ballot((mo4 | ms4) != 0u)) continue;
                uint32_t po, ps;
                rw_wave_reserve2(&sh.n_os, (uint32_t)__popc(mo4), (uint32_t)__popc(ms4), po, ps);
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    if ((mo4 >> q) & 1u) {
                        if (po < RW_GOBS) sh.u.b.o[po] = ((unsigned long long)(~kxq[q]) << 32) | (idx0 + q);
                        po++;
                    }
                    if ((ms4 >> q) & 1u) {
                        if (ps < scap) {
                            if (smode == 3) wk[ps] = kyq[q];
                            else sh.u.b.s[ps] = ((unsigned long long)(~zs_total_key(y[q])) << 32) | (idx0 + q);
                        }
                        ps++;
                    }
                }
            }
        }
        __syncthreads();
        n_o = rw_uni((uint32_t)sh.n_os);
        n_s = rw_uni((uint32_t)(sh.n_os >> 32));
        __syncthreads();   // (the counts are read before they change below)
        const bool many = n_gl > RW_GTIES + Ks || (smode == 1 && Ks <= ZS_KS && n_s > scap);
        if (cut || !(many || n_o > RW_GOBS)) break;
        // Many groups, or many ids, from a threshold on: a row of few distinct
        // values or with a run of equal ones. The thresholds are taken exactly
        // then. Of the observers' groups at theirs only the first Ko are
        // needed (each holds an id at it, and the smallest ids come first);
        // the sampler's list takes the entries above its own and, for the
        // k-th value, Ks places at it (the others count as turned away).
        if (ol) {
            to = max(rw_kth_key(2 * R.words, ng, Ko), kinf + 1u);
            keep = rw_first_ties(2 * R.words, ng, to, Ko);
        }
        if (many && sl && (smode & 1u)) {
            ts = max(rw_kth_key(2 * R.words + ng, ng, Ks), kinf + 1u);
            if (ts > kinf + 1u) pad = ts++;
        }
        __syncthreads();
        if (t == 0) { sh.n_gl = 0; sh.n_os = 0; }
        rw_bar();
        load_groups();   // (again: no registers are held for them meanwhile)
    }
    if (n_gl > RW_GL || n_o > RW_GOBS) return false;
    if ((smode & 1u) && n_s + (pad ? Ks : 0u) > scap) {
        // (the streaming loop would list no k > ZS_KS either)
        if (Ks <= ZS_KS) return false;
        G.s_drop = true;
        n_s = 0;
    } else if (pad) {
        for (uint32_t i = t; i < Ks; i += RW_NT) {
            if (smode == 3) wk[n_s + i] = pad;
            else sh.u.b.s[n_s + i] = ((unsigned long long)(~pad) << 32) | i;
        }
        n_s += Ks;
        rej = max(rej, pad);
    }
    if (ol && n_o < Ko) {
        // fewer than Ko ids above -inf: the smallest ids at -inf follow (at
        // most Ko of the first 64 ids are above it)
        static_assert(2 * ZS_OBS_CAND <= 64, "the first 64 ids hold them");
        if (t < 64) {
            uint32_t w;
            const uint32_t idx0 = t & ~3u;
            const float4 v = rw_fetch4(R, idx0, w);
            float x[4], y[4];
            rw_load4(R, idx0, v, w, x, y, sh);
            const float xi = (t & 3u) == 0 ? x[0] : (t & 3u) == 1 ? x[1] : (t & 3u) == 2 ? x[2] : x[3];
            if (t < R.V && xi == -INFINITY) sh.u.b.o[atomicAdd(reinterpret_cast<uint32_t*>(&sh.n_os), 1u)] = ((unsigned long long)(~kinf) << 32) | t;
        }
        __syncthreads();
        n_o = rw_uni((uint32_t)sh.n_os);
    }
    if (greedy) {
        // the last id whose y equals the maximum: in the last group at it. A
        // NaN restarts the fold (sampler.rs:35-43): then of the ids after the
        // last one, in the rest of its group and in the groups past it
        uint32_t nl = 0;   // the last group with a NaN, plus one
        if (ynan) {
#pragma unroll
            for (int e = 0; e < RW_GPT; e++)
                if (ky[e] == RW_KNAN) nl = t + (uint32_t)e * RW_NT + 1u;
            nl = rw_wave_umax(nl);
            if (zs_lane() == 0) sh.ru[5][wid] = nl;
            __syncthreads();
            nl = 0;
#pragma unroll
            for (int w = 0; w < RW_NW; w++) nl = max(nl, sh.ru[5][w]);
            if (wid == 0) {
                uint32_t w;
                const uint32_t idx0 = ((nl - 1u) << gs) + 4u * (t & qm);
                const float4 v = rw_fetch4(R, idx0, w);
                float x[4], y[4];
                rw_load4(R, idx0, v, w, x, y, sh);
                uint32_t L = 0;   // the last NaN's id, plus one
#pragma unroll
                for (int q = 0; q < 4; q++)
                    if (y[q] != y[q]) L = idx0 + (uint32_t)q + 1u;
                L = rw_wave_umax(L);
                G.gbest = L;
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    if (idx0 + q < L || idx0 + q >= R.V) continue;
                    const unsigned long long c = ((unsigned long long)zs_total_key(y[q] + 0.0f) << 32) | (idx0 + q + 1);
                    G.gbest = c > G.gbest ? c : G.gbest;
                }
            }
        }
        unsigned long long gk = 0;   // the largest maximum of the groups from nl on, and the last group at it, plus one
#pragma unroll
        for (int e = 0; e < RW_GPT; e++) {
            const uint32_t i = t + (uint32_t)e * RW_NT;
            const unsigned long long c = ((unsigned long long)ky[e] << 32) | (i + 1u);
            if (i >= nl && i < ng) gk = c > gk ? c : gk;
        }
        gk = zs_wave_reduce(gk, [](unsigned long long x, unsigned long long y) { return x > y ? x : y; });
        if (zs_lane() == 0) sh.rl[wid] = gk;
        __syncthreads();
        gk = 0;
#pragma unroll
        for (int w = 0; w < RW_NW; w++) gk = sh.rl[w] > gk ? sh.rl[w] : gk;
        if (gk && t <= qm) {
            const uint32_t idx0 = (((uint32_t)gk - 1u) << gs) + 4u * t;
            uint32_t w;
            const float4 v = rw_fetch4(R, idx0, w);
            float x[4], y[4];
            rw_load4(R, idx0, v, w, x, y, sh);
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const unsigned long long c = (gk & 0xffffffff00000000ull) | (idx0 + q + 1);
                if (idx0 + q < R.V && zs_total_key(y[q] + 0.0f) == (uint32_t)(gk >> 32)) G.gbest = c > G.gbest ? c : G.gbest;
            }
        }
    }
    if (tinf) {
        // y / inf is NaN for y = +-inf, which the maxima do not tell: one more
        // read of the row, without lists
        bool bad = false;
        for (uint32_t i0 = 4u * t; i0 < R.V; i0 += NU * 4u * RW_NT) {
            float4 v[NU];
            uint32_t w[NU];
#pragma unroll
            for (int u = 0; u < NU; u++) v[u] = rw_fetch4(R, i0 + (uint32_t)u * 4u * RW_NT, w[u]);
#pragma unroll
            for (int u = 0; u < NU; u++) {
                const uint32_t idx0 = i0 + (uint32_t)u * 4u * RW_NT;
                float x[4], y[4];
                rw_load4(R, idx0, v[u], w[u], x, y, sh);
#pragma unroll
                for (int q = 0; q < 4; q++) bad |= idx0 + q < R.V && (y[q] == INFINITY || y[q] == -INFINITY);
            }
        }
        if (bad) G.fl |= ZS_CF_Z_NAN;
    }
    G.omax = xnan ? -INFINITY : zs_key_to_float(kmo);
    G.ymax = ynan ? -INFINITY : zs_key_to_float(kms);
    G.rejf = rej > kinf ? zs_key_to_float(rej) : -INFINITY;
    G.n_o = n_o;
    G.n_s = n_s;
    if (smode == 2 && n_s > ZS_SMALL_CAP) G.s_over = true;
    __syncthreads();
    return true;
}

// ---------------------------------------------------------------------------
// zs_k_scan: the group maxima of every row, over the whole GPU. One read of
// the logits, 4 16-byte loads in flight per thread; a masked row's loads are
// skipped where 4 ids in a row are disallowed. 32.8 MB (64 x 128256) take 8 us, 4.1
// TB/s, 89 MB of 256 x 151936 with half the rows masked 20 us, 4.7 TB/s with the
// maxima written. (A NaN or few survivors are seen in the maxima: no other statistic
// is needed.)
// ---------------------------------------------------------------------------
#define SC_NT 256
#define SC_IDS (16 * SC_NT)   // ids per workgroup
template <int GS>
__global__ __launch_bounds__(SC_NT) void zs_k_scan(zs_sargs a) {
    const zs_batch& b = a.b;
    const uint32_t r = blockIdx.y, V = b.V, lane = (uint32_t)zs_lane();
    const float* row = b.d_logits + (size_t)r * b.ld;
    const uint32_t* allow = ((b.d_params[r].flags & ZS_ROW_MASKED) && b.d_allow_bits)
                                ? b.d_allow_bits + (size_t)r * b.allow_words : nullptr;
    typedef float sc_f4 __attribute__((ext_vector_type(4)));
    const uint32_t base = blockIdx.x * SC_IDS + 4u * threadIdx.x;
    sc_f4 v[4];
    uint32_t w[4];
    if (allow) {
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const uint32_t id = base + (uint32_t)u * (4u * SC_NT);
            w[u] = id < V ? allow[id >> 5] >> (id & 31u) & 15u : 0u;
        }
    } else {
#pragma unroll
        for (int u = 0; u < 4; u++) w[u] = base + (uint32_t)u * (4u * SC_NT) < V ? 15u : 0u;
    }
#pragma unroll
    for (int u = 0; u < 4; u++) {
        v[u] = sc_f4{-INFINITY, -INFINITY, -INFINITY, -INFINITY};
        if (w[u]) v[u] = *reinterpret_cast<const sc_f4*>(row + base + (uint32_t)u * (4u * SC_NT));
    }
    uint32_t k[4];
#pragma unroll
    for (int u = 0; u < 4; u++) {
        const uint32_t id = base + (uint32_t)u * (4u * SC_NT);
        if (id + 4u > V) w[u] &= id < V ? (1u << (V - id)) - 1u : 0u;
        const float x0 = (w[u] & 1u) ? v[u].x : -INFINITY, x1 = (w[u] & 2u) ? v[u].y : -INFINITY;
        const float x2 = (w[u] & 4u) ? v[u].z : -INFINITY, x3 = (w[u] & 8u) ? v[u].w : -INFINITY;
        const bool nan = __builtin_isunordered(x0, x1) || __builtin_isunordered(x2, x3);
        k[u] = rw_gkey(fmaxf(fmaxf(x0, x1), fmaxf(x2, x3)), nan);
        k[u] = max(k[u], (uint32_t)__builtin_amdgcn_update_dpp(0, (int)k[u], 0xB1, 0xf, 0xf, false));
        k[u] = max(k[u], (uint32_t)__builtin_amdgcn_update_dpp(0, (int)k[u], 0x4E, 0xf, 0xf, false));
        if (GS >= 5) k[u] = max(k[u], (uint32_t)__builtin_amdgcn_update_dpp(0, (int)k[u], 0x141, 0xf, 0xf, false));
        if (GS >= 6) k[u] = max(k[u], (uint32_t)__builtin_amdgcn_update_dpp(0, (int)k[u], 0x140, 0xf, 0xf, false));
    }
    // lane q of a quad stores load q's group (one store for all four)
    constexpr uint32_t LG = 1u << (GS - 2);   // lanes per group
    const uint32_t q = lane & 3u;
    const uint32_t kq = q == 0 ? k[0] : q == 1 ? k[1] : q == 2 ? k[2] : k[3];
    const uint32_t g = (blockIdx.x * SC_IDS + q * (4u * SC_NT) + 4u * threadIdx.x) >> GS;
    if ((lane & (LG - 1u)) < 4u && g < (V + (1u << GS) - 1u) >> GS) a.gmax[(size_t)r * a.gstride + g] = kq;
}

// Group size of the scan: the row kernel holds the maxima of at most RW_GPT
// groups per thread; smaller groups mean fewer ids read twice. 0: rows below
// two of the streaming loop's tiles gain nothing from a second launch, and the
// maxima of rows past about 240000 ids do not fit the LDS beside the bitmap.
uint32_t zs_scan_gshift(uint32_t V) {
    if (V < 2 * RW_G) return 0;
    uint32_t gs = 4;
    while (((V + (1u << gs) - 1u) >> gs) > RW_GPT * RW_NT) gs++;
    if (2u * ((V + 31u) / 32u) + 2u * ((V + (1u << gs) - 1u) >> gs) > RW_DYN_WORDS) return 0;
    return gs;   // at most 6: V <= ZS_MAX_VOCAB
}
static_assert((ZS_MAX_VOCAB >> 6) <= RW_GPT * RW_NT, "groups of 64 ids serve the widest row");

// ---------------------------------------------------------------------------
// zs_k_row
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(RW_NT) void zs_k_row(zs_sargs a) {
    const zs_batch& b = a.b;
    const uint32_t r = rw_block_row(b, blockIdx.x, a.ncu);
    const uint32_t t = threadIdx.x;
    const uint32_t V = b.V;
    rw_shared& sh = rw_sh;
    __shared__ uint32_t cnt_o[3], cnt_s[3];
    __shared__ long long thr_o, thr_s;
    const zs_row_params P = b.d_params[r];
    zs_row_state& st = a.rst[r];
    const float T = P.temperature;
    const bool want_lp = (P.flags & ZS_ROW_LOGPROBS) != 0;
    const bool want_unc = (P.flags & ZS_ROW_UNCERTAINTY) != 0;
    const bool want_obs = want_lp || want_unc;
#ifdef ZS_WALK_DEBUG
    unsigned long long rw_t0 = wall_clock64();
#endif
    const bool greedy = T <= 0.0f;
    const bool tinf = T == INFINITY;   // y / inf is NaN for y = +-inf: checked per element
    const uint32_t* allow = ((P.flags & ZS_ROW_MASKED) && b.d_allow_bits) ? b.d_allow_bits + (size_t)r * b.allow_words
                                                                          : nullptr;
    // ---------------- P0: patches
    const int np = rw_patches(a, r, P, sh);
    RW_T(0);
    rw_row R;
    R.gfl = a.p_flags + (size_t)r * a.pstride;
    R.gy = a.p_y + (size_t)r * a.pstride;
    R.row = b.d_logits + (size_t)r * b.ld;
    R.allow = allow;
    R.V = V;
    R.np = rw_uni((uint32_t)np);
    R.words = (V + 31) / 32;
    R.ldm4 = (uint32_t)min((uint64_t)b.ld - 4, (uint64_t)0xfffffff0u);
    R.allow_or_row = R.allow ? R.allow : reinterpret_cast<const uint32_t*>(R.row);
    R.wmax = R.allow ? R.words - 1 : R.ldm4;
    R.amask = R.allow ? 0u : 15u;
    R.tiles = (V + RW_G - 1) / RW_G;

    // ---------------- P1: statistics and candidate lists
    // The sampler's z = y / T (sampler.rs:47-51) is not formed per element
    // here: division by T > 0 is monotone, so the maximum, the order and the
    // top-k of z follow from those of y (ties created by the rounding are
    // checked when the threshold is set).
    const bool has_topk = P.top_k > 0 && P.top_k < V;
    // sampler list: 1 = top-k by y (k <= ZS_KS), 2 = every y > -inf (the
    // small-survivor check when no top-k applies), 0 = none; from the group
    // maxima also larger k: 1 while the survivors fit the small path, 3 (the
    // keys only, for the threshold) as far as rw_wide_fits
    const bool has_groups = a.gshift && R.np <= ZS_PATCH_LDS;
    const uint32_t kmax1 = has_groups ? (uint32_t)ZS_SMALL_CAP - 1u : (uint32_t)ZS_KS;
    uint32_t smode = greedy ? 0u : (!has_topk ? 2u : P.top_k <= kmax1 ? 1u : has_groups ? 3u : 0u);
    uint32_t Ks = (smode & 1u) ? P.top_k : 0u;
    const uint32_t Ko = want_obs ? (ZS_OBS_CAND < V ? ZS_OBS_CAND : V) : 0u;
    rw_list LO, LS;
    LO.buf = sh.u.b.o; LO.cnt = cnt_o; LO.thr = &thr_o;
    LS.buf = sh.u.b.s; LS.cnt = cnt_s; LS.thr = &thr_s;
    if (t < 3) { cnt_o[t] = 0; cnt_s[t] = 0; }
    if (t == 0) { thr_o = -1; thr_s = -1; }
    float omax = -INFINITY, ymax = -INFINITY;
    uint32_t fl = 0;                // ZS_CF_OBS_NAN, ZS_CF_Z_NAN
    float rejf = -INFINITY;         // largest y turned away from the top-k list
    int last_nan = -1;
    unsigned long long gbest = 0;   // greedy: (key << 32) | (id + 1); ties -> larger id
    uint32_t n_o = 0, n_s = 0;      // entries in the lists (uniform)
    bool s_over = false;            // smode 2: more than ZS_SMALL_CAP values above -inf
    __syncthreads();
    // keys of one element set (observers: -0 and +0 share one key, as equal
    // logprobs rank by id, logprobs.rs:41-51)
    auto keys = [&](const float (&x)[4], const float (&y)[4], uint32_t (&kx)[4], uint32_t (&ky)[4]) {
#pragma unroll
        for (int q = 0; q < 4; q++) {
            kx[q] = zs_total_key(x[q] + 0.0f);
            ky[q] = zs_total_key(y[q]);
        }
    };
    // The lists are synchronised once per group of four tiles: admissions
    // reserve places with a counter slot that rotates over three groups, so a
    // single barrier per group separates its use, its read and its reset.
    uint32_t grp = 0, lastslot = 0;
    bool thr_init = false, p1stop = false;
    if (t < 3) sh.ovf[t] = 0xffffffffu;
    if (t == 0) {
        sh.fthr[0] = sh.fthr[1] = -INFINITY;
        sh.fcut[0] = sh.fcut[1] = -INFINITY;
        sh.inf_lim = 0xffffffffu;
    }
    __syncthreads();
    // A masked row with at most RW_BUF allowed ids (every other x~ and y is
    // -inf) takes its statistics and lists from the allowed ids alone,
    // gathered in index order to row scratch (which the sums reuse): the
    // lists then hold every allowed id (observers) and every y above -inf
    // (sampler), of which the selections take the same first entries as from
    // the whole row. Not for greedy rows (the last maximal element may be a
    // masked -inf), T = inf (a masked y / T is NaN) or rows with fewer than
    // Ko finite x~ (their observers' list ends with -inf ids of the whole
    // row).
    // (the gathered count and whether the gather ran are kept in LDS: few
    // values stay live across the stream below)
    bool gath = false;
    if (t == 0) { sh.g_n = 0; sh.g_done = 0; }
    if (R.allow && !greedy && !tinf) {
        const float* gcx = rw_scratch(a, r);
        const uint32_t gn = rw_gather_allowed(R.row, R.allow, V, R.np, rw_scratch(a, r), R.gfl, R.gy);
        if (t == 0) { sh.g_n = gn; sh.g_done = 1; }
        if (gn && gn <= RW_BUF) {
            uint32_t nf = 0;
            for (uint32_t i = t; i < gn; i += RW_NT) nf += gcx[i] > -INFINITY ? 1u : 0u;
            nf = block_sum_u<RW_NT>(nf, sh.ru[4]);
            gath = rw_uni(nf) >= Ko;
            if (gath && smode == 3) { smode = 0; Ks = 0; }
        }
    }
    RW_T(1);
    // ---- the lists from the group maxima of zs_k_scan
    bool fast = false;
    if (!gath && has_groups) {
        if (Ks > ZS_KS && !rw_wide_fits(Ks, (V + (1u << a.gshift) - 1u) >> a.gshift)) { smode = 0; Ks = 0; }
        rw_gst G = {omax, ymax, rejf, 0ull, 0u, 0u, 0u, false, false};
        fast = rw_groups(a, r, R, greedy, tinf, smode, Ks, Ko, G);
        if (fast) {
            omax = G.omax; ymax = G.ymax; rejf = G.rejf; gbest = G.gbest;
            n_o = G.n_o; n_s = G.n_s; fl = G.fl; s_over = G.s_over;
        }
        if ((!fast && Ks > ZS_KS) || G.s_drop) { smode = 0; Ks = 0; }
    }
    uint32_t g = 0;
    const uint32_t ng = (gath || fast) ? 0u : R.tiles;
    // the admission thresholds in scalar registers: they change only where
    // the lists are set up (first tile) and compacted (outside the stream)
    float r_tfo = -INFINITY, r_tfs = -INFINITY;
    bool r_allo = true, r_alls = true;
    uint32_t r_ilim = 0xffffffffu;
    auto load_thr = [&]() {
        r_tfo = rw_unif(sh.fthr[0]);
        r_tfs = rw_unif(sh.fthr[1]);
        r_allo = rw_uni(thr_o < 0 ? 1u : 0u) != 0u;
        r_alls = rw_uni(thr_s < 0 ? 1u : 0u) != 0u;
        r_ilim = rw_uni(sh.inf_lim);
    };
    if (gath) {
        const float* gcx = rw_scratch(a, r);
        const uint32_t gn = rw_uni(sh.g_n);
        const uint32_t gn4 = (gn + 3) & ~3u;
        const float* gy = gcx + gn4;
        const uint32_t* gid = reinterpret_cast<const uint32_t*>(gy + gn4);
        for (uint32_t i = t; i < gn; i += RW_NT) {
            const float x = gcx[i], y = gy[i];
            const uint32_t id = gid[i];
            omax = fmaxf(omax, x);
            ymax = fmaxf(ymax, y);
            if (x != x) fl |= ZS_CF_OBS_NAN;
            if (y != y) {
                fl |= ZS_CF_Z_NAN;
                last_nan = max(last_nan, (int)id);
            }
            if (Ko) LO.buf[i] = ((unsigned long long)(~zs_total_key(x + 0.0f)) << 32) | id;
            if (smode != 0 && y > -INFINITY) {
                const uint32_t p = atomicAdd(&cnt_s[0], 1u);
                if (smode == 1 || p < ZS_SMALL_CAP) LS.buf[p] = ((unsigned long long)(~zs_total_key(y)) << 32) | id;
            }
        }
        __syncthreads();
        n_o = Ko ? gn : 0u;
        n_s = rw_uni(cnt_s[0]);
        if (smode == 2 && n_s > ZS_SMALL_CAP) s_over = true;
    }
    while (g < ng) {
        auto tile = [&](uint32_t g, int u, const float (&x)[4], const float (&y)[4]) {
            const uint32_t idx0 = g * RW_G + 4 * t;
            // branch-free statistics (ids >= V read -inf: neutral here)
            omax = fmaxf(omax, fmaxf(fmaxf(x[0], x[1]), fmaxf(x[2], x[3])));
            ymax = fmaxf(ymax, fmaxf(fmaxf(y[0], y[1]), fmaxf(y[2], y[3])));
            uint32_t nx = 0, ny = 0;
#pragma unroll
            for (int q = 0; q < 4; q++) {
                nx |= (x[q] != x[q]) ? 1u : 0u;
                ny |= (y[q] != y[q]) ? (1u << q) : 0u;
            }
            if (nx) fl |= ZS_CF_OBS_NAN;
            if (ny) {
                fl |= ZS_CF_Z_NAN;
                last_nan = max(last_nan, (int)(idx0 + 31 - __clz(ny)));
            }
            // valid ids of the thread (the last tile only is partial)
            const uint32_t vm = idx0 + 4 <= V ? 15u : (idx0 >= V ? 0u : (1u << (V - idx0)) - 1u);
            if (tinf) {
                // y / inf is NaN for a real y = +-inf (ids past the range read
                // -inf and are no elements)
#pragma unroll
                for (int q = 0; q < 4; q++)
                    if (((vm >> q) & 1u) && (y[q] == INFINITY || y[q] == -INFINITY)) fl |= ZS_CF_Z_NAN;
            }
            if (greedy) {
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    if (y[q] != y[q] || idx0 + q >= V) continue;
                    // -0.0 and +0.0 compare equal in the reference (partial_cmp)
                    const uint32_t k = zs_total_key(y[q] == 0.0f ? 0.0f : y[q]);
                    const unsigned long long c = ((unsigned long long)k << 32) | (idx0 + q + 1);
                    gbest = c > gbest ? c : gbest;
                }
            }
            if (!thr_init) {
                // initial thresholds (first tile): in every wave the c-th largest
                // thread maximum has at least c elements of that wave at or above
                // it, so the smallest of the waves' values, with c = ceil(K / RW_NW),
                // has at least K elements of this tile at or above it (ids >= V
                // hold key 0)
                thr_init = true;
                if (Ko || Ks) {
                    uint32_t kx[4], ky[4];
                    keys(x, y, kx, ky);
                    uint32_t mo = 0, ms = 0;
#pragma unroll
                    for (int q = 0; q < 4; q++) {
                        if (!((vm >> q) & 1u)) continue;
                        mo = max(mo, kx[q]);
                        ms = max(ms, ky[q]);
                    }
                    const uint32_t so = wave_sort_u32(mo), ss = wave_sort_u32(ms);
                    const int co = max((int)((Ko + RW_NW - 1) / RW_NW), 1), cs = max((int)((Ks + RW_NW - 1) / RW_NW), 1);
                    const uint32_t wo = __shfl(so, 64 - co, 64), ws = __shfl(ss, 64 - cs, 64);
                    // observers: -inf values rank by id, so once this tile holds
                    // Ko of them, a -inf of a larger id than the Ko-th can never
                    // be among the first Ko (masked rows are mostly -inf)
                    uint32_t minf = 0;
#pragma unroll
                    for (int q = 0; q < 4; q++) minf |= (((vm >> q) & 1u) && x[q] == -INFINITY) ? (1u << q) : 0u;
                    const uint32_t ninf = (uint32_t)__popc(minf), winf = wave_incl_scan_u(ninf);
                    if (zs_lane() == 63) sh.ru[4][zs_wid()] = winf;
                    if (zs_lane() == 0) { sh.ru[2][zs_wid()] = wo; sh.ru[3][zs_wid()] = ws; }
                    rw_bar();
                    uint32_t a0 = 0xffffffffu, a1 = 0xffffffffu, ibefore = 0;
#pragma unroll
                    for (int w = 0; w < RW_NW; w++) {
                        a0 = min(a0, sh.ru[2][w]); a1 = min(a1, sh.ru[3][w]);
                        ibefore += (uint32_t)w < (uint32_t)zs_wid() ? sh.ru[4][w] : 0u;
                    }
                    ibefore += winf - ninf;
                    if (Ko && ibefore < Ko && Ko <= ibefore + ninf) {
                        // the (Ko - ibefore)-th set bit of minf
                        uint32_t mm = minf;
                        for (uint32_t k = Ko - ibefore; k > 1; k--) mm &= mm - 1u;
                        sh.inf_lim = idx0 + (uint32_t)(__ffs(mm) - 1);
                    }
                    rw_bar();
                    if (t == 0) {
                        // observers: a bound at or below the key of -inf admits
                        // every id (equal -inf logprobs rank by id). Sampler:
                        // the values above -inf (a k-th value of -inf makes
                        // every finite value a survivor; -inf ids never are)
                        const uint32_t kmin = zs_total_key(-INFINITY);
                        thr_o = a0 > kmin ? (long long)a0 - 1 : -1;
                        thr_s = a1 > kmin ? (long long)a1 - 1 : (long long)kmin;
                        // (as a value, the key below that of +0 is -0, which no
                        // zero exceeds: the value below both zeros then)
                        const uint32_t kneg0 = zs_total_key(-0.0f);
                        sh.fthr[0] = a0 > kmin ? zs_key_to_float(a0 - 1u == kneg0 ? kneg0 - 1u : a0 - 1u) : -INFINITY;
                        sh.fthr[1] = a1 > kmin ? zs_key_to_float(a1 - 1u == kneg0 ? kneg0 - 1u : a1 - 1u) : -INFINITY;
                    }
                    rw_bar();
                    load_thr();
                }
            }
            // admissions, compared as values: a key above the threshold key is a
            // value above the threshold value, -0 and +0 aside (they compare
            // equal: only the value of the k-th entry matters, and observers
            // rank equal values by id) and NaN aside (a NaN row takes no list);
            // a threshold below every key (-1) admits every valid id
            const uint32_t slot = grp % 3;
            uint32_t po = 0, ps = 0;
            {
                const float tfo = r_tfo, tfs = r_tfs;
                const bool allo = r_allo, alls = r_alls;
                const uint32_t ilim = r_ilim;
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    po |= ((x[q] > tfo || allo) && (x[q] != -INFINITY || idx0 + q <= ilim)) ? (1u << q) : 0u;
                    if (smode == 1) {
                        const bool in = y[q] > tfs || alls;
                        ps |= in ? (1u << q) : 0u;
                        if (!in) rejf = fmaxf(rejf, y[q]);
                    }
                }
                po &= Ko ? vm : 0u;
                ps &= vm;
            }
            if (smode == 2 && !s_over) {
                // every value above -inf: one reservation per wave (places past
                // ZS_SMALL_CAP are not written; the count ends the list)
                uint32_t m = 0;
#pragma unroll
                for (int q = 0; q < 4; q++) m |= (y[q] > -INFINITY) ? (1u << q) : 0u;
                m &= vm;
                const uint32_t c = __popc(m);
                uint32_t inc = c;
                for (int d = 1; d < 64; d <<= 1) {
                    const uint32_t o = __shfl_up(inc, d, 64);
                    if (zs_lane() >= d) inc += o;
                }
                const uint32_t wtot = __shfl(inc, 63, 64);
                uint32_t base = 0;
                if (wtot) {
                    if (zs_lane() == 0) base = atomicAdd(&cnt_s[slot], wtot);
                    base = __shfl(base, 0, 64);
                }
                uint32_t p = n_s + base + inc - c;
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    if (!((m >> q) & 1u)) continue;
                    if (p < ZS_SMALL_CAP) LS.buf[p] = ((unsigned long long)(~zs_total_key(y[q])) << 32) | (idx0 + q);
                    p++;
                }
            }
            if (po | ps) {
                uint32_t kx[4], ky[4];
                keys(x, y, kx, ky);
                if (po) rw_admit(LO, &cnt_o[slot], n_o, po, kx, idx0, g, &sh.ovf[slot]);
                if (ps) rw_admit(LS, &cnt_s[slot], n_s, ps, ky, idx0, g, &sh.ovf[slot]);
            }
            if (u != 3) return false;
            // end of the group: counts, overflow, compaction need
            if (t == 0) {
                const uint32_t nx = (grp + 1) % 3;
                cnt_o[nx] = 0;
                cnt_s[nx] = 0;
                sh.ovf[nx] = 0xffffffffu;
            }
            rw_bar();
            n_o += rw_uni(cnt_o[slot]);
            n_s += rw_uni(cnt_s[slot]);
            const uint32_t ovf = rw_uni(sh.ovf[slot]);
            lastslot = slot;
            grp++;
            // more than ZS_SMALL_CAP finite values: the small-survivor list
            // is dropped (its count ended it; nothing to compact)
            if (smode == 2 && !s_over && n_s > ZS_SMALL_CAP) s_over = true;
            p1stop = ovf != 0xffffffffu || n_o > RW_KEEP || (smode == 1 && n_s > RW_KEEP);
            return p1stop;
        };
        // (rows with more patches than the LDS head take the loop that can
        // read the rest from global memory)
        load_thr();
        g = R.np > ZS_PATCH_LDS ? rw_stream<true>(R, sh, g, tile) : rw_stream<false>(R, sh, g, tile);
        if (!p1stop) break;
        p1stop = false;
        // compactions (rare): a list past RW_KEEP is cut to its first K. After
        // an overflow, the entries of the tiles from the first one that lost
        // an entry are dropped; that tile is admitted again element by element
        // with compactions as needed (every round places at least
        // RW_BUF - RW_KEEP entries), and the stream resumes after it (the
        // statistics are maxima and flags, which a second visit does not
        // change).
        __syncthreads();
        const uint32_t ovf = sh.ovf[lastslot];
        const uint32_t idlim = ovf != 0xffffffffu ? ovf * RW_G : 0xffffffffu;
        if (smode == 2 && !s_over && (n_s > ZS_SMALL_CAP || ovf != 0xffffffffu)) s_over = true;
        auto compact_lists = [&](uint32_t lim) {
            if (Ko && (n_o > RW_KEEP || lim != 0xffffffffu))
                n_o = rw_compact(0, LO, min(n_o, (uint32_t)RW_BUF), Ko, lim, &sh.fthr[0], &sh.fcut[0]);
            if (smode == 1 && (n_s > RW_KEEP || lim != 0xffffffffu)) {
                n_s = rw_compact(1, LS, min(n_s, (uint32_t)RW_BUF), Ks, lim, &sh.fthr[1], &sh.fcut[1]);
                rejf = fmaxf(rejf, sh.fcut[1]);   // entries cut count as turned away
            }
        };
        compact_lists(idlim);
        if (t < 3) { cnt_o[t] = 0; cnt_s[t] = 0; sh.ovf[t] = 0xffffffffu; }
        __syncthreads();
        if (ovf != 0xffffffffu && ovf < ng) {
            float x[4], y[4];
            rw_tile(R, sh, ovf, x, y);
            uint32_t kx[4], ky[4];
            keys(x, y, kx, ky);
            const uint32_t idx0 = ovf * RW_G + 4 * t;
            const uint32_t vm = idx0 + 4 <= V ? 15u : (idx0 >= V ? 0u : (1u << (V - idx0)) - 1u);
            uint32_t po = 0, ps = 0;
            for (int round = 0; ; round++) {
                // the tile's elements above the current thresholds, minus those placed
                const float tfo = sh.fthr[0], tfs = sh.fthr[1];
                const bool allo = thr_o < 0, alls = thr_s < 0;
                uint32_t wo = 0, ws = 0;
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    wo |= ((x[q] > tfo || allo) && (x[q] != -INFINITY || idx0 + q <= sh.inf_lim)) ? (1u << q) : 0u;
                    if (smode == 1) {
                        const bool in = y[q] > tfs || alls;
                        ws |= in ? (1u << q) : 0u;
                        if (!in) rejf = fmaxf(rejf, y[q]);
                    }
                }
                wo &= Ko ? vm : 0u;
                ws &= vm;
                if (round == 0) { po = wo; ps = ws; }
                else { po &= wo; ps &= ws; }
                // place what fits (the rest stays in po / ps)
                uint32_t lo = 0, ls = 0;
                {
                    const uint32_t n1 = __popc(po), n2 = __popc(ps);
                    uint32_t p1 = n_o + (n1 ? atomicAdd(&cnt_o[0], n1) : 0u);
                    uint32_t p2 = n_s + (n2 ? atomicAdd(&cnt_s[0], n2) : 0u);
#pragma unroll
                    for (int q = 0; q < 4; q++) {
                        if ((po >> q) & 1u) {
                            if (p1 < RW_BUF) LO.buf[p1] = ((unsigned long long)(~kx[q]) << 32) | (idx0 + q);
                            else lo |= 1u << q;
                            p1++;
                        }
                        if ((ps >> q) & 1u) {
                            if (p2 < RW_BUF) LS.buf[p2] = ((unsigned long long)(~ky[q]) << 32) | (idx0 + q);
                            else ls |= 1u << q;
                            p2++;
                        }
                    }
                }
                po = lo;
                ps = ls;
                __syncthreads();
                n_o = min(n_o + cnt_o[0], (uint32_t)RW_BUF);
                n_s = min(n_s + cnt_s[0], (uint32_t)RW_BUF);
                const bool more = __syncthreads_or((po | ps) != 0u);
                if (t == 0) { cnt_o[0] = 0; cnt_s[0] = 0; }
                if (!more) break;
                compact_lists(0xffffffffu);
                __syncthreads();
            }
            compact_lists(0xffffffffu);   // back below RW_KEEP for the stream
            __syncthreads();
            grp = 0;
            g = ovf + 1;
        } else {
            grp = 0;
            g = g + 1;
        }
    }
    RW_T(2);
    // ---- row statistics (one workgroup reduction)
    {
        omax = wave_max_f(omax);
        ymax = wave_max_f(ymax);
        fl = wave_or_u(fl);
        last_nan = wave_max_i(last_nan);
        rejf = wave_max_f(rejf);
        gbest = zs_wave_reduce(gbest, [](unsigned long long x, unsigned long long y) { return x > y ? x : y; });
        if (zs_lane() == 0) {
            sh.rf[0][zs_wid()] = omax; sh.rf[1][zs_wid()] = ymax;
            sh.ru[0][zs_wid()] = fl; sh.rf[2][zs_wid()] = rejf;
            sh.ru[2][zs_wid()] = (uint32_t)last_nan;
            sh.rl[zs_wid()] = gbest;
        }
        __syncthreads();
        omax = -INFINITY; ymax = -INFINITY; fl = 0; rejf = -INFINITY; last_nan = -1; gbest = 0;
#pragma unroll
        for (int w = 0; w < RW_NW; w++) {
            omax = fmaxf(omax, sh.rf[0][w]); ymax = fmaxf(ymax, sh.rf[1][w]);
            fl |= sh.ru[0][w]; rejf = fmaxf(rejf, sh.rf[2][w]);
            last_nan = max(last_nan, (int)sh.ru[2][w]);
            gbest = sh.rl[w] > gbest ? sh.rl[w] : gbest;
        }
        __syncthreads();
    }
    const float M = rw_unif(omax);
    const float zmax = rw_unif(zs_temper(ymax, T));   // max z = temper(max y): monotone
    const bool special = (fl & ZS_CF_OBS_NAN) || M == INFINITY || M == -INFINITY;
    uint32_t obs_need = 0;
    if (!special && want_obs) obs_need |= ZS_OBS_S;
    if (!special && want_unc) obs_need |= ZS_OBS_H;
    // short lists are sorted whole, the observers' by wave 0 and the sampler's
    // by wave 1 at the same time
    const bool short_o = n_o <= RW_SEL_CAP, short_s = smode == 1 && n_s <= RW_SEL_CAP;
    if (short_o || short_s) {
        if (short_o && Ko && t < 64) rw_wave_sort(sh.u.b.o, n_o);
        if (short_s && t >= 64 && t < 128) rw_wave_sort(sh.u.b.s, n_s);
        __syncthreads();
    }
    // observer candidates: the first Ko entries of the sorted list
    uint32_t n_cand = 0;
    if (Ko) {
        const uint32_t n = short_o ? n_o : rw_select(0, min(n_o, (uint32_t)RW_BUF), Ko, 0xffffffffu);
        n_cand = min(n, Ko);
        if (t < n_cand) {
            sh.cand_id[t] = (uint32_t)sh.u.b.o[t];
            sh.cand_x[t] = zs_key_to_float(~(uint32_t)(sh.u.b.o[t] >> 32));
        }
    }
    RW_T(3);

    // ---------------- sampler decisions
    uint32_t token = 0, mode = ZS_MODE_DONE, status = 0, has_thr = 0, thr_key = 0;
    float thr = -INFINITY;
    if (greedy) {
        // sampler.rs:35-42, max_by over partial_cmp: the last maximal element;
        // a NaN compares Equal, so the fold restarts after the last NaN
        status |= ZS_ST_GREEDY;
        if (last_nan < 0) {
            token = gbest ? (uint32_t)(gbest & 0xffffffffull) - 1u : 0u;
        } else {
            const uint32_t L = (uint32_t)last_nan;
            unsigned long long gb = 0;
            rw_stream<true>(R, sh, 0, [&](uint32_t g, int, const float (&x)[4], const float (&y)[4]) {
                const uint32_t idx0 = g * RW_G + 4 * t;
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    const uint32_t id = idx0 + q;
                    if (id >= V || id <= L || y[q] != y[q]) continue;
                    const uint32_t k = zs_total_key(y[q] == 0.0f ? 0.0f : y[q]);
                    const unsigned long long c = ((unsigned long long)k << 32) | (id + 1);
                    gb = c > gb ? c : gb;
                }
                return false;
            });
            gb = zs_wave_reduce(gb, [](unsigned long long x, unsigned long long y) { return x > y ? x : y; });
            if (zs_lane() == 0) sh.rl[zs_wid()] = gb;
            __syncthreads();
            gb = 0;
#pragma unroll
            for (int w = 0; w < RW_NW; w++) gb = sh.rl[w] > gb ? sh.rl[w] : gb;
            __syncthreads();
            token = gb ? (uint32_t)(gb & 0xffffffffull) - 1u : L;
        }
    } else if ((fl & ZS_CF_Z_NAN) || zmax == INFINITY || zmax == -INFINITY) {
        // exp_sum is NaN: every comparison in the draw fails -> V-1 (sampler.rs:127)
        status |= ZS_ST_NONFINITE;
        token = V - 1;
    } else {
        bool small = false;
        uint32_t nsv = 0;
        if (smode == 1) {
            const uint32_t n = short_s ? n_s : rw_select(1, min(n_s, (uint32_t)RW_BUF), Ks + 1, 0xffffffffu);
            // the k-th largest z is temper(the k-th largest y); a list of
            // fewer than k holds every y above -inf, so the k-th is -inf
            const float yk = n >= Ks ? zs_key_to_float(~(uint32_t)(sh.u.b.s[Ks - 1] >> 32)) : -INFINITY;
            thr = zs_temper(yk, T);
            thr_key = zs_total_key(thr);
            has_thr = 1;
            // every element at the threshold must be listed: after the first
            // k, the next listed y and the largest y turned away must map
            // below it (or the threshold is -inf: every finite value listed)
            bool complete = thr == -INFINITY;
            if (!complete) {
                const float ynext = n > Ks ? zs_key_to_float(~(uint32_t)(sh.u.b.s[Ks] >> 32)) : -INFINITY;
                const float yrej = rejf;
                complete = zs_temper(ynext, T) < thr && zs_temper(yrej, T) < thr;
            }
            if (thr == 0.0f) complete = false;  // the other zero also survives
            if (complete) {
                // survivors: !(z < thr) (sampler.rs:59-63) and above -inf
                if (t < 64) {
                    uint32_t c = 0;
                    for (uint32_t i0 = 0; i0 < Ks; i0 += 64) {
                        const uint32_t i = i0 + t;
                        float zi = -INFINITY;
                        if (i < Ks && i < n) zi = zs_temper(zs_key_to_float(~(uint32_t)(sh.u.b.s[i] >> 32)), T);
                        const bool sv = zi > -INFINITY;
                        const unsigned long long m = __ballot(sv);
                        if (sv) {
                            const uint32_t p = c + __popcll(m & ((1ull << t) - 1ull));
                            sh.sval[p] = zi;
                            sh.sidx[p] = (uint32_t)sh.u.b.s[i];
                        }
                        c += __popcll(m);
                    }
                    if (t == 0) sh.n_surv = c;
                }
                __syncthreads();
                nsv = sh.n_surv;
                small = true;
            }
        } else if (smode == 2 && !s_over) {
            // every y above -inf, unordered (<= ZS_SMALL_CAP); their z
            if (t < 64) {
                uint32_t c = 0;
                for (uint32_t i0 = 0; i0 < n_s; i0 += 64) {
                    const uint32_t i = i0 + t;
                    float zi = -INFINITY;
                    if (i < n_s) zi = zs_temper(zs_key_to_float(~(uint32_t)(sh.u.b.s[i] >> 32)), T);
                    const bool sv = zi > -INFINITY;
                    const unsigned long long m = __ballot(sv);
                    if (sv) {
                        const uint32_t p = c + __popcll(m & ((1ull << t) - 1ull));
                        sh.sval[p] = zi;
                        sh.sidx[p] = (uint32_t)sh.u.b.s[i];
                    }
                    c += __popcll(m);
                }
                if (t == 0) sh.n_surv = c;
            }
            __syncthreads();
            nsv = sh.n_surv;
            small = true;
        } else if (smode == 3) {
            // the k-th largest key among the listed ones (fewer than k: -inf)
            const float yk = n_s >= Ks ? zs_key_to_float(rw_kth_key(0xffffffffu, n_s, Ks)) : -INFINITY;
            thr = zs_temper(yk, T);
            thr_key = zs_total_key(thr);
            has_thr = 1;
        } else if (has_topk) {
            has_thr = 2;   // zs_k_big selects the threshold
        }
        if (small) {
            __syncthreads();
            rw_small(b.d_seed[r], b.d_counter[r], V, P, rw_uni(nsv), zmax, sh);
            __syncthreads();
            token = sh.tok;
            // (documented for the sets of at most ZS_KS, or no top-k)
            if (smode == 2 || Ks <= ZS_KS) status |= ZS_ST_SMALL;
        } else {
            mode = ZS_MODE_BIG;
        }
    }
    __syncthreads();
    RW_T(4);

    // ---------------- the row sums, left to zs_sums.hip: the sampler's S of a
    // big row (on the caller's stream, before the big-row kernels), S_obs
    // (logprobs and uncertainty) and the entropy (on the side stream). A
    // masked row's sums run over its allowed ids, gathered to row scratch
    // (when at most RW_BUF and a quarter of the row are allowed), else over
    // the whole row with its allow bits.
    const bool doA = (obs_need & ZS_OBS_S) != 0;
    const bool doB = mode == ZS_MODE_BIG && has_thr != 2;
    const bool doH = (obs_need & ZS_OBS_H) != 0;
    uint32_t gn = 0;
    if (R.allow && (doA || doB || doH))
        gn = rw_uni(sh.g_done) ? rw_uni(sh.g_n) : rw_gather_allowed(R.row, R.allow, V, R.np, rw_scratch(a, r), R.gfl, R.gy);

    // ---------------- row state for the sums, the big-row kernels and zs_k_final
    if (t == 0) {
        st.rounds = (doB ? (1u << ZS_SUM_SAMP_S) : 0u) | (doA ? (1u << ZS_SUM_OBS_S) : 0u) |
                    (doH ? (1u << ZS_SUM_OBS_H) : 0u);
        st.g_n = gn;
        st.z_max = zmax;
        st.has_thr = has_thr;
        st.thr_key = thr_key;
        st.mode = mode;
        st.token = token;
        st.status = status;
        st.obs_max = M;
        st.obs_special = special ? 1u : 0u;
        st.obs_need = obs_need;
        st.n_cand = n_cand;
        st.klist = 0;
        st.kpend = 0;
        st.kident = 0;
        st.knorm = 0;
        st.samp_S = -0.0f;
        st.obs_S = -0.0f;
        st.obs_H = 0.0f;
    }
    if (t < n_cand) { st.cand_id[t] = sh.cand_id[t]; st.cand_x[t] = sh.cand_x[t]; }
    if (mode == ZS_MODE_BIG) {
        // bucket counts and masses of the top-p walk, accumulated by zs_k_pv
        zs_tp_bucket* bk = a.tp_bk + (size_t)r * ZS_TP_NB;
        for (uint32_t i = t; i < ZS_TP_NB; i += RW_NT) { bk[i].cnt = 0u; bk[i].mass = 0.0f; }
    }
    RW_T(5);
#ifdef ZS_WALK_DEBUG
    if (t == 0) atomicAdd(&rw_dbg[7], 1ull);
#endif
}

#ifdef ZS_WALK_DEBUG
extern "C" int zs_dbg_row_stats(unsigned long long* out) {
    if (hipMemcpyFromSymbol(out, HIP_SYMBOL(rw_dbg), 16 * sizeof(unsigned long long)) != hipSuccess) return -1;
    static unsigned long long zero[16];
    return hipMemcpyToSymbol(HIP_SYMBOL(rw_dbg), zero, sizeof(zero)) == hipSuccess ? 0 : -1;
}
#endif

extern "C" int zs_row_launch(const zs_sargs& a, hipStream_t stream) {
    const uint32_t words = (a.b.V + 31) / 32;
    size_t tail = 2 * rw_bias_words(words);   // rw_patches' bias bitmaps, then the group maxima
    if (a.gshift) {
        const uint32_t ng = (a.b.V + (1u << a.gshift) - 1u) >> a.gshift;
        const dim3 grid((a.b.V + SC_IDS - 1) / SC_IDS, a.b.B);
        if (a.gshift == 4) hipLaunchKernelGGL(zs_k_scan<4>, grid, dim3(SC_NT), 0, stream, a);
        else if (a.gshift == 5) hipLaunchKernelGGL(zs_k_scan<5>, grid, dim3(SC_NT), 0, stream, a);
        else hipLaunchKernelGGL(zs_k_scan<6>, grid, dim3(SC_NT), 0, stream, a);
        tail = std::max(tail, (size_t)2 * ng);
    }
    hipLaunchKernelGGL(zs_k_row, dim3(a.b.B), dim3(RW_NT), (2 * words + tail) * sizeof(uint32_t), stream, a);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}
