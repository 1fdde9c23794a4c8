// SPDX-License-Identifier: MIT
//
// The select pass of the decode: one workgroup per example walks the T steps
// (or the one step of the step API) over the row pass's shortlists.
//
// Per step it stages the step's row statistics and shortlists in LDS, builds
// the candidates (EOS carry-forward; shortlist entries with n-gram blocking
// and the repetition penalty), keeps the best K in an LDS collector under the
// reference's total order (reference src/common.hpp:269-302), and then proves
// the selection exact: a row whose bound could still beat the K-th selected
// candidate is rescanned in full from HBM. The trace, the beam state and the
// prefixes advance as in reference src/decoder.cpp:122-187, 314-350.
//
// Included by one translation unit per input type (select_f32.hip,
// select_f16.hip, select_bf16.hip), which instantiates the kernels of its
// type; select.hip plans and dispatches.
#pragma once

#include <hip/hip_runtime.h>

#include "device_common.hpp"
#include "select_plan.hpp"

namespace dbs_hip {

namespace {

// Rows rescanned since the last reset (read through dbs_hip_profile_read).
__device__ unsigned long long g_rescanned_rows;
// Waits for a step of the overlapped decode that gave up (should stay 0).
__device__ unsigned long long g_wait_timeouts;

// Overlapped decode: waits until the row pass has counted every row of
// example b's step t: one at step 0, else one per beam of the example (the
// row pass reads, and counts, exactly those rows). The count is a relaxed
// hint of when to start reading: each word read afterwards is checked by its
// own tag (wait_tagged). Every wait is bounded (p.wait_ticks of the 100 MHz
// real-time counter; a whole row pass takes milliseconds): the row pass
// never waits on the select pass, so the bound only keeps a fault elsewhere
// from hanging the workgroup. One thread; false when the wait gave up.
__device__ __forceinline__ bool wait_step_rows(const DecodeParams& p, int b, int t) {
    const int need = (t == 0 ? 1 : beams_of(p, b)) + p.wait_extra;
    const int32_t* cnt = p.step_done + static_cast<int64_t>(b) * p.T + t;
    if (__hip_atomic_load(cnt, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) >= need) return true;
    const unsigned long long t0 = __builtin_amdgcn_s_memrealtime();
    while (__hip_atomic_load(cnt, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < need) {
        __builtin_amdgcn_s_sleep(4);
        if (__builtin_amdgcn_s_memrealtime() - t0 > p.wait_ticks) {
            atomicAdd(&g_wait_timeouts, 1ull);
            return false;
        }
    }
    return true;
}

// Split launch of the overlapped decode: whether this launch decodes example
// b. The early launch waits for the example's first row at most
// p.early_ticks and then claims it; the late launch takes what the early one
// left. One thread.
__device__ __forceinline__ bool claim_example(const DecodeParams& p, int b) {
    if (!p.early) return __hip_atomic_load(p.claimed + b, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == 0;
    const int need = 1 + p.wait_extra;
    const int32_t* cnt = p.step_done + static_cast<int64_t>(b) * p.T;
    const unsigned long long t0 = __builtin_amdgcn_s_memrealtime();
    while (__hip_atomic_load(cnt, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < need) {
        __builtin_amdgcn_s_sleep(4);
        if (__builtin_amdgcn_s_memrealtime() - t0 > p.early_ticks) return false;
    }
    __hip_atomic_store(p.claimed + b, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return true;
}

// Overlapped decode: one tagged word of the row pass (RowInfo half or
// shortlist entry), waited for while its tag is 0; false when the wait gave
// up (bounded like wait_step_rows).
__device__ __forceinline__ bool wait_tagged(const DecodeParams& p, const uint32_t* src, uint32_t& lo, uint32_t& hi) {
    if (read_tagged(src, lo, hi)) return true;
    const unsigned long long t0 = __builtin_amdgcn_s_memrealtime();
    while (!read_tagged(src, lo, hi)) {
        __builtin_amdgcn_s_sleep(2);
        if (__builtin_amdgcn_s_memrealtime() - t0 > p.wait_ticks) {
            atomicAdd(&g_wait_timeouts, 1ull);
            return false;
        }
    }
    return true;
}

// The key of the M-th largest of n keys in LDS (n a multiple of kSelectThreads,
// at most 2048; zero keys pad), its low LOW bits zero (at least M keys reach
// it), in every thread of the workgroup: the radix select of mth_largest_key,
// each wavefront counting its quarter, the counts exchanged through part [8]
// (one barrier a bit). The caller's barrier precedes it.
template <int LOW>
__device__ __forceinline__ uint32_t mth_largest_wg(const uint32_t* key, int n, int M, int32_t* part) {
    constexpr int kPer = 2048 / kSelectThreads;
    const int tid = static_cast<int>(threadIdx.x), w = tid >> 6;
    uint32_t k[kPer];
#pragma unroll
    for (int u = 0; u < kPer; ++u) k[u] = u * kSelectThreads < n ? key[u * kSelectThreads + tid] : 0u;
    uint32_t prefix = 0;
    int need = M;
#pragma unroll 1
    for (int bit = 31; bit >= LOW; --bit) {
        const uint32_t want = (prefix >> bit) | 1u;
        int c = 0;
#pragma unroll
        for (int u = 0; u < kPer; ++u) c += __popcll(__ballot((k[u] >> bit) == want));
        int32_t* const slot = part + 4 * (bit & 1);
        if ((tid & 63) == 0) slot[w] = c;
        lds_barrier();
        const int4 all = *reinterpret_cast<const int4*>(slot);
        c = __builtin_amdgcn_readfirstlane(all.x + all.y + all.z + all.w);
        if (c >= need) {
            prefix |= 1u << bit;
        } else {
            need -= c;
        }
    }
    return prefix;
}

struct Lds {
    Cand* buf;        // [sort_cap] the collector
    int32_t* rbuf;    // [kRescanTokens] tokens gathered from one rescanned row
    uint4* key;       // [2 * kRankMax] candidate keys of a rank compaction (kRankMax used; WIDE: [4 * kRankMax])
    bool wide;        // more than kListBeams beams
    int32_t* rank;    // [4 * kRankMax] (WIDE) ranks of a compaction
    int32_t* part;    // [kSelectThreads] partial ranks (or score keys)
    int32_t* surv;    // [64] candidates left by the score pass of a rank compaction
    int32_t* nsurv;   // [1] how many
    float* raw;       // [K] beams after the previous step
    float* nraw;      // [K] beams after this step (also scratch)
    float* rbound;    // [K]
    float* pen;       // [pen_len] length penalty by length
    float* inv;       // [pen_len] 1 / penalty
    int32_t* len;
    int32_t* nlen;
    int32_t* last;
    int32_t* nlast;
    int32_t* ended;
    int32_t* nended;
    int32_t* rcount;  // [K] shortlist entries of the beam's row (-2 not read, -1 no shortlist, -3 failed check)
    int32_t* plen;    // [2K] prefix lengths
    int32_t* nblk;    // [K] n-gram-blocked tokens of each beam
    ShortEntry* sl;   // [K, M + 1] the step's shortlists (see sl_at)
    int32_t* prefix;  // [2, K, P] (LDS) or the example's slice of the workspace
    int32_t* blk;     // [K, P] (LDS) or workspace
    uint32_t* sig;    // [2, K, sig_words] (LDS) prefix signatures, or null
    int sig_words;
    int V;            // vocabulary size (the keys' token field)
    int sig_shift;    // 32 - log2(32 sig_words): hash bits kept
};

// The select pass's barriers order LDS only (lds_barrier): a step's global
// loads (the next step's prefetch) and its trace stores stay in flight across
// them. The beams' prefixes and n-gram-blocked lists live in global memory
// when LDS cannot hold them (long constrained decodes); the barriers after
// they are written then also wait for global memory.
__device__ __forceinline__ void step_barrier(bool lists_global) {
    if (lists_global) __syncthreads();
    else lds_barrier();
}

struct State {
    int gave_up;  // a wait of the overlapped decode gave up
    int first_bad;  // the first invalid row read (t * K + k), else INT_MAX
    int count;
    int any_fail;
    int rcount;
    int overflow;
    uint32_t invalid;
    float tau;
    Cand thr;
};

// Entry i of beam k's shortlist in LDS. Wide beams pad the rows to M + 1
// entries, so the lanes of a wavefront reading entry i of consecutive beams
// spread over the banks.
__device__ __forceinline__ int sl_stride(int K, int M) { return K >= kWideBeam ? M + 1 : M; }
__device__ __forceinline__ int sl_at(int k, int i, int S) { return k * S + i; }

__device__ __forceinline__ float pen_of(const Lds& s, int pen_len, int l, float alpha) {
    const int c = l > 1 ? l : 1;
    return c < pen_len ? s.pen[c] : length_penalty(c, alpha);
}

__device__ __forceinline__ float inv_of(const Lds& s, int pen_len, int l, float alpha) {
    const int c = l > 1 ? l : 1;
    return c < pen_len ? s.inv[c] : 1.0f / length_penalty(c, alpha);
}

struct PrefixView {
    const int32_t* tok;
    int len;
    const uint32_t* sig;  // two bits set for every token of tok[0, len) (a superset filter), or null
    int sig_shift;
};

// The two signature bits of token v: multiplicative hashes to 32 - shift bits.
__device__ __forceinline__ uint32_t sig_bit0(int v, int shift) { return (static_cast<uint32_t>(v) * 0x9E3779B1u) >> shift; }
__device__ __forceinline__ uint32_t sig_bit1(int v, int shift) { return (static_cast<uint32_t>(v) * 0x85EBCA77u + 0x165667B1u) >> shift; }

__device__ __forceinline__ PrefixView prefix_of(const DecodeParams& p, const Lds& s, int b, int k, int cur) {
    if (p.step_mode) {
        const int l = s.len[k];
        const int L = l < 0 ? 0 : (l < p.st_stride ? l : p.st_stride);
        return PrefixView{p.st_prefix + (static_cast<int64_t>(b) * p.K + k) * p.st_stride, L, nullptr, 0};
    }
    return PrefixView{s.prefix + (static_cast<int64_t>(cur) * p.K + k) * p.prefix_cap, s.plen[cur * p.K + k],
                      s.sig ? s.sig + (cur * p.K + k) * s.sig_words : nullptr, s.sig_shift};
}

// Membership of v in a[0, n): eight independent loads in flight per round
// (the list is in LDS or global memory; its latency, not its length, bounds
// the scan).
__device__ __forceinline__ bool in_list(const int32_t* a, int n, int v) {
    int i = 0;
    for (; i + 8 <= n; i += 8) {
        int32_t t[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) t[u] = a[i + u];
        bool hit = false;
#pragma unroll
        for (int u = 0; u < 8; ++u) hit = hit | (t[u] == v);
        if (hit) return true;
    }
    bool hit = false;
    for (; i < n; ++i) hit = hit | (a[i] == v);
    return hit;
}

// Membership of v in a prefix: the signature rules most tokens out with one
// read; the rest are searched.
__device__ __forceinline__ bool in_prefix(const PrefixView& pre, int v) {
    if (pre.sig) {
        const uint32_t h0 = sig_bit0(v, pre.sig_shift), h1 = sig_bit1(v, pre.sig_shift);
        if ((((pre.sig[h0 >> 5] >> (h0 & 31u)) & (pre.sig[h1 >> 5] >> (h1 & 31u))) & 1u) == 0u) return false;
    }
    return in_list(pre.tok, pre.len, v);
}

// The candidate of token v (finite log-prob lp, statically allowed) in the
// row of beam k; false when n-gram blocking removes it. A token of the prefix
// pays the repetition penalty: raw = p + (lp - log(rep)) (reference
// src/decoder.cpp:196-258).
__device__ __forceinline__ bool make_cand(const DecodeParams& p, const Lds& s, const PrefixView& pre, int k,
                                          float praw, float inv_pen, int v, int new_len, float lp, Cand& c) {
    float value = lp;
    if (p.constrained) {
        if (p.ngram == 1) {
            if (in_prefix(pre, v)) return false;
        } else if (p.ngram > 1 && in_list(s.blk + static_cast<int64_t>(k) * p.prefix_cap, s.nblk[k], v)) {
            return false;
        }
        if (p.penalise && in_prefix(pre, v)) value = lp - p.log_rep;
    }
    const float raw = praw + value;
    c = Cand{raw * inv_pen, raw, k, v, new_len, 1};
    return true;
}

__device__ __forceinline__ void sort_cands(Cand* buf, int np) {
    const int tid = static_cast<int>(threadIdx.x);
    for (int kk = 2; kk <= np; kk <<= 1) {
        for (int j = kk >> 1; j > 0; j >>= 1) {
            for (int i = tid; i < np; i += kSelectThreads) {
                const int partner = i ^ j;
                if (partner > i) {
                    const bool desc = (i & kk) == 0;
                    const Cand a = buf[i], c = buf[partner];
                    if (desc ? before(c, a) : before(a, c)) {
                        buf[i] = c;
                        buf[partner] = a;
                    }
                }
            }
            lds_barrier();
        }
    }
}

// The candidate at collector index idx as a 96-bit integer that is larger
// exactly when the candidate comes earlier in the total order, least
// significant word first: (parent, token) as parent * V + token (asc), raw,
// score (desc; no NaN reaches the collector). No two candidates of a
// collector share (parent, token) (a carried beam is not expanded, a rescan
// first drops its row's shortlisted candidates), so length and from_logprob
// never decide; K * V < 2^31 (the argument checks). Dead sentinels (parent
// -1) rank below every other candidate by score and raw (a candidate is
// admitted only if it ranks before the sentinel) and among themselves by
// index, lower first.
__device__ __forceinline__ uint4 cand_key(const Cand& c, int idx, int V) {
    const uint32_t low = c.parent >= 0 ? static_cast<uint32_t>(c.parent) * static_cast<uint32_t>(V) +
                                             static_cast<uint32_t>(c.token)
                                       : static_cast<uint32_t>(idx);
    return make_uint4(0xffffffffu - low, ordered_key(c.raw), ordered_key(c.score), 0u);
}

// rank += (96-bit key j > key i): the borrow out of i - j, kept in VCC
// through the subtraction.
__device__ __forceinline__ void count_above96(int& rank, uint32_t i0, uint32_t i1, uint32_t i2, uint32_t j0,
                                              uint32_t j1, uint32_t j2) {
    uint32_t t;
    asm("v_sub_co_u32 %0, vcc, %2, %5\n\t"
        "v_subb_co_u32 %0, vcc, %3, %6, vcc\n\t"
        "v_subb_co_u32 %0, vcc, %4, %7, vcc\n\t"
        "v_addc_co_u32 %1, vcc, 0, %1, vcc"
        : "=&v"(t), "+v"(rank)
        : "v"(i0), "v"(i1), "v"(i2), "v"(j0), "v"(j1), "v"(j2)
        : "vcc");
}
__device__ __forceinline__ void count_before(int& rank, const uint4& i, const uint4& j) {
    count_above96(rank, i.x, i.y, i.z, j.x, j.y, j.z);
}

// rank += (64-bit key (hi, lo) j > key i): the borrow out of i - j.
__device__ __forceinline__ void count_above64(int& rank, uint32_t ilo, uint32_t ihi, uint32_t jlo, uint32_t jhi) {
    uint32_t t;
    asm("v_sub_co_u32 %0, vcc, %2, %4\n\t"
        "v_subb_co_u32 %0, vcc, %3, %5, vcc\n\t"
        "v_addc_co_u32 %1, vcc, 0, %1, vcc"
        : "=&v"(t), "+v"(rank)
        : "v"(ilo), "v"(ihi), "v"(jlo), "v"(jhi)
        : "vcc");
}

// Keeps the best K of n <= kRankMax collected candidates, in order: every
// candidate's rank is the number of keys above its own, counted by up to four
// waves per candidate over disjoint ranges of the others, and the candidates
// of rank < K move to their rank.
// Past one wavefront of candidates (few beams), a pass over the scores alone
// (the keys' most significant word) comes first: a candidate with K or more
// scores strictly above its own ranks K or later. Every candidate ranked
// before a remaining one has a score at least as high and so remains too:
// the remaining candidates' ranks among themselves are their ranks among all,
// and when at most 64 remain one wavefront ranks them.
__device__ __forceinline__ void compact_by_rank(Lds& s, State& st, int K, int n) {
    const int tid = static_cast<int>(threadIdx.x);
    const int n4 = (n + 3) & ~3;
    const bool by_score = n > 64 && K <= kScoreFilterMaxK;
    Cand c = dead_cand();
    if (tid < n4) {
        if (tid < n) {
            c = s.buf[tid];
            s.key[tid] = cand_key(c, tid, s.V);
        } else {
            s.key[tid] = make_uint4(0u, 0u, 0u, 0u);  // below every key
        }
        if (by_score) s.part[tid] = static_cast<int32_t>(tid < n ? ordered_key(c.score) : 0u);
    }
    if (by_score && tid == 0) s.nsurv[0] = 0;
    lds_barrier();
    if (by_score) {
        if (tid < n) {
            const uint32_t mine = ordered_key(c.score);
            const uint4* sk = reinterpret_cast<const uint4*>(s.part);
            int above = 0;
            int j = 0;
            for (; j + 4 <= n4 / 4; j += 4) {  // four reads in flight
                uint4 w[4];
#pragma unroll
                for (int u = 0; u < 4; ++u) w[u] = sk[j + u];
#pragma unroll
                for (int u = 0; u < 4; ++u)
                    above += (w[u].x > mine) + (w[u].y > mine) + (w[u].z > mine) + (w[u].w > mine);
            }
            for (; j < n4 / 4; ++j) {
                const uint4 w = sk[j];
                above += (w.x > mine) + (w.y > mine) + (w.z > mine) + (w.w > mine);
            }
            if (above < K) {
                const int slot = atomicAdd(s.nsurv, 1);
                if (slot < 64) s.surv[slot] = tid;
            }
        }
        lds_barrier();
        const int ns = __builtin_amdgcn_readfirstlane(s.nsurv[0]);
        if (ns <= 64) {
            if (tid < ns) {
                const int i = s.surv[tid];
                const Cand ci = s.buf[i];
                const uint4 ki = s.key[i];
                int rank = 0;
                for (int j = 0; j < ns; ++j) count_before(rank, ki, s.key[s.surv[j]]);
                if (rank < K) s.buf[rank] = ci;
                if (rank == K - 1 && before(ci, st.thr)) st.thr = ci;
            }
            if (tid == 0) st.count = n < K ? n : K;
            lds_barrier();
            return;
        }
        // many equal scores: every candidate is ranked
    }
    // wave w counts for candidates 64 gi + lane over the gj-th part of the others
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int groups = (n + 63) >> 6;
    const int parts = groups == 1 ? 4 : (groups == 2 ? 2 : 1);
    const int gi = w / parts, gj = w - gi * parts;
    int part = 0;
    if (gi < groups) {
        const int i = 64 * gi + lane;
        const uint4 ki = s.key[i];
        const int span = ((n4 / parts) + 3) & ~3;
        const int j0 = gj * span;
        const int j1 = j0 + span < n4 ? j0 + span : n4;
        int j = j0;
        for (; j + 8 <= j1; j += 8) {  // eight keys in flight
            uint4 w[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) w[u] = s.key[j + u];
#pragma unroll
            for (int u = 0; u < 8; ++u) count_before(part, ki, w[u]);
        }
        for (; j < j1; j += 4) {
            const uint4 a = s.key[j], b2 = s.key[j + 1], c2 = s.key[j + 2], d = s.key[j + 3];
            count_before(part, ki, a);
            count_before(part, ki, b2);
            count_before(part, ki, c2);
            count_before(part, ki, d);
        }
    }
    s.part[tid] = part;
    lds_barrier();
    if (tid < n) {
        const int gi_t = tid >> 6;
        int rank = 0;
        for (int g = 0; g < parts; ++g) rank += s.part[(gi_t * parts + g) * 64 + (tid & 63)];
        if (rank < K) s.buf[rank] = c;
        if (rank == K - 1 && before(c, st.thr)) st.thr = c;
    }
    if (tid == 0) st.count = n < K ? n : K;
    lds_barrier();
}

// The same for n <= 1024 candidates (more than 64 beams: the collector holds K
// to about 2 K of them). Every wavefront keeps all the keys, up to 16 a lane,
// and counts a quarter of the others against them, so that a key is read from
// LDS once, not once per wavefront (a broadcast read of 16 bytes costs the
// LDS as much as 64 distinct ones: with each wavefront counting its own
// candidates, n = 290 took 12.5 us). Bound by the compares of all pairs, n^2 /
// 16 cycles.
constexpr int kWideKeys = kWideRank * kSelectThreads / 64;  // keys per lane
__device__ __forceinline__ void compact_wide(Lds& s, State& st, int K, int n) {
    const int tid = static_cast<int>(threadIdx.x), lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    Cand c[kWideRank];
#pragma unroll
    for (int u = 0; u < kWideRank; ++u) {
        const int i = tid + u * kSelectThreads;
        if (u * kSelectThreads < n) {
            uint4 key = make_uint4(0u, 0u, 0u, 0u);  // below every key
            if (i < n) {
                c[u] = s.buf[i];
                key = cand_key(c[u], i, s.V);
            }
            s.key[i] = key;
            s.rank[i] = 0;
        }
    }
    lds_barrier();
    uint32_t k0[kWideKeys], k1[kWideKeys], k2[kWideKeys];
    int rank[kWideKeys];
#pragma unroll
    for (int u = 0; u < kWideKeys; ++u) {
        rank[u] = 0;
        k0[u] = k1[u] = k2[u] = 0u;
        if (64 * u < n) {
            const uint4 key = s.key[64 * u + lane];
            k0[u] = key.x;
            k1[u] = key.y;
            k2[u] = key.z;
        }
    }
    const int span = ((n + 15) >> 4) << 2;  // a quarter, in fours (the keys past n are zero)
    const int j1 = min(n, (w + 1) * span);
#pragma unroll 1
    for (int j = w * span; j < j1; j += 4) {
        uint4 x[4];
#pragma unroll
        for (int v = 0; v < 4; ++v) x[v] = s.key[j + v];
#pragma unroll
        for (int u = 0; u < kWideKeys; u += 2) {
            if (64 * u < n) {
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    count_above96(rank[u], k0[u], k1[u], k2[u], x[v].x, x[v].y, x[v].z);
                    count_above96(rank[u + 1], k0[u + 1], k1[u + 1], k2[u + 1], x[v].x, x[v].y, x[v].z);
                }
            }
        }
    }
#pragma unroll
    for (int u = 0; u < kWideKeys; ++u)
        if (64 * u + lane < n) atomicAdd(&s.rank[64 * u + lane], rank[u]);
    lds_barrier();
#pragma unroll
    for (int u = 0; u < kWideRank; ++u) {
        const int i = tid + u * kSelectThreads;
        if (i < n) {
            const int r = s.rank[i];
            if (r < K) s.buf[r] = c[u];
            if (r == K - 1 && before(c[u], st.thr)) st.thr = c[u];
        }
    }
    if (tid == 0) st.count = n < K ? n : K;
    lds_barrier();
}

// Sorts the collected candidates, keeps the best K, and raises the admission
// threshold to the K-th kept one when that is better.
__device__ __forceinline__ void compact(Lds& s, State& st, int K) {
    lds_barrier();
    const int n = __builtin_amdgcn_readfirstlane(st.count);
    if (s.wide && n <= kWideRank * kRankMax) {
        compact_wide(s, st, K, n);
        return;
    }
    if (n <= kRankMax) {
        compact_by_rank(s, st, K, n);
        return;
    }
    int np = 1;
    while (np < n) np <<= 1;
    for (int i = n + static_cast<int>(threadIdx.x); i < np; i += kSelectThreads) s.buf[i] = dead_cand();
    lds_barrier();
    sort_cands(s.buf, np);
    if (threadIdx.x == 0) {
        st.count = n < K ? n : K;
        if (st.count == K && before(s.buf[K - 1], st.thr)) st.thr = s.buf[K - 1];
    }
    lds_barrier();
}

// Admits c unless it ranks after the threshold (a candidate offered earlier,
// or the dead sentinel). Equal admits: after a rescan removed the threshold's
// own row from the collector, the threshold itself must come back.
__device__ __forceinline__ void offer(Lds& s, State& st, const Cand& c) {
    if (before(st.thr, c)) return;
    const int slot = atomicAdd(&st.count, 1);
    s.buf[slot] = c;
}

__device__ __forceinline__ void end_round(Lds& s, State& st, int K, int sort_cap) {
    lds_barrier();
    if (st.count > sort_cap - kSelectThreads) compact(s, st, K);
}

// The next float above x (finite or -inf).
__device__ __forceinline__ float next_above(float x) {
    const uint32_t u = f32_bits(x);
    return x == 0.0f ? bits_f32(1u) : bits_f32((u & 0x80000000u) ? u - 1u : u + 1u);
}

// Every candidate of row `row` (beam k) that does not rank after the
// threshold: a sweep over the row gathers the tokens whose score could reach
// it, then their candidates are offered to the collector. With no threshold
// yet, or more tokens than the buffer holds (the first step's one row of a
// wide beam, a step whose threshold is still low), a sweep takes the best
// score of 4 slices of the row per thread first: the keep-th best of those
// 1024 is reached by at least `keep` candidates of this row, so the tokens
// below it are left out (of 32000 at keep = 256 some 300 remain; each 256 past
// the collector's room cost a sort before). More at that score than the buffer
// holds: offered round by round.
// One workgroup reads the row, so a sweep is bound by the latency of its
// batches (kRescanPerThread loads in flight per thread, about 2 us each), and
// the full candidate test is made once per gathered token: inlined for every
// element of a batch it is more code than the instruction cache holds (80 us a
// sweep of 32000).
template <int DT, bool LOGITS>
__device__ __forceinline__ void rescan_row(const DecodeParams& p, Lds& s, State& st, int b, int k, int64_t row, float lse,
                           float praw, float inv_pen, int new_len, const PrefixView& pre, int sort_cap, int keep) {
    const bool mask_eos = new_len < min_length_of(p, b);
    const int V = p.V;
    const int tid = static_cast<int>(threadIdx.x);
    const size_t esz = DT == 0 ? 4 : 2;
    const char* base = static_cast<const char*>(p.x) + static_cast<size_t>(row) * static_cast<size_t>(V) * esz;
    const Cand thr = st.thr;
    float least = -kInf;
    const bool plain = !p.banned && !p.banned_pe && !p.row_mask && !mask_eos && !p.constrained;
    // token v's candidate, unless it is excluded, ranks after the threshold or
    // lies below `least`
    auto candidate = [&](int v, Cand& c) -> bool {
        const float x = load_one<DT>(base, v);
        const float lp = LOGITS ? x - lse : x;
        if (!(lp < kInf) || lp == -kInf) return false;
        if (static_masked(p, b, v, mask_eos)) return false;
        if (p.row_mask && gload(p.row_mask, row * V + v)) return false;
        if (!make_cand(p, s, pre, k, praw, inv_pen, v, new_len, lp, c)) return false;
        return !(c.score < least) && !before(thr, c);
    };
    // A batch's raw scores times `scale`, penalties apart (they only lower a
    // candidate); NaN, which passes no test, where there is no finite entry.
    auto scan = [&](int v0, float scale, float (&value)[kRescanPerThread]) __attribute__((always_inline)) {
        float xs[kRescanPerThread];
#pragma unroll
        for (int j = 0; j < kRescanPerThread; ++j) {  // every load made, from a clamped index
            const int v = v0 + j * kSelectThreads + tid;
            xs[j] = load_one<DT>(base, v < V ? v : V - 1);
        }
#pragma unroll
        for (int j = 0; j < kRescanPerThread; ++j) {
            const float lp = LOGITS ? xs[j] - lse : xs[j];
            const bool in = v0 + j * kSelectThreads + tid < V && lp < kInf && lp > -kInf;
            value[j] = in ? (praw + lp) * scale : __builtin_nanf("");
        }
    };
    int32_t* const tokens = s.rbuf;
#pragma unroll 1
    for (int attempt = thr.parent < 0 ? 1 : 0; attempt < 2; ++attempt) {
        lds_barrier();  // (the buffer and the flags are free)
        if (attempt == 1) {
            float best[4] = {-kInf, -kInf, -kInf, -kInf};
#pragma unroll 1
            for (int v0 = 0; v0 < V; v0 += kSelectThreads * kRescanPerThread) {
                float score[kRescanPerThread];
                scan(v0, inv_pen, score);
                if (plain) {
#pragma unroll
                    for (int j = 0; j < kRescanPerThread; ++j) best[j & 3] = fmaxf(best[j & 3], score[j]);
                } else {
                    uint32_t pass = 0;
#pragma unroll
                    for (int j = 0; j < kRescanPerThread; ++j) pass |= (score[j] > best[j & 3] ? 1u : 0u) << j;
                    while (pass != 0) {
                        const int j = __ffs(static_cast<int>(pass)) - 1;
                        pass &= pass - 1;
                        Cand c;
                        if (!candidate(v0 + j * kSelectThreads + tid, c)) continue;
#pragma unroll
                        for (int u = 0; u < 4; ++u) best[u] = (j & 3) == u ? fmaxf(best[u], c.score) : best[u];
                    }
                }
            }
            uint32_t* const slice = reinterpret_cast<uint32_t*>(s.rbuf);
#pragma unroll
            for (int u = 0; u < 4; ++u) slice[u * kSelectThreads + tid] = ordered_key(best[u]);
            lds_barrier();
            const float at = key_value(mth_largest_wg<0>(slice, 4 * kSelectThreads, keep, s.surv));
            lds_barrier();  // (the slices are read: the buffer is free)
            least = at;
        }
        if (tid == 0) st.rcount = 0;
        lds_barrier();
        // Up to a threshold of this row's penalty the candidates go by raw (the
        // score is a nondecreasing function of it), and the raw of the threshold
        // itself passes only where a token of this row could rank before it:
        // where very many entries have that raw (rows masked with the type's
        // lowest value, rows of one value) all of them would pass by score.
        const bool by_raw = !(least > thr.score) && thr.raw * inv_pen == thr.score;
        auto uniform = [](float x) { return bits_f32(__builtin_amdgcn_readfirstlane(f32_bits(x))); };
        const float scale = uniform(by_raw ? 1.0f : inv_pen);
        const float lowest = uniform(by_raw ? (k <= thr.parent ? thr.raw : next_above(thr.raw)) : fmaxf(least, thr.score));
#pragma unroll 1
        for (int v0 = 0; v0 < V; v0 += kSelectThreads * kRescanPerThread) {
            float value[kRescanPerThread];
            scan(v0, scale, value);
            uint32_t pass = 0;
#pragma unroll
            for (int j = 0; j < kRescanPerThread; ++j) pass |= (value[j] >= lowest ? 1u : 0u) << j;
            while (pass != 0) {
                const int j = __ffs(static_cast<int>(pass)) - 1;
                pass &= pass - 1;
                const int slot = atomicAdd(&st.rcount, 1);
                if (slot < kRescanTokens) tokens[slot] = v0 + j * kSelectThreads + tid;
            }
        }
        lds_barrier();
        const int n = st.rcount;
        if (n <= kRescanTokens) {
            for (int r0 = 0; r0 < n; r0 += kSelectThreads) {
                Cand c;
                if (r0 + tid < n && candidate(tokens[r0 + tid], c)) offer(s, st, c);
                end_round(s, st, keep, sort_cap);
            }
            return;
        }
    }
    for (int v0 = 0; v0 < V; v0 += kSelectThreads) {
        const int v = v0 + tid;
        Cand c;
        if (v < V && candidate(v, c)) offer(s, st, c);
        end_round(s, st, keep, sort_cap);
    }
}

// Entry i of a shortlist in global memory (more than 64 beams: the lists are
// not staged), within its row's count. Overlapped decode: waited for while
// not written yet; a wait that gives up marks the example and reads as -inf.
__device__ __forceinline__ ShortEntry list_entry(const DecodeParams& p, State& st, int64_t row, int i) {
    const uint32_t* src = reinterpret_cast<const uint32_t*>(p.shortlist + row * p.M + i);
    if (p.step_done == nullptr) return p.shortlist[row * p.M + i];
    uint32_t lo = 0, hi = 0;
    if (!read_tagged(src, lo, hi) && !wait_tagged(p, src, lo, hi)) {
        atomicOr(&st.gave_up, 1);
        return ShortEntry{-kInf, 0};
    }
    return ShortEntry{bits_f32(lo), static_cast<int32_t>(hi) - 1};
}

// PF: the next step's RowInfo and shortlists are prefetched into registers
// (chosen on the host: prefetch_fits); a separate instantiation, so the other
// paths keep their register budget.
// HOLD: the kernel claims every accumulation register (a clobber of a255),
// so no wavefront of another kernel fits on its SIMDs beside it: launched
// before a row pass of several workgroups per CU, it keeps its CUs to itself
// (registers it never uses; its own occupancy, one wavefront per SIMD, is
// unchanged).
// WIDE: more than kListBeams beams. The shortlists (shorter than the beams are
// many) stay in global memory: each thread keeps the head of its beams' lists
// in LDS, tau is the K-th largest raw of the heads, and each beam's prefix
// that reaches tau goes to the collector. Most rows give one or two of the K
// selected candidates, so a step reads a few entries per row; the rows that
// give more than their list holds (the first step's one row, a few of the
// next) fail the exactness check and are read in full.
template <int DT, bool LOGITS, bool PF, bool HOLD = false, bool WIDE = false>
__global__ __launch_bounds__(kSelectThreads) void select_kernel(DecodeParams p, SelectLayout L) {
    if constexpr (HOLD) asm volatile("" ::: "a255");
    extern __shared__ __align__(16) unsigned char smem[];
    __shared__ State st;
    if (p.claimed) {
        __shared__ int s_claim;
        if (threadIdx.x == 0) s_claim = claim_example(p, static_cast<int>(blockIdx.x)) ? 1 : 0;
        __syncthreads();
        if (s_claim == 0) return;
    }
    const int K = p.K, T = p.T, M = p.M;
    const int SL = sl_stride(K, M);
    const int b = static_cast<int>(blockIdx.x);
    const int tid = static_cast<int>(threadIdx.x);
    // WIDE: entries of each list's head in LDS, the most of 8, 4, 2 that keep
    // K of them within kHeads (8 leave 1.2 to 1.5 K candidates at tau, 2 leave
    // 2 to 4 K: each list gives few, the best ones up to 80); 0 without lists
    constexpr int kHeadMax = WIDE ? 8 : 1;
    const int hsh = K <= kHeads / 8 ? 3 : (K <= kHeads / 4 ? 2 : 1);
    const int H = WIDE && M >= 8 ? 1 << hsh : 0;

    Lds s;
    s.buf = reinterpret_cast<Cand*>(smem + L.off_buf);
    s.rbuf = reinterpret_cast<int32_t*>(smem + L.off_rbuf);
    s.key = reinterpret_cast<uint4*>(smem + L.off_key);
    s.part = reinterpret_cast<int32_t*>(smem + L.off_key + sizeof(uint4) * (WIDE ? 4 : 2) * kRankMax);
    s.wide = WIDE;
    s.rank = WIDE ? s.part + kSelectThreads + 64 + 4 : nullptr;
    s.surv = s.part + kSelectThreads;
    s.nsurv = s.surv + 64;
    float* f = reinterpret_cast<float*>(smem + L.off_f32);
    s.raw = f;
    s.nraw = f + K;
    s.rbound = f + 2 * K;
    s.pen = f + 3 * K;
    s.inv = f + 3 * K + L.pen_len;
    int32_t* q = reinterpret_cast<int32_t*>(smem + L.off_i32);
    s.len = q;
    s.nlen = q + K;
    s.last = q + 2 * K;
    s.nlast = q + 3 * K;
    s.ended = q + 4 * K;
    s.nended = q + 5 * K;
    s.rcount = q + 6 * K;
    s.plen = q + 7 * K;
    s.nblk = q + 9 * K;
    s.sl = reinterpret_cast<ShortEntry*>(smem + L.off_sl);
    s.prefix = L.prefix_in_lds ? reinterpret_cast<int32_t*>(smem + L.off_prefix)
                               : p.prefix + static_cast<int64_t>(b) * 2 * K * p.prefix_cap;
    s.blk = L.blk_in_lds ? reinterpret_cast<int32_t*>(smem + L.off_blk)
                         : p.blocked + static_cast<int64_t>(b) * K * p.prefix_cap;
    s.sig = L.sig_in_lds && !p.step_mode ? reinterpret_cast<uint32_t*>(smem + L.off_sig) : nullptr;
    s.sig_words = L.sig_words;
    s.V = p.V;
    s.sig_shift = L.sig_words == kSigWordsMax ? 19 : 21;
    const bool lists_global = p.constrained && (!L.prefix_in_lds || !L.blk_in_lds);

    const int steps_b = p.step_mode ? 1 : example_steps(p, b);
    // this example's beams (slots past them stay empty) and EOS token
    const int Kb = beams_of(p, b), eos_b = eos_of(p, b);
    const int T_loop = p.step_mode ? 1 : T;
    const int pen_len = L.pen_len;
    // candidates the collector keeps (the beams, or the relaxed pool), and
    // how many of them are the example's
    const int KP = p.pool_mult > 0 ? K * p.pool_mult : K;
    const int Nb = p.pool_mult > 0 ? Kb * p.pool_mult : Kb;
    for (int l = tid; l < pen_len; l += kSelectThreads) {
        const float pl = length_penalty(l, p.alpha);
        s.pen[l] = pl;
        s.inv[l] = 1.0f / pl;
    }
    // Initial state (reference src/decoder.cpp:46-56) or the caller's (:84-103).
    for (int k = tid; k < K; k += kSelectThreads) {
        if (p.step_mode) {
            const int64_t i = static_cast<int64_t>(b) * K + k;
            s.raw[k] = k < Kb ? p.st_raw[i] : -kInf;
            s.len[k] = p.st_len[i];
            s.ended[k] = p.st_fin[i] != 0;
            const int l = p.st_len[i];
            s.last[k] = (p.st_prefix && l >= 1 && l <= p.st_stride) ? p.st_prefix[i * p.st_stride + (l - 1)] : -1;
        } else {
            s.raw[k] = k == 0 ? 0.0f : -kInf;
            s.len[k] = 0;
            s.ended[k] = 0;
            s.last[k] = -1;
        }
        s.plen[k] = 0;
        s.plen[K + k] = 0;
    }
    if (s.sig)
        for (int i = tid; i < 2 * K * s.sig_words; i += kSelectThreads) s.sig[i] = 0u;
    if (tid == 0) {
        st.invalid = 0;
        st.gave_up = 0;
        st.first_bad = 0x7fffffff;
    }
    lds_barrier();

    // Prefetch (the row pass has finished before this kernel: not the
    // overlapped decode): the next step's RowInfo and shortlists sit at fixed
    // addresses (rows (b, t + 1, k) of every slot), so their loads are issued
    // into registers as soon as a step's own are staged, and land while the
    // step runs.
    constexpr int kPf = PF ? kPfRegs : 1;
    uint4 pf_sl[kPf];
    uint4 pf_info = make_uint4(0u, 0u, 0u, 0u);
    bool have_pf = false;
    auto prefetch = [&](int t_next) {
        const int64_t base = (static_cast<int64_t>(b) * T + t_next) * K;
        if (tid < K) pf_info = reinterpret_cast<const uint4*>(p.rowinfo)[base + tid];
        const uint4* src4 = reinterpret_cast<const uint4*>(p.shortlist + base * M);
        const int n4 = K * M / 2;
#pragma unroll
        for (int u = 0; u < kPf; ++u)
            if (tid + u * kSelectThreads < n4) pf_sl[u] = src4[tid + u * kSelectThreads];
    };

    // Pool entry i of the step starting at pool0 (reference src/decoder.cpp:294-306).
    auto put_pool = [&](int64_t i, const Cand& c) {
        if (p.pool_parents) p.pool_parents[i] = c.parent;
        if (p.pool_tokens) p.pool_tokens[i] = c.token;
        if (p.pool_lengths) p.pool_lengths[i] = c.length;
        if (p.pool_scores) p.pool_scores[i] = c.score;
        if (p.pool_raw) p.pool_raw[i] = c.raw;
        if (p.pool_flp) p.pool_flp[i] = static_cast<uint8_t>(c.flp);
    };
    // A padding step (reference src/c_api.cpp:764-781): no token, no parent.
    auto pad_step = [&](int64_t trace0) {
        for (int k = tid; k < K; k += kSelectThreads) {
            if (p.tokens) p.tokens[trace0 + k] = -1;
            if (p.parents) p.parents[trace0 + k] = -1;
            if (p.lengths) p.lengths[trace0 + k] = 0;
            if (p.scores) p.scores[trace0 + k] = -kInf;
            if (p.raw_scores) p.raw_scores[trace0 + k] = -kInf;
            if (p.from_logprob) p.from_logprob[trace0 + k] = 0;
        }
        if (p.pool_mult > 0) {
            const int64_t pool0 = trace0 / K * KP;
            for (int q = tid; q < KP; q += kSelectThreads) put_pool(pool0 + q, dead_cand());
        }
    };

    int cur = 0;
    for (int t = 0; t < T_loop; ++t) {
        const int64_t trace0 = (static_cast<int64_t>(b) * T + t) * K;  // step mode: T == 1
        if (t >= steps_b) {
            pad_step(trace0);
            continue;
        }
        if (tid == 0) {
            st.count = 0;
            st.any_fail = 0;
            st.tau = -kInf;
            st.thr = dead_cand();
        }
        if (p.step_done) {
            // The row pass runs alongside: wait for this step's rows. After a
            // wait gives up, nothing more of the workspace is read: the
            // example's remaining steps are padding and it is reported
            // invalid.
            if (tid == 0 && !st.gave_up && !wait_step_rows(p, b, t)) st.gave_up = 1;
            lds_barrier();
            if (st.gave_up) {
                pad_step(trace0);
                continue;
            }
        }
        const bool coherent = p.step_done != nullptr;
        // Stage the step: row statistics of the rows read, the shortlists,
        // and the n-gram-blocked tokens of each beam.
        for (int k = tid; k < K; k += kSelectThreads) {
            const float praw = s.raw[k];
            const bool live = praw < kInf && praw > -kInf;
            const bool carried = live && eos_b >= 0 && s.ended[k];
            int cnt = -2;
            float bound = -kInf;
            // WIDE: the head of the beam's list, loaded with its RowInfo, every
            // load from a clamped entry (those past the row's count are not
            // used)
            uint32_t elo[kHeadMax], ehi[kHeadMax];
            if (live && !carried) {
                if constexpr (WIDE) {
                    if (H > 0) {
                        const uint32_t* esrc = reinterpret_cast<const uint32_t*>(p.shortlist + (trace0 + k) * M);
#pragma unroll
                        for (int u = 0; u < kHeadMax; ++u) {
                            const int i = u < H ? u : H - 1;
                            if (coherent) {
                                (void)read_tagged(esrc + 2 * i, elo[u], ehi[u]);
                            } else {
                                elo[u] = esrc[2 * i];
                                ehi[u] = esrc[2 * i + 1];
                            }
                        }
                    }
                }
                RowInfo info;
                if (have_pf) {
                    __builtin_memcpy(&info, &pf_info, sizeof(info));  // k == tid
                } else if (!coherent) {
                    info = p.rowinfo[trace0 + k];
                } else {
                    // the two tagged words (count + 2, invalid + 1), both
                    // loads issued before either is waited for
                    const uint32_t* src = reinterpret_cast<const uint32_t*>(p.rowinfo + trace0 + k);
                    uint32_t lo0 = 0, hi0 = 2, lo1 = 0, hi1 = 1;
                    (void)read_tagged(src, lo0, hi0);
                    (void)read_tagged(src + 2, lo1, hi1);
                    if ((hi0 == 0u && !wait_tagged(p, src, lo0, hi0)) || (hi1 == 0u && !wait_tagged(p, src + 2, lo1, hi1))) {
                        atomicOr(&st.gave_up, 1);
                        lo0 = lo1 = 0;
                        hi0 = 2;
                        hi1 = 1;
                    }
                    info.lse = bits_f32(lo0);
                    info.count = static_cast<int32_t>(hi0) - 2;
                    info.bound = bits_f32(lo1);
                    info.invalid = hi1 - 1u;
                }
                if (info.invalid) {
                    atomicOr(&st.invalid, 1u);
                    atomicMin(&st.first_bad, t * K + k);  // steps in order, beams in order within one
                }
                if (p.row_lse && LOGITS) p.row_lse[trace0 + k] = info.lse;
                cnt = M > 0 ? info.count : -1;
                bound = info.bound;
                s.nraw[k] = info.lse;  // the row's logsumexp, kept for a rescan
            }
            if constexpr (WIDE) {
                if (H > 0) {
#pragma unroll
                    for (int u = 0; u < kHeadMax; ++u) {
                        if (u >= H) break;
                        ShortEntry e{-kInf, 0};
                        if (u < cnt) {
                            const uint32_t* esrc = reinterpret_cast<const uint32_t*>(p.shortlist + (trace0 + k) * M + u);
                            if (coherent && ehi[u] == 0u && !wait_tagged(p, esrc, elo[u], ehi[u])) {
                                atomicOr(&st.gave_up, 1);
                                elo[u] = f32_bits(-kInf);
                                ehi[u] = 1;
                            }
                            e = ShortEntry{bits_f32(elo[u]), static_cast<int32_t>(coherent ? ehi[u] - 1u : ehi[u])};
                        }
                        s.sl[k * H + u] = e;
                    }
                }
            }
            s.rcount[k] = cnt;
            s.rbound[k] = bound;
            if (p.constrained && p.ngram > 1) s.nblk[k] = 0;
        }
        if (coherent) {
            // a shortlist is read only as far as its row's count
            lds_barrier();
            if (st.gave_up) {
                pad_step(trace0);
                continue;
            }
        }
        if constexpr (WIDE) {
            // the lists stay where they are
        } else if (have_pf) {
            const int n4 = K * M / 2;
#pragma unroll
            for (int u = 0; u < kPf; ++u) {
                const int q = tid + u * kSelectThreads;
                if (q < n4) {
                    const int k = (2 * q) / M, i = 2 * q - k * M;
                    uint2* dst = reinterpret_cast<uint2*>(s.sl + sl_at(k, i, SL));
                    dst[0] = make_uint2(pf_sl[u].x, pf_sl[u].y);
                    dst[1] = make_uint2(pf_sl[u].z, pf_sl[u].w);
                }
            }
        } else if (M > 0) {
            const ShortEntry* src = p.shortlist + trace0 * M;
            if (!coherent && (M & 1) == 0 && K * M >= kWideBeam * 16) {
                // 16-byte loads (two entries of one row: with M even the rows'
                // shortlists start 16-byte aligned), eight in flight per
                // thread
                const uint4* src4 = reinterpret_cast<const uint4*>(src);
                const int n4 = K * M / 2;
                for (int i0 = tid; i0 < n4; i0 += 8 * kSelectThreads) {
                    uint4 v[8];
#pragma unroll
                    for (int u = 0; u < 8; ++u)
                        if (i0 + u * kSelectThreads < n4) v[u] = src4[i0 + u * kSelectThreads];
#pragma unroll
                    for (int u = 0; u < 8; ++u) {
                        const int q = i0 + u * kSelectThreads;
                        if (q < n4) {
                            const int k = (2 * q) / M, i = 2 * q - k * M;
                            uint2* dst = reinterpret_cast<uint2*>(s.sl + sl_at(k, i, SL));
                            dst[0] = make_uint2(v[u].x, v[u].y);
                            dst[1] = make_uint2(v[u].z, v[u].w);
                        }
                    }
                }
            } else if (coherent) {
                // The entries the row pass wrote (tag token + 1): eight tagged
                // loads per thread issued together (every one made, from a
                // clamped index), then each entry not yet written waited for.
                const uint32_t* src32 = reinterpret_cast<const uint32_t*>(src);
                const int n = K * M;
                for (int i0 = tid; i0 < n; i0 += kStageTags * kSelectThreads) {
                    uint32_t lo[kStageTags], hi[kStageTags];
#pragma unroll
                    for (int u = 0; u < kStageTags; ++u) {
                        const int i = i0 + u * kSelectThreads;
                        (void)read_tagged(src32 + 2 * (i < n ? i : n - 1), lo[u], hi[u]);
                    }
#pragma unroll
                    for (int u = 0; u < kStageTags; ++u) {
                        const int i = i0 + u * kSelectThreads;
                        if (i >= n) continue;
                        const int k = i / M, j = i - k * M;
                        // a word not yet written is waited for only within its
                        // row's count (the rest are never written)
                        if (hi[u] == 0u) {
                            if (j >= s.rcount[k]) continue;
                            if (!wait_tagged(p, src32 + 2 * i, lo[u], hi[u])) {
                                atomicOr(&st.gave_up, 1);
                                hi[u] = 1;
                            }
                        }
                        ShortEntry e;
                        e.lp = bits_f32(lo[u]);
                        e.token = static_cast<int32_t>(hi[u]) - 1;
                        s.sl[SL == M ? i : sl_at(k, j, SL)] = e;
                    }
                }
            } else {
                for (int i = tid; i < K * M; i += kSelectThreads) s.sl[SL == M ? i : sl_at(i / M, i % M, SL)] = src[i];
            }
        }
        // this step's rows are staged: the next step's loads go out now
        if constexpr (PF) {
            have_pf = t + 1 < steps_b;
            if (have_pf) prefetch(t + 1);
        }
        lds_barrier();
        if (coherent && st.gave_up) {
            pad_step(trace0);
            continue;
        }
        if (p.constrained && p.ngram > 1) {
            // n-gram blocking (reference src/decoder.cpp:196-230): for each
            // read beam, the tokens that followed an earlier occurrence of its
            // last n - 1 tokens; one thread per (beam, prefix position), the
            // list in any order (it is only searched)
            // (a decode's prefixes hold at most t tokens at step t)
            const int n = p.ngram, P = p.prefix_cap, Pt = p.step_mode ? P : min(P, t);
            for (int item = tid; item < K * Pt; item += kSelectThreads) {
                const int k = item / Pt, i = item - k * Pt;
                if (s.rcount[k] == -2) continue;
                const PrefixView pre = prefix_of(p, s, b, k, cur);
                if (i + n > pre.len) continue;
                const int tail = pre.len - (n - 1);
                bool same = true;
                for (int j = 0; j < n - 1; ++j) same = same & (pre.tok[i + j] == pre.tok[tail + j]);
                if (same) {
                    const int slot = atomicAdd(&s.nblk[k], 1);
                    s.blk[static_cast<int64_t>(k) * P + slot] = pre.tok[i + n - 1];
                }
            }
            step_barrier(lists_global);
        }
        // a forced step (uniform over the workgroup): no shortlist is used
        const int forced = p.forced ? gload(p.forced, static_cast<int64_t>(b) * T + t) : -1;
        if constexpr (WIDE) {
            // tau: the K-th largest raw of the rows' heads (to its 20 highest
            // bits, rounded down), reached by at least K real candidates
            if (H > 0 && p.use_tau && forced < 0) {
                const int nv = K * H;
                uint32_t* vk = reinterpret_cast<uint32_t*>(s.key);
                for (int q = tid; q < ((nv + 255) & ~255); q += kSelectThreads) {
                    const int k = q >> hsh;
                    vk[q] = q < nv ? ordered_key(q - k * H < s.rcount[k] ? s.raw[k] + s.sl[q].lp : -kInf) : 0u;
                }
                lds_barrier();
                const float tau = key_value(mth_largest_wg<12>(vk, (nv + 255) & ~255, K, s.surv));
                if (tid == 0) {
                    st.tau = tau > -kInf ? tau : -kInf;  // (a key cut below -inf's reads as NaN)
                    st.rcount = 0;
                    st.overflow = 0;
                }
                lds_barrier();
            }
        } else if (p.use_tau && forced < 0) {
            // Lower bounds of the K-th best expanded raw (unconstrained: raw =
            // fl(p + lp), monotone in lp; every beam expanded has the same
            // length, so this step's shortlisted candidates rank by raw).
            // (a) The first K entries of a shortlist are real candidates with
            // raw >= fl(p + lp_K): at least K reach the largest such value.
            if (tid < 64) {
                float best = -kInf;
                for (int k = tid; k < K; k += 64)
                    if (s.rcount[k] >= K) best = fmaxf(best, s.raw[k] + s.sl[sl_at(k, K - 1, SL)].lp);
                best = wave_max_dpp(best);
                if (tid == 0) st.tau = best;
            }
            // (b) Wide beams: the K-th largest raw among the first kTauHead
            // entries of every row: at least K real candidates reach it.
            // Ranked as 64-bit keys (ordered value bits, then the lower index
            // first), two per broadcast read.
            const int nv = K * kTauHead;  // <= 128 (K <= 64 with a shortlist), even
            uint2* vk = reinterpret_cast<uint2*>(s.key);
            float v = -kInf;
            if (K >= kWideBeam && tid < nv) {
                const int k = tid / kTauHead, i = tid - k * kTauHead;
                v = i < s.rcount[k] ? s.raw[k] + s.sl[sl_at(k, i, SL)].lp : -kInf;
                vk[tid] = make_uint2(0xffffffffu - static_cast<uint32_t>(tid), ordered_key(v));
            }
            if (K >= kWideBeam) lds_barrier();  // (a) and the keys are in
            if (K >= kWideBeam && tid < nv) {
                const uint32_t mlo = 0xffffffffu - static_cast<uint32_t>(tid), mhi = ordered_key(v);
                const uint4* w4 = reinterpret_cast<const uint4*>(vk);
                int rank = 0;
                int j2 = 0;
                for (; j2 + 4 <= nv / 2; j2 += 4) {  // four reads in flight
                    uint4 w[4];
#pragma unroll
                    for (int u = 0; u < 4; ++u) w[u] = w4[j2 + u];
#pragma unroll
                    for (int u = 0; u < 4; ++u) {
                        count_above64(rank, mlo, mhi, w[u].x, w[u].y);
                        count_above64(rank, mlo, mhi, w[u].z, w[u].w);
                    }
                }
                for (; j2 < nv / 2; ++j2) {
                    const uint4 w = w4[j2];
                    count_above64(rank, mlo, mhi, w.x, w.y);
                    count_above64(rank, mlo, mhi, w.z, w.w);
                }
                if (rank == K - 1 && v > st.tau) st.tau = v;
            }
            lds_barrier();
        }

        // Carried-forward beams (reference src/decoder.cpp:131-139).
        for (int k = tid; k < K; k += kSelectThreads) {
            const float praw = s.raw[k];
            const bool live = praw < kInf && praw > -kInf;
            if (live && eos_b >= 0 && s.ended[k]) {
                const int l = s.len[k] > 1 ? s.len[k] : 1;
                const int32_t last = s.last[k];
                const Cand c{praw / pen_of(s, pen_len, l, p.alpha), praw, k, is_eos_of(p, b, last) ? last : eos_b, l,
                             0};
                offer(s, st, c);
            }
        }
        if (forced >= 0) {
            // A forced step (reference src/decoder.cpp:125-167,
            // src/kernels_scalar.cpp:16-26): a read beam's one candidate is
            // the forced token, under every check another candidate meets (a
            // finite log-prob, banned tokens, the EOS mask below min_length,
            // n-gram blocking, the repetition penalty). At most K of them
            // join the carried beams: 2K <= sort_cap. (The host refuses forced
            // tokens outside the vocabulary; the bound keeps the read in the
            // row regardless.)
            for (int k = tid; k < K; k += kSelectThreads) {
                if (s.rcount[k] == -2 || forced >= p.V) continue;
                const int64_t row = p.step_mode ? static_cast<int64_t>(b) * K + k : trace0 + k;
                const float x = load_one<DT>(static_cast<const char*>(p.x) +
                                                 static_cast<size_t>(row) * static_cast<size_t>(p.V) * (DT == 0 ? 4 : 2),
                                             forced);
                const float lp = LOGITS ? x - s.nraw[k] : x;
                const int new_len = s.len[k] + 1;
                if (!(lp < kInf) || lp == -kInf || static_masked(p, b, forced, new_len < min_length_of(p, b))) continue;
                if (p.row_mask && gload(p.row_mask, row * p.V + forced)) continue;
                Cand c;
                if (make_cand(p, s, prefix_of(p, s, b, k, cur), k, s.raw[k], inv_of(s, pen_len, new_len, p.alpha),
                              forced, new_len, lp, c))
                    offer(s, st, c);
            }
        }
        // (at most K offers: the first round of shortlisted offers joins them
        // unless the one-pass path below needs the count)
        if (!WIDE && M > 0 && p.use_tau && K >= kWideBeam && forced < 0) end_round(s, st, KP, L.sort_cap);

        // Shortlisted candidates. Unconstrained wide beams: few reach tau, and
        // when they fit the collector beside what it holds, they are offered
        // in one pass without compaction rounds.
        // A shortlist is sorted (log-prob desc), so the entries reaching tau
        // are a prefix of it: one thread per beam measures its prefix, then
        // offers it.
        // (A sum that overflows to -inf is no candidate: the dead sentinel ranks
        // before it. offer() leaves it out, and so does a tau that is finite.)
        constexpr float kLowestRaw = -3.4028234663852886e38f;
        bool one_pass = false;
        if constexpr (WIDE) {
            if (H > 0 && p.use_tau && forced < 0) {
                // Each beam's entries that reach tau go to the collector, as
                // long as they fit: those of its head by the beam's thread,
                // and where the whole head does, the rest of its list by a
                // wavefront, one entry a lane (a thread walking a list of 80
                // took 40 us a step).
                lds_barrier();  // the carried beams are in
                const float tau = fmaxf(st.tau, kLowestRaw);
                const int base = st.count;
                int32_t* const found = s.nlen;  // the beams whose head does not hold them all (free until the selection)
                auto put = [&](int slot, int k, const ShortEntry& e) __attribute__((always_inline)) {
                    const float raw = s.raw[k] + e.lp;
                    const int new_len = s.len[k] + 1;
                    if (slot < L.sort_cap)
                        s.buf[slot] = Cand{raw * inv_of(s, pen_len, new_len, p.alpha), raw, k, e.token, new_len, 1};
                };
                lds_barrier();  // (the count is read before it grows)
                for (int k = tid; k < K; k += kSelectThreads) {
                    const int cnt = s.rcount[k];
                    const float praw = s.raw[k];
                    int n = 0;
                    while (n < cnt && n < H && !(praw + s.sl[k * H + n].lp < tau)) ++n;
                    if (n == 0) continue;
                    if (n == H && cnt > H) found[atomicAdd(&st.rcount, 1)] = k;
                    const int slot0 = atomicAdd(&st.count, n);
                    for (int i = 0; i < n; ++i) put(slot0 + i, k, s.sl[k * H + i]);
                }
                lds_barrier();
                const int nlong = st.rcount, lane = tid & 63;
                for (int q = tid >> 6; q < nlong; q += kSelectThreads / 64) {
                    const int k = found[q], cnt = s.rcount[k];
                    const float praw = s.raw[k];
                    for (int i0 = H; i0 < cnt; i0 += 64) {
                        const bool in = i0 + lane < cnt;
                        const ShortEntry e = list_entry(p, st, trace0 + k, in ? i0 + lane : cnt - 1);
                        const uint64_t reach = __ballot(in && !(praw + e.lp < tau));
                        const int n = static_cast<int>(__popcll(reach));  // a prefix: the list is sorted
                        if (n > 0) {
                            int slot0 = 0;
                            if (lane == 0) slot0 = atomicAdd(&st.count, n);
                            slot0 = __builtin_amdgcn_readfirstlane(slot0);
                            if (lane < n) put(slot0 + lane, k, e);
                        }
                        if (n < 64) break;
                    }
                }
                lds_barrier();
                one_pass = st.count <= L.sort_cap;
                if (!one_pass) {
                    // too many: only the carried beams stay, and the lists
                    // are offered in rounds
                    lds_barrier();
                    if (tid == 0) st.count = base;
                    lds_barrier();
                }
            }
        } else if (M > 0 && p.use_tau && K >= kWideBeam && forced < 0) {
            // (K <= 64 with a shortlist: lane k of wavefront 0 measures beam
            // k's prefix, eight entries a round; a lane scan places the
            // prefixes at consecutive collector slots, and the four
            // wavefronts copy them, lane k for beam k)
            if (tid < 64) {
                const float tau = fmaxf(st.tau, kLowestRaw);
                const int k = tid;
                int n = 0;
                if (k < K) {
                    const float praw = s.raw[k];
                    const int cnt = s.rcount[k];
                    for (;;) {
                        int reach = 0;
#pragma unroll
                        for (int u = 0; u < 8; ++u)
                            reach += (n + u < cnt && !(praw + s.sl[sl_at(k, n + u, SL)].lp < tau)) ? 1 : 0;
                        n += reach;
                        if (reach < 8) break;
                    }
                }
                const int incl = wave_inclusive_sum(n);
                const int total = __builtin_amdgcn_readlane(incl, 63);
                const int base = st.count;
                s.part[k] = base + incl - n;  // beam k's first collector slot
                s.part[64 + k] = n;
                if (tid == 0) st.rcount = base + total <= L.sort_cap ? base + total : -1;
            }
            lds_barrier();
            one_pass = st.rcount >= 0;
            if (one_pass) {
                const int k = tid & 63, w = tid >> 6;
                const int n = k < K ? s.part[64 + k] : 0;
                if (n > w) {
                    const int slot0 = s.part[k];
                    const float praw = s.raw[k];
                    const int new_len = s.len[k] + 1;
                    const float inv = inv_of(s, pen_len, new_len, p.alpha);
                    for (int i = w; i < n; i += 4) {
                        const ShortEntry e = s.sl[sl_at(k, i, SL)];
                        const float raw = praw + e.lp;
                        s.buf[slot0 + i] = Cand{raw * inv, raw, k, e.token, new_len, 1};
                    }
                }
                if (tid == 0) st.count = st.rcount;
            }
        }
        if constexpr (WIDE) {
            // Constrained, stepped, or too many at once: entry i of every list
            // in turn, best first, until no list's entry could be admitted
            // whatever its token (a list is sorted by log-prob, so neither
            // could its later ones, of which one of the same raw may have a
            // lower token; penalties only lower a candidate).
            if (M > 0 && !one_pass && forced < 0) {
                const float tau = st.tau;
                for (int i = 0; i < M; ++i) {
                    if (tid == 0) st.overflow = 0;
                    lds_barrier();
                    for (int k0 = 0; k0 < K; k0 += kSelectThreads) {
                        const int k = k0 + tid;
                        if (k < K && i < s.rcount[k]) {
                            const int64_t row = p.step_mode ? static_cast<int64_t>(b) * K + k : trace0 + k;
                            const ShortEntry e = list_entry(p, st, row, i);
                            const float praw = s.raw[k];
                            const int new_len = s.len[k] + 1;
                            const float inv = inv_of(s, pen_len, new_len, p.alpha);
                            const float raw0 = praw + e.lp;
                            if (!(raw0 < tau) && !before(st.thr, Cand{raw0 * inv, raw0, k, -1, new_len, 1})) {
                                st.overflow = 1;
                                const PrefixView pre = prefix_of(p, s, b, k, cur);
                                Cand c;
                                if (make_cand(p, s, pre, k, praw, inv, e.token, new_len, e.lp, c)) offer(s, st, c);
                            }
                        }
                        end_round(s, st, KP, L.sort_cap);
                    }
                    const int go = st.overflow;
                    lds_barrier();
                    if (go == 0) break;
                }
            }
        } else if (M > 0 && !one_pass && forced < 0) {
            const float tau = st.tau;
            for (int base = 0; base < K * M; base += kSelectThreads) {
                const int item = base + tid;
                if (item < K * M) {
                    const int k = item / M;
                    const int i = item - k * M;
                    if (i < s.rcount[k]) {
                        const ShortEntry e = s.sl[sl_at(k, i, SL)];
                        const float praw = s.raw[k];
                        if (!(praw + e.lp < tau)) {
                            const int new_len = s.len[k] + 1;
                            const PrefixView pre = prefix_of(p, s, b, k, cur);
                            Cand c;
                            if (make_cand(p, s, pre, k, praw, inv_of(s, pen_len, new_len, p.alpha), e.token, new_len,
                                          e.lp, c))
                                offer(s, st, c);
                        }
                    }
                }
                end_round(s, st, KP, L.sort_cap);
            }
        }
        compact(s, st, KP);

        // Exactness: every candidate left out of a row's shortlist has raw <=
        // fl(p + bound); a row passes when the K-th selected candidate ranks
        // strictly before that bound's score and raw.
        for (int k = tid; k < K; k += kSelectThreads) {
            const int cnt = s.rcount[k];
            if (cnt == -2 || forced >= 0) continue;  // a forced step read its rows whole
            bool fail = cnt < 0;
            if (!fail && s.rbound[k] > -kInf) {
                const float X = s.raw[k] + s.rbound[k];
                if (X > -kInf) {
                    const float SX = X * inv_of(s, pen_len, s.len[k] + 1, p.alpha);
                    const Cand kth = st.count >= Nb ? s.buf[Nb - 1] : dead_cand();
                    fail = !((kth.score > SX) || (kth.score == SX && kth.raw > X));
                }
            }
            if (fail) {
                s.rcount[k] = -3;
                atomicOr(&st.any_fail, 1);
            }
        }
        lds_barrier();
        // (Up to kListBeams beams rows rarely fail, and this is kept out of line:
        // in the steps' path, its loads' registers had the steps' own moved to and
        // from the accumulation registers. Select pass of 4 x 98 x 25 x 12106 f32
        // log-probs 855 us, 772 so, of x 64 937 and 877. Beyond, where the first
        // step's row always fails, out of line costs the rescan 5 %.)
        const int any_fail = __builtin_amdgcn_readfirstlane(st.any_fail);
        if (WIDE ? any_fail != 0 : __builtin_expect(any_fail, 0) != 0) {
            // (64 beams at a time: each wavefront finds the same failed rows)
            uint64_t failed = 0;
            for (int k = 0; k < K; ++k) {
                if ((k & 63) == 0) {
                    const int kl = k + (tid & 63);
                    failed = __ballot(kl < K && s.rcount[kl < K ? kl : 0] == -3);
                }
                if (((failed >> (k & 63)) & 1ull) == 0) continue;
                if (tid == 0) atomicAdd(&g_rescanned_rows, 1ull);
                // No threshold yet, and the rows read so far give one: the rows
                // after need one sweep, not two. (4 x 8 x 20 x 12106 f16, n-gram 3
                // and a penalty, every row read in full: 9.2 ms without, 2.6 so.)
                if (__builtin_amdgcn_readfirstlane(st.thr.parent < 0 && st.count >= KP ? 1 : 0)) compact(s, st, KP);
                // drop the row's shortlisted candidates, then offer the whole row
                for (int i = tid; i < st.count; i += kSelectThreads)
                    if (s.buf[i].parent == k && s.buf[i].flp) s.buf[i] = dead_cand();
                lds_barrier();
                const float praw = s.raw[k];
                const int new_len = s.len[k] + 1;
                const int64_t row = p.step_mode ? static_cast<int64_t>(b) * K + k : trace0 + k;
                const PrefixView pre = prefix_of(p, s, b, k, cur);
                rescan_row<DT, LOGITS>(p, s, st, b, k, row, LOGITS ? s.nraw[k] : 0.0f, praw,
                                       inv_of(s, pen_len, new_len, p.alpha), new_len, pre, L.sort_cap, KP);
            }
            compact(s, st, KP);
        }

        if constexpr (WIDE) {
            if (coherent && st.gave_up) {  // an entry never came
                pad_step(trace0);
                continue;
            }
        }

        // Selection (reference src/decoder.cpp:314-350): the example's best Kb.
        const int nsel = st.count < Kb ? st.count : Kb;
        for (int k = tid; k < K; k += kSelectThreads) {
            const Cand c = k < nsel ? s.buf[k] : dead_cand();
            const int64_t o = trace0 + k;
            if (p.tokens) p.tokens[o] = c.token;
            if (p.parents) p.parents[o] = c.parent;
            if (p.lengths) p.lengths[o] = c.length;
            if (p.scores) p.scores[o] = c.score;
            if (p.raw_scores) p.raw_scores[o] = c.raw;
            if (p.from_logprob) p.from_logprob[o] = static_cast<uint8_t>(c.flp);
            s.nraw[k] = c.raw;
            s.nlen[k] = c.length;
            s.nlast[k] = c.token;
            s.nended[k] = c.parent >= 0 ? (s.ended[c.parent] || is_eos_of(p, b, c.token)) : 0;
            if (p.constrained && !p.step_mode) {
                const int nxt = cur ^ 1;
                s.plen[nxt * K + k] =
                    c.parent >= 0 ? s.plen[cur * K + c.parent] + ((c.flp && c.token >= 0) ? 1 : 0) : 0;
            }
        }
        if (p.pool_mult > 0) {
            // the pool: the example's best Nb, the selection first
            const int npool = st.count < Nb ? st.count : Nb;
            const int64_t pool0 = trace0 / K * KP;
            for (int q = tid; q < KP; q += kSelectThreads) put_pool(pool0 + q, q < npool ? s.buf[q] : dead_cand());
        }
        lds_barrier();
        if (p.constrained && !p.step_mode) {
            // each selected beam: its parent's prefix, then its token, and
            // the signature of both (one pass over every beam's positions)
            const int nxt = cur ^ 1;
            const int P = p.prefix_cap;
            const int Pc = min(P, t + 1);  // the new prefixes' length, at most
            const int W = s.sig ? s.sig_words : 0, W4 = W / 4;  // signatures copied 16 bytes an item
            const int PW = Pc > W4 ? Pc : W4;
            for (int item = tid; item < K * PW; item += kSelectThreads) {
                const int k = item / PW, i = item - k * PW;
                const Cand c = k < nsel ? s.buf[k] : dead_cand();
                if (i < W4) {
                    uint4 w = make_uint4(0u, 0u, 0u, 0u);
                    if (c.parent >= 0) {
                        w = reinterpret_cast<const uint4*>(s.sig + (cur * K + c.parent) * W)[i];
                        if (c.flp && c.token >= 0) {
                            auto set = [&](uint32_t h) {
                                if (static_cast<int>(h >> 7) != i) return;
                                const uint32_t m = 1u << (h & 31u);
                                switch ((h >> 5) & 3u) {
                                    case 0: w.x |= m; break;
                                    case 1: w.y |= m; break;
                                    case 2: w.z |= m; break;
                                    default: w.w |= m; break;
                                }
                            };
                            set(sig_bit0(c.token, s.sig_shift));
                            set(sig_bit1(c.token, s.sig_shift));
                        }
                    }
                    reinterpret_cast<uint4*>(s.sig + (nxt * K + k) * W)[i] = w;
                }
                if (i >= Pc || c.parent < 0) continue;
                const int Lp = s.plen[cur * K + c.parent];
                int32_t* dst = s.prefix + (static_cast<int64_t>(nxt) * K + k) * P;
                if (i < Lp) dst[i] = s.prefix[(static_cast<int64_t>(cur) * K + c.parent) * P + i];
                else if (i == Lp && c.flp && c.token >= 0) dst[Lp] = c.token;
            }
            cur = nxt;
        }
        for (int k = tid; k < K; k += kSelectThreads) {
            s.raw[k] = s.nraw[k];
            s.len[k] = s.nlen[k];
            s.last[k] = s.nlast[k];
            s.ended[k] = s.nended[k];
        }
        step_barrier(lists_global);
    }

    if (st.gave_up) {
        // no hypothesis survives an abandoned decode
        for (int k = tid; k < K; k += kSelectThreads) {
            s.raw[k] = -kInf;
            s.len[k] = 0;
        }
        if (tid == 0 && p.fault) __hip_atomic_store(p.fault, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        lds_barrier();
    }
    // Final scores (reference src/decoder.cpp:179-187) and the state (step mode).
    for (int k = tid; k < K; k += kSelectThreads) {
        const int64_t i = static_cast<int64_t>(b) * K + k;
        if (p.final_scores) p.final_scores[i] = s.raw[k] / pen_of(s, pen_len, s.len[k], p.alpha);
        if (p.final_raw) p.final_raw[i] = s.raw[k];
        if (p.final_lengths) p.final_lengths[i] = s.len[k];
        if (p.step_mode) {
            p.st_raw[i] = s.raw[k];
            p.st_len[i] = s.len[k];
            p.st_fin[i] = static_cast<uint8_t>(s.ended[k] != 0);
        }
    }
    // 1: a row the search read holds NaN or +inf; 2: the decode of the
    // example did not complete (an overlapped wait gave up)
    if (tid == 0 && p.invalid) p.invalid[b] = static_cast<uint8_t>(st.gave_up ? 2 : (st.invalid != 0 ? 1 : 0));
    if (tid == 0 && p.first_invalid) p.first_invalid[b] = st.first_bad == 0x7fffffff ? -1 : st.first_bad;
}

// ---------------------------------------------------------------------------
// The narrow select pass: decodes with at most kNarrowMaxK beams and
// shortlists, not the step API and not n = 1 blocking, take one wavefront
// per example, up to kNarrowWaves examples per workgroup (a CU
// beside a persistent row pass takes one workgroup of the select pass at a
// time, so the overlapped decode leaves about B / kNarrowWaves CUs to it,
// the same number on each XCD). Lane k holds beam
// k's state in registers, and a step has no workgroup barrier and few LDS
// round trips:
//   * RowInfo of each read row (lane k) and the shortlists (LDS);
//   * tau, the largest fl(p_k + lp) over the K-th entries of the beams'
//     shortlists (as in the workgroup pass): at least K candidates reach it,
//     so none below it is selected;
//   * the survivors, each beam's entries that reach tau (a prefix of its
//     shortlist: fl(p_k + lp) is monotone in lp), and the carried-forward
//     beams. Up to 64 are ranked in the lanes (the count of candidates before
//     each one); more go through a running list of the best Kb in lanes
//     0 .. Kb - 1 (insertion in order, as keep_best);
//   * the workgroup pass's exactness check; when a row fails it, the
//     selection is redone through the running list from the passing rows'
//     survivors, the carried-forward beams and every token of the failing
//     rows (the candidate set only grows, so rows that passed still pass);
//   * the trace and the next state.
// With constraints (CON: n-gram blocking of n >= 2, a repetition penalty)
// each beam's prefix lives in LDS with two 32 W-bit signatures (two hashed bits
// per token, and per (n - 1)-gram), all double-buffered and copied from the
// parent's at every step (Prefixes); a step lists a beam's n-gram-blocked
// tokens (one lane per prefix position) where its last (n - 1)-gram may have
// occurred before, and every candidate takes make_cand's value (blocked:
// none; in the prefix: lp - log(rep)). Constraints only lower a value, so the
// row pass's bound still covers every token left out, and tau counts on K of
// a row's first K + nblk entries (a blocked token is one entry at most),
// each worth at least lp - log(rep).
// The kept set is the best Kb of the same candidates under the same total
// order as the workgroup pass, so the trace is the same bit for bit.
// Lane j's candidate, wave-uniform.
__device__ __forceinline__ Cand lane_cand(const Cand& c, int j) {
    Cand r;
    r.score = bits_f32(static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(f32_bits(c.score)), j)));
    r.raw = bits_f32(static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(f32_bits(c.raw)), j)));
    r.parent = __builtin_amdgcn_readlane(c.parent, j);
    r.token = __builtin_amdgcn_readlane(c.token, j);
    r.length = __builtin_amdgcn_readlane(c.length, j);
    r.flp = __builtin_amdgcn_readlane(c.flp, j);
    return r;
}

// The value of lane - 1 (row_shr:1 within a 16-lane row; lane 0 keeps x).
__device__ __forceinline__ int from_lane_below(int x) { return __builtin_amdgcn_update_dpp(x, x, 0x111, 0xf, 0xf, false); }

// The running list: lanes [0, n) hold the best candidates so far, best first
// (dead past what it holds); thr is its last entry (wave-uniform). c
// (wave-uniform) goes in when it ranks before thr.
__device__ __forceinline__ void list_insert(Cand& top, Cand& thr, const Cand& c, int n, int lane) {
    if (!before(c, thr)) return;
    const bool above = lane < n && before(top, c);
    const int pos = __popcll(__builtin_amdgcn_ballot_w64(above));  // the list is sorted: a prefix stays
    Cand prev;
    prev.score = bits_f32(static_cast<uint32_t>(from_lane_below(static_cast<int>(f32_bits(top.score)))));
    prev.raw = bits_f32(static_cast<uint32_t>(from_lane_below(static_cast<int>(f32_bits(top.raw)))));
    prev.parent = from_lane_below(top.parent);
    prev.token = from_lane_below(top.token);
    prev.length = from_lane_below(top.length);
    prev.flp = from_lane_below(top.flp);
    if (lane == pos) top = c;
    else if (lane > pos) top = prev;
    thr = lane_cand(top, n - 1);
}

// Offers every lane's candidate where `offer` is set, in lane order.
__device__ __forceinline__ void list_offer(Cand& top, Cand& thr, const Cand& c, bool offer, int n, int lane) {
    uint64_t m = __builtin_amdgcn_ballot_w64(offer && before(c, thr));
    while (m != 0) {
        const int j = __ffsll(static_cast<long long>(m)) - 1;
        m &= m - 1;
        list_insert(top, thr, lane_cand(c, j), n, lane);
    }
}

// The overlapped decode's words of one step for one wavefront: the step's row
// count (lane 0; a hint of when to read), lane k's RowInfo words and the
// first 64 kNarrowTagLoads shortlist words. Every load is made, from a
// clamped address (a load under a branch is waited for inside it), and the
// caller drops what it does not need; a word not yet written has tag 0.
struct TagWords {
    int have;
    uint32_t ilo0, ihi0, ilo1, ihi1;
    uint32_t lo[kNarrowTagLoads], hi[kNarrowTagLoads];
};

__device__ __forceinline__ void issue_tagged(const DecodeParams& p, int b, int t, int lane, TagWords& w) {
    const int K = p.K, M = p.M;
    const int64_t tr0 = (static_cast<int64_t>(b) * p.T + t) * K;
    w.have = 0;
    if (lane == 0)
        w.have = __hip_atomic_load(p.step_done + static_cast<int64_t>(b) * p.T + t, __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_AGENT);
    const uint32_t* info32 = reinterpret_cast<const uint32_t*>(p.rowinfo + tr0 + (lane < K ? lane : 0));
    (void)read_tagged(info32, w.ilo0, w.ihi0);
    (void)read_tagged(info32 + 2, w.ilo1, w.ihi1);
    const uint32_t* sl32 = reinterpret_cast<const uint32_t*>(p.shortlist + tr0 * M);
#pragma unroll
    for (int u = 0; u < kNarrowTagLoads; ++u) {
        const int q = 64 * u + lane;
        (void)read_tagged(sl32 + 2 * (q < K * M ? q : K * M - 1), w.lo[u], w.hi[u]);
    }
}

// The prefixes of a constrained decode's one-wavefront pass, in LDS: per beam
// one record, a signature of its (n - 1)-grams but the last, one of its
// tokens, and the tokens, in two buffers (the step's and the next). A new
// beam's record is its parent's, copied 16 bytes a lane, a record a time (the
// parent is wave-uniform: no per-lane address arithmetic, 5 x 128 tokens in 20
// LDS operations), with the new token's bits set in place after.
struct Prefixes {
    uint32_t* rec;                // [2][K][R]
    int32_t *blk, *nblk, *plen;   // [K][P] n-gram-blocked tokens, their counts, the lengths of beams that list them
    int K, P, W, R, shift, cur;

    __device__ __forceinline__ uint32_t* gram_sig(int k) const { return rec + (cur * K + k) * R; }
    __device__ __forceinline__ uint32_t* token_sig(int k) const { return gram_sig(k) + W; }
    __device__ __forceinline__ int32_t* tokens(int k) const { return reinterpret_cast<int32_t*>(gram_sig(k) + 2 * W); }
    // Whether the two bits of v are set (if not, v was never added).
    __device__ __forceinline__ bool maybe(const uint32_t* sig, int v) const {
        const uint32_t h0 = sig_bit0(v, shift), h1 = sig_bit1(v, shift);
        return (((sig[h0 >> 5] >> (h0 & 31u)) & (sig[h1 >> 5] >> (h1 & 31u))) & 1u) != 0u;
    }
    __device__ __forceinline__ void add(uint32_t* sig, int v) const {
        const uint32_t h0 = sig_bit0(v, shift), h1 = sig_bit1(v, shift);
        atomicOr(&sig[h0 >> 5], 1u << (h0 & 31u));
        atomicOr(&sig[h1 >> 5], 1u << (h1 & 31u));
    }
    // The last n - 1 of beam k's len tokens, hashed (FNV-1a): the first four
    // reads in flight together.
    __device__ __forceinline__ uint32_t tail_hash(int k, int len, int n) const {
        const int32_t* pre = tokens(k);
        const int q0 = len - (n - 1);
        uint32_t h = 0x811C9DC5u;
        int32_t a[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) a[u] = pre[u < n - 1 ? q0 + u : 0];
#pragma unroll
        for (int u = 0; u < 4; ++u)
            if (u < n - 1) h = (h ^ static_cast<uint32_t>(a[u])) * 0x01000193u;
        for (int u = 4; u < n - 1; ++u) h = (h ^ static_cast<uint32_t>(pre[q0 + u])) * 0x01000193u;
        return h;
    }
    // Each listing beam's blocked tokens (plen[k] its length, -1: none): those
    // that followed an earlier occurrence of its last n - 1 tokens; nblk is
    // zero. One lane per (beam k, position i), eight items per lane a round,
    // every read of a round in flight together (beam k's positions at a
    // power-of-two stride >= t: no division).
    __device__ __forceinline__ void list_blocked(int n, int t, int lane) const {
        const int Pt = min(P, t);
        const int ps = Pt > 1 ? 32 - __builtin_clz(static_cast<uint32_t>(Pt - 1)) : 0, total = K << ps;
        for (int j0 = 0; j0 < total; j0 += 8 * 64) {
            int kk[8], ii[8], tl[8];
            bool on[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                const int j = j0 + 64 * u + lane;
                const int jc = j < total ? j : 0;
                kk[u] = jc >> ps;
                ii[u] = jc & ((1 << ps) - 1);
                const int Lk = plen[kk[u]];
                on[u] = j < total && ii[u] + n <= Lk;  // (a beam that lists none: -1)
                tl[u] = on[u] ? Lk - (n - 1) : 0;
            }
            bool same[8] = {true, true, true, true, true, true, true, true};
            for (int q = 0; q < n - 1; ++q) {
                int32_t a[8], c[8];
#pragma unroll
                for (int u = 0; u < 8; ++u) {
                    const int32_t* pre = tokens(kk[u]);
                    a[u] = pre[on[u] ? ii[u] + q : 0];
                    c[u] = pre[on[u] ? tl[u] + q : 0];
                }
#pragma unroll
                for (int u = 0; u < 8; ++u) same[u] = same[u] && a[u] == c[u];
            }
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                if (on[u] && same[u]) {
                    const int slot = atomicAdd(&nblk[kk[u]], 1);
                    blk[kk[u] * P + slot] = tokens(kk[u])[ii[u] + n - 1];
                }
            }
        }
    }
    // The next buffer: beam k takes the record of its parent (par in lane k
    // stride; none: any record, as it is never read), whose prefix holds at
    // most t tokens; then, where `grows` (one lane of a beam k), token v at
    // position at, and where `gram` the (n - 1)-gram hash gh.
    __device__ __forceinline__ void advance(int par, int t, int lane, int stride, int k, bool grows, int v, int at,
                                            bool gram, uint32_t gh, bool grams) {
        const int first = grams ? 0 : W / 4, last = W / 2 + ((min(P, t) + 3) >> 2);
        const uint4* src = reinterpret_cast<const uint4*>(rec + cur * K * R);
        uint4* dst = reinterpret_cast<uint4*>(rec + (cur ^ 1) * K * R);
        for (int c0 = first; c0 < last; c0 += 64) {
            const int c = min(c0 + lane, last - 1);  // (the lanes past the end repeat the last 16 bytes)
            for (int k0 = 0; k0 < K; k0 += 4) {
                uint4 w[4];
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    const int pk = __builtin_amdgcn_readlane(par, min(k0 + u, K - 1) * stride);
                    w[u] = src[(pk >= 0 ? pk : 0) * (R / 4) + c];
                }
#pragma unroll
                for (int u = 0; u < 4; ++u)
                    if (k0 + u < K) dst[(k0 + u) * (R / 4) + c] = w[u];
            }
        }
        wave_sync();
        cur ^= 1;
        if (grows) {
            tokens(k)[at] = v;
            add(token_sig(k), v);
            if (gram) add(gram_sig(k), static_cast<int>(gh));
        }
        wave_sync();
    }
};

// The steps of a decode of at most kGridBeams beams, the candidates in a
// grid: lane (k, j) = k J + j holds entry j of beam k's shortlist (J = K
// unconstrained, where the entries from K on can be selected only on a tie
// of raws, below; as many as 64 lanes hold with constraints) and every lane of
// beam k its state, so that a step moves nothing between lanes but the
// candidates' keys and the selection, through LDS:
//   * the lane's entry and its row's RowInfo, loaded kGridAhead steps ahead
//     (three words, and unconstrained the entry after the lane's; a step's
//     chain is shorter than a load's latency);
//   * tau, the largest K-th entry's raw: candidates below it are not selected;
//   * the keys of the others, packed in LDS, and each one's rank among them:
//     (raw, parent, token) where every beam is expanded (one length: the score
//     is a nondecreasing function of raw), else (score, raw, parent, token);
//   * the selection, by rank, back into every lane of its beam.
// Loads, and stores through views that drop the lanes that have none, are
// never under a branch, so that a wait for a step's words is a wait for the
// operations before them and leaves the later steps' in flight. Bound by the
// chain of LDS round trips and lane operations, 1.3 us a step: 8 x 32 x 4 x
// 32000 f32 42 us (the general step, 3.1 us: 97).
//
// CON: an entry whose token the beam's signature may hold is looked up in the
// prefix by the whole wavefront, a beam whose last (n - 1)-gram may have
// occurred lists its blocked tokens, and a row's entries from J on are left
// out like those of the list's end: the last one held bounds them. 3.0 us a
// step at 128 steps (the general step, its prefixes rebuilt with per-lane
// addresses and searched by one lane a candidate: 6.0): 64 x 128 x 5 x 50257
// f16, n-gram 3 and a penalty, 860 -> 433 us.
// Returns the first step not taken: steps_b, or a step whose rows need a
// full read or whose words never came (gave_up). s: 64 keys of 16 bytes, then
// the selection (kGridBeams of 16 bytes, over the shortlists).
template <bool CON>
__device__ __forceinline__ int grid_entries(int K) { return CON ? 64 / K : K; }

struct GridState {
    float raw;
    int len, last, ended;
};

struct GridWords {
    uint32_t lp, tok;         // the entry (its tag in tok in the overlapped decode)
    uint32_t nlp, ntok;       // the entry after it (unconstrained)
    uint32_t i0, i1, i2, i3;  // the row's RowInfo (tags in i1 and i3)
};

template <int DT, bool LOGITS, bool CON>
__device__ __forceinline__ int grid_steps(const DecodeParams& p, int b, int t, int steps_b, int Kb, int eos_b,
                                          GridState& g, Prefixes& pre, uint4* s_key, const float* s_pen,
                                          const float* s_inv, int pen_len, int lane, bool& any_invalid, int& first_bad,
                                          bool& gave_up) {
    const int K = p.K, T = p.T, M = p.M;
    const int J = grid_entries<CON>(K);
    const int k = lane / J, j = lane - k * J;
    const bool on = k < K;  // (K J lanes of the grid)
    const int kc = on ? k : 0, jc = on ? min(j, M - 1) : 0;
    constexpr int AHEAD = CON ? kGridAheadCon : kGridAhead;
    const bool coherent = p.step_done != nullptr;
    uint2* const s_key2 = reinterpret_cast<uint2*>(s_key);
    uint4* const s_sel = s_key + 64;
    const bool head = on && j == 0;
    // trace views of this example: lanes with nothing to store use an offset
    // past their end
    const int64_t ex = static_cast<int64_t>(b) * T * K;
    const int trace_bytes = 4 * T * K;
    auto view = [&](void* base, int esz) {
        return __builtin_amdgcn_make_buffer_rsrc(static_cast<char*>(base) + ex * esz, 0, base ? trace_bytes / 4 * esz : 0,
                                                 0x00020000);
    };
    const __amdgpu_buffer_rsrc_t v_tok = view(p.tokens, 4), v_par = view(p.parents, 4), v_len = view(p.lengths, 4),
                                 v_score = view(p.scores, 4), v_raw = view(p.raw_scores, 4),
                                 v_flp = view(p.from_logprob, 1), v_lse = view(LOGITS ? p.row_lse : nullptr, 4);

    GridWords ring[AHEAD];
    auto issue = [&](GridWords& w, int tn) __attribute__((always_inline)) {
        const int64_t row = ex + static_cast<int64_t>(tn < steps_b ? tn : steps_b - 1) * K + kc;
        const uint32_t* e = reinterpret_cast<const uint32_t*>(p.shortlist + row * M + jc);
        const uint32_t* r = reinterpret_cast<const uint32_t*>(p.rowinfo + row);
        // (the entry after the last of a list is the next row's, or past the
        // last row's a word of the workspace's counters: read, not used)
        if (coherent) {
            (void)read_tagged(e, w.lp, w.tok);
            if constexpr (!CON) (void)read_tagged(e + 2, w.nlp, w.ntok);
            (void)read_tagged(r, w.i0, w.i1);
            (void)read_tagged(r + 2, w.i2, w.i3);
        } else {
            // (both entries in one load, 8-byte aligned: a load of its own for
            // the second one cost 0.2 us a step)
            struct __attribute__((packed, aligned(8))) Entries { uint32_t lp, tok, nlp, ntok; };
            if constexpr (CON) {
                const uint2 ev = *reinterpret_cast<const uint2*>(e);
                w.lp = ev.x;
                w.tok = ev.y;
            } else {
                const Entries ev = *reinterpret_cast<const Entries*>(e);
                w.lp = ev.lp;
                w.tok = ev.tok;
                w.nlp = ev.nlp;
                w.ntok = ev.ntok;
            }
            const uint4 iv = *reinterpret_cast<const uint4*>(r);
            w.i0 = iv.x;
            w.i1 = iv.y;
            w.i2 = iv.z;
            w.i3 = iv.w;
        }
    };
    // One step from words w; false: not taken (the state is as before it).
    auto step = [&](GridWords& w, int tt) __attribute__((always_inline)) -> bool {
        const bool live = on && g.raw < kInf && g.raw > -kInf;
        const bool carried = live && eos_b >= 0 && g.ended != 0;
        const bool read = live && !carried;
        uint32_t lpw = w.lp, tokw = w.tok, i0 = w.i0, i1 = w.i1, i2 = w.i2, i3 = w.i3;
        uint32_t nlpw = CON ? 0u : w.nlp;
        const bool last_held = !CON && j == J - 1;  // (its next entry is the row's first not held)
        const uint32_t w_ntok = CON ? 1u : w.ntok;
        issue(w, tt + AHEAD);
        if (coherent) {
            // words not yet written (tag 0) are waited for
            const bool miss_info = read && (i1 == 0u || i3 == 0u);
            const bool miss_next = !CON && last_held && w_ntok == 0u;
            if (__builtin_amdgcn_ballot_w64(miss_info || (read && (tokw == 0u || miss_next))) != 0) {
                const int64_t row = ex + static_cast<int64_t>(tt) * K + kc;
                const uint32_t* e = reinterpret_cast<const uint32_t*>(p.shortlist + row * M + jc);
                const uint32_t* r = reinterpret_cast<const uint32_t*>(p.rowinfo + row);
                bool ok = true;
                if (read) {
                    if (i1 == 0u) ok = wait_tagged(p, r, i0, i1);
                    if (ok && i3 == 0u) ok = wait_tagged(p, r + 2, i2, i3);
                    if (ok && tokw == 0u && jc < static_cast<int>(i1) - 2) ok = wait_tagged(p, e, lpw, tokw);
                    uint32_t tag = 1u;
                    if (ok && miss_next && J < static_cast<int>(i1) - 2) ok = wait_tagged(p, e + 2, nlpw, tag);
                }
                if (__builtin_amdgcn_ballot_w64(!ok) != 0) {
                    gave_up = true;
                    return false;
                }
            }
            i1 -= 2u;
            i3 -= 1u;
            tokw -= 1u;
        }
        const int cnt = static_cast<int>(i1);
        const float lse = bits_f32(i0), bound = bits_f32(i2);
        const uint64_t bad_m = __builtin_amdgcn_ballot_w64(read && i3 != 0u);
        const float inv = (tt + 1 < pen_len) ? s_inv[tt + 1] : 1.0f / length_penalty(tt + 1, p.alpha);
        // the lane's candidate
        const float lp = bits_f32(lpw);
        float raw = g.raw + lp;
        int token = static_cast<int>(tokw);
        bool have = read && j < cnt;
        uint32_t tail = 0u;
        // What bounds the entries past those held. (Unconstrained, the first
        // of them: K others of the row have no lower raw, but log-probs that
        // differ can give one raw, and then the lower token comes first.)
        float left = bound;
        if constexpr (CON) {
            left = j == J - 1 && cnt > J && lp > bound ? lp : bound;
        } else {
            bool first_out = j == J - 1 && cnt > J;
            if constexpr (DT != 0) {
                // 16-bit rows often have one value on both sides of K, which
                // would fail the check below. Where the neighbours of that
                // value (2^-9 of a bfloat16 away at least, 2^-12 of a binary16)
                // are further off than the additions round (2^-22 of the
                // sums), the entries of one raw are in the order of their
                // tokens, and K of the row do come first.
                const float value = LOGITS ? lp + lse : lp;
                const float sums = __builtin_fabsf(g.raw) + __builtin_fabsf(lp) + __builtin_fabsf(lse);
                first_out = first_out && !(nlpw == lpw && __builtin_fabsf(value) * (DT == 1 ? 0x1p-12f : 0x1p-9f) > sums * 0x1p-20f);
            }
            if (first_out) left = bits_f32(nlpw);
        }
        if constexpr (CON) {
            // (a read beam's prefix holds tt tokens)
            const int n = p.ngram;
            bool need = false;
            if (n > 1 && tt >= n - 1) {
                tail = pre.tail_hash(kc, tt, n);
                need = tt >= n && read && pre.maybe(pre.gram_sig(kc), static_cast<int>(tail));
            }
            int nb = 0;
            if (__builtin_amdgcn_ballot_w64(need) != 0) {
                if (on && j == 0) {
                    pre.plen[k] = need ? tt : -1;
                    pre.nblk[k] = 0;
                }
                wave_sync();
                pre.list_blocked(n, tt, lane);
                wave_sync();
                if (on) nb = pre.nblk[kc];
                if (have && nb > 0 && in_list(pre.blk + kc * pre.P, nb, token)) have = false;
            }
            // tau: K of a row's first K + nb entries are not blocked, each
            // worth at least its log-prob less the penalty
            const float tau = wave_max_dpp(read && j < cnt && j == K - 1 + nb ? (p.penalise ? g.raw + (lp - p.log_rep) : raw) : -kInf);
            have = have && !(raw < tau);
            if (p.penalise) {
                uint64_t hits = __builtin_amdgcn_ballot_w64(have && pre.maybe(pre.token_sig(kc), token));
                uint64_t in = 0;
                while (hits != 0) {  // (its latency: one round of LDS reads a hit, up to 64 tokens each)
                    const int l = __ffsll(static_cast<long long>(hits)) - 1;
                    hits &= hits - 1;
                    const int v = __builtin_amdgcn_readlane(token, l);
                    const int32_t* a = pre.tokens(__builtin_amdgcn_readlane(kc, l));
                    bool found = false;
                    for (int c0 = 0; c0 < tt; c0 += 64) found = found || a[min(c0 + lane, tt - 1)] == v;
                    if (__builtin_amdgcn_ballot_w64(found) != 0) in |= 1ull << l;
                }
                if ((in >> lane) & 1ull) raw = g.raw + (lp - p.log_rep);
            }
        } else {
            const float tau = wave_max_dpp(have && j == K - 1 ? raw : -kInf);
            have = have && !(raw < tau);
        }
        float score = raw * inv;
        const uint64_t carried_m = __builtin_amdgcn_ballot_w64(carried);
        if (carried_m != 0) {
            const int l = g.len > 1 ? g.len : 1;
            const float pen = l < pen_len ? s_pen[l] : length_penalty(l, p.alpha);
            if (carried && j == 0) {
                raw = g.raw;
                score = g.raw / pen;
                token = is_eos_of(p, b, g.last) ? g.last : eos_b;
                have = true;
            }
        }
        have = have && (score > -kInf || raw > -kInf);  // ranks before the dead sentinel
        const uint64_t m = __builtin_amdgcn_ballot_w64(have);
        const int n = static_cast<int>(__popcll(m));
        const int before_me = static_cast<int>(__builtin_amdgcn_mbcnt_hi(static_cast<uint32_t>(m >> 32),
                                                                         __builtin_amdgcn_mbcnt_lo(static_cast<uint32_t>(m), 0u)));
        const int pos = have ? before_me : n + (lane - before_me);  // the others: zero keys after them
        const uint32_t low = (static_cast<uint32_t>(k) << 24) | (static_cast<uint32_t>(token) & 0xffffffu);
        const uint32_t k0 = have ? 0xffffffffu - low : 0u, k1 = have ? ordered_key(raw) : 0u;
        int rank = 0;
        if (carried_m == 0) {
            s_key2[pos] = make_uint2(k0, k1);
            wave_sync();
            for (int q = 0; q < n; q += 8) {  // (64 keys: the last round stays within them)
                uint4 x[4];
#pragma unroll
                for (int u = 0; u < 4; ++u) x[u] = s_key[q / 2 + u];
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    count_above64(rank, k0, k1, x[u].x, x[u].y);
                    count_above64(rank, k0, k1, x[u].z, x[u].w);
                }
            }
        } else {
            const uint32_t k2 = have ? ordered_key(score) : 0u;
            s_key[pos] = make_uint4(k0, k1, k2, 0u);
            wave_sync();
            for (int q = 0; q < n; q += 4) {
                uint4 x[4];
#pragma unroll
                for (int u = 0; u < 4; ++u) x[u] = s_key[q + u];
#pragma unroll
                for (int u = 0; u < 4; ++u) count_above96(rank, k0, k1, k2, x[u].x, x[u].y, x[u].z);
            }
        }
        const int nsel = n < Kb ? n : Kb;
        const uint32_t meta = static_cast<uint32_t>(carried ? (g.len > 1 ? g.len : 1) : tt + 1) |
                              (carried ? 0u : 0x40000000u) | (g.ended != 0 ? 0x80000000u : 0u);
        if (have && rank < Kb) s_sel[rank] = make_uint4(f32_bits(score), f32_bits(raw), low, meta);
        wave_sync();
        const uint4 mine = s_sel[kc];
        const uint4 kth = s_sel[Kb - 1];
        // Exactness: every candidate left out of a row's list, those past the
        // last entry held too, has raw <= fl(p + left); the row passes when the
        // Kb-th selected candidate ranks strictly before that score and raw.
        const float ks = nsel >= Kb ? bits_f32(kth.x) : -kInf, kr = nsel >= Kb ? bits_f32(kth.y) : -kInf;
        const float X = g.raw + left;
        const float SX = X * inv;
        const bool fail = read && (cnt < 0 || (X > -kInf && !((ks > SX) || (ks == SX && kr > X))));
        if (__builtin_amdgcn_ballot_w64(fail) != 0) return false;
        if (bad_m != 0) {
            any_invalid = true;
            const int at = tt * K + (__ffsll(static_cast<long long>(bad_m)) - 1) / J;  // steps in order, beams in order
            first_bad = at < first_bad ? at : first_bad;
        }
        const bool sel = on && k < nsel;
        const int parent = sel ? static_cast<int>(mine.z >> 24) : -1;
        const int tok = sel ? static_cast<int>(mine.z & 0xffffffu) : -1;
        const int length = sel ? static_cast<int>(mine.w & 0x3fffffffu) : 0;
        const float sc = sel ? bits_f32(mine.x) : -kInf, rw = sel ? bits_f32(mine.y) : -kInf;
        const int flp = sel ? static_cast<int>((mine.w >> 30) & 1u) : 0;
        const int at = head ? (tt * K + k) * 4 : trace_bytes;
        __builtin_amdgcn_raw_buffer_store_b32(static_cast<uint32_t>(tok), v_tok, at, 0, 0);
        __builtin_amdgcn_raw_buffer_store_b32(static_cast<uint32_t>(parent), v_par, at, 0, 0);
        __builtin_amdgcn_raw_buffer_store_b32(static_cast<uint32_t>(length), v_len, at, 0, 0);
        __builtin_amdgcn_raw_buffer_store_b32(f32_bits(sc), v_score, at, 0, 0);
        __builtin_amdgcn_raw_buffer_store_b32(f32_bits(rw), v_raw, at, 0, 0);
        __builtin_amdgcn_raw_buffer_store_b8(static_cast<uint8_t>(flp), v_flp, at / 4, 0, 0);
        if constexpr (LOGITS)
            __builtin_amdgcn_raw_buffer_store_b32(f32_bits(lse), v_lse, read ? at : trace_bytes, 0, 0);
        if constexpr (CON) {
            const uint32_t gh = static_cast<uint32_t>(__shfl(static_cast<int>(tail), (parent >= 0 ? parent : 0) * J));
            pre.advance(parent, tt, lane, J, kc, head && flp != 0, tok, tt, p.ngram > 1 && tt >= p.ngram - 1, gh,
                        p.ngram > 1);
        }
        g.raw = rw;
        g.len = length;
        g.last = tok;
        g.ended = sel && ((mine.w >> 31) != 0u || is_eos_of(p, b, tok)) ? 1 : 0;
        wave_sync();  // the keys' and the selection's LDS may be reused
        return true;
    };
#pragma unroll
    for (int u = 0; u < AHEAD; ++u) issue(ring[u], t + u);
    for (;;) {
#pragma unroll
        for (int u = 0; u < AHEAD; ++u) {
            if (t >= steps_b) return t;
            if (!step(ring[u], t)) return t;
            ++t;
        }
    }
}

template <int DT, bool LOGITS, bool PF, bool CON>
__device__ __forceinline__ void narrow_example(const DecodeParams& p, int pen_len, int wave_bytes, int sig_words,
                                               unsigned char* smem_all) {
    const int K = p.K, T = p.T, M = p.M, V = p.V;
    // up to kNarrowWaves examples per workgroup, one per wavefront, each with
    // its own LDS; the wavefronts never wait for each other
    const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) >> 6);
    const int b = static_cast<int>(blockIdx.x) * (static_cast<int>(blockDim.x) >> 6) + wave;
    const int lane = static_cast<int>(threadIdx.x) & 63;
    if (b >= p.B) return;
    if (p.claimed) {
        int mine = 1;
        if (lane == 0) mine = claim_example(p, b) ? 1 : 0;
        if (__builtin_amdgcn_readfirstlane(mine) == 0) return;
    }
    unsigned char* smem = smem_all + static_cast<size_t>(wave) * wave_bytes;
    uint4* s_key = reinterpret_cast<uint4*>(smem);                   // [64] rank keys
    ShortEntry* s_sl = reinterpret_cast<ShortEntry*>(smem + 1024);  // [K * M], beam k's list at k * M
    Cand* s_cand = reinterpret_cast<Cand*>(smem + 1024 + sizeof(ShortEntry) * static_cast<size_t>(K) * M);  // [64]
    float* s_pen = reinterpret_cast<float*>(s_cand + 64);  // [pen_len]
    float* s_inv = s_pen + pen_len;                        // [pen_len]
    // Constraints (n-gram blocking, repetition penalty): the beams' prefixes
    Prefixes pre;
    pre.K = K;
    pre.P = p.prefix_cap;
    pre.W = sig_words;
    pre.R = 2 * sig_words + ((p.prefix_cap + 3) & ~3);
    pre.shift = 32 - (31 - __builtin_clz(32 * static_cast<uint32_t>(sig_words > 0 ? sig_words : 1)));
    pre.cur = 0;
    pre.rec = reinterpret_cast<uint32_t*>(
        smem + ((1024 + sizeof(ShortEntry) * static_cast<size_t>(K) * M + sizeof(Cand) * 64 +
                 2 * sizeof(float) * static_cast<size_t>(pen_len) + 15) & ~static_cast<size_t>(15)));
    pre.blk = reinterpret_cast<int32_t*>(pre.rec + 2 * K * pre.R);
    pre.nblk = pre.blk + K * pre.P;
    pre.plen = pre.nblk + K;
    for (int l = lane; l < pen_len; l += 64) {
        const float pl = length_penalty(l, p.alpha);
        s_pen[l] = pl;
        s_inv[l] = 1.0f / pl;
    }
    auto pen_at = [&](int l) {
        const int c = l > 1 ? l : 1;
        return c < pen_len ? s_pen[c] : length_penalty(c, p.alpha);
    };
    auto inv_at = [&](int l) {
        const int c = l > 1 ? l : 1;
        return c < pen_len ? s_inv[c] : 1.0f / length_penalty(c, p.alpha);
    };
    const int steps_b = example_steps(p, b);
    const int Kb = beams_of(p, b), eos_b = eos_of(p, b);
    const bool coherent = p.step_done != nullptr;
    const bool beam = lane < K;
    const Cand dead = dead_cand();

    // beam `lane`'s state (reference src/decoder.cpp:46-56)
    float raw = lane == 0 ? 0.0f : -kInf;
    int len = 0, last = -1;
    bool ended = false;
    bool gave_up = false, any_invalid = false;
    int first_bad = 0x7fffffff;

    // the next step's RowInfo and shortlists (all rows written before this
    // kernel started: not the overlapped decode)
    // (four named registers: an array here would be kept in scratch memory)
    static_assert(kNarrowPf == 4, "four prefetch registers");
    uint4 pf0 = make_uint4(0u, 0u, 0u, 0u), pf1 = pf0, pf2 = pf0, pf3 = pf0, pf_info = pf0;
    auto prefetch = [&](int tn) __attribute__((always_inline)) {
        const int64_t base = (static_cast<int64_t>(b) * T + tn) * K;
        if (beam) pf_info = reinterpret_cast<const uint4*>(p.rowinfo)[base + lane];
        const uint4* src4 = reinterpret_cast<const uint4*>(p.shortlist + base * M);
        const int n4 = K * M / 2;
        if (lane < n4) pf0 = src4[lane];
        if (lane + 64 < n4) pf1 = src4[lane + 64];
        if (lane + 128 < n4) pf2 = src4[lane + 128];
        if (lane + 192 < n4) pf3 = src4[lane + 192];
    };
    bool have_pf = false;
    // Decodes of at most kGridBeams beams: their steps go through grid_steps
    // below, and only those that fail its exactness check (and the padding
    // steps) through the general step. (The test knob for waits that give up
    // forces the general step's counted wait.)
    const bool grid = grid_fits(K, M, T) && p.wait_extra == 0;
    if constexpr (PF) {
        have_pf = steps_b > 0 && !grid;
        if (have_pf) prefetch(0);
    }
    // A step's trace is stored during the next step and its row logsumexps
    // later in the same step, just after the next step's loads go out: stores
    // count in vmcnt like loads, so a wait for a loaded value also waits for
    // every store issued before that load.
    int64_t pend_o = -1;  // the pending trace slot (lanes < K), or none
    Cand pend_c = dead;
    bool pend_lse = false;
    int64_t pend_lse_o = 0;
    float pend_lse_v = 0.0f;
    auto flush = [&]() __attribute__((always_inline)) {
        if (pend_lse) p.row_lse[pend_lse_o] = pend_lse_v;
        if (pend_o >= 0) {
            if (p.tokens) p.tokens[pend_o] = pend_c.token;
            if (p.parents) p.parents[pend_o] = pend_c.parent;
            if (p.lengths) p.lengths[pend_o] = pend_c.length;
            if (p.scores) p.scores[pend_o] = pend_c.score;
            if (p.raw_scores) p.raw_scores[pend_o] = pend_c.raw;
            if (p.from_logprob) p.from_logprob[pend_o] = static_cast<uint8_t>(pend_c.flp);
        }
        pend_lse = false;
        pend_o = -1;
    };
    // overlapped decode: a step's words, loaded a step ahead (spec) while the
    // rows are already written, else at the step
    TagWords tw;
    bool spec = false;
    // Constraints: membership of v in beam k's prefix of length lk (the
    // step's buffer; its signature rules most tokens out with two bits), and
    // the value of token v's log-prob lp in beam k's row (make_cand's rules:
    // false when n-gram blocking removes it, the penalty when it repeats).
    auto in_pre = [&](int k, int lk, int v) -> bool {
        return pre.maybe(pre.token_sig(k), v) && in_list(pre.tokens(k), lk, v);
    };
    auto constrain = [&](int k, int lk, int nbk, int v, float lp, float& val) -> bool {
        if (p.ngram > 1 && in_list(pre.blk + k * pre.P, nbk, v)) return false;
        val = (p.penalise && in_pre(k, lk, v)) ? lp - p.log_rep : lp;
        return true;
    };
    if constexpr (CON) {
        // every prefix starts empty
        for (int k = 0; k < K; ++k)
            for (int i = lane; i < 2 * pre.W; i += 64) pre.gram_sig(k)[i] = 0u;
    }
    // A beam's last n - 1 tokens (its tail), hashed (FNV-1a over the tokens),
    // when it has them: the n-gram list is built only where the tail occurred
    // before, and the tail joins the signature when the beam grows.
    uint32_t tail_h = 0u;
    bool tail_v = false;
    const int gJ = grid_entries<CON>(K);
    const int gk = lane / gJ < K ? lane / gJ : 0;  // the beam of this lane in grid_steps
    wave_sync();

    for (int t = 0; t < T; ++t) {
        if (grid && t < steps_b && !gave_up) {
            GridState g{__shfl(raw, gk), __shfl(len, gk), __shfl(last, gk), __shfl(ended ? 1 : 0, gk)};
            t = grid_steps<DT, LOGITS, CON>(p, b, t, steps_b, Kb, eos_b, g, pre, s_key, s_pen, s_inv, pen_len, lane,
                                            any_invalid, first_bad, gave_up);
            const int src = lane < K ? lane * gJ : 0;
            const float raw_k = __shfl(g.raw, src);  // (every lane shuffles)
            const int ended_k = __shfl(g.ended, src);
            len = __shfl(g.len, src);
            last = __shfl(g.last, src);
            raw = beam ? raw_k : -kInf;
            ended = beam && ended_k != 0;
            if (t >= T) break;
        }
        const int64_t trace0 = (static_cast<int64_t>(b) * T + t) * K;
        bool pad = t >= steps_b || gave_up;
        const bool live = beam && raw < kInf && raw > -kInf;
        const bool carried = live && eos_b >= 0 && ended;
        bool read = !pad && live && !carried;
        int cnt = -2;
        float bound = -kInf, lse = 0.0f;
        bool bad = false, lost = false;
        // Overlapped decode: the step's row count (a hint of when to read),
        // the read rows' RowInfo words and the first shortlist words are
        // loaded together, so a step whose rows are all written costs one
        // round trip; a word not yet written (tag 0) is waited for after.
        const uint32_t* sl32 = reinterpret_cast<const uint32_t*>(p.shortlist + trace0 * M);
        uint32_t* const tlo = tw.lo;
        uint32_t* const thi = tw.hi;
        uint32_t& ilo0 = tw.ilo0;
        uint32_t& ihi0 = tw.ihi0;
        uint32_t& ilo1 = tw.ilo1;
        uint32_t& ihi1 = tw.ihi1;
        if (!pad && coherent) {
            // this step's words: loaded during the last step, or now
            if (!spec) issue_tagged(p, b, t, lane, tw);
            spec = false;
            const int need = (t == 0 ? 1 : Kb) + p.wait_extra;
            if (__builtin_amdgcn_readfirstlane(tw.have) < need) {
                int ok = 1;
                if (lane == 0) ok = wait_step_rows(p, b, t) ? 1 : 0;
                if (__builtin_amdgcn_readfirstlane(ok) == 0) {
                    gave_up = pad = true;
                    read = false;
                }
            }
        }
        if (read) {
            RowInfo info;
            if (have_pf) {
                __builtin_memcpy(&info, &pf_info, sizeof(info));
            } else if (!coherent) {
                info = p.rowinfo[trace0 + lane];
            } else {
                // the two tagged words (count + 2, invalid + 1)
                const uint32_t* info32 = reinterpret_cast<const uint32_t*>(p.rowinfo + trace0 + lane);
                bool ok = ihi0 != 0u || wait_tagged(p, info32, ilo0, ihi0);
                ok = ok && (ihi1 != 0u || wait_tagged(p, info32 + 2, ilo1, ihi1));
                if (!ok) {
                    lost = true;
                    ilo0 = ilo1 = 0;
                    ihi0 = 2;
                    ihi1 = 1;
                }
                info.lse = bits_f32(ilo0);
                info.count = static_cast<int32_t>(ihi0) - 2;
                info.bound = bits_f32(ilo1);
                info.invalid = ihi1 - 1u;
            }
            bad = info.invalid != 0;
            if (p.row_lse && LOGITS) {
                pend_lse = true;
                pend_lse_o = trace0 + lane;
                pend_lse_v = info.lse;
            }
            lse = info.lse;
            cnt = M > 0 ? info.count : -1;
            bound = info.bound;
        }
        const uint64_t bad_m = __builtin_amdgcn_ballot_w64(bad);
        if (bad_m != 0) {
            any_invalid = true;
            const int at = t * K + (__ffsll(static_cast<long long>(bad_m)) - 1);  // steps in order, beams in order
            first_bad = at < first_bad ? at : first_bad;
        }
        if (__builtin_amdgcn_ballot_w64(lost) != 0) gave_up = pad = true;
        if (pad) {
            flush();
            // a padding step (reference src/c_api.cpp:764-781): no token, no parent
            if (beam) {
                if (p.tokens) p.tokens[trace0 + lane] = -1;
                if (p.parents) p.parents[trace0 + lane] = -1;
                if (p.lengths) p.lengths[trace0 + lane] = 0;
                if (p.scores) p.scores[trace0 + lane] = -kInf;
                if (p.raw_scores) p.raw_scores[trace0 + lane] = -kInf;
                if (p.from_logprob) p.from_logprob[trace0 + lane] = 0;
            }
            continue;
        }

        // the shortlists into LDS (an entry past its row's count is never read)
        const ShortEntry* src = p.shortlist + trace0 * M;
        if (have_pf) {
            const int n4 = K * M / 2;
            uint4* dst4 = reinterpret_cast<uint4*>(s_sl);
            if (lane < n4) dst4[lane] = pf0;
            if (lane + 64 < n4) dst4[lane + 64] = pf1;
            if (lane + 128 < n4) dst4[lane + 128] = pf2;
            if (lane + 192 < n4) dst4[lane + 192] = pf3;
        } else if (!coherent) {
            for (int q0 = 0; q0 < K * M; q0 += 8 * 64) {
                ShortEntry e[8];
#pragma unroll
                for (int u = 0; u < 8; ++u) {  // clamped: every load in flight at once
                    const int q = q0 + 64 * u + lane;
                    e[u] = src[q < K * M ? q : K * M - 1];
                }
#pragma unroll
                for (int u = 0; u < 8; ++u)
                    if (q0 + 64 * u + lane < K * M) s_sl[q0 + 64 * u + lane] = e[u];
            }
        } else {
            // the entries the row pass wrote (tag token + 1): the first
            // 64 kNarrowTagLoads were loaded with the RowInfo, the rest are
            // loaded now, kNarrowTagLoads per lane in flight; an entry not
            // yet written is waited for
            // (words written are stored as they are; only when one is not
            // is each lane's row count looked up, to wait for the words
            // within it)
            bool lost_e = false;
            for (int q0 = 0; q0 < K * M; q0 += 64 * kNarrowTagLoads) {
                if (q0 > 0) {
#pragma unroll
                    for (int u = 0; u < kNarrowTagLoads; ++u) {
                        const int q = q0 + 64 * u + lane;
                        (void)read_tagged(sl32 + 2 * (q < K * M ? q : K * M - 1), tlo[u], thi[u]);
                    }
                }
                bool missing = false;
#pragma unroll
                for (int u = 0; u < kNarrowTagLoads; ++u) {
                    const int q = q0 + 64 * u + lane;
                    if (q >= K * M) continue;
                    if (thi[u] != 0u) s_sl[q] = ShortEntry{bits_f32(tlo[u]), static_cast<int32_t>(thi[u]) - 1};
                    else missing = true;
                }
                if (__builtin_amdgcn_ballot_w64(missing) != 0) {
#pragma unroll
                    for (int u = 0; u < kNarrowTagLoads; ++u) {
                        const int q = q0 + 64 * u + lane;
                        const int k = q / M;
                        const int cq = __shfl(cnt, k < K ? k : 0);  // every lane: the shuffle reads other lanes
                        if (q >= K * M || q - k * M >= cq || thi[u] != 0u) continue;
                        if (!wait_tagged(p, sl32 + 2 * q, tlo[u], thi[u])) {
                            lost_e = true;
                            thi[u] = 1;
                        }
                        s_sl[q] = ShortEntry{bits_f32(tlo[u]), static_cast<int32_t>(thi[u]) - 1};
                    }
                }
            }
            if (__builtin_amdgcn_ballot_w64(lost_e) != 0) {
                gave_up = true;
                flush();
                if (beam) {
                    if (p.tokens) p.tokens[trace0 + lane] = -1;
                    if (p.parents) p.parents[trace0 + lane] = -1;
                    if (p.lengths) p.lengths[trace0 + lane] = 0;
                    if (p.scores) p.scores[trace0 + lane] = -kInf;
                    if (p.raw_scores) p.raw_scores[trace0 + lane] = -kInf;
                    if (p.from_logprob) p.from_logprob[trace0 + lane] = 0;
                }
                wave_sync();
                continue;
            }
        }
        // this step's rows are staged: the next step's loads go out, then
        // the pending stores (after the loads, so that waiting for the loads
        // never waits for them)
        if constexpr (PF) {
            have_pf = t + 1 < steps_b && !grid;
            if (have_pf) prefetch(t + 1);
        }
        if (coherent && t + 1 < steps_b && !grid) {
            issue_tagged(p, b, t + 1, lane, tw);
            spec = true;
        }
        flush();
        wave_sync();

        // Constraints: each read beam's n-gram-blocked tokens, the tokens
        // that followed an earlier occurrence of its last n - 1 tokens (one
        // lane per (beam, prefix position); a read beam's prefix holds t
        // tokens)
        int nblk = 0;
        if constexpr (CON) {
            bool need = false;
            if (p.ngram > 1) {
                // the tail, and whether it ended an earlier (n - 1)-gram of
                // the prefix (the signature of those; a hit is checked in full)
                const int n = p.ngram;
                tail_v = read && len >= n - 1;
                tail_h = 0u;
                if (tail_v) {
                    tail_h = pre.tail_hash(lane, len, n);
                    need = len >= n && pre.maybe(pre.gram_sig(lane), static_cast<int>(tail_h));
                }
            }
            if (__builtin_amdgcn_ballot_w64(need) != 0) {
                if (beam) {
                    pre.plen[lane] = need ? len : -1;
                    pre.nblk[lane] = 0;
                }
                wave_sync();
                pre.list_blocked(p.ngram, t, lane);
                wave_sync();
                nblk = beam ? pre.nblk[lane] : 0;
            }
        }

        // tau (every expanded beam has the same length, so this step's
        // shortlisted candidates rank by raw): at least K candidates reach it
        const int new_len = len + 1;
        const float inv = inv_at(new_len);
        float tv = -kInf;
        if constexpr (CON) {
            // K of a row's first K + nblk entries are not blocked (a blocked
            // token is at most one entry), each worth at least its log-prob
            // less the penalty
            if (read && cnt >= K + nblk) {
                const float lpk = s_sl[lane * M + (K - 1 + nblk)].lp;
                tv = raw + (p.penalise ? lpk - p.log_rep : lpk);
            }
        } else {
            if (read && cnt >= K) tv = raw + s_sl[lane * M + (K - 1)].lp;
        }
        const float tau = wave_max_dpp(tv);
        // survivors of beam `lane`: a prefix of its shortlist
        int ns = 0;
        if (read) {
            for (;;) {  // four entries a round, their reads in flight together
                float lp4[4];
#pragma unroll
                for (int u = 0; u < 4; ++u) lp4[u] = ns + u < cnt ? s_sl[lane * M + ns + u].lp : -kInf;
                int reach = 0;
                bool on = true;
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    on = on && ns + u < cnt && !(raw + lp4[u] < tau);
                    reach += on ? 1 : 0;
                }
                ns += reach;
                if (reach < 4) break;
            }
        }
        // the carried-forward candidate (reference src/decoder.cpp:131-139)
        Cand carry = dead;
        if (carried) {
            const int l = len > 1 ? len : 1;
            carry = Cand{raw / pen_at(l), raw, lane, is_eos_of(p, b, last) ? last : eos_b, l, 0};
        }
        const uint64_t carried_m = __builtin_amdgcn_ballot_w64(carried);
        const int incl = wave_inclusive_sum(ns);
        const int nsurv = __builtin_amdgcn_readlane(incl, 63);
        const int ncand = nsurv + static_cast<int>(__popcll(carried_m));

        // the selection: the best Kb candidates, lane k holding the k-th
        Cand sel = dead;
        int nsel = 0;
        // survivor s (< nsurv) as a candidate: beam k with s in [off_k,
        // off_k + ns_k). Every lane calls it (the shuffles read other lanes).
        auto survivor = [&](int s) -> Cand {
            int k = 0;
            for (int kk = 1; kk < K; ++kk)
                if (s >= __builtin_amdgcn_readlane(incl - ns, kk)) k = kk;
            const int i = s - __shfl(incl - ns, k);
            const ShortEntry e = s_sl[k * M + i];
            const int lk = __shfl(len, k), nbk = __shfl(nblk, k);
            float val = e.lp;
            bool ok = true;
            if constexpr (CON) ok = constrain(k, lk, nbk, e.token, e.lp, val);
            const float r = __shfl(raw, k) + val;
            const float ik = __shfl(inv, k);
            const int nlk = __shfl(new_len, k);
            return ok ? Cand{r * ik, r, k, e.token, nlk, 1} : dead;
        };
        if (ncand <= 64) {
            // one candidate per lane, ranked by the count of those before it:
            // lane L < nsurv takes survivor L (of beam k, the last beam whose
            // survivors start at or before L), read from the shortlist;
            // lanes [nsurv, ncand) take the carried beams in beam order
            const int excl = incl - ns;
            int k = 0;
            for (int kk = 1; kk < K; ++kk)
                if (lane >= __builtin_amdgcn_readlane(excl, kk)) k = kk;
            const int ik0 = lane - __shfl(excl, k);
            const ShortEntry e = s_sl[k * M + (lane < nsurv ? ik0 : 0)];
            const float rk = __shfl(raw, k), ivk = __shfl(inv, k);
            const int nlk = __shfl(new_len, k);
            Cand c = dead;
            if (lane < nsurv) {
                if constexpr (CON) {
                    // the log-prob in the score field: the constraints are
                    // applied below, one candidate per lane
                    c = Cand{e.lp, 0.0f, k, e.token, nlk, 1};
                } else {
                    const float r = rk + e.lp;
                    c = Cand{r * ivk, r, k, e.token, nlk, 1};
                }
            }
            if (carried_m != 0) {
                // the (lane - nsurv)-th carried beam
                int src = 0, seen = 0;
                for (int kk = 0; kk < K; ++kk) {
                    if (((carried_m >> kk) & 1ull) == 0) continue;
                    if (seen == lane - nsurv) src = kk;
                    ++seen;
                }
                Cand cb;
                cb.score = bits_f32(static_cast<uint32_t>(__shfl(static_cast<int>(f32_bits(carry.score)), src)));
                cb.raw = bits_f32(static_cast<uint32_t>(__shfl(static_cast<int>(f32_bits(carry.raw)), src)));
                cb.parent = __shfl(carry.parent, src);
                cb.token = __shfl(carry.token, src);
                cb.length = __shfl(carry.length, src);
                cb.flp = __shfl(carry.flp, src);
                if (lane >= nsurv && lane < ncand) c = cb;
            }
            if constexpr (CON) {
                const bool surv = lane < nsurv;  // (the carried-forward beams follow the survivors)
                const int k = surv ? c.parent : 0;
                const float pr = __shfl(raw, k), pi = __shfl(inv, k);
                const int lk = __shfl(len, k), nbk = __shfl(nblk, k);
                if (surv) {
                    float val = c.score;
                    if (constrain(k, lk, nbk, c.token, c.score, val)) {
                        const float r = pr + val;
                        c.score = r * pi;
                        c.raw = r;
                    } else {
                        c = dead;
                    }
                }
            }
            const bool valid = lane < ncand && before(c, dead);
            // Its key, larger exactly when the candidate comes earlier in the
            // total order: score, raw, then (parent, token), which no two of
            // a step's candidates share (a carried beam is not expanded), so
            // length and flp never decide. Parents < 64, tokens < 2^24.
            const uint32_t k2 = ordered_key(c.score), k1 = ordered_key(c.raw);
            const uint32_t k0 = 0xffffffffu - ((static_cast<uint32_t>(c.parent) << 24) |
                                               (static_cast<uint32_t>(c.token) & 0xffffffu));
            s_key[lane] = make_uint4(k0, k1, k2, 0u);
            wave_sync();
            int rank = 0;
            int j = 0;
            for (; j + 4 <= ncand; j += 4) {  // four broadcast reads in flight
                uint4 w[4];
#pragma unroll
                for (int u = 0; u < 4; ++u) w[u] = s_key[j + u];
#pragma unroll
                for (int u = 0; u < 4; ++u) count_above96(rank, k0, k1, k2, w[u].x, w[u].y, w[u].z);
            }
            for (; j < ncand; ++j) {
                const uint4 w = s_key[j];
                count_above96(rank, k0, k1, k2, w.x, w.y, w.z);
            }
            nsel = static_cast<int>(__popcll(__builtin_amdgcn_ballot_w64(valid)));
            nsel = nsel < Kb ? nsel : Kb;
            // each selected candidate to the lane of its rank (lanes not
            // selected write lane 63, which holds no selection: Kb <= 16)
            const int to = 4 * ((valid && rank < Kb) ? rank : 63);
            Cand sc;
            sc.score = bits_f32(static_cast<uint32_t>(__builtin_amdgcn_ds_permute(to, static_cast<int>(f32_bits(c.score)))));
            sc.raw = bits_f32(static_cast<uint32_t>(__builtin_amdgcn_ds_permute(to, static_cast<int>(f32_bits(c.raw)))));
            sc.parent = __builtin_amdgcn_ds_permute(to, c.parent);
            sc.token = __builtin_amdgcn_ds_permute(to, c.token);
            sc.length = __builtin_amdgcn_ds_permute(to, c.length);
            sc.flp = __builtin_amdgcn_ds_permute(to, c.flp);
            if (lane < nsel) sel = sc;
            wave_sync();  // the keys' LDS may be reused
        } else {
            Cand thr = dead;
            for (int s0 = 0; s0 < nsurv; s0 += 64) {
                const bool has = s0 + lane < nsurv;
                const Cand c = survivor(has ? s0 + lane : nsurv - 1);
                list_offer(sel, thr, c, has, Kb, lane);
            }
            list_offer(sel, thr, carry, carried, Kb, lane);
            nsel = static_cast<int>(__popcll(__builtin_amdgcn_ballot_w64(lane < Kb && before(sel, dead))));
        }

        // Exactness: every candidate left out of a row's shortlist has raw <=
        // fl(p + bound); a row passes when the Kb-th selected candidate ranks
        // strictly before that bound's score and raw.
        {
            const Cand kth = nsel >= Kb ? lane_cand(sel, Kb - 1) : dead;
            bool fail = false;
            if (read) {
                fail = cnt < 0;
                if (!fail && bound > -kInf) {
                    const float X = raw + bound;
                    if (X > -kInf) {
                        const float SX = X * inv;
                        fail = !((kth.score > SX) || (kth.score == SX && kth.raw > X));
                    }
                }
            }
            const uint64_t fail_m = __builtin_amdgcn_ballot_w64(fail);
            if (fail_m != 0) {
                if (lane == 0) atomicAdd(&g_rescanned_rows, static_cast<unsigned long long>(__popcll(fail_m)));
                // the passing rows' survivors, the carried-forward beams,
                // then every token of each failing row
                Cand thr = dead;
                sel = dead;
                for (int s0 = 0; s0 < nsurv; s0 += 64) {
                    const bool has = s0 + lane < nsurv;
                    const Cand c = survivor(has ? s0 + lane : nsurv - 1);  // parent in [0, K)
                    list_offer(sel, thr, c, has && ((fail_m >> c.parent) & 1ull) == 0, Kb, lane);
                }
                list_offer(sel, thr, carry, carried, Kb, lane);
                const int min_len = min_length_of(p, b);
                const size_t esz = DT == 0 ? 4 : 2;
                for (uint64_t m = fail_m; m != 0; m &= m - 1) {
                    // beam k's values, in every lane
                    const int k = __ffsll(static_cast<long long>(m)) - 1;
                    const float praw = __shfl(raw, k), lse_k = __shfl(lse, k), inv_k = __shfl(inv, k);
                    const int nl = __shfl(new_len, k), lk = __shfl(len, k), nbk = __shfl(nblk, k);
                    const bool mask_eos = nl < min_len;
                    const char* base = static_cast<const char*>(p.x) +
                                       static_cast<size_t>(trace0 + k) * static_cast<size_t>(V) * esz;
                    for (int v0 = 0; v0 < V; v0 += 64 * kNarrowRescanUnroll) {
                        float xs[kNarrowRescanUnroll];
#pragma unroll
                        for (int u = 0; u < kNarrowRescanUnroll; ++u) {
                            const int v = v0 + 64 * u + lane;
                            xs[u] = load_one<DT>(base, v < V ? v : V - 1);
                        }
#pragma unroll
                        for (int u = 0; u < kNarrowRescanUnroll; ++u) {
                            const int v = v0 + 64 * u + lane;
                            const float lp = LOGITS ? xs[u] - lse_k : xs[u];
                            bool ok = v < V && lp < kInf && lp != -kInf;
                            float val = lp;
                            if constexpr (CON) ok = ok && constrain(k, lk, nbk, v, lp, val);
                            const float r = praw + val;
                            const Cand c{r * inv_k, r, k, v, nl, 1};
                            const bool offer = ok && before(c, thr) && !static_masked(p, b, v, mask_eos);
                            list_offer(sel, thr, c, offer, Kb, lane);
                        }
                    }
                }
                nsel = static_cast<int>(__popcll(__builtin_amdgcn_ballot_w64(lane < Kb && before(sel, dead))));
            }
        }

        // Selection (reference src/decoder.cpp:314-350): the trace and the
        // next state of each slot
        const Cand c = lane < nsel ? sel : dead;
        if (beam) {
            pend_o = trace0 + lane;
            pend_c = c;
        }
        if constexpr (CON) {
            // each selected beam: its parent's prefix and signatures, then its token
            const int par = c.parent;
            const int len_par = __shfl(len, par >= 0 ? par : 0);
            const uint32_t gh_par = static_cast<uint32_t>(__shfl(static_cast<int>(tail_h), par >= 0 ? par : 0));
            const int gv_par = __shfl(tail_v ? 1 : 0, par >= 0 ? par : 0);
            const bool grows = beam && par >= 0 && c.flp && c.token >= 0;
            pre.advance(par, t, lane, 1, lane, grows, c.token, len_par, gv_par != 0, gh_par, p.ngram > 1);
        }
        const int parent_ended = __shfl(ended ? 1 : 0, c.parent >= 0 ? c.parent : 0);
        ended = c.parent >= 0 && (parent_ended != 0 || is_eos_of(p, b, c.token));
        raw = c.raw;
        len = c.length;
        last = c.token;
        wave_sync();
        if (grid) flush();
    }
    flush();

    if (gave_up) {
        // no hypothesis survives an abandoned decode
        raw = -kInf;
        len = 0;
        if (lane == 0 && p.fault) __hip_atomic_store(p.fault, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    // Final scores (reference src/decoder.cpp:179-187).
    if (beam) {
        const int64_t i = static_cast<int64_t>(b) * K + lane;
        if (p.final_scores) p.final_scores[i] = raw / pen_at(len);
        if (p.final_raw) p.final_raw[i] = raw;
        if (p.final_lengths) p.final_lengths[i] = len;
    }
    // 1: a row the search read holds NaN or +inf; 2: the decode of the
    // example did not complete (an overlapped wait gave up)
    if (lane == 0 && p.invalid) p.invalid[b] = static_cast<uint8_t>(gave_up ? 2 : (any_invalid ? 1 : 0));
    if (lane == 0 && p.first_invalid) p.first_invalid[b] = first_bad == 0x7fffffff ? -1 : first_bad;
}

// HOLD: as the workgroup pass's (every register of its SIMDs claimed, so no
// row-pass wavefront joins a CU that holds one of its workgroups): its
// workgroups have kNarrowWaves wavefronts, one per SIMD, and those without an
// example, or done with it, wait at the end for the others. (With fewer
// wavefronts the row pass shared the CU, and 16 examples beside a row pass of
// f32 rows made next to no step until it had ended.)
template <int DT, bool LOGITS, bool PF, bool CON, bool HOLD = false>
__global__ __launch_bounds__(64 * kNarrowWaves) void select_narrow_kernel(DecodeParams p, int pen_len, int wave_bytes,
                                                                         int sig_words) {
    if constexpr (HOLD) asm volatile("" ::: "a255");
    extern __shared__ __align__(16) unsigned char smem_all[];
    narrow_example<DT, LOGITS, PF, CON>(p, pen_len, wave_bytes, sig_words, smem_all);
    if constexpr (HOLD) __syncthreads();
}

template <int DT, bool LOGITS, bool PF, bool HOLD = false, bool WIDE = false>
hipError_t launch_select_variant(const DecodeParams& p, const SelectLayout& L, hipStream_t stream) {
    if (L.smem > 64 * 1024) {
        hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&select_kernel<DT, LOGITS, PF, HOLD, WIDE>),
                                           hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(L.smem));
        if (e != hipSuccess) return e;
    }
    KernelTimer timer(kKindSelect, stream);
    hipLaunchKernelGGL((select_kernel<DT, LOGITS, PF, HOLD, WIDE>), dim3(p.B), dim3(kSelectThreads), L.smem, stream, p, L);
    return hipGetLastError();
}

template <int DT, bool LOGITS, bool CON>
hipError_t launch_select_narrow(const DecodeParams& p, hipStream_t stream) {
    const int pen_len = narrow_pen_len(p);
    const int W = narrow_sig_words(p);
    const int wave_bytes = static_cast<int>(narrow_wave_bytes(p, W));
    // prefetch: rows all written before the kernel starts, shortlists as
    // 16-byte pairs of entries within the prefetch registers
    const bool pf = p.step_done == nullptr && (p.M & 1) == 0 && p.K * p.M <= 2 * 64 * kNarrowPf;
    KernelTimer timer(kKindSelect, stream);
    const int per = p.select_hold ? kNarrowWaves : narrow_per_group(p.B);
    const dim3 grid((p.B + per - 1) / per), block(64 * per);
    const size_t smem = static_cast<size_t>(wave_bytes) * per;
    if (smem > 64 * 1024) {
        hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(pf ? &select_narrow_kernel<DT, LOGITS, true, CON>
                                                                           : &select_narrow_kernel<DT, LOGITS, false, CON>),
                                           hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(smem));
        if (e == hipSuccess)
            e = hipFuncSetAttribute(reinterpret_cast<const void*>(&select_narrow_kernel<DT, LOGITS, false, CON, true>),
                                    hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(smem));
        if (e != hipSuccess) return e;
    }
    // beside a row pass of several workgroups per CU it holds its CUs
    // (p.select_hold)
    if (p.select_hold)
        hipLaunchKernelGGL((select_narrow_kernel<DT, LOGITS, false, CON, true>), grid, block, smem, stream, p, pen_len,
                           wave_bytes, W);
    else if (pf)
        hipLaunchKernelGGL((select_narrow_kernel<DT, LOGITS, true, CON>), grid, block, smem, stream, p, pen_len,
                           wave_bytes, W);
    else
        hipLaunchKernelGGL((select_narrow_kernel<DT, LOGITS, false, CON>), grid, block, smem, stream, p, pen_len,
                           wave_bytes, W);
    return hipGetLastError();
}

template <int DT, bool LOGITS>
hipError_t launch_select_typed(const DecodeParams& p, const SelectLayout& L, hipStream_t stream) {
    if (select_narrow(p))
        return p.constrained ? launch_select_narrow<DT, LOGITS, true>(p, stream)
                             : launch_select_narrow<DT, LOGITS, false>(p, stream);
    // (wide: one instantiation, which holds its CUs whether or not a row pass
    // runs beside it)
    if (p.K > kListBeams) return launch_select_variant<DT, LOGITS, false, true, true>(p, L, stream);
    if (p.select_hold) return launch_select_variant<DT, LOGITS, false, true>(p, L, stream);
    return prefetch_fits(p) ? launch_select_variant<DT, LOGITS, true>(p, L, stream)
                            : launch_select_variant<DT, LOGITS, false>(p, L, stream);
}

hipError_t counter(unsigned long long& symbol, int reset, unsigned long long* value) {
    if (reset) {
        const unsigned long long zero = 0;
        return hipMemcpyToSymbol(HIP_SYMBOL(symbol), &zero, sizeof(zero));
    }
    return hipMemcpyFromSymbol(value, HIP_SYMBOL(symbol), sizeof(*value));
}

}  // namespace

template <int DT>
hipError_t launch_select_dtype(const DecodeParams& p, const SelectLayout& L, hipStream_t stream) {
    return p.from_logits ? launch_select_typed<DT, true>(p, L, stream) : launch_select_typed<DT, false>(p, L, stream);
}

template <int DT>
hipError_t rescan_counter_dtype(int reset, unsigned long long* value) {
    return counter(g_rescanned_rows, reset, value);
}

template <int DT>
hipError_t wait_timeout_counter_dtype(int reset, unsigned long long* value) {
    return counter(g_wait_timeouts, reset, value);
}

}  // namespace dbs_hip
