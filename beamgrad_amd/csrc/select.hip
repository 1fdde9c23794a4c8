// SPDX-License-Identifier: MIT
//
// The select pass: which kernel a decode takes, the LDS plan of the workgroup
// kernel, and the dispatch to the input type's kernels (select_f32.hip,
// select_f16.hip, select_bf16.hip).
#include <hip/hip_runtime.h>

#include <atomic>

#include "select_plan.hpp"

namespace dbs_hip {

std::atomic<int> g_select_kind{0};

bool select_narrow(const DecodeParams& p) {
    if (g_select_kind.load(std::memory_order_relaxed) == 1) return false;
    if (p.step_mode || p.forced || p.pool_mult > 0 || p.M <= 0 || p.K > kNarrowMaxK || p.V > (1 << 24)) return false;
    // constrained: n-gram blocking of n >= 2 and/or a repetition penalty
    // (n = 1 blocking would drop most of a long prefix's shortlist entries)
    if (p.constrained) return p.ngram != 1 && narrow_sig_words(p) > 0;
    return p.use_tau && narrow_wave_bytes(p, 0) <= static_cast<size_t>(kNarrowWaveLds);
}

int select_reserve_cus(const DecodeParams& p, bool persistent) {
    if (!select_narrow(p)) return p.B;
    return persistent ? narrow_groups(p.B) : (p.B + kNarrowWaves - 1) / kNarrowWaves;
}

SelectLayout select_layout(int B, int T, int K, int M, bool constrained, bool step_mode, int prefix_cap, int keep) {
    (void)B;
    SelectLayout L{};
    int sc = 1;
    while (sc < (keep > K ? keep : K) + 2 * kSelectThreads) sc <<= 1;
    L.sort_cap = sc;
    const bool wide = K > kListBeams;
    L.pen_len = step_mode ? 0 : (wide && T + 2 > kWidePenCap ? kWidePenCap : T + 2);
    auto align = [](size_t x) { return (x + 15) & ~static_cast<size_t>(15); };
    size_t off = 0;
    L.off_buf = off;
    off = align(off + sizeof(Cand) * static_cast<size_t>(sc));
    L.off_rbuf = off;
    if (!wide) off = align(off + sizeof(int32_t) * kRescanTokens);
    L.off_key = off;
    off = align(off + sizeof(uint4) * (wide ? kWideRank : 2) * kRankMax + sizeof(int32_t) * (kSelectThreads + 64 + 4) +
                (wide ? sizeof(int32_t) * kWideRank * kRankMax : 0));
    L.off_f32 = off;
    off = align(off + sizeof(float) * (3 * static_cast<size_t>(K) + 2 * static_cast<size_t>(L.pen_len)));
    L.off_i32 = off;
    off = align(off + sizeof(int32_t) * 10 * static_cast<size_t>(K));
    L.off_sl = off;
    // (more than kListBeams beams: the heads of their lists, shared with the
    // rescan buffer, which is used after them)
    if (wide) {
        static_assert(sizeof(ShortEntry) * kHeads >= sizeof(int32_t) * kRescanTokens, "the rescan buffer fits the heads");
        L.off_rbuf = off;
        off = align(off + sizeof(ShortEntry) * kHeads);
    } else {
        off = align(off + sizeof(ShortEntry) * static_cast<size_t>(K) * static_cast<size_t>(K >= kWideBeam ? M + 1 : M));
    }
    const size_t prefix_bytes = sizeof(int32_t) * 2 * static_cast<size_t>(K) * static_cast<size_t>(prefix_cap);
    const size_t blk_bytes = sizeof(int32_t) * static_cast<size_t>(K) * static_cast<size_t>(prefix_cap);
    const size_t budget = 150 * 1024;
    L.prefix_in_lds = 0;
    L.blk_in_lds = 0;
    if (constrained && !step_mode && off + prefix_bytes <= budget) {
        L.prefix_in_lds = 1;
        L.off_prefix = off;
        off = align(off + prefix_bytes);
    }
    if (constrained && off + blk_bytes <= budget) {
        L.blk_in_lds = 1;
        L.off_blk = off;
        off = align(off + blk_bytes);
    }
    L.sig_in_lds = 0;
    L.sig_words = 0;
    for (int words = kSigWordsMax; words >= kSigWordsMax / 4 && !L.sig_in_lds; words /= 4) {
        const size_t sig_bytes = sizeof(uint32_t) * 2 * static_cast<size_t>(K) * words;
        if (L.prefix_in_lds && off + sig_bytes <= budget) {
            L.sig_in_lds = 1;
            L.sig_words = words;
            L.off_sig = off;
            off = align(off + sig_bytes);
        }
    }
    L.smem = off;
    return L;
}

hipError_t launch_select(const DecodeParams& p, const SelectLayout& L, hipStream_t stream) {
    switch (p.dtype) {
        case 0: return launch_select_dtype<0>(p, L, stream);
        case 1: return launch_select_dtype<1>(p, L, stream);
        default: return launch_select_dtype<2>(p, L, stream);
    }
}

namespace {

// The kernels of each input type count for themselves (one translation unit
// each): the sum, or every one reset.
template <class F0, class F1, class F2>
hipError_t summed(F0 f0, F1 f1, F2 f2, int reset, unsigned long long* value) {
    unsigned long long v[3] = {0, 0, 0};
    hipError_t e = f0(reset, &v[0]);
    if (e == hipSuccess) e = f1(reset, &v[1]);
    if (e == hipSuccess) e = f2(reset, &v[2]);
    if (e == hipSuccess && !reset) *value = v[0] + v[1] + v[2];
    return e;
}

}  // namespace

hipError_t wait_timeout_counter(int reset, unsigned long long* value) {
    return summed(wait_timeout_counter_dtype<0>, wait_timeout_counter_dtype<1>, wait_timeout_counter_dtype<2>, reset,
                  value);
}

hipError_t rescan_counter(int reset, unsigned long long* value) {
    return summed(rescan_counter_dtype<0>, rescan_counter_dtype<1>, rescan_counter_dtype<2>, reset, value);
}

}  // namespace dbs_hip
