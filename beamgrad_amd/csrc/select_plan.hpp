// SPDX-License-Identifier: MIT
//
// Sizes and plans of the select pass, shared by its kernels
// (select_kernels.hpp) and the host code that lays out their memory
// (select.hip).
#pragma once

#include "engine.hpp"

namespace dbs_hip {

constexpr int kStageTags = 8;  // tagged shortlist loads per thread in flight (workgroup pass, overlapped decode)

constexpr int kRescanTokens = 3072;  // tokens of one rescanned row gathered before falling back (12 KB)
constexpr int kRescanPerThread = 32;
constexpr int kTauHead = 2;       // entries per row behind the second tau bound
constexpr int kWideBeam = 16;     // beams from which the wide-beam paths pay off
constexpr int kListBeams = 64;    // beams up to which a step's shortlists are staged in LDS, each longer than the beams
constexpr int kHeads = 2048;      // heads of the lists kept in LDS beyond that (two per beam at the most beams, 1024)
constexpr int kWidePenCap = 1024; // lengths with a penalty in LDS there (larger ones are computed)
constexpr int kPfRegs = 12;       // 16-byte prefetch registers per thread (K * M <= 6144)
constexpr int kSigWordsMax = 256;  // words of a beam's prefix signature (8192 bits; 2048 when LDS is short)
constexpr int kScoreFilterMaxK = 32;  // beams up to which a rank compaction first ranks by score alone

// Collector sizes up to this are compacted by a parallel rank (larger ones by
// the bitonic sort).
constexpr int kRankMax = kSelectThreads;
constexpr int kWideRank = 4;  // candidates per thread of the rank compaction beyond kListBeams beams

// The narrow select pass (select_kernels.hpp).
constexpr int kNarrowMaxK = 16;       // the running list lives in one 16-lane DPP row
constexpr int kGridBeams = 8;         // beams whose candidates fit one wavefront's lanes, K of each at least (grid_steps)
constexpr int kGridAhead = 4;         // steps its words are loaded ahead
constexpr int kGridAheadCon = 2;      // with constraints (longer steps, and twice the step's code instead of four times)
constexpr int kNarrowPf = 4;          // 16-byte prefetch registers per lane (K * M <= 512)
constexpr int kNarrowPenCap = 1024;   // lengths with a penalty in LDS (larger ones are computed)
constexpr int kNarrowRescanUnroll = 16;
constexpr int kNarrowTagLoads = 4;    // tagged shortlist loads per lane in flight (overlapped decode)
constexpr int kNarrowWaves = 4;       // examples (wavefronts) per workgroup, at most: one workgroup per CU
constexpr int kXcds = 8;              // MI355X: 8 XCDs of 32 CUs
constexpr int kNarrowWaveLds = 24576; // LDS per wavefront, at most (else the workgroup pass)

// Whether a decode's steps go through the grid of candidates: lists at least
// as long as the beams, and a trace whose byte offsets (an example's, past the
// end included) fit in 31 bits.
constexpr bool grid_fits(int K, int M, int T) {
    return K <= kGridBeams && M >= K && static_cast<int64_t>(T) * K < (1 << 29);
}
static_assert(grid_fits(8, 24, 1 << 25) && !grid_fits(9, 24, 1) && !grid_fits(4, 3, 1), "beams and lists");
static_assert(!grid_fits(8, 24, 1 << 26) && !grid_fits(1, 24, 1 << 29) && grid_fits(1, 24, (1 << 29) - 1), "offsets");

// The prefetch needs the row pass finished before the select pass starts (not
// the overlapped decode, whose rows land while it runs) and a step's
// shortlists within the prefetch registers, as 16-byte pairs of entries.
inline bool prefetch_fits(const DecodeParams& p) {
    return p.step_done == nullptr && !p.step_mode && p.M > 0 && (p.M & 1) == 0 && p.K <= kSelectThreads &&
           p.K * p.M <= 2 * kPfRegs * kSelectThreads;
}

// Workgroups of the narrow pass: a multiple of kXcds (workgroups are dealt
// to the XCDs in turn, and a persistent row pass of CUs - groups workgroups
// leaves groups / kXcds CUs free on each), up to kNarrowWaves examples each.
inline int narrow_groups(int B) { return kXcds * ((B + kXcds * kNarrowWaves - 1) / (kXcds * kNarrowWaves)); }
inline int narrow_per_group(int B) {
    const int g = narrow_groups(B);
    return (B + g - 1) / g;
}

inline int narrow_pen_len(const DecodeParams& p) { return p.T + 2 < kNarrowPenCap ? p.T + 2 : kNarrowPenCap; }

// One wavefront's LDS: rank keys, shortlists, candidates, penalty tables;
// with constraints also signatures of W words per beam, prefixes, n-gram
// lists and per-beam state (the kernel's layout).
inline size_t narrow_wave_bytes(const DecodeParams& p, int W) {
    const size_t K = static_cast<size_t>(p.K), P = static_cast<size_t>(p.prefix_cap);
    size_t n = 1024 + sizeof(ShortEntry) * K * static_cast<size_t>(p.M) + sizeof(Cand) * 64 +
               2 * sizeof(float) * static_cast<size_t>(narrow_pen_len(p));
    n = (n + 15) & ~static_cast<size_t>(15);
    if (p.constrained) {
        const size_t P4 = (P + 3) & ~static_cast<size_t>(3);
        n += sizeof(uint32_t) * 4 * K * static_cast<size_t>(W) + sizeof(int32_t) * (2 * K * P4 + K * P + 2 * K);
    }
    return (n + 15) & ~static_cast<size_t>(15);
}

// Signature words per beam of a constrained decode (the most of 64, 32, 16
// that fit one wavefront's LDS), else 0; 0 for an unconstrained one.
inline int narrow_sig_words(const DecodeParams& p) {
    if (!p.constrained) return 0;
    for (int W = 64; W >= 16; W /= 2)
        if (narrow_wave_bytes(p, W) <= static_cast<size_t>(kNarrowWaveLds)) return W;
    return 0;
}

}  // namespace dbs_hip
