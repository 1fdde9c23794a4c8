// SPDX-License-Identifier: MIT
//
// Row pass for short rows (up to kShortRow entries), logits or log-probs of any
// type and alignment: one wavefront a row, four rows a workgroup, no barrier.
//
// Lane l holds entries v = 64 i + l of the row in registers (read once), so the
// reference's fold lane v mod 256 (src/kernels_scalar.cpp:48-66) is register
// group i mod 4 of one lane, whose terms are added in order from the
// registers; its 256 lane maxima give the maximum and theta, the M-th largest
// (to 20 bits): at least M entries reach it. The survivors are listed by
// ballot in LDS, ranked and published by the wavefront.
//
// What bounds it: the operations of a row (25 an entry for a term, 5 for the
// rest, and some 600 for theta, the logsumexp and the ranks), where a workgroup
// a row spends most of them four times over and waits at its barriers. 64 x 64 x
// 8 rows, log-probs against the one-read pass: f16 of 2000 202 -> 54 us, f32 of
// 3000 190 -> 70, f16 of 6000 234 -> 127; logits against the stream pass: f32 of
// 1000 245 -> 60, f16 of 2000 325 -> 81, bf16 of 6000 400 -> 190. Of 8000 the
// registers leave three wavefronts a SIMD and it gains little (32 x 64 x 8:
// f16 logits 200 -> 163, f32 log-probs 95 -> 113).
#include <hip/hip_runtime.h>

#include "row_helpers.hpp"

namespace dbs_hip {

namespace {

constexpr int kShortThreads = 256;
constexpr int kShortRows = kShortThreads / 64;  // rows per workgroup
constexpr int kShortSurvivors = 256;            // survivors, at most (else the row is read in full)
constexpr int kShortRow = 6144;                 // entries, at most: 96 registers a lane

// The lanes of a ballot before this one.
__device__ __forceinline__ int below(uint64_t m) {
    return static_cast<int>(
        __builtin_amdgcn_mbcnt_hi(static_cast<uint32_t>(m >> 32), __builtin_amdgcn_mbcnt_lo(static_cast<uint32_t>(m), 0u)));
}

// C: entries a lane, a multiple of 8.
template <int DT, bool LOGITS, int C>
__global__ __launch_bounds__(kShortThreads) __attribute__((amdgpu_waves_per_eu(C > 64 ? 2 : 4))) void row_short_kernel(
    DecodeParams p, int64_t rows) {
    __shared__ __align__(16) uint64_t s_keys[kShortRows][kShortSurvivors];
    __shared__ float s_xs[kShortRows][kShortSurvivors];
    constexpr int esz = DT == 0 ? 4 : 2;
    const int lane = static_cast<int>(threadIdx.x) & 63;
    const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) >> 6);
    uint64_t* const s_key = s_keys[wave];
    float* const s_x = s_xs[wave];
    float* const s_acc = reinterpret_cast<float*>(s_key);  // (the sums are read before the survivors are written)
    const int V = p.V, M = p.M;

    const int64_t q = static_cast<int64_t>(blockIdx.x) * kShortRows + wave;
    if (q >= rows) return;
    const int64_t r = row_of_ticket(p, q);
    int b, new_len;
    if (!row_is_read(p, r, b, new_len)) return;

    const uintptr_t a0 = reinterpret_cast<uintptr_t>(p.x) + static_cast<uintptr_t>(r) * static_cast<uintptr_t>(V) * esz;
    const int lead = static_cast<int>(a0 & 3u), bytes = lead + V * esz;
    const __amdgpu_buffer_rsrc_t rs =
        __builtin_amdgcn_make_buffer_rsrc(reinterpret_cast<void*>(a0 - lead), 0, bytes, 0x00020000);
    uint32_t h[C];
#pragma unroll
    for (int i = 0; i < C; ++i)  // (the scalar offset stays within the view; past it loads return zeros)
        h[i] = load_raw<DT>(rs, lead + lane * esz, min(64 * i * esz, bytes));
    float x[C];
#pragma unroll
    for (int i = 0; i < C; ++i) x[i] = raw_value<DT>(h[i]);
#pragma unroll
    for (int i = 0; i < C; ++i)
        if (64 * (i + 1) > V && 64 * i + lane >= V) x[i] = -kInf;

    // The 256 lane maxima and the NaN / +inf flag; a row with NaN or +inf:
    // the maximum of the entries below +inf.
    bool bad = false;
#pragma unroll
    for (int i = 0; i < C; ++i) bad = bad || __builtin_amdgcn_classf(x[i], 0x203);  // sNaN, qNaN, +inf
    const bool any_bad = __builtin_amdgcn_ballot_w64(bad) != 0;
    float top[4] = {-kInf, -kInf, -kInf, -kInf};
    if (any_bad) {
#pragma unroll
        for (int i = 0; i < C; ++i)
            if (x[i] < kInf && x[i] > top[i % 4]) top[i % 4] = x[i];
    } else {
#pragma unroll
        for (int i = 0; i < C; i += 8)
#pragma unroll
            for (int e = 0; e < 4; ++e) top[e] = max3(top[e], x[i + e], x[i + 4 + e]);
    }
    uint32_t k4[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) k4[e] = ordered_key(top[e]);
    const float m = wave_max_dpp(key_value(max(max(k4[0], k4[1]), max(k4[2], k4[3]))));
    const bool do_lse = m > -kInf;
    const bool listing = M > 0 && !any_bad;  // (a flagged row keeps no shortlist)
    float theta = -kInf;
    if (listing) theta = list_threshold<DT>(key_value(mth_largest_key<32, 12>(k4, M)));

    float lse = 0.0f;
    if constexpr (LOGITS) {
        lse = -kInf;
        if (do_lse) {
            float acc[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int i = 0; i < C; ++i) acc[i % 4] = acc[i % 4] + exp_term(m, x[i]);
#pragma unroll
            for (int e = 0; e < 4; ++e) s_acc[64 * e + lane] = acc[e];
            wave_sync();
            const float4 a4 = reinterpret_cast<const float4*>(s_acc)[lane];
            wave_sync();
            float a[4] = {a4.x, a4.y, a4.z, a4.w};
            lse = logsumexp_from(m, lane_tree_sum(a, lane));
        }
    }

    int n = 0;
    if (listing) {
#pragma unroll
        for (int i = 0; i < C; ++i) {
            const bool on = x[i] >= theta;  // (entries past the row hold -inf)
            const uint64_t at = __builtin_amdgcn_ballot_w64(on);
            if (at == 0) continue;
            const int slot = n + below(at);
            if (on && slot < kShortSurvivors) {
                s_key[slot] = survivor_key(x[i], 64 * i + lane);
                s_x[slot] = x[i];
            }
            n += static_cast<int>(__popcll(at));
        }
        // the masked ones leave the list (all at once: their mask bytes are
        // loaded from memory)
        const bool mask_eos = new_len < min_length_of(p, b);
        if (n <= kShortSurvivors && (p.banned || p.banned_pe || mask_eos)) {
            wave_sync();
            int kept = 0;
            for (int i0 = 0; i0 < n; i0 += 64) {
                const int i = i0 + lane < n ? i0 + lane : n - 1;
                const uint64_t key = s_key[i];
                const float xi = s_x[i];
                const int v = static_cast<int>(0xffffffffu - static_cast<uint32_t>(key & 0xffffffffu));
                const bool on = i0 + lane < n && !static_masked(p, b, v, mask_eos);
                const uint64_t at = __builtin_amdgcn_ballot_w64(on);
                wave_sync();
                if (on) {  // (at or before the entries read)
                    s_key[kept + below(at)] = key;
                    s_x[kept + below(at)] = xi;
                }
                kept += static_cast<int>(__popcll(at));
                wave_sync();
            }
            n = kept;
        }
    }
    if (M > 0 && (!listing || n > kShortSurvivors)) n = kSurvivorCap + 1;  // (no shortlist)
    wave_sync();
    finish_row_wave<LOGITS>(p, r, lse, list_bound<DT>(theta), any_bad, s_key, s_x, n, lane);
}

template <int DT, bool LOGITS, int C>
hipError_t launch_short(const DecodeParams& p, int64_t rows, hipStream_t stream) {
    const int64_t grid = (rows + kShortRows - 1) / kShortRows;
    hipLaunchKernelGGL((row_short_kernel<DT, LOGITS, C>), dim3(static_cast<unsigned>(grid)), dim3(kShortThreads), 0, stream,
                       p, rows);
    return hipGetLastError();
}

template <int DT, bool LOGITS>
hipError_t launch_short_typed(const DecodeParams& p, int64_t rows, hipStream_t stream) {
    if (p.V <= 512) return launch_short<DT, LOGITS, 8>(p, rows, stream);
    if (p.V <= 1024) return launch_short<DT, LOGITS, 16>(p, rows, stream);
    if (p.V <= 2048) return launch_short<DT, LOGITS, 32>(p, rows, stream);
    if (p.V <= 3072) return launch_short<DT, LOGITS, 48>(p, rows, stream);
    if (p.V <= 4096) return launch_short<DT, LOGITS, 64>(p, rows, stream);
    return launch_short<DT, LOGITS, 96>(p, rows, stream);
}

}  // namespace

// Where there are rows for every SIMD: one wavefront takes longer over a row
// than four (1024 rows of 4000 bf16 log-probs 14 us against 13, 256 of 1000 f32
// 11 against 10; but 1024 of 2000 f16 11 against 13, 4096 of 4000 18 against 32).
bool row_short_preferred(const DecodeParams& p) {
    const int64_t rows = static_cast<int64_t>(p.B) * (p.step_mode ? 1 : p.T) * p.K;
    return 2 * rows >= p.V;
}

bool row_short_eligible(const DecodeParams& p) { return p.V <= kShortRow && p.M <= 256; }

hipError_t launch_row_short(const DecodeParams& p, int64_t rows, hipStream_t stream) {
    if (rows <= 0) return hipSuccess;
    switch (p.dtype) {
        case 0: return p.from_logits ? launch_short_typed<0, true>(p, rows, stream) : launch_short_typed<0, false>(p, rows, stream);
        case 1: return p.from_logits ? launch_short_typed<1, true>(p, rows, stream) : launch_short_typed<1, false>(p, rows, stream);
        default: return p.from_logits ? launch_short_typed<2, true>(p, rows, stream) : launch_short_typed<2, false>(p, rows, stream);
    }
}

}  // namespace dbs_hip
