// SPDX-License-Identifier: MIT
//
// Row pass that reads a row twice, for rows of any type, size and alignment:
// the logits rows the relay pass does not take, and log-prob rows past the
// one-read pass's registers (which have no logsumexp: the second read only
// finds the survivors).
//
// Each row's logsumexp folds exp(fl(x - max)) into 256 lanes (lane j = v mod
// 256, increasing v; reference src/kernels_scalar.cpp:48-66), so the maximum
// comes first and each lane's sum is one chain. One 256-thread workgroup takes
// a row, several share a CU (one row's loads run beside another's
// arithmetic):
//
//   * first read: 16-byte blocks aligned in memory; the maximum, the NaN / +inf
//     flag and the shortlist threshold theta (the M-th largest of the 256
//     thread maxima: at least M elements reach it);
//   * second read: thread j takes lane j, one element per stripe of 256 (any
//     row alignment), 16 stripes a group with the next group's loads in
//     flight, and adds the exact terms in order;
//   * a group whose maximum reaches theta is recorded, and its elements are
//     read again once the row is folded: some M of V / 16 groups a lane;
//   * the survivors are ranked and published as in the log-prob row pass.
//
// What bounds it. The second read is not served from the Infinity Cache
// (measured: 3.7-4.0 TB/s of rows read twice whatever their number in flight,
// 7.2 TB/s read once), and binary16 and float32 terms cost 25 vector operations
// each (exp_term), 28 an element with the first read's: 2.9 TB/s of binary16
// and 5.8 TB/s of float32 rows at 2.4 GHz (measured, row bytes over time: 8 x 32
// x 8 x 128256 f16 203 us, 2.5 TB/s; 16 x 64 x 4 x 50257 f32 279 us, 2.9 TB/s:
// two reads at 5.9). bfloat16 terms come from a table (7 operations an element
// and 8192 terms a row), 32 x 48 x 5 x 50257 327 us, 2.4 TB/s. Loading 16-bit
// rows by dwords (half the loads, lanes exchanged after) was slower, 238 and
// 337 us. Keeping the row on chip instead
// pays only where the arithmetic leaves room: long bfloat16 rows (a table of the
// terms), which the relay pass takes where alignment allows.
#include <hip/hip_runtime.h>

#include <type_traits>

#include "row_helpers.hpp"

namespace dbs_hip {

namespace {

constexpr int kStThreads = 256;
constexpr int kStGroup = 16;    // stripes per group
// LDS beside the 32 KB term table: four workgroups per CU take 40 KB each.
constexpr int kStRecords = 432;   // groups holding survivors, at most (else the row is read in full)
constexpr int kStSurvivors = 432; // survivors, at most (likewise)
constexpr int kStTableRow = 12000;  // bfloat16 rows from which the term table pays (8192 terms against 5 of 25 operations an element)
constexpr int kStBlocks = 8;    // 16-byte loads in flight per thread in the first read
constexpr int kFirstPolicy = 0;  // (the second read streams, kRowLoadPolicy: 4.0 against 3.7 TB/s)

// TABLE: bfloat16 logits rows long enough for the term table.
template <int DT, bool LOGITS, bool TABLE>
__global__ __launch_bounds__(kStThreads) __attribute__((amdgpu_waves_per_eu(4))) void
row_stream_kernel(DecodeParams p, int64_t rows) {
    __shared__ __align__(16) float s_lut[TABLE ? 2 * kLutHalf : 1];
    __shared__ uint64_t s_key[kStSurvivors];
    __shared__ float s_x[kStSurvivors];
    __shared__ uint32_t s_rec[kStRecords];
    __shared__ __align__(16) uint32_t s_tkey[kStThreads];
    float* const s_acc = reinterpret_cast<float*>(s_tkey);  // (the keys are read before the sums are written)
    __shared__ RowSlot s_slot;
    __shared__ int s_count, s_nrec, s_bad;
    __shared__ float s_m, s_theta, s_lse, s_bound;

    constexpr int kTicketThread = 64;
    constexpr int esz = DT == 0 ? 4 : 2;
    constexpr int epb = 16 / esz;
    const int tid = static_cast<int>(threadIdx.x);
    const int lane = tid & 63;
    const int V = p.V, M = p.M;
    const bool coherent = p.step_done != nullptr;

    int64_t q = 0;
    if (tid == kTicketThread) {
        q = first_ticket(p);
        int b0 = 0, len0 = 0;
        s_slot.r = find_read_row(p, rows, q, b0, len0);
        s_slot.b = b0;
        s_slot.len = len0;
        s_bad = 0;
    }
    __syncthreads();
    int b, new_len;
    int64_t r = read_row_slot(s_slot, b, new_len);

    while (r < rows) {
        const uintptr_t a0 = reinterpret_cast<uintptr_t>(p.x) + static_cast<uintptr_t>(r) * static_cast<uintptr_t>(V) * esz;

        // First read: 16-byte blocks, the first may start before the row and
        // the last end after it (a block holding a row byte crosses no page).
        Extremes<DT> ex;
        {
            const int lead = static_cast<int>(a0 & 15u), lead_e = lead / esz;
            const int nblk = (lead + V * esz + 15) >> 4;
            const __amdgpu_buffer_rsrc_t rs =
                __builtin_amdgcn_make_buffer_rsrc(reinterpret_cast<void*>(a0 - lead), 0, 16 * nblk, 0x00020000);
#pragma unroll 1
            for (int c0 = 0; c0 * kStThreads < nblk; c0 += kStBlocks) {
                v4u32 d[kStBlocks];
#pragma unroll
                for (int u = 0; u < kStBlocks; ++u)
                    d[u] = __builtin_amdgcn_raw_buffer_load_b128(rs, 16 * tid, min(16 * kStThreads * (c0 + u), 16 * nblk),
                                                                 kFirstPolicy);
                const bool inside = (c0 > 0 || lead == 0) && (c0 + kStBlocks) * kStThreads * epb - lead_e <= V;
                if (!inside) {
                    // elements outside the row become -inf
#pragma unroll
                    for (int u = 0; u < kStBlocks; ++u) {
                        const int v0 = ((c0 + u) * kStThreads + tid) * epb - lead_e;
#pragma unroll
                        for (int i = 0; i < epb; ++i) {
                            if (v0 + i >= 0 && v0 + i < V) continue;
                            if constexpr (DT == 0) {
                                d[u][i] = 0xff800000u;
                            } else {
                                const uint32_t ninf = DT == 1 ? 0xfc00u : 0xff80u;
                                const int sh = 16 * (i & 1);
                                d[u][i >> 1] = (d[u][i >> 1] & ~(0xffffu << sh)) | (ninf << sh);
                            }
                        }
                    }
                }
#pragma unroll
                for (int u = 0; u < kStBlocks; ++u) ex.take(d[u]);
            }
        }
        bool bad;
        float tmax = ex.result(bad);
        s_tkey[tid] = ordered_key(tmax);
        if (__any(bad) && lane == 0) s_bad = 1;
        __syncthreads();
        const bool any_bad = s_bad != 0;

        // Second read: lane tid's elements. The view starts at the row's first
        // whole dword.
        const int lead2 = static_cast<int>(a0 & 3u);
        const __amdgpu_buffer_rsrc_t rs =
            __builtin_amdgcn_make_buffer_rsrc(reinterpret_cast<void*>(a0 - lead2), 0, lead2 + V * esz, 0x00020000);
        const int voff = lead2 + tid * esz;
        const int S = (V + 255) >> 8;  // stripes
        auto load_group = [&](uint32_t (&h)[kStGroup], int g) __attribute__((always_inline)) {
#pragma unroll
            for (int u = 0; u < kStGroup; ++u)
                h[u] = load_raw<DT>(rs, voff, min((g * kStGroup + u) * 256 * esz, lead2 + V * esz));
        };
        // (the scalar offset is kept within the view: past it, every lane's load
        // is out of range and returns zero)
        uint32_t h0[kStGroup];  // the first group goes out while the threshold and the table are made
        load_group(h0, 0);
        if (any_bad) {
            // a row with NaN or +inf: the maximum of the entries below +inf
            tmax = -kInf;
            for (int s = 0; s < S; ++s) {
                const float x = raw_value<DT>(load_raw<DT>(rs, voff, s * 256 * esz));
                if (s * 256 + tid < V && x < kInf && x > tmax) tmax = x;
            }
            s_tkey[tid] = ordered_key(tmax);
            __syncthreads();
        }
        if (tid < 64) {
            const uint4 kk = reinterpret_cast<const uint4*>(s_tkey)[tid];
            const uint32_t k4[4] = {kk.x, kk.y, kk.z, kk.w};
            const uint32_t top = max(max(kk.x, kk.y), max(kk.z, kk.w));
            const float m = wave_max_dpp(key_value(top));
            // (to its 20 highest bits, rounded down: at least M elements reach
            // it, and twelve rounds less are waited for)
            const float th = M > 0 ? key_value(mth_largest_key<32, 12>(k4, M)) : -kInf;
            if (tid == 0) {
                s_m = m;
                s_theta = th;
            }
        } else if (tid == kTicketThread) {
            s_nrec = 0;
            s_count = 0;
            publish_next_row(p, rows, q, s_slot);
        }
        __syncthreads();
        if (tid == kTicketThread) s_bad = 0;  // every thread has read it
        const float m = s_m;
        const bool do_lse = m > -kInf;  // (log-probs: a finite entry)
        const bool listing = M > 0 && !any_bad;  // (a flagged row keeps no shortlist)
        const float theta = listing ? list_threshold<DT>(s_theta) : kInf;

        bool table = false;
        if constexpr (TABLE) {
            // terms by bfloat16 pattern (term_slots), where the row fits them
            table = table_fits_fixed(m);
            if (table) {
#pragma unroll 4
                for (int i = tid; i < 2 * kLutHalf; i += kStThreads) {
                    const int k = i & (kLutHalf - 1);
                    const uint32_t sign = i >= kLutHalf ? 0x8000u : 0u;
                    const float x = bits_f32((sign | (k == 0 ? 0u : kFixedBase - 1u + k)) << 16);
                    s_lut[i] = k == kLutHalf - 1 ? 0.0f : exp_term(m, x);
                }
                __syncthreads();
            }
        }

        float acc = 0.0f;
        auto record = [&](float gmax, int g) __attribute__((always_inline)) {
            if (gmax >= theta) {
                const int slot = atomicAdd(&s_nrec, 1);
                if (slot < kStRecords) s_rec[slot] = static_cast<uint32_t>(g * kStThreads + tid);
            }
        };
        // Group g's terms. EDGE: the row ends in it.
        auto fold = [&](const uint32_t (&h)[kStGroup], int g, auto edge) __attribute__((always_inline)) {
            constexpr bool EDGE = decltype(edge)::value;
            float x[kStGroup];
#pragma unroll
            for (int u = 0; u < kStGroup; ++u) {
                x[u] = raw_value<DT>(h[u]);
                if (EDGE && (g * kStGroup + u) * 256 + tid >= V) x[u] = -kInf;
            }
            float gm = max3(x[0], x[1], x[2]);
#pragma unroll
            for (int u = 3; u + 1 < kStGroup; u += 2) gm = max3(gm, x[u], x[u + 1]);
            gm = max3(gm, x[kStGroup - 1], x[kStGroup - 1]);
            if constexpr (LOGITS) {
#pragma unroll
                for (int u = 0; u < kStGroup; ++u) acc = acc + exp_term(m, x[u]);
            }
            record(gm, g);
        };
        auto fold_table = [&](const uint32_t (&h)[kStGroup], int g, auto edge) __attribute__((always_inline)) {
            constexpr bool EDGE = decltype(edge)::value;
            uint32_t w[kStGroup / 2];
            float e[kStGroup];
            float gm = -kInf;
#pragma unroll
            for (int u = 0; u < kStGroup; u += 2) {
                uint32_t lo = h[u], hi = h[u + 1];
                if (EDGE && (g * kStGroup + u) * 256 + tid >= V) lo = 0xff80u;
                if (EDGE && (g * kStGroup + u + 1) * 256 + tid >= V) hi = 0xff80u;
                w[u / 2] = lo | (hi << 16);
                const uint32_t slots = term_slots(w[u / 2]);
                e[u] = s_lut[slots & 0xffffu];
                e[u + 1] = s_lut[slots >> 16];
            }
            if (theta > 0.0f) {
                // a positive threshold: the largest signed pattern decides
                uint32_t pm = w[0];
#pragma unroll
                for (int u = 1; u < kStGroup / 2; ++u) pm = pk_max_i16(pm, w[u]);
                const int best = max(static_cast<int>(static_cast<int16_t>(pm)), static_cast<int>(pm) >> 16);
                gm = best >= 0 ? bits_f32(static_cast<uint32_t>(best) << 16) : -kInf;
            } else {
#pragma unroll
                for (int u = 0; u < kStGroup / 2; ++u) gm = max3(gm, bits_f32(w[u] << 16), bits_f32(w[u] & 0xffff0000u));
            }
#pragma unroll
            for (int u = 0; u < kStGroup; ++u) acc = acc + e[u];
            record(gm, g);
        };
        // Whole groups two at a time, each one's loads in flight while the
        // other folds, then the rest (loads past the row return zeros).
        auto fold_row = [&](auto one) __attribute__((always_inline)) {
            const int G = V / (256 * kStGroup);
            uint32_t h1[kStGroup];
            int g = 0;
#pragma unroll 1
            for (; g + 2 <= G; g += 2) {
                load_group(h1, g + 1);
                one(h0, g, std::false_type{});
                load_group(h0, g + 2);
                one(h1, g + 1, std::false_type{});
            }
            if (g < G) {
                load_group(h1, g + 1);
                one(h0, g, std::false_type{});
                one(h1, g + 1, std::true_type{});
            } else {
                one(h0, g, std::true_type{});
            }
        };
        if (do_lse && (LOGITS || listing)) {
            if (TABLE && table) fold_row(fold_table);
            else fold_row(fold);
        }
        s_acc[tid] = acc;
        __syncthreads();

        // Wavefront 0: the lane tree and the logsumexp; the others: the
        // recorded groups' elements.
        const int nrec = s_nrec;
        const bool keep = listing && nrec <= kStRecords;
        if (tid < 64) {
            float lse = 0.0f;
            if constexpr (LOGITS) {
                float a[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) a[e] = s_acc[4 * tid + e];
                lse = do_lse ? logsumexp_from(m, lane_tree_sum(a, tid)) : -kInf;
            }
            if (tid == 0) s_lse = lse;
        } else if (keep) {
            const bool mask_eos = new_len < min_length_of(p, b);
            for (int i = tid - 64; i < nrec * kStGroup; i += kStThreads - 64) {
                const uint32_t rec = s_rec[i / kStGroup];
                const int s = static_cast<int>(rec >> 8) * kStGroup + i % kStGroup, j = static_cast<int>(rec & 255u);
                const int v = s * 256 + j;
                const float x = raw_value<DT>(load_raw<DT>(rs, lead2 + j * esz + s * 256 * esz, 0));
                if (v < V && x >= theta && !static_masked(p, b, v, mask_eos)) {
                    const int slot = atomicAdd(&s_count, 1);
                    if (slot < kStSurvivors) {
                        s_key[slot] = survivor_key(x, v);
                        s_x[slot] = x;
                    }
                }
            }
        }
        __syncthreads();
        const float lse = s_lse;
        int bn, len_n;
        const int64_t rn = read_row_slot(s_slot, bn, len_n);

        // The shortlist: each survivor's rank is the number of survivors
        // before it (keys are distinct); ranks below M are written in place,
        // rank M is the bound on the rest.
        const int n = s_count;
        const bool listed = keep && n <= kStSurvivors;
        if (listed) {
            ShortEntry* out = p.shortlist + r * M;
            for (int i = tid; i < n; i += kStThreads) {
                const uint64_t ki = s_key[i];
                int rank = 0;
                int j = 0;
                for (; j + 4 <= n; j += 4) {
                    const uint64_t k0 = s_key[j], k1 = s_key[j + 1], k2 = s_key[j + 2], k3 = s_key[j + 3];
                    rank += static_cast<int>(k0 > ki) + static_cast<int>(k1 > ki) + static_cast<int>(k2 > ki) +
                            static_cast<int>(k3 > ki);
                }
                for (; j < n; ++j) rank += static_cast<int>(s_key[j] > ki);
                if (rank < M) {
                    const int32_t tok = static_cast<int32_t>(0xffffffffu - static_cast<uint32_t>(ki & 0xffffffffu));
                    publish_entry(out, rank, LOGITS ? s_x[i] - lse : s_x[i], tok, coherent);
                } else if (rank == M) {
                    s_bound = s_x[i];
                }
            }
        }
        lds_barrier();
        if (tid < 64) {
            RowInfo info;
            info.lse = lse;
            info.invalid = any_bad ? 1u : 0u;
            info.bound = -kInf;
            info.count = 0;
            if (M > 0 && (do_lse || !LOGITS)) {
                if (listed) {
                    info.count = n < M ? n : M;
                    info.bound = n > M ? s_bound : list_bound<DT>(theta);
                    if constexpr (LOGITS) info.bound = info.bound - lse;
                } else {
                    info.count = -1;
                }
            }
            if (tid == 0) publish_rowinfo(p.rowinfo + r, info, coherent);
            signal_row_done(p, r, tid);
        }
        r = rn;
        b = bn;
        new_len = len_n;
    }
}

int g_st_cus[64];

template <int DT, bool LOGITS, bool TABLE = false>
hipError_t launch_st(const DecodeParams& p, int64_t rows, int cus, hipStream_t stream) {
    static const int per_cu = [] {
        int blocks = 0;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&blocks, reinterpret_cast<const void*>(&row_stream_kernel<DT, LOGITS, TABLE>),
                                                         kStThreads, 0) != hipSuccess || blocks < 1)
            blocks = 1;
        return blocks;
    }();
    const int64_t slots = static_cast<int64_t>(cus) * per_cu;
    const int64_t grid = rows < slots ? rows : slots;
    hipLaunchKernelGGL((row_stream_kernel<DT, LOGITS, TABLE>), dim3(static_cast<unsigned>(grid)), dim3(kStThreads), 0, stream, p,
                       rows);
    return hipGetLastError();
}

}  // namespace

bool row_stream_eligible(const DecodeParams& p) {
    // (byte offsets within a row are 31-bit, with room for the last group)
    return p.M <= 256 && p.V < (1 << 28);
}

hipError_t launch_row_stream(const DecodeParams& p, int64_t rows, hipStream_t stream) {
    if (rows <= 0) return hipSuccess;
    int device = 0;
    hipError_t e = hipGetDevice(&device);
    if (e != hipSuccess) return e;
    if (device < 0 || device >= 64) return hipErrorInvalidDevice;
    if (g_st_cus[device] == 0) {
        int cus = 0;
        e = hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device);
        if (e != hipSuccess) return e;
        g_st_cus[device] = cus > 0 ? cus : 1;
    }
    const int held = p.select_hold ? p.reserve_cus : 0;
    const int cus = g_st_cus[device] - held > 0 ? g_st_cus[device] - held : 1;
    if (p.dtype == 2 && p.from_logits && p.V >= kStTableRow) return launch_st<2, true, true>(p, rows, cus, stream);
#define DBS_ST_CASE(DT) \
    return p.from_logits ? launch_st<DT, true>(p, rows, cus, stream) : launch_st<DT, false>(p, rows, cus, stream)
    switch (p.dtype) {
        case 0: DBS_ST_CASE(0);
        case 1: DBS_ST_CASE(1);
        default: DBS_ST_CASE(2);
    }
#undef DBS_ST_CASE
}

}  // namespace dbs_hip
