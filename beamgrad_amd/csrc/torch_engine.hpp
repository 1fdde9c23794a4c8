// SPDX-License-Identifier: MIT
//
// What libdbs_hip exports for this package's torch module alone (not part of
// its C ABIs).
#pragma once

#include <stdint.h>

#include "dbs_cuda.h"

// The least workspace a decode (step_mode 0) or a step takes: beyond 64 beams,
// without the shortlists that dbs_cuda_decode_workspace_size and
// dbs_cuda_decode_step_workspace_size make room for. -1 for invalid arguments.
extern "C" __attribute__((visibility("default"))) int64_t beamgrad_least_workspace(const DBSCudaDecodeArgs* args,
                                                                                   int step_mode, int prefix_stride);

// The beams after one step of the step API, in one launch: from the step's
// outputs and updated state [B, K] (tokens, parents, lengths, raw scores,
// from_logprob, finished) and the sequences before it [B, K, step] (ignored at
// step 0), the sequences after it [B, K, step + 1] as int64 and int32 (the
// parent's tokens, then the one emitted, -1 where none was; a dead slot all
// -1), tokens, parents and lengths as int64, finished and active (finite raw
// score, not finished) as 0/1 bytes, and *any_active (device): whether any beam
// is active. Returns a dbs_cuda status.
extern "C" __attribute__((visibility("default"))) int beamgrad_advance_beams(
    const int32_t* tokens, const int32_t* parents, const int32_t* lengths, const float* raw_scores,
    const uint8_t* from_logprob, const uint8_t* finished, const int64_t* sequences, int batch_size, int beam_size,
    int step, int64_t* sequences_out, int32_t* prefixes_out, int64_t* tokens64, int64_t* parents64, int64_t* lengths64,
    uint8_t* finished_bool, uint8_t* active, int32_t* any_active, void* stream);
