// SPDX-License-Identifier: MIT
//
// The select pass for bfloat16 rows.
#include "select_kernels.hpp"

namespace dbs_hip {

template hipError_t launch_select_dtype<2>(const DecodeParams&, const SelectLayout&, hipStream_t);
template hipError_t rescan_counter_dtype<2>(int, unsigned long long*);
template hipError_t wait_timeout_counter_dtype<2>(int, unsigned long long*);

}  // namespace dbs_hip
