// Host-side launchers of the decode / combine / keep-mask kernels (decode_kernels.hip).
#pragma once
#include "common.h"

namespace fa {
// each returns the hipError_t of the launch as int
int launch_decode_split(const FwdArgs& a, hipStream_t st);
// query heads that a work-group of the decode kernel serves
int decode_heads_per_group(int kv_group);
int launch_combine(const FwdArgs& a, hipStream_t st);
int launch_keep_mask(uint8_t* mask, int B, int H, int Nq, int Nk, uint32_t thr, uint64_t seed, uint64_t offset,
                     hipStream_t st);
}  // namespace fa
