// stack.hpp -- what the resident stack launch (stack.hip) asks of the files whose sums it repeats.
#pragma once
#include "vx_common.hpp"

// mul_mat.hip: waves that share a product's k blocks (and with them the order of its sum)
int vx_gemv_waves(int64_t K, int64_t tokens, int64_t M);
int vx_gemv_dma_slot(int64_t K); // bytes between two rows' images in LDS

// fattn.hip: the key ranges of a decode attention of `tiles` (sequence, KV head) pairs over n_kv keys; false when a switch of
// that file has it run on another kernel.  Whether T tokens of a sequence without a cache run on the column kernel's half tile.
bool vx_fattn_stack_plan(int64_t tiles, int n_kv, bool f16, int * n_splits, int * chunk);
bool vx_fattn_stack_self(int64_t tokens, int64_t gqa);
