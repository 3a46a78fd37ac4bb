// moe.h -- the grouped expert GEMM's arguments (moe.hip, moe_tile.hip).
#pragma once
#include "common.h"

// C[s, n] = T(acc * (scale[e,n]) (+ bias[e,n]) (* topk_w[s])) with
//   acc = sum_k A[s / a_div, k] * B[e, n, k],  B T or int8 [E, N, K]
// for every slot s of every sorted block with expert e != -1; e == -1 zeroes
// the block's rows.
struct MoeArgs {
  void* C;
  const void* A;
  const void* B;
  const void* Bs;   // int8 path: per-channel scales T [E, N]
  const void* bias; // T [E, N] or null
  const float* tw;  // [topk_ids_size] or null
  const int* sorted;
  const int* eids;
  const int* ntpp;
  int K, N, E, tis, top_k, bs, mrw;
  int act;  // 1: gated SiLU output C[s, n] = T(silu(g) u), g / u = weight rows n / N/2 + n
  int a_div;  // slot s reads A row s / a_div
};

// The grouped GEMM on tiles of 32 (int8 only), 64 or 128 rows (moe_tile.hip);
// err: the device flag of out-of-range expert ids.  false: nothing launched,
// the call is outside its contract.  ub_moe_tile_rows: the rows to take for
// these sizes, 0 where k_moe_gemm is faster.
bool ub_moe_tile(const MoeArgs& a, int rows, int dt, bool q8, int* err, hipStream_t s);
int ub_moe_tile_rows(const MoeArgs& a, bool q8);

// The same for decode batches whose blocks leave CUs idle (moe_stream.hip).
bool ub_moe_stream(const MoeArgs& a, int dt, bool q8, int* err, hipStream_t s);
bool ub_moe_stream_pays(const MoeArgs& a, bool q8);
