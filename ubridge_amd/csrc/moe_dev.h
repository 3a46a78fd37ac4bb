// moe_dev.h -- device code shared by the grouped expert GEMMs (moe.hip,
// moe_tile.hip, moe_stream.hip).
#pragma once
#include "moe.h"

namespace {

constexpr uint16_t kElsewhere = 0xffff, kBadExpert = 0xfffe;  // list entries without weights here

// blocks that sorted / experts_ids are sized for
__host__ __device__ inline int max_blocks(const MoeArgs& a) {
  return (int)((a.tis + (long)a.E * (a.bs - 1)) / a.bs);
}

template <int DT>
__device__ __forceinline__ float tof(uint16_t b) {
  if constexpr (DT == UB_BF16) return ub_bf16_to_f32(b);
  else return ub_f16_to_f32(b);
}
template <int DT>
__device__ __forceinline__ uint32_t pack2(float lo, float hi) {
  typedef float f32x2 __attribute__((ext_vector_type(2)));
  const f32x2 v = {lo, hi};
  if constexpr (DT == UB_BF16) {
    typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2));
  } else {
    typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, f16x2));
  }
}
// 8 int8 (two dwords) -> 8 T, exact.
template <int DT>
__device__ __forceinline__ uint4 i8x8_to_t(uint32_t lo, uint32_t hi) {
  uint32_t o[4];
  if constexpr (DT == UB_BF16) {
    typedef signed char i8x4 __attribute__((ext_vector_type(4)));
    const i8x4 L = __builtin_bit_cast(i8x4, lo), H = __builtin_bit_cast(i8x4, hi);
    o[0] = pack2<DT>((float)L[0], (float)L[1]);
    o[1] = pack2<DT>((float)L[2], (float)L[3]);
    o[2] = pack2<DT>((float)H[0], (float)H[1]);
    o[3] = pack2<DT>((float)H[2], (float)H[3]);
  } else {
    // the byte q + 128 under 0x64 is the f16 1024 + (q + 128); minus 1152
    typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
    const f16x2 off = {(_Float16)1152.0f, (_Float16)1152.0f};
    const uint32_t l = lo ^ 0x80808080u, h = hi ^ 0x80808080u, m = 0x64646464u;
    const uint32_t p[4] = {__builtin_amdgcn_perm(m, l, 0x04010400u), __builtin_amdgcn_perm(m, l, 0x04030402u),
                           __builtin_amdgcn_perm(m, h, 0x04010400u), __builtin_amdgcn_perm(m, h, 0x04030402u)};
#pragma unroll
    for (int i = 0; i < 4; i++)
      o[i] = __builtin_bit_cast(uint32_t, (f16x2)(__builtin_bit_cast(f16x2, p[i]) - off));
  }
  return make_uint4(o[0], o[1], o[2], o[3]);
}

// 8 int8 (two dwords) -> 8 T holding q + 128 (exact: 0..255 fit T's
// significand); the caller subtracts 128 * (sum of the A row) after the
// dot.  bf16: 1.75 VALU ops per value: one xor per 4, a byte convert each,
// one pack per 2.
template <int DT>
__device__ __forceinline__ uint4 i8x8_to_t_off(uint32_t lo, uint32_t hi) {
  const uint32_t l = lo ^ 0x80808080u, h = hi ^ 0x80808080u;
  uint32_t o[4];
  if constexpr (DT == UB_BF16) {
    typedef unsigned char u8x4 __attribute__((ext_vector_type(4)));
    const u8x4 L = __builtin_bit_cast(u8x4, l), H = __builtin_bit_cast(u8x4, h);
    o[0] = pack2<DT>((float)L[0], (float)L[1]);
    o[1] = pack2<DT>((float)L[2], (float)L[3]);
    o[2] = pack2<DT>((float)H[0], (float)H[1]);
    o[3] = pack2<DT>((float)H[2], (float)H[3]);
  } else {
    // the byte q + 128 under 0x64 is the f16 1024 + (q + 128)
    typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
    const f16x2 off = {(_Float16)1024.0f, (_Float16)1024.0f};
    const uint32_t m = 0x64646464u;
    const uint32_t p[4] = {__builtin_amdgcn_perm(m, l, 0x04010400u), __builtin_amdgcn_perm(m, l, 0x04030402u),
                           __builtin_amdgcn_perm(m, h, 0x04010400u), __builtin_amdgcn_perm(m, h, 0x04030402u)};
#pragma unroll
    for (int i = 0; i < 4; i++)
      o[i] = __builtin_bit_cast(uint32_t, (f16x2)(__builtin_bit_cast(f16x2, p[i]) - off));
  }
  return make_uint4(o[0], o[1], o[2], o[3]);
}
// acc + the sum of the 8 T values of an MFMA fragment (f32, by v_dot2)
template <int DT>
__device__ __forceinline__ float frag_sum(const uint4& a, float acc) {
  const uint32_t w[4] = {a.x, a.y, a.z, a.w};
#pragma unroll
  for (int i = 0; i < 4; i++) {
    if constexpr (DT == UB_BF16) {
      typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
      const bf16x2 one = {(__bf16)1.0f, (__bf16)1.0f};
      acc = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, w[i]), one, acc, false);
    } else {
      typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
      const f16x2 one = {(_Float16)1.0f, (_Float16)1.0f};
      acc = __builtin_amdgcn_fdot2(__builtin_bit_cast(f16x2, w[i]), one, acc, false);
    }
  }
  return acc;
}

// Cuts the sorted blocks into tiles (consecutive blocks of one expert, G at
// most) and lists tiles [first, first + cap) in LDS: first block and expert of
// each, and the block after the last one.  Called by every thread of an
// NWV-wavefront workgroup; returns the number of tiles there are in all.
// Thread t scans blocks [t C, (t + 1) C).
template <int NWV>
__device__ __forceinline__ int moe_tile_list(const MoeArgs& a, int G, int first, int cap, uint16_t* tab_b,
                                             uint16_t* tab_e, int (*wsum)[NWV]) {
  constexpr int NT = 64 * NWV;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int nblk = min((*a.ntpp + a.bs - 1) / a.bs, max_blocks(a));
  // f(b, e, whether block b starts a tile), given the last run start before b0
  auto walk = [&](int rs, auto f) {
    const int C = (nblk + NT - 1) / NT, b0 = min(nblk, tid * C), b1 = min(nblk, b0 + C);
    int pe = b0 > 0 && b0 < nblk ? a.eids[b0 - 1] : 0;
    for (int b = b0; b < b1; b++) {
      const int e = a.eids[b];
      if (b == 0 || e != pe) rs = b;
      pe = e;
      f(b, e, (b - rs) % G == 0);
    }
    return rs;
  };
  auto scan = [&](int v, int which, bool mx) {  // exclusive scan over the workgroup
    int x = v;
    for (int o = 1; o < 64; o <<= 1) {
      const int u = __shfl_up(x, o, 64);
      if (lane >= o) x = mx ? max(x, u) : x + u;
    }
    if (lane == 63) wsum[which][wave] = x;
    __syncthreads();
    int base = mx ? -1 : 0;
    for (int w = 0; w < wave; w++) base = mx ? max(base, wsum[which][w]) : base + wsum[which][w];
    const int up = __shfl_up(x, 1, 64);
    return lane == 0 ? base : mx ? max(base, up) : base + up;
  };
  const int carry = scan(walk(-1, [](int, int, bool) {}), 0, true);
  int at = 0;
  walk(carry, [&](int, int, bool start) { at += start; });
  at = scan(at, 1, false) - first;
  int tiles = 0;
  for (int w = 0; w < NWV; w++) tiles += wsum[1][w];
  walk(carry, [&](int b, int e, bool start) {
    if (!start) return;
    if (at >= 0 && at <= cap) tab_b[at] = (uint16_t)b;
    if (at >= 0 && at < cap) tab_e[at] = e == -1 ? kElsewhere : e >= 0 && e < a.E ? e : kBadExpert;
    at++;
  });
  if (tid == 0 && tiles - first <= cap) tab_b[tiles - first] = (uint16_t)nblk;
  __syncthreads();
  return tiles;
}

}  // namespace
