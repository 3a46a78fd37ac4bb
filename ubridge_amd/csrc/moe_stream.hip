// moe_stream.hip -- grouped expert GEMM for decode batches: few rows per
// expert, so the product is a stream of the weights of the experts in use
// (gfx950).
//
// Bound by HBM, so shaped for bytes in flight and for every CU having the
// same share of the stream:
//  * The sorted blocks are cut into tiles of 32 rows of one expert; the
//    (tile, column block) items form one list, and every workgroup of the
//    persistent grid takes an equal contiguous run of it, however few experts
//    are in use and however their rows fall.
//  * The W wavefronts of a workgroup split K: wavefront w the 128-element
//    steps w, w + W, ... (at most SP), so a wavefront's activation fragments
//    are the same for every item of a tile and stay in registers; weights
//    go from memory straight to the MFMA operand registers (a load covers
//    64-byte runs of 16 weight rows), the next item's in flight while the
//    current one is multiplied (two register sets, the loop unrolled by two).
//  * v_mfma_f32_16x16x32, weights as the A operand: lane (r, h) ends with
//    weight rows 4 h .. 4 h + 3 of token row r.  The partial sums of the W
//    wavefronts meet in LDS in wavefront order, in one of two buffers by item
//    parity, so one barrier per item suffices.
//  * Within a 128-element step, lane (r, h) takes k = 64 q + 16 h + 8 s .. + 7
//    for product (q, s) on both operands: an int8 row's 16 bytes are one load.
//  * int8 is exact in T; scale, bias and routed weight are applied to the f32
//    sums as in k_moe_gemm.
//
// At one token the chain of dependent loads (block list, slots, activations)
// is most of it: 25 MB of int8 gate/up weights, 2048 -> 2 x 768, 8 experts,
// take 11.8 us (k_moe_gemm 18.5).
#include "lds_dma.h"
#include "moe_dev.h"

#include <algorithm>
#include <type_traits>

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int W = 8, NT = 64 * W;   // wavefronts / threads of a workgroup
constexpr int kTiles = 1024;        // tiles a launch can have
constexpr uint32_t kOOB = 0x80000000u;  // an offset past every buffer: reads zero

__device__ __forceinline__ __amdgpu_buffer_rsrc_t rsrc(const void* base, uint64_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, (int)bytes, 0x00020000);
}
__device__ __forceinline__ uint4 ld16(__amdgpu_buffer_rsrc_t r, uint32_t off) {
  typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
  return __builtin_bit_cast(uint4, (u32x4)__builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0));
}
template <int DT>
__device__ __forceinline__ f32x4 mfma(const uint4& a, const uint4& b, const f32x4& c) {
  if constexpr (DT == UB_BF16)
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b),
                                                   c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b),
                                                  c, 0, 0, 0);
}

// Q8: int8 weights.  ACT: gated SiLU output (gate and up rows of an item's
// columns are its two weight tiles).  SP: 128-element steps of a wavefront, OCC
// wavefronts per SIMD.  RT = 4 (items twice as wide) was level or slower.
template <int DT, bool Q8, bool ACT, int SP, int OCC>
__global__ void __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(OCC, OCC)))
k_moe_stream(MoeArgs a, int* err) {
  constexpr int TM = 2, RT = 2;                      // 16-row token / weight tiles of an item
  constexpr int WB = Q8 ? 1 : 2, U = Q8 ? 2 : 4;     // 16-byte loads of a weight row's step
  constexpr int kTM = 16 * TM, NR = 16 * RT, CT = ACT ? NR / 2 : NR;  // rows, weight rows, columns
  constexpr int NRP = NR + 4;                        // padded row of partial sums
  constexpr int CP = CT / 2, NO_T = (kTM * CP + NT - 1) / NT;  // column pairs; outputs per thread
  static_assert(NT % CP == 0, "a thread keeps its columns");
  __shared__ __attribute__((aligned(16))) float red[2][W * kTM * NRP];
  __shared__ uint16_t tab_b[kTiles + 1], tab_e[kTiles];
  __shared__ int wsum[2][W];
  const int tid = threadIdx.x, lane = tid & 63, r = lane & 15, h = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int K = a.K, N = a.N, bs = a.bs, NO = ACT ? N / 2 : N, ncol = (NO + CT - 1) / CT;
  const int G = gridDim.x;  // a multiple of 8
  const int tiles = moe_tile_list<W>(a, kTM / bs, 0, kTiles, tab_b, tab_e, wsum);
  // equal runs of the items, those of one XCD (workgroup i runs on XCD i % 8) neighbours
  const long total = (long)tiles * ncol;
  const int wg = ((int)blockIdx.x & 7) * (G >> 3) + ((int)blockIdx.x >> 3);
  const int i0 = (int)(total * wg / G), i1 = (int)(total * (wg + 1) / G);
  if (i0 >= i1) return;

  const uint32_t brow = (uint32_t)K * WB;
  const int arows = (a.tis + a.a_div - 1) / a.a_div;
  const __amdgpu_buffer_rsrc_t ra = rsrc(a.A, (uint64_t)arows * K * 2);
  uint32_t ko[SP];  // first element of the wavefront's step i, kOOB past K
#pragma unroll
  for (int i = 0; i < SP; i++) ko[i] = wave + i * W < K / 128 ? (uint32_t)(wave + i * W) * 128u : kOOB;

  typedef uint4 BSet[SP][RT][U];
  struct Ep {  // a thread's column pair: scales and bias (gate, up with ACT)
    uint32_t sc[ACT ? 2 : 1], bv[ACT ? 2 : 1];
  };
  const int c2 = 2 * (tid % CP);
  auto load = [&](BSet& b, Ep& ep, int it) {  // item it's weights; nothing past the run
    const int t = min(it, i1 - 1) / ncol, n0 = (min(it, i1 - 1) - t * ncol) * CT;
    const int e = __builtin_amdgcn_readfirstlane((int)tab_e[t]);
    const bool any = it < i1 && e < a.E;
#pragma unroll
    for (int g = 0; g < (ACT ? 2 : 1); g++) {
      ep.sc[g] = ep.bv[g] = 0;
      if (any && n0 + c2 < NO) {
        const size_t at = (size_t)e * N + g * NO + n0 + c2;
        if constexpr (Q8) ep.sc[g] = *(const uint32_t*)((const uint16_t*)a.Bs + at);
        if (a.bias) ep.bv[g] = *(const uint32_t*)((const uint16_t*)a.bias + at);
      }
    }
    // rows past the expert's lie past the end of the buffer: zero
    const __amdgpu_buffer_rsrc_t rb =
        rsrc((const uint8_t*)a.B + (any ? (size_t)e * N * brow : 0), any ? (uint64_t)N * brow : 0);
#pragma unroll
    for (int i = 0; i < SP; i++)
#pragma unroll
      for (int j = 0; j < RT; j++) {
        const int n = n0 + (ACT && j >= RT / 2 ? NO + 16 * (j - RT / 2) : 16 * j) + r;
#pragma unroll
        for (int u = 0; u < U; u++) {
          // int8: 16 bytes at 64 u + 16 h; 16-bit: 32 bytes per (q, h), u = 2 q + s
          const uint32_t at = Q8 ? 64u * u + 16u * h : 128u * (u >> 1) + 32u * h + 16u * (u & 1);
          b[i][j][u] = ld16(rb, ko[i] == kOOB ? kOOB : (uint32_t)n * brow + ko[i] * WB + at);
        }
      }
  };
  uint4 af[SP][TM][4];
  int slot[NO_T], cur = -1;
  float tw[NO_T];
  auto tile = [&](int t) {  // tile t's activations and the slots of the thread's outputs
    cur = t;
    const int b0 = tab_b[t], rows = (tab_b[t + 1] - b0) * bs;
    auto slot_of = [&](int row) -> int {
      if (row >= rows) return -1;
      const int v = a.sorted[b0 * bs + row];
      return v >= 0 && v < a.tis ? v : -1;
    };
#pragma unroll
    for (int m = 0; m < TM; m++) {
      const int s = slot_of(16 * m + r);
#pragma unroll
      for (int i = 0; i < SP; i++)
#pragma unroll
        for (int u = 0; u < 4; u++)
          af[i][m][u] = ld16(ra, s < 0 || ko[i] == kOOB ? kOOB
                                     : ((uint32_t)(s / a.a_div) * (uint32_t)K + ko[i] + 64u * (u >> 1) + 16u * h + 8u * (u & 1)) * 2u);
    }
#pragma unroll
    for (int x = 0; x < NO_T; x++) {
      const int row = (tid + x * NT) / CP;
      slot[x] = row < kTM ? slot_of(row) : -1;
      tw[x] = a.mrw && slot[x] >= 0 ? a.tw[slot[x]] : 1.f;
    }
  };
  auto mul = [&](const BSet& b, const Ep& ep, int it, int p) {
    f32x4 acc[TM][RT];
#pragma unroll
    for (int j = 0; j < RT; j++) {
#pragma unroll
      for (int m = 0; m < TM; m++) acc[m][j] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int i = 0; i < SP; i++)
#pragma unroll
        for (int u = 0; u < 4; u++) {
          uint4 w;
          if constexpr (Q8) {
            const uint4& x = b[i][j][u >> 1];
            w = (u & 1) ? i8x8_to_t<DT>(x.z, x.w) : i8x8_to_t<DT>(x.x, x.y);
          } else {
            w = b[i][j][u];
          }
#pragma unroll
          for (int m = 0; m < TM; m++) acc[m][j] = mfma<DT>(w, af[i][m][u], acc[m][j]);
        }
    }
#pragma unroll
    for (int m = 0; m < TM; m++)
#pragma unroll
      for (int j = 0; j < RT; j++)
        *(f32x4*)&red[p][(wave * kTM + 16 * m + r) * NRP + 16 * j + 4 * h] = acc[m][j];
    __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): the partial sums are written
    ub_barrier();                        // (the next item's loads stay in flight)
    const int t = it / ncol, n0 = (it - t * ncol) * CT, e = tab_e[t];
    if (n0 + c2 < NO) {
#pragma unroll
      for (int x = 0; x < NO_T; x++) {
        if (slot[x] < 0) continue;
        const int row = (tid + x * NT) / CP;
        float v[ACT ? 2 : 1][2];
#pragma unroll
        for (int g = 0; g < (ACT ? 2 : 1); g++) {
          v[g][0] = v[g][1] = 0.f;
#pragma unroll
          for (int w = 0; w < W; w++) {
            const float2 y = *(const float2*)&red[p][(w * kTM + row) * NRP + g * CT + c2];
            v[g][0] += y.x;
            v[g][1] += y.y;
          }
#pragma unroll
          for (int c = 0; c < 2; c++) {
            // fused explicitly and rounded to f32 before T (the compiler would
            // take one rounding here and two there): the same bits with and
            // without the gate
            const float sc = Q8 ? tof<DT>((uint16_t)(ep.sc[g] >> (16 * c))) : 1.f;
            const float bv = tof<DT>((uint16_t)(ep.bv[g] >> (16 * c)));
            v[g][c] = a.bias ? __builtin_fmaf(v[g][c], sc, bv) : v[g][c] * sc;
            if (a.mrw) v[g][c] *= tw[x];
            asm("" : "+v"(v[g][c]));
          }
        }
        uint32_t o = pack2<DT>(v[0][0], v[0][1]);
        if constexpr (ACT) {  // silu_and_mul on the T-rounded GEMM outputs
          const uint32_t up = pack2<DT>(v[1][0], v[1][1]);
          // converted one at a time and kept apart: the f16 product and its
          // rounding are then one instruction, as in k_silu_and_mul
          uint32_t y[2];
#pragma unroll
          for (int c = 0; c < 2; c++) {
            const float gt = tof<DT>((uint16_t)(o >> (16 * c)));
            const float v = gt / (1.f + expf(-gt)) * tof<DT>((uint16_t)(up >> (16 * c)));
            if constexpr (DT == UB_F16) y[c] = __builtin_bit_cast(uint16_t, (_Float16)v);
            else y[c] = pack2<DT>(v, 0.f) & 0xffff;
            asm("" : "+v"(y[c]));
          }
          o = y[0] | y[1] << 16;
        }
        if (e == kElsewhere) o = 0;  // expert handled elsewhere (expert parallel): zero the rows
        if (e != kBadExpert) *(uint32_t*)((uint16_t*)a.C + (size_t)slot[x] * NO + n0 + c2) = o;
      }
    }
    if (tid == 0 && e == kBadExpert) *err = UB_ERR_INDEX;
  };

  BSet w0, w1;
  Ep e0, e1;
  load(w0, e0, i0);
  for (int it = i0; it < i1; it += 2) {
    if (it / ncol != cur) tile(it / ncol);
    load(w1, e1, it + 1);
    mul(w0, e0, it, 0);
    if (it + 1 >= i1) break;  // uniform
    if ((it + 1) / ncol != cur) tile((it + 1) / ncol);
    load(w0, e0, it + 2);
    mul(w1, e1, it + 1, 1);
  }
}

template <int DT, bool Q8, int SP, int OCC>
void launch(const MoeArgs& a, int* err, hipStream_t s) {
  const unsigned g = 128 * OCC;  // workgroups of 2 wavefronts per SIMD: all of them resident
  if (a.act) k_moe_stream<DT, Q8, true, SP, OCC><<<g, NT, 0, s>>>(a, err);
  else k_moe_stream<DT, Q8, false, SP, OCC><<<g, NT, 0, s>>>(a, err);
}

}  // namespace

// Faster than k_moe_gemm while that kernel's workgroups (about one block per
// expert in use and 32 slots, times its 128-row column blocks) leave CUs idle:
// they are then too few to pull the stream, and each walks all of K.  us,
// k_moe_gemm / this one, at that many workgroups; int8 2048 -> 2 x 768 gate/up
// 96: 18.5 / 11.8, 192: 19.1 / 16.5, 288: 19.4 / 18.8, 456: 28.5 / 29.6, its
// down 128: 9.2 / 8.2, 256: 10.1 / 11.6, 384: 12.5 / 13.2; 2048 -> 2 x 1024 32:
// 18.1 / 9.1, 128: 19.0 / 12.7, its down 128: 11.5 / 9.3; 1024 -> 2 x 2048 64:
// 11.6 / 8.7, 256: 13.1 / 12.9, its down 16: 16.6 / 8.1, 80: 16.9 / 12.3; 2048
// -> 2 x 1408 132: 18.9 / 15.3, its down 96: 13.1 / 11.0, 192: 13.4 / 14.0.
// 16-bit weights fill the CUs with half as many workgroups: 2048 -> 2 x 1024
// 32: 14.9 / 10.3, 64: 16.3 / 12.5, 128: 18.1 / 17.9; 2048 -> 2 x 768 96: 15.4 /
// 15.2; 2048 -> 1024 16: 14.6 / 9.7, 80: 15.7 / 16.4; K <= 1024 level.
bool ub_moe_stream_pays(const MoeArgs& a, bool q8) {
  const long blocks = std::min<long>(a.tis, a.E) + a.tis / 32;
  return blocks * ub_cdiv(a.act ? a.N / 2 : a.N, a.act ? 64 : 128) <= (q8 ? 160 : 64);
}

bool ub_moe_stream(const MoeArgs& a, int dt, bool q8, int* err, hipStream_t s) {
  if (!err || 32 % a.bs != 0 || a.N % 8 != 0 || a.K % 128 != 0 || a.K > 128 * W * 2) return false;
  if (!q8 && a.K <= 128 * W) return false;  // k_moe_gemm is as fast
  // the list holds every tile (at most one per block), numbers in 16 bits
  if (max_blocks(a) > kTiles || a.E >= kBadExpert) return false;
  if ((((uintptr_t)a.A | (uintptr_t)a.B) & 15) != 0 ||
      (((uintptr_t)a.C | (uintptr_t)a.Bs | (uintptr_t)a.bias) & 3) != 0)
    return false;
  // 32-bit buffer offsets, also of an item's rows past the end
  const uint64_t arows = (uint64_t)(a.tis + a.a_div - 1) / a.a_div;
  if (arows * a.K * 2 >= 0x80000000ull || (uint64_t)(a.N + 64) * a.K * (q8 ? 1 : 2) >= 0x80000000ull)
    return false;
  auto go = [&](auto dtc) {
    constexpr int DT = decltype(dtc)::value;
    if (!q8) launch<DT, false, 2, 2>(a, err, s);
    else if (a.K <= 128 * W) launch<DT, true, 1, 4>(a, err, s);
    else launch<DT, true, 2, 2>(a, err, s);
  };
  if (dt == UB_BF16) go(std::integral_constant<int, UB_BF16>{});
  else go(std::integral_constant<int, UB_F16>{});
  return true;
}
