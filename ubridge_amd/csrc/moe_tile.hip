// moe_tile.hip -- grouped expert GEMM on tiles of 32, 64 or 128 rows, for
// batches that fill them (gfx950).
//
// The same operation as k_moe_gemm (moe.hip), which gives every sorted block
// of 32 rows its own workgroup per column tile: a stream of the weights while
// an expert has about one block, but at prefill sizes an expert has tens of
// blocks, and then each of them fetches the expert's weights again, widens
// every int8 weight again for a single row of MFMA tiles, and fills one 32 x
// 32 tile per wavefront.  Here the blocks of one expert are taken together in
// tiles of kTM = 32, 64 or 128 rows, so one widened weight fragment feeds up
// to 4 MFMAs and the weights are fetched a quarter as often; with few rows (32)
// what is left is the persistent grid, whose loads do not stop between tiles.
//
//  * Persistent grid, two workgroups of 4 wavefronts per CU (so the two
//    wavefronts of a SIMD are not held in step by one barrier; one workgroup
//    of 8 measured 1-10% slower).  Each workgroup first cuts the sorted
//    blocks into tiles itself (two scans over experts_ids; consecutive
//    blocks of one expert, at most kTM rows) and keeps the list in LDS, then
//    walks (tile, column block) pairs.
//  * Tile kTM rows x 256 weight rows; a wavefront owns 64 weight rows and
//    all token rows: up to 4 x 2 tiles of v_mfma_f32_32x32x16.  A lane's two
//    columns are adjacent, so a store covers 128-byte runs of two rows.
//    Tiles with at most 96 / 64 / 32 rows run the loop with 3 / 2 / 1 row
//    tiles of 32.  With the gated output a wavefront's two column tiles are the
//    gate and the up rows of the same 32 columns, so silu(g) u is lane-local.
//  * Both operands reach LDS by direct-to-LDS loads through a ring of NS
//    K-step stages (A rows gathered by slot), XOR-swizzled in 16-byte units;
//    within a 32-k pair of MFMAs a lane feeds 16 consecutive k on both
//    operands, so int8 fragments are one 16-byte read per pair.  LDS reads and
//    the widening run one 16-k substep ahead of the MFMAs (reads two ahead
//    spilled), the one barrier per K-step sits before the last substep.  The
//    next pair's rows are fetched during the K loop and its first stages are
//    in flight during the epilogue.
//  * int8 enters as q + 128 (exact in T) and 128 x the sum of the A row is
//    subtracted from the f32 sums, in k_moe_gemm's order of additions: an
//    output has the same bits from every tile height and from that kernel,
//    whatever batch its token is in.  A wavefront sums the rows of one row
//    tile only (its first: the wavefronts start at different row tiles) and
//    the sums meet in LDS.  All four wavefronts summing all rows took 564 us
//    for the whole 4096-token layer below, this way 472, the signed weights
//    with nothing to subtract 472 (but other bits than k_moe_gemm's: 3e-4 of
//    relative 2-norm in a bf16 layer).
//  * scale, bias and routed weight are applied to the f32 sums as in
//    k_moe_gemm.
//
// MI355X, 128 experts of 2048 -> 2 x 768 -> 2048, top-8, us in a graph of
// launches with weights from HBM (k_moe_gemm / 64-row / 128-row tiles), int8 at
// 1024 tokens: gate/up 203 / 124 / 137, down 132 / 77 / 81; at 4096: 582 / -
// / 281, 423 / - / 166 (735 / 620 TFLOP/s); bf16 (k_moe_gemm / 128-row tiles)
// at 1024: 263 / 212, 205 / 110; at 4096: 751 / 348, 704 / 198.  At 4096 int8
// tokens the gate/up launch without its epilogue took 25 us less, with every
// load an L2 hit 34 us less, without the int8 conversion (of the signed
// weights) 26 us less and without all three 200 us: MFMA issue and LDS reads in
// step with a barrier per K-step hold most of it.
#include "lds_dma.h"
#include "moe_dev.h"

#include <algorithm>
#include <type_traits>

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int NWV = 4, kCols = 64 * NWV;  // wavefronts, weight rows of a workgroup
constexpr int kTiles = 512;  // tiles listed in LDS at a time

template <int DT>
__device__ __forceinline__ f32x16 mfma(const uint4& a, const uint4& b, const f32x16& c) {
  if constexpr (DT == UB_BF16)
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a),
                                                   __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a),
                                                  __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
}

template <int DT, bool Q8, int kTM, int BK, int NS>
__global__ void __launch_bounds__(64 * NWV) __attribute__((amdgpu_waves_per_eu(2, 2)))
k_moe_tile(MoeArgs a, int* err) {
  constexpr int NT = 64 * NWV, BN = kCols, SS = BK / 16;
  constexpr int WB = Q8 ? 1 : 2;
  constexpr int RA = BK * 2, UA = RA / 16;    // A row bytes / 16-byte units
  constexpr int RB = BK * WB, UB = RB / 16;   // weight row bytes / units
  constexpr int AB = kTM * RA, BB = BN * RB, STB = AB + BB;
  constexpr int NA = AB / 1024 / NWV, NB = BB / 1024 / NWV, NL = NA + NB;  // loads per wave, stage
  static_assert(kTM == 128 || kTM == 64 || kTM == 32, "rows of a tile");
  static_assert(AB % (1024 * NWV) == 0 && BB % (1024 * NWV) == 0, "loads split evenly");
  static_assert(Q8 ? BK == 64 : BK == 32, "substep schedule");
  constexpr int RPWA = RA >= 256 ? 1 : 256 / RA, RPWB = RB >= 256 ? 1 : 256 / RB;
  auto swa = [](int r) { return (r / RPWA) % UA; };
  auto swb = [](int r) { return (r / RPWB) % UB; };
  __shared__ __attribute__((aligned(16))) uint8_t smem[NS * STB];
  __shared__ uint16_t tab_b[kTiles + 1], tab_e[kTiles];  // first block, expert (>= E: none)
  __shared__ __attribute__((aligned(16))) int srow[2][kTM];   // the tile's slots, -1: padding
  __shared__ __attribute__((aligned(16))) float stw[2][kTM];  // their routed weights
  __shared__ float ssc[2][Q8 ? BN : 1], sbv[2][BN];           // scale / bias of the weight rows
  __shared__ __attribute__((aligned(16))) float srsum[2][Q8 ? kTM : 4];  // int8: sums of the A rows
  __shared__ int wsum[2][NWV];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int K = a.K, N = a.N, bs = a.bs;
  // Output columns: BN per workgroup, or with act BN / 2
  const int NO = a.act ? N / 2 : N, CT = a.act ? BN / 2 : BN;
  const int ncol = (NO + CT - 1) / CT;
  const int l32 = lane & 31, kh = lane >> 5;
  const int nk = K / BK;
  const uint64_t brow = (uint64_t)K * WB;
  const uint32_t sbase = ub_lds_addr(smem);
  const int arows = (a.tis + a.a_div - 1) / a.a_div;
  const ub_u32x4 ra = ub_desc(a.A, (uint64_t)arows * K * 2);
  // weight row of tile row r (wavefront r / 64, column tile j = (r / 32) % 2)
  // and whether its output column exists: with act j = 0 / 1 are the gate and
  // up rows of one output column, otherwise two adjacent columns (N is even)
  auto wrow_of = [&](int r, int n0) -> int {
    if (!a.act) return n0 + (r & ~63) + 2 * (r & 31) + ((r >> 5) & 1);
    const int oc = n0 + 32 * (r >> 6) + (r & 31);
    return (r & 32) ? NO + oc : oc;
  };
  auto wok = [&](int r, int n0) -> bool {
    return a.act ? n0 + 32 * (r >> 6) + (r & 31) < NO : n0 + (r & ~63) + 2 * (r & 31) < N;
  };
  // The workgroup's p-th pair: each round of the grid is handed out so that
  // the workgroups of one XCD (i % 8) take neighbours, which share an
  // expert's weights or a tile's rows in that XCD's L2.
  const int grid = gridDim.x;
  int total = 0;
  auto pair_of = [&](int p) -> int {
    const int base = p - (int)blockIdx.x;
    return base + grid <= total ? base + ((int)blockIdx.x & 7) * (grid >> 3) + ((int)blockIdx.x >> 3) : p;
  };
  // What thread tid holds of pair q for its tile: row tid's slot, weight row
  // tid's scale and bias
  struct Row {
    int slot;
    uint16_t sc, bv;
    float tw;
  };
  auto fetch = [&](int q) -> Row {
    Row x{-1, 0, 0, 1.f};
    const int t = q / ncol, b = tab_b[t], e = tab_e[t], n0 = (q % ncol) * CT;
    if (tid < kTM && tid < (tab_b[t + 1] - b) * bs) {
      const int v = a.sorted[b * bs + tid];
      if (v >= 0 && v < a.tis) {
        x.slot = v;
        if (a.mrw) x.tw = a.tw[v];
      }
    }
    if (e < a.E && wok(tid, n0)) {
      const size_t at = (size_t)e * N + wrow_of(tid, n0);
      if constexpr (Q8) x.sc = ((const uint16_t*)a.Bs)[at];
      if (a.bias) x.bv = ((const uint16_t*)a.bias)[at];
    }
    return x;
  };
  auto put = [&](const Row& x, int buf) {
    if (tid < kTM) {
      srow[buf][tid] = x.slot;
      stw[buf][tid] = x.tw;
    }
    if constexpr (Q8) ssc[buf][tid] = tof<DT>(x.sc);
    sbv[buf][tid] = tof<DT>(x.bv);
  };

  // fragment addresses inside a stage: 16-byte unit of 16-k substep s
  uint32_t aoff[SS], boff[SS];
#pragma unroll
  for (int s = 0; s < SS; s++) {
    const int c = 4 * (s >> 1) + 2 * kh + (s & 1);
    aoff[s] = l32 * RA + ((c ^ swa(l32)) << 4);
    const int r = wave * 64 + l32;
    boff[s] = AB + r * RB + (((Q8 ? 2 * (s >> 1) + kh : c) ^ swb(r)) << 4);
  }

  // lists of more than kTiles tiles are worked off in windows
  for (int first = 0, tiles = 1; first < tiles; first += kTiles) {
  tiles = moe_tile_list<NWV>(a, kTM / bs, first, kTiles, tab_b, tab_e, wsum);
  total = min(tiles - first, kTiles) * ncol;
  int p = blockIdx.x;
  if (p >= total) {
    __syncthreads();  // as the workgroups with pairs: the list is free
    continue;
  }
  // Loads of pair q (its rows in srow[buf]); returns the rows to multiply, 0 where
  // there is nothing to multiply (no rows, an expert elsewhere).
  uint32_t voA[NA], voB[NB];
  ub_u32x4 rb = {0, 0, 0, 0};
  auto issue = [&](int kt, uint32_t st) {
#pragma unroll
    for (int j = 0; j < NB; j++)
      ub_lds_load16_at(rb, st + AB + (j * NWV + wave) * 1024, voB[j], (uint32_t)kt * RB);
#pragma unroll
    for (int j = 0; j < NA; j++)
      ub_lds_load16_at(ra, st + (j * NWV + wave) * 1024, voA[j], (uint32_t)kt * RA);
  };
  auto start = [&](int q, int buf) -> int {
    const int e = tab_e[q / ncol], n0 = (q % ncol) * CT;
    // rows up to the last real one (padding may lie before it, where two
    // neighbouring experts are mapped to the same weights)
    const uint64_t lo = __ballot(lane < kTM && srow[buf][lane] >= 0);
    const uint64_t hi = kTM > 64 ? __ballot(srow[buf][64 % kTM + lane] >= 0) : 0;
    const int nreal = hi ? 128 - __clzll(hi) : lo ? 64 - __clzll(lo) : 0;
    if (e >= a.E || nreal == 0) return 0;
    rb = ub_desc((const uint8_t*)a.B + (size_t)e * N * brow, (uint64_t)N * brow);
#pragma unroll
    for (int j = 0; j < NA; j++) {
      const int u = (j * NWV + wave) * 64 + lane, r = u / UA, c = (u % UA) ^ swa(r);
      const int s = srow[buf][r];
      voA[j] = s >= 0 ? (uint32_t)(((size_t)(s / a.a_div) * K + 8 * c) * 2) : kDmaOOB;
    }
#pragma unroll
    for (int j = 0; j < NB; j++) {
      const int u = (j * NWV + wave) * 64 + lane, r = u / UB, c = (u % UB) ^ swb(r);
      voB[j] = wok(r, n0) ? (uint32_t)((size_t)wrow_of(r, n0) * brow + 16 * c) : kDmaOOB;
    }
#pragma unroll
    for (int j = 0; j < NS; j++)
      if (j < nk) issue(j, sbase + j * STB);
    return nreal;
  };

  put(fetch(pair_of(p)), 0);
  __syncthreads();
  int nreal = start(pair_of(p), 0);
  for (int buf = 0; p < total; p += grid, buf ^= 1) {
    const int q = pair_of(p), n0 = (q % ncol) * CT;
    const bool more = p + grid < total;
    const int qn = more ? pair_of(p + grid) : 0;
    Row nrow{-1, 0, 0, 1.f};
    if (more) nrow = fetch(qn);
    // once every wavefront is past its last read of the ring: the next pair's
    // rows and first loads, in flight during this pair's epilogue
    int nnext = 0;
    auto next = [&]() {
      if (more) put(nrow, buf ^ 1);
      __syncthreads();
      if (more) nnext = start(qn, buf ^ 1);
    };
    auto run = [&](auto tmc) {
      constexpr int TM = decltype(tmc)::value;
      f32x16 acc[TM][2];
#pragma unroll
      for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < 2; j++)
#pragma unroll
          for (int r = 0; r < 16; r++) acc[i][j][r] = 0.f;
      uint4 af[2][TM], bf[2][2], bw[2];
      // int8: each wavefront starts with another row tile (its i-th is tile
      // (i + wave) % TM), whose rows it sums; 16-bit: in order.  Opaque, or an
      // address per tile and substep would be kept and spilled (4096 tokens:
      // 489 us a layer, 472 this way)
      uint32_t tile_of[TM];
#pragma unroll
      for (int i = 0; i < TM; i++) {
        tile_of[i] = Q8 ? (uint32_t)(i + wave) % TM : i;
        if constexpr (Q8) asm("" : "+s"(tile_of[i]));
      }
      float rsum = 0.f;  // sum of the lane's row of tile_of[0] over its k half
      auto read_a = [&](uint32_t st, int s) {
#pragma unroll
        for (int i = 0; i < TM; i++) af[s & 1][i] = ub_lds_read16(st + aoff[s] + 32 * RA * tile_of[i]);
      };
      auto read_b = [&](uint32_t st, int s, uint4 (&to)[2]) {
#pragma unroll
        for (int j = 0; j < 2; j++) to[j] = ub_lds_read16(st + boff[s] + 32 * RB * j);
      };
      auto mfmas = [&](int s) {
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
          for (int j = 0; j < 2; j++) acc[i][j] = mfma<DT>(af[s & 1][i], bf[s & 1][j], acc[i][j]);
      };
      // wait for stage t + 1, free stage t for the loads of step t + NS
      auto turn = [&](int kt, uint32_t cur) {
        __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): the reads of `cur` are done
        if (NS > 2 && kt + NS - 1 < nk) ub_wait_vmcnt<(NS - 2) * NL>();
        else ub_wait_vmcnt<0>();
        ub_barrier();
        if (kt + NS < nk) issue(kt + NS, cur);
      };
      // Stage 0 has landed.  The previous pair's stores were issued after
      // these loads, so the count only makes the wait stricter.
      if (nk >= NS) ub_wait_vmcnt<(NS - 1) * NL>();
      else ub_wait_vmcnt<0>();
      ub_barrier();
      if constexpr (Q8) {
        // widen substep s's 8 k from the pair's raw words
        auto widen = [&](int s) {
#pragma unroll
          for (int j = 0; j < 2; j++) {
            const uint4& w = bw[j];
            bf[s & 1][j] = (s & 1) ? i8x8_to_t_off<DT>(w.z, w.w) : i8x8_to_t_off<DT>(w.x, w.y);
            // pinned here: the converts would otherwise sink to the MFMAs
            asm volatile("" : "+v"(bf[s & 1][j].x), "+v"(bf[s & 1][j].y), "+v"(bf[s & 1][j].z), "+v"(bf[s & 1][j].w));
          }
        };
        // the fragments' sum, pinned here as well (the sums would otherwise
        // sink to the end of the K-step and keep the fragments)
        auto add_rows = [&](int s) {
          rsum = frag_sum<DT>(af[s & 1][0], rsum);
          asm volatile("" : "+v"(rsum));
        };
        // one substep's instructions interleaved: MFMA, LDS read, VALU
        auto sched = [&](auto nreads) {
          constexpr int nread = decltype(nreads)::value;
#pragma unroll
          for (int m = 0; m < 2 * TM; m++) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x100, (nread + 2 * TM - 1) / (2 * TM), 0);
            __builtin_amdgcn_sched_group_barrier(0x002, 16 / TM, 0);
          }
          __builtin_amdgcn_sched_barrier(0);
        };
        read_b(sbase, 0, bw);
        read_a(sbase, 0);
        widen(0);
        for (int k0 = 0; k0 < nk; k0 += NS)
#pragma unroll
          for (int u = 0; u < NS; u++) {  // stage u: constant LDS offsets
            const int kt = k0 + u;
            if (u && kt >= nk) break;
            const uint32_t cur = sbase + u * STB, nxt = sbase + (u + 1) % NS * STB;
            read_a(cur, 1);
            mfmas(0);
            add_rows(0);
            widen(1);
            sched(std::integral_constant<int, TM>{});
            read_b(cur, 2, bw);
            read_a(cur, 2);
            mfmas(1);
            add_rows(1);
            widen(2);
            sched(std::integral_constant<int, TM + 2>{});
            read_a(cur, 3);
            mfmas(2);
            add_rows(2);
            widen(3);
            sched(std::integral_constant<int, TM>{});
            turn(kt, cur);
            read_b(nxt, 0, bw);
            read_a(nxt, 0);
            mfmas(3);
            add_rows(3);
            widen(0);
            sched(std::integral_constant<int, TM + 2>{});
          }
      } else {
        auto sched = [&]() {
#pragma unroll
          for (int m = 0; m < 2 * TM; m++) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x100, (TM + 2 + 2 * TM - 1) / (2 * TM), 0);
          }
          __builtin_amdgcn_sched_barrier(0);
        };
        read_b(sbase, 0, bf[0]);
        read_a(sbase, 0);
        for (int k0 = 0; k0 < nk; k0 += NS)
#pragma unroll
          for (int u = 0; u < NS; u++) {
            const int kt = k0 + u;
            if (u && kt >= nk) break;
            const uint32_t cur = sbase + u * STB, nxt = sbase + (u + 1) % NS * STB;
            read_b(cur, 1, bf[1]);
            read_a(cur, 1);
            mfmas(0);
            sched();
            turn(kt, cur);
            read_b(nxt, 0, bf[0]);
            read_a(nxt, 0);
            mfmas(1);
            sched();
          }
      }
      if constexpr (Q8) {  // read back behind the barrier of next()
        rsum += __shfl_xor(rsum, 32);
        if (wave < TM && kh == 0) srsum[buf][32 * wave + l32] = rsum;
      }
      next();
      // epilogue: register r of tile (i, j): token row 32 tile_of[i] + 8 (r /
      // 4) + 4 kh + r % 4, tile row wave 64 + 32 j + l32 of the weight
      uint16_t* C = (uint16_t*)a.C;
      const bool bias = a.bias != nullptr, mrw = a.mrw != 0;
      float sc[2], bv[2];
#pragma unroll
      for (int j = 0; j < 2; j++) {
        sc[j] = Q8 ? ssc[buf][wave * 64 + 32 * j + l32] : 1.f;
        bv[j] = sbv[buf][wave * 64 + 32 * j + l32];
      }
      const int oc = a.act ? n0 + 32 * wave + l32 : n0 + 64 * wave + 2 * l32;
      if (oc < NO) {
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
          for (int g = 0; g < 4; g++) {
            const int r0 = 32 * tile_of[i] + 8 * g + 4 * kh;
            const int4 s4 = *(const int4*)&srow[buf][r0];
            const float4 t4 = *(const float4*)&stw[buf][r0];
            const float4 q4 = Q8 ? *(const float4*)&srsum[buf][r0] : make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
            for (int x = 0; x < 4; x++) {
              const int s = x == 0 ? s4.x : x == 1 ? s4.y : x == 2 ? s4.z : s4.w;
              const float tw = x == 0 ? t4.x : x == 1 ? t4.y : x == 2 ? t4.z : t4.w;
              const float rs = x == 0 ? q4.x : x == 1 ? q4.y : x == 2 ? q4.z : q4.w;
              float v[2];
#pragma unroll
              for (int j = 0; j < 2; j++) {
                v[j] = acc[i][j][4 * g + x];
                if constexpr (Q8) v[j] = (v[j] - 128.f * rs) * sc[j];
                if (bias) v[j] += bv[j];
                if (mrw) v[j] *= tw;
              }
              const uint32_t o = pack2<DT>(v[0], v[1]);
              if (a.act) {  // silu_and_mul on the T-rounded GEMM outputs
                const float gt = tof<DT>((uint16_t)(o & 0xffff)), up = tof<DT>((uint16_t)(o >> 16));
                const uint16_t y = (uint16_t)(pack2<DT>(gt / (1.f + expf(-gt)) * up, 0.f) & 0xffff);
                if (s >= 0) C[(size_t)s * NO + oc] = y;
              } else if (s >= 0) {
                *(uint32_t*)(C + (size_t)s * NO + oc) = o;
              }
            }
          }
      }
    };
    auto rows = [&](auto tmc) {  // one loop per number of row tiles
      if (nreal <= 32 * (decltype(tmc)::value - 1)) return false;
      run(tmc);
      return true;
    };
    bool done = false;
    if constexpr (kTM == 128)
      done = rows(std::integral_constant<int, 4>{}) || rows(std::integral_constant<int, 3>{}) ||
             rows(std::integral_constant<int, 2>{});
    if constexpr (kTM == 64) done = rows(std::integral_constant<int, 2>{});
    if (!done) done = rows(std::integral_constant<int, 1>{});
    if (!done) {
      __syncthreads();  // every wavefront is past the epilogue that reads the other row buffer
      const int e = tab_e[q / ncol];
      if (e == kElsewhere) {  // expert handled elsewhere (expert parallel): zero the rows
        for (int i = tid; i < kTM * CT; i += NT) {
          const int s = srow[buf][i / CT], n = n0 + i % CT;
          if (s >= 0 && n < NO) ((uint16_t*)a.C)[(size_t)s * NO + n] = 0;
        }
      } else if (tid == 0 && e == kBadExpert) {
        *err = UB_ERR_INDEX;
      }
      next();
    }
    nreal = nnext;
  }
  __syncthreads();  // every wavefront is done with the list and the rows
  }
}

template <int DT, bool Q8, int kTM, int BK, int NS>
void launch(const MoeArgs& a, int* err, hipStream_t s) {
  const int NO = a.act ? a.N / 2 : a.N;
  const long pairs = (long)max_blocks(a) * ub_cdiv(NO, a.act ? kCols / 2 : kCols);  // at most
  const unsigned g = (unsigned)std::min<long>(ub_cdiv(pairs, 8) * 8, 512);
  k_moe_tile<DT, Q8, kTM, BK, NS><<<g, 64 * NWV, 0, s>>>(a, err);
}

}  // namespace

// Rows of the tiles where they pay, 0 where k_moe_gemm is faster; from sizes
// known on the host: an expert's average rows r = slots / E and the (tile,
// column block) pairs, about slots / rows + E / 2 tiles (at least one per
// expert).  Whole layers of 128 / 64 / 8 experts (top-8 2048 -> 2 x 768, top-6
// 2048 -> 2 x 1408, top-2 4096 -> 2 x 1024), us:
//  * taller tiles need rows to fill them.  int8, 128 experts, k_moe_gemm / 32 /
//    64 / 128 rows in turn in one run at r = 2: 123 / 128 / 130 / 147, 3: 133 /
//    131 / 134 / 151, 8: 147 / 141 / 143 / 160, 16: 163 / 165 / 159 / 171, 24:
//    178 / 167 / 173 / 176, 32: 195 / 183 / 185 / 186, 48: 229 / 217 / 190 / 210,
//    64: 267 / 267 / 218 / 229, 96: 351 / 338 / 263 / 246, 128: 441 / 439 / 323 /
//    284; 64 experts at r = 3: 124 / 121 / 123 / 139, 12: 138 / 132 / 133 / 147,
//    24: 160 / 156 / 147 / 156, 48: 212 / 202 / 179 / 182: within 5% of the best
//    up to 64 rows and 7% at 96, as the tiles come out.  16-bit (no widening to
//    share) k_moe_gemm / 64 / 128 rows, 128 experts at r = 4: 247 / 247 / 252, 8:
//    264 / 266 / 273, 16: 279 / 275 / 282, 24: 286 / 301 / 290, 38: 320 / 312 /
//    316, 50: 360 / 327 / 339, 63: 400 / 341 / 350; the two GEMMs alone (64 / 128)
//    at r = 75: 331 / 326, 94: 380 / 344, 150: 487 / 417; 64 experts at r = 14: 235 /
//    239, 28: 260 / 246, 47: 283 / 263, 94: 359 / 316: 64 rows are up to 3% faster
//    below 64 rows of 128 experts, 128 rows up to 20% beyond and for 64 experts.
//  * at least 160 pairs (128 int8 rows: 512): each walks all of K, so few of
//    them leave the chip idle.  8 experts, int8 layer, k_moe_gemm / 32 / 64 / 128
//    rows at r = 32 (gate/up 96 / 64 / 64 pairs) 64 / 71 / 81 / 99, 64 (160 / 96 /
//    64) 84 / 78 / 83 / 111, 128 (- / 160 / 96) 121 / 104 / 92 / 117, 256 (- / 288 /
//    160) 184 / 148 / 129 / 133.  16-bit calls with too few pairs of 128 rows take
//    64: 8 experts at r = 175 (gate/up 119 / 206 pairs), the two GEMMs with 128 / 64
//    rows, 121 / 108.
int ub_moe_tile_rows(const MoeArgs& a, bool q8) {
  const long cols = ub_cdiv(a.act ? a.N / 2 : a.N, a.act ? kCols / 2 : kCols);
  auto pays = [&](int rows, int r, long pairs) {
    return rows % a.bs == 0 && a.tis >= (long)a.E * r &&
           std::max<long>(a.E, a.tis / rows + a.E / 2) * cols >= pairs;
  };
  if (q8) return pays(128, 112, 512) ? 128 : pays(64, 24, 160) ? 64 : pays(32, 3, 160) ? 32 : 0;
  return pays(128, 8, 160) ? 128 : pays(64, 8, 160) ? 64 : 0;
}

bool ub_moe_tile(const MoeArgs& a, int rows, int dt, bool q8, int* err, hipStream_t s) {
  if (!err || rows % a.bs != 0 || a.N % 8 != 0 || a.K % 64 != 0) return false;
  // the list holds block and expert numbers in 16 bits
  if (max_blocks(a) >= 65535 || a.E >= kBadExpert) return false;
  if ((((uintptr_t)a.A | (uintptr_t)a.B) & 15) != 0 || ((uintptr_t)a.C & 3) != 0) return false;
  const uint64_t arows = (uint64_t)(a.tis + a.a_div - 1) / a.a_div;
  if (arows * a.K * 2 >= 0x80000000ull || (uint64_t)a.N * a.K * (q8 ? 1 : 2) >= 0x80000000ull)
    return false;  // 32-bit buffer offsets
  auto go = [&](auto dtc) {
    constexpr int DT = decltype(dtc)::value;
    if (q8) {
      if (rows == 128) launch<DT, true, 128, 64, 2>(a, err, s);
      else if (rows == 64) launch<DT, true, 64, 64, 3>(a, err, s);
      else launch<DT, true, 32, 64, 3>(a, err, s);
    } else {
      if (rows == 128) launch<DT, false, 128, 32, 3>(a, err, s);
      else launch<DT, false, 64, 32, 3>(a, err, s);
    }
  };
  if (dt == UB_BF16) go(std::integral_constant<int, UB_BF16>{});
  else go(std::integral_constant<int, UB_F16>{});
  return true;
}
