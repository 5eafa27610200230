// Row-stationary NT GEMM for the wide projections: K = C = 32 KT channels
// (128, 256 or 384), rows of normalised bf16, few hundred to a few thousand
// output columns.
//   acc = A[64 rows of the wave][K] . W[32 rows of the stage][K]^T
// A workgroup of 4 waves owns 256 rows.  Each wave holds its 64 rows in
// registers for the whole kernel (16 KT VGPRs: 192 at K = 384) and the
// workgroup walks the weight rows, 32 a stage, through two LDS buffers filled
// by direct global -> LDS loads: stage s + 1 streams in while stage s is
// multiplied, one barrier a stage.
//
// Why rows in registers: with K this short a tile that stages both operands
// spends as many LDS cycles as MFMA cycles (64 x 64 per wave) and refills its
// pipeline for every tile.  Here an LDS byte of weights serves 64 rows, half
// the LDS cycles per MFMA, the rows are read once for all their columns, and
// the two workgroups of a CU (256 VGPRs a wave) run out of step, so the
// epilogue of one overlaps the MFMAs of the other.
//
// LDS layout of a stage: KT / 2 sub-tiles of 32 rows x 64 k (128-byte rows),
// slot t of row r holding chunk t ^ (r & 7) (16 bytes), which keeps the
// fragment reads of 8 consecutive rows on distinct bank groups.
#pragma once

#include "common.hpp"

namespace odde {

constexpr int kAsCols = 32;   // weight rows per stage

template <int MB, int KT>
struct AstatShape {
  static constexpr int STAGE = kAsCols * KT * 32;  // bf16 per stage buffer
  static constexpr int LOADS = KT / 2;             // 1 KiB loads per wave and stage
  // two stage buffers and a float per row, in one array: with a second LDS
  // array the compiler tells the two apart, and then waits for every direct
  // load in flight (vmcnt(0)) before a stage's first fragment read
  static constexpr int LDS = 2 * STAGE + 2 * 64 * MB;
  static_assert(KT % 2 == 0, "whole 64-k sub-tiles");
};

template <int KT>
__device__ __forceinline__ float* astat_row_floats(bf16* sm) {
  return reinterpret_cast<float*>(sm + 2 * AstatShape<4, KT>::STAGE);
}

// The lane id, read anew: values derived from the one before the LayerNorm
// would be kept across it, where registers are short, and come back from
// scratch inside the stage loops.
__device__ __forceinline__ int astat_lane() {
  int l;
  asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=v"(l));
  return l;
}

// LayerNorm of the row of MFMA row lane % 16 into row block A_i (statistics
// fp32, two-pass; zeros if !valid, where `row` is any readable row).  kInTurn:
// one block is finished before the next is begun (four at once would need
// 4 x 8 KT floats).
template <bool kInTurn, int KT, typename ZT>
__device__ __forceinline__ void astat_ln_rows(const ZT* row, bool valid,
                                              const float* __restrict__ ln_w,
                                              const float* __restrict__ ln_b, float eps,
                                              Frag<bf16> (&A_i)[KT]) {
  constexpr float kInv = 1.0f / (KT * 32);
  const int g = lane_id() >> 4;
  float x[KT][8];
  float s = 0.f;
#pragma unroll
  for (int t = 0; t < KT; ++t) load8(row + 32 * t + 8 * g, x[t]);
#pragma unroll
  for (int t = 0; t < KT; ++t)
#pragma unroll
    for (int e = 0; e < 8; ++e) s += x[t][e];
  const float mean = group_sum_fast(s) * kInv;
  float q = 0.f;
#pragma unroll
  for (int t = 0; t < KT; ++t)
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      x[t][e] -= mean;
      q += x[t][e] * x[t][e];
    }
  const float rstd = rsqrtf(group_sum_fast(q) * kInv + eps);
#pragma unroll
  for (int t = 0; t < KT; ++t) {
    float w[8], b[8];
    load8(ln_w + 32 * t + 8 * g, w);
    load8(ln_b + 32 * t + 8 * g, b);
#pragma unroll
    for (int e = 0; e < 8; ++e) A_i[t].set(e, valid ? x[t][e] * rstd * w[e] + b[e] : 0.f);
    if constexpr (kInTurn) asm volatile("" : "+v"(A_i[t].v)::"memory");
  }
  if constexpr (kInTurn) __builtin_amdgcn_sched_barrier(0);
}

// Rows of a normalised bf16 matrix: arow(i) is the row of MFMA row lane % 16 in
// row block i.
template <int MB, int KT, typename ARow>
__device__ __forceinline__ void astat_load_rows(ARow arow, int l, Frag<bf16> (&A)[MB][KT]) {
#pragma unroll
  for (int i = 0; i < MB; ++i) {
    const bf16* p = arow(i) + 8 * (l >> 4);
#pragma unroll
    for (int t = 0; t < KT; ++t) A[i][t].load(p + 32 * t);
  }
}

// All rows in registers: what the LayerNorm had to spill comes back here and
// not inside the stage loops.
template <int MB, int KT>
__device__ __forceinline__ void astat_rows_ready(Frag<bf16> (&A)[MB][KT]) {
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int t = 0; t < KT; ++t) asm volatile("" : "+v"(A[i][t].v));
}

// l: astat_lane().  acc[i][j] = row block i times weight rows 16 j .. 16 j + 15 of the stage.
//   kPairCols = true : column (lane % 16) is the row, its 4 values are weight
//                      rows 16 j + 4 (lane / 16) + e;
//   kPairCols = false: the transpose.
// A0 meets the first 16 weight rows, A1 the others.
// AH weight fragments are read ahead.
template <int MB, int KT, bool kPairCols, int AH = 8 / MB>
__device__ __forceinline__ void astat_mult(const bf16* buf, int l, const Frag<bf16> (&A0)[MB][KT],
                                           const Frag<bf16> (&A1)[MB][KT], f32x4 (&acc)[MB][2]) {
  const int g = l >> 4, r16 = l & 15;
  const bf16* p0 = buf + r16 * 64 + ((g ^ (r16 & 7)) * 8);        // even k steps
  const bf16* p1 = buf + r16 * 64 + (((4 + g) ^ (r16 & 7)) * 8);  // odd ones
  // fragment u = (k step u / 2, weight block u % 2): the one read while u is
  // multiplied is u + AH, by default 8 MFMAs ahead
  constexpr int NB = AH + 1;
  Frag<bf16> b[NB];
  auto read = [&](int u) {
    const int t = u >> 1;
    b[u % NB].load(((t & 1) ? p1 : p0) + (t >> 1) * (kAsCols * 64) + (u & 1) * (16 * 64));
  };
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int u = 0; u < AH; ++u) read(u);
#pragma unroll
  for (int u = 0; u < 2 * KT; ++u) {
    if (u + AH < 2 * KT) read(u + AH);
#pragma unroll
    for (int i = 0; i < MB; ++i) {
      const Frag<bf16>& row = (u & 1) ? A1[i][u >> 1] : A0[i][u >> 1];
      if constexpr (kPairCols) mma(acc[i][u & 1], b[u % NB], row);
      else mma(acc[i][u & 1], row, b[u % NB]);
    }
  }
  __builtin_amdgcn_sched_group_barrier(0x100, AH, 0);
#pragma unroll
  for (int u = 0; u + AH < 2 * KT; ++u) {
    __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
    __builtin_amdgcn_sched_group_barrier(0x008, MB, 0);
  }
  __builtin_amdgcn_sched_group_barrier(0x008, AH * MB, 0);
}

template <int MB, int KT, bool kPairCols>
__device__ __forceinline__ void astat_mult(const bf16* buf, int l, const Frag<bf16> (&A)[MB][KT],
                                           f32x4 (&acc)[MB][2]) {
  astat_mult<MB, KT, kPairCols>(buf, l, A, A, acc);
}

// Stages 0 .. nst - 1.  wsrc(st): uniform pointer to the first of the weight
// rows that fill this wave's LDS rows 8 w .. 8 w + 7 of stage st; row_of
// (lane's LDS row, 0 .. 7) its row relative to that pointer (at most 11).
// stage(st, buf) multiplies and stores; it is called by live waves only and
// issues kStores vector stores or more, after which the next stage's loads
// are the only older ones it has to wait for.  sm holds two stage buffers;
// l: astat_lane().  kStores < 0: any number of them, on three stage buffers:
// the loads run two stages ahead, and a stage waits until no more operations
// are out than the next stage's loads.
template <int KT, int kStores, typename WSrc, typename RowOf, typename Stage>
__device__ __forceinline__ void astat_loop(int nst, bool live, bf16* sm, int l, WSrc wsrc, RowOf row_of,
                                           Stage stage) {
  using S = AstatShape<4, KT>;  // the stages do not depend on MB
  constexpr int C = KT * 32, NB = kStores < 0 ? 3 : 2;
  const int lr = l >> 3;
  const int w = __builtin_amdgcn_readfirstlane(wave_id());
  const uint32_t voff = (uint32_t)(row_of(lr) * C + (((l & 7) ^ lr) * 8)) * (uint32_t)sizeof(bf16);
  auto issue = [&](int st) {
    const bf16* src = wsrc(st);
    bf16* dst = sm + (st % NB) * S::STAGE + w * 512;
#pragma unroll
    for (int k = 0; k < S::LOADS; ++k)
      buffer_load_lds16(src, 12 * C * (uint32_t)sizeof(bf16), dst + k * (kAsCols * 64), voff,
                        (uint32_t)k * 128);
  };
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  barrier_nofence();  // the buffers are free (an earlier loop's last stage)
  issue(0);
  if constexpr (kStores < 0) {
    if (nst > 1) issue(1);
    for (int st = 0; st < nst; ++st) {
      if (st + 1 < nst) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(S::LOADS) : "memory");
      else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // own reads of stage st - 1 done
      barrier_nofence();
      if (st + 2 < nst) issue(st + 2);  // the buffer last read in stage st - 1
      __builtin_amdgcn_sched_barrier(0);
      if (live) stage(st, sm + (st % NB) * S::STAGE);
    }
    return;
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  for (int st = 0; st < nst; ++st) {
    if (st) {  // this wave's loads of stage st landed; its last stores may not have
      if (live) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kStores < 0 ? 0 : kStores) : "memory");
      else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // own reads of stage st - 1 done
    barrier_nofence();
    if (st + 1 < nst) issue(st + 1);  // the buffer last read in stage st - 1
    __builtin_amdgcn_sched_barrier(0);  // the loads before the stage's stores
    if (live) stage(st, sm + (st & 1) * S::STAGE);
  }
}

// Column split of a row-stationary grid: 1, 2, 4, .. workgroups share a row
// tile's `stages` (the split divides them) until the grid holds `want`
// workgroups.  Every split reads its rows again, and with a fused LayerNorm
// normalises them again, which soon costs more than idle CUs do: the callers
// say where the line lies.
inline int astat_csplit(int row_tiles, int stages, int want) {
  int s = 1;
  while (row_tiles * s < want && stages % (2 * s) == 0) s *= 2;
  return s;
}

}  // namespace odde
