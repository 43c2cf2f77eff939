// The K loop of the bf16 / fp32 GEMMs whose operands both pass through an LDS
// ring: 4 waves (2 x 2) share a tile of 16 MFC rows by 128 weight rows (the
// mid-size experts launch, the model's projections).
#pragma once

#include "common.h"
#include "ring_blocks.h"

#include <type_traits>

namespace mep {
namespace {

// 16x16x32 bf16 MFMA with the accumulator in VGPRs; src0 = weight
// fragment, src1 = row fragment, so the result is C^T (lane: one row, 4
// consecutive columns).  mfma_first starts a new accumulation (C operand 0).
__device__ __forceinline__ void mfma_acc(f32x4& acc, const u32x4& w, const u32x4& a) {
  asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+v"(acc) : "v"(w), "v"(a));
}
__device__ __forceinline__ void mfma_first(f32x4& acc, const u32x4& w, const u32x4& a) {
  asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, 0" : "=v"(acc) : "v"(w), "v"(a));
}
// Orders later reads of `acc` after every earlier volatile asm (an empty asm
// that claims to rewrite it).  AMDGPU register constraints live in device
// functions only: in a kernel body the host pass parses them as x86 ones.
__device__ __forceinline__ void pin_acc(f32x4& acc) { asm volatile("" : "+v"(acc)); }

// One K-step (64 bytes of every row) of a fragment pair: 32 bf16 in one MFMA,
// or 16 floats in four, MFMA q on elements 4 lg + q of the lane groups (the
// order of grouped_gemm_kernel).
template <int DT>
__device__ __forceinline__ void ring_mfma(f32x4& acc, const u32x4& w, const u32x4& a) {
  if constexpr (DT == MEP_DTYPE_BF16) {
    mfma_acc(acc, w, a);
  } else {
#pragma unroll
    for (int q = 0; q < 4; ++q)
      asm volatile("v_mfma_f32_16x16x4_f32 %0, %1, %2, %0" : "+v"(acc) : "v"(w[q]), "v"(a[q]));
  }
}

namespace ring {
constexpr int NT = 256;
constexpr int WF = 8;                         // weight fragments of a workgroup: 128 weight rows
constexpr int WP = WF / 2;                    // copy passes of 32 weight rows
constexpr int lds_bytes(int mfc) { return 4 * (mfc + WF) * 1024; }

// A thread's part of a copy pass (32 rows, one 128-byte line of each, 8 lanes
// per row): row 16 half + row16, 16-byte chunk `chunk` of the line.
struct Copy {
  int row16, half, chunk;
  __device__ __forceinline__ Copy() {
    const int tid = threadIdx.x;
    row16 = ((tid >> 3) & 3) * 4 + ((tid >> 5) & 3);
    half = tid >> 7;
    chunk = tid & 7;
  }
};
}  // namespace ring

// acc[i][j] = the products of row fragment i and weight fragment j of this
// wave (wave 2 wm + wn: row fragments wm MFC/2 .., weight fragments 4 wn ..)
// over NB blocks of one 128-byte line (two K-steps) per row; NB even, at least
// 4.  load_w(b, i) / load_a(b, i) load block b of this thread's row of pass i;
// wr[b], ar[b] hold blocks 0 .. AHEAD - 1 on entry.  Loads up to two
// blocks past the last one are made and not used (ring::block_at keeps them in
// the row).
//
// Block b (steps 2 b, 2 b + 1), with its first step's fragments and the rows of
// block b + 1 in place:
//   step 2 b: MFMAs; between their groups the weights of block b + 1 go from
//   registers to the ring and step 2 b + 1's fragments come from it (rows into a
//   second set, a weight fragment after its last use); load the weights of
//   block b + 3; barrier: block b + 1 is in the ring, block b's slot free;
//   step 2 b + 1 likewise, with the rows of block b + 2 into that slot, its next
//   fragments from block b + 1; load the rows of block b + 4.
// The writes are the slower side of the LDS (75 B/clk, reads about 200), so they
// are spread over a block's MFMA groups: all at its start they hold up the
// fragment reads behind them (a block of 128 x 128 with one workgroup on a CU
// 1433 -> 1156 cycles, with two 2269 -> 1960; its MFMAs take 512 and 1024).
// No load is under a run-time condition inside a round, so the compiler
// counts the loads in flight exactly; the first round is peeled so that the
// loop is entered in its steady state, and the last one loads nothing.
//
// The ring holds MFMA fragments of 1 KiB, lane (lr, lg)'s 16 bytes in slot
// 16 lg + (lr ^ lg ^ 12 (step & 1)); a copying lane group takes rows 4 apart.
// That keeps both the fragment reads and the copies' writes (8 lanes of a row
// to two steps x four lane groups) on distinct banks.
template <int DT, int MFC, class LoadW, class LoadA>
__device__ __forceinline__ void ring_loop(int NB, unsigned char* s_ring, u32x4 (&wr)[ring::AHEAD][ring::WP],
                                          u32x4 (&ar)[ring::AHEAD][MFC / 2], LoadW load_w, LoadA load_a,
                                          f32x4 (&acc)[MFC / 2][4]) {
  constexpr int MF = MFC / 2, NF = 4, AP = MFC / 2, WP = ring::WP;
  constexpr int STEP = (MFC + ring::WF) * 1024, SLOT = 2 * STEP;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave >> 1, wn = wave & 1;
  const int lr = lane & 15, lg = lane >> 4;
  const ring::Copy cp;
  const int clg = cp.chunk & 3, cstep = cp.chunk >> 2;
  unsigned char* const cdst = s_ring + cstep * STEP + cp.half * 1024 + (16 * clg + (cp.row16 ^ clg ^ (12 * cstep))) * 16;
  auto write_a = [&](int slot, int i, const u32x4& v) {
    *reinterpret_cast<u32x4*>(cdst + slot * SLOT + 2 * i * 1024) = v;
  };
  auto write_w = [&](int slot, int i, const u32x4& v) {
    *reinterpret_cast<u32x4*>(cdst + slot * SLOT + (MFC + 2 * i) * 1024) = v;
  };
#pragma unroll
  for (int i = 0; i < MF; ++i)
#pragma unroll
    for (int j = 0; j < NF; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  const unsigned char* const frag0 = s_ring + (16 * lg + (lr ^ lg)) * 16;
  const unsigned char* const frag1 = s_ring + STEP + (16 * lg + (lr ^ lg ^ 12)) * 16;
  u32x4 a[2][MF], w[NF];
  auto read_a = [&](const unsigned char* at, int h, int i) {
    a[h][i] = *reinterpret_cast<const u32x4*>(at + (wm * MF + i) * 1024);
  };
  auto read_w = [&](const unsigned char* at, int j) {
    w[j] = *reinterpret_cast<const u32x4*>(at + (MFC + wn * NF + j) * 1024);
  };
  constexpr int ROUND = ring::AHEAD;                          // blocks per round: sets and slots are immediates
  static_assert(ROUND == 2, "register sets and ring slots alternate together");
  static_assert(AP <= NF && WP == NF, "a block's writes fit one per MFMA group");
  auto round = [&](int r, auto last_c) {
    constexpr bool LAST = decltype(last_c)::value;
#pragma unroll
    for (int u = 0; u < ROUND; ++u) {
      const int b = r * ROUND + u;
      const bool more = !LAST || u == 0;                      // block b + 1 exists
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const unsigned char* const next = h == 0 ? frag1 + u * SLOT : frag0 + (u ^ 1) * SLOT;
        const bool refill = h == 0 || more;
#pragma unroll
        for (int j = 0; j < NF; ++j) {
#pragma unroll
          for (int i = 0; i < MF; ++i) ring_mfma<DT>(acc[i][j], w[j], a[h][i]);
          if (h == 0 && more) write_w(u ^ 1, j, wr[u ^ 1][j]);
          if (h == 1 && !LAST && j < AP) write_a(u, j, ar[u][j]);
          // (all of the next step's row fragments are used by its first group)
          if (refill && 2 * j < MF) {
            read_a(next, h ^ 1, 2 * j);
            if (2 * j + 1 < MF) read_a(next, h ^ 1, 2 * j + 1);
          }
          if (refill) read_w(next, j);
          asm volatile("" ::: "memory");
        }
        // (the round before the last loads blocks NB and NB + 1 of the rows: unused)
        if (h == 0 && !LAST)
#pragma unroll
          for (int i = 0; i < WP; ++i) wr[u ^ 1][i] = load_w(b + 3, i);
        if (h == 1 && !LAST)
#pragma unroll
          for (int i = 0; i < AP; ++i) ar[u][i] = load_a(b + 4, i);
        if (h == 0 && more) lds_barrier();
      }
    }
  };
#pragma unroll
  for (int i = 0; i < AP; ++i) write_a(0, i, ar[0][i]);
#pragma unroll
  for (int i = 0; i < WP; ++i) write_w(0, i, wr[0][i]);
#pragma unroll
  for (int i = 0; i < WP; ++i) wr[0][i] = load_w(2, i);
#pragma unroll
  for (int i = 0; i < AP; ++i) ar[0][i] = load_a(2, i);
#pragma unroll
  for (int i = 0; i < AP; ++i) write_a(1, i, ar[1][i]);
#pragma unroll
  for (int i = 0; i < AP; ++i) ar[1][i] = load_a(3, i);
  lds_barrier();
#pragma unroll
  for (int i = 0; i < MF; ++i) read_a(frag0, 0, i);
#pragma unroll
  for (int j = 0; j < NF; ++j) read_w(frag0, j);
  std::integral_constant<bool, true> yes;
  std::integral_constant<bool, false> no;
  const int rounds = NB / ROUND;                              // at least 2
  round(0, no);
  for (int r = 1; r < rounds - 1; ++r) round(r, no);
  round(rounds - 1, yes);

  // the MFMAs are inline asm: wait out the last ones before acc is read
  asm volatile("s_nop 7\n\ts_nop 7\n\ts_nop 7" ::: "memory");
#pragma unroll
  for (int i = 0; i < MF; ++i)
#pragma unroll
    for (int j = 0; j < NF; ++j) pin_acc(acc[i][j]);
}

}  // namespace
}  // namespace mep
