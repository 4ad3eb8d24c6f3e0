// What gemm_big.hip and gemm_mid.hip share: loads into LDS through buffer resources, and the write-out of a wave's part of
// a tile.
#pragma once
#include "gemm_big.h"
#include "gemm_epi.h"

namespace {

// 64 lanes x 16 bytes through a buffer resource (byte offset per lane; lanes outside the resource read zeros) into LDS at
// lds + LO + 16 * lane. The whole offset is the lane's, rows included: the resource's range check covers it, while a
// scalar offset beyond the resource's size (a row of the tile past a short matrix) is not what that check is for.
template <int LO>
__device__ __forceinline__ void dma16b(u32x4 rsrc, uint32_t voff, uint32_t lds) {
  asm volatile("s_add_u32 m0, %2, %3\n\ts_nop 0\n\tbuffer_load_dwordx4 %0, %1, 0 offen lds" ::"v"(voff), "s"(rsrc), "s"(lds),
               "n"(LO)
               : "memory", "m0", "scc");
}

// f(IntC<0>), .., f(IntC<N - 1>)
template <int N, int n = 0, typename F>
__device__ __forceinline__ void for_each(F&& f) {
  if constexpr (n < N) {
    f(IntC<n>{});
    for_each<N, n + 1>(f);
  }
}

// Piece n of a wave's write-out (32 rows x 64 columns, the last of a row of pieces 32 columns if FN is odd): its
// 32-column blocks, its 16-byte chunks per output row, the rows of one store instruction
template <int FN, bool GLU, int n>
struct Piece {
  static constexpr int blocks = FN - n % ((FN + 1) / 2) * 2 < 2 ? 1 : 2;
  static constexpr int cpr = (GLU ? 2 : 4) * blocks, rpi = 64 / cpr;
};

// Write-out of a wave's (32 FM) x (32 FN) part of a tile, without barriers: pieces of 32 rows x 64 columns (the last one
// 32 columns wide if FN is odd) through 4 KB of the wave's own LDS at st. Rows of 128 bytes, 16-byte chunks swizzled by
// ((row >> 1) & 7), their 8-byte halves swapped in rows 16 .. 31. A piece is computed while the one before it settles in
// the LDS and the one before that is sent. m0, n0: the tile's first row and column of W, wr, wc: the wave's first row and
// column in it; brow: the tile's bias row in LDS; rows of C and R in whole aligned 16-byte chunks, 32-bit offsets.
template <int FM, int FN, int ACT, int HR, bool LIM>
__device__ __forceinline__ void write_out(const BigGemm& p, const f32x16 (&acc)[FN][FM], int m0, int n0, int wr, int wc,
                                          const float* brow, uint8_t* st, int lane) {
  constexpr bool GLU = ACT == 3;
  constexpr int NPC = (FN + 1) / 2;  // pieces per 32 rows
  const int Ncols = GLU ? p.N / 2 : p.N;
  int ln = lane;
  asm volatile("" : "+v"(ln));  // the lane's addresses are computed here, per tile: hoisted they would spill
  const int lr = ln & 31, hk = ln >> 5;
  const uint32_t put_o = lr * 128 + (((lr >> 1) & 7) << 4) + ((GLU ? (lr >> 4) & 1 : hk ^ ((lr >> 4) & 1)) << 3) + (GLU ? 4 * hk : 0);
  const int nw = n0 + wc, oc = GLU ? nw / 2 : nw;  // first column of W / of the output
  const long obytes = ((long)(p.M - m0 - 1) * p.ldc + Ncols - (GLU ? n0 / 2 : n0)) * 2;
  const uint64_t cu = (uint64_t)(uintptr_t)(p.C + (long)m0 * p.ldc + (GLU ? n0 / 2 : n0));
  uint16_t* cp = reinterpret_cast<uint16_t*>(((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)(cu >> 32)) << 32) |
                                             (uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)cu));
  const __amdgpu_buffer_rsrc_t rc = __builtin_amdgcn_make_buffer_rsrc(
      cp, (short)0, __builtin_amdgcn_readfirstlane((int)(obytes < 0x7ffffff0L ? obytes : 0x7ffffff0L)), 0x00020000);
  constexpr int NP = FM * NPC;
  u32x4 rr[HR ? NP : 1][4];
  if constexpr (HR == 1) {
    for_each<NP>([&](auto nc) {
      constexpr int n = decltype(nc)::value, cpr = Piece<FN, GLU, n>::cpr, rpi = Piece<FN, GLU, n>::rpi;
  #pragma unroll
      for (int u = 0; u < 32 / rpi; u++) {
        int rm = min(m0 + wr + n / NPC * 32 + u * rpi + ln / cpr, p.M - 1);
        if (p.r_rows > 0) rm %= p.r_rows;
        rr[n][u] = *reinterpret_cast<const u32x4*>(p.R + (long)rm * p.ldr + min(nw + n % NPC * 64 + ln % cpr * 8, p.N - 8));
      }
    });
  }
  f32x4 bv[FN][4];
  #pragma unroll
  for (int i = 0; i < FN; i++)
  #pragma unroll
    for (int g = 0; g < 4; g++) bv[i][g] = *reinterpret_cast<const f32x4*>(brow + wc + i * 32 + 8 * g + 4 * hk);
  u32x2 ov[2][8];
  u32x4 gv[2][4];
  auto compute = [&](auto nc) {
    constexpr int n = decltype(nc)::value;
  #pragma unroll
    for (int ii = 0; ii < Piece<FN, GLU, n>::blocks; ii++)
  #pragma unroll
      for (int g = 0; g < 4; g++) {
        const int i = n % NPC * 2 + ii;
        const f32x16& a = acc[i][n / NPC];
        const f32x4 a4 = {a[4 * g], a[4 * g + 1], a[4 * g + 2], a[4 * g + 3]}, &b = bv[i][g];
        if constexpr (ACT == 0)
          ov[n & 1][4 * ii + g] = u32x2{pack2(a4[0] + b[0], a4[1] + b[1]), pack2(a4[2] + b[2], a4[3] + b[3])};
        else
          ov[n & 1][4 * ii + g] = epi_val<ACT, false, 0>(a4, b, u32x2{0u, 0u}, false, nw + i * 32 + 8 * g + 4 * hk,
                                                         LIM ? p.act_ncols : 0);
      }
  };
  auto put = [&](auto nc) {
    constexpr int n = decltype(nc)::value;
  #pragma unroll
    for (int ii = 0; ii < Piece<FN, GLU, n>::blocks; ii++)
  #pragma unroll
      for (int g = 0; g < 4; g++)
        if constexpr (GLU)
          *reinterpret_cast<uint32_t*>(st + (put_o ^ ((2 * ii + (g >> 1)) << 4) ^ ((g & 1) << 3))) = ov[n & 1][4 * ii + g].x;
        else
          *reinterpret_cast<u32x2*>(st + (put_o ^ ((4 * ii + g) << 4))) = ov[n & 1][4 * ii + g];
  };
  auto get = [&](auto nc) {
    constexpr int n = decltype(nc)::value, cpr = Piece<FN, GLU, n>::cpr, rpi = Piece<FN, GLU, n>::rpi;
  #pragma unroll
    for (int u = 0; u < 32 / rpi; u++) {
      const int r = u * rpi + ln / cpr;
      gv[n & 1][u] = *reinterpret_cast<const u32x4*>(st + r * 128 + (((ln % cpr) ^ ((r >> 1) & 7)) << 4));
    }
  };
  auto send = [&](auto nc) {
    constexpr int n = decltype(nc)::value, cpr = Piece<FN, GLU, n>::cpr, rpi = Piece<FN, GLU, n>::rpi;
    constexpr int c = n % NPC * (GLU ? 32 : 64);  // the piece's first output column in the wave's part
    uint32_t vo = (uint32_t)((wr + n / NPC * 32 + ln / cpr) * p.ldc * 2 + ((GLU ? wc / 2 : wc) + c + ln % cpr * 8) * 2);
    vo = oc + c + ln % cpr * 8 < Ncols ? vo : 0x80000000u;
  #pragma unroll
    for (int u = 0; u < 32 / rpi; u++) {
      u32x4 v = gv[n & 1][u];
      if (rpi == 32 ? (ln / cpr) >> 4 & 1 : u * rpi >= 16) v = u32x4{v.z, v.w, v.x, v.y};
      if constexpr (HR == 1) {
  #pragma unroll
        for (int e = 0; e < 4; e++)
          v[e] = pack2(lo_bf(v[e]) + lo_bf(rr[n][u][e]), hi_bf(v[e]) + hi_bf(rr[n][u][e]));
      }
      // the row is in the lane's offset (as in dma16b): rows past M lie past the resource's end and are dropped
      __builtin_amdgcn_raw_buffer_store_b128(v, rc, vo + (uint32_t)(u * rpi) * (uint32_t)p.ldc * 2u, 0, 0);
    }
  };
  for_each<NP + 2>([&](auto nc) {
    constexpr int n = decltype(nc)::value;
    if constexpr (n < NP) compute(nc);
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (n >= 2) send(IntC<n - 2>{});
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (n >= 1 && n <= NP) get(IntC<n - 1>{});
    asm volatile("" ::: "memory");  // a wave's LDS accesses complete in order: the reads see its own writes
    if constexpr (n < NP) put(nc);
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
  });
}

// The fp32 sums of a wave's part to P[m0 + ..][n0 + ..] (row stride ldp, a multiple of 4), 32 x 32 at a time through the
// same 4 KB, in whole 128-byte rows.
template <int FM, int FN>
__device__ __forceinline__ void write_partial(const f32x16 (&acc)[FN][FM], float* P, long ldp, int M, int N, int m0,
                                              int n0, uint8_t* st, int lane) {
  const int lr = lane & 31, hk = lane >> 5;
#pragma unroll
  for (int j = 0; j < FM; j++)
#pragma unroll
    for (int i = 0; i < FN; i++) {
#pragma unroll
      for (int g = 0; g < 4; g++) {
        const f32x16& a = acc[i][j];
        *reinterpret_cast<f32x4*>(st + lr * 128 + (((2 * g + hk) ^ (lr & 7)) << 4)) =
            f32x4{a[4 * g], a[4 * g + 1], a[4 * g + 2], a[4 * g + 3]};
      }
      asm volatile("" ::: "memory");  // a wave's LDS accesses complete in order
      f32x4 v[4];
#pragma unroll
      for (int u = 0; u < 4; u++) {
        const int r = u * 8 + (lane >> 3);
        v[u] = *reinterpret_cast<const f32x4*>(st + r * 128 + (((lane & 7) ^ (r & 7)) << 4));
      }
      asm volatile("" ::: "memory");
      const int n = n0 + 32 * i + 4 * (lane & 7);
#pragma unroll
      for (int u = 0; u < 4; u++) {
        const int m = m0 + 32 * j + u * 8 + (lane >> 3);
        if (m < M && n < N) *reinterpret_cast<f32x4*>(P + (long)m * ldp + n) = v[u];
      }
    }
}

}  // namespace
