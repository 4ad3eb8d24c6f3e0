// What the GEMM kernels share: the workgroup -> tile order and the epilogue of one 4-column group.
#pragma once
#include "common.h"

namespace {

// Tile order. Dispatch sends workgroup b to XCD (b % 8), so each XCD is given a contiguous run of the tile sequence
// (split-major, then tile). Inside a run, tiles go in groups of GM row panels, column-major within a group: the 32
// workgroups an XCD runs at once then share GM panels of A and a few panels of W in that XCD's L2, instead of
// sweeping every row panel of A past one W panel. Grids with at most GM row panels keep plain column-major order.
// GM = 8, and 4 for the 192- and 256-row tiles of large grids (1-3 % faster there than 8; 16 and 32 were slower).
template <int GM = 8>
__device__ __forceinline__ void tile_of(int b, int tiles_m, int tiles_n, int splits, int& tm, int& tn, int& split) {
  const int nt = tiles_m * tiles_n, ntot = nt * splits;
  const int per = ntot / 8, rem = ntot % 8, xcd = b % 8, idx = b / 8;
  const int t = (xcd < rem) ? xcd * (per + 1) + idx : rem * (per + 1) + (xcd - rem) * per + idx;
  const int tile = t % nt;
  split = t / nt;
  const int grp = tile / (GM * tiles_n), first = grp * GM, gs = min(tiles_m - first, GM);
  const int r = tile - grp * GM * tiles_n;
  tm = first + r % gs;
  tn = r / gs;
}

// Epilogue of one 4-column group (output row m, columns n .. n+3) from fp32 sums s: + bias, round to bf16, activation
// ACT (1 GELU-tanh, 2 GELU-erf; rounded again; act_ncols > 0: on columns < act_ncols, < 0: >= -act_ncols), + residual
// (fp32 add, rounded once more). ACT 3 is the gated GELU of interleaved (gate, up) column pairs, written to columns
// n / 2, n / 2 + 1.
template <int V>
struct IntC {
  static constexpr int value = V;
};
// I8: s holds int32 accumulator bits; the linear output is ((float)acc * sa) * sw + bias in fp32 and any GELU applies
// to that fp32 value before the one bf16 rounding (the W8A8 epilogue); a residual is then added to the rounded value.
// HR: 0 / 1 = no residual / a residual, known at compile time; 2 = has_r decides. The activation is computed for every
// column and then selected (act_ncols varies across the lanes of a wave: a branch per group would serialise the
// exp / rcp chains of the groups instead of interleaving them).
template <int ACT, bool I8 = false, int HR = 2>
__device__ __forceinline__ u32x2 epi_val(const f32x4& s, const f32x4& bv, const u32x2& rv, bool has_r, int n,
                                         int act_ncols, float sa = 0.f, const f32x4& sw = f32x4{0.f, 0.f, 0.f, 0.f}) {
  const bool hr = HR == 2 ? has_r : HR == 1;
  float v[4];
  if constexpr (I8) {
    static_assert(ACT != 3, "no gated GELU in the int8 path");
#pragma unroll
    for (int e = 0; e < 4; e++) {
      const float t = (float)__float_as_int(s[e]) * sa;
      v[e] = t * sw[e] + bv[e];
    }
    if constexpr (ACT == 1 || ACT == 2) {
      const bool on = act_ncols <= 0 ? n >= -act_ncols : n < act_ncols;
#pragma unroll
      for (int e = 0; e < 4; e++) {
        const float g = ACT == 1 ? gelu_tanh(v[e]) : gelu_erf(v[e]);
        v[e] = on ? g : v[e];
      }
    }
    if (hr) {
      v[0] = rbf(v[0]) + lo_bf(rv.x);
      v[1] = rbf(v[1]) + hi_bf(rv.x);
      v[2] = rbf(v[2]) + lo_bf(rv.y);
      v[3] = rbf(v[3]) + hi_bf(rv.y);
    }
    return u32x2{pack2(v[0], v[1]), pack2(v[2], v[3])};
  }
#pragma unroll
  for (int e = 0; e < 4; e++) v[e] = rbf(s[e] + bv[e]);
  u32x2 o;
  if constexpr (ACT == 3) {
    o.x = pack2(rbf(gelu_tanh(v[0])) * v[1], rbf(gelu_tanh(v[2])) * v[3]);
    o.y = 0;
  } else {
    if constexpr (ACT == 1 || ACT == 2) {
      // the activation's bf16 rounding: explicit before a residual add, else the final pack's own rounding
      const bool on = act_ncols <= 0 ? n >= -act_ncols : n < act_ncols;
#pragma unroll
      for (int e = 0; e < 4; e++) {
        float g = ACT == 1 ? gelu_tanh(v[e]) : gelu_erf(v[e]);
        if (hr) g = rbf(g);
        v[e] = on ? g : v[e];
      }
    }
    if (hr) {
      v[0] += lo_bf(rv.x);
      v[1] += hi_bf(rv.x);
      v[2] += lo_bf(rv.y);
      v[3] += hi_bf(rv.y);
    }
    o.x = pack2(v[0], v[1]);
    o.y = pack2(v[2], v[3]);
  }
  return o;
}
// Run f(IntC<act>) for the runtime activation code act (0..3).
template <typename F>
__device__ __forceinline__ void with_act(int act, F&& f) {
  switch (act) {
    case 1: f(IntC<1>{}); break;
    case 2: f(IntC<2>{}); break;
    case 3: f(IntC<3>{}); break;
    default: f(IntC<0>{}); break;
  }
}

}  // namespace
