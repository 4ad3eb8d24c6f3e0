// bf16 GEMM for large grids: C[M,N] = epi(A[M,K] . W[N,K]^T + bias[N]), tiles of 256 x 256 or 256 x 192, with the operand
// contract and the roundings of gemm.hip, every sum one fp32 chain in k order (the bits of its one-chain tiles).
//
// One persistent workgroup of 4 waves per CU, one wave per SIMD, each wave a 128 x (BN / 2) quarter of the tile in
// 256 or 192 accumulator registers. What bounded the 8-wave tiles that this replaced (one tile per workgroup, a ring of
// two whole 64-column steps), and what is done about it:
//  * Reads from LDS per MFMA: a 128 x 128 wave tile reads 8 fragments for 16 MFMAs, a 128 x 64 one 6 for 8.
//  * Late loads: a whole-step slot can be refilled only after its last read, so its loads went out in a burst and had
//    one step to land in. Here the unit is a block of 64 rows (32 of each wave row): a step multiplies A block by A
//    block, all of W's fragments in registers, so the blocks of a slot are read, freed and refilled one after another,
//    at most one load instruction per two MFMAs, and a load has one and a half steps to land in. Rows stay 128 bytes in
//    memory and in LDS: a copy with 64-byte rows (32 columns, four slots) made the L1 fetch every line twice (1.35e8
//    instead of 6.7e7 requests to the L2 at 8192^3), which cost more than the longer ring gave.
//  * The ramp at the start of a tile and the write-out at its end, a quarter of the time at K = 1152: the loads of the
//    next tile's first steps are in flight through both, the sums start from the constant 0, and the results leave
//    through a private 4 KB of LDS per wave in three overlapped stages without barriers.
// With one wave per SIMD every instruction between the MFMAs costs issue time (a 32 x 32 x 16 MFMA covers about 6
// vector or 3 scalar instructions, measured), so the issue order is written out and the loads address memory through
// buffer resources: one add per load, and rows past the edge need no clamping. For the same reason the activation
// is not spread over the next tile's steps: 192 waiting values per lane and 10 instructions per value between the
// MFMAs took longer than the write-out they would have hidden (qkv below: 1.35 ms).
// Measured (us, both on one box: the 8-wave tile before -> this one, each the better of both widths):
//   186624 x 3456 x 1152           1495 -> 1319 (1127 TFLOP/s)
//   186624 x 4304 x 1152, GELU     2034 -> 1842
//   186624 x 1152 x 4304, residual 2092 -> 1756
//   186624 x 1152 x 1152, residual  669 ->  522
//   20480 x 6144 x 768, gated GELU  222 ->  196
//   9477 x 3456 x 1152             89.5 -> 75.3
//   8192 x 8192 x 8192              889 ->  807 (1363 TFLOP/s, MFMAs busy 75 % of the cycles)
#include "gemm_out.h"

namespace {

constexpr int BM = 256;
constexpr int BK = 64;   // k columns per step
constexpr int NW = 4;    // waves, 2 x 2

template <int BN, int ACT, int HR, bool LIM>
__global__ __launch_bounds__(256, 1) void gemm_big_kernel(BigGemm p, int tiles_m, int tiles_n) {
  constexpr int WTM = BM / 2, WTN = BN / 2;
  constexpr int FM = WTM / 32, FN = WTN / 32, NM = 4 * FN;  // MFMAs per phase
  static_assert(FM == 4 && (FN == 3 || FN == 4), "four phases per step");
  constexpr bool GLU = ACT == 3;
  constexpr int LPS = 2 * (FM + FN);                          // load instructions per wave and step
  constexpr int NST = FM * FN * (GLU ? 1 : 2);                 // store instructions per wave and tile
  // LDS: two A slots, two W slots at 32 KB steps, the bias rows of up to 4 tiles, 4 KB of staging per wave
  constexpr int SLOT = 32 * 1024, W_O = 2 * SLOT, W_B = BN * BK * 2;
  constexpr int BIAS_O = W_O + SLOT + W_B, EPI_O = BIAS_O + 4 * 1024;
  static_assert(BM * BK * 2 == SLOT && W_B <= SLOT, "LDS map");
  __shared__ __attribute__((aligned(1024))) uint8_t smem[EPI_O + NW * 4096];

  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave & 1, wn = wave >> 1;
  const int lr = lane & 31, hk = lane >> 5;
  const uint32_t sbase = lds_off(smem);
  const int nk = (p.Kw / BK + 1) & ~1;  // steps go in pairs: an odd count takes one more, of zeros (at least 4: the host)

  // this workgroup's tiles: XCD x (= block % 8) owns a contiguous run of the tile sequence, its workgroups take the
  // run's tiles in turn (the workgroups of an XCD work on neighbouring tiles at any time)
  const int nt = tiles_m * tiles_n, nx = min(8, (int)gridDim.x);
  const int xcd = blockIdx.x % nx, stride = ((int)gridDim.x - xcd + nx - 1) / nx;
  const int per = nt / nx, rem = nt % nx;
  const int run0 = xcd * per + min(xcd, rem), run1 = run0 + per + (xcd < rem ? 1 : 0);
  const int t0 = run0 + (int)blockIdx.x / nx;
  if (t0 >= run1) return;
  auto origin = [&](int t, int& m0, int& n0) {  // row groups of 4 tiles, column-major inside a group
    constexpr int GM = 4;
    const int grp = t / (GM * tiles_n), first = grp * GM, gs = min(tiles_m - first, GM);
    const int r = t - grp * GM * tiles_n;
    m0 = (first + r % gs) * BM;
    n0 = r / gs * BN;
  };

  // ---- the two operands' producers: (tile, step, slot) of the next blocks to load, through buffer resources that
  // start at the tile's first row and end with the matrix (rows past the end read as zeros; so do the chunks of A past
  // K and the steps past Kw, whose lanes take an offset outside). Past the last tile they repeat that tile (never
  // read; the loads keep the counts of the waits below true). A load instruction brings 8 rows of 128 bytes; its lanes
  // fetch the 16-byte chunks that belong at their places in the swizzled rows (chunk ^ ((row >> 1) & 7)).
  const int drow = wave * 8 + (lane >> 3), dch = (lane & 7) ^ (((lane >> 4) & 3) | ((wave & 1) << 2));
  const uint32_t va = (uint32_t)(drow * p.lda * 2 + dch * 16), vw = (uint32_t)(drow * p.ldw * 2 + dch * 16);
  const uint32_t a32 = (uint32_t)p.lda * 64, w32 = (uint32_t)p.ldw * 64;  // 32 rows in bytes
  int ak = 0, abias = 0, wt = t0, wk = 0;
  uint32_t alds = sbase + wave * 8 * (BK * 2), wlds = alds + W_O;
  int cm0, cn0, nm0, nn0;  // origins of the tile being multiplied and of the tile W is being loaded for
  uint32_t vak, vwk;       // the lane's offsets at the producers' steps
  u32x4 ra, rw;
  auto resource = [&](const uint16_t* base, long rows, long ld, int width) {
    const long bytes = ((rows - 1) * ld + width) * 2;
    const uint64_t u = (uint64_t)(uintptr_t)base;
    return u32x4{(uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)u),
                 (uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)(u >> 32) & 0xffffu),
                 (uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)(bytes < 0x7ffffff0L ? bytes : 0x7ffffff0L)),
                 0x00020000u};
  };
  auto aim_a = [&]() { ra = resource(p.A + (long)nm0 * p.lda, p.M - nm0, p.lda, p.K); };
  auto aim_w = [&]() {
    origin(wt, nm0, nn0);
    rw = resource(p.W + (long)nn0 * p.ldw, p.N - nn0, p.ldw, p.Kw);
  };
  // half e of the 64 rows of A block j (rows j 32 .. + 31 of each wave row) / of W block i
  auto load_a = [&](auto jc, auto ec) {
    constexpr int j = decltype(jc)::value, e = decltype(ec)::value;
    if (j == 0 && e == 0 && ak == 0 && p.bias)  // the tile's bias row, by every wave to the same place
      dma16s(p.bias, (uint32_t)min(nn0 + 4 * lane, p.N - 4) * 4, sbase + BIAS_O + abias * 1024);
    dma16b<(e * WTM + j * 32) * BK * 2>(ra, vak + (uint32_t)(4 * e + j) * a32, alds);
  };
  auto load_w = [&](auto ic, auto ec) {
    constexpr int i = decltype(ic)::value, e = decltype(ec)::value;
    dma16b<(e * WTN + i * 32) * BK * 2>(rw, vwk + (uint32_t)(FN * e + i) * w32, wlds);
  };
  auto chunk_a = [&]() { vak = ak * BK + dch * 8 < p.K ? va + ak * (BK * 2) : 0x80000000u; };
  auto chunk_w = [&]() { vwk = vw + (wk * BK < p.Kw ? wk * (BK * 2) : 0x80000000u); };
  // (W(k + 2) is loaded in the half step where A(k + 1) is finished, so a tile's W is aimed first)
  auto next_a = [&]() {
    alds ^= SLOT;
    if (++ak == nk) {
      ak = 0;
      abias = (abias + 1) & 3;
      aim_a();
    }
    chunk_a();
  };
  auto next_w = [&]() {
    wlds ^= SLOT;
    if (++wk == nk) {
      wk = 0;
      if (wt + stride < run1) wt += stride;
      aim_w();
    }
    chunk_w();
  };

  f32x16 acc[FN][FM];
  // ---- fragments of one A block and of a step's W blocks (4 substeps each). The next ones overwrite them as soon as the
  // last MFMA that needs them is issued, except the late substeps', which alternate between two places (A: 3; W: 2, 3).
  bf16x8 af[3], a3[2], wf[FN][2], w23[2][FN][2];
  // this lane's address of each substep in the A slot read next and in the next step's W slot; the other slot: ^ SLOT
  uint32_t aa[4], wa[4];
#pragma unroll
  for (int s = 0; s < 4; s++) {
    const int sw = ((2 * s + hk) ^ ((lr >> 1) & 7)) << 4;
    aa[s] = (wm * WTM + lr) * (BK * 2) + sw;
    wa[s] = W_O + (wn * WTN + lr) * (BK * 2) + sw;
  }
  auto flip = [&](uint32_t (&a)[4]) {
#pragma unroll
    for (int s = 0; s < 4; s++) {
      a[s] ^= SLOT;
      asm volatile("" : "+v"(a[s]));
    }
  };
  auto read_a = [&](int buf, int j, int s) {
    const bf16x8 v = as_bf16x8(*reinterpret_cast<const u32x4*>(smem + aa[s] + j * 32 * BK * 2));
    (s < 3 ? af[s < 3 ? s : 0] : a3[buf]) = v;
  };
  auto read_w = [&](int par, int i, int s) {
    const bf16x8 v = as_bf16x8(*reinterpret_cast<const u32x4*>(smem + wa[s] + i * 32 * BK * 2));
    (s < 2 ? wf[i][s & 1] : w23[par][i][s & 1]) = v;
  };

  // ---- a step: four phases, phase ph the MFMAs of A block ph with all W blocks in a fixed order, between them the reads
  // of the next A block and (phases 2, 3) of the next step's W, and the loads. FIRST: the tile's first step.
  int after = 0;  // waits left whose counts include the write-out's stores
  auto step = [&](auto parc, auto firstc) {
    constexpr int par = decltype(parc)::value;
    constexpr bool FIRST = decltype(firstc)::value;
#pragma unroll
    for (int ph = 0; ph < 4; ph++) {
      if (ph % 2 == 0) {
        // what this half step reads has landed once at most the loads of the last two halves (and, for a while, the
        // write-out's stores) are in flight, and this wave has read what it is about to multiply; behind the barrier
        // every wave has, and the loads below may take the places of what was read
        if (after > 0) {
          after--;
          wait_vm<LPS + NST>();
        } else {
          wait_vm<LPS>();
        }
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int t = 0; t < NM; t++) {
        const int s = t / FN, i = t % FN;
        const bf16x8 wv = s < 2 ? wf[i][s & 1] : w23[par][i][s & 1], av = s < 3 ? af[s < 3 ? s : 0] : a3[ph & 1];
        if (FIRST && s == 0) {
          f32x16 z;
#pragma unroll
          for (int e = 0; e < 16; e++) z[e] = 0.f;
          acc[i][ph] = mfma32(wv, av, z);
        } else {
          acc[i][ph] = mfma32(wv, av, acc[i][ph]);
        }
        __builtin_amdgcn_sched_barrier(0);
        // the next A block, each substep behind its last MFMA (the last substep first)
        if (t % FN == 0) read_a((ph + 1) & 1, (ph + 1) & 3, t == 0 ? 3 : t / FN - 1);
        // the next step's W: substeps 2, 3 in phase 2, substeps 0, 1 in phase 3 behind their last MFMAs
        if (ph == 2 && t % 2 == 1) read_w(par ^ 1, t / 4, 2 + t / 2 % 2);
        if (ph == 3 && t >= FN && t < 3 * FN) read_w(par ^ 1, t % FN, t / FN - 1);
        // loads: half 0 A 3, then (next step) A 0, W; half 1 A 1, A 2
        if (ph == 0) {
          if (t == 2) load_a(IntC<3>{}, IntC<0>{});
          if (t == 5) load_a(IntC<3>{}, IntC<1>{});
          if (t == 6) next_a();
          if (t == 8) load_a(IntC<0>{}, IntC<0>{});
          if (t == 11) load_a(IntC<0>{}, IntC<1>{});
        } else if (ph == 1) {
          if (t == 1) load_w(IntC<0>{}, IntC<0>{});
          if (t == 3) load_w(IntC<0>{}, IntC<1>{});
          if (t == 5) load_w(IntC<1>{}, IntC<0>{});
          if (t == 7) load_w(IntC<1>{}, IntC<1>{});
          if (t == 9) load_w(IntC<2>{}, IntC<0>{});
          if (t == 11) load_w(IntC<2>{}, IntC<1>{});
          if constexpr (FN == 4) {
            if (t == 13) load_w(IntC<3>{}, IntC<0>{});
            if (t == 15) load_w(IntC<3>{}, IntC<1>{});
          }
        } else if (ph == 2) {
          if (t == 4) load_a(IntC<1>{}, IntC<0>{});
          if (t == 10) load_a(IntC<1>{}, IntC<1>{});
        } else {
          if (t == 4) load_a(IntC<2>{}, IntC<0>{});
          if (t == 10) load_a(IntC<2>{}, IntC<1>{});
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      if (ph == 1) next_w();
      if (ph == 2) flip(aa);
    }
    flip(wa);
  };

  // ---- prologue: what the halves before step 0 would have loaded for it
  *reinterpret_cast<u32x4*>(smem + BIAS_O + tid * 16) = u32x4{0u, 0u, 0u, 0u};  // no bias: zeros
  aim_w();
  aim_a();
  cm0 = nm0;
  cn0 = nn0;
  chunk_a();
  chunk_w();
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
  auto all_a = [&](auto jc) {
    load_a(jc, IntC<0>{});
    load_a(jc, IntC<1>{});
  };
  auto all_w = [&]() {
    load_w(IntC<0>{}, IntC<0>{});
    load_w(IntC<0>{}, IntC<1>{});
    load_w(IntC<1>{}, IntC<0>{});
    load_w(IntC<1>{}, IntC<1>{});
    load_w(IntC<2>{}, IntC<0>{});
    load_w(IntC<2>{}, IntC<1>{});
    if constexpr (FN == 4) {
      load_w(IntC<3>{}, IntC<0>{});
      load_w(IntC<3>{}, IntC<1>{});
    }
  };
  all_w();
  next_w();
  all_a(IntC<0>{});
  all_a(IntC<1>{});
  all_a(IntC<2>{});
  all_a(IntC<3>{});
  next_a();
  all_a(IntC<0>{});
  all_w();
  next_w();
  all_a(IntC<1>{});
  all_a(IntC<2>{});
  wait_vm<LPS + 4>();  // W(0) and A(0) block 0 (the first instructions but 4) have landed
  __syncthreads();
#pragma unroll
  for (int i = 0; i < FN; i++)
#pragma unroll
    for (int s = 0; s < 4; s++) read_w(0, i, s);
#pragma unroll
  for (int s = 0; s < 4; s++) read_a(0, 0, s);
  flip(wa);

  uint8_t* st = smem + EPI_O + wave * 4096;
  int bias_row = 0;
  for (int t = t0; t < run1; t += stride) {
    step(IntC<0>{}, IntC<1>{});
    step(IntC<1>{}, IntC<0>{});
    for (int ks = 2; ks < nk; ks += 2) {
      step(IntC<0>{}, IntC<0>{});
      step(IntC<1>{}, IntC<0>{});
    }
    const float* brow = reinterpret_cast<const float*>(smem + BIAS_O + bias_row * 1024);
    bias_row = (bias_row + 1) & 3;

    write_out<FM, FN, ACT, HR, LIM>(p, acc, cm0, cn0, wm * WTM, wn * WTN, brow, st, lane);
    after = 3;
    cm0 = nm0;
    cn0 = nn0;
  }
  wait_vm<0>();  // the loads past the last tile land before the workgroup's LDS is given away
}

template <int BN>
hipError_t launch_bn(hipStream_t st, int act, const BigGemm& g) {
  const int tm = (g.M + BM - 1) / BM, tn = (g.N + BN - 1) / BN;
  int dev = 0, cus = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e == hipSuccess) e = hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
  if (e != hipSuccess) return e;
  const long nt = (long)tm * tn;
  if (nt > 0x3fffffffL) return hipErrorInvalidValue;
  const dim3 grid((unsigned)(nt < cus ? nt : cus)), blk(64 * NW);
  auto go = [&](auto kern) {
    hipLaunchKernelGGL(kern, grid, blk, 0, st, g, tm, tn);
    return hipGetLastError();
  };
  const bool lim = g.act_ncols != 0 && g.act_ncols < g.N;
  if (g.R) {
    if (act == 0) return go(gemm_big_kernel<BN, 0, 1, false>);
    if (act == 1) return lim ? go(gemm_big_kernel<BN, 1, 1, true>) : go(gemm_big_kernel<BN, 1, 1, false>);
    return lim ? go(gemm_big_kernel<BN, 2, 1, true>) : go(gemm_big_kernel<BN, 2, 1, false>);
  }
  if (act == 0) return go(gemm_big_kernel<BN, 0, 0, false>);
  if (act == 1) return lim ? go(gemm_big_kernel<BN, 1, 0, true>) : go(gemm_big_kernel<BN, 1, 0, false>);
  if (act == 2) return lim ? go(gemm_big_kernel<BN, 2, 0, true>) : go(gemm_big_kernel<BN, 2, 0, false>);
  return go(gemm_big_kernel<BN, 3, 0, false>);
}

}  // namespace

bool gemm_big_fits(int act, const BigGemm& g) {
  const int nout = act == 3 ? g.N / 2 : g.N;
  constexpr long LD = 1L << 21;
  if (nout % 8 || g.ldc % 8 || ((uintptr_t)g.C & 15) || g.Kw < 4 * BK) return false;
  if (g.R && (g.ldr % 8 || ((uintptr_t)g.R & 15))) return false;
  return g.lda < LD && g.ldw < LD && g.ldc < LD;
}

hipError_t launch_gemm_big(hipStream_t st, int bn, int act, const BigGemm& g) {
  return bn == 192 ? launch_bn<192>(st, act, g) : launch_bn<256>(st, act, g);
}
