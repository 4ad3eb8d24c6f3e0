// bf16 GEMM for grids of about one tile per CU: C[M,N] = epi(A[M,K] . W[N,K]^T + bias[N]) or raw fp32 split-K partials,
// tiles of 128 x 128, 128 x 192 or 128 x 256, with the operand contract and the roundings of gemm.hip. Every sum is one
// fp32 chain in k order: the bits of gemm.hip's one-chain tiles (configs 0-7, 16, 18, 23), not those of its two k groups
// (two chains, joined at the end), which configs 19 and 27 were. Error against 64 bits of 794 x 2048 x 8192 in two splits:
// 2.7e-7 with two chains, 4.0e-7 with one; rounded to bf16 1.65936e-3 either way.
//
// A few hundred rows give about one tile per CU, so a tile's time is the call's. 4 waves (2 x 2, 64 x (BN / 2) each), one
// per SIMD, and what the 8-wave tiles that this replaced left idle between the barriers of a step is filled by writing the
// order out: a step is four substeps of 16 columns, the fragments of a substep are read from LDS two substeps ahead, into
// registers of their own, so the MFMAs run across the barrier; the barrier sits in the middle of the step, behind the
// step's last LDS read, and its slot is refilled right behind it, one load per MFMA. Loads go through buffer resources
// (rows past the edge and steps past the end read zeros: the ring's counts hold without branches).
// What bounds it (128 x 128, K-step of 64, ns, copies for timing with parts taken out): MFMAs alone 213, with the LDS reads
// 253, the loads alone 298 for one workgroup and 380 with 200 of them (200 x 32 KB: 17 TB/s out of the L2s), everything
// together 390-430; the 8-wave tile before 480.
// Tried without gain: a ring of 3 or of 5 slots, lines of the next steps touched ahead (the L2 is not waited for, its rate
// is the limit). The rest of a call is 4 us that do not depend on K: launch, first load, write-out.
// Measured (us, cold weights, one box, the best tile before -> this one):
//   794 x 6144 x 2048  31.7 -> 27.9 (128 x 192; MFMAs alone 10.2)
//   794 x 8192 x 2048, GELU  41.3 -> 35.8 (128 x 256)
//   729 x 4304 x 1152, GELU  16.6 -> 14.3 (128 x 128)
//   729 x 1152 x 592  9.4 -> 8.3;  1280 x 2304 x 768  12.2 -> 10.4;  730 x 6144 x 2048  29.2 -> 27.1
// Where the grid has several tiles per CU the persistent 256-row tiles are better (9477 x 3456 x 1152: 75 against 100).
#include "gemm_mid.h"

#include "gemm_out.h"

namespace {

constexpr int BM = 128;
constexpr int BK = 64;  // k columns per step
constexpr int NW = 4;   // waves, 2 x 2

template <int BN, int ACT, int HR, bool LIM, bool PART>
__global__ __launch_bounds__(256, 1) void gemm_mid_kernel(BigGemm p, int tiles_m, int tiles_n, int splits, int kps,
                                                          float* __restrict__ P, long ldp, long p_split) {
  constexpr int WTM = BM / 2, WTN = BN / 2;
  constexpr int FM = WTM / 32, FN = WTN / 32;
  constexpr int NMF = FM * FN, NRD = FM + FN;  // MFMAs and fragment reads per substep (16 k columns)
  constexpr int LA = BM / 32, LW = BN / 32, LPS = LA + LW;  // load instructions per wave and step
  constexpr int STAGE = (BM + BN) * BK * 2;
  constexpr int S = BN == 128 ? 4 : 3;  // ring slots
  constexpr int BIAS_O = S * STAGE;
  static_assert(NRD <= NMF + 1 && LPS <= 2 * NMF, "reads and loads fit between the MFMAs");
  __shared__ __attribute__((aligned(1024))) uint8_t smem[BIAS_O + 1024];

  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave & 1, wn = wave >> 1;
  const int lr = lane & 31, hk = lane >> 5;
  const uint32_t sbase = lds_off(smem);
  int tm, tn, split;
  tile_of(blockIdx.x, tiles_m, tiles_n, splits, tm, tn, split);
  const int m0 = tm * BM, n0 = tn * BN;
  const int k0 = split * kps, k1 = min(p.Kw / BK, k0 + kps), nk = k1 - k0;

  auto resource = [&](const uint16_t* base, long rows, long ld, int width) {
    const long bytes = ((rows - 1) * ld + width) * 2;
    const uint64_t u = (uint64_t)(uintptr_t)base;
    return u32x4{(uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)u),
                 (uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)(u >> 32) & 0xffffu),
                 (uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)(bytes < 0x7ffffff0L ? bytes : 0x7ffffff0L)),
                 0x00020000u};
  };
  const u32x4 ra = resource(p.A + (long)m0 * p.lda, p.M - m0, p.lda, p.K);
  const u32x4 rw = resource(p.W + (long)n0 * p.ldw, p.N - n0, p.ldw, p.Kw);
  const int drow = wave * 8 + (lane >> 3), dch = (lane & 7) ^ (((lane >> 4) & 3) | ((wave & 1) << 2));
  const uint32_t va = (uint32_t)(drow * p.lda * 2 + dch * 16), vw = (uint32_t)(drow * p.ldw * 2 + dch * 16);
  const uint32_t a32 = (uint32_t)p.lda * 64, w32 = (uint32_t)p.ldw * 64;  // 32 rows in bytes
  const uint32_t lbase = sbase + wave * 8 * (BK * 2);
  // instruction i of the loads of step k into slot offset so: rows 32 i + drow of A, then of W
  uint32_t vak, vwk;
  auto aim = [&](int k) {
    const uint32_t o = (uint32_t)k * (BK * 2);
    vak = k < k1 && k * BK + dch * 8 < p.K ? va + o : 0x80000000u;
    vwk = k < k1 ? vw + o : 0x80000000u;
  };
  auto load = [&](auto ic, uint32_t so) {
    constexpr int i = decltype(ic)::value;
    if constexpr (i < LA)
      dma16b<i * 4096>(ra, vak + (uint32_t)i * a32, lbase + so);
    else
      dma16b<i * 4096>(rw, vwk + (uint32_t)(i - LA) * w32, lbase + so);
  };

  if (!PART && tid < 64) *reinterpret_cast<u32x4*>(smem + BIAS_O + tid * 16) = u32x4{0u, 0u, 0u, 0u};
  if (!PART && p.bias && wave == 0) {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    // past the last column: its last 4 again (stored nowhere)
    dma16s(p.bias, (uint32_t)min(n0 + 4 * lane, p.N - 4) * 4, sbase + BIAS_O);
  }
#pragma unroll
  for (int s = 0; s < S; s++) {
    aim(k0 + s);
    for_each<LPS>([&](auto ic) { load(ic, s * STAGE); });
  }

  f32x16 acc[FN][FM];
#pragma unroll
  for (int i = 0; i < FN; i++)
#pragma unroll
    for (int j = 0; j < FM; j++)
#pragma unroll
      for (int e = 0; e < 16; e++) acc[i][j][e] = 0.f;
  bf16x8 af[4][FM], wf[4][FN];  // the fragments of each substep
  uint32_t aa[4], wa[4];        // this lane's addresses in the slot of offset 0
#pragma unroll
  for (int s = 0; s < 4; s++) {
    const int sw = ((2 * s + hk) ^ ((lr >> 1) & 7)) << 4;
    aa[s] = (wm * WTM + lr) * (BK * 2) + sw;
    wa[s] = (BM + wn * WTN + lr) * (BK * 2) + sw;
  }
  // read r of substep s from the slot at so
  auto read = [&](int s, int r, uint32_t so) {
    if (r < FM)
      af[s][r < FM ? r : 0] = as_bf16x8(*reinterpret_cast<const u32x4*>(smem + aa[s] + so + r * 32 * BK * 2));
    else
      wf[s][r < FM ? 0 : r - FM] = as_bf16x8(*reinterpret_cast<const u32x4*>(smem + wa[s] + so + (r - FM) * 32 * BK * 2));
  };

  wait_vm<(S - 1) * LPS>();
  __syncthreads();
#pragma unroll
  for (int s = 0; s < 2; s++)
#pragma unroll
    for (int r = 0; r < NRD; r++) read(s, r, 0);

  uint32_t cur = 0;
  for (int k = 0; k < nk; k++) {
    const uint32_t nxt = cur + STAGE == S * STAGE ? 0 : cur + STAGE;
    aim(k0 + k + S);
    for_each<4>([&](auto sc) {
      constexpr int s = decltype(sc)::value;
      if constexpr (s == 2) {
        wait_vm<(S - 2) * LPS>();
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
      }
      for_each<NMF>([&](auto tc) {
        constexpr int t = decltype(tc)::value;
        acc[t / FM][t % FM] = mfma32(wf[s][t / FM], af[s][t % FM], acc[t / FM][t % FM]);
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (t < NRD) read((s + 2) & 3, t, s < 2 ? cur : nxt);
        if constexpr (t == NMF - 1 && NRD > NMF) read((s + 2) & 3, NRD - 1, s < 2 ? cur : nxt);
        if constexpr (s >= 2) {
          constexpr int l = (s - 2) * NMF + t;
          if constexpr (l < LPS) load(IntC<l < LPS ? l : 0>{}, cur);
        }
        __builtin_amdgcn_sched_barrier(0);
      });
    });
    cur = nxt;
  }
  wait_vm<0>();
  __syncthreads();
  uint8_t* st = smem + wave * 4096;
  if constexpr (PART)
    write_partial<FM, FN>(acc, P + split * p_split, ldp, p.M, p.N, m0 + wm * WTM, n0 + wn * WTN, st, lane);
  else
    write_out<FM, FN, ACT, HR, LIM>(p, acc, m0, n0, wm * WTM, wn * WTN, reinterpret_cast<const float*>(smem + BIAS_O), st,
                                    lane);
}

template <int BN>
hipError_t launch_bn(hipStream_t st, int act, const BigGemm& g, int splits, float* P, long ldp, long p_split) {
  const int tm = (g.M + BM - 1) / BM, tn = (g.N + BN - 1) / BN, nk = g.Kw / BK;
  const int kps = (nk + splits - 1) / splits;
  const long nt = (long)tm * tn * splits;
  if (nt > 0x7fffffffL) return hipErrorInvalidValue;
  const dim3 grid((unsigned)nt), blk(64 * NW);
  auto go = [&](auto kern) {
    hipLaunchKernelGGL(kern, grid, blk, 0, st, g, tm, tn, splits, kps, P, ldp, p_split);
    return hipGetLastError();
  };
  if (P) return go(gemm_mid_kernel<BN, 0, 0, false, true>);
  const bool lim = g.act_ncols != 0 && g.act_ncols < g.N;
  if (g.R) {
    if (act == 0) return go(gemm_mid_kernel<BN, 0, 1, false, false>);
    if (act == 1) return lim ? go(gemm_mid_kernel<BN, 1, 1, true, false>) : go(gemm_mid_kernel<BN, 1, 1, false, false>);
    return lim ? go(gemm_mid_kernel<BN, 2, 1, true, false>) : go(gemm_mid_kernel<BN, 2, 1, false, false>);
  }
  if (act == 0) return go(gemm_mid_kernel<BN, 0, 0, false, false>);
  if (act == 1) return lim ? go(gemm_mid_kernel<BN, 1, 0, true, false>) : go(gemm_mid_kernel<BN, 1, 0, false, false>);
  if (act == 2) return lim ? go(gemm_mid_kernel<BN, 2, 0, true, false>) : go(gemm_mid_kernel<BN, 2, 0, false, false>);
  return go(gemm_mid_kernel<BN, 3, 0, false, false>);
}

}  // namespace

bool gemm_mid_fits(int act, const BigGemm& g) {
  const int nout = act == 3 ? g.N / 2 : g.N;
  constexpr long LD = 1L << 21;
  if (nout % 8 || g.ldc % 8 || ((uintptr_t)g.C & 15)) return false;
  if (g.R && (g.ldr % 8 || ((uintptr_t)g.R & 15))) return false;
  return g.lda < LD && g.ldw < LD && g.ldc < LD;
}

hipError_t launch_gemm_mid(hipStream_t st, int bn, int act, const BigGemm& g, int splits, float* P, long ldp,
                           long p_split) {
  return bn == 128   ? launch_bn<128>(st, act, g, splits, P, ldp, p_split)
         : bn == 192 ? launch_bn<192>(st, act, g, splits, P, ldp, p_split)
                     : launch_bn<256>(st, act, g, splits, P, ldp, p_split);
}
