// Launch selection for the bf16 MFMA GEMM (kernel in gemm_kernel.hpp).
#include "gemm_kernel.hpp"

namespace blt {

namespace {
// Compute units of the current device (cached per device).
int device_cus() {
  static int cus[64];
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 0;
  if (cus[dev] == 0) {
    int n = 0;
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) return 0;
    cus[dev] = n;
  }
  return cus[dev];
}

template <int BM, int BN, int BK, int WM, int WN, int EPI>
int run_gemm_persistent(const GemmArgs& a, hipStream_t s) {
  const int64_t nb = ((a.M + BM - 1) / BM) * ((a.N + BN - 1) / BN);
  // as many blocks as fit on the CUs at once (256 x 256: one per CU, its LDS
  // holds 160 KB; 128 x 128: two, 80 KB each), a multiple of 8 blocks so each
  // keeps its XCD residue
  int64_t grid = (int64_t)device_cus() * (BM * BN <= 128 * 128 ? 2 : 1);
  grid = grid >= 8 ? grid & ~7 : grid;
  if (grid <= 0 || grid > nb) grid = nb;
  hipLaunchKernelGGL((gemm::gemm_bf16_dma_persistent_kernel<BM, BN, BK, WM, WN, EPI>),
                     dim3((unsigned)grid), dim3(64 * WM * WN), 0, s, a);
  BLT_LAUNCH_CHECK("gemm_bf16_dma_persistent_kernel");
  return 0;
}

// one kernel per epilogue, so each carries only its own registers and code
template <int BM, int BN, int BK, int WM, int WN>
int run_gemm_dma_epi(const GemmArgs& a, hipStream_t s) {
  switch (a.epi) {
    case EPI_BF16: return run_gemm_persistent<BM, BN, BK, WM, WN, EPI_BF16>(a, s);
    case EPI_F32: return run_gemm_persistent<BM, BN, BK, WM, WN, EPI_F32>(a, s);
    case EPI_RESID_F32: return run_gemm_persistent<BM, BN, BK, WM, WN, EPI_RESID_F32>(a, s);
    case EPI_QKV_ROPE:
      // (pick_tile gives QKV no persistent 128 x 128 tiles)
      if constexpr (BM == 256)
        return run_gemm_persistent<BM, BN, BK, WM, WN, EPI_QKV_ROPE>(a, s);
      break;
    case EPI_SILU_GATE: return run_gemm_persistent<BM, BN, BK, WM, WN, EPI_SILU_GATE>(a, s);
  }
  return fail(-2, "gemm: unknown epilogue");
}

template <int BM, int BN, int WM, int WN, int NL, int S, int EPI>
int run_gemm_pipe(const GemmArgs& a, hipStream_t s) {
  const int64_t nb = ((a.M + BM - 1) / BM) * ((a.N + BN - 1) / BN);
  hipLaunchKernelGGL((gemm::gemm_bf16_pipe_kernel<BM, BN, WM, WN, NL, S, EPI>),
                     dim3((unsigned)nb), dim3(64 * (WM * WN + NL)), 0, s, a);
  BLT_LAUNCH_CHECK("gemm_bf16_pipe_kernel");
  return 0;
}

template <int BM, int BN, int WM, int WN, int NL, int S>
int run_gemm_pipe_epi(GemmArgs a, hipStream_t s) {
  // tile groups of 1024 rows: their A rows (1.5 MB at K = 768) stay in an XCD's
  // L2 while it walks the columns.  N <= 1024 with at least as many rows: N
  // fastest (its whole Bt is what stays).
  a.group_m = a.N > 1024 || a.M < a.N ? 1024 / BM : 0;
  switch (a.epi) {
    case EPI_BF16: return run_gemm_pipe<BM, BN, WM, WN, NL, S, EPI_BF16>(a, s);
    case EPI_F32: return run_gemm_pipe<BM, BN, WM, WN, NL, S, EPI_F32>(a, s);
    case EPI_RESID_F32:
      // four waves of 32 x 32 pieces instead of two of 32 x 64: half the MFMA
      // chain per K tile (M = 48, K = 2048: 9.9 -> 8.6 us; K = 768: 6.2 -> 5.5;
      // 8.2 and 5.3 with the fragment reads across K tiles)
      if constexpr (BM == 64 && BN == 64)
        return run_gemm_pipe<64, 64, 2, 2, 4, S, EPI_RESID_F32>(a, s);
      else
        return run_gemm_pipe<BM, BN, WM, WN, NL, S, EPI_RESID_F32>(a, s);
    case EPI_QKV_ROPE: return run_gemm_pipe<BM, BN, WM, WN, NL, S, EPI_QKV_ROPE>(a, s);
    case EPI_SILU_GATE: return run_gemm_pipe<BM, BN, WM, WN, NL, S, EPI_SILU_GATE>(a, s);
  }
  return fail(-2, "gemm: unknown epilogue");
}

// ---- choice of the tile (N % 256 == 0) ---------------------------------------
// The predicted time of a launch on each tile, in us, with n tiles, KT K tiles, f = n
// / CUs, c1 = ceil(f) and c2 = ceil(f / 2), the rounds of one and of two blocks per CU:
//   fix + (k1 c1 + k2 c2 + kf f) KT + e c1 + o c2 + r f
// (k2 and o for the tiles that two blocks of a CU share; e and r by epilogue: the
// tile's own latency and the part that grows with the whole launch's traffic), and for
// a launch with row norms norm f where the tile forms the factors itself, else the
// row_rstd launch.  The constants are fits to 4150 launches on every tile in four
// runs: M = 1 .. 65536, N = 256 .. 12288, K = 64 .. 4096, every epilogue.  Over the
// projections of models (residual, and QKV and SiLU with row norms) the tile it picks
// takes 0.7 % longer than the best of the six on average, 10 % at the 99th percentile;
// a K or N left out of the fit: 0.2 to 1.3 % on average.  25 of those 1744 launches are
// over 3 % slower than on the two persistent tiles alone.  (A fit to K = 768 and 2048
// with one epilogue column for QKV, SiLU and bf16, and without T128x128x2: 1.8 %, 23 %,
// and 114 of them; a model of dim 256 at [4, 8192] took 366 us against 338.)
// Measured us (256 x 256 | picked), N = 768, K = 2048: M = 48: 45.5 | 7.7 (64 x 64);
// 2048: 49.6 | 14.2 (64 x 128); 4096: 51.0 | 20.8 (128 x 128); 8192: 54.7 | 31.5 (128 x
// 256).  All tiles give bit-identical results, so the choice is free of M.
enum Tile { T64x64, T64x128, T128x128, T128x256, T256x256, T128x128x2 };
struct TileCost {
  int bm, bn;
  double fix, k1, k2, kf, o, norm;
  double e[5], r[5];  // by Epilogue
};
// T256x256 and T128x128x2: the persistent two-stage kernel, one and two blocks per CU
constexpr TileCost kTileCost[] = {
    {64, 64, 2.032, 0.119, 0.030, 0.030, 0.926, 0.143,
     {0.357, 0.586, 0.000, 0.650, 0.298}, {0.024, 0.220, 0.711, 0.000, 0.000}},
    {64, 128, 2.179, 0.197, 0.011, 0.065, 0.652, 0.168,
     {0.042, 0.647, 0.528, 0.876, 0.000}, {0.427, 0.473, 1.345, 0.000, 0.160}},
    {128, 128, 1.399, 0.290, 0.000, 0.179, 0.000, 0.548,
     {2.022, 2.753, 1.857, 3.500, 2.059}, {0.548, 1.542, 4.708, 0.000, 0.000}},
    {128, 256, 1.641, 0.390, 0.000, 0.412, 0.000, 1.180,
     {2.282, 4.191, 2.899, 5.930, 2.662}, {1.698, 2.540, 7.192, 0.000, 0.000}},
    {256, 256, 2.722, 1.090, 0.000, 0.593, 0.000, 0.000,
     {2.974, 5.935, 4.000, 7.976, 2.672}, {2.436, 4.503, 15.553, 0.000, 0.288}},
    {128, 128, 2.761, 0.028, 0.404, 0.214, 0.593, 0.000,
     {0.780, 2.537, 1.700, 2.499, 0.401}, {0.223, 0.048, 2.379, 0.000, 0.213}},
};
static_assert(EPI_BF16 == 0 && EPI_F32 == 1 && EPI_RESID_F32 == 2 && EPI_QKV_ROPE == 3 &&
                  EPI_SILU_GATE == 4, "kTileCost's epilogue columns");
// a consumer of norm partials on the persistent tiles needs the row_rstd launch
constexpr double kRowFactorLaunch = 3.4;
bool takes_norm_partials(Tile t) { return t != T256x256 && t != T128x128x2; }
Tile pick_tile(int64_t M, int64_t N, int64_t K, int epi, bool norm) {
  const int cus = device_cus() > 0 ? device_cus() : 256;
  const double KT = (double)(K / 64);
  const int64_t nb256 = ((M + 255) / 256) * (N / 256);
  if (nb256 >= 4 * (int64_t)cus) return T256x256;  // its rounds fill the chip
  // the persistent tile with at least a block per CU; within the fit's error it is
  // kept, since it moves the fewest operand bytes
  const Tile persistent = nb256 < cus ? T128x128x2 : T256x256;
  double best = 0;
  Tile t = T256x256;
  for (int i = 0; i < 6; ++i) {
    if (i == T128x128x2 && epi == EPI_QKV_ROPE) continue;  // (never the least)
    const TileCost& w = kTileCost[i];
    const int64_t n = ((M + w.bm - 1) / w.bm) * ((N + w.bn - 1) / w.bn);
    const double f = (double)n / cus, c1 = (double)((n + cus - 1) / cus),
                 c2 = (double)((n + 2 * cus - 1) / (2 * cus));
    double est = w.fix + (w.k1 * c1 + w.k2 * c2 + w.kf * f) * KT + w.e[epi] * c1 + w.o * c2 +
                 w.r[epi] * f;
    if (norm) est += takes_norm_partials((Tile)i) ? w.norm * f : kRowFactorLaunch;
    if (i == persistent) est *= 0.97;
    if (i == 0 || est < best) {
      best = est;
      t = (Tile)i;
    }
  }
  return t;
}

// a 256-row tile's operand and output rows are addressed with 32-bit byte
// offsets, so their reach must fit
bool tile_reach_fits(const GemmArgs& a) {
  const int64_t two31 = int64_t(1) << 31;
  return 256 * (a.lda > a.ldb ? a.lda : a.ldb) * 2 + a.K * 2 < two31 && 256 * a.ldc * 4 < two31;
}

template <int BM, int BN, int BK, int WM, int WN, int PF, int OCC>
int run_gemm(const GemmArgs& a, hipStream_t s) {
  const int64_t nb = ((a.M + BM - 1) / BM) * ((a.N + BN - 1) / BN);
  hipLaunchKernelGGL((gemm::gemm_bf16_kernel<BM, BN, BK, WM, WN, PF, OCC>), dim3((unsigned)nb),
                     dim3(64 * WM * WN), 0, s, a);
  BLT_LAUNCH_CHECK("gemm_bf16_kernel");
  return 0;
}

}  // namespace

// (dense operands: the model's launches)
bool gemm_takes_norm_partials(int64_t M, int64_t N, int64_t K, int epi, int np) {
  return np % 4 == 0 && np <= 16 && N % 256 == 0 && K * 512 + K * 2 < (int64_t(1) << 31) &&
         N * 1024 < (int64_t(1) << 31) && takes_norm_partials(pick_tile(M, N, K, epi, true));
}

int gemm_tile(int64_t M, int64_t N, int64_t K, int epi) {
  return N % 256 == 0 ? pick_tile(M, N, K, epi, false) : -1;
}

int launch_gemm(const GemmArgs& a_in, hipStream_t s) {
  GemmArgs a = a_in;
  if (a.M == 0 || a.N == 0) return 0;
  a.vec_ok = ((uintptr_t)a.C % 16 == 0) && (a.ldc % 4 == 0);
  if ((a.epi == EPI_BF16 || a.epi == EPI_RESID_F32 || a.epi == EPI_QKV_ROPE ||
       a.epi == EPI_SILU_GATE) && (a.N % 64 != 0 || a.ldc % 4 != 0 || (uintptr_t)a.C % 16 != 0))
    return fail(-2, "gemm: vector epilogues need N % 64 == 0, ldc % 4 == 0, 16-byte aligned C");
  if (a.K % 64 != 0) return fail(-2, "gemm: K must be a multiple of 64");
  if (a.M >= (int64_t(1) << 31) - 256) return fail(-2, "gemm: M must be below 2^31 - 256");
  if (a.epi == EPI_QKV_ROPE && a.rope_cols > 0 &&
      (a.seq_len <= 0 || a.seq_len >= (int64_t(1) << 31)))
    return fail(-2, "gemm: the RoPE epilogue needs 0 < seq_len < 2^31");
  if ((a.xb_out != nullptr) != (a.ss_out != nullptr) ||
      (a.xb_out && (a.epi != EPI_RESID_F32 || a.ss_np * 64 != a.N || (uintptr_t)a.xb_out % 8)))
    return fail(-2, "gemm: norm partials need EPI_RESID_F32, xb_out and ss_out, ss_np = N / 64");
  if (a.col_scale && (!a.xb_out || (uintptr_t)a.col_scale % 16))
    return fail(-2, "gemm: col_scale scales the bf16 copy (xb_out) and must be 16-byte aligned");

  if ((uintptr_t)a.A % 16 != 0 || (uintptr_t)a.Bt % 16 != 0 || a.lda % 8 != 0 || a.ldb % 8 != 0)
    return fail(-2, "gemm: A and Bt rows must be 16-byte aligned (lda, ldb % 8 == 0)");
  if (a.row_ss && (a.row_np % 4 != 0 || a.row_np > 16 || (uintptr_t)a.row_ss % 16 != 0))
    return fail(-2, "gemm: row_ss needs row_np % 4 == 0, row_np <= 16, 16-byte alignment");
  // Wide N (QKV, W1|W3): walk groups of 8 M-tiles so the blocks resident on
  // an XCD share A and Bt tiles in its L2; narrow N (O, W2: 3 tiles): N fastest.
  a.group_m = (a.N + 255) / 256 >= 8 ? 8 : 0;
  // N % 256 == 0: K tiles of 64 moved by LDS DMA, LDS-staged epilogue, on the
  // tile pick_tile chooses.  Otherwise (the 260-wide head, huge strides)
  // 128x128 register-staged tiles over 4 waves.
  if (a.N % 256 == 0 && tile_reach_fits(a)) {
    const Tile t = pick_tile(a.M, a.N, a.K, a.epi, a.row_ss != nullptr);
    if (a.row_ss && !takes_norm_partials(t))
      return fail(-2, "gemm: this launch does not take norm partials");
    switch (t) {
      case T64x64: return run_gemm_pipe_epi<64, 64, 2, 1, 2, 5>(a, s);
      case T64x128: return run_gemm_pipe_epi<64, 128, 2, 2, 4, 3>(a, s);
      case T128x128: return run_gemm_pipe_epi<128, 128, 4, 2, 4, 5>(a, s);
      case T128x256: return run_gemm_pipe_epi<128, 256, 2, 4, 4, 3>(a, s);
      case T128x128x2: return run_gemm_dma_epi<128, 128, 64, 2, 2>(a, s);
      case T256x256: return run_gemm_dma_epi<256, 256, 64, 2, 4>(a, s);
    }
  }
  if (a.row_ss) return fail(-2, "gemm: this launch does not take norm partials");
  return run_gemm<128, 128, 32, 2, 2, 2, 3>(a, s);
}

}  // namespace blt
