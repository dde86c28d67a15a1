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
  // one block per CU (its LDS holds 160 KB), a multiple of 8 blocks so each
  // keeps its XCD residue
  int64_t grid = device_cus();
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
    case EPI_QKV_ROPE: return run_gemm_persistent<BM, BN, BK, WM, WN, EPI_QKV_ROPE>(a, s);
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
// The predicted time of a launch on each tile, in us, with n tiles, c = ceil(n /
// CUs) of them on the fullest CU and KT K tiles:
//   fix + c (k KT + e) + (n / CUs) (kf KT + r)
// e per tile for the epilogue of its class (residual, other), the last term the
// memory traffic that grows with the whole launch (r: the residual's).  The
// constants are fits to the measured times of the four projection shapes of the
// model (N, K = 2304, 768; 768, 768; 4096, 768; 768, 2048) at M = 16 .. 40000; over
// those launches the tile it picks is within 6 % of the best (mean 0.2 %).
// Measured us (256 x 256 | picked), N = 768, K = 2048: M = 48: 47.1 | 8.2 (64 x
// 64); 2048: 52.4 | 15.4 (64 x 128); 4096: 53.0 | 20.5 (128 x 128); 8192: 55.1 |
// 31.2 (128 x 256); 40000: 157 | 157 (128 x 256: 156).  All tiles give
// bit-identical results, so the choice is free of M.
enum Tile { T64x64, T64x128, T128x128, T128x256, T256x256 };
struct TileCost {
  int bm, bn;
  double fix, k, e_resid, e_other, kf, r;
};
constexpr TileCost kTileCost[] = {
    {64, 64, 3.288, 0.153, 0.184, 0.561, 0.027, 1.501},
    {64, 128, 3.824, 0.261, 0.000, 0.001, 0.033, 2.355},
    {128, 128, 0.434, 0.305, 4.394, 3.868, 0.168, 3.480},
    {128, 256, 0.000, 0.463, 7.835, 6.446, 0.186, 3.150},
    {256, 256, 2.954, 1.303, 5.631, 5.373, 0.169, 21.205},
};
// a consumer of norm partials on 256 x 256 tiles needs the row_rstd launch
constexpr double kRowFactorLaunch = 4.5;
Tile pick_tile(int64_t M, int64_t N, int64_t K, bool resid, bool norm) {
  const int cus = device_cus() > 0 ? device_cus() : 256;
  const double KT = (double)(K / 64);
  const int64_t nb256 = ((M + 255) / 256) * (N / 256);
  if (nb256 >= 4 * (int64_t)cus) return T256x256;  // its rounds fill the chip
  double best = 0;
  Tile t = T256x256;
  for (int i = 0; i < 5; ++i) {
    const TileCost& w = kTileCost[i];
    const int64_t n = ((M + w.bm - 1) / w.bm) * ((N + w.bn - 1) / w.bn);
    const double c = (double)((n + cus - 1) / cus), f = (double)n / cus;
    double est = w.fix + c * (w.k * KT + (resid ? w.e_resid : w.e_other)) +
                 f * (w.kf * KT + (resid ? w.r : 0.0));
    if (i == T256x256 && norm) est += kRowFactorLaunch;
    // a full chip of 256 x 256 tiles moves the fewest operand bytes: leave it
    // only for a clear gain
    if (i == T256x256 && nb256 >= cus) est *= 0.95;
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
bool gemm_takes_norm_partials(int64_t M, int64_t N, int64_t K, int np) {
  return np % 4 == 0 && np <= 16 && N % 256 == 0 && K * 512 + K * 2 < (int64_t(1) << 31) &&
         N * 1024 < (int64_t(1) << 31) && pick_tile(M, N, K, false, true) != T256x256;
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
    switch (pick_tile(a.M, a.N, a.K, a.epi == EPI_RESID_F32, a.row_ss != nullptr)) {
      case T64x64: return run_gemm_pipe_epi<64, 64, 2, 1, 2, 5>(a, s);
      case T64x128: return run_gemm_pipe_epi<64, 128, 2, 2, 4, 3>(a, s);
      case T128x128: return run_gemm_pipe_epi<128, 128, 4, 2, 4, 5>(a, s);
      case T128x256: return run_gemm_pipe_epi<128, 256, 2, 4, 4, 3>(a, s);
      case T256x256: break;
    }
    if (a.row_ss) return fail(-2, "gemm: this launch does not take norm partials");
    return run_gemm_dma_epi<256, 256, 64, 2, 4>(a, s);
  }
  if (a.row_ss) return fail(-2, "gemm: this launch does not take norm partials");
  return run_gemm<128, 128, 32, 2, 2, 2, 3>(a, s);
}

}  // namespace blt
