// ns_sampler_loglik.hip -- batched likelihood through the sampler's device code.
#include "ns_sampler_impl.h"

namespace hipns {

// The owned components of a row of U: a lane's slots 8i..8i+7 are 8 consecutive dimensions, read as two
// 16-byte loads where the rows are 16-byte aligned (`vec`, uniform).  Slots beyond D hold 0.5.
template <int LPC, int NJ>
__device__ __forceinline__ void load_row(float (&up)[NJ], const float* U, int64_t row, bool ok, int dps, int D, int nj,
                                         int h, bool vec) {
#pragma unroll
  for (int j = 0; j < NJ; j += 4) {
    const int d = owned_dim<LPC>(h, j);
    if (vec) {
      const bool in = ok && j < nj;  // (then d + 3 < dps: the row stride covers a run's slots)
      const float4 v = in ? *(const float4*)(U + row * dps + d) : make_float4(0.5f, 0.5f, 0.5f, 0.5f);
      up[j] = d < D ? v.x : 0.5f;
      up[j + 1] = d + 1 < D ? v.y : 0.5f;
      up[j + 2] = d + 2 < D ? v.z : 0.5f;
      up[j + 3] = d + 3 < D ? v.w : 0.5f;
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i) up[j + i] = (ok && j < nj && d + i < D) ? U[row * dps + d + i] : 0.5f;
    }
  }
}

// Workgroups of a batched-likelihood launch over `groups` row groups: as many as stay resident by the instance's
// registers and the LDS of a CU, each taking row groups in turn, so that the parameter block is read into LDS
// once per workgroup and not once per 4 wavefronts of rows.  400 000 rows of MVN D=32: 40 -> 24 us, with the
// gradient 63 -> 42.
static unsigned loglik_blocks(int64_t groups, int wpb, int waves_per_simd, size_t lds, const LoglikChip& chip) {
  int64_t per_cu = 4 * waves_per_simd / wpb;
  const int64_t by_lds = lds ? (int64_t)(chip.lds / lds) : per_cu;
  if (per_cu > by_lds) per_cu = by_lds;
  if (per_cu < 1) per_cu = 1;
  const int64_t blocks = (groups + wpb - 1) / wpb, most = chip.cus * per_cu;
  return (unsigned)(blocks < most ? blocks : most);
}

// ---------------------------------------------------------------------------
// batched likelihood (Model.forward over a batch) through the same device code:
// row i of U plays the role of chain i of a single wavefront tile.
// ---------------------------------------------------------------------------
// (the widest regression instances at one wavefront per SIMD: at the 254 VGPRs that the 2-lane one needs, two
// would fit, and a launch that does not fill the chip then has two wavefronts share a SIMD's matrix unit beside
// idle ones: 33000 x 60, 20 000 points in FP32, 1.14 against 2.01 ms)
template <int LPC, int NJ, int FAM, int KT>
__global__ void __launch_bounds__(256)
    __attribute__((amdgpu_waves_per_eu(1, FAM == HIPNS_FAM_LINREG && NJ == 32 ? 1 : 8)))
    k_loglik(const float* U, int64_t B, double* out, const hipns_run_desc_t* runs, hipns_buffers_t Bf, int K,
             LinRegLds lrd) {
  constexpr int CW = HIPNS_WAVE / LPC;
  extern __shared__ float lds[];
  const hipns_run_desc_t run = runs[0];
  const int dps = Bf.dps;
  const int D = run.D;
  const int DPr = ((D + 8 * LPC - 1) / (8 * LPC)) * (8 * LPC);
  const int nj = NJ == 8 ? 8 : DPr / LPC;
  MvnLds mv;
  GmmLds gm;
  LinRegLds lr = lrd;
  lr.split = 1;
  lr.slice = 0;
  const int wpb = blockDim.x / HIPNS_WAVE;
  load_params(FAM, Bf.params + run.param_off, dps, D, K, lds, mv, gm, LPC, &lr, wpb, NJ / 8);
  const int wave = threadIdx.x / HIPNS_WAVE;
  if constexpr (FAM == HIPNS_FAM_LINREG) lr_take_blocks<LPC, NJ>(lr, wave, wpb);
  const int l = lane_id();
  const int c = l % CW, h = l / CW;
  const uint32_t tfm = transform_mask<LPC, NJ>(FAM == HIPNS_FAM_MVN ? mv.tf : gm.tf, h, nj);
  const bool vec = ((uintptr_t)U & 15u) == 0;
  int64_t row = ((int64_t)blockIdx.x * wpb + wave) * CW + c;
  float up[NJ];
  if constexpr (FAM == HIPNS_FAM_LINREG) {
    load_row<LPC, NJ>(up, U, row, row < B, dps, D, nj, h, vec);
    const double L = lik_linreg<LPC, NJ, false, true>(up, nj, D, lr, tfm, wave, wpb, run.log_const);
    if (row < B && h == 0) out[row] = L;
  } else {
    const int64_t stride = (int64_t)gridDim.x * wpb * CW;
    int64_t next = row;
    for (bool first = true;; first = false) {
      // the next rows load while these are evaluated (at one place, the first rows' too: a small batch's time is
      // its instructions' way to the CU)
      const bool more = __any(next < B);
      float nx[NJ];
      if (more) load_row<LPC, NJ>(nx, U, next, next < B, dps, D, nj, h, vec);
      if (!first) {
        double L;
        if constexpr (FAM == HIPNS_FAM_MVN)
          L = lik_mvn<LPC, NJ>(up, nj, D, dps, mv, run.log_const, tfm);
        else
          L = lik_gmm<LPC, NJ, KT>(up, nj, D, gm, tfm);
        if (row < B && h == 0) out[row] = L;
      }
      if (!more) break;
      row = next;
      next += stride;
#pragma unroll
      for (int j = 0; j < NJ; ++j) up[j] = nx[j];
    }
  }
}

// the same with d logL / dU (MVN and mixture families), the device form the gradient-guided chains
// use: grad[row * dps + d] for d < D; the wavefront's gradient scratch follows the parameters in LDS.
// (the 32-slot mixture instances at two wavefronts per SIMD, some spilling up to 128 B a lane: D=100, 400 000
// rows 330 -> 157 us with 6 component rows, 385 -> 267 with 8)
template <int LPC, int NJ, int FAM, int KT>
__global__ void __launch_bounds__(256, FAM == HIPNS_FAM_GMM && NJ == 32 ? 2 : 1)
    k_loglik_grad(const float* U, int64_t B, double* out, float* grad, const hipns_run_desc_t* runs,
                  hipns_buffers_t Bf, int K, int gscr_off) {
  constexpr int CW = HIPNS_WAVE / LPC;
  extern __shared__ float lds[];
  const hipns_run_desc_t run = runs[0];
  const int dps = Bf.dps;
  const int D = run.D;
  const int DPr = ((D + 8 * LPC - 1) / (8 * LPC)) * (8 * LPC);
  const int nj = NJ == 8 ? 8 : DPr / LPC;
  MvnLds mv;
  GmmLds gm;
  LinRegLds lr{};
  const int wpb = blockDim.x / HIPNS_WAVE;
  load_params(FAM, Bf.params + run.param_off, dps, D, K, lds, mv, gm, LPC, &lr, wpb, NJ / 8, true);
  const int wave = threadIdx.x / HIPNS_WAVE;
  const int l = lane_id();
  const int c = l % CW, h = l / CW;
  const uint32_t tfm = transform_mask<LPC, NJ>(FAM == HIPNS_FAM_MVN ? mv.tf : gm.tf, h, nj);
  const bool vec = ((uintptr_t)U & 15u) == 0, vec_out = ((uintptr_t)grad & 15u) == 0;
  const int64_t stride = (int64_t)gridDim.x * wpb * CW;
  float* gscr = lds + gscr_off + (size_t)wave * grad_rows(NJ, LPC) * (CW + 1);
  for (int64_t row = ((int64_t)blockIdx.x * wpb + wave) * CW + c; __any(row < B); row += stride) {
    const bool ok = row < B;
    float up[NJ], g[NJ];
    load_row<LPC, NJ>(up, U, row, ok, dps, D, nj, h, vec);
    double L;
    if constexpr (FAM == HIPNS_FAM_MVN)
      L = lik_mvn<LPC, NJ, true>(up, nj, D, dps, mv, run.log_const, tfm, gscr, g, true);
    else
      L = lik_gmm<LPC, NJ, KT, true>(up, nj, D, gm, tfm, g, true);
    if (ok) {
      if (h == 0) out[row] = L;
#pragma unroll
      for (int j = 0; j < NJ; j += 4) {
        const int d = owned_dim<LPC>(h, j);
        float* dst = grad + row * dps + d;
        if (vec_out && j < nj && d + 3 < D) {
          *(float4*)dst = make_float4(g[j], g[j + 1], g[j + 2], g[j + 3]);
        } else {
#pragma unroll
          for (int i = 0; i < 4; ++i)
            if (j < nj && d + i < D) dst[i] = g[j + i];
        }
      }
    }
  }
}

template <int LPC, int NJ, int FAM, int KT>
static hipError_t launch_loglik_grad_rows(const float* U, int64_t B, double* out, float* grad,
                                          const hipns_run_desc_t* runs, const hipns_buffers_t& Bf, int K, int wpb,
                                          int gscr_off, size_t lds, const LoglikChip& chip, hipStream_t s) {
  static const int waves = waves_by_registers(k_loglik_grad<LPC, NJ, FAM, KT>);
  constexpr int CW = HIPNS_WAVE / LPC;
  dim3 grid(loglik_blocks((B + CW - 1) / CW, wpb, waves, lds, chip)), block(wpb * HIPNS_WAVE);
  hipLaunchKernelGGL((k_loglik_grad<LPC, NJ, FAM, KT>), grid, block, lds, s, U, B, out, grad, runs, Bf, K, gscr_off);
  return hipGetLastError();
}

template <int LPC, int NJ, int FAM>
static hipError_t launch_loglik_grad_one(const float* U, int64_t B, double* out, float* grad,
                                         const hipns_run_desc_t* runs, const hipns_buffers_t& Bf, int K, int wpb,
                                         int gscr_off, size_t lds, const LoglikChip& chip, hipStream_t s) {
  if constexpr (FAM == HIPNS_FAM_GMM) {
    switch (gmm_rows(K)) {
      case 4:
        return launch_loglik_grad_rows<LPC, NJ, FAM, 4>(U, B, out, grad, runs, Bf, K, wpb, gscr_off, lds, chip, s);
      case 6:
        return launch_loglik_grad_rows<LPC, NJ, FAM, 6>(U, B, out, grad, runs, Bf, K, wpb, gscr_off, lds, chip, s);
      default: break;
    }
  }
  constexpr int KT = FAM == HIPNS_FAM_GMM ? HIPNS_MAX_GMM_K : 1;
  return launch_loglik_grad_rows<LPC, NJ, FAM, KT>(U, B, out, grad, runs, Bf, K, wpb, gscr_off, lds, chip, s);
}

template <int FAM>
static hipError_t launch_loglik_grad_fam(const float* U, int64_t B, double* out, float* grad,
                                         const hipns_run_desc_t* runs, const hipns_buffers_t& Bf, int K, int lpc,
                                         int wpb, int dmax, int gscr_off, size_t lds, const LoglikChip& chip,
                                         hipStream_t s) {
  auto call = [&](auto launch) { return launch(U, B, out, grad, runs, Bf, K, wpb, gscr_off, lds, chip, s); };
  if constexpr (FAM == HIPNS_FAM_GMM) {
    if (lpc == 8 && dmax <= 128)
      return call(dmax <= 64 ? launch_loglik_grad_one<8, 8, FAM> : launch_loglik_grad_one<8, 16, FAM>);
  }
  if (lpc == 4 || lpc == 8 || dmax > 64) {
    if (dmax <= 32) return call(launch_loglik_grad_one<4, 8, FAM>);
    if (dmax <= 64) return call(launch_loglik_grad_one<4, 16, FAM>);
    return call(launch_loglik_grad_one<4, 32, FAM>);
  }
  if (dmax <= 16) return call(launch_loglik_grad_one<2, 8, FAM>);
  if (dmax <= 32) return call(launch_loglik_grad_one<2, 16, FAM>);
  return call(launch_loglik_grad_one<2, 32, FAM>);
}

template <int LPC, int NJ, int FAM, int KT>
static hipError_t launch_loglik_rows(const float* U, int64_t B, double* out, const hipns_run_desc_t* runs,
                                     const hipns_buffers_t& Bf, int K, int wpb, size_t lds, const LoglikChip& chip,
                                     hipStream_t s, const LinRegLds& lr) {
  static const int waves = waves_by_registers(k_loglik<LPC, NJ, FAM, KT>);
  constexpr int CW = HIPNS_WAVE / LPC;
  const int64_t groups = (B + CW - 1) / CW;
  // (the regression family reads all its data rows per row group, beside which its parameters are nothing)
  const unsigned blocks =
      FAM == HIPNS_FAM_LINREG ? (unsigned)((groups + wpb - 1) / wpb) : loglik_blocks(groups, wpb, waves, lds, chip);
  dim3 grid(blocks), block(wpb * HIPNS_WAVE);
  hipLaunchKernelGGL((k_loglik<LPC, NJ, FAM, KT>), grid, block, lds, s, U, B, out, runs, Bf, K, lr);
  return hipGetLastError();
}

template <int LPC, int NJ, int FAM>
static hipError_t launch_loglik_one(const float* U, int64_t B, double* out, const hipns_run_desc_t* runs,
                                    const hipns_buffers_t& Bf, int K, int wpb, size_t lds, const LoglikChip& chip,
                                    hipStream_t s, const LinRegLds& lr) {
  if constexpr (FAM == HIPNS_FAM_GMM) {
    switch (gmm_rows(K)) {
      case 4: return launch_loglik_rows<LPC, NJ, FAM, 4>(U, B, out, runs, Bf, K, wpb, lds, chip, s, lr);
      case 6: return launch_loglik_rows<LPC, NJ, FAM, 6>(U, B, out, runs, Bf, K, wpb, lds, chip, s, lr);
      default: break;
    }
  }
  constexpr int KT = FAM == HIPNS_FAM_GMM ? HIPNS_MAX_GMM_K : 1;
  return launch_loglik_rows<LPC, NJ, FAM, KT>(U, B, out, runs, Bf, K, wpb, lds, chip, s, lr);
}

// the same instance choice as the sampler launchers (sampler_nj)
template <int FAM>
static hipError_t launch_loglik_fam(const float* U, int64_t B, double* out, const hipns_run_desc_t* runs,
                                    const hipns_buffers_t& Bf, int K, int lpc, int wpb, int dmax, size_t lds,
                                    const LoglikChip& chip, hipStream_t s, const LinRegLds& lr) {
  if constexpr (FAM == HIPNS_FAM_GMM) {
    if (lpc == 8 && dmax <= 128) {
      if (dmax <= 64) return launch_loglik_one<8, 8, FAM>(U, B, out, runs, Bf, K, wpb, lds, chip, s, lr);
      return launch_loglik_one<8, 16, FAM>(U, B, out, runs, Bf, K, wpb, lds, chip, s, lr);
    }
  }
  if (lpc == 4 || lpc == 8 || dmax > 64) {
    if (dmax <= 32) return launch_loglik_one<4, 8, FAM>(U, B, out, runs, Bf, K, wpb, lds, chip, s, lr);
    if (dmax <= 64) return launch_loglik_one<4, 16, FAM>(U, B, out, runs, Bf, K, wpb, lds, chip, s, lr);
    return launch_loglik_one<4, 32, FAM>(U, B, out, runs, Bf, K, wpb, lds, chip, s, lr);
  }
  if (dmax <= 16) return launch_loglik_one<2, 8, FAM>(U, B, out, runs, Bf, K, wpb, lds, chip, s, lr);
  if (dmax <= 32) return launch_loglik_one<2, 16, FAM>(U, B, out, runs, Bf, K, wpb, lds, chip, s, lr);
  return launch_loglik_one<2, 32, FAM>(U, B, out, runs, Bf, K, wpb, lds, chip, s, lr);
}

// adjoint statistics of the regression likelihood over a batch of points: logL, |r|^2 and y^T r
// per row of U (the host derives d logL / d(log sigma, log tau)).  A workgroup's first wavefront holds one
// group of 64 / LPC points, all of its wavefronts share the data rows.
template <int LPC, int NJ>
__global__ void __launch_bounds__(HIPNS_WAVE * lr_max_waves(NJ))
    k_linreg_stats(const float* U, int64_t B, double* logL, double* rss, double* yr, const hipns_run_desc_t* runs,
                   hipns_buffers_t Bf, LinRegLds lrd) {
  constexpr int CW = HIPNS_WAVE / LPC;
  extern __shared__ float lds[];
  const hipns_run_desc_t run = runs[0];
  const int dps = Bf.dps;
  const int D = run.D;
  const int DPr = ((D + 8 * LPC - 1) / (8 * LPC)) * (8 * LPC);
  const int nj = NJ == 8 ? 8 : DPr / LPC;
  MvnLds mv;
  GmmLds gm;
  LinRegLds lr = lrd;
  lr.split = 1;
  lr.slice = 0;
  load_params(HIPNS_FAM_LINREG, Bf.params + run.param_off, dps, D, 1, lds, mv, gm, LPC, &lr, 1, NJ / 8);
  const int l = lane_id(), wave = threadIdx.x / HIPNS_WAVE;
  const int c = l % CW, h = l / CW;
  lr_take_blocks<LPC, NJ>(lr, wave, blockDim.x / HIPNS_WAVE);
  const int64_t row = (int64_t)blockIdx.x * CW + c;
  float up[NJ];
  const bool ok = wave == 0 && row < B;
#pragma unroll
  for (int j = 0; j < NJ; ++j) {
    int d = owned_dim<LPC>(h, j);
    up[j] = (ok && j < nj && d < D) ? U[row * dps + d] : 0.5f;
  }
  const uint32_t tfm = transform_mask<LPC, NJ>(lr.tf, h, nj);
  double ss = 0.0, sy = 0.0;
  const double L = lik_linreg<LPC, NJ, true>(up, nj, D, lr, tfm, wave, 1, run.log_const, &ss, &sy);
  if (ok && h == 0) {
    logL[row] = L;
    rss[row] = ss;
    yr[row] = sy;
  }
}

hipError_t launch_linreg_stats(const float* U, int64_t B, double* logL, double* rss, double* yr,
                               const hipns_run_desc_t* runs, const hipns_buffers_t& Bf, int lpc, int dmax,
                               int waves, size_t lds, hipStream_t s, const LinRegLds& lr) {
  if (dmax > 64) lpc = 4;
  const int CW = HIPNS_WAVE / lpc;
  dim3 grid((unsigned)((B + CW - 1) / CW)), block(HIPNS_WAVE * waves);
  if (lpc == 2) {
    if (dmax <= 16)
      hipLaunchKernelGGL((k_linreg_stats<2, 8>), grid, block, lds, s, U, B, logL, rss, yr, runs, Bf, lr);
    else if (dmax <= 32)
      hipLaunchKernelGGL((k_linreg_stats<2, 16>), grid, block, lds, s, U, B, logL, rss, yr, runs, Bf, lr);
    else
      hipLaunchKernelGGL((k_linreg_stats<2, 32>), grid, block, lds, s, U, B, logL, rss, yr, runs, Bf, lr);
  } else {
    if (dmax <= 32)
      hipLaunchKernelGGL((k_linreg_stats<4, 8>), grid, block, lds, s, U, B, logL, rss, yr, runs, Bf, lr);
    else if (dmax <= 64)
      hipLaunchKernelGGL((k_linreg_stats<4, 16>), grid, block, lds, s, U, B, logL, rss, yr, runs, Bf, lr);
    else
      hipLaunchKernelGGL((k_linreg_stats<4, 32>), grid, block, lds, s, U, B, logL, rss, yr, runs, Bf, lr);
  }
  return hipGetLastError();
}

hipError_t launch_loglik_grad(const float* U, int64_t B, double* out, float* grad, const hipns_run_desc_t* runs,
                              const hipns_buffers_t& Bf, const hipns_launch_t& L, int dmax, int gscr_off, size_t lds,
                              const LoglikChip& chip, hipStream_t s) {
  const int lpc = L.lanes_per_chain, wpb = L.waves_per_block, K = L.gmm_K;
  if (L.family == HIPNS_FAM_GMM)
    return launch_loglik_grad_fam<HIPNS_FAM_GMM>(U, B, out, grad, runs, Bf, K, lpc, wpb, dmax, gscr_off, lds, chip, s);
  if (L.family == HIPNS_FAM_MVN)
    return launch_loglik_grad_fam<HIPNS_FAM_MVN>(U, B, out, grad, runs, Bf, K, lpc, wpb, dmax, gscr_off, lds, chip, s);
  return hipErrorInvalidValue;
}

hipError_t launch_loglik(const float* U, int64_t B, double* out, const hipns_run_desc_t* runs,
                         const hipns_buffers_t& Bf, const hipns_launch_t& L, int dmax, size_t lds,
                         const LoglikChip& chip, hipStream_t s, const LinRegLds& lr) {
  const int lpc = L.lanes_per_chain, wpb = L.waves_per_block, K = L.gmm_K;
  if (L.family == HIPNS_FAM_GMM)
    return launch_loglik_fam<HIPNS_FAM_GMM>(U, B, out, runs, Bf, K, lpc, wpb, dmax, lds, chip, s, lr);
  if (L.family == HIPNS_FAM_LINREG)
    return launch_loglik_fam<HIPNS_FAM_LINREG>(U, B, out, runs, Bf, K, lpc, wpb, dmax, lds, chip, s, lr);
  return launch_loglik_fam<HIPNS_FAM_MVN>(U, B, out, runs, Bf, K, lpc, wpb, dmax, lds, chip, s, lr);
}

}  // namespace hipns
