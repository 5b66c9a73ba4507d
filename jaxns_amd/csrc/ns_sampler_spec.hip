// ns_sampler_spec.hip -- slice chains of a launch that does not fill the chip: a chain evaluates its
// next proposals together.
#include "ns_sampler_impl.h"

namespace hipns {

// MODE_SLICE of k_sample with `columns` proposals of a chain per step.  A rejected proposal shrinks the
// bracket and the next one is picked from it with the next uniform of the chain's stream, neither of which
// depends on the likelihood; so a chain's next proposals are known before the first is evaluated, and a
// wavefront that would hold few chains has matrix columns for all of them.  Column i of a chain takes the
// i-th from here; the first accepted one is the slice's, and only the evaluations up to it are counted: the
// same points, counts and log L as one proposal per step, bit for bit.
//
// Bound by the latency of one step (about 1.5 us at 8 slots: 600 vector instructions and 8 MFMAs of 64
// cycles, of a wavefront alone on its SIMD).  A slice takes 2.3 evaluations in early shells and 3.6 in late
// ones, so with one proposal per step as many steps, with 8 about 1.05.  One run: D=10, 500 live points 8.06
// -> 4.58 ms; mixture of 4, D=4, with phantoms 4.72 -> 2.80 ms.  The regression family runs it on launches that
// spread their data rows: 16 runs of 512 chains, 4096 x 16, 515 -> 340 ms.
template <int LPC, int NJ, int FAM, int KT>
__global__ void __launch_bounds__(FAM == HIPNS_FAM_LINREG ? HIPNS_WAVE * lr_max_waves(NJ) : 256)
    k_sample_spec(SampleArgs A) {
  constexpr int CW = HIPNS_WAVE / LPC;
  constexpr bool COOP = FAM == HIPNS_FAM_LINREG;  // wavefronts step together and share the data rows
  extern __shared__ float lds[];
  const int r = A.B.run_order ? A.B.run_order[blockIdx.y] : (int)blockIdx.y;
  const hipns_run_desc_t run = A.runs[r];
  hipns_run_state_t* st = A.states + r;
  if (st->done) return;  // uniform across the block
  const int wpb = blockDim.x / HIPNS_WAVE, wave = threadIdx.x / HIPNS_WAVE;
  const int l = lane_id();
  const int c = l % CW, h = l / CW;
  const int m = A.columns;  // a power of two
  const int i = c & (m - 1), g = c / m;  // proposal of the step, chain of the wavefront
  const int cpw = A.chains_per_wave, G = COOP ? A.lr_groups : wpb;  // (the wavefronts past G take rows only)
  if ((int)blockIdx.x * G * cpw >= run.shell) return;  // whole block idle
  const int chain = ((int)blockIdx.x * G + wave) * cpw + g;
  bool alive = wave < G && g < cpw && chain < run.shell;
  const int dps = A.B.dps, D = run.D;
  const int DPr = ((D + 8 * LPC - 1) / (8 * LPC)) * (8 * LPC);
  const int nj = NJ == 8 ? 8 : DPr / LPC;

  MvnLds mv;
  GmmLds gm;
  LinRegLds lr;
  load_params(FAM, A.B.params + run.param_off, dps, D, A.gmm_K, lds, mv, gm, LPC, &lr, COOP ? G : 1, NJ / 8);
  if (COOP) {
    lr.r0 = A.lr_r0;
    lr.split = 1;
    lr.slice = 0;
    // in place before the first step's barriers
    lr.staged = A.lr_r0_off > 0;
    lr.r0l = lds + A.lr_r0_off;
    if (lr.staged) {
      for (int q = threadIdx.x; q < A.lr_npad; q += blockDim.x) lr.r0l[q] = A.lr_r0[q];
    }
    lr.xh = A.lr_xh;
    lr.xl = A.lr_xl;
    lr.xf = A.lr_xf;
    lr.y = nullptr;
    lr.npad = A.lr_npad;
    lr.panels = A.lr_panels;
    lr.terms = A.lr_terms;
    lr_take_blocks<LPC, NJ>(lr, wave, wpb);
  }
  const uint32_t tfm = transform_mask<LPC, NJ>(FAM == HIPNS_FAM_MVN ? mv.tf : gm.tf, h, nj);
  const uint32_t it32 = (uint32_t)st->iteration, k0 = run.seed_lo, k1 = run.seed_hi;
  const int cur = st->buf;
  const double contour = st->contour;
  const int S = run.shell, num_slices = run.num_slices, kph = run.k_phantom;
  const bool midpoint = run.midpoint_shrink != 0;

  // ---- seed point (get_seed_point, uni_slice_sampler.py:343-358)
  float U0[NJ], nv[NJ], up[NJ];
  const int idx = alive ? seed_index_dev(chain, it32, k0, k1, st->first_seed, run.N) : 0;
  const float* src = A.B.live_U[cur] + (run.live_off + idx) * (int64_t)dps;
#pragma unroll
  for (int j = 0; j < NJ; ++j) {
    // (0.5 past the run's dimensions, whatever the row holds there, unless the likelihood masks)
    const int d = owned_dim<LPC>(h, j);
    U0[j] = (alive && j < nj && (lik_masks(FAM, LPC, NJ) || d < D)) ? src[d] : 0.5f;
    nv[j] = 0.0f;
  }
  double logL0 = alive ? A.B.live_logL[cur][run.live_off + idx] : 0.0;

  // alpha = linspace(0.5, 1, num_slices)[s] (uni_slice_sampler.py:422), one table per block
  float* alpha_tab = lds + A.alpha_off;
  for (int q = threadIdx.x; q < num_slices; q += blockDim.x)
    alpha_tab[q] = (float)(num_slices > 1 ? 0.5 + 0.5 * (double)q / (double)(num_slices - 1) : 0.5);
  __syncthreads();

  // ---- drawn ahead, in the wavefront's own LDS: the directions of slices [dir0, dir0 + m), one per column
  // (nj / 4 float4 rows of 64 lanes), and the uniforms of evaluations [4 blk0, 4 (blk0 + m LPC)), one Philox
  // block per lane, a chain's blocks in order
  float* mine = lds + A.ring_off + (size_t)wave * spec_lds_floats(NJ);
  float4* dirs = (float4*)mine;
  uint32_t* picks = (uint32_t*)(mine + NJ * HIPNS_WAVE) + g * m * LPC * 4;
  int dir0 = -m, blk0 = 0, pick_end = 0;
  auto lds_order = [] {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  };

  const int64_t phantom_base =
      kph > 0 ? append_start((st->next_idx + S) % run.max_samples, (int64_t)S * kph, run.max_samples) : 0;
  const int sender = st->sender_node;
  int evals = 0, s = 0, k = 0, cap_hits = 0;  // k: rejected proposals of the slice
  float left = 0.0f, right = 0.0f, t = 0.0f, alpha = 0.5f;
  bool need_begin = true;
  // shrink() with alpha = 1 where the midpoint form is off
  auto cut = [&] {
    const float at = alpha * t;
    left = t < 0.0f ? at : left;
    right = t > 0.0f ? at : right;
  };

  while (COOP ? __syncthreads_or(alive) : __any(alive)) {
    if (__any(alive && evals + m > pick_end)) {
      if (alive) {
        blk0 = evals >> 2;
        pick_end = 4 * (blk0 + m * LPC);
        const int b = i * LPC + h;
        const u32x4 w = philox4x32((uint32_t)chain, it32, (uint32_t)(blk0 + b), RNG_PICK, k0, k1);
        ((uint4*)picks)[b] = make_uint4(w.x, w.y, w.z, w.w);
      }
      lds_order();
    }
    if (__any(alive && need_begin && s - dir0 >= m)) {
      if (alive) {
        dir0 = need_begin ? s : s + 1;
        if (dir0 + i < num_slices) {
          slice_direction<LPC, NJ>(up, chain, it32, dir0 + i, D, nj, h, k0, k1);
#pragma unroll
          for (int j = 0; j < NJ; j += 4)
            dirs[(j / 4) * HIPNS_WAVE + l] = make_float4(up[j], up[j + 1], up[j + 2], up[j + 3]);
        }
      }
      lds_order();
    }
    if (alive) {
      // every LDS read of the step at once (a wavefront alone waits out each latency): the uniforms (those
      // past m, of whatever follows, are not used), the slice's direction and alpha
      const uint32_t* pw = picks + (evals - 4 * blk0);
      uint32_t w[SPEC_COLUMNS_MAX];
#pragma unroll
      for (int q = 0; q < SPEC_COLUMNS_MAX; ++q) w[q] = pw[q];
      const int from = h * CW + g * m + ((s - dir0) & (m - 1));
      float4 v[NJ / 4];
#pragma unroll
      for (int j = 0; j < NJ / 4; ++j) v[j] = dirs[j * HIPNS_WAVE + from];
      const float a = alpha_tab[s];
      if (need_begin) {
        need_begin = false;
        k = 0;
        alpha = midpoint ? a : 1.0f;
#pragma unroll
        for (int j = 0; j < NJ / 4; ++j) {
          nv[4 * j] = v[j].x;
          nv[4 * j + 1] = v[j].y;
          nv[4 * j + 2] = v[j].z;
          nv[4 * j + 3] = v[j].w;
        }
        slice_bracket<LPC, NJ>(U0, nv, left, right);
      } else {
        cut();
      }
      // the picks up to this column's own (_pick_point_in_interval, _shrink_interval,
      // uni_slice_sampler.py:67-111)
      t = pick_t(left, right, u01f(w[0]));
#pragma unroll
      for (int q = 1; q < SPEC_COLUMNS_MAX; ++q) {
        if (q <= i) {
          cut();
          t = pick_t(left, right, u01f(w[q]));
        }
      }
    }
#pragma unroll
    for (int j = 0; j < NJ; ++j) up[j] = point_on_line(U0[j], t, nv[j]);
    double L;
    if constexpr (FAM == HIPNS_FAM_MVN)
      L = lik_mvn<LPC, NJ>(up, nj, D, dps, mv, run.log_const, tfm);
    else if constexpr (FAM == HIPNS_FAM_GMM)
      L = lik_gmm<LPC, NJ, KT>(up, nj, D, gm, tfm);
    else
      L = lik_linreg<LPC, NJ>(up, nj, D, lr, tfm, wave, G, run.log_const);

    // _new_proposal acceptance (uni_slice_sampler.py:160-166); the step cap keeps the seed point
    const bool acc = alive && ((L > contour) || (logL0 == contour && L == contour));
    const bool cap = alive && !acc && k + i + 1 >= A.max_steps;
    const unsigned long long taken = __ballot(acc || cap), capped = __ballot(cap);
    const unsigned mask = (1u << m) - 1u;
    const unsigned mine_taken = (unsigned)(taken >> (g * m)) & mask;  // (lane part 0 of the chain's columns)
    if (alive) {
      if (mine_taken) {
        const int f = __ffs(mine_taken) - 1, from = h * CW + g * m + f;
        evals += f + 1;
        if (((unsigned)(capped >> (g * m)) >> f) & 1u) {
          ++cap_hits;
        } else {
          // the accepted point again from its t: fewer lane exchanges than slots
          const float ta = __shfl(t, from);
          logL0 = __shfl(L, from);
#pragma unroll
          for (int j = 0; j < NJ; ++j) U0[j] = point_on_line(U0[j], ta, nv[j]);
        }
        // phantom samples: x[-(k+1):-1] (uni_slice_sampler.py:432-440), evals 0
        const int pidx = s - (num_slices - 1 - kph);
        if (kph > 0 && pidx >= 0 && s < num_slices - 1 && i == 0) {
          const int64_t si = run.samp_off + phantom_base + (int64_t)chain * kph + pidx;
          float* pd = A.B.samp_U + si * dps;
#pragma unroll
          for (int j = 0; j < NJ; ++j)
            if (j < nj) pd[owned_dim<LPC>(h, j)] = U0[j];
          if (h == 0) {
            A.B.samp_logL[si] = logL0;
            A.B.samp_sender[si] = sender;
            A.B.samp_evals[si] = 0;
            A.B.samp_phantom[si] = 1;
          }
        }
        need_begin = true;
        if (++s == num_slices) {
          alive = false;
          if (i == 0) {
            const int64_t o = run.chain_off + chain;
            float* dst = A.B.new_U + o * dps;
#pragma unroll
            for (int j = 0; j < NJ; ++j)
              if (j < nj) dst[owned_dim<LPC>(h, j)] = U0[j];
            if (h == 0) {
              A.B.new_logL[o] = logL0;
              A.B.new_evals[o] = evals;
            }
          }
        }
      } else {
        // all rejected: on from the last column's bracket and point
        evals += m;
        k += m;
        const int last = h * CW + g * m + m - 1;
        t = __shfl(t, last);
        left = __shfl(left, last);
        right = __shfl(right, last);
      }
    }
  }
  if (cap_hits > 0 && h == 0 && i == 0) {
    atomicAdd((unsigned long long*)&st->cap_hits, (unsigned long long)cap_hits);
    atomicOr(&st->flags, 1);
  }
}

// A call of the instance that a launch takes: the launch itself, or the wavefronts that a SIMD holds of it.
struct SpecCall {
  const SampleArgs* A;  // NULL: the wavefronts
  int R, max_chains, wpb;
  size_t lds;
  hipStream_t s;
  int waves;
  hipError_t err;
};

template <int LPC, int NJ, int FAM, int KT>
static void spec_rows(SpecCall& c) {
  if (!c.A) {
    static const int waves = waves_by_registers(k_sample_spec<LPC, NJ, FAM, KT>);
    c.waves = waves;
    return;
  }
  const int per_block = c.A->chains_per_wave * (FAM == HIPNS_FAM_LINREG ? c.A->lr_groups : c.wpb);
  dim3 grid((c.max_chains + per_block - 1) / per_block, c.R), block(c.wpb * HIPNS_WAVE);
  hipLaunchKernelGGL((k_sample_spec<LPC, NJ, FAM, KT>), grid, block, c.lds, c.s, *c.A);
  c.err = hipGetLastError();
}

template <int LPC, int NJ, int FAM>
static void spec_one(SpecCall& c, int K) {
  if constexpr (FAM == HIPNS_FAM_GMM) {
    switch (gmm_rows(K)) {
      case 4: return spec_rows<LPC, NJ, FAM, 4>(c);
      case 6: return spec_rows<LPC, NJ, FAM, 6>(c);
      default: return spec_rows<LPC, NJ, FAM, HIPNS_MAX_GMM_K>(c);
    }
  } else {
    return spec_rows<LPC, NJ, FAM, 1>(c);
  }
}

// the same instance choice as the sampler launchers (sampler_nj)
template <int FAM>
static void spec_fam(SpecCall& c, int K, int lpc, int dmax) {
  if constexpr (FAM == HIPNS_FAM_GMM) {
    if (lpc == 8 && dmax <= 128) return dmax <= 64 ? spec_one<8, 8, FAM>(c, K) : spec_one<8, 16, FAM>(c, K);
  }
  if (lpc == 4 || lpc == 8 || dmax > 64) {
    if (dmax <= 32) return spec_one<4, 8, FAM>(c, K);
    if (dmax <= 64) return spec_one<4, 16, FAM>(c, K);
    return spec_one<4, 32, FAM>(c, K);
  }
  if (dmax <= 16) return spec_one<2, 8, FAM>(c, K);
  if (dmax <= 32) return spec_one<2, 16, FAM>(c, K);
  return spec_one<2, 32, FAM>(c, K);
}

static void spec_call(SpecCall& c, int family, int K, int lpc, int dmax) {
  if (family == HIPNS_FAM_GMM) return spec_fam<HIPNS_FAM_GMM>(c, K, lpc, dmax);
  if (family == HIPNS_FAM_LINREG) return spec_fam<HIPNS_FAM_LINREG>(c, K, lpc, dmax);
  return spec_fam<HIPNS_FAM_MVN>(c, K, lpc, dmax);
}

hipError_t launch_sampler_spec(const SampleArgs& A, int R, int max_chains, const hipns_launch_t& L, int dmax,
                               size_t lds, hipStream_t s) {
  SpecCall c{&A, R, max_chains, L.waves_per_block, lds, s, 0, hipSuccess};
  spec_call(c, L.family, A.gmm_K, L.lanes_per_chain, dmax);
  return c.err;
}

int sampler_spec_waves(int family, int K, int lpc, int dmax) {
  SpecCall c{};
  spec_call(c, family, K, lpc, dmax);
  return c.waves;
}

}  // namespace hipns
