// ns_sampler_slice.hip -- the sampling kernel's MODE_SLICE instances: UniDimSliceSampler chains of a shell.
#include "ns_sampler_dispatch.h"

namespace hipns {

// clears the heads (join word, step counters) of every cluster of a launch
__global__ void __launch_bounds__(256) k_lr_clear(const hipns_run_desc_t* runs, const hipns_run_state_t* states,
                                                  hipns_buffers_t B, int G, int cw) {
  const int r = blockIdx.y;
  const hipns_run_state_t* st = states + r;
  if (st->done) return;
  constexpr int WORDS = (int)(LR_CLUSTER_HEAD / 4);
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i / WORDS * G * cw >= runs[r].shell) return;
  unsigned char* base = (unsigned char*)(B.live_U[1 - st->buf] + runs[r].live_off * B.dps);
  ((uint32_t*)(base + (size_t)(i / WORDS) * lr_cluster_bytes(G, cw)))[i % WORDS] = 0u;
}

hipError_t launch_sampler_slice(const SampleArgs& A, int R, int max_chains, const hipns_launch_t& L, int dmax,
                                size_t lds_bytes, hipStream_t s) {
  if (L.family == HIPNS_FAM_LINREG && A.lr_split > 1) {
    const int cw = HIPNS_WAVE / L.lanes_per_chain;
    const int clusters = (max_chains + A.lr_groups * cw - 1) / (A.lr_groups * cw);
    const int words = clusters * (int)(LR_CLUSTER_HEAD / 4);
    hipLaunchKernelGGL(k_lr_clear, dim3((words + 255) / 256, R), dim3(256), 0, s, A.runs, A.states, A.B, A.lr_groups,
                       cw);
  }
  return launch_fam<MODE_SLICE>(A, R, max_chains, L, dmax, lds_bytes, s);
}

}  // namespace hipns
