// Wide-head SparseMLA kernels (d_qk = 576, d_v = 512 or 576: the DeepSeek-V3.2
// MLA latent + rope row) and the entry points the C-ABI dispatches to.
#pragma once

#include <hip/hip_runtime.h>

#include "sparse_mla_params.hpp"

namespace dsa {

// Head dims served by the wide kernels: the MLA row with its 512-dim latent as
// V, or the whole row as V (d_v defaults to d_qk when a caller passes none).
inline bool wide_shape(int64_t d_qk, int64_t d_v) { return d_qk == 576 && (d_v == 512 || d_v == 576); }

// Whether rows of this width are the wide kernels' (the backward's workspace and
// passes depend on it).
inline bool wide_row(int64_t d_qk) { return d_qk == 576; }

// How a forward of bf16 rows runs: head tiles per workgroup, splits of the slots and
// the kernel, launch_fwd_wide_bf16's (pipelined; nsplit > 1: p.part_o / p.part_ml hold
// the splits' results) or launch_fwd_wide's.
struct WideFwdPlan {
  int nt, nsplit;
  bool piped;
};
WideFwdPlan wide_fwd_plan(int64_t tgs, int64_t hpg, int64_t d_v, int64_t topk, bool may_split);
// qmx (here and below): Q converted from e4m3 codes and 32-channel block scales as it is loaded.
int launch_fwd_wide_bf16(const FwdParams &p, int64_t d_qk, int64_t d_v, int nt, bool qmx, hipStream_t st);

// Forward over all (token, kv group, nt 32-head tiles) items: e4m3 rows (mx: with one
// scale per 32 channels; nt is chosen here), or bf16 rows.
int launch_fwd_wide(const FwdParams &p, int64_t d_qk, int64_t d_v, int nt, bool fp8, hipStream_t st, bool mx = false,
                    bool qmx = false);
// Backward main pass (P, dS and dQ, then the partial dKV rows at CSR positions); bf16 or e4m3.
int launch_bwd_main_wide(const BwdParams &p, int64_t d_qk, int64_t d_v, bool fp8, bool f32p, hipStream_t st);

}  // namespace dsa
