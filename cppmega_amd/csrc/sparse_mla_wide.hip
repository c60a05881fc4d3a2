// SparseMLA forward for wide heads on gfx950 (d_qk = 576 latent + rope with
// d_v = 512: the DeepSeek-V3.2 MLA row and the reference's default head dims; or
// d_v = 576, what a caller that passes no d_v gets): e4m3 and MXFP8 rows, and
// bf16 rows of kv groups of at most 32 heads.  With one head tile there is
// little to share a row tile with, and this kernel's 57 KiB of LDS lets two
// workgroups hide each other's waits: 601 us at s = 4096, 32 heads, top-k 1024,
// against 885 us for the pipelined kernel that larger groups take.
//
// Reference semantics are those of the narrow kernel:
// cppmega/megatron/sparse_mla_ops/tilelang_sparse_mla_fwd.py:137-290 and
// tilelang_sparse_mla_fwd_fp8.py:187-393 (e4m3).
//
// A wide row does not fit one wave's registers: Q over 576 dims is 144 VGPRs
// per 32 heads and the O accumulator over 512 dims is 256.  So one workgroup of
// four waves owns one (token, kv group, 32-head tile) item and the waves split
// the head dims:
//   * the 32 kv rows of a block (36 KiB) are gathered by all 256 threads into
//     one row-major LDS tile (16-byte chunks, one block ahead in registers);
//   * S^T[slot][head] = K Q^T is split over d_qk: wave w runs k-steps
//     [w * KQ, (w + 1) * KQ) with its quarter of Q resident in registers, writes
//     its fp32 partial tile to LDS, and every wave then sums the four partials
//     in wave order, so all waves hold bit-identical scores and run the same
//     online softmax;
//   * O^T[d][head] += V^T P^T is split over d_v: wave w accumulates every
//     fourth 32-column tile of d_v, t = w + 4q (V^T read with transposing LDS
//     reads in accumulator order, P straight from registers).
#include <type_traits>

#include "dsa_common.hpp"
#include "sparse_mla_gather.hpp"
#include "sparse_mla_params.hpp"
#include "sparse_mla_wide.hpp"
#include "sparse_mla_wide_tile.hpp"

namespace dsa {

// Split form of sum_partials for four waves: wave w sums quarter w (64 lanes x
// 4 floats) of the four partial tiles in the same order and writes it to the
// reduced tile Sr; after a barrier every wave reads the whole reduced tile
// (get_reduced), so each reads 8 KiB of LDS instead of 16.
__device__ __forceinline__ void reduce_quarter(const float *Sp, int stride_w, float *Sr, int w) {
  const int lane = lane_id();
  const f32x4 v0 = *reinterpret_cast<const f32x4 *>(Sp + 0 * stride_w + (w * 64 + lane) * 4);
  const f32x4 v1 = *reinterpret_cast<const f32x4 *>(Sp + 1 * stride_w + (w * 64 + lane) * 4);
  const f32x4 v2 = *reinterpret_cast<const f32x4 *>(Sp + 2 * stride_w + (w * 64 + lane) * 4);
  const f32x4 v3 = *reinterpret_cast<const f32x4 *>(Sp + 3 * stride_w + (w * 64 + lane) * 4);
  f32x4 r;
#pragma unroll
  for (int j = 0; j < 4; ++j) r[j] = ((v0[j] + v1[j]) + v2[j]) + v3[j];
  *reinterpret_cast<f32x4 *>(Sr + (w * 64 + lane) * 4) = r;
}
__device__ __forceinline__ void get_reduced(const float *Sr, float (&s)[16]) {
  const int lane = lane_id();
#pragma unroll
  for (int q4 = 0; q4 < 4; ++q4) {
    const f32x4 v = *reinterpret_cast<const f32x4 *>(Sr + (q4 * 64 + lane) * 4);
#pragma unroll
    for (int j = 0; j < 4; ++j) s[4 * q4 + j] = v[j];
  }
}

// ---------------------------------------------------------------------------
// Forward
// ---------------------------------------------------------------------------
template <int D_QK, int D_V, bool FP8, bool MX = false, int NT = 1>
struct WideFwdLds {
  using C = WideCfg<D_QK, D_V, FP8, 256 * NT>;
  static constexpr int NBLK = D_QK / 32;  // MX scale blocks per row
  static constexpr int OFF_KL = 0;
  static constexpr int OFF_KD = OFF_KL + 32 * C::KL_STRIDE;
  static constexpr int OFF_SC = OFF_KD + (FP8 ? 32 * C::KD_STRIDE : 0);
  static constexpr int OFF_SP = (OFF_SC + (FP8 ? (MX ? NBLK : 1) * 32 * 4 : 0) + 15) / 16 * 16;
  static constexpr int SP_W = 16 * 64;  // floats per wave's partial tile
  static constexpr int OFF_SR = OFF_SP + 4 * NT * SP_W * 4;  // a partial tile per wave
  static constexpr int BYTES = OFF_SR + NT * SP_W * 4;       // a reduced tile per head tile
};

// MX partial scores of one wave over its k-steps [k0, k0 + KQ) of d_qk (k0 of
// parity PAR): every 32-channel block (two k-steps; the wave's first or last
// block may be a half that the neighbouring wave completes) accumulates a fresh
// partial on the e4m3 codes, scaled by kv_scale[slot][block] * q_scale[head][block]
// before it joins sacc.  The block scaling is linear, so the four waves'
// partials still sum to the full score.
template <class C, int PAR>
__device__ __forceinline__ void mx_wave_scores(f32x16 &sacc, const unsigned char *Kl, const long (&qreg)[C::KQ],
                                               const float (&qbs)[C::KQ / 2 + 1], const float *Ksc, int k0,
                                               int l32, int g32) {
  const int cb0 = (k0 - PAR) >> 1;  // first block this wave touches
  f32x16 part;
#pragma unroll
  for (int a = 0; a < 16; ++a) part[a] = 0.0f;
#pragma unroll
  for (int k = 0; k < C::KQ; ++k) {
    const long a = *reinterpret_cast<const long *>(Kl + l32 * C::KL_STRIDE + 16 * (k0 + k) + 8 * g32);
    part = __builtin_amdgcn_mfma_f32_32x32x16_fp8_fp8(a, qreg[k], part, 0, 0, 0);
    if (((k + PAR) & 1) || k == C::KQ - 1) {  // the block of k-step k0 + k ends here (for this wave)
      const int cl = (k + PAR) >> 1;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const f32x4 k4 = *reinterpret_cast<const f32x4 *>(Ksc + (cb0 + cl) * 32 + 8 * i + 4 * g32);
#pragma unroll
        for (int j = 0; j < 4; ++j) sacc[4 * i + j] = fmaf(part[4 * i + j], k4[j] * qbs[cl], sacc[4 * i + j]);
      }
#pragma unroll
      for (int a = 0; a < 16; ++a) part[a] = 0.0f;
    }
  }
}

// NT head tiles per workgroup: waves 4 ht .. 4 ht + 3 own 32-head tile ht of
// the item and split its head dims as described above; all 4 NT waves gather
// (and, e4m3, dequantise) the block's kv rows once for the NT tiles.  QMX: the
// bf16 kernel with Q given as e4m3 codes and one scale per 32 channels,
// converted to bf16 as it is loaded.
template <int D_QK, int D_V, bool FP8, bool MX = false, int NT = 1, bool QMX = false>
__global__ void __launch_bounds__(256 * NT) __attribute__((amdgpu_waves_per_eu(D_V <= 512 ? 2 : 1)))
sparse_mla_fwd_wide_kernel(const FwdParams p) {
  static_assert(!MX || FP8, "MX is an e4m3 mode");
  static_assert(!QMX || !FP8, "QMX converts Q for the bf16 kernel");
  if (p.gate != nullptr && *p.gate != p.gate_run) return;  // workgroup-uniform: the call's other kernel computes it
  using C = WideCfg<D_QK, D_V, FP8, 256 * NT>;
  using L = WideFwdLds<D_QK, D_V, FP8, MX, NT>;
  typedef typename std::conditional<FP8, long, bf16x8>::type qop_t;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];

  const int lane = lane_id(), wv = __builtin_amdgcn_readfirstlane(wave_id());
  const int ht = wv >> 2, w = wv & 3;  // head tile within the item, wave within the tile
  const int g32 = lane >> 5, l32 = lane & 31;
  const int64_t item = xcd_remap(blockIdx.x, gridDim.x);
  const int ntg = (p.ntiles + NT - 1) / NT;  // items per (token, kv group)
  const int tile = (int)(item % ntg) * NT + ht;
  const int64_t rest = item / ntg;
  const int64_t g = rest % p.G;
  const int64_t tok = rest / p.G;
  const int64_t b = tok / p.S;

  unsigned char *Kl = smem + L::OFF_KL;
  unsigned char *Kd = smem + L::OFF_KD;
  float *Ksc = reinterpret_cast<float *>(smem + L::OFF_SC);
  float *Sp = reinterpret_cast<float *>(smem + L::OFF_SP);
  float *Sr = reinterpret_cast<float *>(smem + L::OFF_SR) + ht * L::SP_W;
  const unsigned char *Vsrc = FP8 ? Kd : Kl;
  constexpr int V_STRIDE = FP8 ? C::KD_STRIDE : C::KL_STRIDE;

  const int h_local = tile * 32 + l32;
  const bool head_ok = h_local < p.hpg;
  const int64_t qrow = tok * p.H + g * p.hpg + h_local;
  const int32_t *idx_row = p.idx + (tok * p.G + g) * p.topk;
  const unsigned char *kv_b = p.kv + ((b * p.S_kv) * p.G + g) * C::ROWB;
  // kv scales: [B, S_kv] per row, or MX [B, S_kv, G, D_QK / 32] per (row, block)
  const float *kv_scale_b = !FP8 ? nullptr : (MX ? p.kv_scale + ((b * p.S_kv) * p.G + g) * L::NBLK
                                                 : p.kv_scale + b * p.S_kv);
  const uint32_t sc_pitch = MX ? (uint32_t)(p.G * L::NBLK) : 1u;
  const uint32_t row_pitch = (uint32_t)(p.G * C::ROWB);
  const int nblk = (int)((p.topk + 31) / 32);

  // indices two blocks ahead as raw loads, masked where they are used a block
  // later: the block loop never waits on an index load it has just issued
  const auto idx_rs = slot_rsrc(idx_row, p.topk);
  int idx_cur = slot_index(load_slot_raw(idx_rs, 0, l32), 0, l32, p.topk, p.S_kv);
  int raw_nxt = load_slot_raw(idx_rs, 1, l32);
  typename C::Regs rg;
  wide_issue<C, FP8, MX>(rg, kv_b, kv_scale_b, idx_cur, row_pitch, sc_pitch);

  // this wave's quarter of Q as the B operand: lane = head, 8 consecutive d per k-step
  const int k0 = w * C::KQ;
  qop_t qreg[C::KQ];
#pragma unroll
  for (int k = 0; k < C::KQ; ++k) {
    if constexpr (FP8) {
      qreg[k] = head_ok ? *reinterpret_cast<const long *>(p.q + qrow * D_QK + 16 * (k0 + k) + 8 * g32) : 0l;
    } else if constexpr (QMX) {
      const int d0 = 16 * (k0 + k) + 8 * g32;  // 8 channels of block d0 / 32
      uint2 c8 = {0u, 0u};
      float sc = 0.0f;
      if (head_ok) {
        c8 = *reinterpret_cast<const uint2 *>(p.q + qrow * D_QK + d0);
        sc = p.q_scale[qrow * (D_QK / 32) + (d0 >> 5)];
      }
      qreg[k] = e4m3x8_to_bf16_scaled(c8.x, c8.y, sc);
    } else {
      i32x4 v = {0, 0, 0, 0};
      if (head_ok) v = ld_global_16(p.q + (qrow * D_QK + 16 * (k0 + k) + 8 * g32) * 2);
      qreg[k] = as_bf16x8(v);
    }
  }
  float qsc = 1.0f;
  if constexpr (FP8 && !MX) qsc = p.q_scale[tok];
  const float tscale = p.sl2 * qsc;
  // MX: this lane's head's scales of the blocks this wave's k-steps touch
  // (q_scale [B, S, H, D_QK / 32])
  const int par = (k0 & 1);
  float qbs[C::KQ / 2 + 1];
  if constexpr (MX) {
    const int cb0 = (k0 - par) >> 1;
#pragma unroll
    for (int cl = 0; cl < C::KQ / 2 + 1; ++cl)
      qbs[cl] = (head_ok && cb0 + cl < L::NBLK) ? p.q_scale[qrow * L::NBLK + cb0 + cl] : 0.0f;
  }

  float m_run = kNegBig, l_run = 0.0f;
  f32x16 oacc[C::DTW];
#pragma unroll
  for (int t = 0; t < C::DTW; ++t)
#pragma unroll
    for (int a = 0; a < 16; ++a) oacc[t][a] = 0.0f;

  for (int blk = 0; blk < nblk; ++blk) {
    wide_store<C, FP8, C::NCH_V, C::KD_STRIDE, MX>(rg, Kl, Kd, Ksc);
    const uint64_t vmask = __ballot(idx_cur >= 0);
    __syncthreads();  // the block's rows are in LDS
    const int raw_nn = load_slot_raw(idx_rs, blk + 2, l32);
    const int idx_nxt = slot_index(raw_nxt, blk + 1, l32, p.topk, p.S_kv);
    if (blk + 1 < nblk) wide_issue<C, FP8, MX>(rg, kv_b, kv_scale_b, idx_nxt, row_pitch, sc_pitch);

    // ---- partial S^T = K Q^T over this wave's k-steps ----
    f32x16 sacc;
#pragma unroll
    for (int a = 0; a < 16; ++a) sacc[a] = 0.0f;
    if constexpr (MX) {
      if (par) mx_wave_scores<C, 1>(sacc, Kl, qreg, qbs, Ksc, k0, l32, g32);
      else mx_wave_scores<C, 0>(sacc, Kl, qreg, qbs, Ksc, k0, l32, g32);
    }
#pragma unroll
    for (int k = 0; k < (MX ? 0 : C::KQ); ++k) {
      if constexpr (FP8) {
        const long a = *reinterpret_cast<const long *>(Kl + l32 * C::KL_STRIDE + 16 * (k0 + k) + 8 * g32);
        sacc = __builtin_amdgcn_mfma_f32_32x32x16_fp8_fp8(a, qreg[k], sacc, 0, 0, 0);
      } else {
        const i32x4 a = *reinterpret_cast<const i32x4 *>(Kl + l32 * C::KL_STRIDE + (16 * (k0 + k) + 8 * g32) * 2);
        sacc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(as_bf16x8(a), qreg[k], sacc, 0, 0, 0);
      }
    }
    put_partial(Sp + wv * L::SP_W, sacc);
    __syncthreads();  // all partial tiles written
    reduce_quarter(Sp + 4 * ht * L::SP_W, L::SP_W, Sr, w);
    __syncthreads();  // the head tile's reduced scores are whole
    float s[16];
    get_reduced(Sr, s);

    // ---- online softmax (log2 domain, lazy rescale; identical in every wave) ----
    // this lane's slots are 8i + 4*g32 + j: their valid bits sit at 8i + j of lmask;
    // a block without masked slots (the common case, wave-uniform) skips the tests
    const bool all_valid = (uint32_t)vmask == 0xffffffffu;
    const uint32_t lmask = (uint32_t)vmask >> (4 * g32);
    float xs[16];
    float mloc = kNegBig;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      float ksc4[4] = {1.0f, 1.0f, 1.0f, 1.0f};
      if constexpr (FP8 && !MX) {
        const f32x4 s4 = *reinterpret_cast<const f32x4 *>(Ksc + 8 * i + 4 * g32);
        ksc4[0] = s4[0]; ksc4[1] = s4[1]; ksc4[2] = s4[2]; ksc4[3] = s4[3];
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        float v = s[4 * i + j];
        if constexpr (FP8 && !MX) v *= ksc4[j];
        xs[4 * i + j] = v;  // raw score, scaled inside the exp
      }
    }
    if (!all_valid) {
#pragma unroll
      for (int a = 0; a < 16; ++a)
        if (!((lmask >> (8 * (a >> 2) + (a & 3))) & 1u)) xs[a] = -INFINITY;
    }
#pragma unroll
    for (int a = 0; a < 16; a += 2) mloc = fmaxf(mloc, fmaxf(xs[a], xs[a + 1]));
    mloc = max_halves(mloc) * tscale;
    if (__ballot(mloc > m_run + 8.0f) != 0ull) {
      const float m_new = fmaxf(m_run, mloc);
      const float alpha = exp2_fast(m_run - m_new);
      l_run *= alpha;
      m_run = m_new;
#pragma unroll
      for (int dt = 0; dt < C::DTW; ++dt)
#pragma unroll
        for (int a = 0; a < 16; ++a) oacc[dt][a] *= alpha;
    }
    float t[16];
    float lsum = 0.0f;
#pragma unroll
    for (int a = 0; a < 16; ++a) {
      t[a] = exp2_fast(fmaf(xs[a], tscale, -m_run));
      lsum += t[a];
    }
    lsum = sum_halves(lsum);
    l_run += lsum;

    // ---- O^T[d][head] += V^T[d][slot] P^T[slot][head] on this wave's d_v tiles ----
#pragma unroll
    for (int kc = 0; kc < 2; ++kc) {
      i32x4 pb;
#pragma unroll
      for (int e = 0; e < 4; ++e) pb[e] = (int)pack_bf16x2(t[8 * kc + 2 * e], t[8 * kc + 2 * e + 1]);
      const bf16x8 bop = as_bf16x8(pb);
#pragma unroll
      for (int dt = 0; dt < C::DTW; ++dt) {
        const int tv = w + 4 * dt;
        if (tv < C::DT) {
          const i32x4 av = tr_operand(Vsrc, V_STRIDE, tv * 32, 16 * kc, 8, 4);
          oacc[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(as_bf16x8(av), bop, oacc[dt], 0, 0, 0);
        }
      }
    }
    __syncthreads();  // rows and partial tiles consumed before the next block overwrites them
    idx_cur = idx_nxt;
    raw_nxt = raw_nn;
  }

  // ---- normalise and write: lane = head l32, d = (w + 4*dt)*32 + 8i + 4*g32 + j ----
  if (head_ok) {
    const float inv = l_run > 0.0f ? 1.0f / l_run : 0.0f;
    uint16_t *orow = p.out + qrow * D_V;
#pragma unroll
    for (int dt = 0; dt < C::DTW; ++dt) {
      const int tv = w + 4 * dt;
      if (tv < C::DT) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const i32x2 pk = {(int)pack_bf16x2(oacc[dt][4 * i] * inv, oacc[dt][4 * i + 1] * inv),
                            (int)pack_bf16x2(oacc[dt][4 * i + 2] * inv, oacc[dt][4 * i + 3] * inv)};
          *reinterpret_cast<i32x2 *>(orow + tv * 32 + 8 * i + 4 * g32) = pk;
        }
      }
    }
    if (w == 0 && g32 == 0) p.lse[qrow] = l_run > 0.0f ? log2f(l_run) + m_run : -INFINITY;
  }
}

template <int D_QK, int D_V, bool FP8, bool MX, int NT, bool QMX = false>
static int launch_fwd_wide_nt(const FwdParams &p, hipStream_t st) {
  using L = WideFwdLds<D_QK, D_V, FP8, MX, NT>;
  const size_t lds = L::BYTES;
  if (lds > 64 * 1024) {
    hipError_t e = hipFuncSetAttribute((const void *)sparse_mla_fwd_wide_kernel<D_QK, D_V, FP8, MX, NT, QMX>,
                                       hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return set_error(DSA_ERR_HIP, "sparse_mla_fwd(wide): LDS attribute: %s", hipGetErrorString(e));
  }
  const int64_t nitems = p.B * p.S * p.G * ((p.ntiles + NT - 1) / NT);  // one workgroup per item
  if (nitems >= (1ll << 31)) return set_error(DSA_ERR_INVALID_ARG, "sparse_mla_fwd(wide): grid too large");
  hipLaunchKernelGGL((sparse_mla_fwd_wide_kernel<D_QK, D_V, FP8, MX, NT, QMX>), dim3((unsigned)nitems), dim3(256 * NT),
                     lds, st, p);
  return check_launch("sparse_mla_fwd(wide)");
}

// e4m3: two head tiles per workgroup when a kv group has at least 64 heads (the
// gather and dequantisation of a block serve both), else one.  bf16: nt.
template <int D_QK, int D_V, bool FP8, bool MX = false, bool QMX = false>
static int launch_fwd_wide_t(const FwdParams &p, int nt, hipStream_t st) {
  return (FP8 ? p.ntiles : nt) >= 2 ? launch_fwd_wide_nt<D_QK, D_V, FP8, MX, 2, QMX>(p, st)
                                    : launch_fwd_wide_nt<D_QK, D_V, FP8, MX, 1, QMX>(p, st);
}

int launch_fwd_wide(const FwdParams &p, int64_t d_qk, int64_t d_v, int nt, bool fp8, hipStream_t st, bool mx, bool qmx) {
  if (qmx) {
    if (d_qk == 576 && d_v == 512) return launch_fwd_wide_t<576, 512, false, false, true>(p, nt, st);
    return set_error(DSA_ERR_UNSUPPORTED, "sparse_mla_fwd(wide): no converted-Q kernel for d_qk=%lld d_v=%lld",
                     (long long)d_qk, (long long)d_v);
  }
  if (mx) {
    if (d_qk == 576 && d_v == 512) return launch_fwd_wide_t<576, 512, true, true>(p, nt, st);
    return set_error(DSA_ERR_UNSUPPORTED, "sparse_mla_fwd(wide): no MXFP8 kernel for d_qk=%lld d_v=%lld",
                     (long long)d_qk, (long long)d_v);
  }
  if (d_qk == 576 && d_v == 512)
    return fp8 ? launch_fwd_wide_t<576, 512, true>(p, nt, st) : launch_fwd_wide_t<576, 512, false>(p, nt, st);
  if (d_qk == 576 && d_v == 576)
    return fp8 ? launch_fwd_wide_t<576, 576, true>(p, nt, st) : launch_fwd_wide_t<576, 576, false>(p, nt, st);
  return set_error(DSA_ERR_UNSUPPORTED, "sparse_mla_fwd(wide): no kernel for d_qk=%lld d_v=%lld", (long long)d_qk,
                   (long long)d_v);
}

}  // namespace dsa
