// SparseMLA forward for wide heads, bf16 rows (d_qk = 576; d_v = 512 or 576), on
// gfx950; semantics of cppmega/megatron/sparse_mla_ops/tilelang_sparse_mla_fwd.py:137-290.
//
// One workgroup of NW waves per (token, kv group, NT 32-head tiles, split of the
// slots); per block of 32 slots:
//   S^T (M = slot, N = head): wave = (head tile, one of KP parts of the k-steps),
//     its part of Q resident in registers, K rows from the LDS row tile; the
//     parts meet through LDS;
//   online softmax: a wave takes HW heads of one tile, LPH lanes per head with
//     32 / LPH slots each; P goes to LDS as bf16 [head][slot];
//   O^T[d][head] += V^T P: wave w owns the 16-column tiles w, w + NW, ... of d_v
//     for all heads, V^T by transposed reads of the row tile.
// At 128 heads (NT = 4) a block's rows are fetched once for all of them and the
// products, not LDS or the gather, set the pace: per SIMD 2176 cycles of MFMA a
// block beside about 1700 of LDS.  Registers: O takes 128 and Q 72 of the 256 of
// two waves per SIMD.
// Software pipeline, two barriers a block: block j's S products between the first
// and the second; block j - 1's PV products between the second and the next,
// covering the latency of the exchange and the softmax of block j.  Block j + 1's
// rows are fetched meanwhile by LDS-DMA loads (three row tiles rotate).
//
// Splits: a grid of few tokens (decode) leaves most compute units idle while each
// workgroup walks its top-k alone, so the host may split the slots over nsplit
// workgroups; each leaves its unnormalised fp32 O with its reference maximum m
// and sum l, and fwd_wide_combine_kernel adds them in split order.
#include "dsa_common.hpp"
#include "sparse_mla_gather.hpp"
#include "sparse_mla_params.hpp"
#include "sparse_mla_wide.hpp"
#include "sparse_mla_wide_tile.hpp"

namespace dsa {

template <int D_QK, int D_V, int NT, int NW_>
struct WideFwd {
  static constexpr int NW = NW_, NTHR = 64 * NW, KP = NW / NT;
  static constexpr int FW = NW / 2;                          // the waves that fetch the rows
  using T = DmaTile<D_QK, FW>;
  static constexpr int KS = D_QK / 16 / KP;                  // k-steps per wave: KP i + kq
  static constexpr int NDT = D_V / 16, DTW = (NDT + NW - 1) / NW;
  static constexpr int HEADS = 32 * NT, HW = HEADS / NW;     // heads per wave in the softmax
  static constexpr int LPH = 64 / HW, SPL4 = 8 / LPH;        // lanes per head; 4-slot groups per lane
  static constexpr int SP_W = 32 * 32;
  static constexpr int PT_BYTES = 32 * 32 * 2;               // one tile of P
  static constexpr int OFF_K = 0;
  static constexpr int OFF_SP = OFF_K + 3 * T::BYTES;
  static constexpr int OFF_P = OFF_SP + NW * SP_W * 4;       // two blocks
  static constexpr int OFF_AL = OFF_P + 2 * NT * PT_BYTES;   // [2][HEADS] rescale factors, then [HEADS] 1 / l
  static constexpr int OFF_FL = OFF_AL + 3 * HEADS * 4;      // [2][NW] the waves' rescale flags
  static constexpr int BYTES = OFF_FL + 2 * NW * 4;
  static_assert(D_QK / 16 % KP == 0 && (KP == 2 || KP == 4) && (HW == 8 || HW == 16), "wave split");
  static_assert(BYTES <= 160 * 1024, "wide forward LDS");
};

template <int D_QK, int D_V, int NT, int NW, bool QMX>
__global__ void __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(NW / 4)))
sparse_mla_fwd_wide_bf16_kernel(const FwdParams p) {
  if (p.gate != nullptr && *p.gate != p.gate_run) return;  // workgroup-uniform: the call's other kernel computes it
  using C = WideFwd<D_QK, D_V, NT, NW>;
  using T = typename C::T;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const int lane = lane_id(), w = wave_id();
  const int g32 = lane >> 5, l32 = lane & 31, g16 = lane >> 4, l16 = lane & 15;
  const int64_t item = xcd_remap(blockIdx.x, gridDim.x);
  const int split = (int)(item % p.nsplit);
  const int64_t it = item / p.nsplit;
  const int ntg = (p.ntiles + NT - 1) / NT;
  const int tile0 = (int)(it % ntg) * NT;
  const int64_t tg = it / ntg;
  const int64_t g = tg % p.G, tok = tg / p.G, b = tok / p.S;
  unsigned char *K = smem + C::OFF_K;
  float *Sp = reinterpret_cast<float *>(smem + C::OFF_SP);
  unsigned char *P = smem + C::OFF_P;
  float *AL = reinterpret_cast<float *>(smem + C::OFF_AL);
  int *FL = reinterpret_cast<int *>(smem + C::OFF_FL);

  const int64_t head0 = tok * p.H + g * p.hpg + tile0 * 32;
  const int nheads = p.hpg - tile0 * 32 < C::HEADS ? p.hpg - tile0 * 32 : C::HEADS;
  const unsigned char *kv_b = p.kv + ((b * p.S_kv) * p.G + g) * T::ROWB;
  const uint32_t row_pitch = (uint32_t)(p.G * T::ROWB);
  const i32x4 kv_rs = make_buffer_words(kv_b, (uint32_t)(p.S_kv * p.G * T::ROWB - g * T::ROWB));
  const auto idx_rs = slot_rsrc(p.idx + tg * p.topk, p.topk);
  const uint32_t k_lds = lds_address(K);

  // this workgroup's blocks [b0, b1) of the item's, up to its last valid slot
  int b0 = 0, b1 = valid_blocks<16>(idx_rs, p.topk, p.S_kv);
  if (p.nsplit > 1) {
    const int per = (b1 + p.nsplit - 1) / p.nsplit;
    b0 = split * per < b1 ? split * per : b1;
    b1 = b0 + per < b1 ? b0 + per : b1;
  }
  auto fetch = [&](int tile, int idx) {
    dma_tile_issue<T>(k_lds + (uint32_t)(tile * T::BYTES), kv_rs, idx >= 0 ? (uint32_t)idx * row_pitch : kMaskedOff, w);
  };
  const int idx0 = slot_index(load_slot_raw(idx_rs, b0, l32), b0, l32, p.topk, p.S_kv);
  int idx_nxt = slot_index(load_slot_raw(idx_rs, b0 + 1, l32), b0 + 1, l32, p.topk, p.S_kv);
  uint32_t vm = (uint32_t)__ballot(idx0 >= 0);
  if (w < C::FW) fetch(0, idx0);

  // this wave's part of Q: head l32 of tile ht, k-steps KP i + kq
  const int ht = w / C::KP, kq = w % C::KP;
  i32x4 q[C::KS];
  {
    const int h = 32 * ht + l32;
#pragma unroll
    for (int i = 0; i < C::KS; ++i) {
      const int d0 = 16 * (C::KP * i + kq) + 8 * g32;
      q[i] = i32x4{0, 0, 0, 0};
      if (h < nheads) {
        if constexpr (QMX) {  // e4m3 codes and one scale per 32 channels, converted to bf16
          const uint2 c8 = *reinterpret_cast<const uint2 *>(p.q + (head0 + h) * D_QK + d0);
          q[i] = __builtin_bit_cast(i32x4, e4m3x8_to_bf16_scaled(c8.x, c8.y, p.q_scale[(head0 + h) * (D_QK / 32) + (d0 >> 5)]));
        } else {
          q[i] = ld_global_16(p.q + ((head0 + h) * D_QK + d0) * 2);
        }
      }
    }
  }
  // S operand of k-step KP i + kq: row l32, chunk 2 (KP i + kq) + g32 (KP = 2: i and i + 2 are a panel apart; 4: i and i + 1)
  constexpr int kPh = 4 / C::KP;
  int ka[kPh];
#pragma unroll
  for (int u = 0; u < kPh; ++u) ka[u] = tile_byte(l32, 2 * (C::KP * u + kq) + g32);
  const int et = w * C::HW / 32;  // the head tile this wave's softmax heads are of

  float m_run = kNegBig, l_run = 0.0f;
  f32x4 o[C::DTW][2 * NT];
#pragma unroll
  for (int i = 0; i < C::DTW; ++i)
#pragma unroll
    for (int h = 0; h < 2 * NT; ++h) o[i][h] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

  // O (rescaled where the softmax of buffer `buf` moved a reference maximum) += V^T P of that buffer
  auto pv_step = [&](const unsigned char *Kb, int buf) {
    const int ln = lane_here(), c16 = ln & 15, cg = ln >> 4;
    if (__ballot(FL[buf * NW + (ln & (NW - 1))] != 0) != 0ull) {
#pragma unroll
      for (int h = 0; h < 2 * NT; ++h) {
        const float a = AL[buf * C::HEADS + 16 * h + c16];
#pragma unroll
        for (int i = 0; i < C::DTW; ++i) o[i][h] *= a;
      }
    }
    // V^T of d tile w + NW i: rows 8 cg + (lane % 16) / 4 (+ 4), columns 4 (lane % 4) .. of the tile
    int vt[2];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int c = c16 & 3;
      vt[u] = tile_byte(8 * cg + 4 * u + (c16 >> 2), 2 * (w & 3) + (c >> 1)) + (c & 1) * 8 + (w >> 2) * T::PANEL;
    }
    // P[head][slot]: 64-byte rows, 16-byte chunk c of head h at c ^ ((h >> 2) & 3)
    const int p_rd = buf * NT * C::PT_BYTES + c16 * 64 + ((cg ^ ((c16 >> 2) & 3)) * 16);
    i32x4 av[C::DTW];
#pragma unroll
    for (int i = 0; i < C::DTW; ++i) {
      const i32x2 r0 = ds_read_tr16(Kb + vt[0] + i * (NW / 4) * T::PANEL);
      const i32x2 r1 = ds_read_tr16(Kb + vt[1] + i * (NW / 4) * T::PANEL);
      av[i] = i32x4{r0[0], r0[1], r1[0], r1[1]};
    }
#pragma unroll
    for (int h = 0; h < 2 * NT; ++h) {
      const i32x4 bv = *reinterpret_cast<const i32x4 *>(P + p_rd + (h >> 1) * C::PT_BYTES + (h & 1) * 1024);
#pragma unroll
      for (int i = 0; i < C::DTW; ++i)
        if (C::NDT % NW == 0 || i + 1 < C::DTW || w < C::NDT % NW)
          o[i][h] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(av[i]), as_bf16x8(bv), o[i][h], 0, 0, 0);
    }
  };

  int kb = 0, kp = 0;  // row tiles of block j and of block j - 1
  for (int j = b0; j < b1; ++j) {
    const int kn = kb == 2 ? 0 : kb + 1, cur = (j - b0) & 1;
    const unsigned char *Kj = K + kb * T::BYTES;
    __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): block j's rows, issued a block ago
    __syncthreads();  // block j's rows and block j - 1's P are in LDS; block j - 2's rows are consumed
    const int raw = load_slot_raw(idx_rs, j + 2, l32);
    if (w < C::FW) fetch(kn, idx_nxt);  // block j + 1 (past the last valid: zeros or unused rows)
    f32x16 acc;
#pragma unroll
    for (int a = 0; a < 16; ++a) acc[a] = 0.0f;
#pragma unroll
    for (int i = 0; i < C::KS; ++i) {
      const i32x4 a = *reinterpret_cast<const i32x4 *>(Kj + ka[i % kPh] + (i / kPh) * T::PANEL);
      acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(as_bf16x8(a), as_bf16x8(q[i]), acc, 0, 0, 0);
    }
    put_partial(Sp + w * C::SP_W, acc);
    __syncthreads();  // partial tiles whole

    // softmax: head eh of tile et, 4-slot groups (i, eg) with i = ei .. ei + SPL4 - 1: slots 8 i + 4 eg ..
    const int ln = lane_here(), eh = (w * C::HW) % 32 + (ln & (C::HW - 1));
    const int eq = ln / C::HW, eg = eq & 1, ei = (eq >> 1) * C::SPL4;
    f32x4 s[C::SPL4];
    {
      const float *sp = Sp + et * C::KP * C::SP_W + ((ei * 2 + eg) * 32 + eh) * 4;
#pragma unroll
      for (int u = 0; u < C::SPL4; ++u) {
        s[u] = *reinterpret_cast<const f32x4 *>(sp + u * 256);
#pragma unroll
        for (int k = 1; k < C::KP; ++k) s[u] += *reinterpret_cast<const f32x4 *>(sp + k * C::SP_W + u * 256);
      }
    }
    if (j > b0) pv_step(K + kp * T::BYTES, cur ^ 1);

    // online softmax (log2 domain, lazy rescale)
    float mloc = kNegBig;
#pragma unroll
    for (int u = 0; u < C::SPL4; ++u)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        if (!((vm >> (8 * (ei + u) + 4 * eg + e)) & 1u)) s[u][e] = -INFINITY;
        mloc = fmaxf(mloc, s[u][e]);
      }
#pragma unroll
    for (int off = C::HW; off < 32; off <<= 1) mloc = fmaxf(mloc, __shfl_xor(mloc, off, 64));
    mloc = max_halves(mloc) * p.sl2;
    const bool moved = __ballot(mloc > m_run + 8.0f) != 0ull;  // wave-uniform
    if (moved) {
      const float m_new = fmaxf(m_run, mloc);
      const float alpha = exp2_fast(m_run - m_new);
      l_run *= alpha;
      m_run = m_new;
      if (eq == 0) AL[cur * C::HEADS + et * 32 + eh] = alpha;
    } else if (eq == 0) {
      AL[cur * C::HEADS + et * 32 + eh] = 1.0f;
    }
    if (lane == 0) FL[cur * NW + w] = moved ? 1 : 0;
#pragma unroll
    for (int u = 0; u < C::SPL4; ++u) {
      float t[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        t[e] = exp2_fast(fmaf(s[u][e], p.sl2, -m_run));
        l_run += t[e];
      }
      *reinterpret_cast<i32x2 *>(P + (cur * NT + et) * C::PT_BYTES + eh * 64 + (((ei + u) ^ ((eh >> 2) & 3)) * 16) + eg * 8) =
          i32x2{(int)pack_bf16x2(t[0], t[1]), (int)pack_bf16x2(t[2], t[3])};
    }
    vm = (uint32_t)__ballot(idx_nxt >= 0);
    idx_nxt = slot_index(raw, j + 2, l32, p.topk, p.S_kv);
    kp = kb;
    kb = kn;
  }
  __builtin_amdgcn_s_waitcnt(0x0F70);  // the loads past the last block have landed before the LDS is given up
  // l over the lanes of a head
  const int eh = (w * C::HW) % 32 + (lane & (C::HW - 1)), eq = lane / C::HW;
#pragma unroll
  for (int off = C::HW; off < 32; off <<= 1) l_run += __shfl_xor(l_run, off, 64);
  l_run = sum_halves(l_run);
  if (eq == 0) AL[2 * C::HEADS + et * 32 + eh] = l_run > 0.0f ? 1.0f / l_run : 0.0f;
  __syncthreads();
  if (b1 > b0) pv_step(K + kp * T::BYTES, (b1 - b0 - 1) & 1);

  const int sh = et * 32 + eh;  // this lane's softmax head
  if (p.nsplit > 1) {
    const int64_t row0 = (tg * p.nsplit + split) * p.hpg + tile0 * 32;
    if (eq == 0 && sh < nheads) {
      p.part_ml[(row0 + sh) * 2] = m_run;
      p.part_ml[(row0 + sh) * 2 + 1] = l_run;
    }
    if (b1 > b0) {
#pragma unroll
      for (int i = 0; i < C::DTW; ++i)
        if (C::NDT % NW == 0 || i + 1 < C::DTW || w < C::NDT % NW)
#pragma unroll
          for (int h = 0; h < 2 * NT; ++h)
            if (16 * h + l16 < nheads)
              *reinterpret_cast<f32x4 *>(p.part_o + (row0 + 16 * h + l16) * D_V + (w + NW * i) * 16 + 4 * g16) = o[i][h];
    }
    return;
  }
  // lane = head 16 h + l16, d = 16 tile + 4 g16 ..
#pragma unroll
  for (int h = 0; h < 2 * NT; ++h) {
    const float inv = AL[2 * C::HEADS + 16 * h + l16];
    if (16 * h + l16 < nheads) {
#pragma unroll
      for (int i = 0; i < C::DTW; ++i)
        if (C::NDT % NW == 0 || i + 1 < C::DTW || w < C::NDT % NW)
          *reinterpret_cast<i32x2 *>(p.out + (head0 + 16 * h + l16) * D_V + (w + NW * i) * 16 + 4 * g16) =
              i32x2{(int)pack_bf16x2(o[i][h][0] * inv, o[i][h][1] * inv), (int)pack_bf16x2(o[i][h][2] * inv, o[i][h][3] * inv)};
    }
  }
  if (eq == 0 && sh < nheads) p.lse[head0 + sh] = l_run > 0.0f ? log2f(l_run) + m_run : -INFINITY;
}

// One wave per (token, head): the splits' O and l brought to their largest m and
// added in split order; a split without a valid slot (l = 0) left no O.
template <int D_V>
__global__ void __launch_bounds__(256) fwd_wide_combine_kernel(const FwdParams p) {
  constexpr int NCH = D_V / 4, CPL = (NCH + 63) / 64;  // 16-byte chunks of a row, and per lane
  const int lane = lane_id();
  const int64_t r = (int64_t)blockIdx.x * 4 + wave_id();  // tok * H + head
  if (r >= p.B * p.S * p.H) return;
  const int64_t tok = r / p.H;
  const int h = (int)(r - tok * p.H), g = h / p.hpg;
  const int64_t row0 = (tok * p.G + g) * p.nsplit * p.hpg + (h - g * p.hpg);
  float m = kNegBig;
  for (int s = 0; s < p.nsplit; ++s) {
    const float *ml = p.part_ml + (row0 + (int64_t)s * p.hpg) * 2;
    if (ml[1] > 0.0f) m = fmaxf(m, ml[0]);
  }
  float l = 0.0f;
  f32x4 o[CPL];
#pragma unroll
  for (int c = 0; c < CPL; ++c) o[c] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  for (int s = 0; s < p.nsplit; ++s) {
    const int64_t row = row0 + (int64_t)s * p.hpg;
    const float ls = p.part_ml[row * 2 + 1];
    if (ls == 0.0f) continue;  // wave-uniform (a NaN sum joins, as it does unsplit)
    const float a = exp2_fast(p.part_ml[row * 2] - m);
    l += ls * a;
#pragma unroll
    for (int c = 0; c < CPL; ++c)
      if (lane + 64 * c < NCH) o[c] += a * *reinterpret_cast<const f32x4 *>(p.part_o + row * D_V + (lane + 64 * c) * 4);
  }
  const float inv = l > 0.0f ? 1.0f / l : 0.0f;
#pragma unroll
  for (int c = 0; c < CPL; ++c)
    if (lane + 64 * c < NCH)
      *reinterpret_cast<i32x2 *>(p.out + r * D_V + (lane + 64 * c) * 4) =
          i32x2{(int)pack_bf16x2(o[c][0] * inv, o[c][1] * inv), (int)pack_bf16x2(o[c][2] * inv, o[c][3] * inv)};
  if (lane == 0) p.lse[r] = l > 0.0f ? log2f(l) + m : -INFINITY;
}

template <int D_QK, int D_V, int NT, int NW, bool QMX>
static int launch_wide_bf16(const FwdParams &p, hipStream_t st) {
  using C = WideFwd<D_QK, D_V, NT, NW>;
  const auto kernel = sparse_mla_fwd_wide_bf16_kernel<D_QK, D_V, NT, NW, QMX>;
  const hipError_t e = hipFuncSetAttribute((const void *)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, C::BYTES);
  if (e != hipSuccess) return set_error(DSA_ERR_HIP, "sparse_mla_fwd(wide): LDS attribute: %s", hipGetErrorString(e));
  const int64_t n = p.B * p.S * p.G * ((p.ntiles + NT - 1) / NT) * p.nsplit;
  if (n >= (1ll << 31)) return set_error(DSA_ERR_INVALID_ARG, "sparse_mla_fwd(wide): grid too large");
  hipLaunchKernelGGL(kernel, dim3((unsigned)n), dim3(C::NTHR), C::BYTES, st, p);
  int rc = check_launch("sparse_mla_fwd(wide)");
  if (rc || p.nsplit == 1) return rc;
  hipLaunchKernelGGL(fwd_wide_combine_kernel<D_V>, dim3((unsigned)((p.B * p.S * p.H + 3) / 4)), dim3(256), 0, st, p);
  return check_launch("sparse_mla_fwd(wide combine)");
}

// Microseconds of one launch over tgs (token, kv group) pairs of hpg heads and nblk
// blocks of 32 slots: a workgroup's prologue and epilogue and its time a block, each
// with what 256 workgroups at once add to it, by the rounds that the grid takes on
// 256 compute units.  Fitted to graph-replayed launches of 1 to 2048 tokens, 16 to
// 256 heads, top-32 to top-2048 (the plan that it picks took 0.9% longer than the
// best of the kernels over those, and at most 11% longer).
//   kernel of launch_fwd_wide, one tile: the shortest prologue, and two workgroups
//     share a compute unit (1 token, 128 heads, top-64: 8.8 us; pipelined, four
//     tiles: 19.3); two tiles: half the gathers (100 tokens, 96 heads, top-64:
//     13.7 us; one tile 14.7);
//   pipelined, two or four tiles: a block's rows serve all of them (2048 tokens, 128
//     heads, top-256: 304 us with four tiles, 371 with one, 394 with two; s = 2048,
//     top-k 2048: 1358 us with four, 1957 with two);
//   pipelined with split slots: the combination's launch and, per 2 KiB fp32 row
//     that it reads, its traffic (16 tokens, 128 heads, top-2048: 40 us as two tiles
//     x 8 splits, 49 as four x 16, 130 unsplit; 1 token: 28 us as one x 16, 127
//     unsplit; but 64 tokens, 128 heads, top-256: 37 us as four x 2, 22 as one tile
//     of the other kernel).
static double wide_fwd_us(bool piped, int nt, int64_t nsplit, int64_t tgs, int64_t hpg, int64_t nblk) {
  const int64_t tiles = (hpg + 31) / 32, wg = tgs * ((tiles + nt - 1) / nt) * nsplit;
  const double per = (double)((nblk + nsplit - 1) / nsplit), x = (double)wg / 256;
  if (nsplit > 1) {
    const double rows = (double)(tgs * hpg * nsplit) / 4096;
    if (nt == 1) return 11.0 + 1.46 * per + 1.9 * x + 3.8 * rows;
    return nt == 2 ? 15.6 + 1.65 * per + 2.9 * x + 2.5 * rows : 19.0 + 2.1 * per + 3.0 * x + 2.5 * rows;
  }
  const int64_t full = wg / 256;
  if (!piped && nt == 1) {
    const auto round = [&](double y) {  // y * 256 workgroups, two of them on a compute unit past one each
      if (y <= 0) return 0.0;
      return y <= 1 ? 5.6 + 1.5 * y + (1.7 + 0.1 * y) * per : 8.0 + 2.3 * y + 2.36 * per;
    };
    if (x <= 2) return round(x);
    // more rounds: they run into each other where a workgroup has few blocks
    const int64_t two = full / 2;
    const double flow = round(2) + (x / 2 - 1) * (9.2 + 1.86 * per), apart = (double)two * round(2) + round(x - 2 * (double)two);
    return flow + (apart > flow ? apart - flow : 0.0) * (per < 32 ? per / 32 : 1.0);
  }
  const double f = piped ? (nt == 2 ? 10.0 : 4.7 + 2.6 * (double)(tiles < 4 ? tiles : 4)) : 8.3;
  const double fx = nt == 2 ? 3.3 : 4.0, b = piped ? (nt == 2 ? 1.68 : 2.1) : 1.88, bx = piped ? 0.18 : 0.29;
  const double rest = x - (double)full;
  return (double)full * (f + fx + (b + bx) * per) + (rest > 0 ? f + fx * rest + (b + bx * rest) * per : 0.0);
}

// The kernel, head tiles per workgroup (at most two at d_v = 576: O's registers) and
// splits of the slots, at least four blocks each and within one round, that take
// the least time.
WideFwdPlan wide_fwd_plan(int64_t tgs, int64_t hpg, int64_t d_v, int64_t topk, bool may_split) {
  const int64_t ntiles = (hpg + 31) / 32, nblk = (topk + 31) / 32;
  WideFwdPlan best{1, 1, false};
  double us = wide_fwd_us(false, 1, 1, tgs, hpg, nblk);
  const auto offer = [&](bool piped, int nt, int64_t nsplit) {
    const double t = wide_fwd_us(piped, nt, nsplit, tgs, hpg, nblk);
    if (t < us) {
      us = t;
      best = WideFwdPlan{nt, (int)nsplit, piped};
    }
  };
  if (ntiles >= 2) offer(false, 2, 1);
  for (int nt = 1; nt <= 4; nt *= 2) {
    if (nt > 1 && (ntiles <= nt / 2 || (nt == 4 && d_v != 512))) break;
    if (nt > 1) offer(true, nt, 1);
    const int64_t wg = tgs * ((ntiles + nt - 1) / nt);
    for (int64_t ns = 2; may_split && ns <= nblk / 4 && ns * wg <= 256; ++ns) offer(true, nt, ns);
  }
  return best;
}

int launch_fwd_wide_bf16(const FwdParams &p, int64_t d_qk, int64_t d_v, int nt, bool qmx, hipStream_t st) {
  if (d_qk == 576 && d_v == 512) {
    if (nt == 4) return qmx ? launch_wide_bf16<576, 512, 4, 8, true>(p, st) : launch_wide_bf16<576, 512, 4, 8, false>(p, st);
    if (nt == 2) return qmx ? launch_wide_bf16<576, 512, 2, 8, true>(p, st) : launch_wide_bf16<576, 512, 2, 8, false>(p, st);
    if (!qmx) return launch_wide_bf16<576, 512, 1, 4, false>(p, st);
  }
  if (d_qk == 576 && d_v == 576 && !qmx)
    return nt == 2 ? launch_wide_bf16<576, 576, 2, 8, false>(p, st) : launch_wide_bf16<576, 576, 1, 4, false>(p, st);
  return set_error(DSA_ERR_UNSUPPORTED, "sparse_mla_fwd(wide): no bf16 kernel for d_qk=%lld d_v=%lld", (long long)d_qk,
                   (long long)d_v);
}

}  // namespace dsa
