// SparseMLA backward main pass for wide heads on gfx950 (d_qk = 576 with
// d_v = 512 or 576); semantics of cppmega/megatron/sparse_mla_ops/
// tilelang_sparse_mla_bwd.py:123-419.
//
// Two kernels per pass:
//   1. scores: S, dP, P, dS of every (token, kv group, head, slot) and
//      dQ = dS K.  P and dS leave as bf16 (the rounding at which the products
//      take them) in 2 KiB tiles [head][slot] per (32-slot block, 32-head tile);
//   2. rows: c[slot] = sum_h dS_h Q_h + P_h dO_h over all of the kv group's
//      heads (128 at a time) with Q and dO resident in registers as MFMA
//      operands, written as one fp16 row (scaled by a power of two) or fp32
//      row per (token, slot) at its CSR position.
// One kernel for both would hold Q and dO of at most 32 heads, so each (token,
// slot) would leave four partial rows at 128 heads: 29 GB written and read again
// at s = 4096, h = 128, top-k 2048 (18.0 ms for such a kernel, 5.4 ms for the
// reduction).  P and dS of all heads are 512 bytes per (token, slot), less than
// one partial row's 1152, and buy the sum over heads before the row is stored:
// scores 4.1 ms (2.6 TFLOP of the three products), rows 2.8 ms (11.5 GB of HBM
// traffic), reduction 1.1 ms.  Up to 32 heads there is one row either way; the two
// kernels are no slower there (s = 2048, one kernel and two: 32 heads, top-64 296
// and 279 us, top-512 1093 and 882, top-2048 3765 and 2959; e4m3, top-512 1159 and
// 1122; s = 300, top-64 75 and 75), as each holds fewer operands and the scores run
// in the two-barrier pipeline.
#include <type_traits>

#include "dsa_common.hpp"
#include "sparse_mla_gather.hpp"
#include "sparse_mla_params.hpp"
#include "sparse_mla_wide.hpp"
#include "sparse_mla_wide_tile.hpp"

namespace dsa {

__device__ __forceinline__ f32x4 mfma_16x16x32(i32x4 a, i32x4 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(a), as_bf16x8(b), c, 0, 0, 0);
}

// Delta * sm_scale and LSE of `heads` heads from row head0 (nheads real ones)
// into LD[2 h], LD[2 h + 1]: one wave per head, lane = 8-element chunk.
template <int D_V, int NW>
__device__ __forceinline__ void wide_bwd_stats(const BwdParams &p, float *LD, int64_t head0, int heads, int nheads,
                                               int w) {
  constexpr int VCH = D_V / 8;
  const int lane = lane_id();
  for (int h = w; h < heads; h += NW) {
    float part = 0.0f;
    if (h < nheads) {
      for (int c = lane; c < VCH; c += 64) {
        const i32x4 dv = ld_global_16(p.dO + (head0 + h) * D_V + 8 * c);
        const i32x4 ov = ld_global_16(p.o + (head0 + h) * D_V + 8 * c);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const uint32_t du = (uint32_t)dv[e], ou = (uint32_t)ov[e];
          part += bf16_bits_to_f32(ou & 0xffffu) * bf16_bits_to_f32(du & 0xffffu);
          part += bf16_bits_to_f32(ou >> 16) * bf16_bits_to_f32(du >> 16);
        }
      }
    }
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) part += __shfl_xor(part, off, 64);
    if (lane == 0) {
      float dl = part, lse_h = INFINITY;  // padded heads: P = exp2(x - inf) = 0
      if (h < nheads) {
        if (p.delta != nullptr) dl = p.delta[head0 + h];
        const float l = p.lse[head0 + h];
        lse_h = (l == -INFINITY) ? INFINITY : l;  // all-masked row: zero gradient
      }
      LD[2 * h] = dl * p.scale;
      LD[2 * h + 1] = lse_h;
    }
  }
}

// ---------------------------------------------------------------------------
// Scores and dQ, bf16
// ---------------------------------------------------------------------------
// One workgroup of 4 NT waves per (token, kv group, NT 32-head tiles).
//   S and dP (M = slot, N = head): wave = (matrix, half of the k-steps, head
//     tile), its operand of Q or dO resident in registers; K rows from the tile.
//     The two halves and the two matrices meet through LDS, and each wave then
//     forms P and dS of a quarter of one head tile (lane = head, 4 slots).
//   dQ^T[d][head] += K^T dS: wave w owns the 16-column tiles w, w + 4 NT, ... of
//     d for every head, K^T by transposed reads, dS from the LDS tile.
// Software pipeline, two barriers a block: block j's S / dP products run between
// the first and the second, and block j - 1's dQ products between the second and
// the next, where they cover the latency of the exchange and the softmax of
// block j.  Block j + 1's rows are fetched meanwhile (three row tiles rotate);
// the S waves, which the SIMDs serve first, issue those loads and the P / dS
// stores of block j - 1.
template <int D_QK, int D_V, int NT>
struct WideScores {
  static constexpr int NW = 4 * NT, NTHR = 64 * NW;
  using T = DmaTile<D_QK, 2 * NT>;                           // (filled by the 2 NT S waves)
  static constexpr int KSQ = D_QK / 32, KSV = D_V / 32;      // k-steps of 16 per wave (half of each)
  static constexpr int NDT = D_QK / 16;                      // 16-column tiles of d_qk
  static constexpr int DTW = (NDT + NW - 1) / NW;
  static constexpr int SP_W = 32 * 32;                       // floats per partial tile
  static constexpr int OFF_K = 0;
  static constexpr int OFF_SP = OFF_K + 3 * T::BYTES;
  static constexpr int OFF_PD = OFF_SP + 4 * NT * SP_W * 4;  // [head tile][P, dS][32 heads][32 slots]
  static constexpr int OFF_LD = OFF_PD + 2 * NT * kWidePdBytes;  // (two blocks)
  static constexpr int BYTES = OFF_LD + NT * 32 * 2 * 4;
  static_assert(BYTES <= 160 * 1024 && D_QK % 64 == 0 && D_V % 64 == 0, "wide backward LDS");
};

template <int D_QK, int D_V, int NT>
__global__ void __launch_bounds__(256 * NT) __attribute__((amdgpu_waves_per_eu(NT)))
sparse_mla_bwd_wide_scores_kernel(const BwdParams p) {
  using C = WideScores<D_QK, D_V, NT>;
  using T = typename C::T;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const int lane = lane_id(), w = wave_id(), t = threadIdx.x;
  const int g32 = lane >> 5, l32 = lane & 31, g16 = lane >> 4, l16 = lane & 15;
  const int ntg = (p.htiles + NT - 1) / NT;
  const int64_t item = xcd_remap(blockIdx.x, gridDim.x);
  const int tile0 = (int)(item % ntg) * NT;
  const int64_t tg = item / ntg;  // tok * G + g
  const int64_t g = tg % p.G, tok = tg / p.G, b = tok / p.S;
  unsigned char *K = smem + C::OFF_K;
  float *Sp = reinterpret_cast<float *>(smem + C::OFF_SP);
  unsigned char *PD = smem + C::OFF_PD;
  float *LD = reinterpret_cast<float *>(smem + C::OFF_LD);

  const int64_t head0 = tok * p.H + g * p.hpg + tile0 * 32;
  const int nheads = p.hpg - tile0 * 32 < 32 * NT ? p.hpg - tile0 * 32 : 32 * NT;
  const unsigned char *kv_b = p.kv + ((b * p.S_kv) * p.G + g) * T::ROWB;
  const uint32_t row_pitch = (uint32_t)(p.G * T::ROWB);
  const i32x4 kv_rs = make_buffer_words(kv_b, (uint32_t)(p.S_kv * p.G * T::ROWB - g * T::ROWB));
  const auto idx_rs = slot_rsrc(p.idx + tg * p.topk, p.topk);
  const uint32_t k_lds = lds_address(K);

  const int mat = w / (2 * NT), kh = (w / NT) & 1, ht = w % NT;  // (see below)
  // this wave's share of the rows of a block whose slot indices it holds
  auto fetch = [&](int tile, int idx) {
    dma_tile_issue<T>(k_lds + (uint32_t)(tile * T::BYTES), kv_rs, idx >= 0 ? (uint32_t)idx * row_pitch : kMaskedOff, w);
  };
  const int idx0 = slot_index(load_slot_raw(idx_rs, 0, l32), 0, l32, p.topk, p.S_kv);
  int idx_nxt = slot_index(load_slot_raw(idx_rs, 1, l32), 1, l32, p.topk, p.S_kv);
  const int nblk = valid_blocks(idx_rs, p.topk, p.S_kv);
  uint32_t vm = (uint32_t)__ballot(idx0 >= 0);
  if (mat == 0) fetch(0, idx0);

  // this wave's operand: Q (mat 0) or dO (mat 1) of head tile ht, k-steps 2 i + kh
  i32x4 op[C::KSQ];
  {
    const int h = 32 * ht + l32;
    const bool ok = h < nheads;
    const unsigned char *src = mat == 0 ? p.q + (head0 + h) * (D_QK * 2)
                                        : reinterpret_cast<const unsigned char *>(p.dO) + (head0 + h) * (D_V * 2);
#pragma unroll
    for (int i = 0; i < C::KSQ; ++i) {
      op[i] = i32x4{0, 0, 0, 0};
      if (ok && (i < C::KSV || mat == 0)) op[i] = ld_global_16(src + (16 * (2 * i + kh) + 8 * g32) * 2);
    }
  }
  wide_bwd_stats<D_V, C::NW>(p, LD, head0, 32 * NT, nheads, w);
  // block -1's dS is zero (its dQ products below read row tile 0)
  for (int u = t; u < NT * kWidePdBytes / 16; u += C::NTHR)
    *reinterpret_cast<i32x4 *>(PD + (NT * kWidePdBytes + u * 16)) = i32x4{0, 0, 0, 0};
  __syncthreads();
  // P / dS: this wave takes quarter eq of head tile eh (lane = head, slots 8 eq + 4 g32 ..)
  const int eh = w >> 2, eq = w & 3;
  const float delta_h = LD[2 * (32 * eh + l32)], lse_h = LD[2 * (32 * eh + l32) + 1];

  // S / dP operand of k-step 2 i + kh: row l32, chunk 2 (2 i + kh) + g32; i and i + 2 are a panel apart
  int ka[2];
#pragma unroll
  for (int u = 0; u < 2; ++u) ka[u] = tile_byte(l32, 2 * (2 * u + kh) + g32);
  // K^T of d tile w + NW i: rows 8 g16 + (lane % 16) / 4 (+ 4), columns 4 (lane % 4) .. of the tile
  int kt[2];
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const int row = 8 * g16 + 4 * u + (l16 >> 2), q = l16 & 3;
    kt[u] = tile_byte(row, 2 * (w & 3) + (q >> 1)) + (q & 1) * 8 + (w >> 2) * T::PANEL;
  }
  // dS[head][slot]: 64-byte rows, 16-byte chunk c of head h at c ^ ((h >> 2) & 3)
  const int ds_rd = 2048 + l16 * 64 + ((g16 ^ ((l16 >> 2) & 3)) * 16);
  const int pd_wr = eh * kWidePdBytes + l32 * 64 + ((eq ^ ((l32 >> 2) & 3)) * 16) + g32 * 8;
  // global copy of PD: thread t of the S waves takes chunks t and t + 128 NT
  const int cp_row = (t >> 2) & 31;
  const int cp_src = (t & ~3) * 16 + (((t & 3) ^ ((cp_row >> 2) & 3)) * 16);
  const int64_t nblk_all = (p.topk + 31) / 32;
  unsigned char *pd_g = p.pd + ((tg * nblk_all) * p.htiles + tile0) * (int64_t)kWidePdBytes + t * 16;
  const int64_t pd_step = (int64_t)p.htiles * kWidePdBytes;

  f32x4 dq[C::DTW][2 * NT];
#pragma unroll
  for (int i = 0; i < C::DTW; ++i)
#pragma unroll
    for (int h = 0; h < 2 * NT; ++h) dq[i][h] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

  // dQ products on row tile Kb and the dS of Pb
  auto dq_step = [&](const unsigned char *Kb, const unsigned char *Pb) {
    i32x4 bs[2 * NT];
#pragma unroll
    for (int h = 0; h < 2 * NT; ++h)
      bs[h] = *reinterpret_cast<const i32x4 *>(Pb + (h >> 1) * kWidePdBytes + (h & 1) * 1024 + ds_rd);
#pragma unroll
    for (int i = 0; i < C::DTW; ++i) {
      if (C::NDT % C::NW == 0 || i + 1 < C::DTW || w < C::NDT % C::NW) {
        const i32x2 r0 = ds_read_tr16(Kb + kt[0] + i * (C::NW / 4) * T::PANEL);
        const i32x2 r1 = ds_read_tr16(Kb + kt[1] + i * (C::NW / 4) * T::PANEL);
        const i32x4 a = {r0[0], r0[1], r1[0], r1[1]};
#pragma unroll
        for (int h = 0; h < 2 * NT; ++h) dq[i][h] = mfma_16x16x32(a, bs[h], dq[i][h]);
      }
    }
  };
  auto pd_store = [&](int blk) {
    const unsigned char *Pb = PD + (blk & 1) * NT * kWidePdBytes;
#pragma unroll
    for (int i = 0; i < 2; ++i) {  // (a wave's chunks are of one head tile)
      const int o = 128 * NT * i;
      if (tile0 + ((t + o) >> 8) < p.htiles)
        *reinterpret_cast<i32x4 *>(pd_g + blk * pd_step + o * 16) = *reinterpret_cast<const i32x4 *>(Pb + cp_src + o * 16);
    }
  };

  int kb = 0, kp = 0;  // row tiles of block j (j % 3) and of block j - 1 (any, for j = 0: its dS is zero)
  for (int j = 0; j < nblk; ++j) {
    const int kn = kb == 2 ? 0 : kb + 1;
    const unsigned char *Kj = K + kb * T::BYTES;
    __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): block j's rows, issued a block ago
    __syncthreads();  // block j's rows and block j - 1's P / dS are in LDS; block j - 2's rows are consumed
    const int raw = load_slot_raw(idx_rs, j + 2, l32);
    if (mat == 0) {
      if (j > 0) pd_store(j - 1);
      fetch(kn, idx_nxt);  // block j + 1 (zeros past the last)
    }
    f32x16 acc;
#pragma unroll
    for (int a = 0; a < 16; ++a) acc[a] = 0.0f;
#pragma unroll
    for (int i = 0; i < C::KSV; ++i) {
      const i32x4 a = *reinterpret_cast<const i32x4 *>(Kj + ka[i & 1] + (i >> 1) * T::PANEL);
      acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(as_bf16x8(a), as_bf16x8(op[i]), acc, 0, 0, 0);
    }
    if (C::KSQ > C::KSV && mat == 0) {
#pragma unroll
      for (int i = C::KSV; i < C::KSQ; ++i) {
        const i32x4 a = *reinterpret_cast<const i32x4 *>(Kj + ka[i & 1] + (i >> 1) * T::PANEL);
        acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(as_bf16x8(a), as_bf16x8(op[i]), acc, 0, 0, 0);
      }
    }
    put_partial(Sp + w * C::SP_W, acc);
    __syncthreads();  // partial tiles whole
    const float *sp = Sp + eh * C::SP_W + (eq * 64 + lane) * 4;
    const f32x4 s0 = *reinterpret_cast<const f32x4 *>(sp);
    const f32x4 s1 = *reinterpret_cast<const f32x4 *>(sp + NT * C::SP_W);
    const f32x4 d0 = *reinterpret_cast<const f32x4 *>(sp + 2 * NT * C::SP_W);
    const f32x4 d1 = *reinterpret_cast<const f32x4 *>(sp + 3 * NT * C::SP_W);
    dq_step(K + kp * T::BYTES, PD + ((j & 1) ^ 1) * NT * kWidePdBytes);
    const uint32_t lm = vm >> (8 * eq + 4 * g32);
    float pv[4], ds[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      pv[e] = ((lm >> e) & 1u) ? exp2_fast((s0[e] + s1[e]) * p.sl2 - lse_h) : 0.0f;
      ds[e] = pv[e] * fmaf(d0[e] + d1[e], p.scale, -delta_h);
    }
    unsigned char *Pw = PD + (j & 1) * NT * kWidePdBytes + pd_wr;
    *reinterpret_cast<i32x2 *>(Pw) = i32x2{(int)pack_bf16x2(pv[0], pv[1]), (int)pack_bf16x2(pv[2], pv[3])};
    *reinterpret_cast<i32x2 *>(Pw + 2048) = i32x2{(int)pack_bf16x2(ds[0], ds[1]), (int)pack_bf16x2(ds[2], ds[3])};
    vm = (uint32_t)__ballot(idx_nxt >= 0);
    idx_nxt = slot_index(raw, j + 2, l32, p.topk, p.S_kv);
    kp = kb;
    kb = kn;
  }
  __builtin_amdgcn_s_waitcnt(0x0F70);  // the loads past the last block have landed before the LDS is given up
  __syncthreads();
  if (nblk > 0) {
    dq_step(K + kp * T::BYTES, PD + ((nblk & 1) ^ 1) * NT * kWidePdBytes);
    if (mat == 0) pd_store(nblk - 1);
  }

  // dQ: lane = head 16 h + l16, d = 16 tile + 4 g16 ..
#pragma unroll
  for (int i = 0; i < C::DTW; ++i) {
    if (C::NDT % C::NW == 0 || i + 1 < C::DTW || w < C::NDT % C::NW) {
#pragma unroll
      for (int h = 0; h < 2 * NT; ++h) {
        if (16 * h + l16 < nheads) {
          uint16_t *drow = p.dq + (head0 + 16 * h + l16) * D_QK + (w + C::NW * i) * 16 + 4 * g16;
          *reinterpret_cast<i32x2 *>(drow) = i32x2{(int)pack_bf16x2(dq[i][h][0], dq[i][h][1]),
                                                   (int)pack_bf16x2(dq[i][h][2], dq[i][h][3])};
        }
      }
    }
  }
}

// ---------------------------------------------------------------------------
// Scores and dQ, e4m3
// ---------------------------------------------------------------------------
// One workgroup of four waves per (token, kv group, 32-head tile); S and dP
// (M = head, N = slot) split over their k dims, each wave one quarter, exchanged
// through LDS one after the other and summed by every wave in wave order (all
// waves hold bit-identical P / dS); QK^T on the codes, dP and dQ on rows
// dequantised to bf16.  Wave w owns the 32-column tiles t = w + 4 q of dQ^T.
// LDS: DOL [head][d] dO, LD = LSE (heads 0..31) and Delta * sm_scale (32..63),
// Kl [slot][d] gathered codes, Kd [slot][d] the rows dequantised, Ksc their
// scales, the waves' partial score tiles, one dS[slot][head] tile per wave and
// the P, dS [head][slot] tiles that leave.
template <int D_QK, int D_V>
struct WideBwdLds8 {
  using C = WideCfg<D_QK, D_V, true>;
  static constexpr int DOL_STRIDE = D_V * 2 + 32;
  static constexpr int DS_STRIDE = 32 * 2 + 32;
  static constexpr int KDB_STRIDE = D_QK * 2 + 32;  // whole rows dequantised
  static constexpr int OFF_DOL = 0;
  static constexpr int OFF_LD = OFF_DOL + 32 * DOL_STRIDE;
  static constexpr int OFF_KL = OFF_LD + 64 * 4;
  static constexpr int OFF_KD = OFF_KL + 32 * C::KL_STRIDE;
  static constexpr int OFF_SC = OFF_KD + 32 * KDB_STRIDE;
  static constexpr int OFF_SP = OFF_SC + 32 * 4;
  static constexpr int SP_W = 16 * 64;  // floats per partial tile
  static constexpr int OFF_DS = OFF_SP + 4 * SP_W * 4;
  static constexpr int OFF_PD = OFF_DS + 4 * 32 * DS_STRIDE;
  static constexpr int BYTES = OFF_PD + kWidePdBytes;
  static_assert(BYTES <= 160 * 1024, "wide backward LDS");
};

template <int D_QK, int D_V>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1)))
sparse_mla_bwd_wide_scores8_kernel(const BwdParams p) {
  using C = WideCfg<D_QK, D_V, true>;
  using L = WideBwdLds8<D_QK, D_V>;
  constexpr int DQT = D_QK / 32;          // 32-column tiles of d_qk
  constexpr int DQW = (DQT + 3) / 4;      // tiles per wave (tile t = w + 4 q)
  constexpr int VQ = D_V / 16 / 4;        // dP k-steps per wave
  static_assert((D_V / 16) % 4 == 0, "d_v k-steps split over four waves");
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];

  const int lane = lane_id(), w = __builtin_amdgcn_readfirstlane(wave_id());
  const int g32 = lane >> 5, l32 = lane & 31;
  const int64_t item = xcd_remap(blockIdx.x, gridDim.x);
  const int tile = (int)(item % p.htiles);
  const int64_t rest = item / p.htiles;
  const int64_t g = rest % p.G;
  const int64_t tok = rest / p.G;
  const int64_t b = tok / p.S;

  unsigned char *DOL = smem + L::OFF_DOL;
  float *LD = reinterpret_cast<float *>(smem + L::OFF_LD);
  unsigned char *Kl = smem + L::OFF_KL;
  unsigned char *Kd = smem + L::OFF_KD;
  float *Ksc = reinterpret_cast<float *>(smem + L::OFF_SC);
  float *Sp = reinterpret_cast<float *>(smem + L::OFF_SP);
  unsigned char *DS = smem + L::OFF_DS + w * 32 * L::DS_STRIDE;
  unsigned char *PD = smem + L::OFF_PD;

  const int64_t head0 = tok * p.H + g * p.hpg + tile * 32;
  const int nheads = p.hpg - tile * 32 < 32 ? p.hpg - tile * 32 : 32;
  const int64_t entry0 = (tok * p.G + g) * p.topk;
  const int32_t *idx_row = p.idx + entry0;
  const unsigned char *kv_b = p.kv + ((b * p.S_kv) * p.G + g) * C::ROWB;
  const float *kv_scale_b = p.kv_scale + b * p.S_kv;
  const uint32_t row_pitch = (uint32_t)(p.G * C::ROWB);

  // Indices (two blocks ahead) and rows (one block ahead) are loaded
  // unconditionally through resources that end at the item's top-k, so each wave
  // issues the same loads on every block and the compiler's waits count exactly.
  const auto idx_rs = slot_rsrc(idx_row, p.topk);
  int idx_cur = slot_index(load_slot_raw(idx_rs, 0, l32), 0, l32, p.topk, p.S_kv);
  int raw_nxt = load_slot_raw(idx_rs, 1, l32);
  typename C::Regs rg;
  wide_issue<C, true, false, true>(rg, kv_b, kv_scale_b, idx_cur, row_pitch);
  // blocks up to the last valid slot: the same count in every wave (the loop has workgroup barriers)
  const int nblk = valid_blocks(idx_rs, p.topk, p.S_kv);
  const float qsc = p.q_scale[tok];
  // ---------------- prologue: dO tile, LSE, Delta ----------------
  {
    const int t = threadIdx.x;
    // dO rows and Delta = sum_d O dO: one wave per head, lane = 8-element chunk
    constexpr int VCH = D_V / 8;
    for (int h = w; h < 32; h += 4) {
      float part = 0.0f;
      for (int c = lane; c < VCH; c += 64) {
        i32x4 dv = {0, 0, 0, 0}, ov = {0, 0, 0, 0};
        if (h < nheads) {
          dv = ld_global_16(p.dO + (head0 + h) * D_V + 8 * c);
          ov = ld_global_16(p.o + (head0 + h) * D_V + 8 * c);
        }
        *reinterpret_cast<i32x4 *>(DOL + h * L::DOL_STRIDE + c * 16) = dv;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const uint32_t du = (uint32_t)dv[e], ou = (uint32_t)ov[e];
          part += bf16_bits_to_f32(ou & 0xffffu) * bf16_bits_to_f32(du & 0xffffu);
          part += bf16_bits_to_f32(ou >> 16) * bf16_bits_to_f32(du >> 16);
        }
      }
#pragma unroll
      for (int off = 1; off < 64; off <<= 1) part += __shfl_xor(part, off, 64);
      if (lane == 0) {
        float dl = part;
        if (p.delta != nullptr && h < nheads) dl = p.delta[head0 + h];
        LD[32 + h] = dl * p.scale;
      }
    }
    if (t < 32) {
      float lse_h = INFINITY;  // padded heads: P = exp2(x - inf) = 0
      if (t < nheads) {
        const float l = p.lse[head0 + t];
        lse_h = (l == -INFINITY) ? INFINITY : l;  // all-masked row: zero gradient
      }
      LD[t] = lse_h;
    }
  }

  // e4m3: this wave's quarter of the raw Q codes, the A operand of QK^T (head l32)
  long qA8[C::KQ];
#pragma unroll
  for (int k = 0; k < C::KQ; ++k)
    qA8[k] = l32 < nheads ? *reinterpret_cast<const long *>(p.q + (head0 + l32) * D_QK + 16 * (w * C::KQ + k) + 8 * g32)
                          : 0l;
  f32x16 dqacc[DQW];
#pragma unroll
  for (int q = 0; q < DQW; ++q)
#pragma unroll
    for (int a = 0; a < 16; ++a) dqacc[q][a] = 0.0f;

  const int k0 = w * C::KQ, v0 = w * VQ;
  unsigned char *pd_g = p.pd + (((tok * p.G + g) * ((p.topk + 31) / 32)) * p.htiles + tile) * (int64_t)kWidePdBytes;
  // the first block's rows have landed: nothing is in flight on entry, so the
  // loop's waits follow its own order (s_waitcnt vmcnt(0) with expcnt and
  // lgkmcnt left open, gfx9 encoding)
  __builtin_amdgcn_s_waitcnt(0x0F70);
  for (int blk = 0; blk < nblk; ++blk) {
    wide_store<C, true, C::NCH, L::KDB_STRIDE>(rg, Kl, Kd, Ksc);
    const bool valid = idx_cur >= 0;  // slot 32 blk + l32
    __syncthreads();  // rows (and, on the first block, the prologue tiles) are in LDS
    const int raw_nn = load_slot_raw(idx_rs, blk + 2, l32);
    const int idx_nxt = slot_index(raw_nxt, blk + 1, l32, p.topk, p.S_kv);
    wide_issue<C, true, false, true>(rg, kv_b, kv_scale_b, idx_nxt, row_pitch);  // past the last block too

    // ---- partial S = Q K^T and dP = dO V^T (M = head, N = slot) over this wave's k-steps ----
    f32x16 sacc, dpacc;
#pragma unroll
    for (int a = 0; a < 16; ++a) {
      sacc[a] = 0.0f;
      dpacc[a] = 0.0f;
    }
#pragma unroll
    for (int k = 0; k < C::KQ; ++k) {
      const int d0 = 16 * (k0 + k) + 8 * g32;
      const long kb = *reinterpret_cast<const long *>(Kl + l32 * C::KL_STRIDE + d0);
      sacc = __builtin_amdgcn_mfma_f32_32x32x16_fp8_fp8(qA8[k], kb, sacc, 0, 0, 0);
    }
#pragma unroll
    for (int k = 0; k < VQ; ++k) {
      const int d0 = 16 * (v0 + k) + 8 * g32;
      const i32x4 da = *reinterpret_cast<const i32x4 *>(DOL + l32 * L::DOL_STRIDE + d0 * 2);
      const i32x4 vb = *reinterpret_cast<const i32x4 *>(Kd + l32 * L::KDB_STRIDE + d0 * 2);
      dpacc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(as_bf16x8(da), as_bf16x8(vb), dpacc, 0, 0, 0);
    }
    float s[16], dp[16];
    put_partial(Sp + w * L::SP_W, sacc);
    __syncthreads();  // S partial tiles written
    sum_partials(Sp, L::SP_W, s);
    __syncthreads();  // read before the dP partials reuse the tiles
    put_partial(Sp + w * L::SP_W, dpacc);
    __syncthreads();
    sum_partials(Sp, L::SP_W, dp);

    // ---- P, dS (lane = slot 32 blk + l32, heads 8i + 4*g32 + j; identical in every wave) ----
    const float xs = p.sl2 * qsc * Ksc[l32];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const f32x4 l4 = *reinterpret_cast<const f32x4 *>(LD + 8 * i + 4 * g32);
      const f32x4 d4 = *reinterpret_cast<const f32x4 *>(LD + 32 + 8 * i + 4 * g32);
      float P[4], dS[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        P[j] = valid ? exp2_fast(s[4 * i + j] * xs - l4[j]) : 0.0f;
        dS[j] = P[j] * fmaf(dp[4 * i + j], p.scale, -d4[j]);
      }
      const uint32_t ds0 = pack_bf16x2(dS[0], dS[1]), ds1 = pack_bf16x2(dS[2], dS[3]);
      *reinterpret_cast<i32x2 *>(DS + l32 * L::DS_STRIDE + (8 * i + 4 * g32) * 2) = i32x2{(int)ds0, (int)ds1};
      // the P (wave 0) and dS (wave 1) tiles that leave: [head][slot]
      if (w < 2) {
        const uint32_t v0 = w == 0 ? pack_bf16x2(P[0], P[1]) : ds0, v1 = w == 0 ? pack_bf16x2(P[2], P[3]) : ds1;
        uint16_t *o = reinterpret_cast<uint16_t *>(PD + w * 2048 + (8 * i + 4 * g32) * 64) + l32;
        o[0] = (uint16_t)v0;
        o[32] = (uint16_t)(v0 >> 16);
        o[64] = (uint16_t)v1;
        o[96] = (uint16_t)(v1 >> 16);
      }
    }
    wave_lds_sync();  // this wave's dS tile (and its tile that leaves)
    if (w < 2) {
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int o = w * 2048 + (64 * i + lane) * 16;
        *reinterpret_cast<i32x4 *>(pd_g + (int64_t)blk * p.htiles * kWidePdBytes + o) = *reinterpret_cast<const i32x4 *>(PD + o);
      }
    }

    // ---- dQ^T[d][head] += K^T[d][slot] dS^T[slot][head] on tiles t = w + 4q ----
#pragma unroll
    for (int kc = 0; kc < 2; ++kc) {
      const i32x4 bv = tr_operand(DS, L::DS_STRIDE, 0, 16 * kc, 4, 8);
#pragma unroll
      for (int q = 0; q < DQW; ++q) {
        const int t = w + 4 * q;
        if (t < DQT) {
          const i32x4 av = tr_operand(Kd, L::KDB_STRIDE, t * 32, 16 * kc, 4, 8);
          dqacc[q] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(as_bf16x8(av), as_bf16x8(bv), dqacc[q], 0, 0, 0);
        }
      }
    }

    __syncthreads();  // rows, partial tiles and dS tiles consumed before the next block
    idx_cur = idx_nxt;
    raw_nxt = raw_nn;
  }

  // ---- dQ: lane = head l32, d = t*32 + 8i + 4*g32 + j ----
  if (l32 < nheads) {
    uint16_t *drow = p.dq + (head0 + l32) * D_QK;
#pragma unroll
    for (int q = 0; q < DQW; ++q) {
      const int t = w + 4 * q;
      if (t < DQT) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const i32x2 pk = {(int)pack_bf16x2(dqacc[q][4 * i], dqacc[q][4 * i + 1]),
                            (int)pack_bf16x2(dqacc[q][4 * i + 2], dqacc[q][4 * i + 3])};
          *reinterpret_cast<i32x2 *>(drow + t * 32 + 8 * i + 4 * g32) = pk;
        }
      }
    }
  }
}


// ---------------------------------------------------------------------------
// Partial dKV rows
// ---------------------------------------------------------------------------
// One workgroup of 8 waves per (token, kv group, 128-head group).
// c^T[d][slot] = Q^T dS + dO^T P with M = d, N = slot, K = head: wave w owns the
// 16-column tiles w, w + 8, ... of d (five for waves 0..3 and four for 4..7: an
// even share per SIMD), their Q^T / dO^T operands for all 128 heads in registers, so a
// block reads its 16 KiB of P / dS and writes its 32 rows: it is bound by HBM
// (1.1 KiB written per 0.5 KiB read).  The block's tiles are loaded one block
// ahead, read from LDS by every wave with transposed reads, and the rows are
// staged in LDS so that they leave as whole rows.
template <int D_QK, int D_V, bool F32P>
struct WideRows {
  static constexpr int NW = 8, NTHR = 64 * NW;
  static constexpr int NDT = D_QK / 16, DTW = (NDT + NW - 1) / NW;  // d tiles, and at most per wave
  static constexpr int NDV = D_V / 16, DVW = (NDV + NW - 1) / NW;
  static constexpr int ROWB = D_QK * (F32P ? 4 : 2);
  static constexpr int CS_STRIDE = ROWB + 16;  // an odd number of 16-byte chunks: rows on distinct banks
  static constexpr int RCH = ROWB / 16;
  static constexpr int PD_BYTES = kWideRowTiles * kWidePdBytes;
  static constexpr int OFF_PD = 0;                       // two blocks
  static constexpr int OFF_CS = OFF_PD + 2 * PD_BYTES;
  static constexpr int OFF_MX = OFF_CS + 32 * CS_STRIDE;  // [slot][8, padded to 12] the waves' row maxima
  static constexpr int OFF_POS = OFF_MX + 32 * 12 * 4;
  static constexpr int LOOP_BYTES = OFF_POS + 32 * 4;
  static constexpr int QL_BYTES = 128 * D_QK * 2;         // prologue: Q (then dO) of the group, row-major
  static constexpr int BYTES = LOOP_BYTES > QL_BYTES ? LOOP_BYTES : QL_BYTES;
  static constexpr int RIT = (32 * RCH + NTHR - 1) / NTHR;  // 16-byte row pieces per thread
  static_assert(BYTES <= 160 * 1024, "wide backward LDS");
};

// 128 rows of D elements (bf16, or e4m3 codes times qsc as bf16) from a resource
// that ends at the group's last head (zeros past it), into LDS row-major with
// the chunks swizzled by row_swz.
template <int D, int NTHR, bool FP8>
__device__ __forceinline__ void wide_rows_stage(unsigned char *QL, __amdgpu_buffer_rsrc_t rs, float qsc) {
  constexpr int NCH = D / 8, N = 128 * NCH, IT = (N + NTHR - 1) / NTHR;
  const int t = threadIdx.x;
  i32x4 v[IT];
#pragma unroll
  for (int i = 0; i < IT; ++i) {
    const int u = t + NTHR * i;
    if constexpr (FP8) {
      const auto r = __builtin_amdgcn_raw_buffer_load_b64(rs, u * 8, 0, 0);
      v[i] = __builtin_bit_cast(i32x4, e4m3x8_to_bf16_scaled((uint32_t)r[0], (uint32_t)r[1], qsc));
    } else {
      v[i] = __builtin_bit_cast(i32x4, __builtin_amdgcn_raw_buffer_load_b128(rs, u * 16, 0, 0));
    }
  }
#pragma unroll
  for (int i = 0; i < IT; ++i) {
    const int u = t + NTHR * i, row = u / NCH, c = u - row * NCH;
    if (N % NTHR == 0 || i + 1 < IT || u < N)
      *reinterpret_cast<i32x4 *>(QL + row * (D * 2) + ((c ^ row_swz(row)) * 16)) = v[i];
  }
}

// A operand [16 d of tile dt][32 heads of tile kk] from the staged rows.
template <int D>
__device__ __forceinline__ i32x4 wide_rows_operand(const unsigned char *QL, int dt, int kk) {
  const int lane = lane_id(), g16 = lane >> 4, l16 = lane & 15, q = l16 & 3;
  i32x2 r[2];
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const int row = 32 * kk + 8 * g16 + 4 * u + (l16 >> 2);
    r[u] = ds_read_tr16(QL + row * (D * 2) + (((2 * dt + (q >> 1)) ^ row_swz(row)) * 16) + (q & 1) * 8);
  }
  return i32x4{r[0][0], r[0][1], r[1][0], r[1][1]};
}

template <int D_QK, int D_V, bool FP8, bool F32P>
__global__ void __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2)))
sparse_mla_bwd_wide_rows_kernel(const BwdParams p) {
  using C = WideRows<D_QK, D_V, F32P>;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const int lane = lane_id(), w = wave_id(), t = threadIdx.x;
  const int l32 = lane & 31, g16 = lane >> 4, l16 = lane & 15;
  const int64_t item = xcd_remap(blockIdx.x, gridDim.x);
  const int grp = (int)(item % p.ntiles);
  const int64_t tg = item / p.ntiles;
  const int64_t g = tg % p.G, tok = tg / p.G;
  const int tile0 = grp * kWideRowTiles;
  const int nt = p.htiles - tile0 < kWideRowTiles ? p.htiles - tile0 : kWideRowTiles;  // head tiles of this group
  const int64_t head0 = tok * p.H + g * p.hpg + tile0 * 32;
  const int nheads = p.hpg - tile0 * 32 < 128 ? p.hpg - tile0 * 32 : 128;
  const int64_t n_entries = p.B * p.S * p.G * p.topk;
  const uint32_t trash = (uint32_t)n_entries * (uint32_t)p.ntiles + (uint32_t)(item % kTrashRows);
  const auto idx_rs = slot_rsrc(p.idx + tg * p.topk, p.topk);
  const auto pos_rs = slot_rsrc(p.pos_of + tg * p.topk, p.topk);
  const int nblk = valid_blocks(idx_rs, p.topk, p.S_kv);
  if (nblk == 0) return;  // workgroup-uniform: no valid slot, no row

  // the pass's partial rows, below 4 GiB (the host caps a pass below it)
  const auto row_rs = make_buffer_rsrc(p.partials, ((uint32_t)n_entries * (uint32_t)p.ntiles + kTrashRows) * (uint32_t)C::ROWB);
  typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
  unsigned char *Cs = smem + C::OFF_CS;
  float *MX = reinterpret_cast<float *>(smem + C::OFF_MX);
  uint32_t *Pos = reinterpret_cast<uint32_t *>(smem + C::OFF_POS);

  // P / dS of one block: nt * 4 KiB, thread t takes 16-byte chunks t and t + 512
  const int64_t nblk_all = (p.topk + 31) / 32;
  const uint32_t pd_step = (uint32_t)(p.htiles * kWidePdBytes);
  const auto pd_rs = make_buffer_rsrc(p.pd + ((tg * nblk_all) * p.htiles + tile0) * (int64_t)kWidePdBytes,
                                      (uint32_t)(nblk_all * p.htiles - tile0) * (uint32_t)kWidePdBytes);
  const uint32_t c0 = t < nt * 256 ? (uint32_t)t * 16u : kMaskedOff;
  const uint32_t c1 = t + 512 < nt * 256 ? (uint32_t)(t + 512) * 16u : kMaskedOff;
  i32x4 pv0, pv1;
  auto pd_load = [&](int blk) {
    pv0 = __builtin_bit_cast(i32x4, __builtin_amdgcn_raw_buffer_load_b128(pd_rs, (int)c0, (int)(blk * pd_step), 0));
    pv1 = __builtin_bit_cast(i32x4, __builtin_amdgcn_raw_buffer_load_b128(pd_rs, (int)c1, (int)(blk * pd_step), 0));
  };
  // LDS: chunk c of row r (64-byte rows) at c ^ 2 ((r >> 3) & 1), so that a transposed
  // read's rows 8 g .. 8 g + 3 of two neighbouring g are on distinct banks
  auto pd_put = [&](unsigned char *P) {
    const int r = t >> 2, c = t & 3;  // (512 / 4 = 128 rows on: the same swizzle bit)
    const int d = r * 64 + ((c ^ (((r >> 3) & 1) << 1)) * 16);
    *reinterpret_cast<i32x4 *>(P + d) = pv0;
    *reinterpret_cast<i32x4 *>(P + d + 512 * 16) = pv1;
  };

  // ---- prologue: Q^T and dO^T operands of this wave's d tiles ----
  i32x4 qA[C::DTW][kWideRowTiles], dA[C::DVW][kWideRowTiles];
  {
    float qsc = 1.0f;
    if constexpr (FP8) qsc = p.q_scale[tok];
    wide_rows_stage<D_QK, C::NTHR, FP8>(
        smem, make_buffer_rsrc(p.q + head0 * D_QK * (FP8 ? 1 : 2), (uint32_t)(nheads * D_QK * (FP8 ? 1 : 2))), qsc);
    __syncthreads();
#pragma unroll
    for (int i = 0; i < C::DTW; ++i)
#pragma unroll
      for (int kk = 0; kk < kWideRowTiles; ++kk)
        qA[i][kk] = wide_rows_operand<D_QK>(smem, (w + C::NW * i) % C::NDT, kk);  // (a tile past the last is not used)
    __syncthreads();
    wide_rows_stage<D_V, C::NTHR, false>(smem, make_buffer_rsrc(p.dO + head0 * D_V, (uint32_t)(nheads * D_V * 2)), 1.0f);
    pd_load(0);
    __syncthreads();
#pragma unroll
    for (int i = 0; i < C::DVW; ++i)
#pragma unroll
      for (int kk = 0; kk < kWideRowTiles; ++kk) dA[i][kk] = wide_rows_operand<D_V>(smem, (w + C::NW * i) % C::NDV, kk);
    __syncthreads();
  }

  // B operands: rows (heads) 8 g16 + (lane % 16) / 4 (+ 4), columns (slots) 16 st + 4 (lane % 4) ..
  int bo[2];
#pragma unroll
  for (int st = 0; st < 2; ++st)
    bo[st] = (8 * g16 + (l16 >> 2)) * 64 + (((2 * st + ((l16 & 3) >> 1)) ^ ((g16 & 1) << 1)) * 16) + (l16 & 1) * 8;
  int raw = load_slot_raw(idx_rs, 0, l32), pos = load_slot_raw(pos_rs, 0, l32);

  for (int blk = 0; blk < nblk; ++blk) {
    unsigned char *P = smem + C::OFF_PD + (blk & 1) * C::PD_BYTES;
    pd_put(P);
    const bool wr = slot_index(raw, blk, l32, p.topk, p.S_kv) >= 0 && pos >= 0 && pos < n_entries;
    const uint32_t prow = wr ? (uint32_t)pos * (uint32_t)p.ntiles + (uint32_t)grp : trash;
    __syncthreads();  // this block's P / dS
    pd_load(blk + 1 < nblk ? blk + 1 : blk);
    raw = load_slot_raw(idx_rs, blk + 1, l32);
    pos = load_slot_raw(pos_rs, blk + 1, l32);

    f32x4 acc[C::DTW][2];
#pragma unroll
    for (int i = 0; i < C::DTW; ++i)
#pragma unroll
      for (int st = 0; st < 2; ++st) acc[i][st] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int kk = 0; kk < kWideRowTiles; ++kk) {
      if (kk < nt) {  // uniform
#pragma unroll
        for (int m = 0; m < 2; ++m) {  // P dO, then dS Q
          i32x4 bv[2];
#pragma unroll
          for (int st = 0; st < 2; ++st) {
            const unsigned char *s = P + kk * kWidePdBytes + m * 2048 + bo[st];
            const i32x2 r0 = ds_read_tr16(s), r1 = ds_read_tr16(s + 4 * 64);
            bv[st] = i32x4{r0[0], r0[1], r1[0], r1[1]};
          }
#pragma unroll
          for (int i = 0; i < (m == 0 ? C::DVW : C::DTW); ++i) {
            constexpr int kTiles[2] = {C::NDV, C::NDT};
            if (C::NW * (i + 1) <= kTiles[m] || w + C::NW * i < kTiles[m]) {
#pragma unroll
              for (int st = 0; st < 2; ++st) acc[i][st] = mfma_16x16x32(m == 0 ? dA[i][kk] : qA[i][kk], bv[st], acc[i][st]);
            }
          }
        }
      }
    }

    // acc[i][st][r]: d = 16 (w + 8 i) + 4 g16 + r of slot 16 st + l16 (zeros in a tile past the last)
    float scale[2] = {1.0f, 1.0f};
    if constexpr (!F32P) {
      // fp16 rows: a power of two maps the row's largest magnitude into [2^13, 2^14)
#pragma unroll
      for (int st = 0; st < 2; ++st) {
        float m = 0.0f;
#pragma unroll
        for (int i = 0; i < C::DTW; ++i)
#pragma unroll
          for (int r = 0; r < 4; ++r) m = fmaxf(m, fabsf(acc[i][st][r]));
        m = fmaxf(m, __shfl_xor(m, 16, 64));
        m = max_halves(m);
        if (g16 == 0) MX[(16 * st + l16) * 12 + w] = m;
      }
      if (w == 0 && lane < 32) Pos[lane] = prow;
      __syncthreads();  // the waves' maxima
#pragma unroll
      for (int st = 0; st < 2; ++st) {
        const f32x4 *mr = reinterpret_cast<const f32x4 *>(MX + (16 * st + l16) * 12);
        const f32x4 m0 = mr[0], m1 = mr[1];
        float m = 0.0f;
#pragma unroll
        for (int r = 0; r < 4; ++r) m = fmaxf(m, fmaxf(m0[r], m1[r]));
        const int e = partial_row_exponent(m);
        scale[st] = exp2i(e);
        if (w == 0 && g16 == 0) p.partial_exp[Pos[16 * st + l16]] = (int8_t)e;
      }
    } else {
      if (w == 0 && lane < 32) Pos[lane] = prow;
    }
#pragma unroll
    for (int i = 0; i < C::DTW; ++i) {
      if (C::NW * (i + 1) > C::NDT && w + C::NW * i >= C::NDT) break;
#pragma unroll
      for (int st = 0; st < 2; ++st) {
        const f32x4 a = acc[i][st];
        unsigned char *dst = Cs + (16 * st + l16) * C::CS_STRIDE + ((w + C::NW * i) * 16 + 4 * g16) * (F32P ? 4 : 2);
        if constexpr (F32P) {
          *reinterpret_cast<f32x4 *>(dst) = a;
        } else {
          *reinterpret_cast<i32x2 *>(dst) = i32x2{(int)pack_f16x2(a[0] * scale[st], a[1] * scale[st]),
                                                  (int)pack_f16x2(a[2] * scale[st], a[3] * scale[st])};
        }
      }
    }
    __syncthreads();  // the block's rows are staged
#pragma unroll
    for (int i = 0; i < C::RIT; ++i) {
      const int u = t + C::NTHR * i, row = u / C::RCH, c = u - row * C::RCH;
      if ((32 * C::RCH) % C::NTHR == 0 || i + 1 < C::RIT || u < 32 * C::RCH) {
        const i32x4 v = *reinterpret_cast<const i32x4 *>(Cs + row * C::CS_STRIDE + c * 16);
        const uint32_t o = Pos[row] * (uint32_t)C::ROWB + (uint32_t)c * 16u;
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, v), row_rs, (int)o, 0, 2);  // streaming
      }
    }
    // (F32P: the next block's Cs writes follow its first barrier; Pos likewise)
  }
}

// ---------------------------------------------------------------------------
// Launch
// ---------------------------------------------------------------------------
template <class K>
static int launch_wide_kernel(K kernel, int64_t nitems, int threads, size_t lds, const BwdParams &p, hipStream_t st,
                              const char *what) {
  const hipError_t e = hipFuncSetAttribute((const void *)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  if (e != hipSuccess) return set_error(DSA_ERR_HIP, "%s: LDS attribute: %s", what, hipGetErrorString(e));
  if (nitems >= (1ll << 31)) return set_error(DSA_ERR_INVALID_ARG, "%s: grid too large", what);
  hipLaunchKernelGGL(kernel, dim3((unsigned)nitems), dim3(threads), lds, st, p);
  return check_launch(what);
}

template <int D_QK, int D_V, int NT>
static int launch_scores(const BwdParams &p, int64_t tgs, hipStream_t st) {
  using C = WideScores<D_QK, D_V, NT>;
  return launch_wide_kernel(sparse_mla_bwd_wide_scores_kernel<D_QK, D_V, NT>, tgs * ((p.htiles + NT - 1) / NT), C::NTHR,
                            C::BYTES, p, st, "sparse_mla_bwd(wide scores)");
}

template <int D_QK, int D_V>
static int launch_bwd_wide_t(const BwdParams &p, bool fp8, bool f32p, hipStream_t st) {
  const int64_t tgs = p.B * p.S * p.G;
  int rc;
  if (fp8)
    rc = launch_wide_kernel(sparse_mla_bwd_wide_scores8_kernel<D_QK, D_V>, tgs * p.htiles, 256,
                            WideBwdLds8<D_QK, D_V>::BYTES, p, st, "sparse_mla_bwd(wide scores)");
  else  // two head tiles per workgroup share a block's gather; one where a kv group has no more
    rc = p.htiles >= 2 ? launch_scores<D_QK, D_V, 2>(p, tgs, st) : launch_scores<D_QK, D_V, 1>(p, tgs, st);
  if (rc) return rc;
  const char *what = "sparse_mla_bwd(wide rows)";
  const int64_t n = tgs * p.ntiles;
  const int lds = f32p ? WideRows<D_QK, D_V, true>::BYTES : WideRows<D_QK, D_V, false>::BYTES;
  if (fp8)
    return f32p ? launch_wide_kernel(sparse_mla_bwd_wide_rows_kernel<D_QK, D_V, true, true>, n, 512, lds, p, st, what)
                : launch_wide_kernel(sparse_mla_bwd_wide_rows_kernel<D_QK, D_V, true, false>, n, 512, lds, p, st, what);
  return f32p ? launch_wide_kernel(sparse_mla_bwd_wide_rows_kernel<D_QK, D_V, false, true>, n, 512, lds, p, st, what)
              : launch_wide_kernel(sparse_mla_bwd_wide_rows_kernel<D_QK, D_V, false, false>, n, 512, lds, p, st, what);
}

int launch_bwd_main_wide(const BwdParams &p, int64_t d_qk, int64_t d_v, bool fp8, bool f32p, hipStream_t st) {
  if (d_qk == 576 && d_v == 512) return launch_bwd_wide_t<576, 512>(p, fp8, f32p, st);
  if (d_qk == 576 && d_v == 576) return launch_bwd_wide_t<576, 576>(p, fp8, f32p, st);
  return set_error(DSA_ERR_UNSUPPORTED, "sparse_mla_bwd(wide): no kernel for d_qk=%lld d_v=%lld", (long long)d_qk,
                   (long long)d_v);
}

}  // namespace dsa
