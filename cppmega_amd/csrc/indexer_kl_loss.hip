// DSA indexer KL loss on gfx950: the KL divergence between the head-averaged
// causal attention distribution and the indexer's softmax, without ever
// materialising the [b, np, sq, sk] attention probabilities.
//
// Reference: compute_dsa_indexer_loss_splitk
// (cppmega/megatron/dsa_splitk_indexer_loss.py:328-468), a two-stage Triton
// kernel (stage 1 :57-186 accumulates per-head softmax statistics, stage 2
// :194-322 recomputes q.k, averages the normalised probabilities over heads
// and reduces the KL per position), checked by its test against a clone of
// Megatron's compute_dsa_indexer_loss (tests/test_dsa_splitk_indexer_loss.py:29-83):
//
//   a_h[t, s] = scale * query[t, h] . key[s, h]  (+ sparse top-k mask) (s <= t)
//   P[t, s]   = mean_h softmax_s a_h[t, :]
//   Q[t, s]   = softmax_s (index_scores[t, :] + sparse top-k mask) over all s
//   loss      = coeff * mean_t sum_s P (ln(P + 1e-10) - ln(Q + 1e-10))
//
// Stream-ordered kernels, all deterministic (no atomics outside LDS).  The loss alone
// (dsa_indexer_kl_loss) is 1 to 5; the other entry points are listed below it.
//  1. kl_index_stats_kernel  one wave per (b, t): the log2 normaliser
//     gamma = max + log2(sum exp2(x - max)) of x = index_scores * log2(e) over
//     the row (sparse: over the row's top-k set, built as a bitmask in LDS and
//     written out for the other kernels; with a sparse state also the set's ranks
//     and scores in column order);
//  1a. kl_mask_tiles_kernel  sparse, large calls: the bitmask as lane masks for 2;
//  2. kl_attn_stats_kernel   per (b, head, pair of 256-token blocks): the log2
//     normaliser beta_h[t] of c * q.k (c = scale * log2(e)) over s <= t, on
//     MFMA 32x32x16 bf16 with S^T = K . Q^T (keys on M, tokens on N, so a lane
//     holds 16 keys of one token and row reductions stay in-lane); key chunks
//     are double-buffered in LDS and shared by the 8 waves; a long and a short
//     token block share one workgroup so every workgroup does equal work;
//  3. kl_pass_kernel         per (b, 256- or 128-token block, key chunk): for every head
//     recompute c * q.k, accumulate exp2(c * q.k - beta_h) in registers (the
//     head sum of P), then form the KL terms of the chunk against
//     Q = exp2(index * log2(e) - gamma) and write one partial sum per token;
//  4. kl_rows_kernel         row loss = sum of its chunk partials in chunk order
//     (NaN when the row has no admissible attention column or a NaN index
//     normaliser, as the reference's softmax gives);
//  5. kl_mean_kernel         one workgroup: coeff * mean of the row losses in a
//     fixed summation order.
//
// Gradient with respect to index_scores (dsa_indexer_kl_loss_backward; the
// loss's only path back to the indexer, which Megatron obtains by autograd
// through compute_dsa_indexer_loss).  With Q = softmax(z) over the row's
// columns and P the detached target,
//   dL/dz_s = g * coeff / (B * Sq) * (Q_s * R - P_s * Q_s / (Q_s + 1e-10)),
//   R       = sum_j P_j * Q_j / (Q_j + 1e-10)
// (0 where Q_s = 0: -inf scores and, sparse, columns outside the top-k set;
// NaN over a row whose loss is NaN).  Kernels 1-3 run as above, except that
// the pass kernel writes P into the gradient buffer (s <= t) and one partial
// R per key chunk instead of the KL terms; then
//  6. kl_grad_kernel         one workgroup per row: R in chunk order, then the
//     whole row of the gradient in place over P (16-byte loads and stores).
//
// Loss and gradient together (dsa_indexer_kl_loss_with_grad, what autograd
// takes; dsa_indexer_kl_loss_grad_state leaves the loss out): the gradient is
// linear in g, so one run of the two q.k kernels leaves the loss and a state from
// which dsa_indexer_kl_loss_grad_apply forms the gradient for any g (a backward that
// recomputed would run them again: 565 us at b = 2, s = 4096, 32 heads of 128).
// The state holds
//   v_s = Q_s * R - P_s * Q_s / (Q_s + 1e-10):
// dense, every column (the size of the scores, which then need not be kept):
// kernels 1 to 6, then
//  7. kl_scale_kernel        the gradient, g * coeff / (B * Sq) * v;
// sparse, the columns of the row's top-k set only, in column order (v is 0
// elsewhere), with the set's bitmask: 12 MB instead of 128 MiB at top-256.  Kernels
// 1 to 3, where 3 leaves the set's P at its ranks, then
//  4s. kl_rows_state_kernel  one wave per row: the row's loss and R over the set, v;
//  5, and
//  7s. kl_expand_kernel      the gradient's rows from the bitmask, the ranks and v.
#include "dsa_common.hpp"
#include "wave_ops.hpp"

namespace dsa {
namespace kl {

constexpr int kNT = 256;      // threads per workgroup of the small kernels
constexpr int kMaxW = 1024;   // mask words per row in LDS (sparse: Sk <= 32768)
constexpr float kLn2 = 0.69314718055994531f;
constexpr float kEps = 1e-10f;

template <int D, int NW>
struct Cfg {
  static constexpr int NT = 64 * NW;               // threads per workgroup
  static constexpr int TB = 32 * NW;               // tokens per workgroup (32 per wave)
  static constexpr int KC = D <= 128 ? 128 : 64;   // keys per LDS chunk
  static constexpr int ROWB = D * 2;               // bytes per bf16 key row
  static constexpr int STRIDE = ROWB + 16;         // LDS row pitch (bank spread)
  static constexpr int SUBS = KC / 32;             // 32-key sub-tiles per chunk
  static constexpr int KSTEPS = D / 16;            // MFMA k-steps per q.k
  static constexpr int CPR = ROWB / 16;            // 16-byte pieces per key row
  static constexpr int LOADS = KC * CPR / NT;      // 16-byte loads per thread per chunk
  static_assert(D % 32 == 0 && D <= 256 && KC * CPR % NT == 0, "head dim");
};

struct Params {
  const float *index_scores;      // [B, Sq, Sk]
  const void *topk;               // [B, Sq, K] int32 or int64 (sparse only)
  const unsigned char *query;     // [Sq, B, H, D] bf16
  const unsigned char *key;       // [Sk, B, G, D] bf16
  uint32_t *mask;                 // [B, Sq, W]   top-k bitmask (sparse only)
  uint64_t *tiles;                // [B, ceil(Sq / 32), W, 16] lane masks of the admissible set (sparse only)
  float *gamma;                   // [B, Sq]      index normaliser (log2 units)
  float *beta;                    // [B, H, Sq]   attention normaliser (log2 units)
  float *partial;                 // [B, NC, Sq]  KL partial sums per key chunk
  float *rows;                    // [B, Sq]      per-position KL
  float *loss;                    // [1]
  float *partial_r;               // [B, NC, Sq]  gradient: R partial sums per key chunk
  float *grad;                    // [B, Sq, Sk]  gradient: P (pass kernel), then dL/dz
  const float *grad_loss;         // [1]          upstream gradient of the loss (null: the state's v)
  // sparse state: rows of the top-k set in column order
  int32_t *cpre;                  // [B, Sq, NC + 2] set columns before each key chunk, all, and those at or below the diagonal
  float *pc;                      // [B, Sq, K]   P, then v
  float *xc;                      // [B, Sq, K]   index score
  float *flag;                    // [B, Sq]      NaN for a row whose loss is not finite, else 0
  int64_t B, Sq, Sk, H, G, K, W, NC;
  int KC;                         // keys per chunk
  int64_t NI;                     // KL work items per batch (block, chunk pairs)
  int topk_i64;
  int sparse;
  float c;                        // softmax_scale * log2(e)
  float coeff;
};

// Online log2-sum-exp2 pair: (m, d) represents d * 2^m.  m starts at the
// finite kNegBig so that merging two empty pairs never forms inf - inf.
__device__ __forceinline__ void lse_merge(float &m, float &d, float mo, float dd) {
  const float nm = fmaxf(m, mo);
  d = d * exp2_fast(m - nm) + dd * exp2_fast(mo - nm);
  m = nm;
}

// ---------------------------------------------------------------------------
// 1. index normaliser (and the sparse top-k bitmask)
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(kNT) kl_index_stats_kernel(Params p) {
  __shared__ uint32_t bits[4][kMaxW];
  const int w = wave_id(), lane = lane_id();
  const int64_t row = (int64_t)blockIdx.x * 4 + w;  // b * Sq + t
  if (row >= p.B * p.Sq) return;                      // wave-uniform
  const float *I = p.index_scores + row * p.Sk;
  float m = kNegBig, d = 0.0f;
  if (p.sparse) {
    uint32_t *bw = bits[w];
    for (int i = lane; i < p.W; i += 64) bw[i] = 0u;
    wave_lds_sync();
    for (int64_t j = lane; j < p.K; j += 64) {
      const int64_t s = p.topk_i64 ? static_cast<const int64_t *>(p.topk)[row * p.K + j]
                                   : (int64_t) static_cast<const int32_t *>(p.topk)[row * p.K + j];
      if (s >= 0 && s < p.Sk) atomicOr(&bw[s >> 5], 1u << (s & 31));
    }
    wave_lds_sync();
    const int64_t t = row % p.Sq, last_k = t < p.Sk - 1 ? t : p.Sk - 1;
    const int wpc = p.KC / 32;  // words per key chunk
    int32_t *pre = p.cpre != nullptr ? p.cpre + row * (p.NC + 2) : nullptr;
    int before = 0, adm = 0;  // set columns in the earlier rounds' words; those at or below the diagonal
    for (int i0 = 0; i0 < p.W; i0 += 64) {
      const int i = i0 + lane;
      const bool in = i < p.W;
      uint32_t word = in ? bw[i] : 0u;
      if (in) p.mask[row * p.W + i] = word;
      int at = 0;
      if (pre != nullptr) {  // rank of the word's first column, by a prefix sum over the lanes
        const int n = __popc(word), x = (int)wv::wave_incl_scan((uint32_t)n);
        at = before + x - n;
        before += (int)wv::readlane((uint32_t)x, 63);
        if (in && i % wpc == 0) pre[i / wpc] = at;
        const int64_t lb = last_k - (int64_t)i * 32;  // last admissible bit of the word
        adm += __popc(lb >= 31 ? word : (lb < 0 ? 0u : word & ((2u << lb) - 1u)));
      }
      // each set column once (duplicates in the top-k list count once), four loads in flight
      while (word) {
        int bp[4];
        float x[4];
        int n = 0;
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          bp[u] = word ? __builtin_ctz(word) : 0;
          n += word ? 1 : 0;
          word &= word - 1u;  // (0 stays 0)
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) x[u] = u < n ? I[i * 32 + bp[u]] : -INFINITY;
        if (pre != nullptr) {
#pragma unroll
          for (int u = 0; u < 4; ++u)
            if (u < n) p.xc[row * p.K + at + u] = x[u];
          at += n;
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) x[u] *= kLog2e;
        float nm = fmaxf(m, fmaxf(fmaxf(x[0], x[1]), fmaxf(x[2], x[3])));
        d = d * exp2_fast(m - nm) + exp2_fast(x[0] - nm);
#pragma unroll
        for (int u = 1; u < 4; ++u) d += u < n ? exp2_fast(x[u] - nm) : 0.0f;
        m = nm;
      }
    }
    if (pre != nullptr) {
      adm = (int)wv::wave_reduce((uint32_t)adm, wv::AddU());
      if (lane == 0) {
        pre[p.NC] = before;
        pre[p.NC + 1] = adm;
      }
    }
  } else {
    const uint32_t nbytes = (uint32_t)(p.Sk * 4);
    const auto rs = make_buffer_rsrc(I, nbytes);
    const bool vec = (p.Sk & 3) == 0;  // 16-byte aligned rows
    for (int64_t s0 = 4 * lane; s0 < p.Sk; s0 += 256) {
      f32x4 v;
      if (vec) {
        v = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rs, (int)(s0 * 4), 0, 0));
      } else {
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] = buffer_load_f32(rs, (int)((s0 + j) * 4), 0);
      }
      float x[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) x[j] = s0 + j < p.Sk ? v[j] * kLog2e : -INFINITY;
      const float nm = fmaxf(m, fmaxf(fmaxf(x[0], x[1]), fmaxf(x[2], x[3])));
      d = d * exp2_fast(m - nm) + exp2_fast(x[0] - nm) + exp2_fast(x[1] - nm) + exp2_fast(x[2] - nm) +
          exp2_fast(x[3] - nm);
      m = nm;
    }
  }
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) {
    const float mo = __shfl_xor(m, off, 64), dd = __shfl_xor(d, off, 64);
    lse_merge(m, d, mo, dd);
  }
  // no finite-weight column (all -inf, or an empty top-k set): the reference's
  // softmax is NaN; an inf or NaN score makes d NaN, which propagates
  if (lane == 0) p.gamma[row] = d > 0.0f ? m + __builtin_amdgcn_logf(d) : __builtin_nanf("");
}

// ---------------------------------------------------------------------------
// Shared pieces of the two MFMA kernels
// ---------------------------------------------------------------------------
// B operand (q^T, N = token) of head h for token t: lane half g holds
// elements 16k + 8g .. +8 of the row at k-step k (zero past Sq).
template <int D>
__device__ __forceinline__ void load_q_operand(const Params &p, int64_t b, int64_t h, int64_t t,
                                               bf16x8 (&Q)[Cfg<D, 4>::KSTEPS]) {
  const int g = lane_id() >> 5;
  const bool ok = t < p.Sq;
  const unsigned char *row = p.query + (((ok ? t : 0) * p.B + b) * p.H + h) * (int64_t)(D * 2);
#pragma unroll
  for (int k = 0; k < Cfg<D, 4>::KSTEPS; ++k) {
    i32x4 v = {0, 0, 0, 0};
    if (ok) v = ld_global_16(row + (16 * k + 8 * g) * 2);
    Q[k] = as_bf16x8(v);
  }
}

// Cooperative loads of key chunk [k0, k0 + KC) of (b, group grp) into
// registers; rows at or past Sk read zeros (bounded buffer resource).
template <int D, int NW>
struct ChunkLoader {
  using C = Cfg<D, NW>;
  uint32_t off[C::LOADS];
  uint32_t pitch;
  __device__ ChunkLoader(const Params &p) {
    pitch = (uint32_t)(p.B * p.G * C::ROWB);
#pragma unroll
    for (int l = 0; l < C::LOADS; ++l) {
      const int u = threadIdx.x + C::NT * l;
      off[l] = (uint32_t)(u / C::CPR) * pitch + (uint32_t)(u % C::CPR) * 16u;
    }
  }
  __device__ void load(const Params &p, int64_t b, int64_t grp, int64_t k0, i32x4 (&r)[C::LOADS]) const {
    const int64_t nkeys = p.Sk - k0;
    const uint32_t nb = nkeys > 0 ? (uint32_t)((nkeys - 1) * pitch + C::ROWB) : 0u;
    const unsigned char *base = p.key + ((nkeys > 0 ? k0 : 0) * p.B + b) * p.G * C::ROWB + grp * C::ROWB;
    const auto rs = make_buffer_rsrc(base, nb);
#pragma unroll
    for (int l = 0; l < C::LOADS; ++l)
      r[l] = __builtin_bit_cast(i32x4, __builtin_amdgcn_raw_buffer_load_b128(rs, (int)off[l], 0, 0));
  }
  __device__ static void store(unsigned char *ks, const i32x4 (&r)[C::LOADS]) {
#pragma unroll
    for (int l = 0; l < C::LOADS; ++l) {
      const int u = threadIdx.x + C::NT * l;
      *reinterpret_cast<i32x4 *>(ks + (u / C::CPR) * C::STRIDE + (u % C::CPR) * 16) = r[l];
    }
  }
};

// S^T of sub-tile `sub` (32 keys) of the LDS chunk against the wave's 32
// tokens: acc[4i + j] = q(token lane & 31) . k(key 32 sub + 8i + 4g + j).
template <int D>
__device__ __forceinline__ f32x16 qk_subtile(const unsigned char *ks, int sub, const bf16x8 (&Q)[Cfg<D, 4>::KSTEPS]) {
  using C = Cfg<D, 4>;
  const int lane = lane_id();
  const unsigned char *arow = ks + (sub * 32 + (lane & 31)) * C::STRIDE + (lane >> 5) * 16;
  f32x16 acc;
#pragma unroll
  for (int a = 0; a < 16; ++a) acc[a] = 0.0f;
#pragma unroll
  for (int k = 0; k < C::KSTEPS; ++k) {
    const i32x4 av = *reinterpret_cast<const i32x4 *>(arow + 32 * k);
    acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(as_bf16x8(av), Q[k], acc, 0, 0, 0);
  }
  return acc;
}

// Top-k bitmask word of token t covering keys [key0, key0 + 32) (key0 a
// multiple of 32); all ones in dense mode.
__device__ __forceinline__ uint32_t mask_word(const Params &p, int64_t b, int64_t t, int64_t key0) {
  if (!p.sparse) return 0xffffffffu;
  return t < p.Sq ? p.mask[(b * p.Sq + t) * p.W + (key0 >> 5)] : 0u;
}

// Admissible-column bits of accumulator register a = 4i + j (key
// key0 + 8i + 4g + j) for token t: s <= t, s < Sk, t < Sq and, sparse, in the
// top-k set (bit of `word`).  Word-level: clear the bits past the last
// admissible key, then gather the lane half's four 4-bit groups.
__device__ __forceinline__ uint32_t valid_bits(const Params &p, uint32_t word, int64_t t, int64_t key0) {
  const int g = lane_id() >> 5;
  const int64_t last = (t < p.Sk - 1 ? t : p.Sk - 1) - key0;  // last admissible m
  const uint32_t keep = t >= p.Sq || last < 0 ? 0u : (last >= 31 ? 0xffffffffu : (2u << last) - 1u);
  const uint32_t w = (word & keep) >> (4 * g);
  return (w & 0xfu) | ((w >> 4) & 0xf0u) | ((w >> 8) & 0xf00u) | ((w >> 12) & 0xf000u);
}

// acc if bit a of vb is set, -inf otherwise (sign-extended bit field as a
// select mask: one bfe + one bfi).
__device__ __forceinline__ float keep_or_neginf(float acc, uint32_t vb, int a) {
  const uint32_t m = (uint32_t)(((int32_t)(vb << (31 - a))) >> 31);
  return __uint_as_float((m & __float_as_uint(acc)) | (~m & 0xff800000u));
}

// One v_max3_f32 (a NaN operand is dropped, as fmaxf drops it; its exp2 term
// still joins the sum).  Not for accumulators straight from an MFMA: the wait
// that their first VALU read needs is inserted for instructions the compiler
// knows, not for asm.
__device__ __forceinline__ float max3(float a, float b, float c) {
  float r;
  asm("v_max3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
  return r;
}

// Chunks of KC keys that token block blk (TB tokens) needs: keys up to
// min(last token of the block, Sk - 1).
__device__ __forceinline__ int64_t block_chunks(const Params &p, int64_t blk, int64_t TB, int64_t KC) {
  const int64_t lt = (TB * (blk + 1) < p.Sq ? TB * (blk + 1) : p.Sq) - 1;
  return (lt < p.Sk - 1 ? lt : p.Sk - 1) / KC + 1;
}

// Lane masks of the admissible set (sparse): for 32 tokens and 32 keys, word
// a = 4 i + j holds at bit (32 g + token) whether key 8 i + 4 g + j is in the
// token's top-k set at or below its diagonal: the select operand, straight from
// scalar registers, of accumulator register a in kl_attn_stats_kernel.  One
// transposition serves every head; forming the selects per head from the row
// bitmask takes two VALU operations an element there (174 us with lane masks at
// b = 2, s = 4096, 32 heads of 128; use_lane_masks).  A workgroup takes a (b, 32-token block) and
// every gridDim.y-th group of four words at or below the diagonal.
__global__ void __launch_bounds__(kNT) kl_mask_tiles_kernel(Params p) {
  const int lane = lane_id(), g = lane >> 5, l32 = lane & 31;
  const int64_t NTB = (p.Sq + 31) / 32;
  const int64_t tb = blockIdx.x % NTB, b = blockIdx.x / NTB, t = tb * 32 + l32;
  const int64_t last_t = tb * 32 + 31 < p.Sk - 1 ? tb * 32 + 31 : p.Sk - 1;
  uint64_t *tiles = p.tiles + (b * NTB + tb) * p.W * 16;
  for (int64_t wi = blockIdx.y * (kNT / 64) + wave_id(); wi <= last_t / 32; wi += gridDim.y * (kNT / 64)) {
    const int64_t last = (t < p.Sk - 1 ? t : p.Sk - 1) - wi * 32;
    uint32_t word = t < p.Sq ? p.mask[(b * p.Sq + t) * p.W + wi] : 0u;
    word = last < 0 ? 0u : (last >= 31 ? word : word & ((2u << last) - 1u));
    word >>= 4 * g;
    uint64_t mine = 0;
#pragma unroll
    for (int a = 0; a < 16; ++a) {
      const uint64_t m = __ballot((word >> (8 * (a >> 2) + (a & 3))) & 1u);
      if (lane == a) mine = m;
    }
    if (lane < 16) tiles[wi * 16 + lane] = mine;
  }
}

// ---------------------------------------------------------------------------
// 2. attention normalisers beta_h[t] (log2 units of c * q.k)
// ---------------------------------------------------------------------------
// The admissible set: every column up to the diagonal, or the top-k set by the rows'
// bitmask or by lane masks.
enum StatsSet { kAllColumns, kRowBits, kLaneMasks };

template <int D, int NW, StatsSet SET>
__global__ void __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(NW == 8 ? 4 : 2)))
kl_attn_stats_kernel(Params p) {
  using C = Cfg<D, NW>;
  constexpr int kTB = C::TB;
  __shared__ __attribute__((aligned(16))) unsigned char KS[2][C::KC * C::STRIDE];
  const int w = wave_id(), lane = lane_id(), g = lane >> 5;
  const int64_t NB = (p.Sq + kTB - 1) / kTB, NP = (NB + 1) / 2;
  const int64_t bid = xcd_remap(blockIdx.x, gridDim.x);
  const int64_t pair = bid % NP, bh = bid / NP, h = bh % p.H, b = bh / p.H;
  const int64_t grp = h / (p.H / p.G);
  ChunkLoader<D, NW> ld(p);

  for (int half = 0; half < 2; ++half) {
    const int64_t blk = half == 0 ? NB - 1 - pair : pair;  // the long block first
    if (half == 1 && blk == NB - 1 - pair) break;          // odd NB: middle block once
    const int64_t t0 = blk * kTB, wt0 = t0 + 32 * w, t = wt0 + (lane & 31);
    const int64_t wt_last = wt0 + 31;
    const int64_t kend = p.Sk < t0 + kTB ? p.Sk : t0 + kTB;  // keys s <= last token of the block
    const int nch = (int)((kend + C::KC - 1) / C::KC);
    bf16x8 Q[C::KSTEPS];
    load_q_operand<D>(p, b, h, t, Q);
    float m = kNegBig, d = 0.0f;
    i32x4 kr[C::LOADS];
    __syncthreads();  // the previous block's waves are done with the LDS chunks
    ld.load(p, b, grp, 0, kr);
    ChunkLoader<D, NW>::store(KS[0], kr);
    __syncthreads();
    // lane masks: scalar loads, the tile of 32 keys is 16 words
    typedef const __attribute__((address_space(4))) uint64_t *scalar_u64;
    scalar_u64 tiles = nullptr;
    if constexpr (SET == kLaneMasks)
      if (wt0 < p.Sq) tiles = (scalar_u64)(uintptr_t)(p.tiles + (b * ((p.Sq + 31) / 32) + wt0 / 32) * p.W * 16);
    // row bits: the chunk's words are loaded one chunk ahead
    uint32_t mw[C::SUBS];
#pragma unroll
    for (int sub = 0; sub < C::SUBS; ++sub) mw[sub] = SET == kRowBits ? mask_word(p, b, t, 32 * sub) : 0xffffffffu;
    for (int ci = 0; ci < nch; ++ci) {
      if (ci + 1 < nch) ld.load(p, b, grp, (int64_t)(ci + 1) * C::KC, kr);
      uint32_t mwn[C::SUBS];
      if constexpr (SET == kRowBits) {
#pragma unroll
        for (int sub = 0; sub < C::SUBS; ++sub)
          mwn[sub] = ci + 1 < nch ? mask_word(p, b, t, (int64_t)(ci + 1) * C::KC + 32 * sub) : 0u;
      }
      const unsigned char *ks = KS[ci & 1];
#pragma unroll
      for (int sub = 0; sub < C::SUBS; ++sub) {
        const int64_t key0 = (int64_t)ci * C::KC + 32 * sub;
        if (key0 > wt_last || key0 >= p.Sk || wt0 >= p.Sq) continue;  // wave-uniform: wholly above the diagonal
        const f32x16 acc = qk_subtile<D>(ks, sub, Q);
        // c > 0: max(c * acc) = c * max(acc), and exp2(c * acc - nm) is one fma
        float x[16], lm;
        if constexpr (SET == kLaneMasks) {
#pragma unroll
          for (int a = 0; a < 16; ++a) {
            const uint64_t on = tiles[(key0 >> 5) * 16 + a];
            x[a] = __builtin_amdgcn_inverse_ballot_w64(on) ? acc[a] : -INFINITY;
          }
          lm = x[0];
#pragma unroll
          for (int a = 1; a < 15; a += 2) lm = max3(lm, x[a], x[a + 1]);
          lm = max3(lm, x[15], x[15]);
        } else {
          if (SET == kRowBits || key0 + 31 > wt0 || key0 + 31 >= p.Sk || wt_last >= p.Sq) {
            const uint32_t vb = valid_bits(p, mw[sub], t, key0);
#pragma unroll
            for (int a = 0; a < 16; ++a) x[a] = keep_or_neginf(acc[a], vb, a);
          } else {
#pragma unroll
            for (int a = 0; a < 16; ++a) x[a] = acc[a];
          }
          lm = x[0];
#pragma unroll
          for (int a = 1; a < 16; ++a) lm = fmaxf(lm, x[a]);
        }
        const float nm = fmaxf(m, lm * p.c);
        float s = 0.0f;
#pragma unroll
        for (int a = 0; a < 16; ++a) s += exp2_fast(fmaf(x[a], p.c, -nm));
        d = d * exp2_fast(m - nm) + s;
        m = nm;
      }
      if constexpr (SET == kRowBits) {
#pragma unroll
        for (int sub = 0; sub < C::SUBS; ++sub) mw[sub] = mwn[sub];
      }
      if (ci + 1 < nch) {
        ChunkLoader<D, NW>::store(KS[(ci + 1) & 1], kr);
        __syncthreads();
      }
    }
    // the two lane halves hold the same token's other keys
    const float mo = __shfl_xor(m, 32, 64), dd = __shfl_xor(d, 32, 64);
    lse_merge(m, d, mo, dd);
    if (g == 0 && t < p.Sq)
      p.beta[(b * p.H + h) * p.Sq + t] = d > 0.0f ? m + __builtin_amdgcn_logf(d) : -INFINITY;
  }
}

// ---------------------------------------------------------------------------
// 3. KL partial sums per (token, key chunk)
// ---------------------------------------------------------------------------
// The work per (head, token, key) is one fma, one exp2 (quarter rate) and one
// add beside the products: 384 VALU cycles per 32x32 tile against 256 of MFMA at
// D = 128, so the loop is built to keep the VALU fed: the head's q and k reach
// LDS by coalesced LDS-DMA loads a head ahead (read as operands straight from
// global, q's 32 rows of 16 bytes per instruction cost more address cycles than
// the arithmetic), each wave owns its 32 tokens' q slice, and a wave whose four
// key sub-tiles all count runs the next sub-tile's products under the current
// one's exp2.  256 tokens share a key chunk, or 128 (launch_by_size).  At b = 2, s = 4096,
// 32 heads of 128: 230 us, 315 with the operands read straight from global; the VALU's
// share is about 150 us (544 workgroups are a little over two rounds of 256 compute
// units).
template <int D, int NW>
struct PassCfg {
  using C = Cfg<D, NW>;
  static constexpr int QP = 32 * C::ROWB / 1024;            // 1 KiB pieces of a wave's q slice
  static constexpr int KP = C::KC * C::ROWB / 1024 / NW;    // and of the key chunk, per wave
  static constexpr int OFF_Q = 2 * C::KC * C::ROWB;
  static constexpr int PT_STRIDE = C::KC + 4;               // sparse state: a token's P row in LDS (floats; rows on distinct banks)
  static constexpr int PT_BYTES = 32 * PT_STRIDE * 4;
  static constexpr int LOOP_BYTES = OFF_Q + NW * 32 * C::ROWB;
  static constexpr int BYTES = LOOP_BYTES > NW * PT_BYTES ? LOOP_BYTES : NW * PT_BYTES;
  static_assert(C::KC * C::ROWB % (1024 * NW) == 0 && BYTES <= 160 * 1024, "pass LDS");
  // rows unpadded; 16-byte chunk c of row r at c ^ swz(r): 16 consecutive rows on distinct banks
  __device__ static __forceinline__ int swz(int r) { return C::CPR % 16 == 0 ? (r & 15) : ((r >> 1) & 7); }
  static_assert(C::CPR % 8 == 0, "swizzle within the row");
};

// kOwnKeys: every head has its key head, whose chunk's loads are spread over the
// products as q's are.  kSharedKeys: a group of heads shares one; the next group's
// chunk is fetched at once, by the group's last head, and one barrier serves the
// group (spread conditionally, or at once for every head, the loads cost the former
// case 3 to 7%).  kFarRows: as shared, and a wave's 32 query rows, B * H * D * 2 bytes
// apart, span more than the 4 GiB that the DMA's 32-bit offsets reach (a batch of
// several thousand short sequences): each lane reads its row as operands by 64-bit
// addresses, one sub-tile's products after the other.
enum PassForm { kOwnKeys, kSharedKeys, kFarRows };

// LOSS: the KL partial sums; GRAD: P (p.grad, or the sparse state's p.pc) and the
// R partial sums.
template <int D, int NW, bool LOSS, bool GRAD, PassForm FORM>
__global__ void __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(NW / 4))) kl_pass_kernel(Params p) {
  constexpr bool OWN = FORM == kOwnKeys, FAR = FORM == kFarRows;
  using C = Cfg<D, NW>;
  using PC = PassCfg<D, NW>;
  constexpr int kTB = C::TB;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const int w = wave_id(), lane = lane_id(), g = lane >> 5;
  // Work items are the (b, block, chunk) pairs at or below the diagonal:
  // first every block's full chunks, block-major, then the cheaper diagonal
  // chunks (one per block), so a last partial round of the grid is short
  // work.  The grid is padded to a multiple of 8 so that each XCD takes one
  // contiguous, equal share (consecutive items share a token block's q rows
  // in that XCD's L2).
  const uint32_t NB = (uint32_t)((p.Sq + kTB - 1) / kTB), NI = (uint32_t)p.NI, nb = (uint32_t)p.B;
  const uint32_t bid = (uint32_t)xcd_remap(blockIdx.x, gridDim.x);
  if (bid >= nb * NI) return;
  const uint32_t nfull = NI - NB;  // items per batch before the diagonal ones
  uint32_t bb, bk = 0, cc;
  if (bid < nb * nfull) {
    bb = bid / nfull;
    uint32_t rem = bid - bb * nfull;
    for (;; ++bk) {  // scalar walk over the blocks' full-chunk counts (NB steps at most)
      const uint32_t n = (uint32_t)block_chunks(p, bk, kTB, C::KC) - 1;
      if (rem < n) break;
      rem -= n;
    }
    cc = rem;
  } else {
    const uint32_t r = bid - nb * nfull;
    bb = r / NB;
    bk = r - bb * NB;
    cc = (uint32_t)block_chunks(p, bk, kTB, C::KC) - 1;
  }
  const int64_t b = bb, blk = bk, ci = cc;
  const int64_t t0 = blk * kTB, k0 = ci * C::KC;
  const int64_t wt0 = t0 + 32 * w, t = wt0 + (lane & 31), wt_last = wt0 + 31;

  bool sub_on[C::SUBS];
#pragma unroll
  for (int sub = 0; sub < C::SUBS; ++sub) {
    const int64_t key0 = k0 + 32 * sub;
    sub_on[sub] = key0 <= wt_last && key0 < p.Sk && wt0 < p.Sq;  // wave-uniform
  }

  float P[C::SUBS][16];
#pragma unroll
  for (int sub = 0; sub < C::SUBS; ++sub)
#pragma unroll
    for (int a = 0; a < 16; ++a) P[sub][a] = 0.0f;

  // this lane's source bytes in its wave's pieces of the q slice and of the key chunk
  const uint32_t qpitch = (uint32_t)(p.B * p.H * C::ROWB), kpitch = (uint32_t)(p.B * p.G * C::ROWB);
  uint32_t qo[PC::QP], ko[PC::KP];
#pragma unroll
  for (int i = 0; i < PC::QP; ++i) {
    const int u = 64 * i + lane, r = u / C::CPR;
    qo[i] = (uint32_t)r * qpitch + (uint32_t)(((u - r * C::CPR) ^ PC::swz(r)) * 16);  // (not FAR: below 4 GiB)
  }
#pragma unroll
  for (int i = 0; i < PC::KP; ++i) {
    const int u = 64 * (w * PC::KP + i) + lane, r = u / C::CPR;
    ko[i] = (uint32_t)r * kpitch + (uint32_t)(((u - r * C::CPR) ^ PC::swz(r)) * 16);
  }
  const int64_t nq = p.Sq - wt0 < 32 ? p.Sq - wt0 : 32;  // (rows past Sq and Sk read zeros)
  const uint32_t qbytes = nq > 0 ? (uint32_t)((nq - 1) * qpitch + C::ROWB) : 0u;
  const int64_t nk = p.Sk - k0 < C::KC ? p.Sk - k0 : C::KC;
  const uint32_t kbytes = (uint32_t)((nk - 1) * kpitch + C::ROWB);
  const unsigned char *qb = p.query + (((nq > 0 ? wt0 : 0) * p.B + b) * p.H) * (int64_t)C::ROWB;
  const unsigned char *kbase = p.key + ((k0 * p.B + b) * p.G) * (int64_t)C::ROWB;
  const uint32_t lds = lds_address(smem);
  const uint32_t q_lds = lds + (uint32_t)(PC::OFF_Q + w * 32 * C::ROWB);
  // this wave's loads: its share of a key head's chunk, into buffer kbuf, and its q slice of a head
  const int hpg = OWN ? 1 : (int)(p.H / p.G), H = (int)p.H;
  auto fetch_k = [&](i32x4 krs, int kbuf, int i) {
    lds_dma_16(lds + (uint32_t)(kbuf * C::KC * C::ROWB + (w * PC::KP + i) * 1024), ko[i], krs, 0u);
  };
  auto fetch_q = [&](i32x4 qrs, int i) { lds_dma_16(q_lds + (uint32_t)(i * 1024), qo[i], qrs, 0u); };
  auto key_rs = [&](int grp) { return make_buffer_words(kbase + grp * C::ROWB, kbytes); };
  auto query_rs = [&](int h) { return make_buffer_words(qb + h * C::ROWB, qbytes); };
  constexpr int NK = OWN ? PC::KP : 0, NF = NK + (FAR ? 0 : PC::QP);  // loads spread over a head's products: k's, then q's
  auto fetch = [&](i32x4 krs, i32x4 qrs, int kbuf, int i) {
    if (i < NK) fetch_k(krs, kbuf, i < PC::KP ? i : 0);
    else fetch_q(qrs, i - NK < PC::QP ? i - NK : 0);
  };
  bool all_on = !FAR, any_on = false;  // wave-uniform
#pragma unroll
  for (int sub = 0; sub < C::SUBS; ++sub) {
    all_on = all_on && sub_on[sub];
    any_on = any_on || sub_on[sub];
  }
  // operand of k-step k: row (lane & 31), chunk 2 k + g
  const int l32 = lane & 31;
  auto operand = [&](const unsigned char *tile, int r0, int k) {
    return as_bf16x8(*reinterpret_cast<const i32x4 *>(tile + (r0 + l32) * C::ROWB + (((2 * k + g) ^ PC::swz(l32)) * 16)));
  };
  const float *beta_bt = p.beta + b * p.H * p.Sq + (t < p.Sq ? t : 0);
  i32x4 krs = key_rs(0), qrs = query_rs(0);
#pragma unroll
  for (int i = NK; i < PC::KP; ++i) fetch_k(krs, 0, i);
#pragma unroll
  for (int i = 0; i < NF; ++i) fetch(krs, qrs, 0, i);
  // The previous head's last sub-tile and its normaliser: its exp2 work runs
  // under the next head's first products (before head 0: exp2(-inf) = 0).
  f32x16 cur;
#pragma unroll
  for (int a = 0; a < 16; ++a) cur[a] = 0.0f;
  float bprev = INFINITY, bn = beta_bt[0];
  int grp = 0, left = hpg;  // the head's key group, and its heads still to come
  for (int h = 0; h < H; ++h) {
    __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): this head's q and k, fetched a head ago
    if (OWN || left == hpg) __syncthreads();  // every wave's share of the group's k; the other k buffer is consumed
    const unsigned char *ks = smem + (grp & 1) * C::KC * C::ROWB;
    bf16x8 Q[C::KSTEPS];
#pragma unroll
    for (int k = 0; k < C::KSTEPS; ++k)
      if constexpr (!FAR) Q[k] = operand(smem + PC::OFF_Q + w * 32 * C::ROWB, 0, k);
    if constexpr (FAR) load_q_operand<D>(p, b, h, t, Q);
    const float bh = bn;
    const int hn = h + 1 < H ? h + 1 : h;  // (past the last head: its own again, unused)
    bn = beta_bt[(int64_t)hn * p.Sq];
    qrs = query_rs(hn);
    if (OWN || --left == 0) {  // the last head of its group: the next group's keys
      left = hpg;
      ++grp;
      krs = key_rs(grp < (int)p.G ? grp : grp - 1);
#pragma unroll
      for (int i = NK; i < PC::KP; ++i) fetch_k(krs, grp & 1, i);
    }
    const int kb = grp & 1;
    __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): the q slice is in registers, its LDS free
    if (all_on) {
      // key operands are read two products ahead
      constexpr int kSteps = C::SUBS * C::KSTEPS;
      auto key_operand = [&](int i) { return operand(ks, 32 * (i / C::KSTEPS), i % C::KSTEPS); };
      bf16x8 ring[3];
      ring[0] = key_operand(0);
      ring[1] = key_operand(1);
#pragma unroll
      for (int sub = 0; sub < C::SUBS; ++sub) {
        // sub-tile sub's products, each followed by its share of the exp2 work of the sub-tile before it
        constexpr int kE = 16 / C::KSTEPS > 0 ? (16 + C::KSTEPS - 1) / C::KSTEPS : 1;
        const int ps = sub == 0 ? C::SUBS - 1 : sub - 1;
        const float pb = sub == 0 ? bprev : bh;
        f32x16 nxt;
#pragma unroll
        for (int a = 0; a < 16; ++a) nxt[a] = 0.0f;
#pragma unroll
        for (int k = 0; k < C::KSTEPS; ++k) {
          const int i = sub * C::KSTEPS + k;
          if (i + 2 < kSteps) ring[(i + 2) % 3] = key_operand(i + 2);
          nxt = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ring[i % 3], Q[k], nxt, 0, 0, 0);
#pragma unroll
          for (int e = 0; e < kE; ++e)
            if (k * kE + e < 16) P[ps][k * kE + e] += exp2_fast(fmaf(cur[k * kE + e], p.c, -pb));
          // the next head's loads, spread over the first sub-tiles
          constexpr int kPer = (NF + C::KSTEPS * (C::SUBS - 1) - 1) / (C::KSTEPS * (C::SUBS - 1));
#pragma unroll
          for (int u = 0; u < kPer; ++u) {
            const int f = i * kPer + u;
            if (f < NF) fetch(krs, qrs, kb, f);
          }
          __builtin_amdgcn_sched_barrier(0);  // keep this order
        }
        cur = nxt;
      }
      bprev = bh;
    } else {
#pragma unroll
      for (int i = 0; i < NF; ++i) fetch(krs, qrs, kb, i);
      if (any_on) {
#pragma unroll
        for (int sub = 0; sub < C::SUBS; ++sub) {
          if (!sub_on[sub]) continue;
          f32x16 acc;
#pragma unroll
          for (int a = 0; a < 16; ++a) acc[a] = 0.0f;
#pragma unroll
          for (int k = 0; k < C::KSTEPS; ++k)
            acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(operand(ks, 32 * sub, k), Q[k], acc, 0, 0, 0);
#pragma unroll
          for (int a = 0; a < 16; ++a) P[sub][a] += exp2_fast(fmaf(acc[a], p.c, -bh));
        }
      }
    }
  }
  __builtin_amdgcn_s_waitcnt(0x0F70);  // the last loads have landed before the LDS is given up
  if (all_on) {
#pragma unroll
    for (int a = 0; a < 16; ++a) P[C::SUBS - 1][a] += exp2_fast(fmaf(cur[a], p.c, -bprev));
  }

  const float inv_h = 1.0f / (float)p.H;  // P = (head sum) / H on admissible columns, 0 elsewhere
  const int64_t row = b * p.Sq + (t < p.Sq ? t : 0);
  if (GRAD && p.pc != nullptr) {
    // sparse state: the set columns' P at their rank (kl_rows_state_kernel forms
    // the rest).  P goes through LDS, so that each lane walks the set bits of half
    // its token's words instead of testing every accumulator
    __syncthreads();  // every wave is done with the key chunks
    float *tile = reinterpret_cast<float *>(smem + w * PC::PT_BYTES);
    if (any_on) {
#pragma unroll
      for (int sub = 0; sub < C::SUBS; ++sub)
#pragma unroll
        for (int i = 0; i < 4; ++i)
          *reinterpret_cast<f32x4 *>(tile + l32 * PC::PT_STRIDE + 32 * sub + 8 * i + 4 * g) =
              f32x4{P[sub][4 * i], P[sub][4 * i + 1], P[sub][4 * i + 2], P[sub][4 * i + 3]};
      wave_lds_sync();
      float *crow = p.pc + row * p.K;
      int at = p.cpre[row * (p.NC + 2) + ci];  // rank of the chunk's first set column
      uint32_t words[C::SUBS];
#pragma unroll
      for (int sub = 0; sub < C::SUBS; ++sub) words[sub] = mask_word(p, b, t, k0 + 32 * sub);
#pragma unroll
      for (int sub = 0; sub < C::SUBS; ++sub) {
        if (sub >= C::SUBS / 2 == (g != 0)) {  // lane half 0: the first words, half 1: the last
          const int64_t last = (t < p.Sk - 1 ? t : p.Sk - 1) - (k0 + 32 * sub);  // last admissible bit
          uint32_t word = t >= p.Sq || last < 0 ? 0u : words[sub] & (last >= 31 ? 0xffffffffu : (2u << last) - 1u);
          int r = at;
          while (word) {
            const int bit = __builtin_ctz(word);
            word &= word - 1u;
            crow[r++] = tile[l32 * PC::PT_STRIDE + 32 * sub + bit] * inv_h;
          }
        }
        at += __popc(words[sub]);
      }
    }
    return;
  }
  // admissible bits of this lane's 16 keys per sub-tile
  uint32_t vb[C::SUBS];
#pragma unroll
  for (int sub = 0; sub < C::SUBS; ++sub)
    vb[sub] = sub_on[sub] ? valid_bits(p, mask_word(p, b, t, k0 + 32 * sub), t, k0 + 32 * sub) : 0u;

  // KL terms of the chunk against Q; the index scores of every sub-tile are loaded before any is used
  const float gam = t < p.Sq ? p.gamma[b * p.Sq + t] : 0.0f;
  const float *irow = p.index_scores + b * p.Sq * p.Sk;
  const auto irs = make_buffer_rsrc(irow, (uint32_t)(p.Sq * p.Sk * 4));
  const bool vec = (p.Sk & 3) == 0;  // rows 16-byte aligned: one b128 load per 4 keys
  f32x4 iv[C::SUBS][4];
#pragma unroll
  for (int sub = 0; sub < C::SUBS; ++sub)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      // keys s0 .. s0 + 3 of this lane's row; reads past the row (or past Sq) only feed inadmissible columns
      const int64_t s0 = k0 + 32 * sub + 8 * i + 4 * g;
      if (vec) {
        const uint32_t off = t < p.Sq && s0 < p.Sk ? (uint32_t)((t * p.Sk + s0) * 4) : 0xfffffff0u;
        iv[sub][i] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(irs, (int)off, 0, 0));
      } else {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int64_t s = s0 + j;
          const uint32_t off = (t < p.Sq && s < p.Sk) ? (uint32_t)((t * p.Sk + s) * 4) : 0xfffffff0u;
          iv[sub][i][j] = buffer_load_f32(irs, (int)off, 0);
        }
      }
    }
  float kl = 0.0f, rsum = 0.0f;
  float *grow = GRAD ? p.grad + row * p.Sk : nullptr;
#pragma unroll
  for (int sub = 0; sub < C::SUBS; ++sub) {
    if (!sub_on[sub]) continue;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int64_t s0 = k0 + 32 * sub + 8 * i + 4 * g;
      f32x4 pv;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int a = 4 * i + j;
        const bool on = (vb[sub] >> a) & 1u;
        const float pr = on ? P[sub][a] * inv_h : 0.0f;
        pv[j] = pr;
        if (on) {
          const float q = exp2_fast(fmaf(iv[sub][i][j], kLog2e, -gam));
          if constexpr (LOSS) kl += pr * (__builtin_amdgcn_logf(pr + kEps) - __builtin_amdgcn_logf(q + kEps));
          if constexpr (GRAD) rsum += pr * (q / (q + kEps));
        }
      }
      if (GRAD && t < p.Sq && s0 < p.Sk) {  // 0 off the admissible set
        if (vec) {
          *reinterpret_cast<f32x4 *>(grow + s0) = pv;
        } else {
#pragma unroll
          for (int j = 0; j < 4; ++j)
            if (s0 + j < p.Sk) grow[s0 + j] = pv[j];
        }
      }
    }
  }
  if constexpr (GRAD) {
    rsum = sum_halves(rsum);
    if (g == 0 && t < p.Sq) p.partial_r[(b * p.NC + ci) * p.Sq + t] = rsum;
  }
  if constexpr (LOSS) {
    kl = sum_halves(kl) * kLn2;
    if (g == 0 && t < p.Sq) p.partial[(b * p.NC + ci) * p.Sq + t] = kl;
  }
}

// ---------------------------------------------------------------------------
// 4. row losses, 5. mean
// ---------------------------------------------------------------------------
template <int D>
__global__ void __launch_bounds__(kNT) kl_rows_kernel(Params p) {
  const int64_t row = (int64_t)blockIdx.x * kNT + threadIdx.x;
  if (row >= p.B * p.Sq) return;
  const int64_t b = row / p.Sq, t = row % p.Sq;
  const int64_t last_k = t < p.Sk - 1 ? t : p.Sk - 1;
  const int64_t cmax = last_k / Cfg<D, 4>::KC;
  float s = 0.0f;
  for (int64_t c = 0; c <= cmax; ++c) s += p.partial[(b * p.NC + c) * p.Sq + t];
  const bool no_target = !(p.beta[b * p.H * p.Sq + t] > -INFINITY);
  const float gam = p.gamma[row];
  if (no_target || gam != gam) s = __builtin_nanf("");
  p.rows[row] = s;
}

// 6. gradient row: dL/dz over P in place (one workgroup per (b, t) row)
template <int D>
__global__ void __launch_bounds__(kNT) kl_grad_kernel(Params p) {
  const int64_t row = blockIdx.x;
  const int64_t b = row / p.Sq, t = row % p.Sq;
  const int64_t last_k = t < p.Sk - 1 ? t : p.Sk - 1;  // P is written for s <= last_k
  const int64_t cmax = last_k / Cfg<D, 4>::KC;
  float R = 0.0f;
  for (int64_t c = 0; c <= cmax; ++c) R += p.partial_r[(b * p.NC + c) * p.Sq + t];
  const bool no_target = !(p.beta[b * p.H * p.Sq + t] > -INFINITY);
  const float gam = p.gamma[row];
  const bool nan_row = no_target || gam != gam;
  // (no upstream gradient: v itself, to be scaled by kl_scale_kernel)
  const float gs = p.grad_loss != nullptr ? p.grad_loss[0] * p.coeff / (float)(p.B * p.Sq) : 1.0f;
  const float *zrow = p.index_scores + row * p.Sk;
  float *grow = p.grad + row * p.Sk;
  const uint32_t *mrow = p.sparse ? p.mask + row * p.W : nullptr;
  const bool vec = (p.Sk & 3) == 0;
  for (int64_t s0 = 4 * (int64_t)threadIdx.x; s0 < p.Sk; s0 += 4 * kNT) {
    f32x4 z, pr, out;
    if (vec) {
      z = *reinterpret_cast<const f32x4 *>(zrow + s0);
      pr = s0 <= last_k ? *reinterpret_cast<const f32x4 *>(grow + s0) : f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    } else {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        z[j] = s0 + j < p.Sk ? zrow[s0 + j] : 0.0f;
        pr[j] = s0 + j <= last_k ? grow[s0 + j] : 0.0f;
      }
    }
    const uint32_t mw = mrow ? mrow[s0 >> 5] >> (s0 & 31) : 0xfu;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float q = ((mw >> j) & 1u) ? exp2_fast(fmaf(z[j], kLog2e, -gam)) : 0.0f;
      const float pj = s0 + j <= last_k ? pr[j] : 0.0f;
      out[j] = nan_row ? __builtin_nanf("") : gs * fmaf(q, R, -(pj * (q / (q + kEps))));
    }
    if (vec) {
      *reinterpret_cast<f32x4 *>(grow + s0) = out;
    } else {
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (s0 + j < p.Sk) grow[s0 + j] = out[j];
    }
  }
}

// Sparse state, one wave per row: the row's loss and R over its set columns (a
// fixed order: lane strides, then a tree), then v over P in place.  A twentieth
// of the columns a dense chunk would visit, all lanes busy: the logarithms and
// the division cost 35 K cycles per 256 x 128 chunk in the pass kernel.
template <int D>
__global__ void __launch_bounds__(kNT) kl_rows_state_kernel(Params p) {
  const int lane = lane_id();
  const int64_t row = (int64_t)blockIdx.x * 4 + wave_id();
  if (row >= p.B * p.Sq) return;  // wave-uniform
  const int64_t b = row / p.Sq, t = row % p.Sq;
  const bool no_target = !(p.beta[b * p.H * p.Sq + t] > -INFINITY);
  const float gam = p.gamma[row];
  const bool nan_row = no_target || gam != gam;
  const int32_t *pre = p.cpre + row * (p.NC + 2);
  const int n = pre[p.NC], adm = pre[p.NC + 1];
  float *v = p.pc + row * p.K;
  const float *x = p.xc + row * p.K;
  float kl = 0.0f, R = 0.0f;
  for (int e = lane; e < adm; e += 64) {  // (columns past the diagonal have no target)
    const float q = exp2_fast(fmaf(x[e], kLog2e, -gam)), pe = v[e];
    kl += pe * (__builtin_amdgcn_logf(pe + kEps) - __builtin_amdgcn_logf(q + kEps));
    R += pe * (q / (q + kEps));
  }
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) {
    kl += __shfl_xor(kl, off, 64);
    R += __shfl_xor(R, off, 64);
  }
  if (lane == 0) {
    p.rows[row] = nan_row ? __builtin_nanf("") : kl * kLn2;
    // a NaN or infinite P, from any head, makes R so, and 0 * R (Q is 0 outside the
    // set) every other column's gradient NaN
    p.flag[row] = nan_row || !(fabsf(R) < INFINITY) ? __builtin_nanf("") : 0.0f;
  }
  for (int e = lane; e < n; e += 64) {
    const float q = exp2_fast(fmaf(x[e], kLog2e, -gam));
    const float pe = e < adm ? v[e] : 0.0f;
    v[e] = fmaf(q, R, -(pe * (q / (q + kEps))));
  }
}

// The gradient from the state: g * coeff / (B * Sq) * v.
__global__ void __launch_bounds__(kNT) kl_scale_kernel(const float *v, const float *grad_loss, float *out, int64_t n,
                                                       float coeff, float denom) {
  const float gs = grad_loss[0] * coeff / denom;
  const int64_t i0 = ((int64_t)blockIdx.x * kNT + threadIdx.x) * 4, stride = (int64_t)gridDim.x * kNT * 4;
  for (int64_t i = i0; i < n; i += stride) {
    if (i + 4 <= n) {
      *reinterpret_cast<f32x4 *>(out + i) = gs * *reinterpret_cast<const f32x4 *>(v + i);
    } else {
      for (int64_t j = i; j < n; ++j) out[j] = gs * v[j];
    }
  }
}
// Sparse: one workgroup per row writes every column; a set column's rank is the
// columns before its chunk plus those before it in the chunk's words.
__global__ void __launch_bounds__(kNT) kl_expand_kernel(Params p) {
  const int64_t row = blockIdx.x;
  const float gs = p.grad_loss[0] * p.coeff / (float)(p.B * p.Sq);
  const float off = p.flag[row];  // 0, or NaN over the whole row
  const uint32_t *mrow = p.mask + row * p.W;
  const int32_t *pre = p.cpre + row * (p.NC + 2);
  const float *v = p.pc + row * p.K;
  float *grow = p.grad + row * p.Sk;
  const bool vec = (p.Sk & 3) == 0;
  const int wpc = p.KC / 32;
  for (int64_t s0 = 4 * (int64_t)threadIdx.x; s0 < p.Sk; s0 += 4 * kNT) {
    const int wi = (int)(s0 >> 5), sh = (int)(s0 & 31);
    const uint32_t word = mrow[wi];
    f32x4 out = {gs * off, gs * off, gs * off, gs * off};
    if ((word >> sh) & 0xfu) {
      int at = pre[wi / wpc] + __popc(word & ((1u << sh) - 1u));
      for (int k = wi / wpc * wpc; k < wi; ++k) at += __popc(mrow[k]);
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if ((word >> (sh + j)) & 1u) out[j] = gs * (v[at++] + off);
    }
    if (vec) {
      *reinterpret_cast<f32x4 *>(grow + s0) = out;
    } else {
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (s0 + j < p.Sk) grow[s0 + j] = out[j];
    }
  }
}

__global__ void __launch_bounds__(1024) kl_mean_kernel(Params p) {
  __shared__ float red[1024];
  const int64_t n = p.B * p.Sq;
  float s = 0.0f;
  for (int64_t i = threadIdx.x; i < n; i += 1024) s += p.rows[i];
  red[threadIdx.x] = s;
  __syncthreads();
  for (int off = 512; off >= 1; off >>= 1) {
    if ((int)threadIdx.x < off) red[threadIdx.x] += red[threadIdx.x + off];
    __syncthreads();
  }
  if (threadIdx.x == 0) p.loss[0] = red[0] / (float)n * p.coeff;
}

// ---------------------------------------------------------------------------
// host
// ---------------------------------------------------------------------------
struct Layout {
  size_t mask, tiles, gamma, beta, partial, rows, partial_r, xc, total;
};

// State of dsa_indexer_kl_loss_with_grad: dense v [B, Sq, Sk]; sparse the bitmask,
// the ranks, the row flags and v [B, Sq, K].
struct State {
  size_t v, mask, cpre, flag, total;
};

static size_t align256(size_t x) { return (x + 255) & ~(size_t)255; }

static int64_t chunk_keys(int64_t D) { return D <= 128 ? 128 : 64; }

static State state_layout(int64_t B, int64_t Sq, int64_t Sk, int64_t D, int64_t topk, int sparse) {
  State S{};
  size_t o = 0;
  S.v = o;     o += align256((size_t)(B * Sq * (sparse ? topk : Sk)) * 4);
  if (sparse) {
    S.mask = o;  o += align256((size_t)(B * Sq * ((Sk + 31) / 32)) * 4);
    S.cpre = o;  o += align256((size_t)(B * Sq * ((Sk + chunk_keys(D) - 1) / chunk_keys(D) + 2)) * 4);
    S.flag = o;  o += align256((size_t)(B * Sq) * 4);
  }
  S.total = o;
  return S;
}

// topk > 0: with the sparse state's index scores (its mask lies in the state)
static Layout layout(int64_t B, int64_t Sq, int64_t Sk, int64_t H, int64_t D, int sparse, int64_t topk = 0) {
  const int64_t KC = chunk_keys(D);
  const int64_t W = (Sk + 31) / 32, NC = (Sk + KC - 1) / KC;
  Layout L;
  size_t o = 0;
  L.mask = o;    o += align256(sparse ? (size_t)(B * Sq * W) * 4 : 0);
  L.tiles = o;   o += align256(sparse ? (size_t)(B * ((Sq + 31) / 32) * W) * 128 : 0);
  L.gamma = o;   o += align256((size_t)(B * Sq) * 4);
  L.beta = o;    o += align256((size_t)(B * H * Sq) * 4);
  L.partial = o; o += align256((size_t)(B * NC * Sq) * 4);
  L.rows = o;    o += align256((size_t)(B * Sq) * 4);
  L.partial_r = o; o += align256((size_t)(B * NC * Sq) * 4);
  L.xc = o;      o += align256(sparse ? (size_t)(B * Sq * topk) * 4 : 0);
  L.total = o;
  return L;
}

// (token block, key chunk) pairs of one batch at or below the diagonal.
static int64_t pass_items(const Params &p, int64_t TB, int64_t KC) {
  int64_t n = 0;
  for (int64_t t = 0; t < p.Sq; t += TB) {
    const int64_t lt = (t + TB < p.Sq ? t + TB : p.Sq) - 1;
    n += (lt < p.Sk - 1 ? lt : p.Sk - 1) / KC + 1;
  }
  return n;
}

template <int D, int NW, bool LOSS, bool GRAD, PassForm FORM>
static int launch_pass(const Params &p, int64_t items, hipStream_t st) {
  const auto pass = kl_pass_kernel<D, NW, LOSS, GRAD, FORM>;
  constexpr int lds = PassCfg<D, NW>::BYTES;
  const hipError_t e = hipFuncSetAttribute((const void *)pass, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
  if (e != hipSuccess) return set_error(DSA_ERR_HIP, "kl_pass_kernel: LDS attribute: %s", hipGetErrorString(e));
  hipLaunchKernelGGL(pass, dim3((unsigned)items), dim3(64 * NW), lds, st, p);
  return check_launch("kl_pass_kernel");
}

template <int D, int NWS, int NWP, bool LOSS, bool GRAD>
static int launch_mfma(const Params &p, hipStream_t st) {
  using CS = Cfg<D, NWS>;
  using CP = Cfg<D, NWP>;
  const int64_t NBS = (p.Sq + CS::TB - 1) / CS::TB, NP = (NBS + 1) / 2;
  const dim3 gs((unsigned)(p.B * p.H * NP));
  if (!p.sparse) hipLaunchKernelGGL((kl_attn_stats_kernel<D, NWS, kAllColumns>), gs, dim3(CS::NT), 0, st, p);
  else if (p.tiles == nullptr) hipLaunchKernelGGL((kl_attn_stats_kernel<D, NWS, kRowBits>), gs, dim3(CS::NT), 0, st, p);
  else hipLaunchKernelGGL((kl_attn_stats_kernel<D, NWS, kLaneMasks>), gs, dim3(CS::NT), 0, st, p);
  int rc = check_launch("kl_attn_stats_kernel");
  if (rc) return rc;
  Params q = p;
  q.NI = pass_items(p, CP::TB, CP::KC);
  const int64_t items = (p.B * q.NI + 7) / 8 * 8;
  const int64_t rows = p.Sq < 32 ? p.Sq : 32;  // of a wave
  const bool far = (rows - 1) * p.B * p.H * CP::ROWB + CP::ROWB > (int64_t)0xffffffff;
  if (far) rc = launch_pass<D, NWP, LOSS, GRAD, kFarRows>(q, items, st);
  else if (p.G < p.H) rc = launch_pass<D, NWP, LOSS, GRAD, kSharedKeys>(q, items, st);
  else rc = launch_pass<D, NWP, LOSS, GRAD, kOwnKeys>(q, items, st);
  if (rc) return rc;
  if (p.pc != nullptr) {
    hipLaunchKernelGGL(kl_rows_state_kernel<D>, dim3((unsigned)((p.B * p.Sq + 3) / 4)), dim3(kNT), 0, st, p);
    return check_launch("kl_rows_state_kernel");
  }
  if constexpr (GRAD) {
    hipLaunchKernelGGL(kl_grad_kernel<D>, dim3((unsigned)(p.B * p.Sq)), dim3(kNT), 0, st, p);
    rc = check_launch("kl_grad_kernel");
    if (rc || !LOSS) return rc;
  }
  hipLaunchKernelGGL(kl_rows_kernel<D>, dim3((unsigned)((p.B * p.Sq + kNT - 1) / kNT)), dim3(kNT), 0, st, p);
  return check_launch("kl_rows_kernel");
}

// Checks and Params shared by the loss and its gradient (kernels 1-3).
static int kl_setup(const char *fn, const float *index_scores, const void *topk_indices, int topk_dtype,
                    int64_t topk, const void *query, const void *key, int64_t B, int64_t Sq, int64_t Sk,
                    int64_t H, int64_t G, int64_t D, float softmax_scale, float loss_coeff, int sparse,
                    void *workspace, size_t workspace_bytes, Params &p, bool state = false) {
  DSA_REQUIRE(index_scores && query && key, "%s: null pointer", fn);
  DSA_REQUIRE(B > 0 && Sq > 0 && Sk > 0 && H > 0 && G > 0, "%s: empty shape B=%lld Sq=%lld Sk=%lld H=%lld G=%lld",
              fn, (long long)B, (long long)Sq, (long long)Sk, (long long)H, (long long)G);
  DSA_REQUIRE(H % G == 0, "%s: H=%lld is not a multiple of the key heads G=%lld", fn, (long long)H, (long long)G);
  DSA_REQUIRE(softmax_scale > 0.0f && softmax_scale < INFINITY, "%s: softmax_scale %g must be positive", fn,
              (double)softmax_scale);
  DSA_REQUIRE(D == 64 || D == 128 || D == 192 || D == 256, "%s: head dim %lld not in {64,128,192,256}", fn,
              (long long)D);
  DSA_REQUIRE(B * Sq * Sk < ((int64_t)1 << 29), "%s: B*Sq*Sk=%lld index scores exceed 2 GiB", fn,
              (long long)(B * Sq * Sk));
  DSA_REQUIRE(Sk * B * G * D * 2 < ((int64_t)1 << 31), "%s: key tensor exceeds 2 GiB", fn);
  if (sparse) {
    DSA_REQUIRE(topk_indices && topk > 0, "%s: sparse mode needs top-k indices", fn);
    DSA_REQUIRE(topk_dtype == DSA_DTYPE_I32 || topk_dtype == DSA_DTYPE_I64, "%s: top-k dtype %d is not int32/int64",
                fn, topk_dtype);
    DSA_REQUIRE(Sk <= 32 * kMaxW, "%s: sparse mode supports Sk <= %d (got %lld)", fn, 32 * kMaxW, (long long)Sk);
  }
  const Layout L = layout(B, Sq, Sk, H, D, sparse, state ? topk : 0);
  if (!workspace || workspace_bytes < L.total)
    return set_error(DSA_ERR_WORKSPACE, "%s: workspace %zu bytes < %zu required", fn,
                     workspace ? workspace_bytes : (size_t)0, L.total);
  unsigned char *ws = static_cast<unsigned char *>(workspace);
  p = Params{};
  p.index_scores = index_scores;
  p.topk = topk_indices;
  p.query = static_cast<const unsigned char *>(query);
  p.key = static_cast<const unsigned char *>(key);
  p.mask = reinterpret_cast<uint32_t *>(ws + L.mask);
  p.tiles = reinterpret_cast<uint64_t *>(ws + L.tiles);
  p.gamma = reinterpret_cast<float *>(ws + L.gamma);
  p.beta = reinterpret_cast<float *>(ws + L.beta);
  p.partial = reinterpret_cast<float *>(ws + L.partial);
  p.rows = reinterpret_cast<float *>(ws + L.rows);
  p.partial_r = reinterpret_cast<float *>(ws + L.partial_r);
  p.B = B; p.Sq = Sq; p.Sk = Sk; p.H = H; p.G = G; p.K = sparse ? topk : 0;
  p.W = (Sk + 31) / 32;
  p.KC = (int)chunk_keys(D);
  p.NC = (Sk + p.KC - 1) / p.KC;
  p.xc = reinterpret_cast<float *>(ws + L.xc);
  p.topk_i64 = topk_dtype == DSA_DTYPE_I64;
  p.sparse = sparse ? 1 : 0;
  p.c = softmax_scale * kLog2e;
  p.coeff = loss_coeff;
  return DSA_OK;
}

// Whether the lane masks' launch (3 to 7 us) pays: against the row bitmask they take
// off the statistics 3 us at 134 M scores (b = 2, s = 2048, 16 heads) of 64 or 128
// dims and 9 at 537 M, but -2 to 1 up to 72 M; of 192 or 256 dims, whose registers the
// bitmask's words overfill, 3 to 5 us at 17 M and -3 to 2 up to 8 M.
static bool use_lane_masks(const Params &p, int64_t D) {
  return (double)(p.B * p.H) * (double)p.Sq * (double)p.Sk >= (D <= 128 ? 1e8 : 1.2e7);
}

// The pass with 8 waves a workgroup (256 tokens) or 4 (128).  Four: twice the
// workgroups, which at 64 dims also run two to a compute unit (b = 1, s = 4096, 32
// heads, loss: 191 us, 215 with eight); from 128 dims on the LDS holds one, so half of
// a compute unit's wave slots would stay empty, and they pay only while they all run
// at once (32 heads of 128: s = 2048 125 us, 141 with eight; b = 2 181 and 155).
template <int D, bool LOSS, bool GRAD>
static int launch_by_size(const Params &p, hipStream_t st) {
  if (D == 64 || p.B * pass_items(p, 128, Cfg<D, 4>::KC) <= 256) return launch_mfma<D, 8, 4, LOSS, GRAD>(p, st);
  return launch_mfma<D, 8, D == 64 ? 4 : 8, LOSS, GRAD>(p, st);
}

template <bool LOSS, bool GRAD>
static int kl_launch(Params p, int64_t D, hipStream_t st) {
  hipLaunchKernelGGL(kl_index_stats_kernel, dim3((unsigned)((p.B * p.Sq + 3) / 4)), dim3(kNT), 0, st, p);
  int rc = check_launch("kl_index_stats_kernel");
  if (rc) return rc;
  if (!use_lane_masks(p, D)) p.tiles = nullptr;
  if (p.sparse && p.tiles != nullptr) {
    hipLaunchKernelGGL(kl_mask_tiles_kernel, dim3((unsigned)(p.B * ((p.Sq + 31) / 32)), (unsigned)(p.W < 64 ? (p.W + 7) / 8 : 8)),
                       dim3(kNT), 0, st, p);
    rc = check_launch("kl_mask_tiles_kernel");
    if (rc) return rc;
  }
  switch (D) {
    case 64: return launch_by_size<64, LOSS, GRAD>(p, st);
    case 128: return launch_by_size<128, LOSS, GRAD>(p, st);
    case 192: return launch_by_size<192, LOSS, GRAD>(p, st);
    default:  // (eight q slices and two key chunks would pass 160 KiB)
      return launch_mfma<256, 8, 4, LOSS, GRAD>(p, st);
  }
}

}  // namespace kl
}  // namespace dsa

extern "C" size_t dsa_indexer_kl_loss_workspace_size(int64_t B, int64_t Sq, int64_t Sk, int64_t H, int64_t D,
                                                      int sparse) {
  if (B <= 0 || Sq <= 0 || Sk <= 0 || H <= 0 || D <= 0) return 0;
  return dsa::kl::layout(B, Sq, Sk, H, D, sparse).total;
}

extern "C" int dsa_indexer_kl_loss(const float *index_scores, const void *topk_indices, int topk_dtype,
                                   int64_t topk, const void *query, const void *key, float *loss,
                                   float *row_loss, int64_t B, int64_t Sq, int64_t Sk, int64_t H, int64_t G,
                                   int64_t D, float softmax_scale, float loss_coeff, int sparse,
                                   void *workspace, size_t workspace_bytes, void *stream) {
  using namespace dsa;
  using namespace dsa::kl;
  DSA_REQUIRE(loss, "dsa_indexer_kl_loss: null loss pointer");
  Params p;
  int rc = kl_setup("dsa_indexer_kl_loss", index_scores, topk_indices, topk_dtype, topk, query, key, B, Sq, Sk, H, G,
                    D, softmax_scale, loss_coeff, sparse, workspace, workspace_bytes, p);
  if (rc) return rc;
  if (row_loss) p.rows = row_loss;
  p.loss = loss;
  hipStream_t st = static_cast<hipStream_t>(stream);
  rc = kl_launch<true, false>(p, D, st);
  if (rc) return rc;
  hipLaunchKernelGGL(kl_mean_kernel, dim3(1), dim3(1024), 0, st, p);
  return check_launch("kl_mean_kernel");
}

extern "C" int dsa_indexer_kl_loss_backward(const float *index_scores, const void *topk_indices, int topk_dtype,
                                            int64_t topk, const void *query, const void *key,
                                            const float *grad_loss, float *grad_index_scores, int64_t B, int64_t Sq,
                                            int64_t Sk, int64_t H, int64_t G, int64_t D, float softmax_scale,
                                            float loss_coeff, int sparse, void *workspace, size_t workspace_bytes,
                                            void *stream) {
  using namespace dsa;
  using namespace dsa::kl;
  DSA_REQUIRE(grad_loss && grad_index_scores, "dsa_indexer_kl_loss_backward: null gradient pointer");
  DSA_REQUIRE(grad_index_scores != index_scores, "dsa_indexer_kl_loss_backward: the gradient may not overwrite the scores");
  Params p;
  int rc = kl_setup("dsa_indexer_kl_loss_backward", index_scores, topk_indices, topk_dtype, topk, query, key, B, Sq,
                    Sk, H, G, D, softmax_scale, loss_coeff, sparse, workspace, workspace_bytes, p);
  if (rc) return rc;
  p.grad = grad_index_scores;
  p.grad_loss = grad_loss;
  return kl_launch<false, true>(p, D, static_cast<hipStream_t>(stream));
}

extern "C" size_t dsa_indexer_kl_loss_state_size(int64_t B, int64_t Sq, int64_t Sk, int64_t D, int64_t topk, int sparse) {
  if (B <= 0 || Sq <= 0 || Sk <= 0 || D <= 0 || (sparse && topk <= 0)) return 0;
  return dsa::kl::state_layout(B, Sq, Sk, D, topk, sparse).total;
}

extern "C" size_t dsa_indexer_kl_loss_with_grad_workspace_size(int64_t B, int64_t Sq, int64_t Sk, int64_t H, int64_t D,
                                                                int64_t topk, int sparse) {
  if (B <= 0 || Sq <= 0 || Sk <= 0 || H <= 0 || D <= 0 || (sparse && topk <= 0)) return 0;
  return dsa::kl::layout(B, Sq, Sk, H, D, sparse, sparse ? topk : 0).total;
}

static void kl_bind_state(dsa::kl::Params &p, void *state, const dsa::kl::State &S) {
  unsigned char *s = static_cast<unsigned char *>(state);
  if (!p.sparse) return;
  p.pc = reinterpret_cast<float *>(s + S.v);
  p.mask = reinterpret_cast<uint32_t *>(s + S.mask);
  p.cpre = reinterpret_cast<int32_t *>(s + S.cpre);
  p.flag = reinterpret_cast<float *>(s + S.flag);
}

// loss null: the state alone (the rows' losses are in the workspace then).
static int kl_with_grad(const char *fn, const float *index_scores, const void *topk_indices, int topk_dtype, int64_t topk,
                        const void *query, const void *key, float *loss, float *row_loss, void *state,
                        size_t state_bytes, int64_t B, int64_t Sq, int64_t Sk, int64_t H, int64_t G, int64_t D,
                        float softmax_scale, float loss_coeff, int sparse, void *workspace, size_t workspace_bytes,
                        void *stream) {
  using namespace dsa;
  using namespace dsa::kl;
  Params p;
  int rc = kl_setup(fn, index_scores, topk_indices, topk_dtype, topk, query, key, B, Sq, Sk, H, G, D, softmax_scale,
                    loss_coeff, sparse, workspace, workspace_bytes, p, true);
  if (rc) return rc;
  const State S = state_layout(B, Sq, Sk, D, topk, sparse);
  if (!state || state_bytes < S.total)
    return set_error(DSA_ERR_WORKSPACE, "%s: state %zu bytes < %zu required", fn, state ? state_bytes : (size_t)0, S.total);
  kl_bind_state(p, state, S);
  if (!p.sparse) p.grad = static_cast<float *>(state);
  if (row_loss) p.rows = row_loss;
  p.loss = loss;
  hipStream_t st = static_cast<hipStream_t>(stream);
  rc = kl_launch<true, true>(p, D, st);
  if (rc || !loss) return rc;
  hipLaunchKernelGGL(kl_mean_kernel, dim3(1), dim3(1024), 0, st, p);
  return check_launch("kl_mean_kernel");
}

extern "C" int dsa_indexer_kl_loss_with_grad(const float *index_scores, const void *topk_indices, int topk_dtype,
                                             int64_t topk, const void *query, const void *key, float *loss,
                                             float *row_loss, void *state, size_t state_bytes, int64_t B, int64_t Sq,
                                             int64_t Sk, int64_t H, int64_t G, int64_t D, float softmax_scale,
                                             float loss_coeff, int sparse, void *workspace, size_t workspace_bytes,
                                             void *stream) {
  using namespace dsa;
  DSA_REQUIRE(loss, "dsa_indexer_kl_loss_with_grad: null loss pointer");
  return kl_with_grad("dsa_indexer_kl_loss_with_grad", index_scores, topk_indices, topk_dtype, topk, query, key, loss,
                      row_loss, state, state_bytes, B, Sq, Sk, H, G, D, softmax_scale, loss_coeff, sparse, workspace,
                      workspace_bytes, stream);
}

extern "C" int dsa_indexer_kl_loss_grad_state(const float *index_scores, const void *topk_indices, int topk_dtype,
                                              int64_t topk, const void *query, const void *key, void *state,
                                              size_t state_bytes, int64_t B, int64_t Sq, int64_t Sk, int64_t H,
                                              int64_t G, int64_t D, float softmax_scale, float loss_coeff, int sparse,
                                              void *workspace, size_t workspace_bytes, void *stream) {
  return kl_with_grad("dsa_indexer_kl_loss_grad_state", index_scores, topk_indices, topk_dtype, topk, query, key, nullptr,
                      nullptr, state, state_bytes, B, Sq, Sk, H, G, D, softmax_scale, loss_coeff, sparse, workspace,
                      workspace_bytes, stream);
}

extern "C" int dsa_indexer_kl_loss_grad_apply(const void *state, size_t state_bytes, const float *grad_loss,
                                              float *grad_index_scores, int64_t B, int64_t Sq, int64_t Sk, int64_t D,
                                              int64_t topk, float loss_coeff, int sparse, void *stream) {
  using namespace dsa;
  using namespace dsa::kl;
  const char *fn = "dsa_indexer_kl_loss_grad_apply";
  DSA_REQUIRE(grad_loss && grad_index_scores, "%s: null gradient pointer", fn);
  DSA_REQUIRE(B > 0 && Sq > 0 && Sk > 0 && D > 0 && (!sparse || topk > 0), "%s: empty shape", fn);
  DSA_REQUIRE(B * Sq * Sk < ((int64_t)1 << 29), "%s: B*Sq*Sk=%lld index scores exceed 2 GiB", fn, (long long)(B * Sq * Sk));
  const State S = state_layout(B, Sq, Sk, D, topk, sparse);
  if (!state || state_bytes < S.total)
    return set_error(DSA_ERR_WORKSPACE, "%s: state %zu bytes < %zu required", fn, state ? state_bytes : (size_t)0, S.total);
  hipStream_t st = static_cast<hipStream_t>(stream);
  if (!sparse) {
    const int64_t n = B * Sq * Sk, blocks = (n / 4 + kNT) / kNT;
    hipLaunchKernelGGL(kl_scale_kernel, dim3((unsigned)(blocks < 16384 ? blocks : 16384)), dim3(kNT), 0, st,
                       static_cast<const float *>(state), grad_loss, grad_index_scores, n, loss_coeff, (float)(B * Sq));
    return check_launch("kl_scale_kernel");
  }
  Params p{};
  p.sparse = 1;
  kl_bind_state(p, const_cast<void *>(state), S);
  p.grad = grad_index_scores;
  p.grad_loss = grad_loss;
  p.coeff = loss_coeff;
  p.B = B; p.Sq = Sq; p.Sk = Sk; p.K = topk;
  p.W = (Sk + 31) / 32;
  p.KC = (int)chunk_keys(D);
  p.NC = (Sk + p.KC - 1) / p.KC;
  hipLaunchKernelGGL(kl_expand_kernel, dim3((unsigned)(B * Sq)), dim3(kNT), 0, st, p);
  return check_launch("kl_expand_kernel");
}
