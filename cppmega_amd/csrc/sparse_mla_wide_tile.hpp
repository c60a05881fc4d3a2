// Tile helpers shared by the wide-head (d_qk = 576) forward and backward: the
// register-staged gather of one block's kv rows, the exchange of partial score
// tiles, and the row tiles filled by LDS-DMA loads.
#pragma once

#include "dsa_common.hpp"
#include "sparse_mla_gather.hpp"

namespace dsa {

template <int D_QK, int D_V, bool FP8, int NTHR_ = 256>
struct WideCfg {
  static constexpr int NTHR = NTHR_;               // threads that gather a block
  static constexpr int ELT = FP8 ? 1 : 2;          // bytes per element in HBM
  static constexpr int ROWB = D_QK * ELT;          // bytes per kv row
  static constexpr int NCH = ROWB / 16;            // 16-byte chunks per row
  static constexpr int NCH_V = D_V * ELT / 16;     // chunks of the V prefix
  static constexpr int UNITS = 32 * NCH;           // (row, chunk) units per block
  static constexpr int UPT = (UNITS + NTHR - 1) / NTHR;  // units per thread
  static constexpr int KL_STRIDE = ROWB + 32;      // padded LDS row (conflict-free transposed reads)
  static constexpr int KD_STRIDE = D_V * 2 + 32;   // e4m3: dequantised V rows (bf16)
  static constexpr int KSTEPS = D_QK / 16;         // 32x32x16 k-steps over d_qk
  static constexpr int KQ = KSTEPS / 4;            // S k-steps per wave
  static constexpr int DT = D_V / 32;              // 32-column tiles of d_v
  static constexpr int DTW = (DT + 3) / 4;         // O^T tiles per wave (tile t = w + 4 q, t < DT)
  static_assert(ROWB % 16 == 0 && (D_V * ELT) % 16 == 0, "rows must be whole 16-byte chunks");
  static_assert(KSTEPS % 4 == 0 && D_V % 32 == 0 && D_V <= D_QK, "head dims must split over four waves");
  struct Regs {
    i32x4 v[UPT];
    float sc[UPT];
    uint32_t valid;  // bit i: unit i is a real (unmasked) slot's chunk
  };
};

// Issue the loads of one block's 32 rows: thread t takes units t + NTHR i,
// unit u = chunk u % NCH of row u / NCH.  my_idx is the kv row of slot
// (lane & 31) of this wave (-1: masked).
// kv_scale_b holds one scale per row (sc_pitch 1) or, MX, one per 32-channel
// block of every row (sc_pitch floats apart): a unit loads its own block's.
// UNCOND (the backward): the loads are unconditional, a unit past the block
// (or a masked slot) reading row 0, which wide_store drops, so that every wave
// issues the same loads on every block.
template <class C, bool FP8, bool MX = false, bool UNCOND = false>
__device__ __forceinline__ void wide_issue(typename C::Regs &rg, const unsigned char *kv_b, const float *kv_scale_b,
                                           int my_idx, uint32_t row_pitch, uint32_t sc_pitch = 1u) {
  const int t = threadIdx.x;
  uint32_t valid = 0;
#pragma unroll
  for (int i = 0; i < C::UPT; ++i) {
    const int u = t + C::NTHR * i;
    const int row = (u / C::NCH) & 31;
    const int c = u % C::NCH;
    const int ri = __shfl(my_idx, row, 64);
    const bool exists = (i + 1 < C::UPT) || u < C::UNITS;
    const bool ok = ri >= 0 && exists;
    const uint32_t r = ok ? (uint32_t)ri : 0u;
    if constexpr (UNCOND) {
      rg.v[i] = ld_global_16(kv_b + r * row_pitch + c * 16);
      if constexpr (FP8) rg.sc[i] = kv_scale_b[r * sc_pitch + (MX ? (uint32_t)(c >> 1) : 0u)];
    } else {
      rg.v[i] = i32x4{0, 0, 0, 0};
      if (exists) rg.v[i] = ld_global_16(kv_b + r * row_pitch + c * 16);
      if constexpr (FP8) rg.sc[i] = exists ? kv_scale_b[r * sc_pitch + (MX ? (uint32_t)(c >> 1) : 0u)] : 0.0f;
    }
    valid |= (ok ? 1u : 0u) << i;
  }
  rg.valid = valid;
}

// Store the staged rows: raw bytes row-major into Kl (masked slots zero); for
// e4m3 also the first NCH_D chunks dequantised to bf16 (value * kv_scale, RNE)
// into Kd (row stride KD_STRIDE) and the per-slot scales into Ksc (MX: the
// per-(slot, block) scales, block-major Ksc[block * 32 + slot]).
template <class C, bool FP8, int NCH_D = C::NCH_V, int KD_STRIDE = C::KD_STRIDE, bool MX = false>
__device__ __forceinline__ void wide_store(const typename C::Regs &rg, unsigned char *Kl, unsigned char *Kd,
                                           float *Ksc) {
  const int t = threadIdx.x;
#pragma unroll
  for (int i = 0; i < C::UPT; ++i) {
    const int u = t + C::NTHR * i;
    if ((i + 1 < C::UPT) || u < C::UNITS) {
      const int row = u / C::NCH, c = u % C::NCH;
      const bool ok = (rg.valid >> i) & 1u;
      const i32x4 v = ok ? rg.v[i] : i32x4{0, 0, 0, 0};
      *reinterpret_cast<i32x4 *>(Kl + row * C::KL_STRIDE + c * 16) = v;
      if constexpr (FP8) {
        const float s = ok ? rg.sc[i] : 0.0f;
        if (c < NCH_D) {
          uint32_t wd[8];
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            const f32x2 v2 = e4m3x2_to_f32((uint32_t)v[e >> 1], (e & 1) != 0);
            wd[e] = pack_bf16x2(v2[0] * s, v2[1] * s);
          }
          unsigned char *dst = Kd + row * KD_STRIDE + c * 32;
          *reinterpret_cast<i32x4 *>(dst) = i32x4{(int)wd[0], (int)wd[1], (int)wd[2], (int)wd[3]};
          *reinterpret_cast<i32x4 *>(dst + 16) = i32x4{(int)wd[4], (int)wd[5], (int)wd[6], (int)wd[7]};
        }
        if constexpr (MX) {
          if ((c & 1) == 0) Ksc[(c >> 1) * 32 + row] = s;
        } else if (c == 0) {
          Ksc[row] = s;
        }
      }
    }
  }
}

// Sum of the four waves' partial 32x32 fp32 tiles (stored lane-linear per wave:
// Sp[w][q4][lane][4]) in wave order: the same bits in every wave.
__device__ __forceinline__ void sum_partials(const float *Sp, int stride_w, float (&s)[16]) {
  const int lane = lane_id();
#pragma unroll
  for (int q4 = 0; q4 < 4; ++q4) {
    const f32x4 v0 = *reinterpret_cast<const f32x4 *>(Sp + 0 * stride_w + (q4 * 64 + lane) * 4);
    const f32x4 v1 = *reinterpret_cast<const f32x4 *>(Sp + 1 * stride_w + (q4 * 64 + lane) * 4);
    const f32x4 v2 = *reinterpret_cast<const f32x4 *>(Sp + 2 * stride_w + (q4 * 64 + lane) * 4);
    const f32x4 v3 = *reinterpret_cast<const f32x4 *>(Sp + 3 * stride_w + (q4 * 64 + lane) * 4);
#pragma unroll
    for (int j = 0; j < 4; ++j) s[4 * q4 + j] = ((v0[j] + v1[j]) + v2[j]) + v3[j];
    __builtin_amdgcn_sched_barrier(0);  // bound the loads in flight (register pressure)
  }
}

__device__ __forceinline__ void put_partial(float *dst, const f32x16 &acc) {
  const int lane = lane_id();
#pragma unroll
  for (int q4 = 0; q4 < 4; ++q4)
    *reinterpret_cast<f32x4 *>(dst + (q4 * 64 + lane) * 4) =
        f32x4{acc[4 * q4], acc[4 * q4 + 1], acc[4 * q4 + 2], acc[4 * q4 + 3]};
}


// ---------------------------------------------------------------------------
// Row tiles filled by LDS-DMA loads (bf16 rows)
// ---------------------------------------------------------------------------
// 32 gathered rows of D_QK bf16, written straight into LDS by
// buffer_load_dwordx4 ... lds: no staging registers and no LDS write
// instructions.  One such load fills 1 KiB of consecutive LDS from 64 lanes'
// own addresses: here 8 rows x 128 bytes.  The tile is stored by panels of 128
// bytes of d (64 columns), 32 rows each: chunk c (16 bytes) of row r at byte
//   (c >> 3) * 4096 + r * 128 + ((c & 7) ^ row_swz(r)) * 16,
// so a wave that fetches an 8-row group needs one source address per lane for
// all of its panels (the panel is a scalar offset), and neither the rows' order
// nor a lane's chunk changes between panels.  Rows are 128 bytes apart on the
// 256 bytes of banks; the swizzle permutes the eight chunks such that
//   * 16 consecutive rows read at one chunk (MFMA operand, lane = row) and
//   * rows {8g .. 8g + 3} (or + 4 .. + 7) of two neighbouring g, read at one
//     chunk pair (a transposed read)
// fall on distinct banks.
template <int D_QK, int NW_>
struct DmaTile {
  static constexpr int NW = NW_;                       // waves that fill it (w < NW)
  static constexpr int ROWB = D_QK * 2;
  static constexpr int BYTES = 32 * ROWB;
  static constexpr int PANELS = ROWB / 128, PANEL = 4096;
  static constexpr int RG = 4 / NW;                    // 8-row groups per wave: w, w + NW, ...
  static_assert(ROWB % 128 == 0 && 4 % NW == 0, "whole panels, whole row groups");
};

__device__ __forceinline__ int row_swz(int row) {
  const int x = (row >> 1) & 7;
  return ((x & 1) << 1) | (x & 4) | ((x >> 1) & 1);
}
// Byte of chunk c of row r within a tile (c < 8: an offset that (c >> 3) panels are added to).
__device__ __forceinline__ int tile_byte(int r, int c) { return r * 128 + ((c ^ row_swz(r)) * 16); }

// The lane index as a value the compiler cannot trace: addresses derived from
// it are formed where they are used (a few VALU operations) instead of being
// kept in registers across the block loop, where accumulators and operands leave none to spare.
__device__ __forceinline__ int lane_here() {
  int l = lane_id();
  asm volatile("" : "+v"(l));
  return l;
}

// Fetch 32 rows at byte offsets my_off (held by lane `row`; kMaskedOff: the row
// reads as zeros) into the tile at LDS byte address lds.
template <class T>
__device__ __forceinline__ void dma_tile_issue(uint32_t lds, i32x4 rs, uint32_t my_off, int w) {
  const int lane = lane_here();
#pragma unroll
  for (int i = 0; i < T::RG; ++i) {
    const int rg = w + T::NW * i, row = 8 * rg + (lane >> 3);
    const uint32_t src = (uint32_t)__shfl((int)my_off, row, 64) + (uint32_t)(((lane & 7) ^ row_swz(row)) * 16);
#pragma unroll
    for (int pn = 0; pn < T::PANELS; ++pn) lds_dma_16(lds + (uint32_t)(pn * T::PANEL + rg * 1024), src, rs, (uint32_t)(pn * 128));
  }
}

}  // namespace dsa
