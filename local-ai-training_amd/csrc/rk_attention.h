// Pieces shared by the attention kernels (forward and backward): staged [rows][D] bf16 tiles
// filled by LDS-DMA, the two fragment reads of them, and the owned rows of a wavefront.
//
// Staged tiles are read both by rows (16 bytes per lane) and transposed (8 bytes per lane). The
// 16-byte segments of a row are XOR-swizzled (`seg_swizzle`) so that both reads are free of
// bank conflicts; the swizzle is applied to the DMA's source addresses.
#pragma once

#include "rk_common.h"
#include "rk_lds_dma.h"

namespace rk {

typedef float v16f_a __attribute__((ext_vector_type(16)));
typedef __bf16 v8bf_a __attribute__((ext_vector_type(8)));
typedef __bf16 v2bf_a __attribute__((ext_vector_type(2)));
typedef short v4s_a __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) v4s_a* lds_v4s_a;

constexpr int kAttnRows = 128;    // owned rows (queries or keys) per workgroup, 32 per wavefront
constexpr int kAttnStages = 2;    // a step's products cover the next step's loads

template <int D, int R>
struct AttnTile {
  static constexpr int ROWS = R;
  static constexpr int ROWB = 2 * D;             // bytes per row
  static constexpr int BYTES = ROWS * ROWB;      // one operand's tile
  static constexpr int CHUNKS = BYTES / 1024 / 4;  // 1 KB DMA pieces per wavefront and operand
};

// Physical 16-byte slot of segment `seg` of row `row`: seg ^ f(row). Row reads take one
// segment of 16 consecutive rows (f takes all values over them, with the row's parity in the
// bank for 128-byte rows); transposed reads take 4 adjacent segments of 4 consecutive rows
// (f's high bits differ between them).
template <int D>
__device__ __forceinline__ int seg_swizzle(int row) {
  if constexpr (D == 128) return ((row & 3) << 2) | ((row >> 2) & 3);
  else return (((row >> 1) & 1) << 2) | ((row >> 2) & 3);
}

__device__ __forceinline__ v8bf_a frag_of(uint4 r) { return __builtin_bit_cast(v8bf_a, r); }

__device__ __forceinline__ uint32_t bf16_pair(float lo, float hi) {
  const v2bf_a v = {static_cast<__bf16>(lo), static_cast<__bf16>(hi)};
  return __builtin_bit_cast(uint32_t, v);
}

// Row operand: row `row0 + lane % 32` of a staged tile, features 16 s + 8 (lane / 32) .. + 7.
template <int D>
__device__ __forceinline__ v8bf_a row_frag(const uint8_t* tile, int row0, int s, int lane) {
  const int r = lane & 31, seg = 2 * s + (lane >> 5);
  return frag_of(*reinterpret_cast<const uint4*>(tile + (row0 + r) * (2 * D) +
                                                 16 * (seg ^ seg_swizzle<D>(r))));
}

// Transposed operand: feature 32 dt + lane % 32, rows row0 + {4 h .. + 3, 8 + 4 h .. + 3}.
template <int D>
__device__ __forceinline__ v8bf_a col_frag(const uint8_t* tile, int row0, int dt, int lane) {
  const int g = lane >> 4, sl = lane & 15;
  const int r = 4 * (g >> 1) + (sl >> 2);
  const int seg = 4 * dt + 2 * (g & 1) + ((sl & 3) >> 1);
  v4s_a half[2];
#pragma unroll
  for (int u = 0; u < 2; ++u)
    half[u] = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
        (lds_v4s_a)(tile + (row0 + r + 8 * u) * (2 * D) +
                    16 * (seg ^ seg_swizzle<D>(r + 8 * u)) + 8 * (sl & 1)));
  v8bf_a f;
  __builtin_memcpy(&f, half, sizeof(f));
  return f;
}

// The DMA of one operand's tiles: this wavefront's share of rows row0 .. row0 + ROWS - 1 of a
// head, rows past the descriptor's end read zeros.
template <int D, int R>
struct TileDma {
  __amdgpu_buffer_rsrc_t buf;
  int voff[AttnTile<D, R>::CHUNKS];
  int row_bytes;

  __device__ __forceinline__ TileDma(const uint16_t* base, int64_t stride, int64_t S, int wave,
                                     int lane)
      : buf(make_buffer(base, ((S - 1) * stride + D) * 2)), row_bytes(static_cast<int>(stride) * 2) {
    constexpr int PER = 1024 / (2 * D), SEGS = D / 8;  // rows per DMA, segments per row
#pragma unroll
    for (int c = 0; c < AttnTile<D, R>::CHUNKS; ++c) {
      const int row = (wave * AttnTile<D, R>::CHUNKS + c) * PER + lane / SEGS;
      voff[c] = row * row_bytes + 16 * ((lane % SEGS) ^ seg_swizzle<D>(row));
    }
  }
  __device__ __forceinline__ void issue(uint32_t lds, int row0, int wave) const {
#pragma unroll
    for (int c = 0; c < AttnTile<D, R>::CHUNKS; ++c)
      dma16(buf, lds + 1024 * (wave * AttnTile<D, R>::CHUNKS + c), voff[c], row0 * row_bytes);
  }
};

// The owned row's features 16 s + 8 h .. + 7 for every s: the second operand, in registers.
template <int D>
__device__ __forceinline__ void load_owned(v8bf_a (&f)[D / 16], const uint16_t* base,
                                           int64_t stride, int64_t S, int row, int h) {
  const __amdgpu_buffer_rsrc_t buf = make_buffer(base, ((S - 1) * stride + D) * 2);
  const int rb = static_cast<int>(stride) * 2;
#pragma unroll
  for (int s = 0; s < D / 16; ++s)
    f[s] = frag_of(__builtin_bit_cast(
        uint4, __builtin_amdgcn_raw_buffer_load_b128(buf, row * rb + 32 * s + 16 * h, 0, 0)));
}

// acc[dt][e] = X[row][32 dt + 8 (e / 4) + 4 h + e % 4]: stores factor * acc as bf16.
template <int D>
__device__ __forceinline__ void store_owned(uint16_t* row, const v16f_a (&acc)[D / 32],
                                            float factor, int h) {
#pragma unroll
  for (int dt = 0; dt < D / 32; ++dt)
#pragma unroll
    for (int r = 0; r < 4; ++r)
      *reinterpret_cast<uint2*>(row + 32 * dt + 8 * r + 4 * h) =
          make_uint2(bf16_pair(acc[dt][4 * r] * factor, acc[dt][4 * r + 1] * factor),
                     bf16_pair(acc[dt][4 * r + 2] * factor, acc[dt][4 * r + 3] * factor));
}

__device__ __forceinline__ void pack16(uint4 (&f)[2], const float (&p)[16]) {
#pragma unroll
  for (int s2 = 0; s2 < 2; ++s2)
    f[s2] = make_uint4(bf16_pair(p[8 * s2], p[8 * s2 + 1]), bf16_pair(p[8 * s2 + 2], p[8 * s2 + 3]),
                       bf16_pair(p[8 * s2 + 4], p[8 * s2 + 5]),
                       bf16_pair(p[8 * s2 + 6], p[8 * s2 + 7]));
}

}  // namespace rk
