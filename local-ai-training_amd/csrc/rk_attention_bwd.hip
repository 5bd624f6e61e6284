// Causal self-attention backward of the training step (gfx950), the backward of
// rk_attention_forward (model.py:117-123): from bf16 q, k, v, o, do [B, H, S, D] and the
// forward's log-sum-exp,
//   p_ij = exp(scale q_i . k_j - lse_i)   (j <= i, else 0),     delta_i = do_i . o_i,
//   ds_ij = p_ij (do_i . v_j - delta_i),
//   dq_i = scale sum_j ds_ij k_j,  dk_j = scale sum_i ds_ij q_i,  dv_j = sum_i p_ij do_i.
// Products of bf16 operands summed in float32 (v_mfma_f32_32x32x16_bf16); p and ds enter the
// second products rounded to bf16; scores, exponentials and delta are float32.
//
// Two launches, every output element summed by one wavefront in a fixed order (results
// repeat; no float atomics, no float32 dq buffer to clear and convert):
//  * attn_bwd_dq_kernel: a workgroup owns 128 queries (4 wavefronts x 32) and walks the key
//    tiles up to its diagonal. It also forms delta of its queries and leaves (-lse / scale,
//    -delta) per query in `work` for the second launch.
//  * attn_bwd_dkv_kernel: a workgroup owns 128 keys and walks the query tiles from its
//    diagonal down.
// The scores are computed twice (7 products instead of 5): cheaper than adding float32 dq
// tiles of every key block into memory.
//
// Both use the forward's layout: the product whose result is exponentiated puts the owned
// rows in the MFMA's columns, so a lane holds one owned row (lane % 32) against 16 rows of
// each 32-row tile, and the 8 values of a 16-row half are the next product's second operand
// once its contraction slots stand for rows {4 h .. + 3, 8 + 4 h .. + 3} (h = lane / 32); the
// first operand of that product is read transposed from the staged tile (ds_read_b64_tr_b16)
// with the same slot order. The score and do . v accumulators start at -lse / scale and
// -delta, so neither needs a subtraction per element.
//
// Staged tiles ([rows][D] bf16, row-major, LDS-DMA, three stages, one barrier per step) are
// read both by rows (16 bytes per lane) and transposed (8 bytes per lane). The 16-byte
// segments of a row are XOR-swizzled (`seg_swizzle`) so that both reads are free of bank
// conflicts; the swizzle is applied to the DMA's source addresses.
#include "rk_common.h"
#include "rk_lds_dma.h"

namespace rk {

typedef float v16f_b __attribute__((ext_vector_type(16)));
typedef __bf16 v8bf_b __attribute__((ext_vector_type(8)));
typedef __bf16 v2bf_b __attribute__((ext_vector_type(2)));
typedef short v4s_b __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) v4s_b* lds_v4s_b;

constexpr int kBwdRows = 128;  // owned rows per workgroup
constexpr int kBwdStages = 3;

struct AttnBwdArgs {
  const uint16_t* q;
  const uint16_t* k;
  const uint16_t* v;
  const uint16_t* o;
  const uint16_t* g;  // gradient of o
  int64_t sqb, sqh, sqs, skb, skh, sks, svb, svh, svs, sob, soh, sos, sgb, sgh, sgs;
  const float* lse;  // [B, H, S]
  float* work;       // [2][B * H][Sp]: -lse / scale, -delta (zeros past S)
  uint16_t* dq;
  uint16_t* dk;
  uint16_t* dv;
  int64_t sxb, sxh, sxs;  // strides of dq, dk and dv
  int64_t BH, H, S, Sp;
  float scale, scale_log2, inv_scale;
};

// Staged rows per step: 32 KB of tile pairs in three stages either way.
template <int D>
struct BwdTile {
  static constexpr int ROWS = D == 128 ? 32 : 64;
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

__device__ __forceinline__ v8bf_b frag_of(uint4 r) { return __builtin_bit_cast(v8bf_b, r); }

__device__ __forceinline__ uint32_t bf16_pair(float lo, float hi) {
  const v2bf_b v = {static_cast<__bf16>(lo), static_cast<__bf16>(hi)};
  return __builtin_bit_cast(uint32_t, v);
}

// Row operand: row `row0 + lane % 32` of a staged tile, features 16 s + 8 (lane / 32) .. + 7.
template <int D>
__device__ __forceinline__ v8bf_b row_frag(const uint8_t* tile, int row0, int s, int lane) {
  const int r = lane & 31, seg = 2 * s + (lane >> 5);
  return frag_of(*reinterpret_cast<const uint4*>(tile + (row0 + r) * BwdTile<D>::ROWB +
                                                 16 * (seg ^ seg_swizzle<D>(r))));
}

// Transposed operand: feature 32 dt + lane % 32, rows row0 + {4 h .. + 3, 8 + 4 h .. + 3}.
template <int D>
__device__ __forceinline__ v8bf_b col_frag(const uint8_t* tile, int row0, int dt, int lane) {
  const int g = lane >> 4, sl = lane & 15;
  const int r = 4 * (g >> 1) + (sl >> 2);
  const int seg = 4 * dt + 2 * (g & 1) + ((sl & 3) >> 1);
  v4s_b half[2];
#pragma unroll
  for (int u = 0; u < 2; ++u)
    half[u] = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
        (lds_v4s_b)(tile + (row0 + r + 8 * u) * BwdTile<D>::ROWB +
                    16 * (seg ^ seg_swizzle<D>(r + 8 * u)) + 8 * (sl & 1)));
  v8bf_b f;
  __builtin_memcpy(&f, half, sizeof(f));
  return f;
}

// The DMA of one operand's tiles: this wavefront's share of rows row0 .. row0 + ROWS - 1 of a
// head, rows past the descriptor's end read zeros.
template <int D>
struct TileDma {
  __amdgpu_buffer_rsrc_t buf;
  int voff[BwdTile<D>::CHUNKS];
  int row_bytes;

  __device__ __forceinline__ TileDma(const uint16_t* base, int64_t stride, int64_t S, int wave,
                                     int lane)
      : buf(make_buffer(base, ((S - 1) * stride + D) * 2)), row_bytes(static_cast<int>(stride) * 2) {
    constexpr int PER = 1024 / BwdTile<D>::ROWB, SEGS = D / 8;  // rows per DMA, segments per row
#pragma unroll
    for (int c = 0; c < BwdTile<D>::CHUNKS; ++c) {
      const int row = (wave * BwdTile<D>::CHUNKS + c) * PER + lane / SEGS;
      voff[c] = row * row_bytes + 16 * ((lane % SEGS) ^ seg_swizzle<D>(row));
    }
  }
  __device__ __forceinline__ void issue(uint32_t lds, int row0, int wave) const {
#pragma unroll
    for (int c = 0; c < BwdTile<D>::CHUNKS; ++c)
      dma16(buf, lds + 1024 * (wave * BwdTile<D>::CHUNKS + c), voff[c], row0 * row_bytes);
  }
};

// The owned row's features 16 s + 8 h .. + 7 for every s: the second operand, in registers.
template <int D>
__device__ __forceinline__ void load_owned(v8bf_b (&f)[D / 16], const uint16_t* base,
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
__device__ __forceinline__ void store_owned(uint16_t* row, const v16f_b (&acc)[D / 32],
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

template <int D>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, D == 128 ? 2 : 4)))
void attn_bwd_dq_kernel(AttnBwdArgs a) {
  using T = BwdTile<D>;
  __shared__ __attribute__((aligned(1024))) uint8_t smem[kBwdStages * 2 * T::BYTES];
  const uint32_t lds0 = lds_address(smem);
  const int S = static_cast<int>(a.S);
  const int nqb = (S + kBwdRows - 1) / kBwdRows;
  const int qb = nqb - 1 - static_cast<int>(blockIdx.y);  // longest causal rows first
  const int64_t bh = blockIdx.x, b = bh / a.H, hd = bh - b * a.H;
  const int tid = threadIdx.x, lane = tid & 63, h = lane >> 5, l32 = lane & 31;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int qw0 = qb * kBwdRows + 32 * wave, qi = qw0 + l32;

  const uint16_t* gbase = a.g + b * a.sgb + hd * a.sgh;
  v8bf_b qf[D / 16], gf[D / 16];
  load_owned<D>(qf, a.q + b * a.sqb + hd * a.sqh, a.sqs, S, qi, h);
  load_owned<D>(gf, gbase, a.sgs, S, qi, h);

  // delta of this lane's query: half of the features here, the other half in lane ^ 32
  float dot = 0.0f;
  {
    v8bf_b of[D / 16];
    load_owned<D>(of, a.o + b * a.sob + hd * a.soh, a.sos, S, qi, h);
#pragma unroll
    for (int s = 0; s < D / 16; ++s)
#pragma unroll
      for (int e = 0; e < 8; ++e)
        dot = dot + static_cast<float>(gf[s][e]) * static_cast<float>(of[s][e]);
  }
  dot = dot + __shfl_xor(dot, 32, kWave);
  const bool valid = qi < S;
  const float nlse = valid ? a.lse[bh * a.S + qi] * -a.inv_scale : 0.0f;
  const float ndelta = valid ? -dot : 0.0f;
  if (h == 0) {
    a.work[bh * a.Sp + qi] = nlse;
    a.work[(a.BH + bh) * a.Sp + qi] = ndelta;
  }

  const TileDma<D> kd(a.k + b * a.skb + hd * a.skh, a.sks, S, wave, lane);
  const TileDma<D> vd(a.v + b * a.svb + hd * a.svh, a.svs, S, wave, lane);
  const int last = qb * kBwdRows + kBwdRows < S ? qb * kBwdRows + kBwdRows : S;
  const int steps = (last + T::ROWS - 1) / T::ROWS;
  auto issue = [&](int step) {
    const uint32_t st = lds0 + (step % kBwdStages) * 2 * T::BYTES;
    kd.issue(st, step * T::ROWS, wave);
    vd.issue(st + T::BYTES, step * T::ROWS, wave);
  };

  v16f_b dq[D / 32];
#pragma unroll
  for (int dt = 0; dt < D / 32; ++dt) dq[dt] = v16f_b{};
  issue(0);
  if (steps > 1) issue(1);
  for (int step = 0; step < steps; ++step) {
    if (step + 1 < steps) dma_wait_barrier<2 * T::CHUNKS>();
    else dma_wait_barrier<0>();
    if (step + 2 < steps) issue(step + 2);
    const uint8_t* kt = smem + (step % kBwdStages) * 2 * T::BYTES;
    const uint8_t* vt = kt + T::BYTES;
#pragma unroll
    for (int sub = 0; sub < T::ROWS / 32; ++sub) {
      const int key0 = step * T::ROWS + 32 * sub;
      if (key0 > qw0 || qw0 >= S) continue;  // above this wavefront's diagonal
      v16f_b st, dp;
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        st[e] = nlse;
        dp[e] = ndelta;
      }
#pragma unroll
      for (int s = 0; s < D / 16; ++s)
        st = __builtin_amdgcn_mfma_f32_32x32x16_bf16(row_frag<D>(kt, 32 * sub, s, lane), qf[s], st,
                                                     0, 0, 0);
#pragma unroll
      for (int s = 0; s < D / 16; ++s)
        dp = __builtin_amdgcn_mfma_f32_32x32x16_bf16(row_frag<D>(vt, 32 * sub, s, lane), gf[s], dp,
                                                     0, 0, 0);
      float ds[16];
      const bool diag = key0 == qw0;
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        float p = __builtin_amdgcn_exp2f(st[e] * a.scale_log2);
        if (diag && 8 * (e / 4) + 4 * h + (e % 4) > l32) p = 0.0f;  // key past the query
        ds[e] = p * dp[e];
      }
      uint4 dsf[2];
      pack16(dsf, ds);
#pragma unroll
      for (int s2 = 0; s2 < 2; ++s2)
#pragma unroll
        for (int dt = 0; dt < D / 32; ++dt)
          dq[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
              col_frag<D>(kt, 32 * sub + 16 * s2, dt, lane), frag_of(dsf[s2]), dq[dt], 0, 0, 0);
    }
  }
  if (valid)
    store_owned<D>(a.dq + b * a.sxb + hd * a.sxh + static_cast<int64_t>(qi) * a.sxs, dq, a.scale, h);
}

template <int D>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, D == 128 ? 2 : 4)))
void attn_bwd_dkv_kernel(AttnBwdArgs a) {
  using T = BwdTile<D>;
  constexpr int ROWF = 2 * T::ROWS;  // staged floats per step: -lse / scale, then -delta
  constexpr int STAGE = 2 * T::BYTES + 512;
  __shared__ __attribute__((aligned(1024))) uint8_t smem[kBwdStages * STAGE];
  const uint32_t lds0 = lds_address(smem);
  const int S = static_cast<int>(a.S);
  const int64_t bh = blockIdx.x, b = bh / a.H, hd = bh - b * a.H;
  const int k0 = static_cast<int>(blockIdx.y) * kBwdRows;  // the first keys have the longest walk
  const int tid = threadIdx.x, lane = tid & 63, h = lane >> 5, l32 = lane & 31;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int kw0 = k0 + 32 * wave, kj = kw0 + l32;

  v8bf_b kf[D / 16], vf[D / 16];
  load_owned<D>(kf, a.k + b * a.skb + hd * a.skh, a.sks, S, kj, h);
  load_owned<D>(vf, a.v + b * a.svb + hd * a.svh, a.svs, S, kj, h);

  const TileDma<D> qd(a.q + b * a.sqb + hd * a.sqh, a.sqs, S, wave, lane);
  const TileDma<D> gd(a.g + b * a.sgb + hd * a.sgh, a.sgs, S, wave, lane);
  // row statistics: one 4-byte DMA per wavefront and step. 32-row steps: lanes 0..31 take
  // -lse / scale, lanes 32..63 -delta (every wavefront writes the same bytes, so that all
  // count the same loads in flight); 64-row steps: even wavefronts take the one, odd the other.
  const int64_t plane = a.BH * a.Sp;
  const __amdgpu_buffer_rsrc_t rbuf = make_buffer(a.work, 2 * plane * 4);
  const bool second = T::ROWS == 32 ? h != 0 : (wave & 1) != 0;
  const int rvoff = static_cast<int>(((second ? plane : 0) + bh * a.Sp +
                                      (T::ROWS == 32 ? l32 : lane)) * 4);
  const uint32_t rdst = T::ROWS == 32 ? 0 : 256 * (wave & 1);
  const int step0 = k0 / T::ROWS, steps = (S + T::ROWS - 1) / T::ROWS - step0;
  auto issue = [&](int step) {
    const uint32_t st = lds0 + (step % kBwdStages) * STAGE;
    const int row0 = (step0 + step) * T::ROWS;
    dma4(rbuf, st + 2 * T::BYTES + rdst, rvoff, row0 * 4);
    qd.issue(st, row0, wave);
    gd.issue(st + T::BYTES, row0, wave);
  };

  v16f_b dk[D / 32], dv[D / 32];
#pragma unroll
  for (int dt = 0; dt < D / 32; ++dt) {
    dk[dt] = v16f_b{};
    dv[dt] = v16f_b{};
  }
  issue(0);
  if (steps > 1) issue(1);
  for (int step = 0; step < steps; ++step) {
    if (step + 1 < steps) dma_wait_barrier<2 * T::CHUNKS + 1>();
    else dma_wait_barrier<0>();
    if (step + 2 < steps) issue(step + 2);
    const uint8_t* qt = smem + (step % kBwdStages) * STAGE;
    const uint8_t* gt = qt + T::BYTES;
    const float* rows = reinterpret_cast<const float*>(gt + T::BYTES);
#pragma unroll
    for (int sub = 0; sub < T::ROWS / 32; ++sub) {
      const int qs = (step0 + step) * T::ROWS + 32 * sub;
      if (qs < kw0 || qs >= S) continue;  // above this wavefront's diagonal, or past the end
      v16f_b st, dp;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float4 nl = *reinterpret_cast<const float4*>(rows + 32 * sub + 8 * r + 4 * h);
        const float4 nd =
            *reinterpret_cast<const float4*>(rows + ROWF / 2 + 32 * sub + 8 * r + 4 * h);
        st[4 * r] = nl.x; st[4 * r + 1] = nl.y; st[4 * r + 2] = nl.z; st[4 * r + 3] = nl.w;
        dp[4 * r] = nd.x; dp[4 * r + 1] = nd.y; dp[4 * r + 2] = nd.z; dp[4 * r + 3] = nd.w;
      }
#pragma unroll
      for (int s = 0; s < D / 16; ++s)
        st = __builtin_amdgcn_mfma_f32_32x32x16_bf16(row_frag<D>(qt, 32 * sub, s, lane), kf[s], st,
                                                     0, 0, 0);
#pragma unroll
      for (int s = 0; s < D / 16; ++s)
        dp = __builtin_amdgcn_mfma_f32_32x32x16_bf16(row_frag<D>(gt, 32 * sub, s, lane), vf[s], dp,
                                                     0, 0, 0);
      float p[16], ds[16];
      // the diagonal tile, and the last tile of a ragged S: queries before the key or past the end
      const bool edge = qs == kw0 || qs + 32 > S;
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        p[e] = __builtin_amdgcn_exp2f(st[e] * a.scale_log2);
        const int qi = qs + 8 * (e / 4) + 4 * h + (e % 4);
        if (edge && (qi < kj || qi >= S)) {
          p[e] = 0.0f;
          dp[e] = 0.0f;
        }
        ds[e] = p[e] * dp[e];
      }
      uint4 pf[2], dsf[2];
      pack16(pf, p);
      pack16(dsf, ds);
#pragma unroll
      for (int s2 = 0; s2 < 2; ++s2)
#pragma unroll
        for (int dt = 0; dt < D / 32; ++dt)
          dv[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
              col_frag<D>(gt, 32 * sub + 16 * s2, dt, lane), frag_of(pf[s2]), dv[dt], 0, 0, 0);
#pragma unroll
      for (int s2 = 0; s2 < 2; ++s2)
#pragma unroll
        for (int dt = 0; dt < D / 32; ++dt)
          dk[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
              col_frag<D>(qt, 32 * sub + 16 * s2, dt, lane), frag_of(dsf[s2]), dk[dt], 0, 0, 0);
    }
  }
  if (kj < S) {
    const int64_t off = b * a.sxb + hd * a.sxh + static_cast<int64_t>(kj) * a.sxs;
    store_owned<D>(a.dk + off, dk, a.scale, h);
    store_owned<D>(a.dv + off, dv, 1.0f, h);
  }
}

static int64_t padded_rows(int64_t S) { return (S + kBwdRows - 1) / kBwdRows * kBwdRows; }

template <int D>
static void launch_bwd(const AttnBwdArgs& a, hipStream_t stream) {
  const dim3 grid(static_cast<unsigned>(a.BH), static_cast<unsigned>(a.Sp / kBwdRows));
  attn_bwd_dq_kernel<D><<<grid, 256, 0, stream>>>(a);
  attn_bwd_dkv_kernel<D><<<grid, 256, 0, stream>>>(a);
}

}  // namespace rk

using namespace rk;

extern "C" int64_t rk_attention_backward_work(int64_t B, int64_t H, int64_t S) {
  if (B <= 0 || H <= 0 || S <= 0) return 0;
  return 2 * B * H * padded_rows(S);
}

extern "C" int rk_attention_backward(const uint16_t* q, int64_t sqb, int64_t sqh, int64_t sqs,
                                     const uint16_t* k, int64_t skb, int64_t skh, int64_t sks,
                                     const uint16_t* v, int64_t svb, int64_t svh, int64_t svs,
                                     const uint16_t* o, int64_t sob, int64_t soh, int64_t sos,
                                     const uint16_t* g, int64_t sgb, int64_t sgh, int64_t sgs,
                                     const float* lse, int64_t B, int64_t H, int64_t S, int64_t D,
                                     float scale, uint16_t* dq, uint16_t* dk, uint16_t* dv,
                                     int64_t sxb, int64_t sxh, int64_t sxs, float* work,
                                     void* stream) {
  clear_error();
  if (B < 0 || H < 0 || S < 0) return fail(RK_ERR_ARG, "negative size");
  if (D != 64 && D != 128) return fail(RK_ERR_UNSUPPORTED, "head size %lld (64 or 128 only)",
                                       static_cast<long long>(D));
  if (B == 0 || H == 0 || S == 0) return RK_OK;
  if (!(scale > 0.0f)) return fail(RK_ERR_ARG, "scale must be positive");
  if (!q || !k || !v || !o || !g || !lse || !dq || !dk || !dv || !work)
    return fail(RK_ERR_ARG, "null pointer");
  const void* in16[] = {q, k, v, o, g};
  for (const void* p : in16)
    if (!aligned16(p)) return fail(RK_ERR_UNSUPPORTED, "q, k, v, o, g need 16-byte alignment");
  const void* out8[] = {dq, dk, dv};
  for (const void* p : out8)
    if (reinterpret_cast<uintptr_t>(p) & 7)
      return fail(RK_ERR_UNSUPPORTED, "dq, dk, dv need 8-byte alignment");
  const int64_t strides[] = {sqb, sqh, sqs, skb, skh, sks, svb, svh, svs,
                             sob, soh, sos, sgb, sgh, sgs, sxb, sxh, sxs};
  for (int64_t st : strides)
    if (st < 0 || st % 8 != 0)
      return fail(RK_ERR_UNSUPPORTED, "strides must be non-negative multiples of 8 elements");
  // buffer offsets are 32-bit: one head's rows up to the padded S, and the row statistics,
  // must lie below 2^31 bytes
  const int64_t rows[] = {sqs, sks, svs, sos, sgs};
  const int64_t Sp = padded_rows(S);
  for (int64_t st : rows)
    if (((Sp + 64) * st + D) * 2 >= (int64_t{1} << 31))
      return fail(RK_ERR_UNSUPPORTED, "sequence extent exceeds 2^31 bytes per head");
  if (B * H > 0x7fffffff || Sp / kBwdRows > 65535 || 2 * B * H * Sp * 4 >= (int64_t{1} << 31))
    return fail(RK_ERR_UNSUPPORTED, "row statistics exceed 2^31 bytes");
  AttnBwdArgs a{q,   k,   v,   o,   g,   sqb, sqh, sqs, skb, skh, sks, svb,
                svh, svs, sob, soh, sos, sgb, sgh, sgs, lse, work, dq,  dk,
                dv,  sxb, sxh, sxs, B * H, H,  S,   Sp,  scale, scale * 1.4426950408889634f,
                1.0f / scale};
  if (D == 64) launch_bwd<64>(a, as_stream(stream));
  else launch_bwd<128>(a, as_stream(stream));
  return launch_status("attention_backward");
}
