// Causal self-attention backward of the training step (gfx950), the backward of
// rk_attention_forward at head size 128 (model.py:117-123): from bf16 q, k, v, o, do [B, H, S, D]
// and the forward's log-sum-exp,
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
// Tiles are staged by LDS-DMA in two stages, one barrier per step (rk_attention.h). Heads run
// fastest over the blocks: where their number is a multiple of 8, the blocks of one head share an
// XCD's L2.
//
// B 8, H 16, S 1024: 73 + 92 us, 120 GFLOP at 730 TFLOP/s, against 293 us for torch's
// memory-efficient backward (its kernel, the delta pass, and the float32 dq buffer cleared and
// converted). Per score a wavefront issues 7 VALU slots (two products, exp2 at a quarter rate,
// half of two bf16 conversions) beside 64 MFMA cycles; what is left is waiting for LDS: every
// product reads its first operand from it, 1 KB per MFMA.
#include "rk_attention.h"

namespace rk {


constexpr int kBwdD = 128;                // head size
typedef AttnTile<kBwdD, 32> BwdTile;      // staged rows per step: 16 KB per tile pair

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

__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2)))
void attn_bwd_dq_kernel(AttnBwdArgs a) {
  constexpr int D = kBwdD;
  using T = BwdTile;
  __shared__ __attribute__((aligned(1024))) uint8_t smem[kAttnStages * 2 * T::BYTES];
  const uint32_t lds0 = lds_address(smem);
  const int S = static_cast<int>(a.S);
  const int nqb = (S + kAttnRows - 1) / kAttnRows;
  const int blk = static_cast<int>(blockIdx.x / a.BH);  // heads fastest
  const int qb = nqb - 1 - blk;                         // longest causal rows first
  const int64_t bh = blockIdx.x - blk * a.BH, b = bh / a.H, hd = bh - b * a.H;
  const int tid = threadIdx.x, lane = tid & 63, h = lane >> 5, l32 = lane & 31;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int qw0 = qb * kAttnRows + 32 * wave, qi = qw0 + l32;

  const uint16_t* gbase = a.g + b * a.sgb + hd * a.sgh;
  v8bf_a qf[D / 16], gf[D / 16];
  load_owned<D>(qf, a.q + b * a.sqb + hd * a.sqh, a.sqs, S, qi, h);
  load_owned<D>(gf, gbase, a.sgs, S, qi, h);

  // delta of this lane's query: half of the features here, the other half in lane ^ 32
  float dot = 0.0f;
  {
    v8bf_a of[D / 16];
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

  const TileDma<D, T::ROWS> kd(a.k + b * a.skb + hd * a.skh, a.sks, S, wave, lane);
  const TileDma<D, T::ROWS> vd(a.v + b * a.svb + hd * a.svh, a.svs, S, wave, lane);
  const int last = qb * kAttnRows + kAttnRows < S ? qb * kAttnRows + kAttnRows : S;
  const int steps = (last + T::ROWS - 1) / T::ROWS;
  auto issue = [&](int step) {
    const uint32_t st = lds0 + (step % kAttnStages) * 2 * T::BYTES;
    kd.issue(st, step * T::ROWS, wave);
    vd.issue(st + T::BYTES, step * T::ROWS, wave);
  };

  v16f_a dq[D / 32];
#pragma unroll
  for (int dt = 0; dt < D / 32; ++dt) dq[dt] = v16f_a{};
  issue(0);
  for (int step = 0; step < steps; ++step) {
    dma_wait_barrier<0>();
    if (step + 1 < steps) issue(step + 1);
    const uint8_t* kt = smem + (step % kAttnStages) * 2 * T::BYTES;
    const uint8_t* vt = kt + T::BYTES;
    const int key0 = step * T::ROWS;
    if (key0 > qw0 || qw0 >= S) continue;  // above this wavefront's diagonal
    v16f_a st, dp;
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      st[e] = nlse;
      dp[e] = ndelta;
    }
#pragma unroll
    for (int s = 0; s < D / 16; ++s)
      st = __builtin_amdgcn_mfma_f32_32x32x16_bf16(row_frag<D>(kt, 0, s, lane), qf[s], st,
                                                   0, 0, 0);
#pragma unroll
    for (int s = 0; s < D / 16; ++s)
      dp = __builtin_amdgcn_mfma_f32_32x32x16_bf16(row_frag<D>(vt, 0, s, lane), gf[s], dp,
                                                   0, 0, 0);
    // the masks sit in one uniform branch, apart from the arithmetic (a condition per element
    // became a branch per element)
    if (key0 == qw0) {  // the diagonal tile: keys past the query
#pragma unroll
      for (int e = 0; e < 16; ++e)
        if (8 * (e / 4) + 4 * h + (e % 4) > l32) st[e] = -INFINITY;
    }
    float ds[16];
#pragma unroll
    for (int e = 0; e < 16; ++e) ds[e] = __builtin_amdgcn_exp2f(st[e] * a.scale_log2) * dp[e];
    uint4 dsf[2];
    pack16(dsf, ds);
#pragma unroll
    for (int s2 = 0; s2 < 2; ++s2)
#pragma unroll
      for (int dt = 0; dt < D / 32; ++dt)
        dq[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
            col_frag<D>(kt, 16 * s2, dt, lane), frag_of(dsf[s2]), dq[dt], 0, 0, 0);
  }
  if (valid)
    store_owned<D>(a.dq + b * a.sxb + hd * a.sxh + static_cast<int64_t>(qi) * a.sxs, dq, a.scale, h);
}

__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2)))
void attn_bwd_dkv_kernel(AttnBwdArgs a) {
  constexpr int D = kBwdD;
  using T = BwdTile;
  constexpr int STAGE = 2 * T::BYTES + 256;  // two tiles, 32 -lse / scale, 32 -delta
  // The owned V rows stay in LDS (32 KB, read again each step): with both K and V beside the dk
  // and dv accumulators in registers the loop spilled at two wavefronts per SIMD (156 us at
  // B 8, H 16, S 1024; 92 us this way).
  constexpr int VTILE = kAttnRows * T::ROWB;
  __shared__ __attribute__((aligned(1024))) uint8_t smem[VTILE + kAttnStages * STAGE];
  const uint32_t lds0 = lds_address(smem) + VTILE;
  const int S = static_cast<int>(a.S);
  const int blk = static_cast<int>(blockIdx.x / a.BH);  // heads fastest
  const int64_t bh = blockIdx.x - blk * a.BH, b = bh / a.H, hd = bh - b * a.H;
  const int k0 = blk * kAttnRows;  // the first keys have the longest walk
  const int tid = threadIdx.x, lane = tid & 63, h = lane >> 5, l32 = lane & 31;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int kw0 = k0 + 32 * wave, kj = kw0 + l32;

  v8bf_a kf[D / 16];
  load_owned<D>(kf, a.k + b * a.skb + hd * a.skh, a.sks, S, kj, h);
  const TileDma<D, T::ROWS> vd(a.v + b * a.svb + hd * a.svh, a.svs, S, wave, lane);
#pragma unroll
  for (int t = 0; t < kAttnRows / T::ROWS; ++t)
    vd.issue(lds_address(smem) + t * T::BYTES, k0 + t * T::ROWS, wave);

  const TileDma<D, T::ROWS> qd(a.q + b * a.sqb + hd * a.sqh, a.sqs, S, wave, lane);
  const TileDma<D, T::ROWS> gd(a.g + b * a.sgb + hd * a.sgh, a.sgs, S, wave, lane);
  // row statistics: one 4-byte DMA per step, lanes 0..31 take -lse / scale, lanes 32..63 -delta
  // (every wavefront writes the same bytes)
  const int64_t plane = a.BH * a.Sp;
  const __amdgpu_buffer_rsrc_t rbuf = make_buffer(a.work, 2 * plane * 4);
  const int rvoff = static_cast<int>(((h != 0 ? plane : 0) + bh * a.Sp + l32) * 4);
  const int step0 = k0 / T::ROWS, steps = (S + T::ROWS - 1) / T::ROWS - step0;
  auto issue = [&](int step) {
    const uint32_t st = lds0 + (step % kAttnStages) * STAGE;
    const int row0 = (step0 + step) * T::ROWS;
    dma4(rbuf, st + 2 * T::BYTES, rvoff, row0 * 4);
    qd.issue(st, row0, wave);
    gd.issue(st + T::BYTES, row0, wave);
  };

  v16f_a dk[D / 32], dv[D / 32];
#pragma unroll
  for (int dt = 0; dt < D / 32; ++dt) {
    dk[dt] = v16f_a{};
    dv[dt] = v16f_a{};
  }
  issue(0);
  for (int step = 0; step < steps; ++step) {
    dma_wait_barrier<0>();
    if (step + 1 < steps) issue(step + 1);
    const uint8_t* qt = smem + VTILE + (step % kAttnStages) * STAGE;
    const uint8_t* gt = qt + T::BYTES;
    const float* rows = reinterpret_cast<const float*>(gt + T::BYTES);
    const int qs = (step0 + step) * T::ROWS;
    if (qs < kw0) continue;  // above this wavefront's diagonal
    v16f_a st, dp;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const float4 nl = *reinterpret_cast<const float4*>(rows + 8 * r + 4 * h);
      const float4 nd =
          *reinterpret_cast<const float4*>(rows + T::ROWS + 8 * r + 4 * h);
      st[4 * r] = nl.x; st[4 * r + 1] = nl.y; st[4 * r + 2] = nl.z; st[4 * r + 3] = nl.w;
      dp[4 * r] = nd.x; dp[4 * r + 1] = nd.y; dp[4 * r + 2] = nd.z; dp[4 * r + 3] = nd.w;
    }
#pragma unroll
    for (int s = 0; s < D / 16; ++s)
      st = __builtin_amdgcn_mfma_f32_32x32x16_bf16(row_frag<D>(qt, 0, s, lane), kf[s], st,
                                                   0, 0, 0);
#pragma unroll
    for (int s = 0; s < D / 16; ++s)
      dp = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
          row_frag<D>(gt, 0, s, lane),
          row_frag<D>(smem, 32 * wave, s, lane), dp, 0, 0, 0);
    // the diagonal tile, and the last tile of a ragged S: queries before the key or past the end
    if (qs == kw0 || qs + 32 > S) {
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const int qi = qs + 8 * (e / 4) + 4 * h + (e % 4);
        if (qi < kj || qi >= S) {
          st[e] = -INFINITY;
          dp[e] = 0.0f;
        }
      }
    }
    float p[16], ds[16];
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      p[e] = __builtin_amdgcn_exp2f(st[e] * a.scale_log2);
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
            col_frag<D>(gt, 16 * s2, dt, lane), frag_of(pf[s2]), dv[dt], 0, 0, 0);
#pragma unroll
    for (int s2 = 0; s2 < 2; ++s2)
#pragma unroll
      for (int dt = 0; dt < D / 32; ++dt)
        dk[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
            col_frag<D>(qt, 16 * s2, dt, lane), frag_of(dsf[s2]), dk[dt], 0, 0, 0);
  }
  if (kj < S) {
    const int64_t off = b * a.sxb + hd * a.sxh + static_cast<int64_t>(kj) * a.sxs;
    store_owned<D>(a.dk + off, dk, a.scale, h);
    store_owned<D>(a.dv + off, dv, 1.0f, h);
  }
}

static int64_t padded_rows(int64_t S) { return (S + kAttnRows - 1) / kAttnRows * kAttnRows; }

static void launch_bwd(const AttnBwdArgs& a, hipStream_t stream) {
  const dim3 grid(static_cast<unsigned>(a.BH * (a.Sp / kAttnRows)));
  attn_bwd_dq_kernel<<<grid, 256, 0, stream>>>(a);
  attn_bwd_dkv_kernel<<<grid, 256, 0, stream>>>(a);
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
  if (D != kBwdD)
    return fail(RK_ERR_UNSUPPORTED, "head size %lld (128 only)", static_cast<long long>(D));
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
  if (2 * B * H * Sp * 4 >= (int64_t{1} << 31))  // (also bounds the grid)
    return fail(RK_ERR_UNSUPPORTED, "row statistics exceed 2^31 bytes");
  AttnBwdArgs a{q,   k,   v,   o,   g,   sqb, sqh, sqs, skb, skh, sks, svb,
                svh, svs, sob, soh, sos, sgb, sgh, sgs, lse, work, dq,  dk,
                dv,  sxb, sxh, sxs, B * H, H,  S,   Sp,  scale, scale * 1.4426950408889634f,
                1.0f / scale};
  launch_bwd(a, as_stream(stream));
  return launch_status("attention_backward");
}
