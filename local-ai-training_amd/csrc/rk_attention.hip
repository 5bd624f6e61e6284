// Causal self-attention forward of the training step (flash form, gfx950), for the model's
// F.scaled_dot_product_attention(q, k, v, is_causal=True) (model.py:117-123): bf16 q, k, v
// [B, H, S, D] (any batch / head / position strides, unit feature stride), D = 64 or 128.
// Writes o (bf16) and the per-query log-sum-exp lse = log(sum_j exp(s_j)) of the scaled
// scores s_j = (q . k_j) * scale, float32 [B, H, S], the pair the backward takes
// (rk_attention_bwd.hip; torch's memory-efficient attention backward takes the same).
//
// One workgroup = 4 wavefronts = 128 queries of one (batch, head); steps of 64 keys are staged
// in LDS by DMA, K and V both row-major (rk_attention.h). Each wavefront owns 32 queries and
// computes S^T = K . Q^T with v_mfma_f32_32x32x16_bf16, K rows as the first operand and its Q
// rows (held in registers) as the second, so a lane holds all the scores of ONE query (its
// lane index mod 32) for 16 keys of each 32-key tile (the partner lane l ^ 32 holds the
// other 16): the softmax's row max and row sum are a lane's own values plus one xor-32
// exchange. The online softmax runs in base 2 (scores times scale * log2 e, exp2). The
// output accumulates transposed, O^T = V^T . P^T: the 8 probabilities a lane holds for
// one 16-key MFMA step are exactly the second operand that step needs, once the
// operand's k slots are mapped to keys {16 s + 4 h + 0..3, 16 s + 8 + 4 h + 0..3}
// (h = lane / 32, the accumulator's own row order), and the first operand reads V transposed
// (ds_read_b64_tr_b16) with the same slot order. The probabilities enter the product rounded
// to bf16; their sum stays float32. Causal tiles above a wavefront's diagonal are skipped; the
// diagonal step is masked per element. Every global load goes through a buffer descriptor
// bounded by the (batch, head) extent, so positions past S read zeros without a test.
//
// Staging V transposed through registers (16 VALU permutes and 8-byte LDS writes per piece) and
// its conflicts held the kernel at 36.7 us (B 32, H 8, S 512, D 64) and 112 us (B 8, H 16,
// S 1024, D 128); both tiles by DMA and V read transposed take 21.2 and 59 us. What is left is
// about the wavefront's exponentials (7 issue slots per score, as much as its MFMAs at D 128,
// twice them at D 64) and the operands it reads (26 us for 134 MB at 5.2 TB/s).
#include "rk_attention.h"

namespace rk {

struct AttnArgs {
  const uint16_t* q;
  const uint16_t* k;
  const uint16_t* v;
  int64_t sqb, sqh, sqs;  // element strides (feature stride 1)
  int64_t skb, skh, sks;
  int64_t svb, svh, svs;
  uint16_t* o;
  int64_t sob, soh, sos;
  float* lse;  // [B, H, S]
  int64_t bh0, BH;  // this launch's (batch, head) pairs: bh0 .. bh0 + BH - 1
  int64_t H, S;
  float scale_log2;  // scale * log2(e)
};

// op over a lane and its partner lane ^ 32 (the two halves of a query's keys).
__device__ __forceinline__ float half_max(float v) {
  const uint32_t b = __float_as_uint(v);
  const auto r = __builtin_amdgcn_permlane32_swap(b, b, false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float half_sum(float v) {
  const uint32_t b = __float_as_uint(v);
  const auto r = __builtin_amdgcn_permlane32_swap(b, b, false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// R keys are staged per step, U of them make one update of the running max and sum. The U keys'
// probabilities are rounded to bf16 relative to the max after them, so U is part of the result's
// rounding, which int8 rows downstream turn into differences of 1%: 64 at D = 64, 32 at D = 128.
// With 64 at D = 128 too, B 8, H 16, S 1024 took 55-59 us against 59-61, B 2, H 8, S 2048 48
// against 52. R is 64, but 32 at D = 128 up to 32 positions: one step either way, in half the
// LDS, so twice the blocks of a CU (8192 heads of 8 positions 35 us against 56).
template <int D, int R, int U>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 4)))
void attn_fwd_kernel(AttnArgs a) {
  using T = AttnTile<D, R>;
  constexpr int UT = U / 32;
  __shared__ __attribute__((aligned(1024))) uint8_t smem[kAttnStages * 2 * T::BYTES];
  const uint32_t lds0 = lds_address(smem);
  // positions fit 32 bits (checked by the host, with the row offsets of S + 128 rows)
  const int S = static_cast<int>(a.S);
  const int nqb = (S + kAttnRows - 1) / kAttnRows;
  // heads fastest: with BH a multiple of 8, one head stays on an XCD
  const int blk = static_cast<int>(blockIdx.x / a.BH);
  const int qb = nqb - 1 - blk;  // longest causal rows first
  const int64_t bh = a.bh0 + blockIdx.x - blk * a.BH, b = bh / a.H, hd = bh - b * a.H;
  const int tid = threadIdx.x, lane = tid & 63, h = lane >> 5, l32 = lane & 31;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int qw0 = qb * kAttnRows + 32 * wave, qi = qw0 + l32;  // this lane's query

  v8bf_a qf[D / 16];
  load_owned<D>(qf, a.q + b * a.sqb + hd * a.sqh, a.sqs, S, qi, h);
  const TileDma<D, R> kd(a.k + b * a.skb + hd * a.skh, a.sks, S, wave, lane);
  const TileDma<D, R> vd(a.v + b * a.svb + hd * a.svh, a.svs, S, wave, lane);
  const int last = qb * kAttnRows + kAttnRows < S ? qb * kAttnRows + kAttnRows : S;
  const int steps = (last + R - 1) / R;
  auto issue = [&](int step) {
    const uint32_t st = lds0 + (step % kAttnStages) * 2 * T::BYTES;
    kd.issue(st, step * R, wave);
    vd.issue(st + T::BYTES, step * R, wave);
  };

  float m = -INFINITY, l = 0.0f;
  v16f_a o[D / 32];
#pragma unroll
  for (int dt = 0; dt < D / 32; ++dt) o[dt] = v16f_a{};
  issue(0);
  for (int step = 0; step < steps; ++step) {
    dma_wait_barrier<0>();
    if (step + 1 < steps) issue(step + 1);
    const uint8_t* kt = smem + (step % kAttnStages) * 2 * T::BYTES;
    const uint8_t* vt = kt + T::BYTES;
    if (step * R > qw0 + 31) continue;  // above this wavefront's diagonal
    // S^T: lane holds keys step R + 32 t + 8 (e / 4) + 4 h + e % 4 of its query
    v16f_a sc[R / 32];
#pragma unroll
    for (int t = 0; t < R / 32; ++t) {
      sc[t] = v16f_a{};
#pragma unroll
      for (int s = 0; s < D / 16; ++s)
        sc[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(row_frag<D>(kt, 32 * t, s, lane), qf[s],
                                                        sc[t], 0, 0, 0);
    }
    if (step * R + R - 1 > qw0) {  // some key of the step lies past some query
#pragma unroll
      for (int t = 0; t < R / 32; ++t)
#pragma unroll
        for (int e = 0; e < 16; ++e)
          if (step * R + 32 * t + 8 * (e / 4) + 4 * h + (e % 4) > qi) sc[t][e] = -INFINITY;
    }
    // The updates' probabilities first, then their products: the only branches (a rescale) then
    // lie between products, and the exponentials of one update overlap the next one's.
    float alpha[R / U], ps[R / U];
    uint4 pf[R / 32][2];
#pragma unroll
    for (int u = 0; u < R / U; ++u) {
      float mx = -INFINITY;
#pragma unroll
      for (int t = u * UT; t < (u + 1) * UT; ++t)
#pragma unroll
        for (int e = 0; e < 16; ++e) mx = fmaxf(mx, sc[t][e]);
      mx = half_max(mx);
      // the running max in base-2 units (scale * log2 e > 0 commutes with max)
      const float mnew = fmaxf(m, mx * a.scale_log2);
      const float mref = mnew == -INFINITY ? 0.0f : mnew;  // a row with no key yet
      alpha[u] = __builtin_amdgcn_exp2f(m - mref);
      m = mnew;
      ps[u] = 0.0f;
#pragma unroll
      for (int t = u * UT; t < (u + 1) * UT; ++t) {
        float p[16];
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          p[e] = __builtin_amdgcn_exp2f(__builtin_fmaf(sc[t][e], a.scale_log2, -mref));
          ps[u] = ps[u] + p[e];
        }
        pack16(pf[t], p);
      }
    }
#pragma unroll
    for (int u = 0; u < R / U; ++u) {
      // keys above the diagonal: alpha is 1 and every p zero, but their values may not be finite
      if (step * R + u * U > qw0 + 31) break;
      // rescale only when some query's running max grew (alpha == 1 exactly otherwise:
      // exp2(0) = 1), which after the first keys is rare
      if (__any(alpha[u] != 1.0f)) {
#pragma unroll
        for (int dt = 0; dt < D / 32; ++dt)
#pragma unroll
          for (int e = 0; e < 16; ++e) o[dt][e] = o[dt][e] * alpha[u];
      }
      l = l * alpha[u] + half_sum(ps[u]);
#pragma unroll
      for (int t = u * UT; t < (u + 1) * UT; ++t)
#pragma unroll
        for (int s2 = 0; s2 < 2; ++s2)
#pragma unroll
          for (int dt = 0; dt < D / 32; ++dt)
            o[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                col_frag<D>(vt, 32 * t + 16 * s2, dt, lane), frag_of(pf[t][s2]), o[dt], 0, 0, 0);
    }
  }

  if (qi < S) {
    store_owned<D>(a.o + b * a.sob + hd * a.soh + static_cast<int64_t>(qi) * a.sos, o, 1.0f / l, h);
    if (h == 0) a.lse[bh * a.S + qi] = (m + __log2f(l)) * 0.69314718055994531f;
  }
}

// Keys and values of a prompt into their cache, one 16-byte vector of each per thread, the rows
// behind them cleared in the same pass: two strided copies and two strided clears before (29 us
// a layer at 4 sequences x 777 positions x 16 heads x 128; 10.4 us in one launch).
__global__ __launch_bounds__(256) void kv_append_kernel(
    const uint4* k, int64_t skb, int64_t skh, int64_t sks, const uint4* v, int64_t svb,
    int64_t svh, int64_t svs, uint4* keys, uint4* values, uint32_t H, uint32_t S, uint32_t rows,
    uint32_t per_row, uint32_t max_len, uint32_t start) {
  const uint32_t i = blockIdx.x * 256 + threadIdx.x;  // the host bounds rows * per_row
  const uint32_t row = i / per_row, piece = i - row * per_row;
  if (row >= rows) return;
  const uint32_t bh = blockIdx.y, b = bh / H, h = bh - b * H;
  uint4 kv = make_uint4(0, 0, 0, 0), vv = kv;
  if (row < S) {
    kv = k[b * skb + h * skh + row * sks + piece];
    vv = v[b * svb + h * svh + row * svs + piece];
  }
  const int64_t to = (static_cast<int64_t>(bh) * max_len + start + row) * per_row + piece;
  keys[to] = kv;
  values[to] = vv;
}

}  // namespace rk

using namespace rk;

extern "C" int rk_kv_append(const void* k, int64_t skb, int64_t skh, int64_t sks, const void* v,
                            int64_t svb, int64_t svh, int64_t svs, void* keys, void* values,
                            int elem_size, int64_t B, int64_t H, int64_t S, int64_t D,
                            int64_t max_len, int64_t start, int64_t clear_to, void* stream) {
  clear_error();
  if (B < 0 || H < 0 || S < 0 || D <= 0) return fail(RK_ERR_ARG, "invalid cache shape");
  if (start < 0 || start + S > max_len || clear_to > max_len)
    return fail(RK_ERR_ARG, "positions past the cache");
  if (elem_size != 2 && elem_size != 4) return fail(RK_ERR_UNSUPPORTED, "2 or 4 byte elements");
  const int64_t end = clear_to > start + S ? clear_to : start + S;
  if (B == 0 || H == 0 || end == start) return RK_OK;
  if (!keys || !values || (S > 0 && (!k || !v))) return fail(RK_ERR_ARG, "null pointer");
  const int64_t per = 16 / elem_size;  // elements per vector
  const int64_t strides[] = {skb, skh, sks, svb, svh, svs, D};
  for (int64_t st : strides)
    if (st < 0 || st % per != 0)
      return fail(RK_ERR_UNSUPPORTED, "cache rows and strides must be whole 16-byte vectors");
  if (!aligned16(k) || !aligned16(v) || !aligned16(keys) || !aligned16(values))
    return fail(RK_ERR_UNSUPPORTED, "keys and values need 16-byte alignment");
  const int64_t rows = end - start, pieces = rows * (D / per);
  if (B * H > 65535 || pieces >= (int64_t{1} << 31) || max_len >= (int64_t{1} << 31))
    return fail(RK_ERR_UNSUPPORTED, "cache too large for one launch");
  const dim3 grid(static_cast<unsigned>((pieces + 255) / 256), static_cast<unsigned>(B * H));
  kv_append_kernel<<<grid, 256, 0, as_stream(stream)>>>(
      static_cast<const uint4*>(k), skb / per, skh / per, sks / per, static_cast<const uint4*>(v),
      svb / per, svh / per, svs / per, static_cast<uint4*>(keys), static_cast<uint4*>(values),
      static_cast<uint32_t>(H), static_cast<uint32_t>(S), static_cast<uint32_t>(rows),
      static_cast<uint32_t>(D / per), static_cast<uint32_t>(max_len),
      static_cast<uint32_t>(start));
  return launch_status("kv_append");
}

extern "C" int rk_attention_forward(const uint16_t* q, int64_t sqb, int64_t sqh, int64_t sqs,
                                    const uint16_t* k, int64_t skb, int64_t skh, int64_t sks,
                                    const uint16_t* v, int64_t svb, int64_t svh, int64_t svs,
                                    int64_t B, int64_t H, int64_t S, int64_t D, float scale,
                                    uint16_t* o, int64_t sob, int64_t soh, int64_t sos,
                                    float* lse, void* stream) {
  clear_error();
  if (B < 0 || H < 0 || S < 0) return fail(RK_ERR_ARG, "negative size");
  if (D != 64 && D != 128) return fail(RK_ERR_UNSUPPORTED, "head size %lld (64 or 128 only)",
                                       static_cast<long long>(D));
  if (B == 0 || H == 0 || S == 0) return RK_OK;
  if (!q || !k || !v || !o || !lse) return fail(RK_ERR_ARG, "null pointer");
  if (!aligned16(q) || !aligned16(k) || !aligned16(v) || (reinterpret_cast<uintptr_t>(o) & 7))
    return fail(RK_ERR_UNSUPPORTED, "q, k, v need 16-byte and o 8-byte alignment");
  const int64_t strides[] = {sqb, sqh, sqs, skb, skh, sks, svb, svh, svs, sob, soh, sos};
  for (int64_t st : strides)
    if (st < 0 || st % 8 != 0)
      return fail(RK_ERR_UNSUPPORTED, "strides must be non-negative multiples of 8 elements");
  // buffer offsets are 32-bit: the rows of one (batch, head) up to S + 128 (the last key
  // block's padding) must lie below 2^31 bytes
  const int64_t rows = S + 128;
  if ((rows * sqs + D) * 2 >= (int64_t{1} << 31) || (rows * sks + D) * 2 >= (int64_t{1} << 31) ||
      (rows * svs + D) * 2 >= (int64_t{1} << 31))
    return fail(RK_ERR_UNSUPPORTED, "sequence extent exceeds 2^31 bytes per head");
  // a launch holds fewer than 2^24 blocks (2^32 threads): more heads take several
  const int64_t nqb = (S + kAttnRows - 1) / kAttnRows, per = ((int64_t{1} << 24) - 1) / nqb;
  if (B * H > 0x7fffffff || per == 0) return fail(RK_ERR_ARG, "grid too large");
  AttnArgs a{q, k, v, sqb, sqh, sqs, skb, skh, sks, svb, svh, svs, o, sob, soh, sos, lse,
             0, 0, H, S, scale * 1.4426950408889634f};
  for (; a.bh0 < B * H; a.bh0 += a.BH) {
    a.BH = B * H - a.bh0 < per ? B * H - a.bh0 : per;
    const dim3 grid(static_cast<unsigned>(a.BH * nqb));
    if (D == 64) attn_fwd_kernel<64, 64, 64><<<grid, 256, 0, as_stream(stream)>>>(a);
    else if (S <= 32) attn_fwd_kernel<128, 32, 32><<<grid, 256, 0, as_stream(stream)>>>(a);
    else attn_fwd_kernel<128, 64, 32><<<grid, 256, 0, as_stream(stream)>>>(a);
  }
  return launch_status("attention_forward");
}
