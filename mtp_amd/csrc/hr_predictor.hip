// Forward of the reference's HiddenResidualExpertPredictor
// (src/mtp_expert_prefetch/training/hidden_residual.py:44-106) in bf16, plus the residual
// combination logits = prior + scale * residual (train_hidden_residual_predictor_smoke.py:446)
// and the top-k experts of every (example, future delta):
//
//   z  = bf16(x . W_enc^T + b_enc)                    encoder Linear (fp32 sums)
//   a  = bf16(silu(z))                                SiLU
//   s  = bf16(LayerNorm(a) * ln_w + ln_b)             LayerNorm over the width (fp32 statistics)
//   c_d = bf16(bf16(s + E_layer[layer]) + E_delta[d]) context per future delta d
//   g_d = bf16(silu(c_d))
//   r_d = g_d . W_cls^T + b_cls                       classifier (fp32 sums), fp32
//   out_d = prior_d + scale * r_d                     (prior optional), top-k by (value, id)
//
// Every Linear input is bf16 (the dtype of a bf16 model's activations), and both Linear layers sum
// exact products in fp32, on v_mfma_f32_16x16x32_bf16 or in the router's canonical order
// (routing.h:logits_tile). At these sizes a call is bound by launches and by each kernel's chain
// of loads, not by bytes or arithmetic. Two forms (hr_split chooses):
//  - two launches: the encoder, then everything per 16 context rows (hr_rows_kernel): 160 examples
//    of the default shape (hidden 2048, width 256, 4 deltas, 256 experts, top-16) 19 us on the GPU
//    and 22 us a call, which the host's work bounds (four launches: 29 to 53 us);
//  - four launches for few rows of a large classifier, which one workgroup of the first form would
//    read alone: the encoder, the context rows, the classifier over many workgroups, the
//    selection: one example and delta of width 1024 with 512 experts 20.8 us on the GPU and 29 a
//    call (46 and 46 in two launches).
// The error against 64 bits is the same (3.7e-3 to 4.2e-3 of the residual over 3 to 640 examples
// and widths 128 to 512: the bf16 activations).
#include <math.h>
#include <stdio.h>

#include "launch.h"
#include "routing.h"

namespace {

typedef __bf16 bf16x8_h __attribute__((ext_vector_type(8)));
MOE_DEV f32x4 mfma16(u32x4 a, u32x4 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_h, a),
                                                 __builtin_bit_cast(bf16x8_h, b), c, 0, 0, 0);
}

MOE_DEV float bf16_round(float v) { return bf16_to_f32(f32_to_bf16_rne(v)); }

constexpr int kMaxWidth = 1024;
// Up to this many examples the encoder runs as the router's GEMV: a 16-row MFMA tile would be
// partly padding (width 256: 1 example 3.3 against 4.9 us, 16 examples 4.9 against 6.0, 40 the same).
constexpr int kEncFew = 16;

// z[n][j] = x_n . W_enc[j] (fp32): a 16 x 16 (example x output) tile per workgroup, its four waves a
// quarter of K each (added in wave order). A wave has 16 k-steps of both operands in flight at
// once (all of its K at hidden 2048), so a tile takes about one memory latency; 16 x 16 tiles put the
// most workgroups on the chip (160 at 160 examples). Lane (r, kq) reads row r at k = 32 step + 8 kq;
// rows and chunks out of range read zeros without a memory access.
constexpr int kEncWaves = 4, kEncSteps = 16;
__global__ __launch_bounds__(64 * kEncWaves) void hr_encoder_kernel(
    const uint16_t* __restrict__ x, int N, int H, const uint16_t* __restrict__ enc_w, int W,
    float* __restrict__ z) {
  __shared__ f32x4 part[kEncWaves][64];
  const int lane = threadIdx.x & 63, r = lane & 15, kq = lane >> 4;
  const int wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int tiles_w = (W + 15) / 16;
  const int n0 = (int)(blockIdx.x / tiles_w) * 16, j0 = (int)(blockIdx.x % tiles_w) * 16;
  const __amdgpu_buffer_rsrc_t xr = buf_rsrc(x, (uint32_t)N * (uint32_t)H * 2u);
  const __amdgpu_buffer_rsrc_t wr = buf_rsrc(enc_w, (uint32_t)W * (uint32_t)H * 2u);
  const uint32_t xo = n0 + r < N ? (uint32_t)(n0 + r) * (uint32_t)H * 2u : kOutOfRange;
  const uint32_t wo = j0 + r < W ? (uint32_t)(j0 + r) * (uint32_t)H * 2u : kOutOfRange;
  const int steps = (H + 31) / 32, per_wave = (steps + kEncWaves - 1) / kEncWaves;
  const int s_end = min(steps, (wv + 1) * per_wave);
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  for (int s0 = wv * per_wave; s0 < s_end; s0 += kEncSteps) {
    u32x4 a[kEncSteps], b[kEncSteps];
#pragma unroll
    for (int i = 0; i < kEncSteps; ++i) {
      const int k = 32 * (s0 + i) + 8 * kq;
      const uint32_t ko = s0 + i < s_end && k < H ? (uint32_t)k * 2u : kOutOfRange;
      a[i] = buf_ld128(xr, (xo + ko) | ((xo | ko) & kOutOfRange));
      b[i] = buf_ld128(wr, (wo + ko) | ((wo | ko) & kOutOfRange));
    }
    __builtin_amdgcn_sched_barrier(0);  // every load before the first wait
#pragma unroll
    for (int i = 0; i < kEncSteps; ++i) acc = mfma16(a[i], b[i], acc);
  }
  part[wv][lane] = acc;
  __syncthreads();
  if (wv != 0) return;
#pragma unroll
  for (int w = 1; w < kEncWaves; ++w) acc = acc + part[w][lane];
#pragma unroll
  for (int i = 0; i < 4; ++i) {  // D[4 kq + i][r]
    const int n = n0 + 4 * kq + i, j = j0 + r;
    if (n < N && j < W) z[(int64_t)n * (W + 1) + j] = acc[i];
  }
}

// NW consecutive dwords at byte offset `off`, one load.
template <int NW>
MOE_DEV void ld_words(__amdgpu_buffer_rsrc_t r, uint32_t off, uint32_t (&o)[NW]) {
  static_assert(NW == 1 || NW == 2 || NW == 4, "one buffer load");
  if constexpr (NW == 4) {
    const u32x4 v = buf_ld128(r, off);
#pragma unroll
    for (int j = 0; j < 4; ++j) o[j] = v[j];
  } else if constexpr (NW == 2) {
    const u32x2 v = buf_ld64(r, off);
    o[0] = v[0];
    o[1] = v[1];
  } else {
    o[0] = buf_ld32(r, off);
  }
}

// 16 context rows r = n * F + d per workgroup, one wave per row: SiLU, LayerNorm (fp32
// statistics), embeddings and SiLU of the row into LDS as bf16; the 16 x E classifier tile on MFMA
// (wave w the expert tiles w, w + 16); then v = (prior ? prior[r] : 0) + scale_n * logits[r],
// optionally written to out, and the top-k of v by (value, lower id), again one wave per row, so
// that the 16 selections of a workgroup run side by side (each is a serial chain of top_k rounds).
// What bounds it is the memory round trips of that chain, so every operand of the context row, the
// prior, the bias and the first classifier steps are loaded together, four columns a lane, two up to
// width 128 (one
// column a lane with the loads behind their range checks: one example 12.4 us against 10.6 at
// width 256, 20.3 against 14.2 at width 512), and a wave keeps kRing classifier steps in flight.
// NC, MAXC: 64-lane columns of the width and of the experts. The F rows of one example repeat its
// LayerNorm: cheaper than another launch. 64 VGPRs where that fits: two workgroups per CU (5120
// rows of width 64 at four columns a lane 29.5 us, with one workgroup 32.0).
constexpr int kRows = 16;
template <int NC, int MAXC>
__global__ __launch_bounds__(64 * kRows, NC + MAXC <= 8 ? 8 : 4) void hr_rows_kernel(
    const float* __restrict__ z, int rows, int F, const int32_t* __restrict__ layer_ids,
    moe_hr_predictor_params_v1 p, const float* __restrict__ prior, float scale,
    const float* __restrict__ scale_per_example, int top_k, float* __restrict__ out,
    int32_t* __restrict__ ids) {
  constexpr int kG = 64 * NC + 8, kL = 64 * MAXC + 4;  // row strides (16-byte rows, odd quads)
  constexpr int TPW = MAXC / 4;                        // expert tiles per wave
  constexpr int CPL = NC < 4 ? NC : 4, NQ = NC / CPL;  // columns of a load, loads per lane
  // classifier k-steps of 32: in all, in the ring of a wave, and of these loaded before the context
  constexpr int kSteps = 2 * NC, kRing = 16 / TPW < kSteps ? 16 / TPW : kSteps,
                kFirst = 8 / TPW < kRing ? 8 / TPW : kRing;
  __shared__ __attribute__((aligned(16))) uint16_t s_g[kRows * kG];
  __shared__ float s_l[kRows * kL];
  const int lane = threadIdx.x & 63, r16 = lane & 15, kq = lane >> 4;
  const int wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int W = p.width, E = p.num_experts;
  const int row = (int)blockIdx.x * kRows + wv;
  const bool live = row < rows;  // wave-uniform
  const int n = live ? row / F : 0, d = live ? row % F : 0;
  const int layer = layer_ids[n];
  const bool layer_ok = layer >= 0 && layer < p.num_layers;  // else the embedding reads zeros
  const float sc = scale_per_example ? scale_per_example[n] : scale;

  // The context row's operands (lane: columns CPL (lane + 64 i) ..; past the width zeros, without a
  // memory access), the prior, the classifier's bias and its first chunk: one memory latency.
  const uint32_t wb = (uint32_t)W * 2u;
  const __amdgpu_buffer_rsrc_t zr = buf_rsrc(z + (int64_t)n * (W + 1), 2u * wb);
  const __amdgpu_buffer_rsrc_t br = buf_rsrc(p.enc_b, 2u * wb);
  const __amdgpu_buffer_rsrc_t lwr = buf_rsrc(p.ln_w, wb), lbr = buf_rsrc(p.ln_b, wb);
  const __amdgpu_buffer_rsrc_t ler =
      buf_rsrc(p.layer_emb + (int64_t)(layer_ok ? layer : 0) * W, layer_ok ? wb : 0u);
  const __amdgpu_buffer_rsrc_t der = buf_rsrc(p.delta_emb + (int64_t)d * W, wb);
  uint32_t zq[NQ][CPL], bq[NQ][CPL], lw[NQ][CPL / 2], lb[NQ][CPL / 2], le[NQ][CPL / 2],
      de[NQ][CPL / 2];
#pragma unroll
  for (int i = 0; i < NQ; ++i) {
    const uint32_t o = (uint32_t)(CPL * 2 * (lane + 64 * i));
    ld_words(zr, 2u * o, zq[i]);
    ld_words(br, 2u * o, bq[i]);
    ld_words(lwr, o, lw[i]);
    ld_words(lbr, o, lb[i]);
    ld_words(ler, o, le[i]);
    ld_words(der, o, de[i]);
  }
  const __amdgpu_buffer_rsrc_t pr = buf_rsrc(prior ? prior + (int64_t)(live ? row : 0) * E : nullptr,
                                             prior && live ? (uint32_t)E * 4u : 0u);
  float pv[MAXC], cb[TPW];
#pragma unroll
  for (int c = 0; c < MAXC; ++c)
    pv[c] = __uint_as_float(buf_ld32(pr, (uint32_t)(lane + 64 * c) * 4u));
  const __amdgpu_buffer_rsrc_t cbr = buf_rsrc(p.cls_b, (uint32_t)E * 4u);
#pragma unroll
  for (int t = 0; t < TPW; ++t)
    cb[t] = __uint_as_float(buf_ld32(cbr, (uint32_t)(16 * (wv + 16 * t) + r16) * 4u));
  const __amdgpu_buffer_rsrc_t cr = buf_rsrc(p.cls_w, (uint32_t)E * wb);
  u32x4 b[kRing][TPW];
  auto load_cls = [&](int i) {  // k-step i into its place in the ring
    const int k = 32 * i + 8 * kq;
    const uint32_t ko = k < W ? (uint32_t)k * 2u : kOutOfRange;
#pragma unroll
    for (int t = 0; t < TPW; ++t) {
      const int e = 16 * (wv + 16 * t) + r16;
      const uint32_t eo = e < E ? (uint32_t)e * wb : kOutOfRange;
      b[i % kRing][t] = buf_ld128(cr, (eo + ko) | ((eo | ko) & kOutOfRange));
    }
  };
#pragma unroll
  for (int i = 0; i < kFirst; ++i) load_cls(i);
  __builtin_amdgcn_sched_barrier(0);

  float a[NQ][CPL], sum = 0.0f;
#pragma unroll
  for (int i = 0; i < NQ; ++i)
#pragma unroll
    for (int j = 0; j < CPL; ++j) {
      const float zb = bf16_round(__uint_as_float(zq[i][j]) + __uint_as_float(bq[i][j]));
      a[i][j] = bf16_round(zb / (1.0f + expf(-zb)));  // past the width silu(0) = 0
      sum += a[i][j];
    }
  const float mean = bfly_sum(sum) / (float)W;
  float sq = 0.0f;
#pragma unroll
  for (int i = 0; i < NQ; ++i)
#pragma unroll
    for (int j = 0; j < CPL; ++j) {
      const float dv = CPL * (lane + 64 * i) < W ? a[i][j] - mean : 0.0f;
      sq = __builtin_fmaf(dv, dv, sq);
    }
  const float var = bfly_sum(sq) / (float)W;
  const float rstd = 1.0f / sqrtf(var + p.ln_eps);
#pragma unroll
  for (int i = 0; i < NQ; ++i) {
    const uint32_t in = 0u - (uint32_t)(CPL * (lane + 64 * i) < W);
    uint32_t g[CPL / 2];
#pragma unroll
    for (int w = 0; w < CPL / 2; ++w) {
      uint32_t half[2];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        auto el = [&](uint32_t v) { return h ? bf16hi_to_f32(v) : bf16lo_to_f32(v); };
        const float s = bf16_round((a[i][2 * w + h] - mean) * rstd * el(lw[i][w]) + el(lb[i][w]));
        const float sl = bf16_round(s + el(le[i][w]));
        const float c = bf16_round(sl + el(de[i][w]));
        half[h] = f32_to_bf16_rne(c / (1.0f + expf(-c)));
      }
      g[w] = (half[0] | (half[1] << 16)) & in;
    }
    uint16_t* dst = s_g + wv * kG + CPL * (lane + 64 * i);
    if constexpr (CPL == 4)
      *reinterpret_cast<u32x2*>(dst) = u32x2{g[0], g[1]};
    else
      *reinterpret_cast<uint32_t*>(dst) = g[0];
  }
#pragma unroll
  for (int i = kFirst; i < kRing; ++i) load_cls(i);
  // A barrier without __syncthreads' fence, which would also wait for the loads in flight.
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  __builtin_amdgcn_s_barrier();
  __atomic_signal_fence(__ATOMIC_SEQ_CST);

  // classifier: A row r16 at k = 32 step + 8 kq from LDS
  f32x4 acc[TPW];
#pragma unroll
  for (int t = 0; t < TPW; ++t) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i0 = 0; i0 < kSteps; i0 += 4) {
    u32x4 av[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) av[i] = ld128(s_g + r16 * kG + 32 * (i0 + i) + 8 * kq);
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int t = 0; t < TPW; ++t) acc[t] = mfma16(av[i], b[(i0 + i) % kRing][t], acc[t]);
    if (i0 + kRing < kSteps) {
#pragma unroll
      for (int i = 0; i < 4; ++i) load_cls(i0 + i + kRing);
      __builtin_amdgcn_sched_barrier(0);  // the ring's loads here, not at their use
    }
  }
#pragma unroll
  for (int t = 0; t < TPW; ++t) {
    const int e = 16 * (wv + 16 * t) + r16;
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (e < E) s_l[(4 * kq + i) * kL + e] = acc[t][i] + cb[t];
  }
  __syncthreads();
  if (!live) return;

  uint32_t key[MAXC];
#pragma unroll
  for (int c = 0; c < MAXC; ++c) {
    const int e = lane + 64 * c;
    const float v = e < E ? pv[c] + sc * s_l[wv * kL + e] : 0.0f;
    if (out && e < E) out[(int64_t)row * E + e] = v;
    key[c] = topk_ord(v) & (0u - (uint32_t)(e < E));
  }
  int my_i;
  uint32_t my_key;
  topk_select_keys<MAXC>(key, top_k, lane, my_i, my_key);
  if (lane < top_k) ids[(int64_t)row * top_k + lane] = my_i;
}

constexpr int kCtxThreads = 256;
constexpr int kCtxMaxPerThread = kMaxWidth / kCtxThreads;

// Fixed-order sum over the workgroup: per-thread value -> wave butterfly -> waves in order.
MOE_DEV float block_sum(float v, float* red) {
  v = bfly_sum(v);
  const int wv = threadIdx.x >> 6;
  __syncthreads();
  if ((threadIdx.x & 63) == 0) red[wv] = v;
  __syncthreads();
  float s = 0.0f;
  for (int w = 0; w < kCtxThreads / 64; ++w) s += red[w];
  return s;
}

// One workgroup per example n: the encoder output row z[n] (fp32 dot, stride W + 1) -> the
// future_window context rows g[n * F + d] (bf16).
__global__ __launch_bounds__(kCtxThreads) void hr_context_kernel(
    const float* __restrict__ z, int N, int W, const float* __restrict__ enc_b,
    const uint16_t* __restrict__ ln_w, const uint16_t* __restrict__ ln_b, float ln_eps,
    const int32_t* __restrict__ layer_ids, int num_layers, const uint16_t* __restrict__ layer_emb,
    const uint16_t* __restrict__ delta_emb, int F, uint16_t* __restrict__ g) {
  __shared__ float red[kCtxThreads / 64];
  const int n = blockIdx.x;
  const int tid = threadIdx.x;
  float a[kCtxMaxPerThread];
  float sum = 0.0f;
#pragma unroll
  for (int i = 0; i < kCtxMaxPerThread; ++i) {
    const int j = tid + kCtxThreads * i;
    a[i] = 0.0f;
    if (j < W) {
      const float zb = bf16_round(z[(int64_t)n * (W + 1) + j] + enc_b[j]);
      a[i] = bf16_round(zb / (1.0f + expf(-zb)));
      sum += a[i];
    }
  }
  const float mean = block_sum(sum, red) / (float)W;
  float sq = 0.0f;
#pragma unroll
  for (int i = 0; i < kCtxMaxPerThread; ++i) {
    const int j = tid + kCtxThreads * i;
    if (j < W) {
      const float d = a[i] - mean;
      sq = __builtin_fmaf(d, d, sq);
    }
  }
  const float var = block_sum(sq, red) / (float)W;
  const float rstd = 1.0f / sqrtf(var + ln_eps);
  const int layer = layer_ids[n];
  const bool layer_ok = layer >= 0 && layer < num_layers;  // else the embedding reads zeros
#pragma unroll
  for (int i = 0; i < kCtxMaxPerThread; ++i) {
    const int j = tid + kCtxThreads * i;
    if (j >= W) continue;
    const float s = bf16_round((a[i] - mean) * rstd * bf16_to_f32(ln_w[j]) + bf16_to_f32(ln_b[j]));
    const float le = layer_ok ? bf16_to_f32(layer_emb[(int64_t)layer * W + j]) : 0.0f;
    const float sl = bf16_round(s + le);
    for (int d = 0; d < F; ++d) {
      const float c = bf16_round(sl + bf16_to_f32(delta_emb[(int64_t)d * W + j]));
      g[((int64_t)n * F + d) * W + j] = (uint16_t)f32_to_bf16_rne(c / (1.0f + expf(-c)));
    }
  }
}

// One wave per row r = n * F + d: v = (prior ? prior[r] : 0) + scale_n * logits[r], optionally
// written to out, and the top-k of v by (value, lower id).
template <int MAXC>
__global__ __launch_bounds__(256) void hr_select_kernel(
    const float* __restrict__ logits, int rows, int F, int E, const float* __restrict__ prior,
    float scale, const float* __restrict__ scale_per_example, int top_k,
    float* __restrict__ out, int32_t* __restrict__ ids) {
  const int lane = threadIdx.x & 63;
  const int r = blockIdx.x * 4 + __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  if (r >= rows) return;
  const float sc = scale_per_example ? scale_per_example[r / F] : scale;
  const __amdgpu_buffer_rsrc_t lr = buf_rsrc(logits + (int64_t)r * (E + 1), (uint32_t)E * 4u);
  const __amdgpu_buffer_rsrc_t pr = buf_rsrc(prior ? prior + (int64_t)r * E : nullptr,
                                             prior ? (uint32_t)E * 4u : 0u);
  uint32_t key[MAXC];
#pragma unroll
  for (int c = 0; c < MAXC; ++c) {
    const int e = lane + 64 * c;
    const float l = __uint_as_float(buf_ld32(lr, (uint32_t)e * 4u));
    const float p = __uint_as_float(buf_ld32(pr, (uint32_t)e * 4u));
    const float v = p + sc * l;
    if (out && e < E) out[(int64_t)r * E + e] = v;
    key[c] = topk_ord(v) & (0u - (uint32_t)(e < E));
  }
  int my_i;
  uint32_t my_key;
  topk_select_keys<MAXC>(key, top_k, lane, my_i, my_key);
  if (lane < top_k) ids[(int64_t)r * top_k + lane] = my_i;
}

}  // namespace

namespace {
int64_t a256(int64_t v) { return (v + 255) & ~int64_t(255); }

// Whether the context rows, the classifier and the selection are launches of their own, from both
// forms' times over widths 64 to 1024, 64 to 512 experts and 1 to 5120 rows:
//  - never up to width 512 and 256 KB of classifier: a launch costs the host 3 us, which the
//    classifier's reading alone by a CU does not reach (one example, width 512, 256 experts: 22.4
//    against 27.9 us a call, 18.2 against 16.0 on the GPU);
//  - beyond, up to 64 rows (the small tiles of launch_router_logits; width 768, 256 experts, 64 rows
//    28.4 against 31.8 us a call, 160 rows 34.9 against 32), and up to 512 where the width is a
//    multiple of 512, which the classifier's 8 x 8 tiles need (width 1024, 256 rows 29.1 against
//    34.7, 1024 rows 50.0 against 45.9);
//  - always where a bf16 array starts at an odd element: the context kernel loads single ones.
bool hr_split(const moe_hr_predictor_params_v1& p, int64_t rows) {
  const uintptr_t bases =
      reinterpret_cast<uintptr_t>(p.ln_w) | reinterpret_cast<uintptr_t>(p.ln_b) |
      reinterpret_cast<uintptr_t>(p.layer_emb) | reinterpret_cast<uintptr_t>(p.delta_emb);
  if (bases & 3u) return true;
  if (p.width <= 512 && p.width * p.num_experts <= 128 * 1024) return false;
  return rows <= (p.width % 512 == 0 ? 512 : 64);
}
}  // namespace

// Workspace sections: z [N][W + 1] fp32; in the split form also g [N * F][W] bf16 and logits
// [N * F][E + 1] fp32.
int64_t hr_predictor_workspace(int N, const moe_hr_predictor_params_v1& p) {
  const int64_t rows = (int64_t)N * p.future_window, z = a256((int64_t)N * (p.width + 1) * 4);
  return hr_split(p, rows) ? z + a256(rows * p.width * 2) + a256(rows * (p.num_experts + 1) * 4) : z;
}

hipError_t launch_hr_predictor(const uint16_t* x, int N, int H, const int32_t* layer_ids,
                               const moe_hr_predictor_params_v1& p, const float* prior, float scale,
                               const float* scale_per_example, int top_k, void* workspace,
                               float* out, int32_t* ids, hipStream_t stream) {
  const int W = p.width, F = p.future_window, E = p.num_experts, rows = N * F;
  char* ws = static_cast<char*>(workspace);
  float* z = reinterpret_cast<float*>(ws);
  hipError_t err;
  if (N <= kEncFew) {
    err = launch_router_logits(x, N, H, p.enc_w, W, nullptr, nullptr, z, stream);
  } else {
    hipLaunchKernelGGL(hr_encoder_kernel, dim3(((N + 15) / 16) * ((W + 15) / 16)),
                       dim3(64 * kEncWaves), 0, stream, x, N, H, p.enc_w, W, z);
    err = hipGetLastError();
  }
  if (err != hipSuccess) return err;
  if (hr_split(p, rows)) {
    uint16_t* g = reinterpret_cast<uint16_t*>(ws + a256((int64_t)N * (W + 1) * 4));
    float* lg = reinterpret_cast<float*>(ws + a256((int64_t)N * (W + 1) * 4) +
                                         a256((int64_t)rows * W * 2));
    hipLaunchKernelGGL(hr_context_kernel, dim3(N), dim3(kCtxThreads), 0, stream, z, N, W, p.enc_b,
                       p.ln_w, p.ln_b, p.ln_eps, layer_ids, p.num_layers, p.layer_emb, p.delta_emb,
                       F, g);
    if ((err = hipGetLastError()) != hipSuccess) return err;
    // classifier over the context rows, bias added, row stride E + 1
    err = launch_router_logits(g, rows, W, p.cls_w, E, nullptr, p.cls_b, lg, stream);
    if (err != hipSuccess) return err;
    auto select = [&](auto kernel) {
      hipLaunchKernelGGL(kernel, dim3((rows + 3) / 4), dim3(256), 0, stream, lg, rows, F, E, prior,
                         scale, scale_per_example, top_k, out, ids);
      return hipGetLastError();
    };
    return E <= 256 ? select(hr_select_kernel<4>) : select(hr_select_kernel<8>);
  }
  auto go = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3((rows + kRows - 1) / kRows), dim3(64 * kRows), 0, stream, z,
                       rows, F, layer_ids, p, prior, scale, scale_per_example, top_k, out, ids);
    return hipGetLastError();
  };
  if (E <= 256) {
    if (W <= 128) return go(hr_rows_kernel<2, 4>);
    if (W <= 256) return go(hr_rows_kernel<4, 4>);
    return W <= 512 ? go(hr_rows_kernel<8, 4>) : go(hr_rows_kernel<16, 4>);
  }
  if (W <= 128) return go(hr_rows_kernel<2, 8>);
  if (W <= 256) return go(hr_rows_kernel<4, 8>);
  return W <= 512 ? go(hr_rows_kernel<8, 8>) : go(hr_rows_kernel<16, 8>);
}

namespace {
int hr_fail(int code, const char* msg) {
  snprintf(moe_error_buffer(), kErrorBufferBytes, "hidden-residual predictor: %s", msg);
  return code;
}

int hr_check(int32_t N, const moe_hr_predictor_params_v1* p, int32_t top_k) {
  if (!p) return hr_fail(MOE_ERR_NULL, "params is NULL");
  if (!p->enc_w || !p->enc_b || !p->ln_w || !p->ln_b || !p->layer_emb || !p->delta_emb ||
      !p->cls_w || !p->cls_b)
    return hr_fail(MOE_ERR_NULL, "a parameter pointer is NULL");
  if (N < 0) return hr_fail(MOE_ERR_SHAPE, "N < 0");
  if (p->hidden <= 0 || p->hidden % 8 != 0) return hr_fail(MOE_ERR_SHAPE, "hidden % 8 != 0");
  if (p->width < 64 || p->width > kMaxWidth || p->width % 8 != 0)
    return hr_fail(MOE_ERR_SHAPE, "width must be a multiple of 8 in [64, 1024]");
  if (p->num_layers < 1 || p->future_window < 1 || p->future_window > 64)
    return hr_fail(MOE_ERR_SHAPE, "num_layers >= 1 and future_window in [1, 64]");
  if (p->num_experts < 1 || p->num_experts > 512 || top_k < 1 || top_k > p->num_experts ||
      top_k > 64)
    return hr_fail(MOE_ERR_SHAPE, "num_experts in [1, 512] and top_k in [1, min(E, 64)]");
  if (!(p->ln_eps >= 0.0f)) return hr_fail(MOE_ERR_SHAPE, "ln_eps must be >= 0");
  // 32-bit offsets of the buffers and of the four-launch form's sections (asked of either form, so
  // that what is refused does not depend on which one a size takes)
  const int64_t lim = int64_t(1) << 31;
  if ((int64_t)N * p->hidden * 2 >= lim || (int64_t)p->width * p->hidden * 2 >= lim ||
      (int64_t)N * p->future_window * p->width * 2 >= lim ||
      (int64_t)N * p->future_window * (p->num_experts + 1) * 4 >= lim)
    return hr_fail(MOE_ERR_SHAPE, "sizes beyond 2 GiB buffers");
  return MOE_OK;
}
}  // namespace

extern "C" {

int64_t moe_hr_predictor_workspace_bytes_v1(int32_t N, const moe_hr_predictor_params_v1* params) {
  if (!params || N < 0) return -1;
  return hr_predictor_workspace(N, *params);
}

int moe_hr_predictor_v1(const uint16_t* hidden, int32_t N, const int32_t* layer_ids,
                        const moe_hr_predictor_params_v1* params, const float* prior,
                        float residual_scale, const float* scale_per_example, int32_t top_k,
                        void* workspace, int64_t workspace_bytes, float* logits_out,
                        int32_t* topk_ids, void* stream) {
  int rc = hr_check(N, params, top_k);
  if (rc) return rc;
  if (N == 0) return MOE_OK;
  if (!hidden || !layer_ids || !workspace || !topk_ids)
    return hr_fail(MOE_ERR_NULL, "NULL hidden, layer_ids, workspace or topk_ids");
  if (workspace_bytes < hr_predictor_workspace(N, *params))
    return hr_fail(MOE_ERR_WORKSPACE, "workspace too small");
  if (!workspace_aligned(workspace)) return hr_fail(MOE_ERR_WORKSPACE, "workspace must be 256-byte aligned");
  const hipError_t e = launch_hr_predictor(hidden, N, params->hidden, layer_ids, *params, prior,
                                           residual_scale, scale_per_example, top_k, workspace,
                                           logits_out, topk_ids, (hipStream_t)stream);
  if (e != hipSuccess) {
    snprintf(moe_error_buffer(), kErrorBufferBytes, "hidden-residual predictor: HIP error %d (%s)",
             (int)e, hipGetErrorString(e));
    return MOE_ERR_HIP + ((int)e % 100);
  }
  return MOE_OK;
}

}  // extern "C"
