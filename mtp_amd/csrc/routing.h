// Device building blocks of the routing stage, shared by the standalone kernels (router.hip,
// align.hip) and the fused decode routing kernel.
//
// logits_tile: fp32 logits of a TT x TE (token x router-row) tile by one wave in the canonical
//   order (chunk q of 8 bf16 -> lane q % 64; per lane increasing q then k with fma from +0.0f;
//   lanes combined by v += shfl_xor(v, m), m = 32 .. 1). The CPU oracle reproduces this order.
// topk_token: one wave selects the top-k of one token's logits (larger logit first, equal logits
//   -> lower id; vLLM topk_softmax(renormalize=True) semantics,
//   src/mtp_expert_prefetch/tracing/vllm_router_trace.py:4201-4225).
// align_block: one 1024-thread block turns top-k ids into the block-padded expert-grouped slot
//   layout (vLLM moe_align_block_size format, vllm_router_trace.py:19647-19660): experts
//   ascending, slots ascending inside an expert, each group padded to BM with the sentinel
//   num_slots, unused blocks tagged -1.
#pragma once

#include "common.h"

// ---------------------------------------------------------------------------- logits
// NV <= 64 (a power of two) values of partial sums per lane, summed over the lanes by a
// transposed butterfly: at the step of lane mask m every lane keeps the half of its values whose
// index bit matches its own lane bit and adds the partner's (lane ^ m) copy of the same values;
// once one value is left, the remaining masks are plain butterfly steps. Every addition is the
// one the butterfly v += shfl_xor(v, m) makes at that lane (the same two operands, and fp32
// addition is commutative), so the sums are bit-identical to it, with NV - 1 exchanges plus the
// plain steps instead of 6 NV. Afterwards a[0] of lane l is the sum of value l / (64 / NV).
template <int M, int HALF, int N>
MOE_DEV void fold_step(float (&a)[N], int lane) {
  if constexpr (HALF == 0) {
    a[0] = a[0] + xor_partner<M>(a[0]);
  } else {
    const bool up = (lane & M) != 0;
#pragma unroll
    for (int v = 0; v < HALF; ++v) {
      if constexpr (M == 32) {
        const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a[v]),
                                                        __float_as_uint(a[v + HALF]), false, false);
        a[v] = __uint_as_float(r[0]) + __uint_as_float(r[1]);
      } else if constexpr (M == 16) {
        const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(a[v]),
                                                        __float_as_uint(a[v + HALF]), false, false);
        a[v] = __uint_as_float(r[0]) + __uint_as_float(r[1]);
      } else {
        const float keep = up ? a[v + HALF] : a[v];
        a[v] = keep + xor_partner<M>(up ? a[v] : a[v + HALF]);
      }
    }
  }
}
template <int NV>
MOE_DEV void fold_partials(float (&a)[NV], int lane) {
  fold_step<32, NV / 2>(a, lane);
  fold_step<16, NV / 4>(a, lane);
  fold_step<8, NV / 8>(a, lane);
  fold_step<4, NV / 16>(a, lane);
  fold_step<2, NV / 32>(a, lane);
  fold_step<1, NV / 64>(a, lane);
}

template <int TT, int TE>
MOE_DEV void logits_tile(const uint16_t* __restrict__ x, int T, int H, const uint16_t* __restrict__ W,
                         int E, const uint16_t* __restrict__ shared_w, const float* __restrict__ bias,
                         float* __restrict__ logits, int t0, int e0, int lane) {
  const int rows = E + (shared_w ? 1 : 0);
  // Buffer loads: a token or router row outside the tile's range, and chunks past H, read zeros
  // without a memory access, so every iteration issues the same loads (exact wait counts).
  // t0 and e0 are wave-uniform: the resources and row offsets live in scalar registers.
  const __amdgpu_buffer_rsrc_t xr = buf_rsrc(x, (uint32_t)T * (uint32_t)H * 2u);
  const __amdgpu_buffer_rsrc_t wr = buf_rsrc(W, (uint32_t)E * (uint32_t)H * 2u);
  const __amdgpu_buffer_rsrc_t sr = buf_rsrc(shared_w, shared_w ? (uint32_t)H * 2u : 0u);
  uint32_t xo[TT], wo[TE];
#pragma unroll
  for (int i = 0; i < TT; ++i) xo[i] = (t0 + i < T) ? (uint32_t)(t0 + i) * (uint32_t)H * 2u : kOutOfRange;
#pragma unroll
  for (int j = 0; j < TE; ++j) {
    const int e = e0 + j;
    wo[j] = e < E ? (uint32_t)e * (uint32_t)H * 2u : (e == E && shared_w ? 0u : kOutOfRange);
  }
  float acc[TT][TE];
#pragma unroll
  for (int i = 0; i < TT; ++i)
#pragma unroll
    for (int j = 0; j < TE; ++j) acc[i][j] = 0.0f;

  // Lane l owns chunks q = l, l + 64, ... (8 bf16 each) and accumulates them in increasing q;
  // NI iterations of loads are in flight before their arithmetic.
  constexpr int NI = 4;
  const int nq = H / 8;
  for (int q0 = 0; q0 < nq; q0 += 64 * NI) {
    u32x4 xv[NI][TT], wv[NI][TE];
#pragma unroll
    for (int it = 0; it < NI; ++it) {
      const int q = q0 + 64 * it + lane;
      const uint32_t qo = q < nq ? (uint32_t)q * 16u : kOutOfRange;
#pragma unroll
      for (int i = 0; i < TT; ++i) xv[it][i] = buf_ld128(xr, (xo[i] + qo) | (qo & kOutOfRange));
#pragma unroll
      for (int j = 0; j < TE; ++j)
        wv[it][j] = buf_ld128(e0 + j == E ? sr : wr, (wo[j] + qo) | (qo & kOutOfRange));
    }
    __builtin_amdgcn_sched_barrier(0);  // every load of the NI iterations before the first wait
#pragma unroll
    for (int it = 0; it < NI; ++it) {
      if (q0 + 64 * it + lane >= nq) continue;  // no arithmetic past H (keeps the fma chain exact)
#pragma unroll
      for (int el = 0; el < 8; ++el) {
        float wf[TE];
#pragma unroll
        for (int j = 0; j < TE; ++j)
          wf[j] = (el & 1) ? bf16hi_to_f32(wv[it][j][el >> 1]) : bf16lo_to_f32(wv[it][j][el >> 1]);
#pragma unroll
        for (int i = 0; i < TT; ++i) {
          const uint32_t xd = xv[it][i][el >> 1];
          const float xf = (el & 1) ? bf16hi_to_f32(xd) : bf16lo_to_f32(xd);
#pragma unroll
          for (int j = 0; j < TE; ++j) acc[i][j] = __builtin_fmaf(xf, wf[j], acc[i][j]);
        }
      }
    }
  }
#pragma unroll
  for (int i = 0; i < TT; ++i)
#pragma unroll
    for (int j = 0; j < TE; ++j) {
      float v = acc[i][j];
      v = bfly_sum(v);
      acc[i][j] = v;
    }
  if (lane == 0) {
#pragma unroll
    for (int i = 0; i < TT; ++i)
#pragma unroll
      for (int j = 0; j < TE; ++j) {
        const int t = t0 + i, e = e0 + j;
        if (t < T && e < rows) {
          float v = acc[i][j];
          if (bias && e < E) v = v + bias[e];
          logits[(int64_t)t * (E + 1) + e] = v;
        }
      }
  }
}

// logits_tile for H <= 2048 with the TT token rows in LDS (x_lds [TT][H] bf16, rows t0 ..
// t0 + TT - 1 of the batch), in two phases: load() issues every chunk of the wave's TE router
// rows (no dependence on x), compute_store() runs the same chunks per lane, fma order and
// butterfly as logits_tile, so the logits are bit-identical to logits_tile on the same rows.
// AUX: cache policy of the weight loads.
template <int TT, int TE, int NI_ = 4, int AUX = 0>
struct LdsLogitsTile {
  static constexpr int NI = NI_;  // 64 * NI chunks of 8 columns
  u32x4 wv[NI][TE];

  MOE_DEV void load(int H, const uint16_t* __restrict__ W, int E,
                    const uint16_t* __restrict__ shared_w, int e0, int lane) {
    const __amdgpu_buffer_rsrc_t wr = buf_rsrc(W, (uint32_t)E * (uint32_t)H * 2u);
    const __amdgpu_buffer_rsrc_t sr = buf_rsrc(shared_w, shared_w ? (uint32_t)H * 2u : 0u);
    const int nq = H / 8;
#pragma unroll
    for (int j = 0; j < TE; ++j) {
      const int e = e0 + j;
      const uint32_t wo =
          e < E ? (uint32_t)e * (uint32_t)H * 2u : (e == E && shared_w ? 0u : kOutOfRange);
#pragma unroll
      for (int it = 0; it < NI; ++it) {
        const int q = 64 * it + lane;
        const uint32_t qo = q < nq ? (uint32_t)q * 16u : kOutOfRange;
        wv[it][j] = buf_ld128<AUX>(e == E ? sr : wr, (wo + qo) | (qo & kOutOfRange));
      }
    }
  }

  // acc[i * TE + j]: the lane's partial of (token i, row j) over its chunks.
  MOE_DEV void partials(const uint16_t* x_lds, int H, int lane, float (&acc)[TT * TE]) const {
    const int nq = H / 8;
#pragma unroll
    for (int v = 0; v < TT * TE; ++v) acc[v] = 0.0f;
#pragma unroll
    for (int it = 0; it < NI; ++it) {
      const int q = 64 * it + lane;
      if (q >= nq) continue;
      u32x4 xv[TT];
#pragma unroll
      for (int i = 0; i < TT; ++i) xv[i] = ld128(x_lds + i * H + 8 * q);
#pragma unroll
      for (int el = 0; el < 8; ++el) {
        float wf[TE];
#pragma unroll
        for (int j = 0; j < TE; ++j)
          wf[j] = (el & 1) ? bf16hi_to_f32(wv[it][j][el >> 1]) : bf16lo_to_f32(wv[it][j][el >> 1]);
#pragma unroll
        for (int i = 0; i < TT; ++i) {
          const uint32_t xd = xv[i][el >> 1];
          const float xf = (el & 1) ? bf16hi_to_f32(xd) : bf16lo_to_f32(xd);
#pragma unroll
          for (int j = 0; j < TE; ++j)
            acc[i * TE + j] = __builtin_fmaf(xf, wf[j], acc[i * TE + j]);
        }
      }
    }
  }

  MOE_DEV void compute_store(const uint16_t* x_lds, int T, int H, int E, bool has_shared,
                             const float* __restrict__ bias, float* __restrict__ logits, int t0,
                             int e0, int lane) const {
    const int rows = E + (has_shared ? 1 : 0);
    float acc[TT * TE];
    partials(x_lds, H, lane, acc);
#pragma unroll
    for (int v = 0; v < TT * TE; ++v) acc[v] = bfly_sum(acc[v]);
    if (lane == 0) {
#pragma unroll
      for (int i = 0; i < TT; ++i)
#pragma unroll
        for (int j = 0; j < TE; ++j) {
          const int t = t0 + i, e = e0 + j;
          if (t < T && e < rows) {
            float v = acc[i * TE + j];
            if (bias && e < E) v = v + bias[e];
            logits[(int64_t)t * (E + 1) + e] = v;
          }
        }
    }
  }
};

// ---------------------------------------------------------------------------- top-k
// 32-bit order key of a logit: unsigned order = logit order, with -0 equal to +0 and NaN (key 1)
// below every number; key 0 marks "not a candidate" (already selected, or past E).
MOE_DEV uint32_t topk_ord(float v) {
  uint32_t u = __float_as_uint(v);
  if ((u & 0x7FFFFFFFu) == 0u) u = 0u;  // -0 -> +0
  u = (u & 0x80000000u) ? ~u : (u | 0x80000000u);
  return ((__float_as_uint(v) & 0x7FFFFFFFu) > 0x7F800000u) ? 1u : u;
}

// The logit of a key (a NaN for key 1; +0 for either zero).
MOE_DEV float topk_ord_value(uint32_t o) {
  return __uint_as_float((o & 0x80000000u) ? (o & 0x7FFFFFFFu) : ~o);
}

// DPP move with 0 in the lanes a row mask leaves out (0 is the identity of unsigned max, so the
// move and the max fuse into one v_max_u32_dpp).
#define MOE_DPP(v, ctrl, rmask) \
  (uint32_t) __builtin_amdgcn_update_dpp(0, (int)(v), ctrl, rmask, 0xF, false)

// Wave-wide maximum through DPP (quad xor 1, quad xor 2, half-row mirror, row mirror,
// row_bcast15, row_bcast31); the result is read from lane 63 and is wave-uniform.
MOE_DEV uint32_t wave_max_u32(uint32_t v) {
  v = max(v, MOE_DPP(v, 0xB1, 0xF));   // quad_perm(1,0,3,2)
  v = max(v, MOE_DPP(v, 0x4E, 0xF));   // quad_perm(2,3,0,1)
  v = max(v, MOE_DPP(v, 0x141, 0xF));  // row_half_mirror
  v = max(v, MOE_DPP(v, 0x140, 0xF));  // row_mirror
  v = max(v, MOE_DPP(v, 0x142, 0xA));  // row_bcast15 into rows 1, 3
  v = max(v, MOE_DPP(v, 0x143, 0xC));  // row_bcast31 into rows 2, 3
  return (uint32_t)__builtin_amdgcn_readlane((int)v, 63);
}

// One wave: the top_k (<= 64) largest keys, larger key first and equal keys by lower id (the
// reference's tie rule made explicit). key[c] of lane l belongs to id l + 64 c; key 0 marks
// "not a candidate" (there must be at least top_k candidates). A round is a 32-bit wave
// maximum plus one ballot per column to find the lowest id holding it; the selected keys are
// cleared to 0. Lane r < top_k receives the r-th selection (id, key).
template <int MAXC>
MOE_DEV void topk_select_keys(uint32_t (&key)[MAXC], int top_k, int lane, int& my_i,
                              uint32_t& my_key) {
  my_key = 0u;
  my_i = 0;
  for (int r = 0; r < top_k; ++r) {
    uint32_t m = key[0];
#pragma unroll
    for (int c = 1; c < MAXC; ++c) m = max(m, key[c]);
    m = wave_max_u32(m);
    int sel = -1;  // lowest id whose key is the maximum (wave-uniform)
#pragma unroll
    for (int c = 0; c < MAXC; ++c) {
      const uint64_t b = __ballot(key[c] == m);
      if (sel < 0 && b != 0) sel = 64 * c + __ffsll((long long)b) - 1;
    }
#pragma unroll
    for (int c = 0; c < MAXC; ++c)
      if (lane + 64 * c == sel) key[c] = 0u;
    if (lane == r) {
      my_i = sel;
      my_key = m;
    }
  }
}

// One wave: the top_k (<= 64) largest of row[0..E) (E <= 64 * MAXC), larger logit first and
// equal logits by lower id. Lane r < top_k receives the r-th selection (id, logit). Every logit
// is loaded at once (lanes past E read zeros without a memory access and are masked out).
template <int MAXC>
MOE_DEV void topk_select(const float* __restrict__ row, int E, int top_k, int lane, int& my_i,
                         float& my_v) {
  const __amdgpu_buffer_rsrc_t rr = buf_rsrc(row, (uint32_t)E * 4u);
  float v[MAXC];
#pragma unroll
  for (int c = 0; c < MAXC; ++c) v[c] = __uint_as_float(buf_ld32(rr, (uint32_t)(lane + 64 * c) * 4u));
  uint32_t key[MAXC];
#pragma unroll
  for (int c = 0; c < MAXC; ++c)  // masked with an AND: a select of a loaded value would become
                                  // a branch around the load with a wait inside it
    key[c] = topk_ord(v[c]) & (0u - (uint32_t)(lane + 64 * c < E));
  uint32_t my_key;
  topk_select_keys<MAXC>(key, top_k, lane, my_i, my_key);
  my_v = (lane < top_k) ? topk_ord_value(my_key) : 0.0f;
}

// Renormalised weight of lane r's selection: exp(l_r - l_0) / sum_{j < k} exp(l_j - l_0), the sum
// in selection order. Called by a whole wave (the lane reads are v_readlane, not LDS permutes).
MOE_DEV float topk_weight(float my_v, int top_k, int lane) {
  const float vmax = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(my_v), 0));
  const float ex = (lane < top_k) ? expf(my_v - vmax) : 0.0f;
  float s = 0.0f;
  for (int r = 0; r < top_k; ++r)
    s = s + __int_as_float(__builtin_amdgcn_readlane(__float_as_int(ex), r));
  return ex / s;
}

// One wave: top-k of row[0..E) (E <= 64 * MAXC). Writes ids[t*k + r], weights[t*k + r]
// (r < k) and, when has_shared, weights[T*k + t] = sigmoid(row[E]). Optionally mirrors the ids
// to ids_lds.
template <int MAXC>
MOE_DEV void topk_token(const float* __restrict__ row, int E, int top_k, int has_shared, int T,
                        int t, int lane, int32_t* __restrict__ ids, float* __restrict__ weights,
                        int* ids_lds, int32_t* ids_mirror = nullptr) {
  // row[E] when has_shared, else zero; issued with the selection's loads
  const float g = __uint_as_float(
      buf_ld32(buf_rsrc(row, (uint32_t)(E + (has_shared ? 1 : 0)) * 4u), (uint32_t)E * 4u));
  int my_i;
  float my_v;
  topk_select<MAXC>(row, E, top_k, lane, my_i, my_v);
  const float w = topk_weight(my_v, top_k, lane);
  if (lane < top_k) {
    ids[(int64_t)t * top_k + lane] = my_i;
    weights[(int64_t)t * top_k + lane] = w;
    if (ids_lds) ids_lds[t * top_k + lane] = my_i;
    if (ids_mirror) ids_mirror[(int64_t)t * top_k + lane] = my_i;
  }
  if (has_shared && lane == 0) weights[(int64_t)T * top_k + t] = 1.0f / (1.0f + expf(-g));
}

// One wave: top-k of row[0..E) into LDS only (ids_lds[r], w_lds[r] for r < top_k), the same
// selection and weights as topk_token.
template <int MAXC>
MOE_DEV void topk_token_lds(const float* __restrict__ row, int E, int top_k, int lane, int* ids_lds,
                            float* w_lds) {
  int my_i;
  float my_v;
  topk_select<MAXC>(row, E, top_k, lane, my_i, my_v);
  const float w = topk_weight(my_v, top_k, lane);
  if (lane < top_k) {
    ids_lds[lane] = my_i;
    w_lds[lane] = w;
  }
}

// topk_token / topk_token_lds for any E <= 512 (a uniform branch on E).
MOE_DEV void topk_token_any(const float* __restrict__ row, int E, int top_k, int has_shared, int T,
                            int t, int lane, int32_t* __restrict__ ids,
                            float* __restrict__ weights, int* ids_lds,
                            int32_t* ids_mirror = nullptr) {
  if (E <= 256)
    topk_token<4>(row, E, top_k, has_shared, T, t, lane, ids, weights, ids_lds, ids_mirror);
  else
    topk_token<8>(row, E, top_k, has_shared, T, t, lane, ids, weights, ids_lds, ids_mirror);
}
MOE_DEV void topk_token_lds_any(const float* __restrict__ row, int E, int top_k, int lane,
                                int* ids_lds, float* w_lds) {
  if (E <= 256)
    topk_token_lds<4>(row, E, top_k, lane, ids_lds, w_lds);
  else
    topk_token_lds<8>(row, E, top_k, lane, ids_lds, w_lds);
}

// ---------------------------------------------------------------------------- align
constexpr int kAlignWaves = 16;   // align_block needs blockDim.x == 1024
constexpr int kMaxGroups = 513;   // 512 routed experts + the shared expert

struct AlignSmem {
  int cnt[kAlignWaves][kMaxGroups];
  int off[kMaxGroups];
  int pad[kMaxGroups];
  int wtot[16];
};

// Inclusive prefix sum over the 64 lanes of a wave through DPP: row shifts by 1, 2, 4 and 8
// (a lane whose source lies before its row keeps 0), then row_bcast15 into rows 1 and 3 and
// row_bcast31 into rows 2 and 3. Six dependent VALU operations instead of six LDS permutes.
MOE_DEV int wave_incl_sum(int v) {
  v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xF, 0xF, false);  // row_shr:1
  v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xF, 0xF, false);  // row_shr:2
  v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xF, 0xF, false);  // row_shr:4
  v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xF, 0xF, false);  // row_shr:8
  v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xA, 0xF, false);  // row_bcast15
  v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xC, 0xF, false);  // row_bcast31
  return v;
}

// Exclusive prefix sum of v over the threads of a workgroup of at most 16 waves, in thread order,
// and the total. wtot: 16 ints of LDS. Every thread of the workgroup calls it (it synchronises);
// wtot may be reused only after a further barrier.
MOE_DEV int block_excl_sum(int v, int* wtot, int& total) {
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, nw = (blockDim.x + 63) >> 6;
  const int incl = wave_incl_sum(v);
  if (lane == 63) wtot[w] = incl;
  __syncthreads();
  int before = 0, tot = 0;
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const int t = i < nw ? wtot[i] : 0;
    tot += t;
    before += i < w ? t : 0;
  }
  total = tot;
  return before + incl - v;
}

// Division by the (wave-uniform) align block size for n >= 0: a shift when it is a power of two,
// as the kernels' block sizes are, else an integer division (a uniform branch).
struct BlockDiv {
  int bm, sh;
  MOE_DEV explicit BlockDiv(int b) : bm(b), sh((b & (b - 1)) == 0 ? __builtin_ctz(b) : -1) {}
  MOE_DEV int div(int n) const { return sh >= 0 ? (n >> sh) : n / bm; }
  MOE_DEV int pad(int n) const { return div(n + bm - 1) * bm; }  // n rounded up to blocks
};

MOE_DEV int slot_expert(const int32_t* topk_ids, int routed, int E, int f) {
  if (f < routed) {
    const int e = topk_ids[f];
    return (e >= 0 && e < E) ? e : -1;
  }
  return E;  // shared slot
}

// Experts of kAlignIds consecutive chunks of a wave's slot range (slot f = base + 64 u + lane,
// u < kAlignIds), -1 past hi or for an id outside [0, E). The id loads are buffer loads issued
// together (slots past the routed ones read zeros without a memory access), so a batch costs one
// memory latency instead of one per slot.
constexpr int kAlignIds = 8;

MOE_DEV void align_ids(__amdgpu_buffer_rsrc_t ir, int routed, int E, int base, int hi, int lane,
                       int (&e)[kAlignIds]) {
  int raw[kAlignIds];
#pragma unroll
  for (int u = 0; u < kAlignIds; ++u) {
    const int f = base + 64 * u + lane;
    raw[u] = (int)buf_ld32(ir, (f < routed && f < hi) ? (uint32_t)f * 4u : kOutOfRange);
  }
#pragma unroll
  for (int u = 0; u < kAlignIds; ++u) {
    const int f = base + 64 * u + lane;
    const bool routed_ok = f < routed && f < hi && raw[u] >= 0 && raw[u] < E;
    const bool shared = f >= routed && f < hi;  // the shared slots follow the routed ones
    e[u] = routed_ok ? raw[u] : (shared ? E : -1);
  }
}

// Slots of a 64-slot chunk with this lane's expert (e < 0: no slot), from one ballot per id bit.
MOE_DEV uint64_t expert_peers(int e) {
  const bool valid = e >= 0;
  uint64_t peers = __ballot(valid);
#pragma unroll
  for (int bit = 0; bit < 10; ++bit) {
    const bool b = valid && ((e >> bit) & 1);
    const uint64_t bal = __ballot(b);
    peers &= b ? bal : ~bal;
  }
  return peers;
}

// topk_ids in global memory. One workgroup, so what bounds it is its chain of dependent steps.
// Up to kAlignHeld chunks of 64 slots per wave (4096 slots) a wave's ids stay in registers from the
// one load on: the ballot match ranks a chunk's slots and leaves the wave's counts behind, one
// pass over the groups turns the counts into bases, and the slots, the padding and the block ids
// are stored together after the last barrier (a barrier between stores waits for the earlier
// ones). Against counting with LDS atomics, loading the ids a second time and ranking them after
// the padding's stores: eight layers of 48 tokens (64 experts, top-4) 168.5 -> 163.5 us, of 64
// tokens (256 experts, top-8) 524 -> 514 us; one layer of 203 tokens 98.7 -> 97.7 us. Larger
// inputs keep that form: their slots' stores are better spread between the ranks (8192 slots of 512
// experts 13.2 against 15.0 us held, 5000 10.7 against 11.3, 3000 9.1 against 9.0).
// With fill_tail false the entries past the padded total are left as they are, as in align_wave.
constexpr int kAlignHeld = 4;
MOE_DEV void align_block(const int32_t* topk_ids, int T, int top_k, int E, int has_shared, int BM,
                         int cap, int32_t* __restrict__ sorted, int32_t* __restrict__ eids,
                         int32_t* __restrict__ ntpp, AlignSmem& sm, bool fill_tail) {
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int routed = T * top_k;
  const int n_slots = routed + (has_shared ? T : 0);
  const int G = E + (has_shared ? 1 : 0);
  const BlockDiv bd(BM);
  const int per_wave = (((n_slots + kAlignWaves - 1) / kAlignWaves) + 63) / 64 * 64;
  const int lo = min(w * per_wave, n_slots), hi = min(lo + per_wave, n_slots);
  const bool held = per_wave <= 64 * kAlignHeld;  // uniform over the workgroup
  const __amdgpu_buffer_rsrc_t ir = buf_rsrc(topk_ids, (uint32_t)routed * 4u);
  const uint64_t lt_mask = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
  int eb[kAlignIds], rank[kAlignHeld];
  if (held) align_ids(ir, routed, E, lo, hi, lane, eb);
  // every wave clears and fills its own counters: LDS operations of one wave complete in order
  for (int g = lane; g < G; g += 64) sm.cnt[w][g] = 0;
  __builtin_amdgcn_wave_barrier();
  if (held) {
#pragma unroll
    for (int u = 0; u < kAlignHeld; ++u) {
      if (lo + 64 * u >= hi) break;  // uniform over the wave
      const int e = eb[u];
      const uint64_t peers = expert_peers(e);
      const int before = (u > 0 && e >= 0) ? sm.cnt[w][e] : 0;
      rank[u] = before + __popcll(peers & lt_mask);
      __builtin_amdgcn_wave_barrier();  // every lane has read the old count
      if (e >= 0 && (peers & lt_mask) == 0) sm.cnt[w][e] = before + __popcll(peers);
      __builtin_amdgcn_wave_barrier();
    }
  } else {
    for (int base = lo; base < hi; base += 64 * kAlignIds) {
      int e[kAlignIds];
      align_ids(ir, routed, E, base, hi, lane, e);
#pragma unroll
      for (int u = 0; u < kAlignIds; ++u) {
        if (base + 64 * u >= hi) break;  // uniform
        if (e[u] >= 0) atomicAdd(&sm.cnt[w][e[u]], 1);
      }
    }
  }
  __syncthreads();
  // Thread g: group g's size, the exclusive scan of the padded sizes over the groups, and the
  // waves' bases in place of their counts; pad[] keeps the end of the group's real slots.
  int tp;
  {
    int c[kAlignWaves], tot = 0;
#pragma unroll
    for (int v = 0; v < kAlignWaves; ++v) {
      c[v] = tid < G ? sm.cnt[v][tid] : 0;
      tot += c[v];
    }
    const int off = block_excl_sum(bd.pad(tot), sm.wtot, tp);
    if (tid < G) {
      sm.off[tid] = off;
      sm.pad[tid] = off + tot;
      int run = off;
#pragma unroll
      for (int v = 0; v < kAlignWaves; ++v) {
        sm.cnt[v][tid] = run;
        run += c[v];
      }
    }
  }
  __syncthreads();
  const int limit = cap * BM;
  // Stable scatter: ranges in wave order, slots in order inside a range.
  if (held) {
#pragma unroll
    for (int u = 0; u < kAlignHeld; ++u) {
      if (lo + 64 * u >= hi) break;  // uniform over the wave
      if (eb[u] >= 0) {
        const int pos = sm.cnt[w][eb[u]] + rank[u];
        if (pos < limit) sorted[pos] = lo + 64 * u + lane;
      }
    }
  }
  // Four threads per group write its padding sentinels with 16-byte stores (scalar stores for an
  // unaligned head or tail) and its block ids; a group's padded end is the next group's offset.
  const bool vec = (reinterpret_cast<uintptr_t>(sorted) & 15u) == 0;
  for (int g = tid >> 2; g < G; g += 256) {
    const int sub = tid & 3;
    const int off = sm.off[g], real_end = sm.pad[g];
    const int end = g + 1 < G ? sm.off[g + 1] : tp;
    const int fend = min(end, limit);
    const int a4 = vec ? min((real_end + 3) & ~3, fend) : fend;  // vector part [a4, v_end)
    const int v_end = a4 + ((fend - a4) & ~3);
    if (sub == 0) {
      for (int p = real_end; p < a4; ++p) sorted[p] = n_slots;
      for (int p = v_end; p < fend; ++p) sorted[p] = n_slots;
    }
    const i32x4 sent = {n_slots, n_slots, n_slots, n_slots};
    for (int p = a4 + 4 * sub; p < v_end; p += 16) *reinterpret_cast<i32x4*>(&sorted[p]) = sent;
    const int bend = min(bd.div(end), cap);
    for (int b = bd.div(off) + sub; b < bend; b += 4) eids[b] = g;
  }
  if (fill_tail) {
    for (int b = bd.div(tp) + tid; b < cap; b += 1024) eids[b] = -1;
    for (int p = tp + tid; p < limit; p += 1024) sorted[p] = n_slots;
  }
  if (tid == 0) *ntpp = tp;
  if (held) return;

  for (int base0 = lo; base0 < hi; base0 += 64 * kAlignIds) {
    align_ids(ir, routed, E, base0, hi, lane, eb);
#pragma unroll
    for (int u = 0; u < kAlignIds; ++u) {
      const int base = base0 + 64 * u;
      if (base >= hi) break;  // uniform: the rest of the batch lies past the wave's range
      const int e = eb[u];
      const uint64_t peers = expert_peers(e);
      if (e >= 0) {
        const int pos = sm.cnt[w][e] + __popcll(peers & lt_mask);
        if (pos < limit) sorted[pos] = base + lane;
      }
      // wave-local LDS update after every lane has read the old base
      __builtin_amdgcn_wave_barrier();
      if (e >= 0 && (peers & lt_mask) == 0) sm.cnt[w][e] += __popcll(peers);
      __builtin_amdgcn_wave_barrier();
    }
  }
}

// Single-wave align for at most 64 slots (decode step sizes) in blocks of 16; same output as
// align_block up to the padded total, past which nothing is written (the decode kernels never read
// there: every block checks the padded total first). Lane f holds slot f: the slots of one expert
// are found with a ballot match over the expert id bits and the lowest lane of each group is its
// leader. Each leader writes its group's padded size into an LDS table indexed by group id; one
// exclusive scan of the table by the wave gives every group's offset (groups in ascending id
// order), so the cost does not grow with the number of distinct experts. The table's runs are held
// in registers between the two passes, and the layout is put together in LDS and stored in whole
// lines (eight layers of 8 tokens 265 -> 260 us).
constexpr int kAlignWaveMaxSlots = 64;
constexpr int kAlignWaveBlock = 16;
constexpr int kAlignWaveRun = (kMaxGroups + 63) / 64;  // groups per lane
struct AlignWaveSmem {
  int pad[64 * kAlignWaveRun];
  __attribute__((aligned(16))) int sorted[kAlignWaveMaxSlots * kAlignWaveBlock];
};

MOE_DEV void align_wave(const int32_t* topk_ids, int T, int top_k, int E, int has_shared, int cap,
                        int32_t* __restrict__ sorted, int32_t* __restrict__ eids,
                        int32_t* __restrict__ ntpp, int lane, AlignWaveSmem& sm) {
  constexpr int BM = kAlignWaveBlock;
  const int routed = T * top_k;
  const int n_slots = routed + (has_shared ? T : 0);
  const int e = (lane < n_slots) ? slot_expert(topk_ids, routed, E, lane) : -1;
  const bool valid = e >= 0;
#pragma unroll
  for (int i = 0; i < kAlignWaveRun; ++i) sm.pad[64 * i + lane] = 0;
  const i32x4 sent = {n_slots, n_slots, n_slots, n_slots};
#pragma unroll
  for (int i = 0; i < BM / 4; ++i) *reinterpret_cast<i32x4*>(&sm.sorted[4 * (64 * i + lane)]) = sent;
  const uint64_t peers = expert_peers(e);
  const uint64_t lt_mask = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
  const int rank = __popcll(peers & lt_mask);
  const bool leader = valid && rank == 0;
  const int padded = (__popcll(peers) + BM - 1) / BM * BM;
  __builtin_amdgcn_wave_barrier();  // one wave: LDS operations complete in order
  if (leader) sm.pad[e] = padded;
  __builtin_amdgcn_wave_barrier();
  // lane l owns the table's run of kAlignWaveRun groups
  int run[kAlignWaveRun], local = 0;
#pragma unroll
  for (int i = 0; i < kAlignWaveRun; ++i) run[i] = sm.pad[kAlignWaveRun * lane + i];
#pragma unroll
  for (int i = 0; i < kAlignWaveRun; ++i) local += run[i];
  const int incl = wave_incl_sum(local);
  const int total = __builtin_amdgcn_readlane(incl, 63);
  int at = incl - local;
  __builtin_amdgcn_wave_barrier();
#pragma unroll
  for (int i = 0; i < kAlignWaveRun; ++i) {
    sm.pad[kAlignWaveRun * lane + i] = at;
    at += run[i];
  }
  __builtin_amdgcn_wave_barrier();
  const int off = valid ? sm.pad[e] : 0;
  if (valid) sm.sorted[off + rank] = lane;  // off + rank < total <= 16 n_slots
  if (leader) {
    const int b1 = min((off + padded) / BM, cap);
    for (int b = off / BM; b < b1; ++b) eids[b] = e;
  }
  __builtin_amdgcn_wave_barrier();
  const int end = min(total, cap * BM);
  for (int p = 4 * lane; p < end; p += 256)
    *reinterpret_cast<i32x4*>(&sorted[p]) = *reinterpret_cast<const i32x4*>(&sm.sorted[p]);
  if (lane == 0) *ntpp = total;
}
