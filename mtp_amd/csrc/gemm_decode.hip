// Decode path (token batches up to a few hundred slots): grouped int4 GEMM on MFMA with the
// int4 weights dequantised in registers directly into the MFMA B operand.
//
// Tile = 16 slots (the M dimension of v_mfma_f32_16x16x32_bf16) x 16*CT columns x a K range,
// computed by one wave.
//
// B operand: lane l of a wave holds, for k-step s (32 k), the packed int32 row
// r = s*4 + (l >> 4) at columns cl .. cl + CT - 1 with cl = c0 + CT*(l & 15) (one 8- or 16-byte
// nontemporal load; 16 lanes read 16*CT*4 contiguous bytes of a row). One packed int32 is
// exactly the 8 k-values one lane contributes to a 16x16x32 MFMA, so each int32 becomes one B
// fragment: bf16 "magic" pairs 128 + q built from two byte planes of the word (weight_frag)
// give the k order [0,2,4,6,1,3,5,7]; the A fragment (activations) is loaded as 8 consecutive
// bf16 and permuted to the same order (v_perm), so the dot products are unchanged. N-subtile j
// of a lane holds column cl + j.
//
// Zero point and scale are applied per quantisation group g on fp32 partial sums:
//   y[m, n] = sum_g s[g, n] * ( sum_{k in g} x[m, k] (128 + q[k, n]) - (128 + z[g, n]) X[m, g] )
// with X[m, g] = sum_{k in g} x[m, k] produced by one extra MFMA against an all-ones B.
// All weight products are exact; the only difference from the reference's dequantise-then-
// matmul is that the reference rounds each (q - z) * s to bf16 first.
//
// Kernels:
//  * gemm_decode_kernel: block = one 16-slot expert block x one column tile; KS waves split K
//    and are summed through LDS in wave order (deterministic).
//    W1 (gate_up): A = x[token(slot)], gate and up tiles, epilogue h = bf16(silu(g) * u).
//    W2 (down):    A = h[slot], epilogue ys[slot, n] = w[slot] * y (fp32).
//  * w2_token_sum_kernel (up to 8 tokens): block = one token x one column tile, wave i =
//    the token's routed slot i (or its shared slot); the weighted rows are summed in slot order
//    inside the block, so no separate sum kernel runs.
// Arithmetic references: src/mtp_expert_prefetch/tracing/vllm_wna16_group_plan.py:367-486,
// src/mtp_expert_prefetch/repack/gptq_unpack.py:88-131, 247-256, and the moe_sum order of
// src/mtp_expert_prefetch/tracing/vllm_router_trace.py:19801-19804.
#include <math.h>

#include <type_traits>

#include "common.h"
#include "launch.h"
#include "routing.h"

namespace {

typedef __bf16 bf16x8_v __attribute__((ext_vector_type(8)));

constexpr int kBM = kDecodeBlockM;  // 16 slots
constexpr int kW2Groups = 4;        // fused W2: 64-column groups of the output per wave
constexpr uint32_t kOnes = 0x3F803F80u;

enum { DEC_W1 = 1, DEC_W2 = 2 };

MOE_DEV bf16x8_v as_frag(uint32_t a, uint32_t b, uint32_t c, uint32_t d) {
  u32x4 v = {a, b, c, d};
  return __builtin_bit_cast(bf16x8_v, v);
}

// B fragment of one packed int32 (8 k of one column) in the k order [0,2,4,6,1,3,5,7]: the
// nibbles are split into two byte planes (even nibbles q0 q2 q4 q6, odd nibbles q1 q3 q5 q7),
// and each bf16 pair (128 + q_a, 128 + q_b) is one byte permute of a plane with the magic
// exponent byte 0x43: 7 VALU operations per word.
constexpr uint32_t kMagicBytes = 0x43434343u;
MOE_DEV bf16x8_v weight_frag(uint32_t w) {
  const uint32_t ev = w & 0x0F0F0F0Fu;         // bytes q0, q2, q4, q6
  const uint32_t od = (w >> 4) & 0x0F0F0F0Fu;  // bytes q1, q3, q5, q7
  return as_frag(__builtin_amdgcn_perm(ev, kMagicBytes, 0x00050004u),   // (q0, q2)
                 __builtin_amdgcn_perm(ev, kMagicBytes, 0x00070006u),   // (q4, q6)
                 __builtin_amdgcn_perm(od, kMagicBytes, 0x00050004u),   // (q1, q3)
                 __builtin_amdgcn_perm(od, kMagicBytes, 0x00070006u));  // (q5, q7)
}

// A fragment of 8 consecutive bf16 activations (d0 = x0|x1<<16, ..., d3 = x6|x7<<16) in the
// k order of weight_frag: (x0,x2), (x4,x6), (x1,x3), (x5,x7).
MOE_DEV bf16x8_v act_frag(const u32x4 d) {
  return as_frag(__builtin_amdgcn_perm(d[1], d[0], 0x05040100u),
                 __builtin_amdgcn_perm(d[3], d[2], 0x05040100u),
                 __builtin_amdgcn_perm(d[1], d[0], 0x07060302u),
                 __builtin_amdgcn_perm(d[3], d[2], 0x07060302u));
}

// Everything one lane needs for one quantisation group (SPG MFMA k-steps of 32): activations
// and packed weights, and the group's scales and zeros.
template <int NP, int SPG, int CT>
struct GroupAW {
  u32x4 a[SPG];                 // 8 consecutive bf16 activations per k-step
  uint32_t w[NP][SPG][CT];      // packed int4 rows, CT columns
};
template <int NP, int CT>
struct GroupSZ {
  uint32_t s[NP][CT / 2];       // fp16 scale pairs of the CT columns
  uint32_t z[NP];               // packed zeros word holding the CT columns
};

// A operand of one lane: resource over the activation rows and the byte offset of
// (this lane's row, first k of the wave's slice + 8 * kq), kOutOfRange for a padding row.
struct AView {
  __amdgpu_buffer_rsrc_t r;
  uint32_t off;
};

// One wave's view of a K slice [k0, k0 + NGW*G) of the NP projections at columns
// cl .. cl + CT - 1. Every load is a buffer load from a uniform resource with a 32-bit lane
// offset; padding rows load zeros with no memory access, so the same instructions run on every
// path.
template <int NP, int SPG, int CT>
struct DecodeTile {
  __amdgpu_buffer_rsrc_t qr[NP], sr[NP], zr[NP];
  AView a;
  uint32_t qoff, soff, zoff;        // lane offsets of group 0
  uint32_t qgrp, sgrp, zgrp, qrow;  // bytes per group (qweight, scales, zeros), per packed row
  int G, zshift;

  MOE_DEV DecodeTile(const ProjDev (&pj)[NP], AView av, int NOUT, int G_, int k0, int cl,
                     int kq)
      : a(av), G(G_), zshift(4 * (cl & 7)) {
#pragma unroll
    for (int p = 0; p < NP; ++p) {
      qr[p] = buf_rsrc(pj[p].qweight);
      sr[p] = buf_rsrc(pj[p].scales);
      zr[p] = buf_rsrc(pj[p].qzeros);
    }
    qrow = (uint32_t)NOUT * 4u;
    qoff = (uint32_t)(k0 / 8 + kq) * qrow + (uint32_t)cl * 4u;
    soff = (uint32_t)((k0 / G) * NOUT + cl) * 2u;
    zoff = (uint32_t)((k0 / G) * (NOUT / 8) + (cl >> 3)) * 4u;
    qgrp = (uint32_t)(G / 8) * qrow;
    sgrp = (uint32_t)NOUT * 2u;
    zgrp = (uint32_t)(NOUT / 8) * 4u;
  }

  // A lane's offsets stay the same for the whole slice; what moves from group to group and from
  // k-step to k-step is uniform and goes into the loads' scalar offset (with the scales in the ring
  // and one projection's group sums at a time: 190 -> 178 VGPRs in W1 with four columns per lane;
  // eight layers of 64 tokens 509.6 -> 506.6 us, one layer of 203 95.2 -> 94.6 us).
  MOE_DEV void load_aw(GroupAW<NP, SPG, CT>& B, int gi) const {
    const uint32_t ug = (uint32_t)gi;
#pragma unroll
    for (int s = 0; s < SPG; ++s)
      B.a[s] = buf_ld128(a.r, a.off + (uint32_t)(64 * s), ug * (uint32_t)G * 2u);
#pragma unroll
    for (int p = 0; p < NP; ++p) {
#pragma unroll
      for (int s = 0; s < SPG; ++s) {  // weights are streamed once: nontemporal
        const uint32_t so = ug * qgrp + (uint32_t)(4 * s) * qrow;
        if constexpr (CT == 2) {
          const u32x2 v = buf_ld64<kBufNontemporal>(qr[p], qoff, so);
          B.w[p][s][0] = v[0];
          B.w[p][s][1] = v[1];
        } else {
          const u32x4 v = buf_ld128<kBufNontemporal>(qr[p], qoff, so);
#pragma unroll
          for (int j = 0; j < 4; ++j) B.w[p][s][j] = v[j];
        }
      }
    }
  }

  MOE_DEV void load_sz(GroupSZ<NP, CT>& B, int gi) const {
    const uint32_t ug = (uint32_t)gi;
#pragma unroll
    for (int p = 0; p < NP; ++p) {
      if constexpr (CT == 2) {
        B.s[p][0] = buf_ld32(sr[p], soff, ug * sgrp);
      } else {
        const u32x2 v = buf_ld64(sr[p], soff, ug * sgrp);
        B.s[p][0] = v[0];
        B.s[p][1] = v[1];
      }
      B.z[p] = buf_ld32(zr[p], zoff, ug * zgrp);  // shifted at use: no wait here
    }
  }

  // acc[p*CT + j] += s * (sum_k x (128 + q) - (128 + z) * sum_k x) over one group.
  MOE_DEV void compute(const GroupAW<NP, SPG, CT>& B, const GroupSZ<NP, CT>& Z,
                       f32x4 (&acc)[NP * CT]) const {
    const bf16x8_v ones = as_frag(kOnes, kOnes, kOnes, kOnes);
    f32x4 tx = {0.f, 0.f, 0.f, 0.f};
    bf16x8_v av[SPG];
#pragma unroll
    for (int s = 0; s < SPG; ++s) {
      av[s] = act_frag(B.a[s]);
      tx = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av[s], ones, tx, 0, 0, 0);
    }
    // one projection after the other: the group sums of one are held at a time
#pragma unroll
    for (int p = 0; p < NP; ++p) {
      f32x4 tmp[CT];
#pragma unroll
      for (int j = 0; j < CT; ++j) tmp[j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int s = 0; s < SPG; ++s) {
#pragma unroll
        for (int j = 0; j < CT; ++j)
          tmp[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av[s], weight_frag(B.w[p][s][j]),
                                                           tmp[j], 0, 0, 0);
      }
#pragma unroll
      for (int j = 0; j < CT; ++j) {
        const uint32_t s2 = Z.s[p][j >> 1];
        const float sc = f16_to_f32((j & 1) ? (s2 >> 16) : (s2 & 0xFFFFu));
        const float zb = kMagicBias + (float)((Z.z[p] >> (zshift + 4 * j)) & 0xFu);
#pragma unroll
        for (int i = 0; i < 4; ++i)
          acc[p * CT + j][i] =
              __builtin_fmaf(sc, __builtin_fmaf(-zb, tx[i], tmp[j][i]), acc[p * CT + j][i]);
      }
    }
  }
};

// Compile-time loop: f(std::integral_constant<int, I>) for I in [B, E).
template <int B, int E, typename F>
MOE_DEV void static_for(F&& f) {
  if constexpr (B < E) {
    f(std::integral_constant<int, B>{});
    static_for<B + 1, E>(f);
  }
}

// One wave: acc[p*CT + j] += A[16 rows, k0 : k0+klen] . W_p[k0 : k0+klen, cl + j] for the NP
// projections over a slice of exactly NGW groups, as straight-line code with a ring of DEPTH
// buffers (DEPTH == NGW: all loads up front): groups g + 1 .. g + DEPTH - 1 are in flight while
// group g is multiplied. Without a loop back-edge each wait is for exactly the group about to be
// multiplied, whatever the ring depth.
template <int NP, int SPG, int CT, int NGW, int DEPTH>
MOE_DEV void decode_tile(const DecodeTile<NP, SPG, CT>& tile, f32x4 (&acc)[NP * CT]) {
  static_assert(DEPTH >= 1 && DEPTH <= NGW, "ring depth within the slice");
  GroupSZ<NP, CT> sz[DEPTH];
  GroupAW<NP, SPG, CT> ring[DEPTH];
  static_for<0, DEPTH - 1>([&](auto gc) {
    tile.load_sz(sz[gc.value], gc.value);
    tile.load_aw(ring[gc.value], gc.value);
  });
  static_for<0, NGW>([&](auto gc) {
    constexpr int g = gc.value;
    if constexpr (g + DEPTH - 1 < NGW) {
      __builtin_amdgcn_s_setprio(2);  // issue the stage's loads ahead of the other waves' math
      tile.load_sz(sz[(g + DEPTH - 1) % DEPTH], g + DEPTH - 1);
      tile.load_aw(ring[(g + DEPTH - 1) % DEPTH], g + DEPTH - 1);
      __builtin_amdgcn_s_setprio(0);
    }
    __builtin_amdgcn_sched_barrier(0);  // this stage's loads before the wait for group g
    tile.compute(ring[g % DEPTH], sz[g % DEPTH], acc);
  });
}

MOE_DEV void projections(const ExpertsDev& ed, int mode, bool is_shared, ProjDev* pj) {
  if (mode == DEC_W1) {
    pj[0] = is_shared ? ed.sgate : ed.gate;
    pj[1] = is_shared ? ed.sup : ed.up;
  } else {
    pj[0] = is_shared ? ed.sdown : ed.down;
  }
}

// Block = one 16-slot expert block x (16 * CT) columns; KS waves split K evenly (each slice a
// whole number of quantisation groups) and are summed through LDS in wave order. Every wave adds
// and finishes its share of the tile (EPW of a lane's four rows x JPW of its columns): with wave 0
// alone doing it, the sums, SiLUs and stores of the whole tile were a serial tail of each
// workgroup (eight layers: of one token 160 -> 156 us, of 64 518 -> 508 us; of 48 with 64 experts
// 159 -> 153 us; one layer of 203 tokens 97.4 -> 95.5 us).
// A wave's slice has exactly NGW groups, loaded through an NB-deep ring (NB == NGW: all up front).
// FW2 (W1 on the slot grid, CT == 2): W2 fused in. The block's 32 h columns are the K rows
// [32 x, 32 x + 32) of the down projection (inside one quantisation group); after the W1
// epilogue every wave multiplies the block's h rows (from LDS) by its kW2Groups x 64 output
// columns and writes the weighted fp32 partial rows ys[slot][x][n] (partial_sum adds them).
// The workgroup of a dropped expert writes zero rows, so every partial row is written.
template <int MODE, int SPG, int KS, int CT, int NB, int NGW, bool FW2 = false>
__global__ __launch_bounds__(64 * KS) void gemm_decode_kernel(
    const uint16_t* __restrict__ act, ExpertsDev ed, SlotsDev sd,
    const int32_t* __restrict__ sorted, const int32_t* __restrict__ eids,
    const int32_t* __restrict__ ntpp, const float* __restrict__ topk_w,
    uint16_t* __restrict__ h_out, float* __restrict__ ys, SlotGrid sg) {
  constexpr int NP = (MODE == DEC_W1) ? 2 : 1;  // projections (gate, up) or (down)
  constexpr int NT = NP * CT;                    // MFMA N-subtiles per lane
  constexpr int TW = 16 * CT;                    // columns per block
  static_assert(!FW2 || (MODE == DEC_W1 && CT == 2), "fused W2: W1 blocks of 32 columns");
  constexpr int EPW = KS >= 4 ? 1 : 4 / KS;             // rows per lane that a wave finishes
  constexpr int JPW = KS > 4 ? CT * 4 / KS : CT;        // columns per lane that it finishes
  static_assert(JPW >= 1 && EPW * JPW * KS == 4 * CT, "an even share of the tile for every wave");
  __shared__ float red[KS > 1 ? KS * NT * 4 * 64 : 1];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // uniform: scalar K-slice offsets
  const int el0 = KS >= 4 ? wave * 4 / KS : wave * EPW;  // this wave's share of the tile
  const int j0 = KS > 4 ? (wave % (KS / 4)) * JPW : 0;
  constexpr int NF = FW2 ? 4 : EPW;  // fused W2: every wave writes all the rows
  int e, f_m, f_out[NF];  // expert; A row of this lane; the D rows of this lane that it writes
  __shared__ float s_w[kSlotGridMaxSlots + kTopkAlignMaxTokens];  // slot grid: routed weights
  if (sg.active) {
    // Slot grid (SlotGrid in launch.h): slots from the routed ids, no align pass.
    __shared__ int s_ids[kSlotGridMaxSlots];
    __shared__ int s_rows[kBM];
    const int E = ed.num_experts, routed = sd.T * sd.top_k, n_slots = sd.num_slots;
    if (sg.logits) {  // every workgroup computes the same top-k of the (at most 8) tokens
      for (int t = wave; t < sd.T; t += KS) {
        const float* row = sg.logits + (int64_t)t * (E + 1);
        const bool shared = n_slots > routed;  // row[E] is the shared gate's logit
        const float g = __uint_as_float(
            buf_ld32(buf_rsrc(row, (uint32_t)(E + (shared ? 1 : 0)) * 4u), (uint32_t)E * 4u));
        topk_token_lds_any(row, E, sd.top_k, lane, s_ids + t * sd.top_k, s_w + t * sd.top_k);
        if (shared && lane == 0) s_w[routed + t] = 1.0f / (1.0f + expf(-g));
      }
    } else {
      if (tid < routed) s_ids[tid] = sg.ids[tid];
      if (FW2 && tid < n_slots) s_w[tid] = sg.weights[tid];
    }
    __syncthreads();
    if (sg.logits && blockIdx.x == 0 && blockIdx.y == 0) {  // publish for W2 and the caller
      if (tid < routed) sg.ids[tid] = s_ids[tid];
      if (tid < n_slots) sg.weights[tid] = s_w[tid];
    }
    const int b = blockIdx.y;  // slot index
    auto expert_of = [&](int f) { return f < routed ? s_ids[f] : E; };
    e = expert_of(b);
    const uint64_t mask = __ballot(lane < n_slots && expert_of(lane) == e);
    const int rank_b = __popcll(mask & ((1ull << b) - 1));  // occurrences of e before slot b
    if constexpr (!FW2) {
      if (rank_b % kBM != 0 || !expert_ok(ed, e)) return;  // uniform over the workgroup
    } else {
      if (rank_b % kBM != 0) return;  // a dropped expert still writes its (zero) partial rows
    }
    const int rank = __popcll(mask & ((1ull << lane) - 1));
    if (wave == 0 && ((mask >> lane) & 1) && rank >= rank_b && rank < rank_b + kBM)
      s_rows[rank - rank_b] = lane;
    const int cnt = min(__popcll(mask) - rank_b, kBM);
    __syncthreads();
    f_m = (lane & 15) < cnt ? s_rows[lane & 15] : n_slots;
#pragma unroll
    for (int i = 0; i < NF; ++i) {
      const int r = 4 * (lane >> 4) + (FW2 ? 0 : el0) + i;
      f_out[i] = r < cnt ? s_rows[r] : n_slots;
    }
    if constexpr (FW2) {
      if (!expert_ok(ed, e)) {  // dropped slots: zero partial rows for this column block
        const int H = ed.hidden, q4 = H / 4;
        for (int i = tid; i < cnt * q4; i += blockDim.x)
          *reinterpret_cast<float4*>(ys + ((int64_t)s_rows[i / q4] * gridDim.x + blockIdx.x) * H +
                                     4 * (i % q4)) = float4{0.f, 0.f, 0.f, 0.f};
        return;
      }
    }
  } else {
    // Block metadata: every load below is in bounds for any b < gridDim.y, so all of them are
    // issued together (one memory latency before the first weight load, not a chain).
    const int b = blockIdx.y;
    const int n_padded = *ntpp;
    e = eids[b];
    f_m = sorted[b * kBM + (lane & 15)];
#pragma unroll
    for (int i = 0; i < NF; ++i) f_out[i] = sorted[b * kBM + 4 * (lane >> 4) + el0 + i];
    if (b * kBM >= n_padded || !expert_ok(ed, e)) return;
  }

  const int G = ed.group;
  const int K = (MODE == DEC_W1) ? ed.hidden : ed.inter;
  const int NOUT = (MODE == DEC_W1) ? ed.inter : ed.hidden;
  const bool is_shared = (e == ed.num_experts);
  const int64_t row = is_shared ? 0 : expert_row(ed, e);
  ProjDev pj[NP];
  projections(ed, MODE, is_shared, pj);
#pragma unroll
  for (int p = 0; p < NP; ++p)
    pj[p] = proj_row(pj[p], is_shared ? 0 : ed.row_stride, row, K / 8, K / G, NOUT);

  const int kslice = K / KS;
  const int kw0 = wave * kslice;
  const int m = lane & 15, kq = lane >> 4;
  const bool valid_m = (unsigned)f_m < (unsigned)sd.num_slots;
  const uint32_t arow = valid_m ? ((MODE == DEC_W1) ? (uint32_t)slot_token(sd, f_m) : (uint32_t)f_m) : 0u;
  const uint32_t a_rows = (MODE == DEC_W1) ? (uint32_t)sd.T : (uint32_t)sd.num_slots;
  const AView av{buf_rsrc(act, a_rows * (uint32_t)K * 2u),
                 valid_m ? (arow * (uint32_t)K + (uint32_t)(kw0 + 8 * kq)) * 2u : kOutOfRange};
  const int cl = blockIdx.x * TW + CT * m;  // this lane's first column
  const DecodeTile<NP, SPG, CT> tile(pj, av, NOUT, G, kw0, cl, kq);

  // FW2: the down projection's words, scales and zeros for this wave's output columns, loaded
  // with the W1 stream. Lane (c = lane & 15, kq) takes packed row x * 4 + kq (TW == 32) and the
  // 4 columns n0 + 4 c .. + 3 of each 64-column group: word t is the B fragment of MFMA tile t.
  [[maybe_unused]] u32x4 w2q[FW2 ? kW2Groups : 1];
  [[maybe_unused]] u32x2 w2s[FW2 ? kW2Groups : 1];
  [[maybe_unused]] uint32_t w2z[FW2 ? kW2Groups : 1];
  [[maybe_unused]] int w2n0 = 0;
  if constexpr (FW2) {
    const int I = ed.inter, H = ed.hidden;
    ProjDev pd[1];
    projections(ed, DEC_W2, is_shared, pd);
    pd[0] = proj_row(pd[0], is_shared ? 0 : ed.row_stride, row, I / 8, I / G, H);
    const int k0 = blockIdx.x * TW, g2 = k0 / G;
    w2n0 = wave * (kW2Groups * 64) + 4 * m;
    const __amdgpu_buffer_rsrc_t q2 = buf_rsrc(pd[0].qweight), s2 = buf_rsrc(pd[0].scales),
                                 z2 = buf_rsrc(pd[0].qzeros);
#pragma unroll
    for (int gi = 0; gi < kW2Groups; ++gi) {
      const uint32_t n = (uint32_t)(w2n0 + 64 * gi);
      w2q[gi] = buf_ld128<kBufNontemporal>(q2, ((uint32_t)(k0 / 8 + kq) * (uint32_t)H + n) * 4u);
      w2s[gi] = buf_ld64(s2, ((uint32_t)g2 * (uint32_t)H + n) * 2u);
      w2z[gi] = buf_ld32(z2, ((uint32_t)g2 * (uint32_t)(H / 8) + (n >> 3)) * 4u);
    }
    __builtin_amdgcn_sched_barrier(0);  // issued here, with the W1 stream, not at their use
  }

  // the rows' routed weights, in flight with the weight stream (their first use is the epilogue)
  [[maybe_unused]] float w_out[EPW];
  if constexpr (MODE == DEC_W2) {
    const __amdgpu_buffer_rsrc_t wr = buf_rsrc(topk_w, (uint32_t)sd.num_slots * 4u);
#pragma unroll
    for (int i = 0; i < EPW; ++i)  // a padding row's offset lies past the end: zero
      w_out[i] = __uint_as_float(buf_ld32(wr, (uint32_t)f_out[i] * 4u));
    __builtin_amdgcn_sched_barrier(0);
  }

  f32x4 acc[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
  decode_tile<NP, SPG, CT, NGW, NB>(tile, acc);

  // This wave's share: fin[p][i][j] = element el0 + i of N-subtile j0 + j of projection p, the
  // waves' partial sums added in wave order.
  float fin[NP][EPW][JPW];
  if constexpr (KS > 1) {
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i) red[((wave * NT + t) * 4 + i) * 64 + lane] = acc[t][i];
    __syncthreads();
#pragma unroll
    for (int p = 0; p < NP; ++p)
#pragma unroll
      for (int i = 0; i < EPW; ++i)
#pragma unroll
        for (int j = 0; j < JPW; ++j) {
          const float* src = red + ((p * CT + j0 + j) * 4 + el0 + i) * 64 + lane;
          float v = src[0];
#pragma unroll
          for (int w = 1; w < KS; ++w) v += src[w * NT * 4 * 64];
          fin[p][i][j] = v;
        }
  } else {
#pragma unroll
    for (int p = 0; p < NP; ++p)
#pragma unroll
      for (int i = 0; i < EPW; ++i)
#pragma unroll
        for (int j = 0; j < JPW; ++j) fin[p][i][j] = acc[p * CT + j][i];
  }

  if constexpr (FW2) {
    // h rows of the block (bf16, as W1 writes them) into LDS as [16 rows][32 columns]
    __shared__ __attribute__((aligned(16))) uint16_t s_h[kBM * TW];
#pragma unroll
    for (int i = 0; i < EPW; ++i) {
      int f = f_out[0];  // f_out[el0 + i] without an indexed register read
#pragma unroll
      for (int r = 1; r < NF; ++r) f = el0 + i == r ? f_out[r] : f;
      const bool real = (unsigned)f < (unsigned)sd.num_slots;
#pragma unroll
      for (int j = 0; j < JPW; ++j)
        s_h[(4 * kq + el0 + i) * TW + CT * m + j0 + j] =
            real ? (uint16_t)f32_to_bf16_rne(silu_f32(fin[0][i][j]) * fin[1][i][j]) : 0;
    }
    __syncthreads();
    // A: row m, k 8 kq .. 8 kq + 7 of the block's 32 h columns; X[row] = sum of the row's h
    const u32x4 hv = ld128(s_h + m * TW + 8 * kq);
    const bf16x8_v av2 = act_frag(hv);
    const f32x4 tx = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
        av2, as_frag(kOnes, kOnes, kOnes, kOnes), f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    const int H = ed.hidden, nct = gridDim.x;
    float wrow[4];
#pragma unroll
    for (int el = 0; el < 4; ++el)
      wrow[el] = (unsigned)f_out[el] < (unsigned)sd.num_slots ? s_w[f_out[el]] : 0.0f;
#pragma unroll
    for (int gi = 0; gi < kW2Groups; ++gi) {
      f32x4 d[4];
#pragma unroll
      for (int t = 0; t < 4; ++t)
        d[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av2, weight_frag(w2q[gi][t]),
                                                       f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
      const int n = w2n0 + 64 * gi;
      float sc[4], zb[4];
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        sc[t] = f16_to_f32(t & 2 ? ((t & 1) ? (w2s[gi][1] >> 16) : (w2s[gi][1] & 0xFFFFu))
                                 : ((t & 1) ? (w2s[gi][0] >> 16) : (w2s[gi][0] & 0xFFFFu)));
        zb[t] = kMagicBias + (float)((w2z[gi] >> (4 * ((n & 7) + t))) & 0xFu);
      }
#pragma unroll
      for (int el = 0; el < 4; ++el) {
        const int f = f_out[el];
        if ((unsigned)f >= (unsigned)sd.num_slots) continue;
        float4 v;
        v.x = wrow[el] * (sc[0] * __builtin_fmaf(-zb[0], tx[el], d[0][el]));
        v.y = wrow[el] * (sc[1] * __builtin_fmaf(-zb[1], tx[el], d[1][el]));
        v.z = wrow[el] * (sc[2] * __builtin_fmaf(-zb[2], tx[el], d[2][el]));
        v.w = wrow[el] * (sc[3] * __builtin_fmaf(-zb[3], tx[el], d[3][el]));
        *reinterpret_cast<float4*>(ys + ((int64_t)f * nct + blockIdx.x) * H + n) = v;
      }
    }
    return;
  }

  // D[i][j] of a 16x16 tile: lane j + 16*(i/4), element i%4 -> row 4*(lane>>4)+el; N-subtile t
  // of projection p holds column cl + t.
#pragma unroll
  for (int i = 0; i < EPW; ++i) {
    const int f = f_out[i];
    if ((unsigned)f >= (unsigned)sd.num_slots) continue;
    const int64_t o = (int64_t)f * NOUT + cl + j0;
    if constexpr (MODE == DEC_W1) {
      float hv[JPW];
#pragma unroll
      for (int j = 0; j < JPW; ++j) hv[j] = silu_f32(fin[0][i][j]) * fin[1][i][j];
      if constexpr (JPW == 1) {
        h_out[o] = (uint16_t)f32_to_bf16_rne(hv[0]);
      } else if constexpr (JPW == 2) {
        *reinterpret_cast<uint32_t*>(h_out + o) = pack_bf16x2(hv[0], hv[1]);
      } else {
        *reinterpret_cast<u32x2*>(h_out + o) =
            u32x2{pack_bf16x2(hv[0], hv[1]), pack_bf16x2(hv[2], hv[3])};
      }
    } else {
      const float w = w_out[i];
      if constexpr (JPW == 1) {
        ys[o] = w * fin[0][i][0];
      } else if constexpr (JPW == 2) {
        *reinterpret_cast<float2*>(ys + o) = float2{w * fin[0][i][0], w * fin[0][i][1]};
      } else {
        *reinterpret_cast<float4*>(ys + o) = float4{w * fin[0][i][0], w * fin[0][i][1],
                                                    w * fin[0][i][2], w * fin[0][i][3]};
      }
    }
  }
}

// Token-major W2 + weighted sum: block (column tile, token t); wave i < top_k handles routed slot
// t*top_k + i, wave top_k (when present) the shared slot T*top_k + t. A = h[slot] in MFMA row 0
// (the other 15 rows are zero); the block adds the waves' w[slot] * y rows in slot order.
template <int SPG, int CT, int NGW, int NB>
__global__ __launch_bounds__(64 * kTokenSumMaxWaves) void w2_token_sum_kernel(
    const uint16_t* __restrict__ h, ExpertsDev ed, SlotsDev sd, const int32_t* __restrict__ ids,
    const float* __restrict__ topk_w, uint16_t* __restrict__ out) {
  constexpr int TW = 16 * CT;
  __shared__ float part[kTokenSumMaxWaves][TW];
  const int t = blockIdx.y;
  const int lane = threadIdx.x & 63;
  const int i = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));  // uniform: the slot's
                                                                         // resources in SGPRs
  const int nwaves = blockDim.x >> 6;
  const bool is_shared = i >= sd.top_k;
  const int f = is_shared ? sd.T * sd.top_k + t : t * sd.top_k + i;
  const int e = is_shared ? ed.num_experts : ids[f];
  const bool ok = is_shared || routed_ok(ed.expert_row, ed.num_experts, e);
  const int G = ed.group, K = ed.inter, NOUT = ed.hidden;
  const int m = lane & 15, kq = lane >> 4;
  const int cl = blockIdx.x * TW + CT * m;
  const float w = ok ? topk_w[f] : 0.0f;  // in flight with the weight stream

  f32x4 acc[CT];
#pragma unroll
  for (int j = 0; j < CT; ++j) acc[j] = f32x4{0.f, 0.f, 0.f, 0.f};
  if (ok) {  // wave-uniform: a dropped slot contributes nothing
    const int64_t row = is_shared ? 0 : expert_row(ed, e);
    ProjDev pj[1];
    projections(ed, DEC_W2, is_shared, pj);
    pj[0] = proj_row(pj[0], is_shared ? 0 : ed.row_stride, row, K / 8, K / G, NOUT);
    const AView av{buf_rsrc(h, (uint32_t)sd.num_slots * (uint32_t)K * 2u),
                   m == 0 ? ((uint32_t)f * (uint32_t)K + (uint32_t)(8 * kq)) * 2u : kOutOfRange};
    const DecodeTile<1, SPG, CT> tile(pj, av, NOUT, G, 0, cl, kq);
    decode_tile<1, SPG, CT, NGW, NB>(tile, acc);
  }
  if (lane < 16) {  // row 0 of the tile: lanes 0..15, element 0
#pragma unroll
    for (int j = 0; j < CT; ++j) part[i][CT * lane + j] = w * acc[j][0];
  }
  __syncthreads();
  if (i == 0 && lane < TW) {
    float s = 0.0f;
    for (int v = 0; v < nwaves; ++v) s += part[v][lane];
    const int c = blockIdx.x * TW + lane;
    out[(int64_t)t * NOUT + c] = (uint16_t)f32_to_bf16_rne(s);
  }
}

// Every buffer offset the decode kernels form (activation rows, one expert's qweight, scales
// and zeros) stays below kOutOfRange.
bool decode_offsets_fit(const ExpertsDev& ed, const SlotsDev& sd) {
  const int64_t lim = kOutOfRange;
  return (int64_t)sd.T * ed.hidden * 2 < lim && (int64_t)sd.num_slots * ed.inter * 2 < lim &&
         (int64_t)ed.hidden * ed.inter / 2 < lim;
}

template <int MODE, int SPG, int KS, int CT, int NB, int NGW>
hipError_t launch_cfg(const uint16_t* act, const ExpertsDev& ed, const SlotsDev& sd,
                      const int32_t* sorted, const int32_t* eids, const int32_t* ntpp, int cap,
                      const float* topk_w, uint16_t* h, float* ys, const SlotGrid& sg,
                      hipStream_t stream) {
  const int NOUT = (MODE == DEC_W1) ? ed.inter : ed.hidden;
  if (!decode_offsets_fit(ed, sd)) return hipErrorInvalidValue;
  const dim3 grid(NOUT / (16 * CT), sg.active ? sd.num_slots : cap);
  hipLaunchKernelGGL((gemm_decode_kernel<MODE, SPG, KS, CT, NB, NGW>), grid, dim3(64 * KS), 0,
                     stream, act, ed, sd, sorted, eids, ntpp, topk_w, h, ys, sg);
  return hipGetLastError();
}

// Tile of a decode GEMM: ks waves over K, 16 * ct columns.
struct DecodeCfg {
  int ks, ct;
};

// Every configuration that pick_decode_cfg gives for hidden in {512, 1024, 1536, 2048},
// intermediate in {256, 512, 1024} and groups of 32 SPG.
template <int MODE, int SPG>
hipError_t launch_decode_cfg(const uint16_t* act, const ExpertsDev& ed, const SlotsDev& sd,
                             const int32_t* sorted, const int32_t* eids, const int32_t* ntpp,
                             int cap, const float* topk_w, uint16_t* h, float* ys, DecodeCfg c,
                             const SlotGrid& sg, hipStream_t stream) {
  const int K = (MODE == DEC_W1) ? ed.hidden : ed.inter;
  const int NOUT = (MODE == DEC_W1) ? ed.inter : ed.hidden;
  if (NOUT % (16 * c.ct) != 0 || K % (c.ks * ed.group) != 0) return hipErrorInvalidValue;
  const int ngw = K / (c.ks * ed.group);
#define MOE_DEC(KSV, CTV, NGWV)                                                                \
  if (c.ks == KSV && c.ct == CTV && ngw == NGWV)                                               \
    return launch_cfg<MODE, SPG, KSV, CTV, (NGWV < 2 ? NGWV : 2), NGWV>(                       \
        act, ed, sd, sorted, eids, ntpp, cap, topk_w, h, ys, sg, stream);
#define MOE_DEC2(KSV, NGWV) MOE_DEC(KSV, 2, NGWV) MOE_DEC(KSV, 4, NGWV)
  if constexpr (MODE == DEC_W1) {
    if constexpr (SPG == 2) { MOE_DEC2(4, 2) MOE_DEC2(4, 4) MOE_DEC2(4, 6) MOE_DEC2(4, 8) }
    if constexpr (SPG == 4) { MOE_DEC2(4, 1) MOE_DEC2(4, 2) MOE_DEC2(4, 3) MOE_DEC2(4, 4) }
    if constexpr (SPG == 8) { MOE_DEC2(4, 1) MOE_DEC2(4, 2) MOE_DEC(2, 2, 1) MOE_DEC2(2, 3) }
    MOE_DEC(8, 2, 1)
    if constexpr (SPG <= 4) { MOE_DEC(8, 2, 2) }
    if constexpr (SPG == 2) { MOE_DEC(8, 2, 3) MOE_DEC(8, 2, 4) }
  } else {
    MOE_DEC(4, 4, 1)
    if constexpr (SPG <= 4) { MOE_DEC(4, 4, 2) }
    if constexpr (SPG == 2) { MOE_DEC(4, 4, 4) }
    if constexpr (SPG >= 4) { MOE_DEC(2, 4, 1) }
    if constexpr (SPG == 8) { MOE_DEC(1, 4, 1) }
  }
#undef MOE_DEC2
#undef MOE_DEC
  return hipErrorInvalidValue;
}

// Configuration by problem size, from sweeps over hidden 512 .. 2048, intermediate 256 .. 1024,
// groups of 64 .. 256 and 4 .. 203 tokens (times of eight layers, 128 or 256 experts):
//  - Four waves over K wherever the groups divide by four: now that all of a block's waves finish
//    its tile, more waves cost no longer tail (W2 of 64 tokens, K 512: four waves of one group
//    491.7 us, two of two 497.5, one of four 505).
//  - A wave's groups unrolled with a 2-deep ring: all other forms are slower, a runtime loop by
//    most (W1 of 32 tokens 393 against 446 us; W1 with K 2048 in groups of 256, 48 tokens, 636
//    against 773); deeper rings and more waves per SIMD too.
//  - W1 with four columns per lane (half the activation loads per weight) from about 700
//    workgroups of that size on (32 tokens: 393 against 409 us with two), and where they are
//    about one for each of the 256 CUs (hidden 2048, 4 tokens: 192.5 against 205.8); between
//    these some CUs would get one such workgroup and others two (8 tokens: 267 against 257), and
//    below there are too few. The workgroups are estimated from the experts that an even routing
//    reaches. K of 512 is too short to gain from it (64 tokens: 239 against 234 us).
//  - Where an expert has 8 rows and more, blocks are full and experts have several: four columns
//    from 500 workgroups on, at K of 512 too (a layer of hidden 2048, intermediate 512: 1200
//    tokens, top-2, 16 experts 71.1 against 81.3 us, 128 tokens, top-8, 64 experts 58.5 against
//    62.2; hidden 512: 256 tokens, top-8, 64 experts 48.9 against 53.0). Not with two waves (6
//    groups of 256), whose four-column form has one wave per SIMD: 46.9 against 50.6 there.
//  - Up to 16 slots W1 takes eight waves: nothing but latency counts there.
template <int MODE>
DecodeCfg pick_decode_cfg(const ExpertsDev& ed, const SlotsDev& sd) {
  const int K = (MODE == DEC_W1) ? ed.hidden : ed.inter;
  const int groups = K / ed.group;
  DecodeCfg c{groups % 4 == 0 ? 4 : (groups % 2 == 0 ? 2 : 1), 4};
  if (MODE == DEC_W1) {
    const float E = (float)ed.num_experts;
    const float reached = E * (1.0f - powf(fmaxf(0.0f, 1.0f - (float)sd.top_k / E), (float)sd.T));
    const float wgs = reached * (float)(ed.inter / 64);
    if (K <= 512 || wgs < 220.0f || (wgs > 300.0f && wgs < 700.0f)) c.ct = 2;
    const float slots = (float)sd.T * (float)sd.top_k;
    const float blocks = fmaxf(reached, slots / 16.0f + reached / 2.0f);
    if (c.ks == 4 && slots >= 8.0f * reached && blocks * (float)(ed.inter / 64) >= 500.0f) c.ct = 4;
    if (sd.num_slots <= 16 && groups % 8 == 0) c = DecodeCfg{8, 2};
  }
  return c;
}

template <int SPG, int CT, int NGW, int NB>
hipError_t launch_token_sum(const uint16_t* h, const ExpertsDev& ed, const SlotsDev& sd,
                            const int32_t* ids, const float* topk_w, uint16_t* out,
                            hipStream_t stream) {
  const int has_shared = sd.num_slots > sd.T * sd.top_k ? 1 : 0;
  const dim3 grid(ed.hidden / (16 * CT), sd.T);
  hipLaunchKernelGGL((w2_token_sum_kernel<SPG, CT, NGW, NB>), grid, dim3(64 * (sd.top_k + has_shared)),
                     0, stream, h, ed, sd, ids, topk_w, out);
  return hipGetLastError();
}

}  // namespace

namespace {
template <int MODE>
hipError_t launch_decode_picked(const uint16_t* act, const ExpertsDev& ed, const SlotsDev& sd,
                                const int32_t* sorted, const int32_t* eids, const int32_t* ntpp,
                                int cap, const float* topk_w, uint16_t* h, float* ys,
                                const SlotGrid& sg, hipStream_t stream) {
  auto launch = [&](auto spg, DecodeCfg c) {
    return launch_decode_cfg<MODE, decltype(spg)::value>(act, ed, sd, sorted, eids, ntpp, cap,
                                                         topk_w, h, ys, c, sg, stream);
  };
  DecodeCfg c = pick_decode_cfg<MODE>(ed, sd);
  switch (ed.group) {
    case 64: return launch(std::integral_constant<int, 2>{}, c);
    case 128: return launch(std::integral_constant<int, 4>{}, c);
    case 256: return launch(std::integral_constant<int, 8>{}, c);
    default: return hipErrorInvalidValue;
  }
}
}  // namespace

hipError_t launch_w1_decode_mfma(const uint16_t* x, const ExpertsDev& ed, const SlotsDev& sd,
                                 const int32_t* sorted, const int32_t* eids, const int32_t* ntpp,
                                 int cap, uint16_t* h, hipStream_t stream) {
  return launch_decode_picked<DEC_W1>(x, ed, sd, sorted, eids, ntpp, cap, nullptr, h, nullptr,
                                      SlotGrid{0, nullptr, nullptr, nullptr}, stream);
}

hipError_t launch_w2_decode_mfma(const uint16_t* h, const ExpertsDev& ed, const SlotsDev& sd,
                                 const int32_t* sorted, const int32_t* eids, const int32_t* ntpp,
                                 int cap, const float* topk_w, float* ys, hipStream_t stream) {
  return launch_decode_picked<DEC_W2>(h, ed, sd, sorted, eids, ntpp, cap, topk_w, nullptr, ys,
                                      SlotGrid{0, nullptr, nullptr, nullptr}, stream);
}

hipError_t launch_w1_decode_slotgrid(const uint16_t* x, const ExpertsDev& ed, const SlotsDev& sd,
                                     const SlotGrid& sg, uint16_t* h, hipStream_t stream) {
  if (!sg.active || !slot_grid_fits(sd.T, sd.top_k, sd.num_slots > sd.T * sd.top_k ? 1 : 0))
    return hipErrorInvalidValue;
  return launch_decode_picked<DEC_W1>(x, ed, sd, nullptr, nullptr, nullptr, 0, nullptr, h,
                                      nullptr, sg, stream);
}

hipError_t launch_w2_decode_slotgrid(const uint16_t* h, const ExpertsDev& ed, const SlotsDev& sd,
                                     const SlotGrid& sg, float* ys, hipStream_t stream) {
  if (!sg.active || sg.logits ||
      !slot_grid_fits(sd.T, sd.top_k, sd.num_slots > sd.T * sd.top_k ? 1 : 0))
    return hipErrorInvalidValue;
  return launch_decode_picked<DEC_W2>(h, ed, sd, nullptr, nullptr, nullptr, 0, sg.weights, nullptr,
                                      ys, sg, stream);
}

// W1 + fused W2 partials on the slot grid: group 128, one wave per two groups of K = hidden
// (all loads up front), and hidden = 4 x 64 output columns per wave.
bool w1w2_fused_fits(const ExpertsDev& ed, const SlotsDev& sd) {
  const int H = ed.hidden, ks = H / 256;
  return ed.group == 128 && H % 256 == 0 && (ks == 2 || ks == 4 || ks == 8) &&
         ed.inter % 32 == 0 && decode_offsets_fit(ed, sd) &&
         slot_grid_fits(sd.T, sd.top_k, sd.num_slots > sd.T * sd.top_k ? 1 : 0) &&
         (int64_t)sd.num_slots * (ed.inter / 32) * H * 4 < kOutOfRange;
}

hipError_t launch_w1w2_slotgrid(const uint16_t* x, const ExpertsDev& ed, const SlotsDev& sd,
                                const SlotGrid& sg, float* part, hipStream_t stream) {
  if (!sg.active || !w1w2_fused_fits(ed, sd)) return hipErrorInvalidValue;
  const dim3 grid(ed.inter / 32, sd.num_slots);
  switch (ed.hidden / 256) {
#define MOE_W1W2(KSV)                                                                          \
  case KSV:                                                                                    \
    hipLaunchKernelGGL((gemm_decode_kernel<DEC_W1, 4, KSV, 2, 2, 2, true>), grid,             \
                       dim3(64 * KSV), 0, stream, x, ed, sd, nullptr, nullptr, nullptr,        \
                       nullptr, nullptr, part, sg);                                            \
    return hipGetLastError();
    MOE_W1W2(2) MOE_W1W2(4) MOE_W1W2(8)
#undef MOE_W1W2
    default: return hipErrorInvalidValue;
  }
}

bool w2_token_sum_fits(const ExpertsDev& ed, const SlotsDev& sd) {
  const int has_shared = sd.num_slots > sd.T * sd.top_k ? 1 : 0;
  return sd.T >= 1 && sd.T <= kTokenSumMaxTokens && sd.top_k + has_shared <= kTokenSumMaxWaves &&
         ed.hidden % 32 == 0 && ed.inter % ed.group == 0;
}

hipError_t launch_w2_token_sum(const uint16_t* h, const ExpertsDev& ed, const SlotsDev& sd,
                               const int32_t* ids, const float* topk_w, uint16_t* out,
                               hipStream_t stream) {
  if (!w2_token_sum_fits(ed, sd) || !decode_offsets_fit(ed, sd)) return hipErrorInvalidValue;
  // K of 256 and 512: all of a slot's groups in flight at once; K of 1024: 512 k of them.
#define MOE_TOKEN_SUM(G, K, NGW, NB)     \
  if (ed.group == G && ed.inter == K)    \
    return launch_token_sum<G / 32, 2, NGW, NB>(h, ed, sd, ids, topk_w, out, stream);
  MOE_TOKEN_SUM(64, 256, 4, 4) MOE_TOKEN_SUM(64, 512, 8, 8) MOE_TOKEN_SUM(64, 1024, 16, 8)
  MOE_TOKEN_SUM(128, 256, 2, 2) MOE_TOKEN_SUM(128, 512, 4, 4) MOE_TOKEN_SUM(128, 1024, 8, 4)
  MOE_TOKEN_SUM(256, 256, 1, 1) MOE_TOKEN_SUM(256, 512, 2, 2) MOE_TOKEN_SUM(256, 1024, 4, 2)
#undef MOE_TOKEN_SUM
  return hipErrorInvalidValue;
}
