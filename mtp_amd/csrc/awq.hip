// AWQ int4 checkpoints behind the GPTQ kernels: an exact load-time repack into the reference's
// GPTQ layout (qweight int32 [E, K/8, N] packed along K, qzeros int32 [E, K/G, N/8] packed
// along N, scales fp16 [E, K/G, N]). Only nibbles and scale bits move, so every dequantised
// weight (q - z) * s is unchanged.
//
// Source layouts:
//  * MOE_AWQ_WNA16: vLLM's int4 fused-MoE layout that the reference serves its AWQ checkpoint
//    with (src/mtp_expert_prefetch/tracing/vllm_wna16_group_plan.py:394-470): B uint8
//    [E, N, K/2], q(k, n) in nibble k % 2 of byte (n, k / 2); zero points uint8 [E, N/2, K/G],
//    z(g, n) in nibble n % 2 of byte (n / 2, g), or none (zero 8); scales [E, N, K/G] in fp16 or
//    bf16. The bytes of one (n, 8 k) run are exactly one GPTQ word, so qweight is a transpose of
//    32-bit words.
//  * MOE_AWQ_GEMM: the AutoAWQ GEMM checkpoint layout: qweight int32 [E, K, N/8] and qzeros
//    int32 [E, K/G, N/8] packed along N in the order [0, 2, 4, 6, 1, 3, 5, 7]; scales fp16
//    [E, K/G, N].
// A bf16 scale outside [2^-17, 65504] (not exact in fp16) sets *status to 1; 0 means every
// value moved exactly.
//
// Byte and integer moves, bound by HBM. One launch holds the three tensors (workgroup ranges:
// zeros, scales, then the far larger qweight, so that the small parts end inside it), after the
// one that clears the status. Measured on 256 experts of 2048 x 512 (wna16, 280 MB): 175 + 9 + 5 us
// for the three one-thread-per-word kernels before -> 47 us (5.9 TB/s); the call, which waits
// for the status, 212 -> 73 us.
#include <stdio.h>

#include "common.h"
#include "launch.h"

namespace {

constexpr int kThreads = 256;
constexpr int kTile = 64;  // qweight words per side of a transposed tile

struct AwqArgs {
  const void* qw;
  const void* qz;
  const uint16_t* sc;
  int32_t* oq;
  int32_t* oz;
  uint16_t* os;
  int32_t* status;
  int E, K8, N, NG, sc_bf16;
  unsigned zero_blocks, scale_blocks;
  unsigned first;  // workgroup index of the launch's first workgroup
  int q_vec, s_vec;  // wide accesses fit the bases and strides of qweight / scales
};

// MOE_AWQ_WNA16 qweight: per expert the transpose of a [N, K8] matrix of words. A workgroup turns
// a 64 x 64 tile through LDS (rows padded by one word), 16-byte loads along K8 and 16-byte stores
// along N; one thread per word read 64 lines per wave load, each a quarter of a KB or more apart.
MOE_DEV void qweight_wna16(const AwqArgs& a, unsigned block) {
  __shared__ uint32_t s[kTile * (kTile + 1)];
  const int tr = (a.K8 + kTile - 1) / kTile, tn = (a.N + kTile - 1) / kTile;
  const int r0 = (int)(block % tr) * kTile, n0 = (int)(block / tr % tn) * kTile;
  const int64_t e = block / ((unsigned)tr * tn);
  const uint32_t* src = static_cast<const uint32_t*>(a.qw) + e * a.N * a.K8;
  int32_t* dst = a.oq + e * a.K8 * a.N;
  const int tid = threadIdx.x;
  if (a.q_vec) {  // K8 % 4 == 0 and N % 8 == 0: a quad is in range or out of it as a whole
    const int l = 4 * (tid & 15), h = tid >> 4;
    u32x4 v[4] = {};
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int n = n0 + h + 16 * u;
      if (n < a.N && r0 + l < a.K8) v[u] = ld128_nt(src + (int64_t)n * a.K8 + r0 + l);
    }
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
      for (int i = 0; i < 4; ++i) s[(h + 16 * u) * (kTile + 1) + l + i] = v[u][i];
    __syncthreads();
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int r = h + 16 * u;
      if (r0 + r >= a.K8 || n0 + l >= a.N) continue;
      u32x4 o;
#pragma unroll
      for (int i = 0; i < 4; ++i) o[i] = s[(l + i) * (kTile + 1) + r];
      *reinterpret_cast<u32x4*>(dst + (int64_t)(r0 + r) * a.N + n0 + l) = o;
    }
    return;
  }
  const int l = tid & 63, h = tid >> 6;
  for (int n = h; n < kTile; n += kThreads / 64)
    if (n0 + n < a.N && r0 + l < a.K8)
      s[n * (kTile + 1) + l] = src[(int64_t)(n0 + n) * a.K8 + r0 + l];
  __syncthreads();
  for (int r = h; r < kTile; r += kThreads / 64)
    if (r0 + r < a.K8 && n0 + l < a.N)
      dst[(int64_t)(r0 + r) * a.N + n0 + l] = (int32_t)s[l * (kTile + 1) + r];
}

// 8 x 8 nibble transpose: nibble j of word m becomes nibble m of word j.
MOE_DEV void nibble_transpose(uint32_t (&v)[8]) {
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const uint32_t x = v[j], y = v[j + 4];
    v[j] = (x & 0xFFFFu) | (y << 16);
    v[j + 4] = (x >> 16) | (y & 0xFFFF0000u);
  }
#pragma unroll
  for (int h = 0; h < 8; h += 4)
#pragma unroll
    for (int j = h; j < h + 2; ++j) {
      const uint32_t x = v[j], y = v[j + 2];
      v[j] = (x & 0x00FF00FFu) | ((y & 0x00FF00FFu) << 8);
      v[j + 2] = ((x >> 8) & 0x00FF00FFu) | (y & 0xFF00FF00u);
    }
#pragma unroll
  for (int j = 0; j < 8; j += 2) {
    const uint32_t x = v[j], y = v[j + 1];
    v[j] = (x & 0x0F0F0F0Fu) | ((y & 0x0F0F0F0Fu) << 4);
    v[j + 1] = ((x >> 4) & 0x0F0F0F0Fu) | (y & 0xF0F0F0F0u);
  }
}

// nibble i of an AutoAWQ word holds column 8 c + kAwqOrder[i]; column j sits at nibble kAwqInv[j]
constexpr int kAwqInv[8] = {0, 4, 1, 5, 2, 6, 3, 7};

// MOE_AWQ_GEMM qweight: a thread takes the 8 words of 8 k and 8 columns (one word per k) and
// turns their nibbles into the 8 columns' words; every source word is read once.
MOE_DEV void qweight_gemm(const AwqArgs& a, unsigned block) {
  const int C = a.N / 8;
  const int64_t i = (int64_t)block * kThreads + threadIdx.x;
  if (i >= (int64_t)a.E * a.K8 * C) return;
  const int64_t er = i / C, c = i % C;  // er = e * K8 + r
  const uint32_t* src = static_cast<const uint32_t*>(a.qw) + er * 8 * C + c;
  uint32_t v[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) v[j] = src[(int64_t)j * C];
  nibble_transpose(v);
  int32_t* dst = a.oq + er * a.N + 8 * c;
  if (a.q_vec) {
#pragma unroll
    for (int h = 0; h < 8; h += 4)
      *reinterpret_cast<u32x4*>(dst + h) = u32x4{v[kAwqInv[h]], v[kAwqInv[h + 1]],
                                                 v[kAwqInv[h + 2]], v[kAwqInv[h + 3]]};
  } else {
#pragma unroll
    for (int j = 0; j < 8; ++j) dst[j] = (int32_t)v[kAwqInv[j]];
  }
}

// One thread per word of the zero points (under 1 % of the bytes).
template <int LAYOUT>
MOE_DEV void qzeros(const AwqArgs& a, unsigned block) {
  const int64_t C = a.N / 8, NG = a.NG;
  const int64_t i = (int64_t)block * kThreads + threadIdx.x;
  if (i >= (int64_t)a.E * NG * C) return;
  const int64_t e = i / (NG * C), rem = i % (NG * C);
  const int64_t g = rem / C, c = rem % C;  // GPTQ word (g, c): z(g, 8 c + j) at nibble j
  uint32_t w = 0;
  if (!a.qz) {
    w = 0x88888888u;  // symmetric checkpoint: zero point 8
  } else if (LAYOUT == MOE_AWQ_WNA16) {
    const uint8_t* s = static_cast<const uint8_t*>(a.qz);
#pragma unroll
    for (int j = 0; j < 4; ++j)  // columns 8c + 2j, 8c + 2j + 1 share byte (4c + j, g)
      w |= (uint32_t)s[(e * (a.N / 2) + 4 * c + j) * NG + g] << (8 * j);
  } else {
    const uint32_t v = static_cast<const uint32_t*>(a.qz)[i];
#pragma unroll
    for (int j = 0; j < 8; ++j) w |= ((v >> (4 * kAwqInv[j])) & 0xFu) << (4 * j);
  }
  a.oz[i] = (int32_t)w;
}

// fp16 bits of a bf16 value, exact for magnitudes in [2^-17, 65504] and zero; else *bad = 1
// (a plain store: every writer stores the same value).
MOE_DEV uint16_t bf16_to_f16_exact(uint16_t b, int32_t* bad) {
  const float f = bf16_to_f32(b);
  const _Float16 h = (_Float16)f;
  if (!((float)h == f)) *bad = 1;
  return __builtin_bit_cast(uint16_t, h);
}

// Scales. s_vec: MOE_AWQ_WNA16 with NG % 8 == 0: a thread turns 2 columns x 8 groups (two 16-byte
// loads, eight 4-byte stores, consecutive over the lanes); MOE_AWQ_GEMM: 8 values in place order.
// Otherwise one thread per value.
template <int LAYOUT>
MOE_DEV void scales(const AwqArgs& a, unsigned block) {
  const int64_t i = (int64_t)block * kThreads + threadIdx.x;
  const int64_t total = (int64_t)a.E * a.NG * a.N;
  if (!a.s_vec) {
    if (i >= total) return;
    const int64_t n = i % a.N, eg = i / a.N, e = eg / a.NG, g = eg % a.NG;
    const uint16_t v = LAYOUT == MOE_AWQ_WNA16 ? a.sc[(e * a.N + n) * a.NG + g] : a.sc[i];
    a.os[i] = a.sc_bf16 ? bf16_to_f16_exact(v, a.status) : v;
    return;
  }
  if constexpr (LAYOUT == MOE_AWQ_WNA16) {
    if (i >= total / 16) return;
    const int64_t np = i % (a.N / 2), eg = i / (a.N / 2);
    const int64_t e = eg / (a.NG / 8), g = 8 * (eg % (a.NG / 8)), n = 2 * np;
    u32x4 v[2];
#pragma unroll
    for (int u = 0; u < 2; ++u) v[u] = ld128(a.sc + (e * a.N + n + u) * a.NG + g);
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      uint32_t p = 0;
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        uint16_t b = (uint16_t)(v[u][k >> 1] >> (16 * (k & 1)));
        if (a.sc_bf16) b = bf16_to_f16_exact(b, a.status);
        p |= (uint32_t)b << (16 * u);
      }
      *reinterpret_cast<uint32_t*>(a.os + (e * a.NG + g + k) * a.N + n) = p;
    }
  } else {  // fp16 only
    if (i < total / 8) *reinterpret_cast<u32x4*>(a.os + 8 * i) = ld128(a.sc + 8 * i);
  }
}

template <int LAYOUT>
__global__ __launch_bounds__(kThreads) void awq_repack_kernel(AwqArgs a) {
  unsigned b = a.first + blockIdx.x;
  if (b < a.zero_blocks) return qzeros<LAYOUT>(a, b);
  b -= a.zero_blocks;
  if (b < a.scale_blocks) return scales<LAYOUT>(a, b);
  b -= a.scale_blocks;
  if constexpr (LAYOUT == MOE_AWQ_WNA16)
    qweight_wna16(a, b);
  else
    qweight_gemm(a, b);
}

__global__ void awq_status_clear(int32_t* status) { *status = 0; }

int64_t blocks_for(int64_t n) { return (n + kThreads - 1) / kThreads; }

bool aligned(const void* p, uintptr_t bytes) {
  return (reinterpret_cast<uintptr_t>(p) & (bytes - 1)) == 0;
}

}  // namespace

extern "C" {

int moe_awq_to_gptq_v1(int32_t layout, const void* qweight, const void* qzeros,
                       const uint16_t* scales, int32_t scales_bf16, int32_t num_experts,
                       int32_t in_features, int32_t out_features, int32_t group_size,
                       const moe_gptq_proj_v1* out, int32_t* status, void* stream) {
  auto err = [](int code, const char* msg) {
    snprintf(moe_error_buffer(), kErrorBufferBytes, "awq_to_gptq: %s", msg);
    return code;
  };
  if (layout != MOE_AWQ_WNA16 && layout != MOE_AWQ_GEMM) return err(MOE_ERR_UNSUPPORTED, "layout");
  if (!qweight || !scales || !out || !out->qweight || !out->qzeros || !out->scales || !status)
    return err(MOE_ERR_NULL, "NULL pointer");
  if (layout == MOE_AWQ_GEMM && (!qzeros || scales_bf16))
    return err(MOE_ERR_UNSUPPORTED, "the AutoAWQ GEMM layout has zero points and fp16 scales");
  const int K = in_features, N = out_features, G = group_size, E = num_experts;
  if (E < 1 || K < 8 || N < 8 || K % 8 || N % 8 || G < 8 || K % G)
    return err(MOE_ERR_SHAPE, "need K % 8 == 0, N % 8 == 0, G | K");
  hipStream_t s = (hipStream_t)stream;
  hipLaunchKernelGGL(awq_status_clear, dim3(1), dim3(1), 0, s, status);
  const bool wna16 = layout == MOE_AWQ_WNA16;
  // out names the caller's GPTQ tensors (the descriptor is the read-only one the kernels take)
  AwqArgs a{qweight, qzeros, scales, const_cast<int32_t*>(out->qweight),
            const_cast<int32_t*>(out->qzeros), const_cast<uint16_t*>(out->scales), status, E,
            K / 8, N, K / G, scales_bf16 ? 1 : 0, 0u, 0u, 0u, 0, 0};
  // wide accesses where bases and row strides allow them (N % 8 == 0 always); the narrow forms
  // move the same words one at a time
  a.q_vec = aligned(a.oq, 16) && (!wna16 || (aligned(qweight, 16) && a.K8 % 4 == 0));
  a.s_vec = wna16 ? aligned(scales, 16) && aligned(a.os, 4) && a.NG % 8 == 0
                  : aligned(scales, 16) && aligned(a.os, 16);
  const int64_t ns = (int64_t)E * a.NG * N;
  const int64_t zb = blocks_for(ns / 8),
                sb = blocks_for(a.s_vec ? ns / (wna16 ? 16 : 8) : ns),
                qb = wna16 ? (int64_t)E * ((a.K8 + kTile - 1) / kTile) * ((N + kTile - 1) / kTile)
                           : blocks_for((int64_t)E * a.K8 * (N / 8));
  a.zero_blocks = (unsigned)zb;
  a.scale_blocks = (unsigned)sb;
  // one launch holds under 2^32 threads
  constexpr int64_t kMaxBlocks = int64_t(1) << 23;
  for (int64_t first = 0, total = zb + sb + qb; first < total; first += kMaxBlocks) {
    a.first = (unsigned)first;
    const dim3 grid((unsigned)(total - first < kMaxBlocks ? total - first : kMaxBlocks));
    if (wna16)
      hipLaunchKernelGGL(awq_repack_kernel<MOE_AWQ_WNA16>, grid, dim3(kThreads), 0, s, a);
    else
      hipLaunchKernelGGL(awq_repack_kernel<MOE_AWQ_GEMM>, grid, dim3(kThreads), 0, s, a);
  }
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) {
    snprintf(moe_error_buffer(), kErrorBufferBytes, "awq_to_gptq: HIP error %d (%s)", (int)e,
             hipGetErrorString(e));
    return MOE_ERR_HIP + ((int)e % 100);
  }
  return MOE_OK;
}

}  // extern "C"
