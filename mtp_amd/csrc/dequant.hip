// GPTQ int4 -> bf16 dequantisation (load-time utility path).
//
// Follows src/mtp_expert_prefetch/repack/gptq_unpack.py:88-131:
//   W[k, n] = bf16_rne( (float(q[k, n]) - float(z[g(k), n])) * float(s[g(k), n]) )
// The fp32 product is exact (|q - z| <= 15 times an fp16), so the only rounding is the
// final cast (RNE to bf16 or fp16, none for fp32), which makes the result bit-identical to the
// reference for every output dtype.
//
// Bound by HBM: the dense result is 8 (fp32: 16) times the packed words per projection.
#include "common.h"
#include "launch.h"

namespace {

MOE_DEV float dequant1(uint32_t w, int j, float z, float s) {
  return ((float)((w >> (4 * j)) & 0xFu) - z) * s;
}

template <int OUT>
MOE_DEV uint32_t bits16(float v) {
  return OUT == 0 ? f32_to_bf16_rne(v) : (uint32_t)__builtin_bit_cast(uint16_t, (_Float16)v);
}

// The 8 consecutive k of one column to out[0..8): 16 (fp32: 32) aligned bytes.
template <int OUT>
MOE_DEV void store8(void* out_v, int64_t idx, const float (&v)[8]) {
  if constexpr (OUT == 2) {
    f32x4* o = reinterpret_cast<f32x4*>(static_cast<float*>(out_v) + idx);
    o[0] = f32x4{v[0], v[1], v[2], v[3]};
    o[1] = f32x4{v[4], v[5], v[6], v[7]};
  } else {
    u32x4 o;
#pragma unroll
    for (int p = 0; p < 4; ++p) o[p] = bits16<OUT>(v[2 * p]) | (bits16<OUT>(v[2 * p + 1]) << 16);
    *reinterpret_cast<u32x4*>(static_cast<uint16_t*>(out_v) + idx) = o;
  }
}

// Tile of kTileR packed rows (256 k) x kTileC columns per 256-thread workgroup. The packed words
// come in with 16-byte loads along the columns. Linear layout ([N, K]): they turn through LDS (8 KB,
// rows padded by one word: both sides free of bank conflicts beyond the two passes of a
// 64-lane access), so that 32 lanes write 512 (fp32: 1024) consecutive bytes of one output row;
// written straight from the column-wise loads the lanes' 16 bytes lie 2 K bytes apart and every
// store is 64 partial lines. Transposed layout ([K, N]): no turn, a thread writes its 4
// columns of each of the 8 k. G % 8 == 0, so without g_idx a word lies in one group. With g_idx
// (IDX) the tile's scales and zeros of all ng <= kMaxIdxGroups groups are held in LDS.
// Measured, 64 experts of 2048 x 512 (170 MB for bf16): bf16 linear 117.5 -> 32-39 us (one thread
// per word before; 4.4-5.3 TB/s, at the rate of a large copy), transposed 29 us, fp32 67 / 54 us.
constexpr int kTileR = 32, kTileC = 64, kMaxIdxGroups = 64;

template <int OUT, bool LINEAR, bool IDX>
__global__ __launch_bounds__(256) void dequant_tile_kernel(ProjDev p,
                                                           const int32_t* __restrict__ g_idx,
                                                           int K, int N, int G,
                                                           void* __restrict__ out) {
  __shared__ uint32_t s_w[LINEAR ? kTileR * (kTileC + 1) : 1];
  __shared__ uint32_t s_sz[IDX ? kMaxIdxGroups * (kTileC + 1) : 1];  // scale bits | zero << 16
  __shared__ int s_g[IDX ? kTileR * 8 : 1];
  const int tid = threadIdx.x;
  const int n0 = blockIdx.x * kTileC, r0 = blockIdx.y * kTileR;
  const int64_t e = blockIdx.z;
  const int K8 = K / 8, ng = K / G, G8 = G / 8;
  const int32_t* qw = p.qweight + e * K8 * N;
  const int32_t* qz = p.qzeros + e * ng * (N / 8);
  const uint16_t* sc = p.scales + e * ng * N;
  // 16 threads x 4 columns per packed row, 16 rows per pass (N % 8 == 0: a quad is in range or
  // out of it as a whole)
  const int cq = 4 * (tid & 15), rq = tid >> 4;
  const bool col_ok = n0 + cq < N;
  u32x4 w[2] = {};
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const int r = r0 + rq + 16 * u;
    if (col_ok && r < K8) w[u] = ld128(qw + (int64_t)r * N + n0 + cq);
  }
  if constexpr (IDX) {
    for (int i = tid; i < ng * kTileC; i += 256) {
      const int g = i / kTileC, c = i % kTileC, n = n0 + c;
      if (n < N) {
        const uint32_t z = ((uint32_t)qz[g * (N / 8) + n / 8] >> (4 * (n & 7))) & 0xFu;
        s_sz[g * (kTileC + 1) + c] = (uint32_t)sc[g * N + n] | (z << 16);
      }
    }
    const int k = 8 * r0 + tid;
    if (k < K) {
      const int g = g_idx[e * K + k];
      s_g[tid] = g < 0 ? 0 : (g >= ng ? ng - 1 : g);
    }
  }
  if constexpr (LINEAR) {
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int i = 0; i < 4; ++i) s_w[(rq + 16 * u) * (kTileC + 1) + cq + i] = w[u][i];
  }
  if constexpr (LINEAR || IDX) __syncthreads();

  // scale and zero of word (tile row rr, tile column c), element j
  auto scale_zero = [&](int rr, int c, int j, float& s, float& z) {
    const uint32_t v = s_sz[s_g[8 * rr + j] * (kTileC + 1) + c];
    s = f16_to_f32(v & 0xFFFFu);
    z = (float)(v >> 16);
  };
  if constexpr (LINEAR) {
    const int rr = tid & (kTileR - 1), r = r0 + rr;
    if (r >= K8) return;
#pragma unroll
    for (int u = 0; u < kTileC / 8; ++u) {
      const int c = (tid >> 5) + 8 * u, n = n0 + c;
      if (n >= N) break;
      const uint32_t word = s_w[rr * (kTileC + 1) + c];
      float v[8], s, z;
      if constexpr (!IDX) {
        const int g = r / G8;
        s = f16_to_f32(sc[g * N + n]);
        z = (float)(((uint32_t)qz[g * (N / 8) + n / 8] >> (4 * (n & 7))) & 0xFu);
      }
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        if constexpr (IDX) scale_zero(rr, c, j, s, z);
        v[j] = dequant1(word, j, z, s);
      }
      store8<OUT>(out, (e * N + n) * K + 8 * r, v);
    }
  } else {
    if (!col_ok) return;
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int rr = rq + 16 * u, r = r0 + rr;
      if (r >= K8) break;
      float s[4], z[4];
      if constexpr (!IDX) {
        const int g = r / G8;
        const u32x2 s4 = *reinterpret_cast<const u32x2*>(sc + g * N + n0 + cq);
        const uint32_t zw = (uint32_t)qz[g * (N / 8) + (n0 + cq) / 8] >> (4 * (cq & 7));
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          s[i] = f16_to_f32((s4[i >> 1] >> (16 * (i & 1))) & 0xFFFFu);
          z[i] = (float)((zw >> (4 * i)) & 0xFu);
        }
      }
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        float v[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          if constexpr (IDX) scale_zero(rr, cq + i, j, s[i], z[i]);
          v[i] = dequant1(w[u][i], j, z[i], s[i]);
        }
        const int64_t o = (e * K + 8 * r + j) * N + n0 + cq;
        if constexpr (OUT == 2)
          *reinterpret_cast<f32x4*>(static_cast<float*>(out) + o) = f32x4{v[0], v[1], v[2], v[3]};
        else
          *reinterpret_cast<u32x2*>(static_cast<uint16_t*>(out) + o) =
              u32x2{bits16<OUT>(v[0]) | (bits16<OUT>(v[1]) << 16),
                    bits16<OUT>(v[2]) | (bits16<OUT>(v[3]) << 16)};
      }
    }
  }
}

// Any group size, group count and base alignment, and small stacks: one thread per packed word.
template <int OUT>  // 0 bf16, 1 fp16, 2 fp32
__global__ __launch_bounds__(256) void dequant_kernel(ProjDev p, const int32_t* __restrict__ g_idx,
                                                      int K, int N, int G, int linear,
                                                      void* __restrict__ out_v) {
  const int n = blockIdx.x * blockDim.x + threadIdx.x;
  const int r = blockIdx.y;
  const int64_t e = blockIdx.z;
  if (n >= N) return;
  const int ngroups = K / G;
  const uint32_t w = (uint32_t)p.qweight[(e * (K / 8) + r) * N + n];
  const int32_t* zrow = p.qzeros + e * ngroups * (N / 8);
  const uint16_t* srow = p.scales + e * ngroups * N;
  float v[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const int k = 8 * r + j;
    int g = g_idx ? g_idx[e * K + k] : k / G;
    g = g < 0 ? 0 : (g >= ngroups ? ngroups - 1 : g);
    const uint32_t z = ((uint32_t)zrow[g * (N / 8) + n / 8] >> (4 * (n & 7))) & 0xFu;
    v[j] = dequant1(w, j, (float)z, f16_to_f32(srow[g * N + n]));
  }
  if (linear) {
    store8<OUT>(out_v, (e * N + n) * K + 8 * r, v);
    return;
  }
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const int64_t o = (e * K + 8 * r + j) * N + n;
    if constexpr (OUT == 2)
      static_cast<float*>(out_v)[o] = v[j];
    else
      static_cast<uint16_t*>(out_v)[o] = (uint16_t)bits16<OUT>(v[j]);
  }
}

// Whether the tile kernel is the faster one, from both kernels' times over 2^14 to 2^22 packed
// words of 8 to 2048 k and 8 to 2048 columns (in ps beyond a launch of 3.4 us). The
// one-thread-per-word kernel takes 10 per word (7 in long rows of words) and 3 per thread, and 256
// threads cover a row's columns. The tile kernel takes a fixed chain of loads, LDS and stores, plus
// a share per tile of 32 packed rows x 64 columns, full or not, and with g_idx of the tile's table.
// bf16 linear: 1 expert of 512 x 512 3.7 against 6.1 us, 2 of 2048 x 512 8.0 against 6.8, 4 of them
// 11.1 against 7.4, 256 of 24 x 512 8.7 against 16.0.
bool tile_pays(int64_t E, int64_t K, int64_t N, int64_t G, bool linear, bool fp32, bool idx) {
  const int64_t words = E * (K / 8) * N, threads = E * (K / 8) * ((N + 255) / 256 * 256);
  const int64_t tiles = E * ((K / 8 + kTileR - 1) / kTileR) * ((N + kTileC - 1) / kTileC);
  int64_t base, per_tile;
  if (linear) {
    base = fp32 ? 1400000 : 2600000;
    per_tile = fp32 ? 2700 : 4900;
  } else if (fp32) {
    base = idx ? 3300000 : 1300000;
    per_tile = 500;
  } else {  // stores of 8 bytes: partial lines where the columns end inside a tile
    base = idx ? 8000000 : (N % kTileC ? 6000000 : 2200000);
    per_tile = 2000;
  }
  if (idx) per_tile += 160 * (K / G);
  return (N >= 1024 ? 7 : 10) * words + 3 * threads > base + per_tile * tiles;
}

template <int OUT>
hipError_t launch_out(const ProjDev& p, const int32_t* g_idx, int E, int K, int N, int G,
                      int linear, void* out, hipStream_t stream) {
  const uintptr_t bases = reinterpret_cast<uintptr_t>(p.qweight) |
                          reinterpret_cast<uintptr_t>(p.scales) | reinterpret_cast<uintptr_t>(out);
  // The tile kernel where its accesses fit (its loads and stores are up to 16 bytes wide, its
  // words lie in one group (without g_idx) and its group table (with g_idx) holds
  // kMaxIdxGroups) and where it pays.
  const bool tile = (bases & 15u) == 0 && (g_idx ? K / G <= kMaxIdxGroups : G % 8 == 0) &&
                    tile_pays(E, K, N, G, linear != 0, OUT == 2, g_idx != nullptr);
  if (!tile) {
    hipLaunchKernelGGL(dequant_kernel<OUT>, dim3((N + 255) / 256, K / 8, E), dim3(256), 0, stream,
                       p, g_idx, K, N, G, linear, out);
    return hipGetLastError();
  }
  const dim3 grid((N + kTileC - 1) / kTileC, (K / 8 + kTileR - 1) / kTileR, E);
  auto go = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, grid, dim3(256), 0, stream, p, g_idx, K, N, G, out);
    return hipGetLastError();
  };
  if (g_idx) return linear ? go(dequant_tile_kernel<OUT, true, true>)
                           : go(dequant_tile_kernel<OUT, false, true>);
  return linear ? go(dequant_tile_kernel<OUT, true, false>)
                : go(dequant_tile_kernel<OUT, false, false>);
}

}  // namespace

hipError_t launch_dequant(const ProjDev& p, const int32_t* g_idx, int E, int K, int N, int G,
                          int linear, int out_dtype, void* out, hipStream_t stream) {
  switch (out_dtype) {
    case 0: return launch_out<0>(p, g_idx, E, K, N, G, linear, out, stream);
    case 1: return launch_out<1>(p, g_idx, E, K, N, G, linear, out, stream);
    case 2: return launch_out<2>(p, g_idx, E, K, N, G, linear, out, stream);
    default: return hipErrorInvalidValue;
  }
}
