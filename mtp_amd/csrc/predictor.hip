// Expert-demand predictor: per layer head l, a bf16 MLP  hidden -> D (SiLU) -> E logits, then
// the top-k experts of every (head, token).
//
// The reference's predictor (src/mtp_expert_prefetch/training/hidden_residual.py:44-106,
// Linear -> SiLU -> ... -> Linear(w, E), one prediction per layer) is simplified, as the offload
// workload specifies, to a two-layer bf16 MLP per layer with random weights whose top-16 experts
// drive the prefetch of that layer. All heads run in three launches: the first products of every
// head as one [T, L*D] product (w1 heads are contiguous rows) with SiLU into a head-major
// activation, the second products with the head on grid.y, and one wave per (head, token) for the
// top-k. Both products use the canonical fp32 dot order of the router (routing.h:logits_tile);
// the hidden activation is SiLU in fp32 rounded once to bf16 (the bf16 Linear output dtype).
#include "launch.h"
#include "routing.h"

namespace {

// bf16(silu(v)).
MOE_DEV uint16_t silu_bf16(float v) { return (uint16_t)f32_to_bf16_rne(v / (1.0f + expf(-v))); }

// x[head][t][:] . W[head][n][:] for the 4 waves x TE rows n of a workgroup, head = blockIdx.y, and
// the token tiles of its per_wg tokens: every wave issues the loads of its
// weight rows, then each tile of TT token rows passes through LDS, so a weight row is read once
// for per_wg tokens and the whole 8 KB of a wave's rows is in flight at once (bound by HBM up
// to about 4 tokens, by the fp32 FMAs beyond). 40 heads (2048 -> 1024 -> 256, 189 MB) per call:
// 4 tokens 116.7 -> 50.6 us (the row read from memory once per token before), 1 token 37.5 us, 16
// tokens 89 us. Two rows per wave (four: 58.3 us at 4 tokens, one: 57.4) and nontemporal
// weight loads (53.5 -> 50.6).
// ACT: out is bf16 [n / D][T][D] = silu(z); else fp32 [head][T][N + 1].
constexpr int kRowsTE = 2;
template <int TT, int NI, bool ACT>
__global__ __launch_bounds__(256) void mlp_rows_kernel(const uint16_t* __restrict__ x,
                                                       int64_t x_head, int T, int K,
                                                       const uint16_t* __restrict__ W,
                                                       int64_t w_head, int N, int D, int per_wg,
                                                       void* __restrict__ out_v) {
  __shared__ __attribute__((aligned(16))) uint16_t s_x[TT * NI * 512];
  constexpr int NV = TT * kRowsTE;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int64_t head = blockIdx.y;
  const int row_blocks = (N + 4 * kRowsTE - 1) / (4 * kRowsTE);
  const int n0 = ((int)blockIdx.x % row_blocks * 4 + wave) * kRowsTE;
  LdsLogitsTile<TT, kRowsTE, NI, kBufNontemporal> tile;
  tile.load(K, W + head * w_head, N, nullptr, n0, lane);
  const __amdgpu_buffer_rsrc_t xr = buf_rsrc(x + head * x_head, (uint32_t)T * (uint32_t)K * 2u);
  const int t_begin = (int)blockIdx.x / row_blocks * per_wg;
  const int t_end = min(T, t_begin + per_wg);
  for (int t0 = t_begin; t0 < t_end; t0 += TT) {
    if (t0 > t_begin) __syncthreads();  // the previous tile is read
    // the tile's rows are contiguous; past the last token the loads read zeros
#pragma unroll
    for (int u = 0; u < (TT * NI + 3) / 4; ++u) {
      const int o = 8 * (tid + 256 * u);
      if (o < TT * K)
        *reinterpret_cast<u32x4*>(s_x + o) = buf_ld128(xr, ((uint32_t)t0 * K + o) * 2u);
    }
    __syncthreads();
    float acc[NV];
    tile.partials(s_x, K, lane, acc);
    fold_partials(acc, lane);
    const int v = lane / (64 / NV), t = t0 + v / kRowsTE, n = n0 + v % kRowsTE;
    if (lane % (64 / NV) == 0 && t < t_end && n < N) {
      if constexpr (ACT)
        static_cast<uint16_t*>(out_v)[((int64_t)(n / D) * T + t) * D + n % D] = silu_bf16(acc[0]);
      else
        static_cast<float*>(out_v)[(head * T + t) * (N + 1) + n] = acc[0];
    }
  }
}

// The same products for any K: one wave per TT x TE tile, out[head][t][n] fp32 (row stride N + 1).
template <int TT, int TE>
__global__ __launch_bounds__(256) void mlp_logits_kernel(
    const uint16_t* __restrict__ x, int64_t x_head, int T, int K, const uint16_t* __restrict__ W,
    int64_t w_head, int N, float* __restrict__ out, int64_t out_head) {
  const int lane = threadIdx.x & 63;
  const int wave = blockIdx.x * (blockDim.x >> 6) + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int tiles_n = (N + TE - 1) / TE;
  const int t0 = (wave / tiles_n) * TT;
  const int n0 = (wave % tiles_n) * TE;
  if (t0 >= T) return;
  const int64_t head = blockIdx.y;
  logits_tile<TT, TE>(x + head * x_head, T, K, W + head * w_head, N, nullptr, nullptr,
                      out + head * out_head, t0, n0, lane);
}

// a[l][t][j] = bf16(silu(z[t][l * D + j])), z with row stride L * D + 1.
__global__ void silu_bf16_kernel(const float* __restrict__ z, int T, int L, int D,
                                 uint16_t* __restrict__ a) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t per_head = (int64_t)T * D;
  if (i >= per_head * L) return;
  const int64_t l = i / per_head, r = i % per_head;
  const int64_t t = r / D, j = r % D;
  a[i] = silu_bf16(z[t * ((int64_t)L * D + 1) + l * D + j]);
}

// One wave per (head, token): logits row (head * T + t) of z2, ids/scores [head][t][top_k].
__global__ __launch_bounds__(256) void predictor_topk_kernel(const float* __restrict__ logits,
                                                             int T, int L, int E, int top_k,
                                                             int32_t* __restrict__ ids,
                                                             float* __restrict__ scores) {
  const int lane = threadIdx.x & 63;
  const int w = blockIdx.x * (blockDim.x >> 6) + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (w >= T * L) return;
  const int l = w / T, t = w % T;
  const int64_t head_off = (int64_t)l * T * top_k;
  topk_token_any(logits + (int64_t)w * (E + 1), E, top_k, 0, T, t, lane, ids + head_off,
             scores + head_off, nullptr);
}

template <int TT, int TE>
hipError_t launch_mlp_logits(const uint16_t* x, int64_t x_head, int T, int K, const uint16_t* W,
                             int64_t w_head, int N, float* out, int64_t out_head, int heads,
                             hipStream_t stream) {
  const int64_t tiles = (int64_t)((T + TT - 1) / TT) * ((N + TE - 1) / TE);
  hipLaunchKernelGGL((mlp_logits_kernel<TT, TE>), dim3((unsigned)((tiles + 3) / 4), heads),
                     dim3(256), 0, stream, x, x_head, T, K, W, w_head, N, out, out_head);
  return hipGetLastError();
}

// The tiled products hold K in at most four 512-column steps per lane.
constexpr int kRowsMaxK = 2048;
constexpr int kMaxTokensPerWg = 32, kWantedWgs = 1024;

template <int NI, bool ACT>
hipError_t launch_mlp_rows(const uint16_t* x, int64_t x_head, int T, int K, const uint16_t* W,
                           int64_t w_head, int N, int D, void* out, int heads,
                           hipStream_t stream) {
  const unsigned row_blocks = (N + 4 * kRowsTE - 1) / (4 * kRowsTE);
  // Tokens per workgroup: its token tiles run one after the other, so with few rows they are dealt to
  // more workgroups, down to one tile each, until there are four per CU (the weight rows then come
  // from L2 again). One head (2048 -> 1024 -> 256): 32 tokens 31.7 us at 32 per workgroup, 13.8 so;
  // 8 heads 43.9 -> 38.2. Wanting 512 is slower (40 heads of 512, 32 tokens 52.7 against 51.0 us),
  // 2048 reads the weights too often (8 heads, 8 tokens 22.4 against 19.4).
  int per_wg = kMaxTokensPerWg;
  while (per_wg > 4 && (int64_t)row_blocks * heads * ((T + per_wg - 1) / per_wg) < kWantedWgs)
    per_wg /= 2;
  const dim3 grid(row_blocks * ((T + per_wg - 1) / per_wg), heads);
  auto go = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, grid, dim3(256), 0, stream, x, x_head, T, K, W, w_head, N, D, per_wg,
                       out);
    return hipGetLastError();
  };
  // the token tile nearest to the batch: rows of a larger one would be zeros. 4 tokens at most:
  // tiles of 8 cost registers (8 tokens 68.2 vs 61.7 us a call, 16 tokens 98.1 vs 88.7)
  if (T == 1) return go(mlp_rows_kernel<1, NI, ACT>);
  if (T == 2) return go(mlp_rows_kernel<2, NI, ACT>);
  return go(mlp_rows_kernel<4, NI, ACT>);
}

}  // namespace

hipError_t launch_predictor(const uint16_t* h, int T, int H, int L, const uint16_t* w1, int D,
                            const uint16_t* w2, int E, int top_k, float* z1, uint16_t* a,
                            float* z2, int32_t* ids, float* scores, hipStream_t stream) {
  const int LD = L * D;
  hipError_t err;
  if (H <= kRowsMaxK) {
    err = H <= 1024 ? launch_mlp_rows<2, true>(h, 0, T, H, w1, 0, LD, D, a, 1, stream)
                    : launch_mlp_rows<4, true>(h, 0, T, H, w1, 0, LD, D, a, 1, stream);
  } else {
    err = launch_mlp_logits<1, 2>(h, 0, T, H, w1, 0, LD, z1, 0, 1, stream);
    if (err != hipSuccess) return err;
    const int64_t n = (int64_t)T * LD;
    hipLaunchKernelGGL(silu_bf16_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, stream,
                       z1, T, L, D, a);
    err = hipGetLastError();
  }
  if (err != hipSuccess) return err;
  const int64_t x2 = (int64_t)T * D, w2h = (int64_t)E * D;
  if (D <= 1024)
    err = launch_mlp_rows<2, false>(a, x2, T, D, w2, w2h, E, D, z2, L, stream);
  else if (D <= kRowsMaxK)
    err = launch_mlp_rows<4, false>(a, x2, T, D, w2, w2h, E, D, z2, L, stream);
  else
    err = launch_mlp_logits<1, 2>(a, x2, T, D, w2, w2h, E, z2, (int64_t)T * (E + 1), L, stream);
  if (err != hipSuccess) return err;
  hipLaunchKernelGGL(predictor_topk_kernel, dim3((T * L + 3) / 4), dim3(256), 0, stream, z2, T, L,
                     E, top_k, ids, scores);
  return hipGetLastError();
}
