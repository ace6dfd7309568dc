// Edge featurisation and edge embedding.
//
// Features per edge slot (residue r, neighbour j = idx[r,k]):
//   [0,16)    positional one-hot linear: W_pos[d, class] + b_pos[d],
//             class = 65 across chains, else clamp(res_r - res_j, +-32) + 32
//             (cpp/modules/mpnn/edge_rbf_features_scalar.cpp:45-76);
//   [16,416)  for each of the 25 atom pairs (query atom of r, neighbour atom
//             of j; cpp/primitives/compute/atom_pair_distance_scalar.cpp:21-72)
//             16 Gaussian RBFs of D = sqrt(sum (n - q)^2 + 1e-6) with centres
//             2 + f * 20/15 and 2 sigma^2 from sigma = 20 / (16 / 0.70710678)
//             (rbf_scalar.cpp:10-35, edge_rbf_features_scalar.cpp:135-137);
//             zero when either atom is missing; the whole row is zero for an
//             invalid neighbour. Float operations follow the reference order
//             with contraction disabled, so features are bit-identical to
//             the CPU path.
// Edge embedding (inverse_fold_scalar.cpp:236-279):
//   h_E = W_e . LayerNorm(W_edge . f) + b_e  (W_edge has no bias),
// fused in one kernel: a 16-slot tile of features is built in LDS, multiplied by W_edge, normalised and multiplied by W_e without leaving the
// CU, all in the reference's rounding order (h_E is bit-identical).
#include "device_math.hpp"
#include "edge_chunk.hpp"
#include "pmpnn_internal.hpp"

namespace hkbs {
namespace {

__global__ __launch_bounds__(256) void edge_features_kernel(ModelDev m, const float* __restrict__ coords,
                                                            const uint8_t* __restrict__ src,
                                                            const int32_t* __restrict__ resid,
                                                            const int32_t* __restrict__ chain,
                                                            const int32_t* __restrict__ idx, int L, int K,
                                                            float* __restrict__ features) {
  const size_t task = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  const size_t S = (size_t)L * K;
  if (task >= S * 26) return;
  const size_t slot = task / 26;
  const int c = static_cast<int>(task % 26);
  const int r = static_cast<int>(slot / K);
  float out[16];
  edge_chunk(m, coords, src, resid, chain, L, r, idx[slot], c, out);
  float* dst = features + slot * kEdgeIn + c * 16;
#pragma unroll
  for (int f = 0; f < 16; ++f) dst[f] = out[f];
}

constexpr int kTile = 16;  // edge slots per workgroup of eight waves, 16 output columns each
constexpr int kTileThreads = 512;
constexpr int kLdF = kEdgeIn + 4;  // floats per row of the features, and of a 128-wide tile (both 4 mod 32)
constexpr int kLdX = kH + 4;

// h_E = W_e . LN(W_edge . f) + b_e in the reference's rounding order
// (sequential sums without FMA, Welford LayerNorm), on the encoder's edge
// tiles (seq_rows_mfma). The tile's 16 x 26 chunks of 16 features are built in
// one round, a chunk per thread.
__global__ __launch_bounds__(kTileThreads, 6) void edge_embed_kernel(ModelDev m, const float* __restrict__ coords,
                                                                     const uint8_t* __restrict__ src,
                                                                     const int32_t* __restrict__ resid,
                                                                     const int32_t* __restrict__ chain,
                                                                     const int32_t* __restrict__ idx, int L, int K,
                                                                     float* __restrict__ h_e) {
#pragma clang fp contract(off)
  static_assert(26 * kTile <= kTileThreads && kEdgeIn == 26 * 16 && kLdF % 32 == 4 && kLdX % 32 == 4, "tile sizes");
  __shared__ __attribute__((aligned(16))) float F[kTile * kLdF];
  __shared__ __attribute__((aligned(16))) float X[kTile * kLdX];
  __shared__ float mean[kTile], inv[kTile];
  __shared__ float tbl[17];
  const size_t S = (size_t)L * K;
  const size_t slot0 = (size_t)blockIdx.x * kTile;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int row0 = 4 * (lane >> 4), c = 16 * wave + (lane & 15);
  float4 ring[kQuadRing];
  seq_ring_fill(ring, m.edge_q);
  if (threadIdx.x < 17) tbl[threadIdx.x] = kExpNegTable[threadIdx.x];
  __syncthreads();
  if (threadIdx.x < 26 * kTile) {
    const int row = threadIdx.x % kTile, chunk = threadIdx.x / kTile;
    const size_t slot = slot0 + row;
    const int r = slot < S ? static_cast<int>(slot / K) : 0;
    const int j = slot < S ? idx[slot] : -1;
    float out[16];
    edge_chunk(m, coords, src, resid, chain, L, r, j, chunk, out, tbl);  // zeros when j is not a residue
#pragma unroll
    for (int b = 0; b < 4; ++b)  // k-quad order of the chunk's 16 inputs
      *reinterpret_cast<float4*>(F + row * kLdF + 16 * chunk + 4 * b) =
          make_float4(out[b], out[4 + b], out[8 + b], out[12 + b]);
  }
  __syncthreads();
  float acc[4] = {0.0F, 0.0F, 0.0F, 0.0F};
  seq_rows_mfma<kEdgeIn / 16>(acc, F, kLdF, m.edge_q, ring, m.We_q);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    X[(row0 + i) * kLdX + c] = acc[i];
    acc[i] = 0.0F;
  }
  __syncthreads();
  if (threadIdx.x < kTile) welford_stats_row(X + threadIdx.x * kLdX, mean + threadIdx.x, inv + threadIdx.x);
  __syncthreads();
  float* N = F;  // the normalised rows in k-quad order, where the features were
  {
    const int row = threadIdx.x >> 5, q = threadIdx.x & 31;
    const float4 x = *reinterpret_cast<const float4*>(X + row * kLdX + 4 * q);
    const float4 gm = *reinterpret_cast<const float4*>(m.ne_g + 4 * q), bt = *reinterpret_cast<const float4*>(m.ne_b + 4 * q);
    const float mu = mean[row], is = inv[row];
    float* p = N + row * kLdX + kquad(4 * q);
    p[0] = (x.x - mu) * is * gm.x + bt.x;
    p[4] = (x.y - mu) * is * gm.y + bt.y;
    p[8] = (x.z - mu) * is * gm.z + bt.z;
    p[12] = (x.w - mu) * is * gm.w + bt.w;
  }
  __syncthreads();
  seq_rows_mfma<kH / 16, (kEdgeIn / 16) % kQuadRing>(acc, N, kLdX, m.We_q, ring, m.We_q);
  const float be = m.We_b[c];
#pragma unroll
  for (int i = 0; i < 4; ++i)
    if (slot0 + row0 + i < S) h_e[(slot0 + row0 + i) * kH + c] = acc[i] + be;
}

}  // namespace

hipError_t launch_edge_features(const ModelDev& m, const float* coords, const uint8_t* atom_src,
                                const int32_t* resid, const int32_t* chain, const int32_t* idx, int L, int K,
                                float* features, hipStream_t stream) {
  const size_t tasks = (size_t)L * K * 26;
  if (tasks == 0) return hipSuccess;
  edge_features_kernel<<<(unsigned)((tasks + 255) / 256), 256, 0, stream>>>(m, coords, atom_src, resid, chain,
                                                                           idx, L, K, features);
  return hipGetLastError();
}

hipError_t launch_edge_embed(const ModelDev& m, const float* coords, const uint8_t* atom_src,
                             const int32_t* resid, const int32_t* chain, const int32_t* idx, int L, int K,
                             float* h_e, hipStream_t stream) {
  const size_t S = (size_t)L * K;
  if (S == 0) return hipSuccess;
  edge_embed_kernel<<<(unsigned)((S + kTile - 1) / kTile), kTileThreads, 0, stream>>>(m, coords, atom_src, resid, chain,
                                                                            idx, L, K, h_e);
  return hipGetLastError();
}

}  // namespace hkbs
