// Learned double-excitation proposal: inference (bf16 MFMA, gfx950),
// training (fp32 forward/backward, Adam) and heat-bath training samples.
#include "mlp.hpp"

#include <cmath>
#include <cstdio>
#include <cstring>
#include <vector>

namespace fqm {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kBlock = 256;

#define MLP_HIP(call)                                                                                   \
  do {                                                                                                  \
    hipError_t err_ = (call);                                                                           \
    if (err_ != hipSuccess) {                                                                           \
      fprintf(stderr, "fqmc mlp: %s failed: %s (%s:%d)\n", #call, hipGetErrorString(err_), __FILE__, \
              __LINE__);                                                                                \
      return FQ_ERR_DEVICE;                                                                             \
    }                                                                                                   \
  } while (0)

inline int64_t ceil_div(int64_t a, int64_t b) { return (a + b - 1) / b; }
inline unsigned blocks(int64_t n) { return static_cast<unsigned>(std::max<int64_t>(1, ceil_div(n, kBlock))); }

// float -> bfloat16 bits, round to nearest even (NaN kept quiet).
__host__ __device__ inline uint16_t f2bf(float x) {
  uint32_t u;
  memcpy(&u, &x, 4);
  if ((u & 0x7fffffffu) > 0x7f800000u) return 0x7fc0;
  u += 0x7fffu + ((u >> 16) & 1u);
  return static_cast<uint16_t>(u >> 16);
}
__device__ inline float gelu_f(float z) { return 0.5f * z * (1.0f + erff(z * 0.70710678118654752f)); }
__device__ inline float gelu_g(float z) {
  return 0.5f * (1.0f + erff(z * 0.70710678118654752f)) + z * expf(-0.5f * z * z) * 0.39894228040143268f;
}

// ---- inference ---------------------------------------------------------------
// A block takes 16 RT determinants through the three layers; its four wavefronts
// split the output columns (column tile t of 16 to wavefront t % 4), so every
// weight is read by one wavefront of the block, straight from L2 into the
// operand registers of v_mfma_f32_16x16x32_bf16 (lane l feeds A[row l%16]
// [k 8(l/16)..+7] and B[k 8(l/16)..+7][col l%16], the weights being stored
// transposed, [N][K], and holds D[rows 4(l/16)..+3][col l%16]).  The
// activations (bf16) sit in one LDS buffer that a layer reads, barrier,
// overwrites; rows are 264 apart so that a fragment's 16 rows spread over the
// banks.  Every output accumulates its K slabs in order, whatever RT, so both
// instances give the same bits.  RT = 1 for lists of at most kFewRows, which
// fill at most two blocks per CU and are bound by the latency of the weights;
// RT = 4 reads them once per 64 rows.  (Staging every weight slab in LDS between
// two barriers took 79 us for a list of a few determinants at nbasis 80; 20 us
// now.  65536 determinants: 288 -> 117 us, 145 TFLOP/s.)
constexpr int kActLd = kHidden + 8;
constexpr int64_t kFewRows = 8192;
constexpr int kColTiles = kHidden / 16 / 4;  // column tiles of a wavefront

// acc[r][c]: rows 16 r.. times column tile 4 c + wave of the layer.
template <int RT>
__device__ __forceinline__ void layer_mfma(const uint16_t* act, int K, const uint16_t* __restrict__ Wt, int ntiles,
                                           f32x4 (&acc)[RT][kColTiles], int wave, int lane) {
  const int kq = (lane >> 4) * 8, cl = lane & 15;
#pragma unroll
  for (int r = 0; r < RT; ++r)
#pragma unroll
    for (int c = 0; c < kColTiles; ++c) acc[r][c] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll 8
  for (int k0 = 0; k0 < K; k0 += 32) {
    bf16x8 b[kColTiles];
#pragma unroll
    for (int c = 0; c < kColTiles; ++c) {
      const int t = 4 * c + wave < ntiles ? 4 * c + wave : 0;
      b[c] = *reinterpret_cast<const bf16x8*>(Wt + static_cast<int64_t>(t * 16 + cl) * K + k0 + kq);
    }
#pragma unroll
    for (int r = 0; r < RT; ++r) {
      const bf16x8 a = *reinterpret_cast<const bf16x8*>(act + (r * 16 + cl) * kActLd + k0 + kq);
#pragma unroll
      for (int c = 0; c < kColTiles; ++c) acc[r][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b[c], acc[r][c], 0, 0, 0);
    }
  }
}

template <int RT>
__global__ __launch_bounds__(kBlock) void k_mlp_infer(int nb, int k1, int n3, int d_out,
                                                      const uint64_t* __restrict__ det, int64_t cap, int64_t n,
                                                      const int64_t* __restrict__ idx,
                                                      const double* __restrict__ eps,
                                                      const uint16_t* __restrict__ w1t, const float* __restrict__ b1,
                                                      const uint16_t* __restrict__ w2t, const float* __restrict__ b2,
                                                      const uint16_t* __restrict__ w3t, const float* __restrict__ b3,
                                                      float* __restrict__ tab, int64_t ld,
                                                      const int64_t* __restrict__ pn) {
  constexpr int R = 16 * RT;
  __shared__ __attribute__((aligned(16))) uint16_t act[R * kActLd];
  const int64_t row0 = static_cast<int64_t>(blockIdx.x) * R;
  if (pn) n = *pn < n ? *pn : n;  // n is a bound
  if (row0 >= n) return;
  for (int el = threadIdx.x; el < R * k1; el += blockDim.x) {
    const int r = el / k1, c = el - r * k1;
    const int64_t d = row0 + r;
    float x = 0.0f;
    if (d < n && c < 2 * nb) {
      const int o = c < nb ? c : c - nb;
      const int64_t src = idx ? idx[d] : d;
      const bool occ = (det[static_cast<int64_t>(o >> 6) * cap + src] >> (o & 63)) & 1;
      x = occ ? (c < nb ? 1.0f : static_cast<float>(eps[o])) : 0.0f;
    }
    act[r * kActLd + c] = f2bf(x);
  }
  __syncthreads();
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, cl = lane & 15, orow = (lane >> 4) * 4;
  f32x4 acc[RT][kColTiles];
  auto hidden = [&](const float* __restrict__ bias) {  // GELU of the layer's output into the buffer it was read from
    __syncthreads();
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
      for (int c = 0; c < kColTiles; ++c) {
        const int col = (4 * c + wave) * 16 + cl;
#pragma unroll
        for (int q = 0; q < 4; ++q)
          act[(r * 16 + orow + q) * kActLd + col] = f2bf(gelu_f(acc[r][c][q] + bias[col]));
      }
    __syncthreads();
  };
  layer_mfma<RT>(act, k1, w1t, kHidden / 16, acc, wave, lane);
  hidden(b1);
  layer_mfma<RT>(act, kHidden, w2t, kHidden / 16, acc, wave, lane);
  hidden(b2);
  const int nt3 = n3 / 16;
  layer_mfma<RT>(act, kHidden, w3t, nt3, acc, wave, lane);
#pragma unroll
  for (int r = 0; r < RT; ++r)
#pragma unroll
    for (int c = 0; c < kColTiles; ++c) {
      const int t = 4 * c + wave, col = t * 16 + cl;
      if (t >= nt3 || col >= d_out) continue;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int64_t d = row0 + r * 16 + orow + q;
        if (d < n) {
          const float z = acc[r][c][q] + b3[col];
          tab[d * ld + col] = expf(fminf(fmaxf(z, -kClip), kClip));
        }
      }
    }
}

// bf16 inference copies: w1t[n][k] = W1[k][n] (k < d_in, else 0), w2t[n][k] =
// W2[k][n], w3t[n][k] = W3[k][n] (n < d_out, else 0).
__global__ void k_mlp_pack(int d_in, int k1, int d_out, int n3, const float* __restrict__ p, int64_t o_w1,
                           int64_t o_w2, int64_t o_w3, uint16_t* __restrict__ w1t, uint16_t* __restrict__ w2t,
                           uint16_t* __restrict__ w3t) {
  const int64_t t = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  const int64_t n1 = static_cast<int64_t>(kHidden) * k1, n2 = static_cast<int64_t>(kHidden) * kHidden;
  const int64_t n3t = static_cast<int64_t>(n3) * kHidden;
  if (t < n1) {
    const int n = static_cast<int>(t / k1), k = static_cast<int>(t % k1);
    w1t[t] = k < d_in ? f2bf(p[o_w1 + static_cast<int64_t>(k) * kHidden + n]) : 0;
  } else if (t < n1 + n2) {
    const int64_t u = t - n1;
    const int n = static_cast<int>(u / kHidden), k = static_cast<int>(u % kHidden);
    w2t[u] = f2bf(p[o_w2 + static_cast<int64_t>(k) * kHidden + n]);
  } else if (t < n1 + n2 + n3t) {
    const int64_t u = t - n1 - n2;
    const int n = static_cast<int>(u / kHidden), k = static_cast<int>(u % kHidden);
    w3t[u] = n < d_out ? f2bf(p[o_w3 + static_cast<int64_t>(k) * d_out + n]) : 0;
  }
}

// ---- training (fp32) ------------------------------------------------------------
__global__ void k_mlp_feat(int64_t ns, int nb, int d_in, const uint64_t* __restrict__ sdet, int64_t bcap,
                           const double* __restrict__ eps, float* __restrict__ x) {
  const int64_t t = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (t >= ns * d_in) return;
  const int64_t s = t / d_in;
  const int c = static_cast<int>(t % d_in);
  const int o = c < nb ? c : c - nb;
  const bool occ = (sdet[static_cast<int64_t>(o >> 6) * bcap + s] >> (o & 63)) & 1;
  x[t] = occ ? (c < nb ? 1.0f : static_cast<float>(eps[o])) : 0.0f;
}

// C[M][N] = A[M][K] op(B)[K][N] on fp32 matrix cores, op(B)[k][j] = TB ?
// B[j][k] : B[k][j].  A block makes a 64x64 tile of C, each of its four waves a
// 32x32 quarter as 2x2 tiles of v_mfma_f32_16x16x4_f32 (lane l feeds
// A[row l%16][k l/16] and B[k l/16][col l%16] and holds D[rows 4(l/16)..+3]
// [col l%16]).  K goes in slabs of 32 staged through LDS, the next slab's
// loads in flight while a slab is multiplied (a slab's 32 MFMAs take ~1000
// cycles, about one trip to L2).  Rows of Bs are 80 floats apart, so the four
// k groups of a fragment read 4 x 16 different banks.  The accumulation order
// is fixed by the tile shape, so results are deterministic.
// The epilogue is fused (kEpiBias: C = acc + bias; kEpiGelu: Z = acc + bias,
// C = gelu(Z); kEpiGeluBwd: C = acc * gelu'(Z)), which saves each hidden
// layer's separate pass over its 16384 x 256 activations.  At 16384 samples
// and nbasis 80 a product takes 31-36 us (43-60 TFLOP/s), bound by the LDS
// staging between barriers at 4 waves a block.
constexpr int kGemmTile = 64, kGemmSlab = 32;
constexpr int kGemmPer = kGemmTile * kGemmSlab / kBlock;  // elements of each operand a thread stages per slab
enum GemmEpilogue { kEpiBias, kEpiGelu, kEpiGeluBwd };

struct GemmTiles {
  float As[kGemmTile][kGemmSlab + 1];
  float Bs[kGemmSlab][kGemmTile + 16];
};
// acc += the staged slab's product for this wave's quarter (wr, wc).
__device__ __forceinline__ void gemm_slab(const GemmTiles& t, int lane, int wr, int wc, f32x4 (&acc)[2][2]) {
#pragma unroll
  for (int kk = 0; kk < kGemmSlab; kk += 4) {
    const int kq = kk + (lane >> 4);
    float av[2], bv[2];
#pragma unroll
    for (int a = 0; a < 2; ++a) av[a] = t.As[wr + a * 16 + (lane & 15)][kq];
#pragma unroll
    for (int b = 0; b < 2; ++b) bv[b] = t.Bs[kq][wc + b * 16 + (lane & 15)];
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
      for (int b = 0; b < 2; ++b) acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x4f32(av[a], bv[b], acc[a][b], 0, 0, 0);
  }
}

template <bool TB, GemmEpilogue E>
__global__ __launch_bounds__(kBlock) void k_gemm_mfma(int M, int N, int K, const float* __restrict__ A, int lda,
                                                      const float* __restrict__ B, int ldb,
                                                      const float* __restrict__ bias, float* __restrict__ Z,
                                                      float* __restrict__ C, int ldc) {
  __shared__ GemmTiles sm;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int i0 = blockIdx.y * kGemmTile, j0 = blockIdx.x * kGemmTile;
  const int wr = (wave >> 1) * 32, wc = (wave & 1) * 32;
  f32x4 acc[2][2];
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b) acc[a][b] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  float ra[kGemmPer], rb[kGemmPer];
  auto fetch = [&](int k0) {
#pragma unroll
    for (int q = 0; q < kGemmPer; ++q) {
      const int e = q * kBlock + tid;
      const int r = e >> 5, ka = k0 + (e & 31);  // consecutive threads along k
      ra[q] = (i0 + r < M && ka < K) ? A[static_cast<int64_t>(i0 + r) * lda + ka] : 0.0f;
      const int c = TB ? (e >> 5) : (e & 63), kb = k0 + (TB ? (e & 31) : (e >> 6));
      rb[q] = (j0 + c < N && kb < K)
                  ? (TB ? B[static_cast<int64_t>(j0 + c) * ldb + kb] : B[static_cast<int64_t>(kb) * ldb + j0 + c])
                  : 0.0f;
    }
  };
  fetch(0);
  for (int k0 = 0; k0 < K; k0 += kGemmSlab) {
    __syncthreads();  // the previous slab has been read
#pragma unroll
    for (int q = 0; q < kGemmPer; ++q) {
      const int e = q * kBlock + tid;
      sm.As[e >> 5][e & 31] = ra[q];
      if (TB)
        sm.Bs[e & 31][e >> 5] = rb[q];
      else
        sm.Bs[e >> 6][e & 63] = rb[q];
    }
    __syncthreads();
    if (k0 + kGemmSlab < K) fetch(k0 + kGemmSlab);
    gemm_slab(sm, lane, wr, wc, acc);
  }
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int gi = i0 + wr + a * 16 + (lane >> 4) * 4 + r, gj = j0 + wc + b * 16 + (lane & 15);
        if (gi >= M || gj >= N) continue;
        const int64_t o = static_cast<int64_t>(gi) * ldc + gj;
        if constexpr (E == kEpiGeluBwd) {
          C[o] = acc[a][b][r] * gelu_g(Z[o]);
        } else {
          const float z = acc[a][b][r] + bias[gj];
          if constexpr (E == kEpiGelu) {
            Z[o] = z;
            C[o] = gelu_f(z);
          } else {
            C[o] = z;
          }
        }
      }
}

// The three weight gradients act^T D (act [B][M], D [B][N], B samples) and bias
// gradients (column sums of D) in one launch: a block takes one 64x64 tile of
// one gradient over one chunk of the samples and writes it to that chunk's
// copy of the parameter vector; k_sum_splits adds the chunks in order.
// The gradients have only 12 + 16 + 12 tiles (nbasis 80), which without the
// split left 216 of the 256 CUs idle behind 1024 serial slabs: at 16384
// samples the three products and the column sums (then a kernel of one thread
// per column) took 18.4 of a training step's 19.5 ms, with 32 chunks 80 us
// (65 TFLOP/s; a large fp32 product reaches 153 here).
// Bias sums come from the D values the first row of tiles stages anyway.
struct WGrad {
  const float* act;
  const float* d;
  int M, N;
  int64_t o_w, o_b;  // offsets of the gradient and the bias gradient in the parameter vector
  int first;         // first tile of this gradient (tiles are numbered over all three)
};
struct WGrads {
  WGrad g[3];
  int tiles;
};
__global__ __launch_bounds__(kBlock) void k_wgrad(WGrads w, int64_t ns, int64_t chunk, int64_t stride,
                                                  float* __restrict__ part) {
  __shared__ GemmTiles sm;
  __shared__ float cs[kBlock];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int tile = blockIdx.x;
  const WGrad g = tile >= w.g[2].first ? w.g[2] : tile >= w.g[1].first ? w.g[1] : w.g[0];
  const int tn = (g.N + kGemmTile - 1) / kGemmTile, t = tile - g.first;
  const int i0 = (t / tn) * kGemmTile, j0 = (t % tn) * kGemmTile;
  const int64_t s0 = blockIdx.y * chunk, s1 = s0 + chunk < ns ? s0 + chunk : ns;
  float* out = part + static_cast<int64_t>(blockIdx.y) * stride;
  const int wr = (wave >> 1) * 32, wc = (wave & 1) * 32;
  f32x4 acc[2][2];
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b) acc[a][b] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  float ra[kGemmPer], rb[kGemmPer], csum = 0.0f;
  const int c = tid & 63;  // this thread's row of act^T and column of D
  auto fetch = [&](int64_t k0) {
#pragma unroll
    for (int q = 0; q < kGemmPer; ++q) {
      const int64_t k = k0 + q * (kBlock / 64) + wave;
      ra[q] = (i0 + c < g.M && k < s1) ? g.act[k * g.M + i0 + c] : 0.0f;
      rb[q] = (j0 + c < g.N && k < s1) ? g.d[k * g.N + j0 + c] : 0.0f;
    }
  };
  fetch(s0);
  for (int64_t k0 = s0; k0 < s1; k0 += kGemmSlab) {
    __syncthreads();
#pragma unroll
    for (int q = 0; q < kGemmPer; ++q) {
      const int kk = q * (kBlock / 64) + wave;
      sm.As[c][kk] = ra[q];
      sm.Bs[kk][c] = rb[q];
      csum += rb[q];
    }
    __syncthreads();
    if (k0 + kGemmSlab < s1) fetch(k0 + kGemmSlab);
    gemm_slab(sm, lane, wr, wc, acc);
  }
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int gi = i0 + wr + a * 16 + (lane >> 4) * 4 + r, gj = j0 + wc + b * 16 + (lane & 15);
        if (gi < g.M && gj < g.N) out[g.o_w + static_cast<int64_t>(gi) * g.N + gj] = acc[a][b][r];
      }
  if (i0 == 0) {  // block-uniform
    cs[tid] = csum;
    __syncthreads();
    if (wave == 0 && j0 + c < g.N) out[g.o_b + j0 + c] = (cs[c] + cs[64 + c]) + (cs[128 + c] + cs[192 + c]);
  }
}
// The gradient of each parameter: its chunks' partial sums in order.
__global__ void k_sum_splits(int64_t n, int64_t stride, int nsplit, const float* __restrict__ part,
                             float* __restrict__ g) {
  const int64_t t = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (t >= n) return;
  float acc = 0.0f;
#pragma unroll 8
  for (int z = 0; z < nsplit; ++z) acc += part[z * stride + t];
  g[t] = acc;
}
// Fixed-order sum of n doubles on one block (kSumBlock threads: 16384 values
// are 16 loads a thread, all in flight; 16.6 us with 256 threads, 4.7 now).
constexpr int kSumBlock = 1024;
__global__ __launch_bounds__(kSumBlock) void k_dsum(int64_t n, const double* __restrict__ x, double* __restrict__ out) {
  __shared__ double sh[kSumBlock];
  double acc = 0.0;
#pragma unroll 8
  for (int64_t i = threadIdx.x; i < n; i += kSumBlock) acc = acc + x[i];
  sh[threadIdx.x] = acc;
  __syncthreads();
  for (int k = kSumBlock / 2; k > 0; k >>= 1) {
    if (threadIdx.x < k) sh[threadIdx.x] = sh[threadIdx.x] + sh[threadIdx.x + k];
    __syncthreads();
  }
  if (threadIdx.x == 0) *out = sh[0];
}

// Weighted NLL of each sample's double under the network distribution and its
// gradient with respect to the logits (d3) and to the affinity rows of the
// sample's two holes (dth: row i then row j, nb each), one wavefront per sample.
// The network component sums four paths (h1, h2, p1, p2): the first particle
// p1 is drawn with h1's affinity over the unoccupied orbitals (normaliser
// Z1(h1)), its partner p2 with h2's affinity over p1's partner class (Z2).
// A sample flagged flat (sflat, may be null) is scored as a determinant the
// network does not run on: hole and particle weights 1 (logits 0), so only the
// affinity receives its gradient.
// Lane l holds orbitals l + 1 and l + 65 (nbasis <= 128): the rows of logits
// and affinities are read and the gradients written coalesced, each exponential
// is evaluated once, and 16384 samples are 16384 wavefronts.  (One thread per
// sample walked its rows twice at one wavefront per CU: 190 -> 21 us at 16384
// samples and nbasis 80, 142 -> 13 us at 4096 and 52.)
constexpr int kLossOrbs = 2;  // orbitals per lane
__device__ __forceinline__ double wave_dsum(double x) {
#pragma unroll
  for (int d = 32; d > 0; d >>= 1) x = x + __shfl_xor(x, d, 64);
  return x;
}
__global__ __launch_bounds__(kBlock) void k_mlp_loss_grad(
    fqd::Sys s, int64_t ns, int nb, int d_out, const uint64_t* __restrict__ sdet, int64_t bcap,
    const int32_t* __restrict__ sexc, const double* __restrict__ sw, const int32_t* __restrict__ sflat,
    const double* __restrict__ wsum, const float* __restrict__ z3, const float* __restrict__ th,
    float* __restrict__ d3, float* __restrict__ dth, double* __restrict__ sloss, const double* __restrict__ sh,
    int variance) {
  const int lane = threadIdx.x & 63;
  const int64_t t = static_cast<int64_t>(blockIdx.x) * (kBlock / 64) + (threadIdx.x >> 6);
  if (t >= ns) return;  // whole wavefront
  const float* z = z3 + t * d_out;
  float* d = d3 + t * d_out;
  float* gth = dth + t * 2 * nb;
  if (!(sw[t] > 0.0)) {
    for (int c = lane; c < d_out; c += 64) d[c] = 0.0f;
    for (int c = lane; c < 2 * nb; c += 64) gth[c] = 0.0f;
    if (lane == 0) sloss[t] = 0.0;
    return;
  }
  const double wt = sw[t] / *wsum;
  uint64_t f[FQ_MAX_WORDS] = {0, 0};
  for (int w = 0; w < s.W; ++w) f[w] = sdet[static_cast<int64_t>(w) * bcap + t];
  const int i = sexc[4 * t], j = sexc[4 * t + 1], a = sexc[4 * t + 2], b = sexc[4 * t + 3];
  const bool flat = sflat && sflat[t];
  auto clip = [](float x) { return static_cast<double>(fminf(fmaxf(x, -kClip), kClip)); };
  const fqd::PartnerClass cb = fqd::partner_class(s, i, j, a), ca = fqd::partner_class(s, i, j, b);
  auto in_class = [&](const fqd::PartnerClass& c, int o, int x) {
    return c.ok && o != x && fqd::ims_of(o) == c.ims && s.orb_sym[o - 1] == c.sym;
  };
  // e: hole weight of an occupied orbital; wi, wj: f_o A[i][o], f_o A[j][o] of an unoccupied one
  double e[kLossOrbs], wi[kLossOrbs], wj[kLossOrbs];
  float zh_[kLossOrbs], zp_[kLossOrbs], ti[kLossOrbs], tj[kLossOrbs];
  bool occ[kLossOrbs], inb[kLossOrbs], ina[kLossOrbs];
  // Z1(i), Z1(j); Z2 of holes i, j over b's class given a first (zbi, zbj) and a's given b (zai, zaj)
  double zh = 0.0, z1i = 0.0, z1j = 0.0, zbi = 0.0, zbj = 0.0, zai = 0.0, zaj = 0.0;
#pragma unroll
  for (int k = 0; k < kLossOrbs; ++k) {
    const int o = lane + 1 + 64 * k;
    e[k] = wi[k] = wj[k] = 0.0;
    zh_[k] = zp_[k] = ti[k] = tj[k] = 0.0f;
    occ[k] = inb[k] = ina[k] = false;
    if (o <= nb) {
      zh_[k] = z[o - 1];
      zp_[k] = z[nb + o - 1];
      ti[k] = th[(i - 1) * nb + o - 1];
      tj[k] = th[(j - 1) * nb + o - 1];
      occ[k] = (f[k] >> lane) & 1;
      if (occ[k]) {
        e[k] = flat ? 1.0 : exp(clip(zh_[k]));
      } else {
        const double v = flat ? 1.0 : exp(clip(zp_[k]));
        wi[k] = v * exp(clip(ti[k]));
        wj[k] = v * exp(clip(tj[k]));
        inb[k] = in_class(cb, o, a);
        ina[k] = in_class(ca, o, b);
      }
    }
    zh = zh + e[k];
    z1i = z1i + wi[k];
    z1j = z1j + wj[k];
    zbi = zbi + (inb[k] ? wi[k] : 0.0);
    zbj = zbj + (inb[k] ? wj[k] : 0.0);
    zai = zai + (ina[k] ? wi[k] : 0.0);
    zaj = zaj + (ina[k] ? wj[k] : 0.0);
  }
  zh = wave_dsum(zh);
  z1i = wave_dsum(z1i);
  z1j = wave_dsum(z1j);
  zbi = wave_dsum(zbi);
  zbj = wave_dsum(zbj);
  zai = wave_dsum(zai);
  zaj = wave_dsum(zaj);
  static_assert(kLossOrbs == 2, "an orbital's value is in one of two registers");
  auto at = [](const double(&v)[kLossOrbs], int o) { return __shfl(o > 64 ? v[1] : v[0], (o - 1) & 63, 64); };
  const double ei = at(e, i), ej = at(e, j);
  const double wia = at(wi, a), wib = at(wi, b), wja = at(wj, a), wjb = at(wj, b);
  const double pij = ei / zh * ej / (zh - ei), pji = ej / zh * ei / (zh - ej);
  const double t1 = pij * (wia / z1i) * (wjb / zbj);  // (i, j, a, b)
  const double t2 = pij * (wib / z1i) * (wja / zaj);  // (i, j, b, a)
  const double t3 = pji * (wja / z1j) * (wib / zbi);  // (j, i, a, b)
  const double t4 = pji * (wjb / z1j) * (wia / zai);  // (j, i, b, a)
  const double q = t1 + t2 + t3 + t4;
  const double r1 = t1 / q, r2 = t2 / q, r3 = t3 / q, r4 = t4 / q;
  // the sample's loss and the factor of its -log q gradient: the NLL weighted
  // by wt, or the spawning-variance term wt |H| / q, whose gradient is the NLL
  // gradient weighted by that term
  const double c = variance ? wt * sh[t] / q : wt;
  if (lane == 0) sloss[t] = variance ? c : wt * -log(q);
#pragma unroll
  for (int k = 0; k < kLossOrbs; ++k) {
    const int o = lane + 1 + 64 * k;
    if (o > nb) continue;
    double gu = 0.0, gi = 0.0, gj = 0.0;
    if (occ[k]) {
      double gij = -e[k] / zh - (o != i ? e[k] / (zh - ei) : 0.0);
      double gji = -e[k] / zh - (o != j ? e[k] / (zh - ej) : 0.0);
      if (o == i || o == j) {
        gij += 1.0;
        gji += 1.0;
      }
      gu = (r1 + r2) * gij + (r3 + r4) * gji;
    } else {
      const double da = o == a ? 1.0 : 0.0, db = o == b ? 1.0 : 0.0;
      gi = r1 * (da - wi[k] / z1i) + r2 * (db - wi[k] / z1i) + r3 * (db - (inb[k] ? wi[k] / zbi : 0.0)) +
           r4 * (da - (ina[k] ? wi[k] / zai : 0.0));
      gj = r1 * (db - (inb[k] ? wj[k] / zbj : 0.0)) + r2 * (da - (ina[k] ? wj[k] / zaj : 0.0)) +
           r3 * (da - wj[k] / z1j) + r4 * (db - wj[k] / z1j);
    }
    const bool in_h = !flat && fabsf(zh_[k]) < kClip, in_p = !flat && fabsf(zp_[k]) < kClip;
    d[o - 1] = in_h ? static_cast<float>(-c * gu) : 0.0f;
    d[nb + o - 1] = in_p ? static_cast<float>(-c * (gi + gj)) : 0.0f;
    gth[o - 1] = fabsf(ti[k]) < kClip ? static_cast<float>(-c * gi) : 0.0f;
    gth[nb + o - 1] = fabsf(tj[k]) < kClip ? static_cast<float>(-c * gj) : 0.0f;
  }
  for (int k = 2 * nb + lane; k < d_out; k += 64) d[k] = 0.0f;
}

// Affinity gradient, deterministic: block c adds, in sample order, the row
// gradients of the samples [c*chunk, (c+1)*chunk) to its copy of the table in
// LDS (thread o owns column o of every row) and writes it to part[c];
// k_aff_grad_sum adds the chunks in order.  Each sample's rows are read once,
// eight samples' loads in flight.  (A block per (hole, chunk) read every sample
// once per hole: 80 -> 18 us at 16384 samples and nbasis 80, 102 -> 22 us at
// 4096 and 52.)
constexpr int kAffAhead = 8;
__global__ __launch_bounds__(kHidden / 2) void k_aff_grad_part(int64_t ns, int nb, int64_t chunk,
                                                               const int32_t* __restrict__ sexc,
                                                               const double* __restrict__ sw,
                                                               const float* __restrict__ dth,
                                                               float* __restrict__ part) {
  extern __shared__ float tab[];  // nb x nb
  const int o = threadIdx.x;
  const int64_t s0 = blockIdx.x * chunk, s1 = s0 + chunk < ns ? s0 + chunk : ns;
  if (o < nb) {  // no barrier: a thread touches its own column only
    for (int h = 0; h < nb; ++h) tab[h * nb + o] = 0.0f;
    for (int64_t t0 = s0; t0 < s1; t0 += kAffAhead) {
      int hi[kAffAhead], hj[kAffAhead];  // 0: sample not used
      float gi[kAffAhead], gj[kAffAhead];
#pragma unroll
      for (int u = 0; u < kAffAhead; ++u) {
        const int64_t t = t0 + u < s1 ? t0 + u : s1 - 1;
        const bool use = t0 + u < s1 && sw[t] > 0.0;
        hi[u] = use ? sexc[4 * t] : 0;
        hj[u] = use ? sexc[4 * t + 1] : 0;
        gi[u] = dth[t * 2 * nb + o];
        gj[u] = dth[t * 2 * nb + nb + o];
      }
#pragma unroll
      for (int u = 0; u < kAffAhead; ++u) {
        if (hi[u]) {
          tab[(hi[u] - 1) * nb + o] += gi[u];
          tab[(hj[u] - 1) * nb + o] += gj[u];
        }
      }
    }
    float* out = part + static_cast<int64_t>(blockIdx.x) * nb * nb;
    for (int h = 0; h < nb; ++h) out[h * nb + o] = tab[h * nb + o];
  }
}

// 64 elements a block, its four wavefronts each adding a quarter of the chunks in order.
__global__ __launch_bounds__(kBlock) void k_aff_grad_sum(int nb, int nchunk, const float* __restrict__ part,
                                                         float* __restrict__ g) {
  __shared__ float sh[kBlock];
  const int64_t n = static_cast<int64_t>(nb) * nb;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int64_t k = static_cast<int64_t>(blockIdx.x) * 64 + lane;
  const int per = (nchunk + 3) / 4, c0 = wave * per, c1 = c0 + per < nchunk ? c0 + per : nchunk;
  float acc = 0.0f;
  if (k < n) {
#pragma unroll 8
    for (int c = c0; c < c1; ++c) acc += part[c * n + k];
  }
  sh[threadIdx.x] = acc;
  __syncthreads();
  if (wave == 0 && k < n) g[k] = (sh[lane] + sh[64 + lane]) + (sh[128 + lane] + sh[192 + lane]);
}

// Everything the generator reads of the affinity, one wavefront per (hole h,
// table): table 0 the whole row, table 1 + c the members of spin/irrep class c
// (in the class table's order).  The stored affinity is exp(clamp(theta, -60,
// 60)) rounded to float; its sums (rs, crs) are taken in row or member order,
// and the alias tables repeat generate_alias_tables' steps (fqd::build_alias)
// with the weights and its two stacks in LDS and the current top of "over" in
// a register.  Block 0 also writes the class bit masks.  (Table, sums and alias
// tables as three kernels, one thread per row or table with the stacks in
// scratch memory, took 142 us at nbasis 80; this takes 17.)
constexpr int kMaxAlias = 128;
__global__ __launch_bounds__(64) void k_aff_tables(int nb, const float* __restrict__ th, float* __restrict__ aff,
                                                   const int* __restrict__ nbss, const int* __restrict__ ssbf,
                                                   int nsym_pg, int max_sym_spin, double* __restrict__ rs,
                                                   double* __restrict__ crs, uint64_t* __restrict__ cmask,
                                                   double* __restrict__ au, int* __restrict__ ak,
                                                   double* __restrict__ cu, int* __restrict__ ck) {
  __shared__ double u[kMaxAlias];
  __shared__ int alias[kMaxAlias];
  __shared__ uint8_t under[kMaxAlias], over[kMaxAlias];
  const int ncls = 2 * nsym_pg, lane = threadIdx.x;
  const int h = blockIdx.x / (1 + ncls), c = blockIdx.x % (1 + ncls) - 1;
  if (blockIdx.x == 0 && lane < ncls) {
    uint64_t mw[FQ_MAX_WORDS] = {0, 0};
    for (int k = 0; k < nbss[lane]; ++k) {
      const int o = ssbf[lane * max_sym_spin + k] - 1;
      if (o < 64)
        mw[0] |= uint64_t{1} << o;
      else
        mw[1] |= uint64_t{1} << (o - 64);
    }
    for (int w = 0; w < FQ_MAX_WORDS; ++w) cmask[lane * FQ_MAX_WORDS + w] = mw[w];
  }
  const int n = c < 0 ? nb : nbss[c];
  for (int q = lane; q < n; q += 64) {
    const int o = c < 0 ? q : ssbf[c * max_sym_spin + q] - 1;
    const float a = static_cast<float>(exp(static_cast<double>(fminf(fmaxf(th[h * nb + o], -kClip), kClip))));
    u[q] = static_cast<double>(a);
    if (c < 0) aff[h * nb + q] = a;
  }
  __syncthreads();
  double tot = 0.0;
  for (int q = 0; q < n; ++q) tot = tot + u[q];
  if (lane == 0) {
    if (c < 0)
      rs[h] = tot;
    else
      crs[h * ncls + c] = tot;
  }
  if (n == 0) return;  // whole block
  __syncthreads();
  const double scale = static_cast<double>(n) / tot;
  int nunder = 0, nover = 0;  // the same in every lane
  for (int q0 = 0; q0 < n; q0 += 64) {
    const int q = q0 + lane;
    bool lo = false;
    if (q < n) {
      u[q] = u[q] * scale;
      lo = u[q] <= 1.0;
      alias[q] = q + 1;
    }
    const unsigned long long bl = __ballot(q < n && lo), bh = __ballot(q < n && !lo), below = (1ull << lane) - 1;
    if (q < n) {
      if (lo)
        under[nunder + __popcll(bl & below)] = static_cast<uint8_t>(q + 1);
      else
        over[nover + __popcll(bh & below)] = static_cast<uint8_t>(q + 1);
    }
    nunder += __popcll(bl);
    nover += __popcll(bh);
  }
  __syncthreads();
  if (lane == 0 && nover > 0) {
    int ov = over[nover - 1];
    double uo = u[ov - 1];
    while (nover > 0 && nunder > 0) {
      const int un = under[--nunder];
      alias[un - 1] = ov;
      uo = uo - (1.0 - u[un - 1]);
      if (uo < 1.0) {
        u[ov - 1] = uo;
        under[nunder++] = static_cast<uint8_t>(ov);
        if (--nover > 0) {
          ov = over[nover - 1];
          uo = u[ov - 1];
        }
      }
    }
    if (nover > 0) u[ov - 1] = uo;
  }
  __syncthreads();
  const int64_t o0 = c < 0 ? static_cast<int64_t>(h) * nb : (static_cast<int64_t>(h) * ncls + c) * max_sym_spin;
  for (int q = lane; q < n; q += 64) {
    (c < 0 ? au : cu)[o0 + q] = u[q];
    (c < 0 ? ak : ck)[o0 + q] = alias[q];
  }
}

// Adam over all parameters; those from o_th on (the affinity) with their own rate.
__global__ void k_adam(int64_t n, int64_t o_th, float* __restrict__ p, const float* __restrict__ g,
                       float* __restrict__ m, float* __restrict__ v, float lr_net, float lr_aff, float c1, float c2) {
  const int64_t t = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (t >= n) return;
  const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
  const float lr = t < o_th ? lr_net : lr_aff;
  const float gt = g[t];
  const float mt = b1 * m[t] + (1.0f - b1) * gt;
  const float vt = b2 * v[t] + (1.0f - b2) * gt * gt;
  m[t] = mt;
  v[t] = vt;
  p[t] = p[t] - lr * (mt / c1) / (sqrtf(vt / c2) + eps);
}

// ---- heat-bath training samples -------------------------------------------------
__global__ void k_det_weight(int64_t n, int64_t cap, int S, const int64_t* __restrict__ pop, int shift,
                             int64_t* __restrict__ out) {
  const int64_t d = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (d >= n) return;
  int64_t w = 1;
  for (int q = 0; q < S; ++q) {
    const int64_t p = pop[q * cap + d];
    w += (p < 0 ? -p : p) >> shift;
  }
  out[d] = w;
}

// One heat-bath training sample per thread; its determinant is flagged flat
// when even rounded up it makes fewer than min_att attempts (the network does
// not run on it in production).  Blocks of one wavefront, the generator's nel
// on-the-fly weights in a column of LDS each: 16384 samples are one wavefront
// per CU, so the chain of dependent reads (the search of the list, the tables)
// sets the time: 60 us, 82 with the weights in scratch memory.
constexpr int kSampleBlock = 64;
__global__ __launch_bounds__(kSampleBlock) void k_hb_sample(fqd::Sys s, const uint64_t* __restrict__ det, int64_t cap, int64_t n,
                            const int64_t* __restrict__ cum, const int64_t* __restrict__ dw, int64_t min_att,
                            int64_t ns, uint64_t seed, uint32_t step, uint64_t* __restrict__ sdet, int64_t bcap,
                            int32_t* __restrict__ sexc, double* __restrict__ sw, int32_t* __restrict__ sflat,
                            double* __restrict__ sh) {
  extern __shared__ double hb_lds[];
  const int64_t t = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (t >= ns) return;
  fqd::Philox rng(seed, static_cast<uint32_t>(t), static_cast<uint32_t>(t >> 32), step ^ (fqd::kDrawTrain << 24));
  const int64_t total = cum[n];
  const int64_t target = static_cast<int64_t>(rng.next() * static_cast<double>(total));
  int64_t lo = 0, hi = n - 1;  // last d with cum[d] <= target
  while (lo < hi) {
    const int64_t mid = (lo + hi + 1) >> 1;
    if (cum[mid] <= target)
      lo = mid;
    else
      hi = mid - 1;
  }
  uint64_t f[FQ_MAX_WORDS] = {0, 0};
  FQ_FOR_WORDS(w, s.W) f[w] = det[static_cast<int64_t>(w) * cap + lo];
  fqd::Excit conn;
  double h = 0.0, pgen = 1.0;
  fqd::gen_heat_bath(s, rng, f, conn, h, pgen, fqd::HbBuf{hb_lds + threadIdx.x, kSampleBlock});
  FQ_FOR_WORDS(w, s.W) sdet[static_cast<int64_t>(w) * bcap + t] = f[w];
  const bool use = conn.nexcit == 2 && h != 0.0;
  sexc[4 * t] = conn.from[0];
  sexc[4 * t + 1] = conn.from[1];
  sexc[4 * t + 2] = conn.to[0];
  sexc[4 * t + 3] = conn.to[1];
  sw[t] = use ? fabs(h) / pgen : 0.0;
  sh[t] = use ? fabs(h) : 0.0;
  sflat[t] = dw[lo] < min_att ? 1 : 0;  // dw = 1 + sum of floor|N|
}

template <class T>
int dalloc(T** p, int64_t count) {
  if (count < 1) count = 1;
  return hipMalloc(reinterpret_cast<void**>(p), sizeof(T) * static_cast<size_t>(count)) == hipSuccess
             ? FQ_OK
             : FQ_ERR_NOMEM;
}
template <class T>
void dfree(T*& p) {
  if (p) (void)hipFree(p);
  p = nullptr;
}

template <bool TB, GemmEpilogue E>
void gemm(int M, int N, int K, const float* A, int lda, const float* B, int ldb, const float* bias, float* Z,
          float* C, int ldc, hipStream_t st) {
  hipLaunchKernelGGL((k_gemm_mfma<TB, E>), dim3(static_cast<unsigned>(ceil_div(N, kGemmTile)),
                                               static_cast<unsigned>(ceil_div(M, kGemmTile))),
                     dim3(kBlock), 0, st, M, N, K, A, lda, B, ldb, bias, Z, C, ldc);
}

// splitmix64 -> standard normal (Box--Muller) for parameter initialisation.
struct HostNormal {
  uint64_t x;
  uint64_t next_u64() {
    uint64_t z = (x += 0x9E3779B97F4A7C15ULL);
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ULL;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBULL;
    return z ^ (z >> 31);
  }
  double uniform() { return (static_cast<double>(next_u64() >> 11) + 0.5) * (1.0 / 9007199254740992.0); }
  double normal() { return std::sqrt(-2.0 * std::log(uniform())) * std::cos(6.283185307179586 * uniform()); }
};

}  // namespace

int mlp_alloc(Mlp& m, int nb, int W, int64_t bcap) {
  m.nb = nb;
  m.d_in = m.d_out = 2 * nb;
  m.k1 = static_cast<int>(ceil_div(m.d_in, 32) * 32);
  m.n3 = static_cast<int>(ceil_div(m.d_out, 16) * 16);
  if (m.k1 > kHidden || m.n3 > kHidden) return FQ_ERR_ARG;
  m.o_w1 = 0;
  m.o_b1 = m.o_w1 + static_cast<int64_t>(m.d_in) * kHidden;
  m.o_w2 = m.o_b1 + kHidden;
  m.o_b2 = m.o_w2 + static_cast<int64_t>(kHidden) * kHidden;
  m.o_w3 = m.o_b2 + kHidden;
  m.o_b3 = m.o_w3 + static_cast<int64_t>(kHidden) * m.d_out;
  m.o_th = m.o_b3 + m.d_out;
  m.nparams = m.o_th + static_cast<int64_t>(nb) * nb;
  m.bcap = bcap;
  m.nchunk = static_cast<int>(ceil_div(bcap, kAffChunk));
  int rc = FQ_OK;
  rc |= dalloc(&m.p, m.nparams);
  rc |= dalloc(&m.g, m.nparams);
  rc |= dalloc(&m.m, m.nparams);
  rc |= dalloc(&m.v, m.nparams);
  rc |= dalloc(&m.w1t, static_cast<int64_t>(kHidden) * m.k1);
  rc |= dalloc(&m.w2t, static_cast<int64_t>(kHidden) * kHidden);
  rc |= dalloc(&m.w3t, static_cast<int64_t>(m.n3) * kHidden);
  rc |= dalloc(&m.x, bcap * m.d_in);
  rc |= dalloc(&m.z1, bcap * kHidden);
  rc |= dalloc(&m.a1, bcap * kHidden);
  rc |= dalloc(&m.z2, bcap * kHidden);
  rc |= dalloc(&m.a2, bcap * kHidden);
  rc |= dalloc(&m.z3, bcap * m.d_out);
  rc |= dalloc(&m.d3, bcap * m.d_out);
  rc |= dalloc(&m.d2, bcap * kHidden);
  rc |= dalloc(&m.d1, bcap * kHidden);
  rc |= dalloc(&m.sdet, bcap * W);
  rc |= dalloc(&m.sexc, bcap * 4);
  rc |= dalloc(&m.sw, bcap);
  rc |= dalloc(&m.sh, bcap);
  rc |= dalloc(&m.sflat, bcap);
  rc |= dalloc(&m.sloss, bcap);
  rc |= dalloc(&m.dsum, 2);
  rc |= dalloc(&m.aff, static_cast<int64_t>(nb) * nb);
  rc |= dalloc(&m.dth, bcap * 2 * nb);
  rc |= dalloc(&m.aff_part, static_cast<int64_t>(m.nchunk) * nb * nb);
  rc |= dalloc(&m.gpart, static_cast<int64_t>(kGradSplits) * m.o_th);
  return rc == FQ_OK ? FQ_OK : FQ_ERR_NOMEM;
}

void mlp_free(Mlp& m) {
  dfree(m.p);
  dfree(m.g);
  dfree(m.m);
  dfree(m.v);
  dfree(m.w1t);
  dfree(m.w2t);
  dfree(m.w3t);
  dfree(m.x);
  dfree(m.z1);
  dfree(m.a1);
  dfree(m.z2);
  dfree(m.a2);
  dfree(m.z3);
  dfree(m.d3);
  dfree(m.d2);
  dfree(m.d1);
  dfree(m.sdet);
  dfree(m.sexc);
  dfree(m.sw);
  dfree(m.sh);
  dfree(m.sflat);
  dfree(m.sloss);
  dfree(m.dsum);
  dfree(m.aff);
  dfree(m.rs);
  dfree(m.crs);
  dfree(m.cmask);
  dfree(m.au);
  dfree(m.ak);
  dfree(m.cu);
  dfree(m.ck);
  dfree(m.dth);
  dfree(m.aff_part);
  dfree(m.gpart);
  dfree(m.scum);
  dfree(m.swts);
  m.scum_cap = 0;
}

int mlp_refresh(Mlp& m, hipStream_t st) {
  const int64_t total = static_cast<int64_t>(kHidden) * m.k1 + static_cast<int64_t>(kHidden) * kHidden +
                        static_cast<int64_t>(m.n3) * kHidden;
  hipLaunchKernelGGL(k_mlp_pack, dim3(blocks(total)), dim3(kBlock), 0, st, m.d_in, m.k1, m.d_out, m.n3, m.p, m.o_w1,
                     m.o_w2, m.o_w3, m.w1t, m.w2t, m.w3t);
  if (m.nbss)
    hipLaunchKernelGGL(k_aff_tables, dim3(static_cast<unsigned>(m.nb * (1 + 2 * m.nsym_pg))), dim3(64), 0, st, m.nb,
                       m.p + m.o_th, m.aff, m.nbss, m.ssbf, m.nsym_pg, m.max_sym_spin, m.rs, m.crs, m.cmask, m.au,
                       m.ak, m.cu, m.ck);
  MLP_HIP(hipGetLastError());
  return FQ_OK;
}

int mlp_set_classes(Mlp& m, const int* nbss, const int* ssbf, int nsym_pg, int max_sym_spin) {
  m.nbss = nbss;
  m.ssbf = ssbf;
  m.nsym_pg = nsym_pg;
  m.max_sym_spin = max_sym_spin;
  int rc = dalloc(&m.rs, m.nb);
  rc |= dalloc(&m.crs, static_cast<int64_t>(m.nb) * 2 * nsym_pg);
  rc |= dalloc(&m.cmask, static_cast<int64_t>(2) * nsym_pg * FQ_MAX_WORDS);
  rc |= dalloc(&m.au, static_cast<int64_t>(m.nb) * m.nb);
  rc |= dalloc(&m.ak, static_cast<int64_t>(m.nb) * m.nb);
  rc |= dalloc(&m.cu, static_cast<int64_t>(m.nb) * 2 * nsym_pg * max_sym_spin);
  rc |= dalloc(&m.ck, static_cast<int64_t>(m.nb) * 2 * nsym_pg * max_sym_spin);
  return rc == FQ_OK ? FQ_OK : FQ_ERR_NOMEM;
}

int mlp_set(Mlp& m, const float* host, hipStream_t st) {
  MLP_HIP(hipMemcpyAsync(m.p, host, sizeof(float) * m.nparams, hipMemcpyHostToDevice, st));
  MLP_HIP(hipMemsetAsync(m.m, 0, sizeof(float) * m.nparams, st));
  MLP_HIP(hipMemsetAsync(m.v, 0, sizeof(float) * m.nparams, st));
  m.adam_t = 0;
  int rc = mlp_refresh(m, st);
  if (rc != FQ_OK) return rc;
  MLP_HIP(hipStreamSynchronize(st));
  return FQ_OK;
}

int mlp_init(Mlp& m, uint64_t seed, hipStream_t st) {
  std::vector<float> h(static_cast<size_t>(m.nparams), 0.0f);
  HostNormal rng{seed ^ 0x5DEECE66DULL};
  auto fill = [&](int64_t off, int64_t count, double sd) {
    for (int64_t k = 0; k < count; ++k) h[off + k] = static_cast<float>(sd * rng.normal());
  };
  fill(m.o_w1, static_cast<int64_t>(m.d_in) * kHidden, 1.0 / std::sqrt(static_cast<double>(m.d_in)));
  fill(m.o_w2, static_cast<int64_t>(kHidden) * kHidden, 1.0 / std::sqrt(static_cast<double>(kHidden)));
  // small output layer: the initial proposal is close to uniform
  fill(m.o_w3, static_cast<int64_t>(kHidden) * m.d_out, 0.1 / std::sqrt(static_cast<double>(kHidden)));
  return mlp_set(m, h.data(), st);
}

int mlp_infer(const Mlp& m, const fqd::Sys& s, const uint64_t* det, int64_t cap, int64_t n, float* tab,
              hipStream_t st, const int64_t* idx, const int64_t* pn, int64_t like) {
  if (n <= 0) return FQ_OK;
  const int rt = (pn ? std::min(like, n) : n) <= kFewRows ? 1 : 4;
  hipLaunchKernelGGL(rt == 1 ? k_mlp_infer<1> : k_mlp_infer<4>, dim3(static_cast<unsigned>(ceil_div(n, 16 * rt))),
                     dim3(kBlock), 0, st, m.nb, m.k1, m.n3, m.d_out, det, cap, n, idx, s.sp_eigv, m.w1t, m.p + m.o_b1,
                     m.w2t, m.p + m.o_b2, m.w3t, m.p + m.o_b3, tab, static_cast<int64_t>(m.d_out), pn);
  MLP_HIP(hipGetLastError());
  return FQ_OK;
}

int mlp_train_step(Mlp& m, const fqd::Sys& s, int64_t ns, double lr, bool apply, hipStream_t st) {
  if (ns < 1 || ns > m.bcap) return FQ_ERR_ARG;
  const int H = kHidden, di = m.d_in, dout = m.d_out, B = static_cast<int>(ns);
  hipLaunchKernelGGL(k_mlp_feat, dim3(blocks(ns * di)), dim3(kBlock), 0, st, ns, m.nb, di, m.sdet, m.bcap,
                     s.sp_eigv, m.x);
  gemm<false, kEpiGelu>(B, H, di, m.x, di, m.p + m.o_w1, H, m.p + m.o_b1, m.z1, m.a1, H, st);
  gemm<false, kEpiGelu>(B, H, H, m.a1, H, m.p + m.o_w2, H, m.p + m.o_b2, m.z2, m.a2, H, st);
  gemm<false, kEpiBias>(B, dout, H, m.a2, H, m.p + m.o_w3, dout, m.p + m.o_b3, nullptr, m.z3, dout, st);
  hipLaunchKernelGGL(k_dsum, dim3(1), dim3(kSumBlock), 0, st, ns, m.sw, m.dsum);
  hipLaunchKernelGGL(k_mlp_loss_grad, dim3(blocks(ns * 64)), dim3(kBlock), 0, st, s, ns, m.nb, dout, m.sdet, m.bcap,
                     m.sexc, m.sw, m.sflat, m.dsum, m.z3, m.p + m.o_th, m.d3, m.dth, m.sloss, m.sh, m.objective);
  hipLaunchKernelGGL(k_dsum, dim3(1), dim3(kSumBlock), 0, st, ns, m.sloss, m.dsum + 1);
  const int nchunk = static_cast<int>(ceil_div(ns, kAffChunk));
  const int64_t na = static_cast<int64_t>(m.nb) * m.nb;
  hipLaunchKernelGGL(k_aff_grad_part, dim3(static_cast<unsigned>(nchunk)), dim3(kHidden / 2),
                     sizeof(float) * static_cast<size_t>(na), st, ns, m.nb, static_cast<int64_t>(kAffChunk), m.sexc,
                     m.sw, m.dth, m.aff_part);
  hipLaunchKernelGGL(k_aff_grad_sum, dim3(static_cast<unsigned>(ceil_div(na, 64))), dim3(kBlock), 0, st, m.nb, nchunk,
                     m.aff_part, m.g + m.o_th);
  // backward
  gemm<true, kEpiGeluBwd>(B, H, dout, m.d3, dout, m.p + m.o_w3, dout, nullptr, m.z2, m.d2, H, st);
  gemm<true, kEpiGeluBwd>(B, H, H, m.d2, H, m.p + m.o_w2, H, nullptr, m.z1, m.d1, H, st);
  // weight and bias gradients: chunks of at least 4 slabs of samples, at most kGradSplits of them
  const int64_t chunk = std::max<int64_t>(4 * kGemmSlab, ceil_div(ceil_div(ns, kGradSplits), kGemmSlab) * kGemmSlab);
  const int nsplit = static_cast<int>(ceil_div(ns, chunk));
  WGrads wg;
  wg.g[0] = WGrad{m.x, m.d1, di, H, m.o_w1, m.o_b1, 0};
  wg.g[1] = WGrad{m.a1, m.d2, H, H, m.o_w2, m.o_b2, 0};
  wg.g[2] = WGrad{m.a2, m.d3, H, dout, m.o_w3, m.o_b3, 0};
  wg.tiles = 0;
  for (auto& g : wg.g) {
    g.first = wg.tiles;
    wg.tiles += static_cast<int>(ceil_div(g.M, kGemmTile) * ceil_div(g.N, kGemmTile));
  }
  hipLaunchKernelGGL(k_wgrad, dim3(static_cast<unsigned>(wg.tiles), static_cast<unsigned>(nsplit)), dim3(kBlock), 0, st,
                     wg, ns, chunk, m.o_th, m.gpart);
  hipLaunchKernelGGL(k_sum_splits, dim3(blocks(m.o_th)), dim3(kBlock), 0, st, m.o_th, m.o_th, nsplit, m.gpart, m.g);
  MLP_HIP(hipGetLastError());
  if (apply) {
    m.adam_t += 1;
    const float c1 = static_cast<float>(1.0 - std::pow(0.9, static_cast<double>(m.adam_t)));
    const float c2 = static_cast<float>(1.0 - std::pow(0.999, static_cast<double>(m.adam_t)));
    hipLaunchKernelGGL(k_adam, dim3(blocks(m.nparams)), dim3(kBlock), 0, st, m.nparams, m.o_th, m.p, m.g, m.m, m.v,
                       static_cast<float>(lr), static_cast<float>(lr * kAffLrScale), c1, c2);
    MLP_HIP(hipGetLastError());
    return mlp_refresh(m, st);
  }
  return FQ_OK;
}

int mlp_sample(Mlp& m, const fqd::Sys& s, const uint64_t* det, const int64_t* pop, int64_t cap, int64_t n,
               int64_t ns, int64_t min_att, uint64_t seed, uint32_t step, hipStream_t st,
               int (*scan)(void* ctx, const int64_t* in, int64_t* out, int64_t n), void* scan_ctx) {
  if (n < 1 || ns < 1 || ns > m.bcap) return FQ_ERR_ARG;
  if (m.scum_cap < n + 1) {
    dfree(m.scum);
    dfree(m.swts);
    m.scum_cap = 0;
    if (dalloc(&m.scum, n + 1) != FQ_OK || dalloc(&m.swts, n + 1) != FQ_OK) return FQ_ERR_NOMEM;
    m.scum_cap = n + 1;
  }
  int shift = 0;
  while ((int64_t{1} << shift) < s.rf) ++shift;
  // per-determinant weights, their exclusive prefix (total at scum[n]), then the samples
  hipLaunchKernelGGL(k_det_weight, dim3(blocks(n)), dim3(kBlock), 0, st, n, cap, s.S, pop, shift, m.swts);
  int rc = scan(scan_ctx, m.swts, m.scum, n);
  if (rc != FQ_OK) return rc;
  hipLaunchKernelGGL(k_hb_sample, dim3(static_cast<unsigned>(ceil_div(ns, kSampleBlock))), dim3(kSampleBlock),
                     sizeof(double) * static_cast<size_t>(s.nel) * kSampleBlock, st, s, det, cap, n, m.scum, m.swts, min_att,
                     ns, seed, step, m.sdet, m.bcap, m.sexc, m.sw, m.sflat, m.sh);
  MLP_HIP(hipGetLastError());
  return FQ_OK;
}

}  // namespace fqm
