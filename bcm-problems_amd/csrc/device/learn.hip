// Learned initial guess: a small MLP trained on the GPU with hand-written
// BF16 MFMA kernels, and the POD bases its outputs are coefficients in.
//
// MLP: nin -> nh (tanh) -> nh (tanh) -> nout (linear). Weights are kept as
// FP32 masters with BF16 copies; every product runs on the matrix cores as
// v_mfma_f32_16x16x32_bf16 (BF16 operands, FP32 accumulation): activations
// and gradients are rounded to BF16 as they are loaded into the MFMA, the
// results stay FP32. Training is full-batch Adam on a mean-squared loss.
//
// POD: for each right-hand side the basis is the leading left singular
// vectors of the snapshot matrix S (n x k, FP64), from a randomized range
// finder with power iterations and Cholesky-QR orthonormalisation: every
// product with S runs on the device (tall-skinny FP64 kernels), only r x r
// and r x k matrices (r <= 96) reach the host.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <random>

#include "dev_common.hpp"
#include "learn.hpp"

namespace bcm {

namespace {

typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef unsigned short v8u __attribute__((ext_vector_type(8)));
typedef float v4f __attribute__((ext_vector_type(4)));

// float -> bf16, round to nearest even (NaN kept quiet).
__device__ __forceinline__ unsigned short f2bf(float f) {
  uint32_t u = __float_as_uint(f);
  if ((u & 0x7fffffffu) > 0x7f800000u) return (unsigned short)((u >> 16) | 0x40u);
  u += 0x7fffu + ((u >> 16) & 1u);
  return (unsigned short)(u >> 16);
}

__device__ __forceinline__ float ldf(const float* p, size_t i) { return p[i]; }
__device__ __forceinline__ float ldf(const unsigned short* p, size_t i) {
  return __uint_as_float((uint32_t)p[i] << 16);
}

// C(i,j) = epilogue(sum_k A(i,k) B(k,j)) with A(i,k) = A[i*ars + k*acs] and
// B(k,j) = B[k*brs + j*bcs] (strides express the transposes). One wave per
// 16 x 16 tile of C, K in steps of 32 (zero padded). Epilogue: + bias[j],
// then tanh (act == 1), then * (1 - D(i,j)^2) with D(i,j) = dmul[i*ldd + j].
template <class TA, class TB>
__global__ __launch_bounds__(256) void k_gemm_bf16(int M, int N, int K, const TA* __restrict__ A, int ars, int acs,
                                                   const TB* __restrict__ B, int brs, int bcs, float* __restrict__ C,
                                                   int ldc, const float* __restrict__ bias, int act,
                                                   const float* __restrict__ dmul, int ldd) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int tiles_n = (N + 15) >> 4;
  const int tiles = ((M + 15) >> 4) * tiles_n;
  const int tile = blockIdx.x * 4 + wave;
  if (tile >= tiles) return;  // wave-uniform: no block-level synchronisation below
  const int tm = tile / tiles_n, tn = tile - tm * tiles_n;
  const int r = lane & 15, g = lane >> 4;
  const int ia = tm * 16 + r;  // row of A this lane feeds
  const int jb = tn * 16 + r;  // column of B this lane feeds
  v4f acc = {0.f, 0.f, 0.f, 0.f};
  // split K: wave group blockIdx.y adds the K range [kz0, kz1) into its own
  // partial tile (C + blockIdx.y * M * ldc); no epilogue then
  const int kper = (((K + gridDim.y - 1) / gridDim.y) + 31) / 32 * 32;
  const int kz0 = blockIdx.y * kper, kz1 = min(K, kz0 + kper);
  C += (size_t)blockIdx.y * M * ldc;
  for (int k0 = kz0; k0 < kz1; k0 += 32) {
    v8u av, bv;
#pragma unroll
    for (int t = 0; t < 8; ++t) {
      const int k = k0 + 8 * g + t;
      av[t] = (ia < M && k < kz1) ? f2bf(ldf(A, (size_t)ia * ars + (size_t)k * acs)) : (unsigned short)0;
      bv[t] = (jb < N && k < kz1) ? f2bf(ldf(B, (size_t)k * brs + (size_t)jb * bcs)) : (unsigned short)0;
    }
    acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8bf, av), __builtin_bit_cast(v8bf, bv), acc,
                                                  0, 0, 0);
  }
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    const int i = tm * 16 + 4 * g + t, j = tn * 16 + r;
    if (i < M && j < N) {
      float v = acc[t];
      if (bias) v += bias[j];
      if (act == 1) v = tanhf(v);
      if (dmul) {
        const float d = dmul[(size_t)i * ldd + j];
        v *= 1.0f - d * d;
      }
      C[(size_t)i * ldc + j] = v;
    }
  }
}

// Column sums db[j] = sum_i dz[i*ld + j] in two deterministic passes: block
// (tile, chunk) adds rows [chunk*rows_per, ...) of 64 columns (4 row phases
// per column, combined in a fixed order) into part[chunk*N + j]; k_colsum_fin
// adds the chunks in order.
constexpr int kColChunks = 32;
__global__ __launch_bounds__(256) void k_colsum(int M, int N, const float* __restrict__ dz, int ld,
                                                float* __restrict__ part) {
  __shared__ float sm[4][64];
  const int c = threadIdx.x & 63, ph = threadIdx.x >> 6;
  const int j = blockIdx.x * 64 + c;
  const int per = (M + kColChunks - 1) / kColChunks;
  const int i0 = blockIdx.y * per, i1 = min(M, i0 + per);
  float s = 0.f;
  if (j < N)
    for (int i = i0 + ph; i < i1; i += 4) s += dz[(size_t)i * ld + j];
  sm[ph][c] = s;
  __syncthreads();
  if (ph == 0 && j < N) part[(size_t)blockIdx.y * N + j] = ((sm[0][c] + sm[1][c]) + sm[2][c]) + sm[3][c];
}

__global__ void k_colsum_fin(int N, const float* __restrict__ part, float* __restrict__ db) {
  const int j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= N) return;
  float s = 0.f;
  for (int k = 0; k < kColChunks; ++k) s += part[(size_t)k * N + j];
  db[j] = s;
}

void colsum(hipStream_t s, int M, int N, const float* dz, int ld, float* db, float* part) {
  hipLaunchKernelGGL(k_colsum, dim3((N + 63) / 64, kColChunks), dim3(256), 0, s, M, N, dz, ld, part);
  hipLaunchKernelGGL(k_colsum_fin, dim3((N + 255) / 256), dim3(256), 0, s, N, part, db);
  BCM_HIP(hipGetLastError());
}

// dy = 2 (y - t) / (M N); per-block partials of sum (y - t)^2.
__global__ __launch_bounds__(256) void k_mse(int64_t total, const float* __restrict__ y, const float* __restrict__ t,
                                             float scale, float* __restrict__ dy, double* partials) {
  double acc[1] = {0.0};
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += stride) {
    const float d = y[i] - t[i];
    dy[i] = scale * d;
    acc[0] += (double)d * (double)d;
  }
  block_partials<1>(acc, partials);
}

__global__ __launch_bounds__(256) void k_sum_to(const double* partials, int nb, double scale, double* out) {
  const double s = sum_partials(partials, nb, 1, 0);
  if (threadIdx.x == 0) *out = s * scale;
}

// Adam step over all parameters; refreshes the bf16 copies of the weights.
__global__ void k_adam(int64_t n, float* __restrict__ w, const float* __restrict__ gr, float* __restrict__ m,
                       float* __restrict__ v, unsigned short* __restrict__ wb, const unsigned char* __restrict__ is_w,
                       const int64_t* __restrict__ wb_index, float lr, float b1, float b2, float eps, float c1,
                       float c2) {
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
    const float g = gr[i];
    const float mi = b1 * m[i] + (1.f - b1) * g;
    const float vi = b2 * v[i] + (1.f - b2) * g * g;
    m[i] = mi;
    v[i] = vi;
    const float wi = w[i] - lr * (mi / c1) / (sqrtf(vi / c2) + eps);
    w[i] = wi;
    if (is_w[i]) wb[wb_index[i]] = f2bf(wi);
  }
}

__global__ void k_to_bf16(int64_t n, const float* __restrict__ w, unsigned short* __restrict__ wb) {
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) wb[i] = f2bf(w[i]);
}

// ---- the network in fused kernels ----
//
// At the sizes a guess model has (a few hundred neurons, up to some thousand
// cells) a training step is 1 GFLOP over 1 MB: as one launch per product, bias
// sum and reduction (21 of them) it took 263 us at 1024 x 4-256-256-384, all of
// it launches and gathers of 2-byte operands. It is now three launches:
//  * k_mlp_chain: 16 rows of the batch per workgroup through the whole network,
//    the loss, and back through the activations; rows stay in LDS.
//  * k_mlp_wgrad: all weight and bias gradients and the loss sum.
//  * k_mlp_adam.
// Operands are kept as MFMA fragments, so that every load is 16 bytes a lane
// and consecutive over the wave. A fragment holds, for 16 columns j and 32
// steps k of the contraction, lane (j % 16) + 16 * (k % 32 / 8) its 8 values k
// % 8; columns and steps past the end are zero. Weights are packed once per
// update (for the products and, transposed, for the way back); activations and
// their gradients are written as fragments over the rows of the batch.
// Chosen where the rows of a workgroup fit 63 KB of LDS; larger networks
// take one product after another (k_gemm_bf16).
constexpr int kFrag = 512;            // values of a fragment
constexpr int kChainWaves = 16;       // most waves of a workgroup: one 16-column tile per wave and pass

__host__ __device__ constexpr int up16(int n) { return (n + 15) & ~15; }
__host__ __device__ constexpr int up32(int n) { return (n + 31) & ~31; }

// Offset of element (k, j) in fragments of `ks` steps of 32 per column tile.
__device__ __forceinline__ size_t frag_at(int k, int j, int ks) {
  return ((size_t)(j >> 4) * ks + (k >> 5)) * kFrag + (size_t)((j & 15) + 16 * ((k & 31) >> 3)) * 8 + (k & 7);
}

// Sizes and the packed weights: f[l] for the product with W_l, r[l] (layers 1
// and 2) for the product with its transpose.
struct MlpDims {
  int nin, nh, nout;
  int64_t w_off[3], b_off[3];
  int64_t f[3], r[3];
};

__device__ __forceinline__ void pack_weight(const MlpDims& d, int64_t i, unsigned short v, unsigned short* pk) {
  for (int l = 0; l < 3; ++l) {
    if (i < d.w_off[l] || i >= d.b_off[l]) continue;
    const int nj = l == 2 ? d.nout : d.nh, nk = l == 0 ? d.nin : d.nh;
    const int e = (int)(i - d.w_off[l]), k = e / nj, j = e - k * nj;
    pk[d.f[l] + frag_at(k, j, up32(nk) >> 5)] = v;
    if (l > 0) pk[d.r[l] + frag_at(j, k, up32(nj) >> 5)] = v;
  }
}

__global__ void k_mlp_pack(int64_t n, MlpDims d, const float* __restrict__ w, unsigned short* __restrict__ pk) {
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) pack_weight(d, i, f2bf(w[i]), pk);
}

// What a pass over the batch leaves for the gradients: fragments over the rows
// (the k of the gradient products) and per-16-row sums.
struct MlpTape {
  unsigned short *x, *h1, *h2, *dz1, *dz2, *dy;
  float* colpart;    // per row tile: column sums of dz1, dz2, dy
  double* losspart;  // per row tile: sum of squared errors
};

// Up to kChainHeld fragments of column tile tn, from step k0 on. A layer is a
// few steps long, so a workgroup's time is the latency of its weights (the
// other XCDs' last update, from beyond the L2): a wave loads a whole group at
// once, and the first group of the next layer while it works on this one.
constexpr int kChainHeld = 8;
struct ChainHeld {
  v8u b[kChainHeld];
};
__device__ __forceinline__ ChainHeld chain_load(const unsigned short* __restrict__ w, int ks, int tiles, int tn,
                                                int k0) {
  ChainHeld h;
  const v8u* wp = reinterpret_cast<const v8u*>(w + (size_t)tn * ks * kFrag) + (threadIdx.x & 63);
#pragma unroll
  for (int q = 0; q < kChainHeld; ++q) {
    h.b[q] = v8u{};
    if (tn < tiles && k0 + q < ks) h.b[q] = wp[(k0 + q) * 64];
  }
  return h;
}
__device__ __forceinline__ ChainHeld chain_first(const unsigned short* __restrict__ w, int ks, int tiles) {
  return chain_load(w, ks, tiles, __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), 0);
}

// acc of the tiles tn = wave, wave + waves, ... of A (16 rows in LDS, ks
// steps of 32) times packed weights, handed to `epi(tn, acc)`; `held` is the
// wave's chain_first of these weights.
template <class F>
__device__ __forceinline__ void chain_product(const unsigned short* a, int lda, const unsigned short* __restrict__ w,
                                              int ks, int tiles, ChainHeld held, F epi) {
  const int lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
  const unsigned short* ar = a + r * lda + 8 * g;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), waves = blockDim.x >> 6;
  for (int tn = wave; tn < tiles; tn += waves) {
    v4f acc = {0.f, 0.f, 0.f, 0.f};
    for (int k0 = 0; k0 < ks; k0 += kChainHeld) {
      if (tn != wave || k0) held = chain_load(w, ks, tiles, tn, k0);
#pragma unroll
      for (int q = 0; q < kChainHeld; ++q)
        if (k0 + q < ks) {
          const v8u av = *reinterpret_cast<const v8u*>(ar + 32 * (k0 + q));
          acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8bf, av),
                                                        __builtin_bit_cast(v8bf, held.b[q]), acc, 0, 0, 0);
        }
    }
    epi(tn, acc);
  }
}

// This lane's four rows (4g .. 4g + 3 of the tile at m0) of column tile tn as
// a fragment over ms steps of 32 rows.
__device__ __forceinline__ void store_frag(unsigned short* f, int tn, int ms, int m0, const float (&v)[4]) {
  const int lane = threadIdx.x & 63, m = (m0 & 31) + 4 * (lane >> 4);
  ushort4 b;
  b.x = f2bf(v[0]);
  b.y = f2bf(v[1]);
  b.z = f2bf(v[2]);
  b.w = f2bf(v[3]);
  const size_t o = ((size_t)tn * ms + (m0 >> 5)) * kFrag + (size_t)((lane & 15) + 16 * (m >> 3)) * 8 + (m & 7);
  *reinterpret_cast<ushort4*>(f + o) = b;
}

// Sums over the tile's 16 rows (valid in lanes < 16).
__device__ __forceinline__ float tile_colsum(const float (&v)[4]) {
  float s = (v[0] + v[1]) + (v[2] + v[3]);
  s += __shfl_xor(s, 16);
  s += __shfl_xor(s, 32);
  return s;
}

// LDS bytes of a chain workgroup: h1 and h2 in FP32, the BF16 operands x, h1
// (then dz2), h2 and dy, rows 8 values apart in the banks.
size_t chain_lds(int nin, int nh, int nout) {
  return (size_t)16 * (2 * 4 * up16(nh) + 2 * (up32(nin) + 8 + 2 * (up32(nh) + 8) + up32(nout) + 8));
}

// Tile tile0 + blockIdx.x of 16 rows of the batch: out = MLP(x), or to train the
// loss against t, the activations' gradients and the tape. A forward pass has as
// many waves as the widest layer has tiles, so that a small network leaves room
// for other workgroups: 65536 rows through 1-1-1 took 80 us with 16 waves (13 as
// separate products), 9 now; through 4-32-96 89 (54), 29 now.
template <bool kTrain>
__global__ __launch_bounds__(64 * kChainWaves) void k_mlp_chain(int tile0, int M, int ms, MlpDims d,
                                                                const float* __restrict__ p,
                                                                const unsigned short* __restrict__ pk,
                                                                const float* __restrict__ x, const float* __restrict__ t,
                                                                float* __restrict__ out, float scale, MlpTape tape) {
  extern __shared__ __align__(16) char smem[];
  const int hc = up16(d.nh), lx = up32(d.nin) + 8, lh = up32(d.nh) + 8, ly = up32(d.nout) + 8;
  float* h1f = reinterpret_cast<float*>(smem);
  float* h2f = h1f + 16 * hc;
  unsigned short* xb = reinterpret_cast<unsigned short*>(h2f + 16 * hc);
  unsigned short* h1b = xb + 16 * lx;
  unsigned short* h2b = h1b + 16 * lh;
  unsigned short* dyb = h2b + 16 * lh;
  const int lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
  const int tile = tile0 + blockIdx.x, m0 = tile * 16, nt = blockDim.x;
  const int ki = up32(d.nin) >> 5, kh = up32(d.nh) >> 5, ko = up32(d.nout) >> 5, th = hc >> 4, to = up16(d.nout) >> 4;
  const ChainHeld w1 = chain_first(pk + d.f[0], ki, th), w2 = chain_first(pk + d.f[1], kh, th);
  // operands: x in BF16, eight values at a time, zeros in the padding that no product writes
  for (int e = threadIdx.x; e < 2 * lx; e += nt) {
    const int i = e / (lx >> 3), k0 = (e - i * (lx >> 3)) * 8;
    const float* xr = x + (size_t)(m0 + i) * d.nin + k0;
    v8u b{};
#pragma unroll
    for (int k = 0; k < 8; ++k)
      if (m0 + i < M && k0 + k < d.nin) b[k] = f2bf(xr[k]);
    reinterpret_cast<v8u*>(xb)[e] = b;
  }
  for (int e = threadIdx.x; e < 2 * (2 * lh + ly); e += nt) reinterpret_cast<v8u*>(h1b)[e] = v8u{};
  __syncthreads();
  if (kTrain) {  // x over the rows, for dW1
    for (int e = threadIdx.x; e < 16 * up16(d.nin); e += nt) {
      const int k = e >> 4, i = e & 15;
      tape.x[frag_at(m0 + i, k, ms)] = xb[i * lx + k];
    }
  }
  auto hidden = [&](const unsigned short* a, int lda, int ks, int l, const ChainHeld& held, float* hf,
                    unsigned short* hb, unsigned short* frag) {
    const float* b = p + d.b_off[l];
    chain_product(a, lda, pk + d.f[l], ks, th, held, [&](int tn, v4f acc) {
      const int j = tn * 16 + r;
      const float bj = j < d.nh ? b[j] : 0.f;
      float v[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        v[q] = j < d.nh && m0 + 4 * g + q < M ? tanhf(acc[q] + bj) : 0.f;
        hf[(4 * g + q) * hc + j] = v[q];
        hb[(4 * g + q) * lh + j] = f2bf(v[q]);
      }
      if (kTrain) store_frag(frag, tn, ms, m0, v);
    });
    __syncthreads();
  };
  hidden(xb, lx, ki, 0, w1, h1f, h1b, tape.h1);
  const ChainHeld w3 = chain_first(pk + d.f[2], kh, to);
  hidden(h1b, lh, kh, 1, w2, h2f, h2b, tape.h2);
  const ChainHeld r3 = chain_first(pk + d.r[2], ko, kTrain ? th : 0);
  double loss = 0.0;
  float* cp = kTrain ? tape.colpart + (size_t)tile * (2 * d.nh + d.nout) : nullptr;
  {
    const float* b = p + d.b_off[2];
    chain_product(h2b, lh, pk + d.f[2], kh, to, w3, [&](int tn, v4f acc) {
      const int j = tn * 16 + r;
      const float bj = j < d.nout ? b[j] : 0.f;
      float v[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int i = m0 + 4 * g + q;
        const bool in = i < M && j < d.nout;
        const float y = acc[q] + bj;
        v[q] = 0.f;
        if (!kTrain) {
          if (in) out[(size_t)i * d.nout + j] = y;
        } else if (in) {
          const float e = y - t[(size_t)i * d.nout + j];
          loss += (double)e * (double)e;
          v[q] = scale * e;
        }
        if (kTrain) dyb[(4 * g + q) * ly + j] = f2bf(v[q]);
      }
      if (kTrain) {
        store_frag(tape.dy, tn, ms, m0, v);
        const float s = tile_colsum(v);
        if (lane < 16 && j < d.nout) cp[2 * d.nh + j] = s;
      }
    });
  }
  if (!kTrain) return;
  const ChainHeld r2 = chain_first(pk + d.r[1], kh, th);
  __shared__ double ls[kChainWaves];
  for (int o = 32; o > 0; o >>= 1) loss += __shfl_down(loss, o);
  if (lane == 0) ls[threadIdx.x >> 6] = loss;
  __syncthreads();
  if (threadIdx.x == 0) {
    double s = 0.0;
    for (int w = 0; w < nt >> 6; ++w) s += ls[w];
    tape.losspart[tile] = s;
  }
  // dz2 = (dy W3^T) * (1 - h2^2) into h1's operand, dz1 = (dz2 W2^T) * (1 - h1^2)
  chain_product(dyb, ly, pk + d.r[2], ko, th, r3, [&](int tn, v4f acc) {
    const int j = tn * 16 + r;
    float v[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const float h = h2f[(4 * g + q) * hc + j];
      v[q] = j < d.nh && m0 + 4 * g + q < M ? acc[q] * (1.0f - h * h) : 0.f;
      h1b[(4 * g + q) * lh + j] = f2bf(v[q]);
    }
    store_frag(tape.dz2, tn, ms, m0, v);
    const float s = tile_colsum(v);
    if (lane < 16 && j < d.nh) cp[d.nh + j] = s;
  });
  __syncthreads();
  chain_product(h1b, lh, pk + d.r[1], kh, th, r2, [&](int tn, v4f acc) {
    const int j = tn * 16 + r;
    float v[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const float h = h1f[(4 * g + q) * hc + j];
      v[q] = j < d.nh && m0 + 4 * g + q < M ? acc[q] * (1.0f - h * h) : 0.f;
    }
    store_frag(tape.dz1, tn, ms, m0, v);
    const float s = tile_colsum(v);
    if (lane < 16 && j < d.nh) cp[j] = s;
  });
}

// Gradients from the tape. Workgroups [0, ntile): one 16 x 16 tile of dW3 =
// H2^T dY, dW2 = H1^T dZ2 or dW1 = X^T dZ1, its rows of the batch split over
// the four waves and added in order (1 KB operands a load, all from L2), 1024
// rows of a wave at a time, so that the FP32 sums of long batches stay short. Then
// ones of 64 columns of the bias gradients (tiles of 16 rows, added in FP64), and
// one for the loss.
__global__ __launch_bounds__(256) void k_mlp_wgrad(int ms, int mt, MlpDims d, MlpTape tape, float* __restrict__ grad,
                                                   double loss_scale, double* loss) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int th = up16(d.nh) >> 4, to = up16(d.nout) >> 4, ti = up16(d.nin) >> 4;
  const int n3 = th * to, n2 = th * th, n1 = ti * th;
  int b = blockIdx.x;
  if (b < n3 + n2 + n1) {
    __shared__ float part[4][256];
    const unsigned short *A, *Bm;
    int l, tj, ni, nj;
    if (b < n3) { l = 2; A = tape.h2; Bm = tape.dy; tj = to; ni = d.nh; nj = d.nout; }
    else if (b < n3 + n2) { b -= n3; l = 1; A = tape.h1; Bm = tape.dz2; tj = th; ni = d.nh; nj = d.nh; }
    else { b -= n3 + n2; l = 0; A = tape.x; Bm = tape.dz1; tj = th; ni = d.nin; nj = d.nh; }
    const int bi = b / tj, bj = b - bi * tj;
    const v8u* ap = reinterpret_cast<const v8u*>(A + (size_t)bi * ms * kFrag) + lane;
    const v8u* bp = reinterpret_cast<const v8u*>(Bm + (size_t)bj * ms * kFrag) + lane;
    v4f sum = {0.f, 0.f, 0.f, 0.f};
    for (int k0 = wave; k0 < ms; k0 += 4 * 32) {
      v4f acc = {0.f, 0.f, 0.f, 0.f};
      const int k1 = min(ms, k0 + 4 * 32);
#pragma unroll 8
      for (int k = k0; k < k1; k += 4)
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8bf, ap[(size_t)k * 64]),
                                                      __builtin_bit_cast(v8bf, bp[(size_t)k * 64]), acc, 0, 0, 0);
      sum += acc;
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) part[wave][(4 * (lane >> 4) + q) * 16 + (lane & 15)] = sum[q];
    __syncthreads();
    const int e = threadIdx.x, i = bi * 16 + (e >> 4), j = bj * 16 + (e & 15);
    if (i < ni && j < nj)
      grad[d.w_off[l] + (size_t)i * nj + j] = ((part[0][e] + part[1][e]) + part[2][e]) + part[3][e];
    return;
  }
  b -= n3 + n2 + n1;
  const int ncol = 2 * d.nh + d.nout, nb = (ncol + 63) / 64;
  if (b < nb) {
    __shared__ double sm[4][64];
    const int c = b * 64 + lane;
    double s = 0.0;
    if (c < ncol)
#pragma unroll 8
      for (int k = wave; k < mt; k += 4) s += (double)tape.colpart[(size_t)k * ncol + c];
    sm[wave][lane] = s;
    __syncthreads();
    if (wave == 0 && c < ncol) {
      const int64_t o = c < d.nh ? d.b_off[0] + c : c < 2 * d.nh ? d.b_off[1] + c - d.nh : d.b_off[2] + c - 2 * d.nh;
      grad[o] = (float)(((sm[0][lane] + sm[1][lane]) + sm[2][lane]) + sm[3][lane]);
    }
    return;
  }
  const double s = sum_partials(tape.losspart, mt, 1, 0);
  if (threadIdx.x == 0 && loss) *loss = s * loss_scale;
}

// Adam step over all parameters; refreshes the packed weights.
__global__ void k_mlp_adam(int64_t n, MlpDims d, float* __restrict__ w, const float* __restrict__ gr,
                           float* __restrict__ m, float* __restrict__ v, unsigned short* __restrict__ pk, float lr,
                           float b1, float b2, float eps, float c1, float c2) {
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
    const float g = gr[i];
    const float mi = b1 * m[i] + (1.f - b1) * g;
    const float vi = b2 * v[i] + (1.f - b2) * g * g;
    m[i] = mi;
    v[i] = vi;
    const float wi = w[i] - lr * (mi / c1) / (sqrtf(vi / c2) + eps);
    w[i] = wi;
    pack_weight(d, i, f2bf(wi), pk);
  }
}

// ---- FP64 tall-skinny products for the POD ----

// Partial C_s = X(rows of split s)^T Y(rows of split s): X n x p, Y n x q
// (column-major, leading dimension n); C tile 32 x 32 per block, 256
// threads x 4 outputs; rows staged through LDS in chunks of 64.
__global__ __launch_bounds__(256) void k_tsmm(int64_t n, int p, int q, const double* __restrict__ X,
                                              const double* __restrict__ Y, int64_t rows_per_split,
                                              double* __restrict__ part) {
  __shared__ double xs[64][33];
  __shared__ double ys[64][33];
  const int i0 = blockIdx.x * 32, j0 = blockIdx.y * 32;
  const int64_t r0 = (int64_t)blockIdx.z * rows_per_split;
  const int64_t r1 = std::min<int64_t>(n, r0 + rows_per_split);
  const int t = threadIdx.x;
  const int ci = t & 31, cj = (t >> 5) * 4;  // outputs (ci, cj..cj+3)
  double acc[4] = {0.0, 0.0, 0.0, 0.0};
  for (int64_t rb = r0; rb < r1; rb += 64) {
    for (int e = t; e < 64 * 32; e += 256) {
      const int rr = e & 63, cc = e >> 6;
      const int64_t row = rb + rr;
      xs[rr][cc] = (row < r1 && i0 + cc < p) ? X[(size_t)(i0 + cc) * n + row] : 0.0;
      ys[rr][cc] = (row < r1 && j0 + cc < q) ? Y[(size_t)(j0 + cc) * n + row] : 0.0;
    }
    __syncthreads();
#pragma unroll 8
    for (int rr = 0; rr < 64; ++rr) {
      const double xv = xs[rr][ci];
#pragma unroll
      for (int u = 0; u < 4; ++u) acc[u] += xv * ys[rr][cj + u];
    }
    __syncthreads();
  }
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const int i = i0 + ci, j = j0 + cj + u;
    if (i < p && j < q) part[((size_t)blockIdx.z * q + j) * p + i] = acc[u];
  }
}

// C = sum over splits of the partials (fixed order), column-major p x q.
__global__ void k_tsmm_sum(int p, int q, int splits, const double* __restrict__ part, double* __restrict__ C) {
  const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= (int64_t)p * q) return;
  double s = 0.0;
  for (int z = 0; z < splits; ++z) s += part[(size_t)z * p * q + e];
  C[e] = s;
}

// Y(n x q) = X(n x p) C(p x q), column-major; 16 columns of Y per block row,
// C staged through LDS in chunks of 64 rows.
__global__ __launch_bounds__(256) void k_mm(int64_t n, int p, int q, const double* __restrict__ X,
                                            const double* __restrict__ Cm, double* __restrict__ Y, int64_t ldy) {
  __shared__ double cs[64][16];
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int j0 = blockIdx.y * 16;
  double acc[16];
#pragma unroll
  for (int u = 0; u < 16; ++u) acc[u] = 0.0;
  for (int k0 = 0; k0 < p; k0 += 64) {
    for (int e = threadIdx.x; e < 64 * 16; e += blockDim.x) {
      const int kk = e & 63, u = e >> 6;
      cs[kk][u] = (k0 + kk < p && j0 + u < q) ? Cm[(size_t)(j0 + u) * p + k0 + kk] : 0.0;
    }
    __syncthreads();
    if (i < n) {
      const int kn = std::min(64, p - k0);
      for (int kk = 0; kk < kn; ++kk) {
        const double xv = X[(size_t)(k0 + kk) * n + i];
#pragma unroll
        for (int u = 0; u < 16; ++u) acc[u] += xv * cs[kk][u];
      }
    }
    __syncthreads();
  }
  if (i < n) {
#pragma unroll
    for (int u = 0; u < 16; ++u)
      if (j0 + u < q) Y[(size_t)(j0 + u) * ldy + i] = acc[u];
  }
}

int grid1(int64_t n, int cap = 4096) { return (int)std::max<int64_t>(1, std::min<int64_t>((n + 255) / 256, cap)); }

// C(i,j) = sum over s of the split-K partial tiles P[s*M*N + i*N + j], in order.
__global__ void k_ksum(int M, int N, int ks, const float* __restrict__ P, float* __restrict__ C, int ldc) {
  const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= (int64_t)M * N) return;
  float v = 0.f;
  for (int z = 0; z < ks; ++z) v += P[(size_t)z * M * N + e];
  const int i = (int)(e / N), j = (int)(e - (int64_t)i * N);
  C[(size_t)i * ldc + j] = v;
}

template <class TA, class TB>
void gemm(hipStream_t s, int M, int N, int K, const TA* A, int ars, int acs, const TB* B, int brs, int bcs, float* C,
          int ldc, const float* bias, int act, const float* dmul, int ldd, DevBuf* kscratch = nullptr) {
  const int tiles = ((M + 15) / 16) * ((N + 15) / 16);
  // few output tiles over a long K (the weight gradients): split K so that the
  // whole device works, then add the partial tiles in a fixed order
  int ks = 1;
  if (kscratch && !bias && !act && !dmul) {
    const int waves = (tiles + 3) / 4 * 4;
    ks = std::max(1, std::min({16, K / 128, (4 * 256 * 4) / std::max(1, waves)}));
  }
  if (ks == 1) {
    hipLaunchKernelGGL((k_gemm_bf16<TA, TB>), dim3((tiles + 3) / 4), dim3(256), 0, s, M, N, K, A, ars, acs, B, brs,
                       bcs, C, ldc, bias, act, dmul, ldd);
    BCM_HIP(hipGetLastError());
    return;
  }
  const size_t part = (size_t)M * N;
  if (kscratch->bytes < part * ks * 4) kscratch->alloc(part * ks * 4);
  float* P = kscratch->as<float>();
  hipLaunchKernelGGL((k_gemm_bf16<TA, TB>), dim3((tiles + 3) / 4, ks), dim3(256), 0, s, M, N, K, A, ars, acs, B, brs,
                     bcs, P, N, (const float*)nullptr, 0, (const float*)nullptr, 0);
  hipLaunchKernelGGL(k_ksum, dim3((unsigned)((part + 255) / 256)), dim3(256), 0, s, M, N, ks, P, C, ldc);
  BCM_HIP(hipGetLastError());
}

MlpDims mlp_dims(const Mlp& m) {
  MlpDims d{};
  d.nin = m.nin;
  d.nh = m.nh;
  d.nout = m.nout;
  int64_t o = 0;
  for (int l = 0; l < 3; ++l) {
    d.w_off[l] = m.w_off[l];
    d.b_off[l] = m.b_off[l];
    const int nk = l == 0 ? m.nin : m.nh, nj = l == 2 ? m.nout : m.nh;
    d.f[l] = o;
    o += (int64_t)up16(nj) * up32(nk);
    d.r[l] = o;
    if (l > 0) o += (int64_t)up16(nk) * up32(nj);
  }
  return d;
}

int64_t packed_values(const Mlp& m) {
  const MlpDims d = mlp_dims(m);
  return d.r[2] + (int64_t)up16(m.nh) * up32(m.nout);
}

}  // namespace

// ---------------------------------------------------------------------------
// MLP

Mlp::Mlp(int nin_, int nh_, int nout_, uint64_t seed) : nin(nin_), nh(nh_), nout(nout_) {
  if (nin < 1 || nh < 1 || nout < 1 || nin > 4096 || nh > 4096 || nout > 4096)
    throw Error(kErrArg, "mlp: layer sizes must be in 1..4096");
  const int fan_in[3] = {nin, nh, nh}, fan_out[3] = {nh, nh, nout};
  int64_t off = 0, woff = 0;
  for (int l = 0; l < 3; ++l) {
    w_off[l] = off;
    off += (int64_t)fan_in[l] * fan_out[l];
    b_off[l] = off;
    off += fan_out[l];
    wb_off[l] = woff;
    woff += (int64_t)fan_in[l] * fan_out[l];
  }
  nparam = off;
  nweight = woff;
  std::vector<float> h(nparam, 0.0f);
  std::mt19937_64 g(seed);
  for (int l = 0; l < 3; ++l) {  // Glorot-uniform weights, zero biases
    const double lim = std::sqrt(6.0 / (fan_in[l] + fan_out[l]));
    std::uniform_real_distribution<double> u(-lim, lim);
    for (int64_t i = 0; i < (int64_t)fan_in[l] * fan_out[l]; ++i) h[w_off[l] + i] = (float)u(g);
  }
  params.alloc(nparam * 4);
  grads.alloc(nparam * 4);
  m1.alloc(nparam * 4);
  m2.alloc(nparam * 4);
  fused = chain_lds(nin, nh, nout) <= (size_t)63 << 10;
  if (fused) {
    wpk.alloc(packed_values(*this) * 2);
    set_params(h.data());
    return;
  }
  wbf.alloc(nweight * 2);
  std::vector<unsigned char> isw(nparam, 0);
  std::vector<int64_t> idx(nparam, 0);
  for (int l = 0; l < 3; ++l)
    for (int64_t i = 0; i < (int64_t)fan_in[l] * fan_out[l]; ++i) {
      isw[w_off[l] + i] = 1;
      idx[w_off[l] + i] = wb_off[l] + i;
    }
  is_w.upload(isw.data(), isw.size());
  wb_index.upload(idx.data(), idx.size() * 8);
  set_params(h.data());
}

void Mlp::set_params(const float* host) {
  BCM_HIP(hipMemcpy(params.p, host, nparam * 4, hipMemcpyHostToDevice));
  BCM_HIP(hipMemset(m1.p, 0, nparam * 4));
  BCM_HIP(hipMemset(m2.p, 0, nparam * 4));
  BCM_HIP(hipMemset(grads.p, 0, nparam * 4));
  if (fused) {
    BCM_HIP(hipMemset(wpk.p, 0, wpk.bytes));
    hipLaunchKernelGGL(k_mlp_pack, dim3(grid1(nparam)), dim3(256), 0, nullptr, nparam, mlp_dims(*this),
                       params.as<const float>(), wpk.as<unsigned short>());
  }
  for (int l = 0; l < 3 && !fused; ++l) {
    const int64_t cnt = b_off[l] - w_off[l];
    hipLaunchKernelGGL(k_to_bf16, dim3(grid1(cnt)), dim3(256), 0, nullptr, cnt, params.as<float>() + w_off[l],
                       wbf.as<unsigned short>() + wb_off[l]);
  }
  BCM_HIP(hipDeviceSynchronize());
  step = 0;
}

void Mlp::ensure_batch(int M) {
  if (M <= cap_batch) return;
  if (fused) {  // the tape: fragments over the rows, padded to whole steps of 32
    const size_t m32 = up32(M), mt = m32 / 16;
    const size_t frags = m32 * (up16(nin) + 4 * (size_t)up16(nh) + up16(nout)) * 2;
    tape.alloc(mt * 8 + frags + mt * (2 * (size_t)nh + nout) * 4);
    cap_batch = M;
    return;
  }
  h1.alloc((size_t)M * nh * 4);
  h2.alloc((size_t)M * nh * 4);
  y.alloc((size_t)M * nout * 4);
  dz1.alloc((size_t)M * nh * 4);
  dz2.alloc((size_t)M * nh * 4);
  dy.alloc((size_t)M * nout * 4);
  partials.alloc(4096 * 8 + 64);
  colpart.alloc((size_t)kColChunks * std::max(nh, nout) * 4);
  cap_batch = M;
}

// One pass of the chain over the batch; t == nullptr: out = MLP(x) only.
void Mlp::chain(hipStream_t s, int M, const float* x, const float* t, float* out, double* loss_dev) {
  const MlpDims d = mlp_dims(*this);
  const int ms = up32(M) >> 5, mt = t ? 2 * ms : (M + 15) / 16;
  MlpTape tp{};
  if (t) {
    ensure_batch(M);
    const size_t m32 = up32(M);
    tp.losspart = tape.as<double>();
    unsigned short* f = reinterpret_cast<unsigned short*>(tp.losspart + mt);
    tp.x = f;
    tp.h1 = tp.x + m32 * up16(nin);
    tp.h2 = tp.h1 + m32 * up16(nh);
    tp.dz1 = tp.h2 + m32 * up16(nh);
    tp.dz2 = tp.dz1 + m32 * up16(nh);
    tp.dy = tp.dz2 + m32 * up16(nh);
    tp.colpart = reinterpret_cast<float*>(tp.dy + m32 * up16(nout));
  }
  const double total = (double)M * nout;
  const int th = up16(nh) / 16, to = up16(nout) / 16, ti = up16(nin) / 16;
  int waves = t ? kChainWaves : std::min(kChainWaves, std::max(th, to));
  // 16 waves fit a compute unit at these registers: many workgroups leave none of it idle
  if (mt > 1024)
    while (waves & (waves - 1)) waves &= waves - 1;
  constexpr int kMostTiles = 1 << 21;  // of 1024 threads: a launch takes less than 2^32
  for (int tile = 0; tile < mt; tile += kMostTiles)
    hipLaunchKernelGGL(t ? k_mlp_chain<true> : k_mlp_chain<false>, dim3(std::min(kMostTiles, mt - tile)), dim3(64 * waves),
                       chain_lds(nin, nh, nout), s, tile, M, ms, d, params.as<const float>(),
                       wpk.as<const unsigned short>(), x, t, out, 2.0f / (float)((int64_t)M * nout), tp);
  if (t) {
    const int grid = th * to + th * th + ti * th + (2 * nh + nout + 63) / 64 + 1;
    hipLaunchKernelGGL(k_mlp_wgrad, dim3(grid), dim3(256), 0, s, ms, mt, d, tp, grads.as<float>(), 1.0 / total,
                       loss_dev);
  }
  BCM_HIP(hipGetLastError());
}

void Mlp::forward(hipStream_t s, int M, const float* x, float* out) {
  if (fused) {
    if (!out) throw Error(kErrArg, "mlp: the forward pass of a fused network needs an output");
    // A workgroup writes its rows of out while others still read x: where the
    // two share memory, x is read from a copy.
    const size_t nx = (size_t)M * nin, ny = (size_t)M * nout;
    if (out < x + nx && x < out + ny) {
      if (xcopy.bytes < nx * 4) xcopy.alloc(nx * 4);
      BCM_HIP(hipMemcpyAsync(xcopy.p, x, nx * 4, hipMemcpyDeviceToDevice, s));
      x = xcopy.as<const float>();
    }
    chain(s, M, x, nullptr, out, nullptr);
    return;
  }
  ensure_batch(M);
  const float* P = params.as<float>();
  const unsigned short* W = wbf.as<unsigned short>();
  gemm(s, M, nh, nin, x, nin, 1, W + wb_off[0], nh, 1, h1.as<float>(), nh, P + b_off[0], 1, (const float*)nullptr, 0);
  gemm(s, M, nh, nh, h1.as<const float>(), nh, 1, W + wb_off[1], nh, 1, h2.as<float>(), nh, P + b_off[1], 1,
       (const float*)nullptr, 0);
  gemm(s, M, nout, nh, h2.as<const float>(), nh, 1, W + wb_off[2], nout, 1, out ? out : y.as<float>(), nout,
       P + b_off[2], 0, (const float*)nullptr, 0);
}

void Mlp::backward(hipStream_t s, int M, const float* x, const float* t, double* loss_dev) {
  if (fused) {
    chain(s, M, x, t, nullptr, loss_dev);
    return;
  }
  forward(s, M, x, nullptr);
  float* G = grads.as<float>();
  const unsigned short* W = wbf.as<unsigned short>();
  const int64_t total = (int64_t)M * nout;
  const int nb = grid1(total, 4096);
  hipLaunchKernelGGL(k_mse, dim3(nb), dim3(256), 0, s, total, y.as<const float>(), t, 2.0f / (float)total,
                     dy.as<float>(), partials.as<double>());
  if (loss_dev)
    hipLaunchKernelGGL(k_sum_to, dim3(1), dim3(256), 0, s, partials.as<const double>(), nb, 1.0 / (double)total,
                       loss_dev);
  // layer 3: dW3 = H2^T dY, db3 = colsum(dY), dZ2 = (dY W3^T) * (1 - H2^2)
  gemm(s, nh, nout, M, h2.as<const float>(), 1, nh, dy.as<const float>(), nout, 1, G + w_off[2], nout,
       (const float*)nullptr, 0, (const float*)nullptr, 0, &kpart);
  colsum(s, M, nout, dy.as<const float>(), nout, G + b_off[2], colpart.as<float>());
  gemm(s, M, nh, nout, dy.as<const float>(), nout, 1, W + wb_off[2], 1, nout, dz2.as<float>(), nh,
       (const float*)nullptr, 0, h2.as<const float>(), nh);
  // layer 2
  gemm(s, nh, nh, M, h1.as<const float>(), 1, nh, dz2.as<const float>(), nh, 1, G + w_off[1], nh,
       (const float*)nullptr, 0, (const float*)nullptr, 0, &kpart);
  colsum(s, M, nh, dz2.as<const float>(), nh, G + b_off[1], colpart.as<float>());
  gemm(s, M, nh, nh, dz2.as<const float>(), nh, 1, W + wb_off[1], 1, nh, dz1.as<float>(), nh, (const float*)nullptr,
       0, h1.as<const float>(), nh);
  // layer 1
  gemm(s, nin, nh, M, x, 1, nin, dz1.as<const float>(), nh, 1, G + w_off[0], nh, (const float*)nullptr, 0,
       (const float*)nullptr, 0, &kpart);
  colsum(s, M, nh, dz1.as<const float>(), nh, G + b_off[0], colpart.as<float>());
}

void Mlp::adam(hipStream_t s, float lr) {
  ++step;
  const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
  const float c1 = 1.0f - std::pow(b1, (float)step), c2 = 1.0f - std::pow(b2, (float)step);
  if (fused) {
    hipLaunchKernelGGL(k_mlp_adam, dim3(grid1(nparam)), dim3(256), 0, s, nparam, mlp_dims(*this), params.as<float>(),
                       grads.as<const float>(), m1.as<float>(), m2.as<float>(), wpk.as<unsigned short>(), lr, b1, b2,
                       eps, c1, c2);
    BCM_HIP(hipGetLastError());
    return;
  }
  hipLaunchKernelGGL(k_adam, dim3(grid1(nparam)), dim3(256), 0, s, nparam, params.as<float>(), grads.as<float>(),
                     m1.as<float>(), m2.as<float>(), wbf.as<unsigned short>(), is_w.as<unsigned char>(),
                     wb_index.as<int64_t>(), lr, b1, b2, eps, c1, c2);
  BCM_HIP(hipGetLastError());
}

// ---------------------------------------------------------------------------
// FP64 products for the POD

void tsmm(hipStream_t s, int64_t n, int p, int q, const double* X, const double* Y, double* C, DevBuf& scratch) {
  const int splits = (int)std::max<int64_t>(1, std::min<int64_t>(64, n / 2048));
  const int64_t rows = (n + splits - 1) / splits;
  const size_t need = (size_t)splits * p * q * 8;
  if (scratch.bytes < need) scratch.alloc(need);
  hipLaunchKernelGGL(k_tsmm, dim3((p + 31) / 32, (q + 31) / 32, splits), dim3(256), 0, s, n, p, q, X, Y, rows,
                     scratch.as<double>());
  hipLaunchKernelGGL(k_tsmm_sum, dim3(((int64_t)p * q + 255) / 256), dim3(256), 0, s, p, q, splits,
                     scratch.as<const double>(), C);
  BCM_HIP(hipGetLastError());
}

void mm(hipStream_t s, int64_t n, int p, int q, const double* X, const double* Cm, double* Y, int64_t ldy) {
  hipLaunchKernelGGL(k_mm, dim3((unsigned)((n + 255) / 256), (q + 15) / 16), dim3(256), 0, s, n, p, q, X, Cm, Y, ldy);
  BCM_HIP(hipGetLastError());
}

}  // namespace bcm
