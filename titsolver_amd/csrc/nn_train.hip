// Dense layers of the network's training: forward and input-gradient products
// with the weights resident in LDS, and weight gradients.
//
// The layers are tall and narrow (141,000 edge rows by 80 to 160 columns for
// an 18,000-node sample), so they are bound by the rows' bytes.  What kept
// the general tiled GEMM (nn_kernels.hip) far from that were its operands
// transposed into LDS two bytes at a time for every 64 x 64 tile, its passes
// over FP32 intermediates (gradient, activation derivative, column sums, edge
// sums) and, for the weight gradients, 136 workgroups.  Here a workgroup packs
// the weights once as MFMA fragments and walks row tiles, whose fragments come
// straight from global memory, and the neighbouring element-wise passes are
// the product's epilogue; a weight gradient's operands are transposed 8 x 8 in
// registers and its row slices are summed by one pass at the end.
//
// One loss and gradient of an 18,000-node sample: 2,980 us before, 970 us.
#include "nn_kernels.hpp"

#include <algorithm>

namespace tit_amd {

namespace {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(16))) float f32x16;

constexpr int kFrag = 512;  // BF16 elements of one MFMA operand fragment
constexpr int NT = 256;
constexpr int kWaves = NT / 64;

__device__ __forceinline__ bf16x8 ld8(const bf16* p) {
  return *reinterpret_cast<const bf16x8*>(p);
}
__device__ __forceinline__ f32x16 mfma(bf16x8 a, bf16x8 b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

// Rows [M x 16 KS] times weights [16 KS x N], N <= 32 NB.  A wave takes 32
// rows at a time; fragment layouts as in nn_kernels.hip: A[m = l % 32]
// [k = 8 (l / 32) + i], B[k][n = l % 32], C[m = 8 j + 4 (l / 32) + i][n] in
// accumulator element 4 j + i.
template <int KS, int N>
__global__ __launch_bounds__(NT) void k_dense(DenseArgs g) {
  constexpr int NB = (N + 31) / 32;
  __shared__ __attribute__((aligned(16))) bf16 s_w[NB * KS * kFrag];
  __shared__ float s_sum[kWaves][NB * 32];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int h = lane >> 5, col = lane & 31;
  for (int u = tid; u < NB * KS * 64; u += NT) {
    const int f = u >> 6, l = u & 63;
    const int n = 32 * (f / KS) + (l & 31), k = 16 * (f % KS) + 8 * (l >> 5);
    bf16x8 v = {};
    if (n < N) {
      if (g.trans) {
        v = ld8(g.W + static_cast<size_t>(n) * g.ldw + k);
      } else {
#pragma unroll
        for (int t = 0; t < 8; ++t) v[t] = g.W[static_cast<size_t>(k + t) * g.ldw + n];
      }
    }
    *reinterpret_cast<bf16x8*>(s_w + u * 8) = v;
  }
  __syncthreads();
  float sum[NB];
#pragma unroll
  for (int nb = 0; nb < NB; ++nb) sum[nb] = 0.0f;
  const int tiles = (g.M + 31) / 32;
  for (int t = blockIdx.x * kWaves + wave; t < tiles; t += gridDim.x * kWaves) {
    const int m0 = 32 * t;
    const bf16* row = g.A + static_cast<size_t>(min(m0 + col, g.M - 1)) * g.lda + 8 * h;
    bf16x8 a[KS];
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) a[ks] = ld8(row + 16 * ks);
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
      const int n = 32 * nb + col;
      f32x16 acc = {};
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) acc = mfma(a[ks], ld8(s_w + ((nb * KS + ks) * 64 + lane) * 8), acc);
      const bool in_n = n < N;
      const float bias = g.bias && in_n ? g.bias[n] : 0.0f;
      if (g.bpre) {  // the gradient through the activation, its column sums
        float pre[16];  // all loads in flight together
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          const int m = min(m0 + 8 * (e >> 2) + 4 * h + (e & 3), g.M - 1);
          pre[e] = g.bpre[static_cast<size_t>(m) * N + (in_n ? n : 0)];
        }
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          const int m = m0 + 8 * (e >> 2) + 4 * h + (e & 3);
          if (m >= g.M || !in_n) continue;
          const float d = acc[e] * nn_act_grad(pre[e]);
          g.out16[static_cast<size_t>(m) * g.ldo16 + n] = static_cast<bf16>(d);
          sum[nb] += d;
        }
        continue;
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        float y[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int m = m0 + 8 * j + 4 * h + i;
          const float x = g.bias ? acc[4 * j + i] + bias : acc[4 * j + i];
          y[i] = g.act == kActHswish ? nn_act(x) : x;
          if (m >= g.M || !in_n) continue;
          if (g.pre) g.pre[static_cast<size_t>(m) * N + n] = x;
          if (g.out32) g.out32[static_cast<size_t>(m) * g.ldo32 + n] = y[i];
          if (g.out16) g.out16[static_cast<size_t>(m) * g.ldo16 + n] = static_cast<bf16>(y[i]);
        }
        if (g.group16) {
          // the sum of eight rows (an edge group), in row order: the lower
          // half's four, then the upper half's
          static_assert(kGroupRows == 8, "four rows of each half");
          float s = 0.0f;
          if (h == 0) s = ((s + y[0]) + y[1]) + y[2] + y[3];
          s = __shfl(s, col);
          if (h == 1) s = ((s + y[0]) + y[1]) + y[2] + y[3];
          const int r = (m0 >> 3) + j;
          if (h == 1 && 8 * r < g.M && in_n) {
            g.group16[static_cast<size_t>(r) * g.ldg + g.colg + n] = static_cast<bf16>(s);
          }
        }
      }
    }
  }
  if (g.colsum) {
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
      const float s = sum[nb] + __shfl_xor(sum[nb], 32);
      if (h == 0) s_sum[wave][32 * nb + col] = s;
    }
    __syncthreads();
    for (int n = tid; n < N; n += NT) {
      float s = 0.0f;
      for (int w = 0; w < kWaves; ++w) s += s_sum[w][n];
      atomicAdd(g.colsum + n, s);
    }
  }
}

// d = dy act'(pre) for edge rows whose upstream row is shared by `group` of
// them; BF16, and its column sums.  A thread keeps its column.
constexpr int kEdgeRows = 256;
template <int N>
__global__ __launch_bounds__(NT) void k_edge_grad(int M, const float* dy, int ld_dy, int group,
                                                  const float* pre, bf16* d16, float* colsum) {
  static_assert(NT % N == 0, "a thread keeps its column");
  __shared__ float s_sum[NT];
  const int n = threadIdx.x % N, r0 = threadIdx.x / N, step = NT / N;
  float sum = 0.0f;
  const int beg = blockIdx.x * kEdgeRows, end = min(M, beg + kEdgeRows);
#pragma unroll 8
  for (int m = beg + r0; m < end; m += step) {
    const float d = dy[static_cast<size_t>(m / group) * ld_dy + n] *
                    nn_act_grad(pre[static_cast<size_t>(m) * N + n]);
    d16[static_cast<size_t>(m) * N + n] = static_cast<bf16>(d);
    sum += d;
  }
  s_sum[threadIdx.x] = sum;
  __syncthreads();
  if (threadIdx.x < static_cast<unsigned>(N)) {
    float s = 0.0f;
    for (int k = 0; k < step; ++k) s += s_sum[k * N + n];
    atomicAdd(colsum + n, s);
  }
}

// ---- weight gradients -------------------------------------------------------------

constexpr int kRows = 64;               // rows of one step
constexpr int kRowPad = kRows + 8;      // padded LDS row (144 B)

// Eight rows x eight columns of a row-major BF16 matrix (leading dimension
// ld) into LDS as tile[column][row]; rows past `end` are zero.
__device__ __forceinline__ void put_transposed(bf16* tile, const bf16* src, int ld, int c8, int k0,
                                               int k8, int end) {
  typedef __attribute__((ext_vector_type(4))) uint32_t u32x4;
  u32x4 r[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int k = k0 + 8 * k8 + i;
    r[i] = u32x4{0u, 0u, 0u, 0u};
    if (k < end) {
      r[i] = *reinterpret_cast<const u32x4*>(src + static_cast<size_t>(k) * ld + 8 * c8);
    }
  }
#pragma unroll
  for (int c = 0; c < 8; ++c) {
    u32x4 o;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      o[w] = __builtin_amdgcn_perm(r[2 * w + 1][c >> 1], r[2 * w][c >> 1],
                                   (c & 1) ? 0x07060302u : 0x05040100u);
    }
    *reinterpret_cast<u32x4*>(tile + (8 * c8 + c) * kRowPad + 8 * k8) = o;
  }
}

// dW[32 MB x 32 NB] of rows [beg, end) of X (M columns) and dY (N columns)
// into this slice's partial (row-major M x N).  NB == 4: wave w takes output
// columns 32 w ..; NB == 1: wave w takes output rows 32 w .. .
template <int M, int N>
__global__ __launch_bounds__(NT) void k_wgrad(int K, const bf16* X, const bf16* dY,
                                              int slice_rows, float* part) {
  constexpr int MB = (M + 31) / 32, NB = (N + 31) / 32;
  static_assert(M % 8 == 0 && N % 8 == 0 && (NB == kWaves || (NB == 1 && MB <= kWaves)),
                "the waves cover the output");
  __shared__ __attribute__((aligned(16))) bf16 sX[32 * MB * kRowPad];
  __shared__ __attribute__((aligned(16))) bf16 sY[32 * NB * kRowPad];
  constexpr int BM = NB == 1 ? 1 : MB;  // output blocks of a wave
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int h = lane >> 5, col = lane & 31;
  const int beg = blockIdx.x * slice_rows, end = min(K, beg + slice_rows);
  // columns past M or N stay zero
  for (int u = tid; u < 32 * MB * kRowPad / 8; u += NT) reinterpret_cast<uint4*>(sX)[u] = make_uint4(0, 0, 0, 0);
  for (int u = tid; u < 32 * NB * kRowPad / 8; u += NT) reinterpret_cast<uint4*>(sY)[u] = make_uint4(0, 0, 0, 0);
  f32x16 acc[BM];
#pragma unroll
  for (int b = 0; b < BM; ++b) acc[b] = f32x16{};
  constexpr int cx = M / 8, cy = N / 8;
  for (int k0 = beg; k0 < end; k0 += kRows) {
    __syncthreads();
    for (int u = tid; u < (cx + cy) * 8; u += NT) {
      const int k8 = u / (cx + cy), c = u % (cx + cy);
      if (c < cx) {
        put_transposed(sX, X, M, c, k0, k8, end);
      } else {
        put_transposed(sY, dY, N, c - cx, k0, k8, end);
      }
    }
    __syncthreads();
#pragma unroll
    for (int kk = 0; kk < kRows; kk += 16) {
      const int nb = NB == 1 ? 0 : wave;
      const bf16x8 b = ld8(sY + (32 * nb + col) * kRowPad + kk + 8 * h);
#pragma unroll
      for (int q = 0; q < BM; ++q) {
        const int mb = NB == 1 ? wave : q;
        if (mb < MB) {
          acc[q] = mfma(ld8(sX + (32 * mb + col) * kRowPad + kk + 8 * h), b, acc[q]);
        }
      }
    }
  }
  float* out = part + static_cast<size_t>(blockIdx.x) * M * N;
#pragma unroll
  for (int q = 0; q < BM; ++q) {
    const int mb = NB == 1 ? wave : q, nb = NB == 1 ? 0 : wave;
    const int n = 32 * nb + col;
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      const int m = 32 * mb + 8 * (e >> 2) + 4 * h + (e & 3);
      if (m < M && n < N) out[m * N + n] = acc[q][e];
    }
  }
}

// g += the slices' partials, every weight matrix of the network in one
// launch: one workgroup per 256 weights of one matrix.
__global__ __launch_bounds__(NT) void k_wgrad_sum(WgradTable t, float* g) {
  uint32_t b = blockIdx.x;
  int q = 0;
  while (q + 1 < t.n && b >= t.first_block[q + 1]) ++q;
  const uint32_t i = (b - t.first_block[q]) * NT + threadIdx.x;
  if (i >= t.size[q]) return;
  const float* p = t.part[q] + i;
  float s[4] = {};
  int k = 0;
  for (; k + 4 <= t.slices[q]; k += 4) {
#pragma unroll
    for (int u = 0; u < 4; ++u) s[u] += p[static_cast<size_t>(k + u) * t.size[q]];
  }
  for (; k < t.slices[q]; ++k) s[0] += p[static_cast<size_t>(k) * t.size[q]];
  g[t.dst[q] + i] += (s[0] + s[1]) + (s[2] + s[3]);
}

}  // namespace

// The waves' row tiles: four workgroups per CU at most (three fit the LDS of
// the widest layers, whose weights take 40 KB), two where each ends with an
// atomic per column (11.5 ns each on one address).
template <int K, int N>
void dense(hipStream_t s, const DenseArgs& g) {
  static_assert(K % 16 == 0, "whole MFMA steps");
  if (g.M <= 0) return;
  const int wgs = (g.M + 32 * kWaves - 1) / (32 * kWaves);
  k_dense<K / 16, N><<<std::min(wgs, g.colsum ? 512 : 1024), NT, 0, s>>>(g);
}
template void dense<80, 128>(hipStream_t, const DenseArgs&);
template void dense<128, 128>(hipStream_t, const DenseArgs&);
template void dense<160, 128>(hipStream_t, const DenseArgs&);
template void dense<128, 16>(hipStream_t, const DenseArgs&);
template void dense<16, 128>(hipStream_t, const DenseArgs&);
template void dense<128, 160>(hipStream_t, const DenseArgs&);
template void dense<128, 80>(hipStream_t, const DenseArgs&);

template <int N>
void edge_grad(hipStream_t s, int M, const float* dy, int ld_dy, int group, const float* pre,
               bf16* d16, float* colsum) {
  if (M <= 0) return;
  k_edge_grad<N><<<(M + kEdgeRows - 1) / kEdgeRows, NT, 0, s>>>(M, dy, ld_dy, group, pre, d16,
                                                               colsum);
}
template void edge_grad<128>(hipStream_t, int, const float*, int, int, const float*, bf16*,
                             float*);

int wgrad_slices(size_t K) {
  return static_cast<int>(std::clamp<size_t>((K + kRows - 1) / kRows, 1, 256));
}

template <int M, int N>
void wgrad_part(hipStream_t s, size_t K, const bf16* X, const bf16* dY, float* part) {
  const int slices = wgrad_slices(K);
  // whole steps per slice; the last slices may be empty (their partial is 0)
  const int per = static_cast<int>((K + slices - 1) / slices + kRows - 1) / kRows * kRows;
  k_wgrad<M, N><<<slices, NT, 0, s>>>(static_cast<int>(K), X, dY, per, part);
}
template void wgrad_part<80, 128>(hipStream_t, size_t, const bf16*, const bf16*, float*);
template void wgrad_part<128, 128>(hipStream_t, size_t, const bf16*, const bf16*, float*);
template void wgrad_part<160, 128>(hipStream_t, size_t, const bf16*, const bf16*, float*);
template void wgrad_part<128, 16>(hipStream_t, size_t, const bf16*, const bf16*, float*);

void wgrad_sum(hipStream_t s, WgradTable& t, float* g) {
  uint32_t blocks = 0;
  for (int q = 0; q < t.n; ++q) {
    t.first_block[q] = blocks;
    blocks += (t.size[q] + NT - 1) / NT;
  }
  if (blocks) k_wgrad_sum<<<blocks, NT, 0, s>>>(t, g);
}

}  // namespace tit_amd
