// Dense-layer building blocks of the learned step: a BF16 MFMA GEMM with
// fused epilogues, and the small element-wise / graph kernels around it.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace tit_amd {

typedef __bf16 bf16;

enum NnAct { kActNone = 0, kActHswish = 1 };

// The network's activation, hard-swish x min(max(x / 6 + 1/2, 0), 1): three
// full-rate VALU operations (an FMA, a clamp, a product), used by every
// layer (training GEMM epilogues, the derivative, the fused inference kernel).
__device__ __forceinline__ float nn_gate(float x) {
  return __builtin_amdgcn_fmed3f(__builtin_fmaf(x, 1.0f / 6.0f, 0.5f), 0.0f, 1.0f);
}
__device__ __forceinline__ float nn_act(float x) { return x * nn_gate(x); }
// 0 below -3, x / 3 + 1/2 on (-3, 3), 1 above 3
__device__ __forceinline__ float nn_act_grad(float x) {
  const float g = nn_gate(x);
  return (x > -3.0f && x < 3.0f) ? __builtin_fmaf(x, 1.0f / 6.0f, g) : g;
}

// C[M x N] = act(op(A)[M x K] . op(B)[K x N] + bias + G1[r1[m]] + G2[r2[m]])
// with BF16 operands and FP32 accumulation.  op(A) is A (row-major, lda) or,
// with transA, the transpose of a row-major K x M matrix; likewise for B.
// Outputs (any may be null): pre (FP32 before the activation), out32 (FP32
// after), out16 (BF16 after).  With accumulate, out32 += result through
// atomics (split-K over k_splits slices of K; out32 must hold the running
// sum).
struct GemmArgs {
  int M = 0, N = 0, K = 0;
  const bf16* A = nullptr;
  int lda = 0;
  bool transA = false;
  const bf16* B = nullptr;
  int ldb = 0;
  bool transB = false;
  const float* bias = nullptr;
  const float* G1 = nullptr;  // row-gathered addends, ld = N
  const uint32_t* r1 = nullptr;
  const float* G2 = nullptr;
  const uint32_t* r2 = nullptr;
  int act = kActNone;
  float* pre = nullptr;
  int ldpre = 0;
  float* out32 = nullptr;
  int ldo32 = 0;
  bf16* out16 = nullptr;
  int ldo16 = 0;
  bool accumulate = false;
  int k_splits = 1;
};

void gemm_bf16(hipStream_t s, const GemmArgs& g);

// col_sum[n] += sum_m in[m][n].
void column_sum(hipStream_t s, int M, int N, const float* in, float* col_sum);
// Adam on FP32 master weights, refreshing the BF16 copy.
void adam_update(hipStream_t s, int n, float* w, bf16* w16, const float* g,
                 float* m, float* v, float lr, float b1, float b2, float eps,
                 float bc1, float bc2);
void fill_f32(hipStream_t s, size_t n, float* p, float value);

// ---- dense layers of the training (nn_train.hip) -----------------------------
// out = act(A . B + bias), A M x K row-major BF16, B = W (K x N row-major) or,
// with trans, the transpose of the row-major N x K matrix W.  K and N are the
// network's layer sizes: nn_train.hip instantiates them, another pair does not
// link.  pre (M x N): the value before the activation;
// group16: BF16 sums of every kGroupRows rows of the output.  With bpre (M x N):
// out16 = (A . B) act'(bpre), colsum[n] += its column sums; out16 may be A.
constexpr int kGroupRows = 8;
struct DenseArgs {
  int M = 0;
  const bf16* A = nullptr;
  int lda = 0;
  const bf16* W = nullptr;
  int ldw = 0;
  bool trans = false;
  const float* bias = nullptr;
  int act = kActNone;
  float* pre = nullptr;
  bf16* out16 = nullptr;
  int ldo16 = 0;
  float* out32 = nullptr;
  int ldo32 = 0;
  bf16* group16 = nullptr;
  int ldg = 0, colg = 0;
  const float* bpre = nullptr;
  float* colsum = nullptr;
};
template <int K, int N>
void dense(hipStream_t s, const DenseArgs& g);
// d16[m][n] = dy[m / group][n] act'(pre[m][n]) (M x N), colsum[n] += its
// column sums.
template <int N>
void edge_grad(hipStream_t s, int M, const float* dy, int ld_dy, int group, const float* pre,
               bf16* d16, float* colsum);
// Partial products X^T dY (X: K x M, dY: K x N, BF16 row-major) over
// wgrad_slices(K) row slices, M x N each; wgrad_sum adds every listed
// matrix's slices to its place in the gradient.
int wgrad_slices(size_t K);
template <int M, int N>
void wgrad_part(hipStream_t s, size_t K, const bf16* X, const bf16* dY, float* part);
struct WgradTable {
  static constexpr int kMax = 10;
  int n = 0;
  const float* part[kMax];
  int slices[kMax];
  uint32_t size[kMax], dst[kMax], first_block[kMax];
};
void wgrad_sum(hipStream_t s, WgradTable& t, float* g);

}  // namespace tit_amd
