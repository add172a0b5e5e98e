// Arguments of one (batched, split-K) GEMM C[m][n] = bias[n] + sum_k A(m,k) B(k,n),
// shared by the fp32-MFMA kernels of linear.hip and the bf16 ones of
// gemm_split.hip.
#pragma once
#include "wha_launch.hpp"

namespace wha {

struct GemmArgs {
  const float* a;
  int64_t a_sm, a_sk;  // A(m,k) = a[m*a_sm + k*a_sk]
  const float* b;
  int64_t b_sn, b_sk;  // B(k,n) = b[n*b_sn + k*b_sk]
  float* c;
  int64_t ldc;         // C(m,n) = c[m*ldc + n]  (or the split-K partial [z][M][N])
  const float* bias;   // [N] or nullptr
  int M, N, K;
  int k_chunk;         // k range per split (multiple of the stage depth)
  bool c_vec;          // c, ldc and c_sb allow 128-bit stores
  bool accumulate;     // C += result instead of C = result
  int batch = 1;       // independent GEMMs, operands offset by the strides below
  int splits = 1;      // blockIdx.z = batch index * splits + split index
  int64_t a_sb = 0, b_sb = 0, c_sb = 0, bias_sb = 0;
  bool a_vec = false;  // A's base, batch stride and row stride along its contiguous
  bool b_vec = false;  // direction are 16-byte multiples (set by gemm_t, gemm_split); same for B
  // Row sums of A over the k range (A row-contiguous only, i.e. the weight-gradient
  // GEMM, where they are the bias gradient): rowsum[bt*rowsum_sb + m] = sum_k A(m,k),
  // written by the blocks of the first column tile; with split-K each split writes
  // rowsum_part[(bt*splits + split)*M + m] and the reduce adds the splits in order.
  float* rowsum = nullptr;
  int64_t rowsum_sb = 0;
  float* rowsum_part = nullptr;
  // bytes of one batch's A and B that the VEC loads may touch (the buffer
  // descriptors' extents; set by gemm_dma_ok, gemm_vec_ok)
  uint32_t a_bytes = 0, b_bytes = 0;
};

inline bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

// Sums the split-K partial tiles ws [batch * splits][M][N] into C (bias, accumulate).
hipError_t gemm_reduce(const GemmArgs& g, const float* ws, hipStream_t stream);

// gemm_split.hip.  gemm_split_ok / _dw_ok: the size rules under which these kernels run.
struct GemmPick {
  int bm, bn, splits;
};
bool gemm_split_ok(int64_t M, int64_t N, int64_t K, int64_t batch);
bool gemm_split_dw_ok(int64_t M, int64_t N, int64_t K, int64_t batch);
GemmPick gemm_pick(int M, int N, int K, int batch, bool rows_contiguous, int max_splits, int min_k);
template <bool A_KC, bool B_KC>
hipError_t gemm_split(const GemmArgs& g, const GemmPick& t, float* ws, const char* name, hipStream_t stream);

}  // namespace wha
