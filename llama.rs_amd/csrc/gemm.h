// gemm.h — batched prefill products Y = X W^T on int8 MFMA (ops.rs:150-313,
// integer semantics of RUST_LLAMA_BATCH_INT=1).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "matvec.h"
#include "rlh_format.h"

namespace rlh {

struct GemmArgs {
  DevMat w;        // rows x cols, tiled layout (rlh_format.h)
  Q8Tiles x;       // n Q8 activation rows in 32-token tiles (rlh_format.h)
  uint32_t n;      // tokens
  float* y;        // y[t * rows + r] = total (nullable)
  float* resid;    // resid[t * rows + r] += total (nullable)
  uint32_t n_tt;   // token tiles of the launched variant
  uint32_t n_rt;   // its row tiles of all segments
  // optional second and third segments of the same type and columns (the q, k
  // and v products of a layer in one launch): row tiles from n_rt1 on belong
  // to w2 and write y2, those from n_rt2 on to w3 and y3 (no residual)
  DevMat w2, w3;
  float *y2, *y3;
  uint32_t n_rt1;  // row tiles of w (n_rt when there is no second segment)
  uint32_t n_rt2;  // row tiles of w and w2
};

bool gemm_supported(uint32_t ty);
// Raises the kernels' dynamic LDS limits (once, before the first launch).
bool gemm_set_max_lds();
// Y[n][rows] (token-major) for the n activation rows; cols % 256 == 0.
void launch_gemm(hipStream_t st, const DevMat& w, const Q8Tiles& x, uint32_t n, float* y, float* resid);
// Two or three products of one activation in one launch: Y[n][w.rows],
// Y2[n][w2.rows] and (w3 not null) Y3[n][w3->rows], all weights of the same
// supported type and columns.
bool gemm_pair_supported(const DevMat& w, const DevMat& w2);
void launch_gemm_pair(hipStream_t st, const DevMat& w, const DevMat& w2, const Q8Tiles& x, uint32_t n, float* y,
                      float* y2, const DevMat* w3 = nullptr, float* y3 = nullptr);
// Weight types without an integer batch path (Q5_K, Q4_1, Q5_0, Q5_1, F16,
// BF16, F32): matmul_batch's f32 route on the f32 activations x[n][cols]; the
// tokens from n4 on (the last n % 4 of the whole batch; all of them for F32
// weights) take the single-token dot order.
bool gemm_f32_supported(uint32_t ty);
void launch_gemm_f32(hipStream_t st, const DevMat& w, const float* x, uint32_t n, uint32_t n4, float* y,
                     float* resid);
// Two or three of them with one activation in one launch (same type and columns).
bool gemm_f32_pair_supported(const DevMat& w, const DevMat& w2);
void launch_gemm_f32_pair(hipStream_t st, const DevMat& w, const DevMat& w2, const float* x, uint32_t n, uint32_t n4,
                          float* y, float* y2, const DevMat* w3 = nullptr, float* y3 = nullptr);

}  // namespace rlh
