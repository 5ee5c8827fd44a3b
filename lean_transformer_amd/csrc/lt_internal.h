// Internal launchers shared between the translation units of libleanffn.
#pragma once
#include "lt_gemm.h"

// 16-bit vectors -> fp32
struct WidenJobs {
  const void* in[6];
  float* out[6];
  int count[6];
  int n;
};
int lt_widen(const WidenJobs& jobs, hipStream_t stream);
// fp32 tensors -> 16 bits, up to MAX of them in one launch
struct CastJobs {
  static constexpr int MAX = 8;
  const float* in[MAX];
  void* out[MAX];
  int64_t count[MAX];
  unsigned first[MAX];  // first workgroup of each job; the number of workgroups where there is none
  unsigned vec;         // bit j: job j moves 8 elements a lane (16-byte aligned)
  int n;
};
int lt_cast_launch(CastJobs& jobs, hipStream_t stream);
// LayerNorm forward.  y may be null (statistics only).  w, b: fp32, or 16 bits where the output (tail: the input) is.  tail: apply dropout,
// then add `residual` (dtype res_dtype).  widen: vectors that the same launch widens for the kernels behind it.
int lt_ln_forward(int64_t T, int H, float eps, int x_dtype, const void* x, int w_dtype, const void* w, const void* b, int y_dtype,
                  void* y, float* stats, int res_dtype, const void* residual, const DropoutParams* drop, bool tail,
                  hipStream_t stream, const WidenJobs* widen = nullptr);
size_t lt_ln_backward_workspace(int64_t T, int H);
// w_room: H floats for a 16-bit weight where the kernel taken reads it in fp32; dw_dtype: type of dweight and dbias
int lt_ln_backward(int64_t T, int H, int x_dtype, const void* x, const float* stats, int w_dtype, const void* w, float* w_room,
                   int dy_dtype, const void* dy, int dx_dtype, const void* residual_grad, void* dx, int dw_dtype, void* dweight,
                   void* dbias, void* workspace, size_t workspace_bytes, hipStream_t stream, ColReduceQueue* defer = nullptr);
// column sums, in sum_dtype
size_t lt_colsum_workspace(int64_t rows, int cols);
int lt_colsum(int64_t rows, int cols, int64_t ld, int dtype, const void* in, void* out, int sum_dtype, void* workspace,
              size_t workspace_bytes, hipStream_t stream, ColReduceQueue* defer = nullptr);
int lt_act_forward(int64_t T, int64_t I, int gated, int act, int dtype, const void* pre, void* hid, hipStream_t stream);
int lt_act_backward(int64_t T, int64_t I, int gated, int act, int dtype, const void* pre, const void* dhid, void* dpre,
                    hipStream_t stream);
int lt_dropout_cast_colsum(int64_t rows, int cols, int in_dtype, const void* in, int out_dtype, void* out,
                           const DropoutParams& drop, void* colsum, int sum_dtype, void* workspace, size_t workspace_bytes,
                           hipStream_t stream, ColReduceQueue* defer = nullptr);
int lt_dropout_cast(int64_t n, int in_dtype, const void* in, int out_dtype, void* out, const DropoutParams& drop,
                    hipStream_t stream);
int lt_dropout_mask_launch(int64_t n, uint8_t* keep, const DropoutParams& drop, hipStream_t stream);
