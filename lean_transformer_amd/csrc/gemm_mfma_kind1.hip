// Instantiates the tiled bf16 GEMM kernels with the EPI_ACT_FWD epilogue (dense layouts and block-sparse products).
#include "gemm_mfma_kernels.h"

int lt_mfma_launch_dense_kind1(const GemmProblem& p, int io_dtype, hipStream_t stream) {
  return launch_layout<EPI_ACT_FWD>(p, io_dtype, stream);
}

int lt_mfma_launch_sparse_kind1(const GemmProblem& p, hipStream_t stream) { return launch_sparse<EPI_ACT_FWD>(p, stream); }
