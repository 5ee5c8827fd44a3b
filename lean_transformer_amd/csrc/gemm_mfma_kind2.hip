// Instantiates the tiled bf16 GEMM kernels with the EPI_ACT_BWD epilogue (dense layouts).
#include "gemm_mfma_kernels.h"

int lt_mfma_launch_dense_kind2(const GemmProblem& p, int io_dtype, hipStream_t stream) {
  return launch_layout<EPI_ACT_BWD>(p, io_dtype, stream);
}
