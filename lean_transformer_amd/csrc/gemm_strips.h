// Epilogue of a wavefront's 64 x 64 sub-tile of a copy-based kernel: the 128 x 128 tiles (gemm_mid.hip) and the block-sparse walks
// (gemm_walk.hip).  Needs gemm_mfma_kernels.h.
#pragma once

namespace {

// Strips of 32 rows x 64 columns, transposed through `stage`, 8 KiB of LDS of this wavefront's own, and read back 8 columns per lane;
// what a strip reads from memory is requested before it is staged.  Accumulator register r of a 32 x 32 block is row
// 8 (r / 4) + 4 (lane / 32) + r % 4, column lane % 32; columns of rows with bit 2 set are staged 32 further on (banks).
// Rows m_first .. + 63, columns n_first .. + 63 of the result; PAIR (gated forward): acc[i][0] are gate columns n_first .. + 31,
// acc[i][1] the matching linear ones.  slice: of a split reduction.
template <int KIND, typename TX, int ACT, bool PAIR>
__device__ __forceinline__ void strip_epilogue(const f32x16 (&acc)[2][2], const GemmProblem& p, const int slice, float* stage,
                                               const int64_t m_first, const int64_t n_first, const int lane) {
  EpiParams epi = p.epi;
  if (KIND == EPI_STORE && p.ksplit > 1) epi.out = reinterpret_cast<float*>(epi.out) + (int64_t)slice * p.split_stride;
  epi.bias = nullptr;
  auto staged = [&](int row, int col) -> float* { return &stage[row * 64 + (col ^ (((row >> 2) & 1) << 5))]; };
  float colsum[16];  // EPI_ACT_BWD: column sums of the dpre values this lane writes
#pragma unroll
  for (int e = 0; e < 16; e++) colsum[e] = 0.f;
  constexpr int PER_ROW = PAIR ? 4 : 8, ROWS = 64 / PER_ROW, NIT = 32 / ROWS;
  const int c = (lane % PER_ROW) * 8;
  const int64_t n = n_first + c;
  const bool in_n = n < p.N;  // N is a multiple of 8
  float bias0[8], bias1[8];
#pragma unroll
  for (int e = 0; e < 8; e++) bias0[e] = bias1[e] = 0.f;
  if (p.epi.bias && in_n) {
    load8(p.epi.bias + n, bias0);
    if constexpr (PAIR) load8(p.epi.bias + epi.inter + n, bias1);
  }
  // WHOLE (forward, activation fixed): every row and column exists.  A strip's values are then read back before the first is used,
  // with no branch around a row.  Paired walk, row by row behind a branch against this: hidden 4096, tiled butterfly, T 4096 296 us, 290;
  // T 2048 143, 138; 128 x 128 tiles, [512, 2048] x 8192 27.1, 26.4.
  auto strips = [&](auto W) __attribute__((always_inline)) {
    constexpr bool WHOLE = decltype(W)::value;
#pragma unroll
    for (int i = 0; i < 2; i++) {
      const int64_t mrow0 = m_first + i * 32 + lane / PER_ROW;
      EpiLoad in[NIT];
      if constexpr (KIND == EPI_ACT_BWD || KIND == EPI_OUT) {
#pragma unroll
        for (int it = 0; it < NIT; it++)
          in[it] = epi_load8<KIND, TX>(epi, min(mrow0 + it * ROWS, p.M - 1), in_n ? n : 0, true);
      }
      __builtin_amdgcn_wave_barrier();
#pragma unroll
      for (int j = 0; j < 2; j++)
#pragma unroll
        for (int r = 0; r < 16; r++) *staged(8 * (r >> 2) + 4 * (lane >> 5) + (r & 3), j * 32 + (lane & 31)) = acc[i][j][r];
      __builtin_amdgcn_wave_barrier();
      auto read8 = [&](int it, int col, const float (&bias)[8], float (&v)[8]) __attribute__((always_inline)) {
        const float* sv = staged(it * ROWS + lane / PER_ROW, col);
        const f32x4 lo = *reinterpret_cast<const f32x4*>(sv), hi = *reinterpret_cast<const f32x4*>(sv + 4);
#pragma unroll
        for (int e = 0; e < 4; e++) {
          v[e] = lo[e] + bias[e];
          v[4 + e] = hi[e] + bias[4 + e];
        }
      };
      if constexpr (WHOLE) {
        float v[NIT][8], vl[NIT][8];
#pragma unroll
        for (int it = 0; it < NIT; it++) {
          read8(it, c, bias0, v[it]);
          if constexpr (PAIR) read8(it, 32 + c, bias1, vl[it]);
        }
#pragma unroll
        for (int it = 0; it < NIT; it++) epi_act_fwd8_fixed<PAIR, ACT>(epi, mrow0 + it * ROWS, n, v[it], vl[it]);
      } else {
#pragma unroll
        for (int it = 0; it < NIT; it++) {
          const int64_t m = mrow0 + it * ROWS;
          float v[8];
          read8(it, c, bias0, v);
          if constexpr (PAIR) {
            float vl[8];
            read8(it, 32 + c, bias1, vl);
            if (in_n && m < p.M) epi_act_fwd_gated8<ACT>(epi, m, n, v, vl);
          } else if (in_n && m < p.M) {
            if constexpr (KIND == EPI_STORE) epi_store8(epi, m, n, v);
            else if constexpr (KIND == EPI_ACT_FWD) epi_act_fwd8<ACT>(epi, m, n, v);
            else if constexpr (KIND == EPI_ACT_BWD) epi_act_bwd8_loaded<ACT>(epi, m, n, v, in[it], colsum);
            else epi_out8_loaded<TX>(epi, m, n, v, in[it]);
          }
        }
      }
    }
  };
  if constexpr (KIND == EPI_ACT_FWD && ACT >= 0) {
    if (m_first + 64 <= p.M && n_first + (PAIR ? 32 : 64) <= p.N) strips(std::true_type{});
    else strips(std::false_type{});
  } else {
    strips(std::false_type{});
  }
  if constexpr (KIND == EPI_ACT_BWD) {
    if (epi.colsum) {  // lanes l, l + 8, ... hold the same columns; one partial row per 64 rows of the result
#pragma unroll
      for (int e = 0; e < 16; e++)
#pragma unroll
        for (int mask = 8; mask < 64; mask <<= 1) colsum[e] += __shfl_xor(colsum[e], mask, 64);
      if (lane < 8 && in_n && m_first < p.M) {
        float* dst = epi.colsum + (m_first / 64) * epi.ld_pre + n;
        float lo[8], hi[8];
#pragma unroll
        for (int e = 0; e < 8; e++) {
          lo[e] = colsum[e];
          hi[e] = colsum[8 + e];
        }
        store8(dst, lo);
        if (epi.gated) store8(dst + epi.inter, hi);
      }
    }
  }
}

}  // namespace
