// Products of up to 64 rows with a weight matrix (token-by-token generation):  C[m, n] = sum_k A[m, k] W[n, k], both operands k-major,
// fp32 or 16-bit, with the forward epilogues fused.
//
// What bounds it: the weights, which are read once (403 MB per token at hidden 4096, gated: 70 us at 5.8 TB/s); a 256 x 256 tile
// spends all its time on a few rows, and leaves most CUs without a tile (hidden 4096, one token: 220 us for the block; 88 now, its two
// launches 55 and 31 us = 4.9 and 4.4 TB/s).  So the reduction
// is split over the wavefronts of a workgroup: a workgroup owns 16 NT rows of W (gated up-projection: half of them gate rows, half
// the matching linear rows), wavefront w takes the 128-byte k-blocks w, w + W, ... of all of them, and the partial sums meet in
// LDS at the end, in wavefront order, so that a result is the same at every run.  A block is fetched 128 contiguous bytes per 8 lanes
// into registers, DEPTH blocks ahead, and goes through a buffer in LDS that belongs to the wavefront alone (no barrier in the loop)
// into the layout of v_mfma_f32_16x16x32 (fp32: v_mfma_f32_16x16x4, plain fp32 arithmetic), W as the first operand, so that a
// lane ends up with 4 consecutive columns of one row.  Blocks past the end of the reduction arrive as zeros.
//
// LayerNorm in front of an up-projection of a few rows (FfnStream::ln_weight) is part of it: every workgroup normalises them, from its XCD's
// L2, behind its first requests for weights, and keeps them in LDS, up to 32 KiB, where the loop reads them.  A launch of its own takes 4 -
// 9 us for a row or two: three trips to memory, one behind another.  (Rows normalised block by block on their way through the loop took more
// registers: one workgroup on a CU where there had been two, one row, hidden 3776 79 us -> 84.)
//
// The same kernel computes the thin products of a low-rank term, hid = x L1^T and g L2, with the roles exchanged (THIN): the rows of the
// activation are streamed as the weights are, once, against up to 64 rows of the factor, which comes out of L2; L2, whose rows are k, goes through
// LDS as it is and is transposed by the reads (ds_read_b64_tr_b16).  128 x 128 tiles leave half or more of such a tile empty and most CUs
// without one, or pay for a sum of slices.  lt_gemm_thin_selected has the line and both sides.
#include <algorithm>

#include "lt_internal.h"

namespace {

template <typename TI> struct StreamMfma {  // 16-bit
  static __device__ __forceinline__ f32x4 run(const lt_u32x4& a, const lt_u32x4& b, f32x4 c) {
    return LT_MFMA_16X16X32(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c);
  }
};
template <> struct StreamMfma<float> {
  static __device__ __forceinline__ f32x4 run(const lt_u32x4& a, const lt_u32x4& b, f32x4 c) {
    const f32x4 fa = __builtin_bit_cast(f32x4, a), fb = __builtin_bit_cast(f32x4, b);
#pragma unroll
    for (int e = 0; e < 4; e++) c = __builtin_amdgcn_mfma_f32_16x16x4f32(fa[e], fb[e], c, 0, 0, 0);
    return c;
  }
};

struct NoLn {};
// the 16-byte words of 8 consecutive elements, in fp32
template <typename T> __device__ __forceinline__ void widened(const lt_u32x4* w, float (&v)[8]) {
  if constexpr (sizeof(T) == 2) unpack_bf16x8(w[0], v);
  else {
#pragma unroll
    for (int i = 0; i < 8; i++) v[i] = __builtin_bit_cast(f32x4, w[i / 4])[i % 4];
  }
}

// MT: 16-row tiles of A (M <= 16 MT), NT: 16-row tiles of W per workgroup, WAVES: wavefronts per workgroup
// XT, VT: with LayerNorm, the types of its input and of its parameters (NoLn: A is used as it is)
// THIN: 1, 2: the result is stored transposed, out[n, m]; 2: A is mn-major, element (m, k) at ptr[k * ld + m]
template <typename TI, int KIND, typename TX, int MT, int NT, int WAVES, typename XT = NoLn, typename VT = NoLn, int THIN = 0>
__global__ __launch_bounds__(64 * WAVES) __attribute__((amdgpu_waves_per_eu(std::is_same<XT, NoLn>::value ? 1 : WAVES / 2 < 4 ? 2 : 4)))
void gemm_stream_kernel(GemmProblem p, FfnStream ffn) {
  constexpr bool LN = !std::is_same<XT, NoLn>::value;
  constexpr int TILES = LN ? NT : NT + MT, LOADS = 2 * TILES;  // per block and wavefront, 1 KiB each
  constexpr int DEPTH = LOADS <= 10 ? 3 : 2;             // blocks in flight (registers)
  constexpr int STAGE = TILES * 16 * 8;                  // 16-byte words: TILES * 16 rows of 128 bytes
  constexpr int PAIRS = NT * MT;                         // 16 x 16 results
  static_assert(PAIRS * 64 <= STAGE, "the partial sums take the place of the staged blocks");
  __shared__ lt_u32x4 smem[WAVES * STAGE];
  __shared__ lt_u32x4 ln_rows[LN ? LT_STREAM_LN_BYTES / 16 + 16 * MT : 1];
  char* const rows = reinterpret_cast<char*>(ln_rows);

  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const bool gated = KIND == EPI_ACT_FWD && p.epi.gated;
  const int M = (int)p.M;
  const int64_t N = p.N;  // gated: gate columns
  const int own = gated ? NT / 2 : NT;  // tiles of output columns
  const int64_t n0 = (int64_t)blockIdx.x * own * 16;

  // 16-byte piece j of a block: row j * 8 + lane / 8 of [W tiles, A tiles], piece lane % 8 of its 128 bytes.  Rows past the last one
  // read the last one again; they only feed results that are not stored.
  const int row_in = lane >> 3;
  const uint32_t k_bytes = (uint32_t)(p.K[0] * sizeof(TI));
  const char* const w_base = reinterpret_cast<const char*>(p.B[0].ptr) + n0 * p.B[0].ld * (int64_t)sizeof(TI);
  const char* const w_base2 = w_base + (gated ? N * p.B[0].ld * (int64_t)sizeof(TI) : 0);  // the linear half
  const char* const a_base = reinterpret_cast<const char*>(p.A[0].ptr);
  uint32_t off[LOADS];
#pragma unroll
  for (int j = 0; j < LOADS; j++) {
    if (j < 2 * NT) {
      const int tile = j >> 1, t = gated && tile >= NT / 2 ? tile - NT / 2 : tile;
      const int64_t n = min(n0 + t * 16 + (j & 1) * 8 + row_in, N - 1) - n0;
      off[j] = (uint32_t)(n * p.B[0].ld * (int64_t)sizeof(TI));
    } else if constexpr (THIN == 2) {  // piece j * 64 + lane of a block's 64 k x 2 MT pieces of 8 columns; past the last column the last 8 again
      off[j] = (uint32_t)(min((((j - 2 * NT) * 64 + lane) % (2 * MT)) * 8, M - 8) * (int)sizeof(TI));
    } else {
      off[j] = (uint32_t)(min((j - 2 * NT) * 8 + row_in, M - 1) * p.A[0].ld * (int64_t)sizeof(TI));
    }
  }
  // (THIN == 2) k of that piece inside its block, and the piece's place in a row of LDS: 16 rows are read at once, 32 bytes of each
  auto thin_k = [&](int j) { return ((j - 2 * NT) * 64 + lane) / (2 * MT); };
  auto thin_slot = [](int k, int c) { return k * 2 * MT + (MT == 4 ? c ^ (((k >> 1 & 1) << 1) | ((k >> 3 & 1) << 2)) : MT == 2 ? c ^ ((k >> 3 & 1) << 1) : c); };
  const uint32_t my_k = (uint32_t)(lane & 7) * 16;
  auto fetch = [&](uint32_t block, lt_u32x4 (&r)[LOADS]) __attribute__((always_inline)) {
    const uint32_t k = min(block * 128 + my_k, k_bytes - 16);
#pragma unroll
    for (int j = 0; j < LOADS; j++) {
      if constexpr (THIN == 2) {
        if (j >= 2 * NT) {
          const uint32_t row = min(block * 64 + thin_k(j), (uint32_t)p.K[0] - 1);
          r[j] = *reinterpret_cast<const lt_u32x4*>(a_base + (size_t)(off[j] + row * (uint32_t)(p.A[0].ld * sizeof(TI))));
          continue;
        }
      }
      const char* base = j >= 2 * NT ? a_base : (NT > 1 && j >= NT) ? w_base2 : w_base;
      r[j] = *reinterpret_cast<const lt_u32x4*>(base + (size_t)(off[j] + k));
    }
  };

  f32x4 acc[NT][MT];
#pragma unroll
  for (int i = 0; i < NT; i++)
#pragma unroll
    for (int j = 0; j < MT; j++) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  lt_u32x4* const stage = smem + wave * STAGE;
  // row r keeps its 16-byte piece c in slot c ^ (r / 2) % 8: the 16 rows a quarter of the wavefront reads cover all 64 banks
  auto slot = [](int r, int c) { return r * 8 + (c ^ ((r >> 1) & 7)); };
  // (LayerNorm) the normalised rows, a 16-byte piece more than a row apart (banks)
  const uint32_t row_bytes = k_bytes + 16;
  auto consume = [&](uint32_t block, const lt_u32x4 (&r)[LOADS]) __attribute__((always_inline)) {
    const bool inside = block * 128 + my_k < k_bytes;
#pragma unroll
    for (int j = 0; j < LOADS; j++) {
      lt_u32x4 v = r[j];
      if constexpr (THIN == 2) {
        if (j >= 2 * NT) {
          const bool live = block * 64 + thin_k(j) < (uint32_t)p.K[0];
#pragma unroll
          for (int e = 0; e < 4; e++) v[e] = live ? v[e] : 0u;
          stage[NT * 128 + thin_slot(thin_k(j), ((j - 2 * NT) * 64 + lane) % (2 * MT))] = v;
          continue;
        }
      }
#pragma unroll
      for (int e = 0; e < 4; e++) v[e] = inside ? v[e] : 0u;
      stage[slot(j * 8 + row_in, lane & 7)] = v;
    }
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int s = 0; s < 2; s++) {
      const int c = (lane >> 4) + 4 * s;
      lt_u32x4 w[NT], a[MT];
#pragma unroll
      for (int i = 0; i < NT; i++) w[i] = stage[slot(i * 16 + (lane & 15), c)];
#pragma unroll
      for (int j = 0; j < MT; j++) {
        if constexpr (LN) {
          const uint32_t k = block * 128 + c * 16;
          const bool in_row = k < k_bytes;
          a[j] = *reinterpret_cast<const lt_u32x4*>(rows + min(j * 16 + (lane & 15), M - 1) * row_bytes + (in_row ? k : 0));
#pragma unroll
          for (int e = 0; e < 4; e++) a[j][e] = in_row ? a[j][e] : 0u;
        } else if constexpr (THIN == 2) {
          union { lt_u32x4 v; s16x4 h[2]; } u;
          const int col = j * 16 + 4 * (lane & 3);
#pragma unroll
          for (int h = 0; h < 2; h++) {
            const int k = s * 32 + 8 * (lane >> 4) + 4 * h + ((lane & 15) >> 2);
            const bf16* src = reinterpret_cast<const bf16*>(stage + NT * 128 + thin_slot(k, col >> 3)) + (col & 7);
            u.h[h] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)(src));
          }
          a[j] = u.v;
        } else {
          a[j] = stage[slot((NT + j) * 16 + (lane & 15), c)];
        }
      }
#pragma unroll
      for (int i = 0; i < NT; i++)
#pragma unroll
        for (int j = 0; j < MT; j++) acc[i][j] = THIN ? StreamMfma<TI>::run(a[j], w[i], acc[i][j]) : StreamMfma<TI>::run(w[i], a[j], acc[i][j]);
    }
    __builtin_amdgcn_wave_barrier();
  };

  lt_u32x4 regs[DEPTH][LOADS];
  const uint32_t blocks = (k_bytes + 127) / 128;
#pragma unroll
  for (int d = 0; d < DEPTH; d++) fetch(wave + d * WAVES, regs[d]);
  if constexpr (LN) {
    // 8 elements a lane and piece, all wavefronts on a row and ROWS rows at a time: few registers, and gain and shift are read once
    constexpr int PIECES = LT_STREAM_LN_MAX_H / (512 * WAVES) > 0 ? LT_STREAM_LN_MAX_H / (512 * WAVES) : 1;
    constexpr int ROWS = 4;
    constexpr int XW = (int)sizeof(XT) / 2, VW = (int)sizeof(VT) / 2;  // 16-byte words of 8 elements
    __shared__ float row_sums[2][ROWS][WAVES];
    const int H = (int)p.K[0];
    const float inv_h = 1.0f / (float)H;
    auto column = [&](int i) { return ((i * WAVES + wave) * 64 + lane) * 8; };
    lt_u32x4 gain_words[PIECES][VW], shift_words[PIECES][VW];
#pragma unroll
    for (int i = 0; i < PIECES; i++)
      if (column(i) < H)
#pragma unroll
        for (int k = 0; k < VW; k++) {
          gain_words[i][k] = reinterpret_cast<const lt_u32x4*>(reinterpret_cast<const VT*>(ffn.ln_weight) + column(i))[k];
          shift_words[i][k] = reinterpret_cast<const lt_u32x4*>(reinterpret_cast<const VT*>(ffn.ln_bias) + column(i))[k];
        }
    for (int row0 = 0; row0 < M; row0 += ROWS) {
      lt_u32x4 words[ROWS][PIECES][XW];
      float sums[ROWS], mean[ROWS], rstd[ROWS];
#pragma unroll
      for (int r = 0; r < ROWS; r++)
        if (row0 + r < M)
#pragma unroll
          for (int i = 0; i < PIECES; i++)
            if (column(i) < H)
#pragma unroll
              for (int k = 0; k < XW; k++)
                words[r][i][k] = reinterpret_cast<const lt_u32x4*>(reinterpret_cast<const XT*>(a_base) + (row0 + r) * p.A[0].ld + column(i))[k];
      // sums[r] over the workgroup: lanes 16 r .. 16 r + 15 take over row r, a third of the exchanges of four sums one by one
      auto totals = [&](int turn, float (&out)[ROWS]) __attribute__((always_inline)) {
        const bool upper = lane & 32, odd = lane & 16;
        float t[2];
#pragma unroll
        for (int r = 0; r < 2; r++) {
          t[r] = upper ? sums[2 + r] : sums[r];
          t[r] += __shfl_xor(upper ? sums[r] : sums[2 + r], 32, 64);
        }
        float one = odd ? t[1] : t[0];
        one += __shfl_xor(odd ? t[0] : t[1], 16, 64);
#pragma unroll
        for (int mask = 8; mask; mask >>= 1) one += __shfl_xor(one, mask, 64);
        if ((lane & 15) == 0) row_sums[turn][lane >> 4][wave] = one;
        __syncthreads();  // (the buffer is written again two barriers on)
        one = row_sums[turn][lane >> 4][lane & (WAVES - 1)];
#pragma unroll
        for (int mask = WAVES / 2; mask; mask >>= 1) one += __shfl_xor(one, mask, 64);
#pragma unroll
        for (int r = 0; r < ROWS; r++) out[r] = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, one), 16 * r));
      };
#pragma unroll
      for (int r = 0; r < ROWS; r++) {
        sums[r] = 0.f;
        if (row0 + r >= M) continue;
#pragma unroll
        for (int i = 0; i < PIECES; i++)
          if (column(i) < H) {
            float v[8];
            widened<XT>(words[r][i], v);
#pragma unroll
            for (int e = 0; e < 8; e++) sums[r] += v[e];
          }
      }
      totals(0, mean);
#pragma unroll
      for (int r = 0; r < ROWS; r++) {
        sums[r] = 0.f;
        if (row0 + r >= M) continue;
        mean[r] *= inv_h;
#pragma unroll
        for (int i = 0; i < PIECES; i++)
          if (column(i) < H) {
            float v[8];
            widened<XT>(words[r][i], v);
#pragma unroll
            for (int e = 0; e < 8; e++) sums[r] += (v[e] - mean[r]) * (v[e] - mean[r]);
          }
      }
      totals(1, rstd);
#pragma unroll
      for (int r = 0; r < ROWS; r++) {
        if (row0 + r >= M) break;
        rstd[r] = 1.0f / sqrtf(rstd[r] * inv_h + ffn.ln_eps);
#pragma unroll
        for (int i = 0; i < PIECES; i++)
          if (column(i) < H) {
            float v[8], gain[8], shift[8];
            widened<XT>(words[r][i], v);
            widened<VT>(gain_words[i], gain);
            widened<VT>(shift_words[i], shift);
#pragma unroll
            for (int e = 0; e < 8; e++) v[e] = (v[e] - mean[r]) * rstd[r] * gain[e] + shift[e];
            store8(reinterpret_cast<TI*>(rows + (row0 + r) * row_bytes) + column(i), v);
          }
        if (blockIdx.x == 0 && threadIdx.x == 0) reinterpret_cast<float2*>(ffn.ln_stats)[row0 + r] = make_float2(mean[r], rstd[r]);
      }
    }
    __syncthreads();
  }
  for (uint32_t b = wave; b < blocks; b += DEPTH * WAVES) {
#pragma unroll
    for (int d = 0; d < DEPTH; d++) {
      consume(b + d * WAVES, regs[d]);
      fetch(b + (d + DEPTH) * WAVES, regs[d]);
    }
  }

  // ---- partial sums of the wavefronts, then the epilogue: lane = row lane % 16 of A's tile, columns 4 (lane / 16) .. + 3 of W's
  __syncthreads();
  f32x4* const sums = reinterpret_cast<f32x4*>(smem);
#pragma unroll
  for (int i = 0; i < NT; i++)
#pragma unroll
    for (int j = 0; j < MT; j++) sums[(wave * PAIRS + i * MT + j) * 64 + lane] = acc[i][j];
  __syncthreads();
  auto total = [&](int pair, float (&v)[4]) __attribute__((always_inline)) {
    f32x4 t = sums[pair * 64 + lane];
#pragma unroll
    for (int w = 1; w < WAVES; w++) t += sums[(w * PAIRS + pair) * 64 + lane];
#pragma unroll
    for (int e = 0; e < 4; e++) v[e] = t[e];
  };
  constexpr bool PRECISE = sizeof(TI) == 4;
  const EpiParams& e = p.epi;
  auto load_bias = [&](int64_t i, float (&b)[4]) __attribute__((always_inline)) {
    if (ffn.bias_half) load4(reinterpret_cast<const bf16*>(e.bias) + i, b);
    else load4(e.bias + i, b);
  };
  for (int q = wave; q < own * MT; q += WAVES) {
    if constexpr (THIN) {  // the lane's four values are consecutive m
      const int64_t m = (q % MT) * 16 + (lane >> 4) * 4, n = n0 + (q / MT) * 16 + (lane & 15);
      if (m >= M || n >= N) continue;  // (M is a multiple of 8)
      float v[4];
      total(q, v);
      store4(reinterpret_cast<bf16*>(e.out) + n * e.ldo + m, v);
      continue;
    }
    const int64_t m = (q % MT) * 16 + (lane & 15), n = n0 + (q / MT) * 16 + (lane >> 4) * 4;
    if (m >= M || n >= N) continue;  // (N is a multiple of 4)
    float v[4], bias[4] = {0.f, 0.f, 0.f, 0.f};
    total(q, v);
    if (e.bias) load_bias(n, bias);
#pragma unroll
    for (int i = 0; i < 4; i++) v[i] += bias[i];
    if constexpr (KIND == EPI_STORE) {
      if (e.out_dtype == LT_F32) store4(reinterpret_cast<float*>(e.out) + m * e.ldo + n, v);
      else store4(reinterpret_cast<bf16*>(e.out) + m * e.ldo + n, v);
    } else if constexpr (KIND == EPI_ACT_FWD) {
      TI* pre = reinterpret_cast<TI*>(e.pre) + m * e.ld_pre + n;
      float h[4];
#pragma unroll
      for (int i = 0; i < 4; i++) {
        v[i] = to_f32(from_f32<TI>(v[i]));  // the activation sees the stored (rounded) pre-activation, as backward will
        h[i] = act_value<PRECISE>(e.act, v[i]);
      }
      store4(pre, v);
      if (gated) {
        float l[4], lb[4] = {0.f, 0.f, 0.f, 0.f};
        total(q + own * MT, l);
        if (e.bias) load_bias(e.inter + n, lb);
#pragma unroll
        for (int i = 0; i < 4; i++) {
          l[i] = to_f32(from_f32<TI>(l[i] + lb[i]));
          h[i] *= l[i];
        }
        store4(pre + e.inter, l);
      }
      store4(reinterpret_cast<TI*>(e.hid) + m * e.ld_hid + n, h);
    } else {
      const int64_t idx = m * e.ldy + n;
      if (e.drop.p > 0.f) {
        bool keep[4];
        dropout_keep4(e.drop, idx, keep);
#pragma unroll
        for (int i = 0; i < 4; i++) v[i] = keep[i] ? v[i] * e.drop.scale : 0.f;
      }
      if (e.x) {
        float r[4];
        load4(reinterpret_cast<const TX*>(e.x) + idx, r);
#pragma unroll
        for (int i = 0; i < 4; i++) v[i] += r[i];
      }
      store4(reinterpret_cast<TX*>(e.y) + idx, v);
    }
  }
}

template <typename TI, int KIND, typename TX, int MT, int NT, int WAVES>
int launch(const GemmProblem& p, const FfnStream& ffn, bool gated, hipStream_t stream) {
  const int64_t cols = 16 * (gated ? NT / 2 : NT);
  const dim3 grid((unsigned)((p.N + cols - 1) / cols)), block(64 * WAVES);
  if constexpr (KIND == EPI_ACT_FWD && MT == 1) {
    if (ffn.ln_weight) {
      if constexpr (sizeof(TI) == 4)
        hipLaunchKernelGGL((gemm_stream_kernel<TI, KIND, TX, MT, NT, WAVES, float, float>), grid, block, 0, stream, p, ffn);
      else if (!ffn.ln_half)
        hipLaunchKernelGGL((gemm_stream_kernel<TI, KIND, TX, MT, NT, WAVES, float, float>), grid, block, 0, stream, p, ffn);
      else if (ffn.x_dtype == LT_F32)
        hipLaunchKernelGGL((gemm_stream_kernel<TI, KIND, TX, MT, NT, WAVES, float, bf16>), grid, block, 0, stream, p, ffn);
      else
        hipLaunchKernelGGL((gemm_stream_kernel<TI, KIND, TX, MT, NT, WAVES, bf16, bf16>), grid, block, 0, stream, p, ffn);
      LT_LAUNCH_CHECK();
      return LT_OK;
    }
  }
  hipLaunchKernelGGL((gemm_stream_kernel<TI, KIND, TX, MT, NT, WAVES>), grid, block, 0, stream, p, ffn);
  LT_LAUNCH_CHECK();
  return LT_OK;
}

// Workgroup shape.  Many rows of W: four tiles of them per workgroup, which reads A once for 64 of them ([1, 4096] x [32768, 4096]:
// 52.8 us = 5.1 TB/s, two tiles 61.3).  Few: one tile, and more wavefronts share its reduction ([24, 16384] x [4096, 16384]: 35.6 us
// against 39.5 with two tiles, [48, 6400] x [1600, 6400]: 15.3 against 18.3).  Between: two, eight wavefronts ([24, 2048] x [8192,
// 2048]: 8.7 us, 13.6 with one tile; [48, 2048]: 11.6, 18.8).
template <typename TI, int KIND, typename TX> int launch_shape(const GemmProblem& p, const FfnStream& ffn, hipStream_t stream) {
  const bool gated = KIND == EPI_ACT_FWD && p.epi.gated;
  const int64_t rows = gated ? 2 * p.N : p.N;
  const bool many = rows >= 512 * 64, few = rows <= 4096 && !gated;  // (a gated workgroup pairs two tiles)
  if (p.M <= 16) {
    if (many) return launch<TI, KIND, TX, 1, 4, 4>(p, ffn, gated, stream);
    if (few) return launch<TI, KIND, TX, 1, 1, 16>(p, ffn, gated, stream);
    return launch<TI, KIND, TX, 1, 2, 8>(p, ffn, gated, stream);
  }
  if (p.M <= 32) {
    if (many) return launch<TI, KIND, TX, 2, 4, 4>(p, ffn, gated, stream);
    if (few) return launch<TI, KIND, TX, 2, 1, 16>(p, ffn, gated, stream);
    return launch<TI, KIND, TX, 2, 2, 8>(p, ffn, gated, stream);
  }
  if (many) return launch<TI, KIND, TX, 4, 4, 4>(p, ffn, gated, stream);
  if (few) return launch<TI, KIND, TX, 4, 1, 8>(p, ffn, gated, stream);
  return launch<TI, KIND, TX, 4, 2, 8>(p, ffn, gated, stream);
}

template <int MT, int NT, int WAVES> int launch_thin_shape(const GemmProblem& q, hipStream_t stream) {
  const dim3 grid((unsigned)((q.N + 16 * NT - 1) / (16 * NT))), block(64 * WAVES);
  if (q.A[0].kmajor)
    hipLaunchKernelGGL((gemm_stream_kernel<bf16, EPI_STORE, float, MT, NT, WAVES, NoLn, NoLn, 1>), grid, block, 0, stream, q, FfnStream{});
  else
    hipLaunchKernelGGL((gemm_stream_kernel<bf16, EPI_STORE, float, MT, NT, WAVES, NoLn, NoLn, 2>), grid, block, 0, stream, q, FfnStream{});
  LT_LAUNCH_CHECK();
  return LT_OK;
}

template <typename TI> int launch_kind(const GemmProblem& p, const FfnStream& ffn, int kind, int io_dtype, hipStream_t stream) {
  if (kind == EPI_STORE) return launch_shape<TI, EPI_STORE, float>(p, ffn, stream);
  if (kind == EPI_ACT_FWD) return launch_shape<TI, EPI_ACT_FWD, float>(p, ffn, stream);
  if constexpr (sizeof(TI) == 2)
    if (io_dtype == LT_BF16) return launch_shape<TI, EPI_OUT, bf16>(p, ffn, stream);
  return launch_shape<TI, EPI_OUT, float>(p, ffn, stream);
}

}  // namespace

bool lt_gemm_stream_supported(const GemmProblem& p, int kind, int dtype, int io_dtype) {
  const EpiParams& e = p.epi;
  const int64_t piece = dtype == LT_F32 ? 4 : 8, bytes = dtype == LT_F32 ? 4 : 2;  // elements per 16 bytes
  if (p.sp.mode != SPARSE_NONE || p.nseg != 1 || p.ksplit > 1 || p.variant || kind == EPI_ACT_BWD) return false;
  if (p.M < 1 || p.M > 64 || p.N < 1 || p.K[0] < 1 || !p.A[0].kmajor || !p.B[0].kmajor) return false;
  if (dtype == LT_F32 && kind == EPI_OUT && io_dtype != LT_F32) return false;
  // 16-byte pieces of every row, 4 columns per store
  if (p.N % 4 || p.K[0] % piece || p.A[0].ld % piece || p.B[0].ld % piece || !lt_aligned(p.A[0].ptr, 16) || !lt_aligned(p.B[0].ptr, 16))
    return false;
  // 32-bit byte offsets inside a workgroup's rows and along k (the blocks asked for run up to 2 x 3 x 16 past the end before they are clamped)
  if (64 * std::max(p.A[0].ld, p.B[0].ld) * bytes >= (int64_t)1 << 31) return false;
  if ((p.N + 7) / 8 > 0x7fffffff) return false;
  if (e.bias && !lt_aligned(e.bias, 16)) return false;
  if (kind == EPI_STORE) return e.ldo % 4 == 0 && lt_aligned(e.out, 16);
  if (kind == EPI_ACT_FWD)
    return e.ld_pre % 4 == 0 && e.ld_hid % 4 == 0 && e.inter % 4 == 0 && (!e.gated || e.inter == p.N) && e.hid &&
           lt_aligned(e.pre, 16) && lt_aligned(e.hid, 16);
  return e.ldy % 4 == 0 && lt_aligned(e.y, 16) && (!e.x || lt_aligned(e.x, 16));
}

// Rows: graph replays, a LayerNorm launch against this, us: bf16, gated: [1, 512] 16.5, 12.7; [1, 2048] 40.0, 32.4; [4, 1024] 24.1, 19.6; [8,
// 768] 20.7, 18.7; [8, 1024] 24.6, 22.7; [12, 1024] 24.6, 25.7; [16, 1024] 25.3, 28.9; fp32: [4, 2048] 47.7, 47.1; [8, 1024] 30.3, 32.8.
bool lt_stream_ln_supported(int64_t M, int64_t H, int x_dtype, int dtype, bool ln_half) {
  if (M > (dtype == LT_F32 ? 4 : 8) || H % 8 || H > LT_STREAM_LN_MAX_H || M * H * (int64_t)lt_dtype_size(dtype) > LT_STREAM_LN_BYTES) return false;
  return dtype == LT_F32 ? x_dtype == LT_F32 && !ln_half : ln_half || x_dtype == LT_F32;
}

int lt_launch_gemm_stream(const GemmProblem& p, int kind, int dtype, int io_dtype, hipStream_t stream, const FfnStream* ffn_) {
  LT_REQUIRE(lt_gemm_stream_supported(p, kind, dtype, io_dtype), LT_ERR_UNSUPPORTED, "streaming gemm does not take this problem");
  const FfnStream ffn = ffn_ ? *ffn_ : FfnStream{};
  LT_REQUIRE(!ffn.ln_weight || (kind == EPI_ACT_FWD && lt_stream_ln_supported(p.M, p.K[0], ffn.x_dtype, dtype, ffn.ln_half)),
             LT_ERR_UNSUPPORTED, "streaming gemm does not take this LayerNorm");
  LtProfileScope scope("gemm_stream", lt_gemm_flops(p, kind), 0.0, stream);
  return dtype == LT_F32 ? launch_kind<float>(p, ffn, kind, io_dtype, stream) : launch_kind<bf16>(p, ffn, kind, io_dtype, stream);
}

// [M, N] of up to 64 columns, a k-major A of more rows than that, 16-bit operands and result
bool lt_gemm_thin_supported(const GemmProblem& p, int dtype) {
  const EpiParams& e = p.epi;
  if (dtype != LT_BF16 || p.sp.mode != SPARSE_NONE || p.nseg != 1 || p.ksplit > 1 || p.variant || e.bias || e.out_dtype != LT_BF16) return false;
  if (p.M <= 64 || p.N < 8 || p.N > 64 || p.N % 8 || p.K[0] < 8 || p.K[0] % 8 || !p.A[0].kmajor) return false;
  if (p.A[0].ld % 8 || p.B[0].ld % 8 || !lt_aligned(p.A[0].ptr, 16) || !lt_aligned(p.B[0].ptr, 16) || e.ldo % 4 || !lt_aligned(e.out, 8))
    return false;
  // 32-bit byte offsets: inside a workgroup's rows, over the whole factor
  if (64 * p.A[0].ld * 2 >= (int64_t)1 << 31 || (p.B[0].kmajor ? p.N : p.K[0]) * p.B[0].ld * 2 >= (int64_t)1 << 31 || p.K[0] >= (int64_t)1 << 29)
    return false;
  return p.M < (int64_t)1 << 28;  // 16 threads a row (8 wavefronts on 32 rows), less than 2^32 a launch
}

// 128 x 128 tiles (with the sum of their slices) and this, us, operands from memory.  Up to 16 columns: [500, 16] over 768 11.9, 8.2; over 8192
// 18.5, 11.4; [4000, 16] over 1024 15.4, 7.7; over 4096 20.8, 13.0; [16384, 16] over 768 11.6, 11.2; over 2048 25.3, 19.8; over 4096 29.8, 30.4.  More
// rows are several rounds of short workgroups: [24000, 16] over 512 12.0, 13.1; [50000, 16] over 256 13.1, 15.4; [65000, 16] over 64 9.1, 11.5, over
// 1024 29.8, 31.9; from 65537 on the other side is 256 x 256 tiles: [66000, 16] over 256 33, 17; [131072, 16] over 256 35, 25, over 1024 71, 44.  32:
// [4000, 32] over 2304 18.2, 11.9; [8192, 32] over 4096 26.4, 22.1; [12000, 32] over 768 13.1, 13.3.  64 columns, where the factor is read from L2
// more often: [500, 64] over 1024 15.6, 10.1; [4000, 64] over 1024 13.5, 9.8; over 2048 17.6, 13.7; over 4096 20.6, 19.0, but 17.1, 18.4 with the
// activation still in the caches; over 8192 26.4, 29.0 (52.4 where the caller has no room for slices); [16384, 64] over 1024 16.6, 17.2.
bool lt_gemm_thin_selected(const GemmProblem& p, int dtype, bool can_split) {
  if (!lt_gemm_thin_supported(p, dtype)) return false;
  if (p.N <= 16) return p.M <= 8192 || (p.K[0] <= 3072 && (p.M <= 16384 || p.M > 65536));
  return p.M <= 8192 && (p.K[0] <= (p.N <= 32 ? 4096 : 2048) || !can_split);
}

int lt_launch_gemm_thin(const GemmProblem& p, hipStream_t stream) {
  LT_REQUIRE(lt_gemm_thin_supported(p, LT_BF16), LT_ERR_UNSUPPORTED, "thin gemm does not take this problem");
  GemmProblem q = p;  // the factor as A, the activation as the streamed operand
  q.M = p.N; q.N = p.M;
  q.A[0] = p.B[0]; q.B[0] = p.A[0];
  LtProfileScope scope("gemm_thin", lt_gemm_flops(p, EPI_STORE), 0.0, stream);
  // One tile of rows a workgroup while its workgroups run at once, two a CU with up to 16 columns, else one ([4000, 16] over 4096 12.3 us, two
  // tiles 14.5; [8192, 16] over 1024 11.3, 8.8; [8192, 64] over 1024 15.2, 10.2; [4000, 64] over 4096 18.8, 19.1).
  const bool wide = p.M > (p.N <= 16 ? 8191 : 4096);
  if (p.N <= 16) return wide ? launch_thin_shape<1, 2, 8>(q, stream) : launch_thin_shape<1, 1, 16>(q, stream);
  if (p.N <= 32) return wide ? launch_thin_shape<2, 2, 8>(q, stream) : launch_thin_shape<2, 1, 16>(q, stream);
  return wide ? launch_thin_shape<4, 2, 8>(q, stream) : launch_thin_shape<4, 1, 8>(q, stream);
}
