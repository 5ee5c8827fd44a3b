// Tiled 16-bit products of a middling number of rows (65 to about a thousand: a prompt, a short training batch; gradients of small
// factors): 128 x 128 tiles, operands copied global -> LDS, the operand layouts and fused epilogues of the copy-based 256 x 256 kernel.
//
// What bounds it: 256 x 256 tiles of [512, 8192] are 64 workgroups for 256 CUs, each walking the whole reduction; four times as many
// tiles fill the chip, at the price of LDS bandwidth: a wavefront's 64 x 64 sub-tile reads as many cycles of LDS as it has of
// matrix instructions, so a chip full of 256 x 256 tiles is faster over a long reduction (the lines: mid_selected in gemm_mfma_bf16.hip).  A grid of at most
// one workgroup per CU keeps four 64-k stages of both operands in LDS (128 KiB), three of them on their way; a larger one two
// stages, and two workgroups share a CU.  Measured, 256 x 256 tiles against these: [512, 8192] over 2048 43 us, 21 (805 TFLOP/s); [1024,
// 4096] over 16384 276, 137 (1000 TFLOP/s); [768, 3072] over 768 22, 11.
//
// LDS layouts, swizzles and the transposing read of an mn-major operand are those of gemm_mfma_kernels.h.  Every copy tests for the
// end of the reduction (the buffer unit returns zeros past the descriptor's size), so that whole, ragged and absent stages go through
// the same straight-line code.
#include "gemm_mfma_kernels.h"
#include "gemm_staged.h"
#include "gemm_strips.h"

namespace {

constexpr int MID = 128;  // tile rows and columns

// copies of one operand: 64 k x 128 rows per stage, 4 per wavefront
template <bool KM> struct MidOperand {
  static constexpr int LOADS = 4;
  static constexpr uint32_t RECORDS = 0xfffffc00u, OUTSIDE = 0xfffffe00u;
  uint32_t off[LOADS];
  const char* base;
  int64_t unit_bytes;

  // row0: first row (k-major) or column of the tile, of `limit`; past the end the last row / the last 8 columns are copied again.
  // pair_rows > 0 (gated): tile row r is weight row row0 + 32 (r / 64) + r % 32, plus pair_rows where r % 64 >= 32.
  __device__ __forceinline__ void setup(const GemmOperand& op, int64_t row0, int64_t limit, int64_t pair_rows, int wave, int lane) {
    const int64_t ld = op.ld;
    const char* ptr = reinterpret_cast<const char*>(op.ptr);
#pragma unroll
    for (int j = 0; j < LOADS; j++) {
      const int q = (wave * LOADS + j) * 64 + lane;  // 16-byte slot of the stage
      if constexpr (KM) {
        const int row = q >> 3, c = (q & 7) ^ swz_km(row);
        const int local = pair_rows > 0 ? (row >> 6) * 32 + (row & 31) : row;
        int64_t g = min(row0 + local, limit - 1) - row0;
        if (pair_rows > 0) g += ((row >> 5) & 1) * pair_rows;
        off[j] = (uint32_t)((g * ld + c * 8) * 2);
      } else {
        const int kr = q >> 4, c = (q & 15) ^ swz_mn(kr);
        off[j] = (uint32_t)((kr * ld + min(row0 + c * 8, limit - 8) - row0) * 2);
      }
    }
    base = KM ? ptr + row0 * ld * 2 : ptr + row0 * 2;
    unit_bytes = KM ? 64 * 2 : 64 * ld * 2;
  }
  // copies J0 .. J1 - 1 of the 64 k from u * 64 on; pieces at or past k_limit arrive as zeros
  template <int J0, int J1> __device__ __forceinline__ void issue(int u, bf16* dst, int wave, int lane, int k_limit) const {
    const __amdgpu_buffer_rsrc_t rsrc =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(base + u * unit_bytes), 0, (int)RECORDS, 0x00020000);
#pragma unroll
    for (int j = J0; j < J1; j++) {
      const int q = (wave * LOADS + j) * 64 + lane;
      const int k = u * 64 + (KM ? ((q & 7) ^ swz_km(q >> 3)) * 8 : q >> 4);
      const uint32_t o = k < k_limit ? off[j] : OUTSIDE;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (__attribute__((address_space(3))) void*)(dst + (wave * LOADS + j) * 512), 16,
                                               (int)o, 0, 0, 0);
    }
  }
};

// workgroup v of a product's tiles_m x tiles_n tiles and slices
template <bool A_KM, bool B_KM, int KIND, typename TX, int ACT, int STAGES>
__device__ __forceinline__ void mid_workgroup(const GemmProblem& p, const int tiles_m, const int tiles_n, const int v) {
  static_assert(STAGES == 2 || STAGES == 4, "stages");
  constexpr int ELEMS = MID * 64;
  // an array per stage and operand: the compiler can prove that copies and reads do not alias
  __shared__ __attribute__((aligned(1024))) bf16 a0[ELEMS];
  __shared__ __attribute__((aligned(1024))) bf16 a1[ELEMS];
  __shared__ __attribute__((aligned(1024))) bf16 a2[ELEMS];
  __shared__ __attribute__((aligned(1024))) bf16 a3[ELEMS];
  __shared__ __attribute__((aligned(1024))) bf16 b0[ELEMS];
  __shared__ __attribute__((aligned(1024))) bf16 b1[ELEMS];
  __shared__ __attribute__((aligned(1024))) bf16 b2[ELEMS];
  __shared__ __attribute__((aligned(1024))) bf16 b3[ELEMS];
  auto a_buf = [&](auto S) -> bf16* {
    constexpr int s = decltype(S)::value % STAGES;
    return s == 0 ? a0 : s == 1 ? a1 : s == 2 ? a2 : a3;
  };
  auto b_buf = [&](auto S) -> bf16* {
    constexpr int s = decltype(S)::value % STAGES;
    return s == 0 ? b0 : s == 1 ? b1 : s == 2 ? b2 : b3;
  };

  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int wm = wave >> 1, wn = wave & 1;
  const bool gated = KIND == EPI_ACT_FWD && p.epi.gated;

  // each XCD takes a contiguous range of tiles, GROUP_M tile rows at a time
  const bool split = KIND == EPI_STORE && p.ksplit > 1;
  int pid, slice = 0, later = (v >> 3) & 7;  // (later: steps that a workgroup starts behind its neighbour on the XCD)
  if (split) {
    const bool tiles_first = A_KM && lt_split_tiles_first(p.M, p.N, p.K[0]);
    const lt_split_place at = tiles_first ? lt_split_by_tile(v, tiles_m * tiles_n, p.ksplit) : lt_split_by_slice(v, tiles_m * tiles_n, p.ksplit);
    pid = __builtin_amdgcn_readfirstlane(at.tile);
    slice = __builtin_amdgcn_readfirstlane(at.slice);
    if (tiles_first) later = pid & 7;
  } else {
    pid = lt_xcd_order(v, tiles_m * tiles_n);
  }
  const int in_group = GROUP_M * tiles_n, first_m = pid / in_group * GROUP_M, group_m = min(tiles_m - first_m, GROUP_M);
  const int64_t m0 = (int64_t)(first_m + pid % in_group % group_m) * MID;
  const int64_t n0 = (int64_t)(pid % in_group / group_m) * (gated ? MID / 2 : MID);

  // this workgroup's stages: first .. first + total of the reduction (a slice of them), walked from `rot` on and around:
  // with a power-of-two leading dimension the rows of a k-major tile otherwise lie on the same memory channels, chip-wide
  const int all = (int)((p.K[0] + 63) / 64);
  int first = 0, total = all;
  if (split) {
    const int per = (all + p.ksplit - 1) / p.ksplit;
    first = min(all, slice * per);
    total = min(per, all - first);
  }
  const int rot = total > 0 ? (int)((unsigned)((v & 7) * (total >> 3) + later) % (unsigned)total) : 0;
  const int k_limit = (int)p.K[0];
  MidOperand<A_KM> ca;
  MidOperand<B_KM> cb;
  ca.setup(p.A[0], m0, p.M, 0, wave, lane);
  cb.setup(p.B[0], n0, p.N, gated ? p.N : 0, wave, lane);
  // copies J0 .. J1 - 1 (A's four, then B's) of step t
  auto copy = [&](auto S, int t, auto J0_, auto J1_) __attribute__((always_inline)) {
    constexpr int j0 = decltype(J0_)::value, j1 = decltype(J1_)::value;
    int u = t + rot;
    if (u >= total) u -= total;
    u = t < total ? first + u : all;  // (past the last step: zeros)
    if constexpr (j0 < 4) ca.template issue<j0, (j1 < 4 ? j1 : 4)>(u, a_buf(S), wave, lane, k_limit);
    if constexpr (j1 > 4) cb.template issue<(j0 > 4 ? j0 - 4 : 0), j1 - 4>(u, b_buf(S), wave, lane, k_limit);
  };

  f32x16 acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; i++)
#pragma unroll
    for (int j = 0; j < 2; j++)
#pragma unroll
      for (int r = 0; r < 16; r++) acc[i][j][r] = 0.f;
  auto frag_km = [&](const bf16* buf, int base, int kk) -> bf16x8 {
    const int row = base + (lane & 31);
    return *reinterpret_cast<const bf16x8*>(&buf[(row * 8 + ((kk * 2 + (lane >> 5)) ^ swz_km(row))) * 8]);
  };
  auto frag_mn = [&](const bf16* tile, int base, int kk) -> bf16x8 {
    union { bf16x8 v; s16x4 h[2]; } u;
    const int i16 = lane & 15, col = base + ((lane >> 4) & 1) * 16 + 4 * (i16 & 3);
#pragma unroll
    for (int s = 0; s < 2; s++) {
      const int kr = kk * 16 + 8 * (lane >> 5) + 4 * s + (i16 >> 2);
      const bf16* src = &tile[kr * MID + ((((col >> 3) ^ swz_mn(kr)) << 3) | (col & 7))];
      u.h[s] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)(src));
    }
    return u.v;
  };
  bf16x8 fa[2][2], fb[2][2];
  auto load = [&](auto S, auto KK, auto F) __attribute__((always_inline)) {
    constexpr int kk = decltype(KK)::value, f = decltype(F)::value;
#pragma unroll
    for (int i = 0; i < 2; i++) {
      if constexpr (A_KM) fa[f][i] = frag_km(a_buf(S), wm * 64 + i * 32, kk);
      else fa[f][i] = frag_mn(a_buf(S), wm * 64 + i * 32, kk);
      if constexpr (B_KM) fb[f][i] = frag_km(b_buf(S), wn * 64 + i * 32, kk);
      else fb[f][i] = frag_mn(b_buf(S), wn * 64 + i * 32, kk);
    }
  };
  auto multiply = [&](auto F) __attribute__((always_inline)) {
    constexpr int f = decltype(F)::value;
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
      for (int j = 0; j < 2; j++) acc[i][j] = LT_MFMA_32X32X16(fa[f][i], fb[f][j], acc[i][j]);
  };
  using Loop = StagedLoop<STAGES, 8, 2 * (A_KM ? 1 : 2) + 2 * (B_KM ? 1 : 2)>;
  Loop::start(0, copy, load);
  Loop::run(0, total, copy, load, multiply);
  wait_copies_and_barrier<0>();

  // ---- epilogue (strip_epilogue)
  float* const stage = reinterpret_cast<float*>(wave == 0 ? a0 : wave == 1 ? a1 : wave == 2 ? b0 : b1);
  if constexpr (KIND == EPI_ACT_FWD) {
    if (gated) strip_epilogue<KIND, TX, ACT, true>(acc, p, slice, stage, m0 + wm * 64, n0 + wn * 32, lane);
    else strip_epilogue<KIND, TX, ACT, false>(acc, p, slice, stage, m0 + wm * 64, n0 + wn * 64, lane);
  } else {
    strip_epilogue<KIND, TX, ACT, false>(acc, p, slice, stage, m0 + wm * 64, n0 + wn * 64, lane);
  }
}

template <bool A_KM, bool B_KM, int KIND, typename TX, int ACT, int STAGES>
__global__ __launch_bounds__(256) void gemm_bf16_mid_kernel(GemmProblem p, int tiles_m, int tiles_n) {
  mid_workgroup<A_KM, B_KM, KIND, TX, ACT, STAGES>(p, tiles_m, tiles_n, (int)(blockIdx.y * gridDim.x + blockIdx.x));
}

// several weight gradients in one launch (both operands mn-major, plain store): workgroups first[j] .. first[j + 1] - 1 are product j's
struct MidGroup {
  GemmProblem p[LT_MID_GROUP_MAX];
  int tiles_m[LT_MID_GROUP_MAX], tiles_n[LT_MID_GROUP_MAX];
  unsigned first[LT_MID_GROUP_MAX];  // (the number of workgroups where there is no product)
};
__global__ __launch_bounds__(256) void gemm_bf16_mid_group_kernel(MidGroup g) {
  int j = 0;
#pragma unroll
  for (int k = 1; k < LT_MID_GROUP_MAX; k++) j += blockIdx.x >= g.first[k];
  mid_workgroup<false, false, EPI_STORE, float, -1, 4>(g.p[j], g.tiles_m[j], g.tiles_n[j], (int)(blockIdx.x - g.first[j]));
}

template <bool A_KM, bool B_KM, int KIND, typename TX> int launch_mid(const GemmProblem& p, hipStream_t stream) {
  const bool gated = KIND == EPI_ACT_FWD && p.epi.gated;
  const int tiles_m = (int)((p.M + MID - 1) / MID), tiles_n = (int)((p.N + (gated ? 63 : 127)) / (gated ? 64 : 128));
  const int slices = p.ksplit > 1 ? p.ksplit : 1;
  const dim3 grid((unsigned)(tiles_m * tiles_n), (unsigned)slices), block(256);
  with_activation<KIND>(p, [&](auto ACT) {
    if (tiles_m * tiles_n * slices <= 256)
      hipLaunchKernelGGL((gemm_bf16_mid_kernel<A_KM, B_KM, KIND, TX, decltype(ACT)::value, 4>), grid, block, 0, stream, p, tiles_m, tiles_n);
    else
      hipLaunchKernelGGL((gemm_bf16_mid_kernel<A_KM, B_KM, KIND, TX, decltype(ACT)::value, 2>), grid, block, 0, stream, p, tiles_m, tiles_n);
  });
  LT_LAUNCH_CHECK();
  return LT_OK;
}

}  // namespace

bool lt_gemm_mid_supported(const GemmProblem& p, int kind) {
  return p.nseg == 1 && p.sp.mode == SPARSE_NONE && p.variant == 0 && p.K[0] < (int64_t)1 << 30 &&
         lt_gemm_mfma_supported(p, kind) && dma_offsets_fit(p, kind);
}

int lt_launch_gemm_mid(const GemmProblem& p, int kind, int io_dtype, hipStream_t stream) {
  LT_REQUIRE(lt_gemm_mid_supported(p, kind), LT_ERR_UNSUPPORTED, "128 x 128 gemm does not take this problem");
  const bool b_km = p.B[0].kmajor;
  if (kind == EPI_STORE && !p.A[0].kmajor) return launch_mid<false, false, EPI_STORE, float>(p, stream);
  if (kind == EPI_STORE) return b_km ? launch_mid<true, true, EPI_STORE, float>(p, stream) : launch_mid<true, false, EPI_STORE, float>(p, stream);
  if (kind == EPI_ACT_FWD) return launch_mid<true, true, EPI_ACT_FWD, float>(p, stream);
  if (kind == EPI_ACT_BWD) return launch_mid<true, false, EPI_ACT_BWD, float>(p, stream);
  return io_dtype == LT_BF16 ? launch_mid<true, true, EPI_OUT, bf16>(p, stream) : launch_mid<true, true, EPI_OUT, float>(p, stream);
}

int lt_launch_gemm_mid_group(const GemmProblem* problems, int n, hipStream_t stream) {
  LT_REQUIRE(n > 0 && n <= LT_MID_GROUP_MAX, LT_ERR_BAD_ARG, "128 x 128 gemms in one launch: %d of them", n);
  MidGroup g;
  memset(&g, 0, sizeof(g));
  unsigned total = 0;
  double flops = 0.0;
  for (int j = 0; j < LT_MID_GROUP_MAX; j++) {
    g.first[j] = total;
    if (j >= n) continue;
    const GemmProblem& p = problems[j];
    LT_REQUIRE(!p.A[0].kmajor && !p.B[0].kmajor && lt_gemm_mid_supported(p, EPI_STORE), LT_ERR_UNSUPPORTED,
               "128 x 128 gemms in one launch: product %d is none of them", j);
    g.p[j] = p;
    g.tiles_m[j] = (int)((p.M + MID - 1) / MID);
    g.tiles_n[j] = (int)((p.N + MID - 1) / MID);
    total += (unsigned)(g.tiles_m[j] * g.tiles_n[j] * (p.ksplit > 1 ? p.ksplit : 1));
    flops += lt_gemm_flops(p, EPI_STORE);
  }
  for (int j = n; j < LT_MID_GROUP_MAX; j++) g.first[j] = total;
  LT_REQUIRE(total <= 256, LT_ERR_UNSUPPORTED, "128 x 128 gemms in one launch: %u workgroups", total);
  LtProfileScope scope("gemm_mid_tn_store", flops, 0.0, stream);
  hipLaunchKernelGGL(gemm_bf16_mid_group_kernel, dim3(total), dim3(256), 0, stream, g);
  LT_LAUNCH_CHECK();
  return LT_OK;
}
