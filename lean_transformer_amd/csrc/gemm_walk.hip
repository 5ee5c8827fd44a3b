// Block-sparse forward products and input gradients over 64 x 64 blocks (SparseWalk modes FWD / DX) on the matrix cores: a workgroup
// owns 256 tokens x one block column and walks that column's list, one 64-k block of both operands per step, the low-rank term's
// blocks behind it.  256 x 64 tiles in four wavefronts of 64 x 64; operands copied global -> LDS, epilogues of gemm_strips.h.
//
// What bounds it: a step moves 40 KiB into LDS (640 cycles of the CU's path to L2) and reads 64 KiB of it (512 cycles) for 512 cycles of
// matrix instructions, so the three have to run under each other; in a wide layer the gathers' traffic between L2 and memory, and the
// epilogues of the activation.  The list sits in registers (a lane an entry, read with v_readlane): no step waits for an index.  A
// grid of at most one workgroup per CU keeps four steps in LDS (160 KiB); a larger one two, and two workgroups share a CU, so that
// one's epilogue runs under the other's walk (four steps and one workgroup there: 20 - 40 % longer).  Measured, against tiles
// staged through registers one step ahead with the index read from memory in every step:
//   hidden 4096 -> 16384 gated, stretched butterfly, rank 128, T 4096: down-projection 124 us, 103; dh + dGeGLU 251, 240; du 203, 150
//   hidden 1024 -> 4096 gated, tiled butterfly, rank 64, T 4000: up-projection + GeGLU 79 us, 57; down 37, 26; dh 72, 54; du 57, 33
#include "gemm_mfma_kernels.h"
#include "gemm_staged.h"
#include "gemm_strips.h"

namespace {

constexpr int LISTED = 128;  // steps whose blocks are held in registers, two of them with an entry per lane, at a time

// PH == 2 (gated forward): gate block tn and the matching linear block tn + groups, walked one after the other into accumulators of
// their own and paired in the epilogue.
template <int SP, int KIND, typename TX, int ACT, int PH, int STAGES>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(STAGES == 2 ? 2 : 1)))
void gemm_walk_kernel(GemmProblem p, int tiles_m, int groups) {
  static_assert(SP == SPARSE_FWD || SP == SPARSE_DX, "walks");
  static_assert(PH == 1 || (PH == 2 && SP == SPARSE_FWD && KIND == EPI_ACT_FWD), "two phases: gated forward");
  static_assert(STAGES == 2 || STAGES == 4, "stages");
  constexpr int A_ELEMS = 256 * 64, B_ELEMS = 64 * 64, A_LOADS = 8, B_LOADS = 2;
  constexpr uint32_t RECORDS = DmaOperand<true>::RECORDS, OUTSIDE = DmaOperand<true>::OUTSIDE;
  constexpr bool B_KM = SP == SPARSE_FWD;
  // an array per stage and operand: the compiler can prove that copies and reads do not alias
  __shared__ __attribute__((aligned(1024))) bf16 a0[A_ELEMS];
  __shared__ __attribute__((aligned(1024))) bf16 a1[A_ELEMS];
  __shared__ __attribute__((aligned(1024))) bf16 a2[A_ELEMS];
  __shared__ __attribute__((aligned(1024))) bf16 a3[A_ELEMS];
  __shared__ __attribute__((aligned(1024))) bf16 b0[B_ELEMS];
  __shared__ __attribute__((aligned(1024))) bf16 b1[B_ELEMS];
  __shared__ __attribute__((aligned(1024))) bf16 b2[B_ELEMS];
  __shared__ __attribute__((aligned(1024))) bf16 b3[B_ELEMS];
  auto a_buf = [&](auto S) -> bf16* {
    constexpr int s = decltype(S)::value % STAGES;
    return s == 0 ? a0 : s == 1 ? a1 : s == 2 ? a2 : a3;
  };
  auto b_buf = [&](auto S) -> bf16* {
    constexpr int s = decltype(S)::value % STAGES;
    return s == 0 ? b0 : s == 1 ? b1 : s == 2 ? b2 : b3;
  };
#ifdef LT_TILE_TIMING
  unsigned long long* const tile_stamps = p.tile_stamps ? p.tile_stamps + (size_t)blockIdx.x * 8 : nullptr;
#endif
  LT_TILE_STAMP(0);
  LT_TILE_STAMP_REALTIME(4);

  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  // The workgroups of one token tile gather column blocks of the same 256 activation rows (a few MiB that stay in the XCD's L2)
  // while every block column has a weight list of its own, so one XCD's concurrent workgroups (workgroup i runs on XCD i % 8) take
  // one token tile and consecutive block columns.
  const int num_pid = tiles_m * groups;
  const int pid = lt_xcd_order((int)blockIdx.x, num_pid);
  const int tm = pid / groups, tn = pid % groups;
  const int64_t m0 = (int64_t)tm * 256, n0 = (int64_t)tn * 64;

  const SparseWalk& sp = p.sp;
  const int steps = SP == SPARSE_FWD ? sp.blocks_per_out : sp.blocks_per_in;  // the list
  const int low_k = p.nseg > 1 ? (int)p.K[1] : 0;                             // the low-rank term's reduction
  const int total = steps + (low_k + 63) / 64;
  const int padded = (total + STAGES - 1) / STAGES * STAGES;  // steps a phase takes (those past `total` copy zeros, unread)

  // Entry of the list taken at step t (SparseWalk::walk_run).  Token tiles start an eighth of the list apart: the rows of an activation
  // block lie a power of two apart, on few memory channels, and the tiles of one block column would ask for theirs at the same
  // time.  hidden 4096, T 4096, all from the first entry against this: down-projection 108 us, 103; dh 248, 240; du 154, 150; both products
  // of a tiled butterfly's forward pass 434, 404.  The price: a row's terms are added in an order that depends on the tile it is in, so
  // that equal rows may differ in their last bits from tile to tile (the dense kernels' staggered walks do the same).  Starts that go
  // by the block column instead would not, and measured 459 for the 404.
  const int first = (tm & 7) * steps / 8;
  auto walk_entry = [&](int t) __attribute__((always_inline)) {
    t += first;
    if (t >= steps) t -= steps;
    if (sp.walk_run <= 1) return t;
    const int runs = steps / sp.walk_run;
    return (t % runs) * sp.walk_run + t / runs;
  };
  // Steps g of the workgroup: phase g / padded, step g % padded of it.  In registers for steps base .. base + 127: the activation
  // column block and the weight block; of a low-rank step -1 - (its number in the term) and the phase (past the end: a number whose
  // k are all past the term's reduction).
  int base = 0, a_lo, a_hi, b_lo, b_hi;
  auto entry_of = [&](int g, int& a_block, int& b_block) __attribute__((always_inline)) {
    const int ph = PH == 2 && g >= padded ? 1 : 0, t = g - ph * padded, e = walk_entry(min(t, steps - 1));
    if constexpr (SP == SPARSE_FWD) {
      b_block = sp.forward_indices[(int64_t)(tn + ph * groups) * steps + e];
      a_block = b_block / sp.blocks_per_in;
    } else {
      b_block = tn * steps + e;
      a_block = (int)sp.backward_indices[b_block];
    }
    if (t >= steps) {
      a_block = -1 - (t < total ? t - steps : (low_k + 63) / 64);
      b_block = ph;
    }
  };
  auto load_list = [&](int from) __attribute__((always_inline)) {
    base = from;
    entry_of(from + lane, a_lo, b_lo);
    entry_of(from + 64 + lane, a_hi, b_hi);
  };
  load_list(0);

  // Copies: row and byte offset inside a row's 128 bytes of this lane's 16-byte pieces; rows past M repeat the last one (their results
  // are not stored).  The two steps of a copy's swizzle alternate, so there are two offsets per operand at most.
  uint32_t a_row[A_LOADS], b_row[B_LOADS], a_piece[2], b_piece[2];
  int a_k[2], b_k[B_LOADS];  // k of the pieces inside the step
#pragma unroll
  for (int j = 0; j < A_LOADS; j++) {
    const int q = (wave * A_LOADS + j) * 64 + lane, row = q >> 3, c = (q & 7) ^ swz_km(row);
    a_row[j] = (uint32_t)min((int64_t)row, p.M - 1 - m0);
    if (j < 2) {
      a_piece[j] = (uint32_t)c * 16;
      a_k[j] = c * 8;
    }
  }
#pragma unroll
  for (int j = 0; j < B_LOADS; j++) {
    const int q = (wave * B_LOADS + j) * 64 + lane, row = q >> 3, c = (q & 7) ^ (B_KM ? swz_km(row) : swz_mn_cols<64>(row));
    b_row[j] = (uint32_t)row;
    b_piece[j] = (uint32_t)c * 16;
    b_k[j] = B_KM ? c * 8 : row;
  }
  const int64_t lda1 = low_k ? p.A[1].ld : 0, ldb1 = low_k ? p.B[1].ld : 0;
  const char* const a_base = reinterpret_cast<const char*>(sp.act) + m0 * sp.ld_act * 2;
  const char* const a_base1 = reinterpret_cast<const char*>(p.A[1].ptr) + m0 * lda1 * 2;
  const char* const b_base = reinterpret_cast<const char*>(sp.weight);
  const char* const b_base1 = reinterpret_cast<const char*>(p.B[1].ptr) + (B_KM ? n0 * ldb1 * 2 : n0 * 2);
  const int64_t phase_bytes = B_KM ? p.N * ldb1 * 2 : 0, term_bytes = B_KM ? 128 : 128 * ldb1;  // per phase and per step of the low-rank term
  // Copies J0 .. J1 - 1 (A's eight, then B's two) of step g into the buffers of position S; past the last step, zeros.  Without a branch
  // (the kinds of steps differ in scalars only): one would keep the copies from spreading between the matrix instructions.
  auto copy = [&](auto S, int g, auto J0_, auto J1_) __attribute__((always_inline)) {
    constexpr int j0 = decltype(J0_)::value, j1 = decltype(J1_)::value;
    const int l = g - base, h = (l << 25) >> 31;  // (all ones in the second register)
    auto entry = [&](int lo, int hi) __attribute__((always_inline)) {
      const int x = __builtin_amdgcn_readlane(lo, l & 63), y = __builtin_amdgcn_readlane(hi, l & 63);
      return x ^ ((x ^ y) & h);
    };
    const int ea = entry(a_lo, a_hi), eb = entry(b_lo, b_hi);
    const int low = ea >> 31, unit = ea ^ low;  // all ones for a low-rank step; its number, or the column block
    auto either = [&](int64_t list, int64_t term) __attribute__((always_inline)) { return list ^ ((list ^ term) & (int64_t)low); };
    const int limit = 64 + ((low_k - 64 - unit * 64) & low);  // of the step's 64 k
    auto outside = [&](int k) __attribute__((always_inline)) { return (uint32_t)((limit - 1 - k) >> 31) & OUTSIDE; };
    if constexpr (j0 < A_LOADS) {
      const char* const a = reinterpret_cast<const char*>(either((int64_t)a_base, (int64_t)a_base1) + (int64_t)unit * 128);
      const uint32_t pitch = (uint32_t)either(sp.ld_act, lda1) * 2;
      const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(a), 0, (int)RECORDS, 0x00020000);
      const uint32_t mask[2] = {outside(a_k[0]), outside(a_k[1])};
#pragma unroll
      for (int j = j0; j < (j1 < A_LOADS ? j1 : A_LOADS); j++) {
        const uint32_t o = max(__umul24(a_row[j], pitch) + a_piece[j & 1], mask[j & 1]);
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (__attribute__((address_space(3))) void*)(a_buf(S) + (wave * A_LOADS + j) * 512), 16,
                                                 (int)o, 0, 0, 0);
      }
    }
    if constexpr (j1 > A_LOADS) {
      const char* const b = reinterpret_cast<const char*>(either((int64_t)b_base, (int64_t)b_base1) + (int64_t)eb * either(8192, phase_bytes) +
                                                          (int64_t)(unit & low) * term_bytes);
      const uint32_t pitch = (uint32_t)either(64, ldb1) * 2;
      const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(b), 0, (int)RECORDS, 0x00020000);
#pragma unroll
      for (int j = (j0 > A_LOADS ? j0 - A_LOADS : 0); j < j1 - A_LOADS; j++) {
        const uint32_t o = max(__umul24(b_row[j], pitch) + b_piece[j], outside(b_k[j]));
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (__attribute__((address_space(3))) void*)(b_buf(S) + (wave * B_LOADS + j) * 512), 16,
                                                 (int)o, 0, 0, 0);
      }
    }
  };

  f32x16 acc[2][2], acc2[2][2];  // (acc2: the linear block's)
#pragma unroll
  for (int i = 0; i < 2; i++)
#pragma unroll
    for (int j = 0; j < 2; j++)
#pragma unroll
      for (int r = 0; r < 16; r++) acc[i][j][r] = acc2[i][j][r] = 0.f;
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
      const bf16* src = &tile[kr * 64 + ((((col >> 3) ^ swz_mn_cols<64>(kr)) << 3) | (col & 7))];
      u.h[s] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)(src));
    }
    return u.v;
  };
  bf16x8 fa[2][2], fb[2][2];
  auto load = [&](auto S, auto KK, auto F) __attribute__((always_inline)) {
    constexpr int kk = decltype(KK)::value, f = decltype(F)::value;
#pragma unroll
    for (int i = 0; i < 2; i++) {
      fa[f][i] = frag_km(a_buf(S), wave * 64 + i * 32, kk);
      if constexpr (B_KM) fb[f][i] = frag_km(b_buf(S), i * 32, kk);
      else fb[f][i] = frag_mn(b_buf(S), i * 32, kk);
    }
  };
  LT_TILE_STAMP(1);
  using Loop = StagedLoop<STAGES, A_LOADS + B_LOADS, 2 + 2 * (B_KM ? 1 : 2)>;
  auto multiply_into = [&](f32x16 (&c)[2][2], auto F) __attribute__((always_inline)) {
    constexpr int f = decltype(F)::value;
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
      for (int j = 0; j < 2; j++) c[i][j] = LT_MFMA_32X32X16(fa[f][i], fb[f][j], c[i][j]);
  };
  // steps from .. from + count - 1, LISTED at a time; the pipeline runs on where the registers hold them all
  const bool one_list = PH * padded <= LISTED;
  auto walk = [&](int from, int count, f32x16 (&c)[2][2]) __attribute__((always_inline)) {
    for (int g = from; g < from + count; g += LISTED) {
      if (g > 0 && !one_list) {
        wait_copies_and_barrier<0>();
        load_list(g);
      }
      if (g == 0 || !one_list) Loop::start(g, copy, load);
      Loop::run(g, min(LISTED, from + count - g), copy, load, [&](auto F) __attribute__((always_inline)) { multiply_into(c, F); });
    }
  };
  walk(0, PH == 2 ? padded : total, acc);
  if constexpr (PH == 2) walk(padded, total, acc2);
  wait_copies_and_barrier<0>();
  LT_TILE_STAMP(2);

  float* const stage = reinterpret_cast<float*>(a0) + wave * 2048;
  if constexpr (PH == 2) {
    lt_static_for<2>([&](auto J) __attribute__((always_inline)) {
      constexpr int j = decltype(J)::value;
      const f32x16 pair[2][2] = {{acc[0][j], acc2[0][j]}, {acc[1][j], acc2[1][j]}};
      strip_epilogue<KIND, TX, ACT, true>(pair, p, 0, stage, m0 + wave * 64, n0 + j * 32, lane);
    });
  } else {
    strip_epilogue<KIND, TX, ACT, false>(acc, p, 0, stage, m0 + wave * 64, n0, lane);
  }
  LT_TILE_STAMP(3);
  LT_TILE_STAMP_REALTIME(5);
}

template <int SP, int KIND, typename TX, int PH> int launch_walk(const GemmProblem& problem, hipStream_t stream) {
  GemmProblem p = problem;
#ifdef LT_TILE_TIMING
  // launch number i of the process writes region i % 4 (8192 workgroups each) of its own buffer
  if (const char* e = getenv("LT_TILE_TIMING_BUFFER_SPARSE"))
    p.tile_stamps = (unsigned long long*)(strtoull(e, nullptr, 0) + (size_t)(lt_tile_timing_launch_counter()++ % 4) * 8192 * 64);
#endif
  const int tiles_m = (int)((p.M + 255) / 256), groups = (int)(p.N / 64);
  const dim3 grid((unsigned)(tiles_m * groups)), block(256);
  with_activation<KIND>(p, [&](auto ACT) {
    if (tiles_m * groups <= 256)
      hipLaunchKernelGGL((gemm_walk_kernel<SP, KIND, TX, decltype(ACT)::value, PH, 4>), grid, block, 0, stream, p, tiles_m, groups);
    else
      hipLaunchKernelGGL((gemm_walk_kernel<SP, KIND, TX, decltype(ACT)::value, PH, 2>), grid, block, 0, stream, p, tiles_m, groups);
  });
  LT_LAUNCH_CHECK();
  return LT_OK;
}

}  // namespace

int lt_launch_gemm_walk(const GemmProblem& p, int kind, int io_dtype, hipStream_t stream) {
  if (p.sp.mode == SPARSE_DX) {
    if (kind == EPI_STORE) return launch_walk<SPARSE_DX, EPI_STORE, float, 1>(p, stream);
    if (kind == EPI_ACT_BWD) return launch_walk<SPARSE_DX, EPI_ACT_BWD, float, 1>(p, stream);
  } else if (p.sp.mode == SPARSE_FWD) {
    if (kind == EPI_STORE) return launch_walk<SPARSE_FWD, EPI_STORE, float, 1>(p, stream);
    // (gated: p.N counts the gate columns; one workgroup per token tile and gate block)
    if (kind == EPI_ACT_FWD && p.epi.gated) return launch_walk<SPARSE_FWD, EPI_ACT_FWD, float, 2>(p, stream);
    if (kind == EPI_ACT_FWD) return launch_walk<SPARSE_FWD, EPI_ACT_FWD, float, 1>(p, stream);
    if (kind == EPI_OUT && io_dtype == LT_BF16) return launch_walk<SPARSE_FWD, EPI_OUT, bf16, 1>(p, stream);
    if (kind == EPI_OUT) return launch_walk<SPARSE_FWD, EPI_OUT, float, 1>(p, stream);
  }
  LT_FAIL(LT_ERR_UNSUPPORTED, "block-sparse walk: epilogue %d does not go with mode %d", kind, p.sp.mode);
}
