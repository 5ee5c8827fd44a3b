// Any-shape GEMM with fused epilogues: fp32 or 16-bit operands with arbitrary leading dimensions and either operand
// transposed, 16-bit matrix-core arithmetic with fp32 accumulation.  This is the kernel of the fp32 path, of every shape the
// tiled 16-bit kernel does not take (sizes that are not multiples of 8), and -- with a SparseWalk -- of the block-sparse matmul
// for any block size: a group of workgroups (blockIdx.y) then walks the index table of one output block / input block / weight
// block and treats each active block as one k-segment.
//
// fp32 operands.  The fp32 matrix instruction runs at 1/16 of the 16-bit one's rate.  A float has 24 significant bits, a bfloat16
// 8 and the same exponent range, so every operand element is split without error into three bfloat16 planes, x = x1 + x2 + x3:
// x1 is x truncated, x2 the remainder (16 bits, exact in fp32) rounded, x3 the rest (8 bits, exact).  A product of two floats
// is nine products of planes, each of them exact in fp32; the six with a weight of 2^-16 or more are accumulated
// (x1 y1, x1 y2, x2 y1, x2 y2, x1 y3, x3 y1), and all nine where the whole reduction is one step.  What is left out, x2 y3 + x3 y2 +
// x3 y3, is at most 2^-7 2^-16 2 = 2^-22 of |x y| and 2^-24.5 of it on average with random sign, the size of the one rounding that
// every fp32 accumulation makes, and the matrix unit adds 16 products per such rounding instead of 2.  x1 y1 has accumulators of its
// own: added to the whole sum, 16 products of 2^-16 are less than half a unit in its last place once a reduction of one sign has
// a few thousand terms, and are lost every time (|x| |y| of normal numbers over 8192: 89 x 2^-24 off, 24 with the fp32 instruction).
// Below 2^-110 an element's last plane is subnormal and loses bits below 2^-133.  The 16-bit instruction rounds
// what it aligns away towards minus infinity (a bias of 0.1 - 0.2 units in the last place per instruction, measured), which
// sums over many rows of a result would collect (a bias gradient is one over all tokens); odd rows of A are therefore negated
// on the way in and odd rows of the result on the way out, so that the bias alternates.
// An infinity has no such planes (inf - inf) and gives NaN; an element that comes out as NaN is therefore computed again, in fp32
// arithmetic from the operands in memory, as the epilogue takes it up (a NaN among its operands ends that where it is met).
// What bounds it: at 4096^3 a full round of workgroups runs at 1.2 PFLOP/s of bfloat16 products, what the tiled 16-bit kernel
// reaches on the same data (the clock under load); smaller products lose to a last round that is not full and to the start and
// end of a tile.  4096^3: 1411 us with the fp32 instruction, 752 with one set of accumulators, 763 with two; a training step of T = 4096,
// hidden 768: 2263 us, 1150, 1266; 2-norm error of 4096^3 against float64 1.15e-6, 1.01e-6, 0.39e-6.  16-bit operands, 4096^3: 1591 us, 221.
//
// Work decomposition: 256 threads = 4 wavefronts in a 2 x 2 grid over a (64 FM) x 128 output tile; each wavefront owns FM x 2
// MFMA blocks of 32 x 32.  Operand tiles of BK k-steps are staged in LDS as 16-byte pieces of 8 consecutive k, [plane][k / 8][row],
// which is what a lane of the matrix instruction reads; a piece is fetched by one thread (two 16-byte loads of a k-major operand,
// eight coalesced loads of an mn-major one), split in registers and written with one 16-byte LDS write per plane.  The fetches
// of the next step are in flight (in registers) while the matrix cores work on the current one; two LDS buffers, one barrier
// per step.
#include <type_traits>

#include "lt_gemm.h"

namespace {

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bfloat8;
typedef __attribute__((__vector_size__(2 * sizeof(float)))) float f32x2;
typedef __attribute__((__vector_size__(2 * sizeof(__bf16)))) __bf16 bfloat2;

// how operands of type TI go to the matrix cores: planes per element, k per LDS stage, the fragment type and instruction
template <typename TI> struct Operand {  // 16-bit: as they are
  static constexpr int PLANES = 1, BK = 32, PRODUCTS = 1;
  typedef bf16x8 Frag;
  static __device__ __forceinline__ f32x16 mfma(Frag a, Frag b, f32x16 c) { return LT_MFMA_32X32X16(a, b, c); }
  static constexpr int A_PLANE[1] = {0}, B_PLANE[1] = {0};
};
template <> struct Operand<float> {
  static constexpr int PLANES = 3, BK = 16, PRODUCTS = 9;
  typedef bfloat8 Frag;
  static __device__ __forceinline__ f32x16 mfma(Frag a, Frag b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
  }
  // smallest first; FEW: the first three belong to short reductions only
  static constexpr int A_PLANE[9] = {2, 1, 2, 2, 0, 1, 1, 0, 0}, B_PLANE[9] = {2, 2, 1, 0, 2, 1, 0, 1, 0}, FEW = 3;
};

// 8 consecutive k of one row, as fetched
template <typename TI> struct Piece {
  TI v[8];
};

// piece -> its planes as 16-byte words; flip (fp32): sign bit to flip in every element
__device__ __forceinline__ void split_piece(const Piece<bf16>& f, uint32_t, lt_u32x4 (&out)[1]) {
  union { lt_u32x4 u; bf16 h[8]; } t;
#pragma unroll
  for (int e = 0; e < 8; e++) t.h[e] = f.v[e];
  out[0] = t.u;
}
__device__ __forceinline__ void split_piece(const Piece<float>& f, uint32_t flip, lt_u32x4 (&out)[3]) {
#pragma unroll
  for (int e = 0; e < 4; e++) {
    const uint32_t b0 = __builtin_bit_cast(uint32_t, f.v[2 * e]) ^ flip, b1 = __builtin_bit_cast(uint32_t, f.v[2 * e + 1]) ^ flip;
    out[0][e] = __builtin_amdgcn_perm(b1, b0, 0x07060302u);  // the upper halves, element 2 e in the lower 16 bits
    const float r0 = __builtin_bit_cast(float, b0) - __builtin_bit_cast(float, b0 & 0xffff0000u);
    const float r1 = __builtin_bit_cast(float, b1) - __builtin_bit_cast(float, b1 & 0xffff0000u);
    const uint32_t second = __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{r0, r1}, bfloat2));
    out[1][e] = second;
    const float s0 = r0 - __builtin_bit_cast(float, second << 16), s1 = r1 - __builtin_bit_cast(float, second & 0xffff0000u);
    out[2][e] = __builtin_amdgcn_perm(__builtin_bit_cast(uint32_t, s1), __builtin_bit_cast(uint32_t, s0), 0x07060302u);
  }
}

template <typename TI> struct Segment {
  const TI* A;
  const TI* B;
  int64_t lda, ldb, K;
};

// up to 4 consecutive elements p[0 .. count), all of them with one access where `vec` says that alignment allows it
template <typename T> __device__ __forceinline__ void load_few(const T* p, bool vec, int count, float (&v)[4]) {
  if (vec) {
    load4(p, v);
  } else {
#pragma unroll
    for (int e = 0; e < 4; e++) v[e] = e < count ? to_f32(p[e]) : 0.f;
  }
}
template <typename T> __device__ __forceinline__ void store_few(T* p, bool vec, int count, const float (&v)[4]) {
  if (vec) {
    store4(p, v);
  } else {
#pragma unroll
    for (int e = 0; e < 4; e++)
      if (e < count) p[e] = from_f32<T>(v[e]);
  }
}

// body(row, in0, in1) for each of N rows, rolled: the rows' inputs move up one place per turn (registers cannot be indexed)
template <int N, typename F> __device__ __forceinline__ void lt_rolled_rows(F&& body, float (&in0)[N][4], float (&in1)[N][4]) {
#pragma unroll 1
  for (int it = 0; it < N; it++) {
    body(it, in0[0], in1[0]);
#pragma unroll
    for (int k = 0; k + 1 < N; k++)
#pragma unroll
      for (int e = 0; e < 4; e++) {
        in0[k][e] = in0[k + 1][e];
        in1[k][e] = in1[k + 1][e];
      }
  }
}

// A_KM, B_KM: layout of the operands (of every k-segment).  A block-sparse walk has the layout of its mode.
template <typename TI, bool A_KM, bool B_KM, int KIND, typename TC, typename TX, int FM>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu((FM == 1 ? 4 : 3) - (sizeof(TI) == 4)))) void gemm_generic_kernel(GemmProblem p, int tiles_m, int tiles_n) {
  typedef Operand<TI> Op;
  typedef typename Op::Frag Frag;
  constexpr int BM = 64 * FM, BN = 128, BK = Op::BK, CH = BK / 8, PLANES = Op::PLANES;
  // 16-byte pieces per (plane, k chunk): 4 more than rows, so that the chunks of one row land on different banks
  constexpr int A_ROWS = BM + 4, B_ROWS = BN + 4;
  constexpr int A_WORDS = PLANES * CH * A_ROWS, B_WORDS = PLANES * CH * B_ROWS;  // pieces per buffer
  constexpr int STAGE_LD = 64 + 8;  // floats per staged row of the epilogue: 4 rows apart land 32 banks apart
  constexpr int LOOP_BYTES = 2 * (A_WORDS + B_WORDS) * 16, STAGE_BYTES = 4 * 32 * STAGE_LD * 4;
  __shared__ __attribute__((aligned(16))) char smem[LOOP_BYTES > STAGE_BYTES ? LOOP_BYTES : STAGE_BYTES];
  lt_u32x4* const lds = reinterpret_cast<lt_u32x4*>(smem);
  auto a_tile = [&](int buf) { return lds + buf * A_WORDS; };
  auto b_tile = [&](int buf) { return lds + 2 * A_WORDS + buf * B_WORDS; };

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave >> 1, wn = wave & 1;
  const bool gated = (KIND == EPI_ACT_FWD) && p.epi.gated;
  // Tile: the hardware hands workgroup i to XCD i % 8; each XCD takes a contiguous range of tiles, 8 tile rows at a time, so that
  // the tiles it works on share few operand panels through its L2.
  int pid = blockIdx.x;
  const int num_pid = tiles_m * tiles_n;
  if ((num_pid & 7) == 0) pid = (pid & 7) * (num_pid >> 3) + (pid >> 3);
  const int in_group = 8 * tiles_n, first_m = pid / in_group * 8, group_m = min(tiles_m - first_m, 8);
  const int64_t m0 = (int64_t)(first_m + pid % in_group % group_m) * BM;
  // gated forward: a tile holds 64 gate columns and the 64 matching linear columns, split per wavefront so that one wavefront
  // owns both members of a pair: tile column c -> wavefront c / 64, MFMA block (c % 64) / 32 = half, offset c % 32
  const int64_t n0 = (int64_t)(pid % in_group / group_m) * (gated ? BN / 2 : BN);

  // ---- problem seen by this workgroup: dense, or one group of a block-sparse walk
  const SparseWalk& sp = p.sp;
  const int group = blockIdx.y;
  const int b = sp.block;
  int64_t M = p.M, N = p.N;  // bounds of the local tile coordinates
  int64_t n_off = 0;         // global column of local column 0 (epilogue indices)
  int nseg = p.nseg;
  EpiParams epi = p.epi;
  if (sp.mode == SPARSE_FWD) {
    N = b; n_off = (int64_t)group * b; nseg = sp.blocks_per_out + (p.nseg > 1);
  } else if (sp.mode == SPARSE_DX) {
    N = b; n_off = (int64_t)group * b; nseg = sp.blocks_per_in + (p.nseg > 1);
  } else if (sp.mode == SPARSE_DW) {
    M = b; N = b; nseg = 1;
    epi.out = reinterpret_cast<char*>(epi.out) + (int64_t)group * b * b * (epi.out_dtype == LT_F32 ? 4 : 2);
    epi.ldo = b;
  }
  if (m0 >= M || n0 >= N) return;  // whole workgroup

  auto segment = [&](int s) __attribute__((always_inline)) -> Segment<TI> {
    Segment<TI> g;
    if (sp.mode == SPARSE_NONE) {
      g.A = reinterpret_cast<const TI*>(p.A[s].ptr); g.lda = p.A[s].ld;
      g.B = reinterpret_cast<const TI*>(p.B[s].ptr); g.ldb = p.B[s].ld;
      g.K = p.K[s];
    } else if (sp.mode == SPARSE_FWD) {
      if (s < sp.blocks_per_out) {
        const int f = sp.forward_indices[(int64_t)group * sp.blocks_per_out + s];
        const int ib = f / sp.blocks_per_in;
        g.A = reinterpret_cast<const TI*>(sp.act) + (int64_t)ib * b; g.lda = sp.ld_act;
        g.B = reinterpret_cast<const TI*>(sp.weight) + (int64_t)f * b * b; g.ldb = b;
        g.K = b;
      } else {  // low-rank: hid [M, r] x second[out, r]^T restricted to this output block
        g.A = reinterpret_cast<const TI*>(p.A[1].ptr); g.lda = p.A[1].ld;
        g.B = reinterpret_cast<const TI*>(p.B[1].ptr) + n_off * p.B[1].ld; g.ldb = p.B[1].ld;
        g.K = p.K[1];
      }
    } else if (sp.mode == SPARSE_DX) {
      if (s < sp.blocks_per_in) {
        const int64_t ob = sp.backward_indices[(int64_t)group * sp.blocks_per_in + s];
        g.A = reinterpret_cast<const TI*>(sp.act) + ob * b; g.lda = sp.ld_act;
        // B(n = input column c, k = output row rho) = W4[ib, a, rho, c]: k strided by b
        g.B = reinterpret_cast<const TI*>(sp.weight) + ((int64_t)group * sp.blocks_per_in + s) * b * b; g.ldb = b;
       
        g.K = b;
      } else {  // low-rank: g_hid [M, r] x first[r, in] restricted to this input block
        g.A = reinterpret_cast<const TI*>(p.A[1].ptr); g.lda = p.A[1].ld;
        g.B = reinterpret_cast<const TI*>(p.B[1].ptr) + n_off; g.ldb = p.B[1].ld;
        g.K = p.K[1];
      }
    } else {  // SPARSE_DW: rows = output row rho of block ob, columns = input column c of block ib, reduce over tokens
      const int ib = group / sp.blocks_per_in;
      const int64_t ob = sp.backward_indices[group];
      g.A = reinterpret_cast<const TI*>(sp.act) + ob * b; g.lda = sp.ld_act;
      g.B = reinterpret_cast<const TI*>(sp.act2) + (int64_t)ib * b; g.ldb = sp.ld_act2;
      g.K = sp.tokens;
    }
    return g;
  };

  f32x16 acc[FM][2], rest[FM][2];  // rest (fp32): the products of planes below the first
#pragma unroll
  for (int i = 0; i < FM; i++)
#pragma unroll
    for (int j = 0; j < 2; j++)
#pragma unroll
      for (int r = 0; r < 16; r++) acc[i][j][r] = rest[i][j][r] = 0.f;

  // ---- main loop.  Step t multiplies LDS buffer t & 1 while the fetches of step t + 2 are in flight into register set t & 1; then the
  //      pieces of step t + 1 (set (t + 1) & 1) are split and written to the other buffer.  The two to four workgroups of a CU
  //      overlap each other's matrix and vector work: placing the split between the matrix instructions of the same wavefront
  //      measured the same.
  constexpr int A_PIECES = (BM * CH + 255) / 256, B_PIECES = BN * CH / 256;  // per thread and step
  static_assert(BN * CH % 256 == 0 && (BM * CH % 256 == 0 || BM * CH == 128), "pieces divide over the threads");
  constexpr bool A_ALL = BM * CH % 256 == 0;  // every thread has pieces of A
  // the cursor: segment and k of the next step to be fetched
  int seg = 0;
  Segment<TI> g = segment(0);
  int64_t k0 = 0, slice_k0 = 0, slice_k1 = g.K;
  if (sp.mode == SPARSE_NONE && p.ksplit > 1) {
    // split reduction (one k-segment, EPI_STORE): slice blockIdx.y walks a whole number of k-steps and stores fp32 partial
    // sums at epi.out + slice * split_stride
    const int64_t steps = (g.K + BK - 1) / BK, per = (steps + p.ksplit - 1) / p.ksplit * BK;
    k0 = min(g.K, (int64_t)blockIdx.y * per);
    g.K = min(g.K, k0 + per);
    slice_k0 = k0;
    slice_k1 = g.K;
    epi.out = reinterpret_cast<float*>(epi.out) + (int64_t)blockIdx.y * p.split_stride;
  }
  int total = 0;  // steps (an empty slice: one step of zeros)
  if (sp.mode == SPARSE_NONE) {
    total = max(1, (int)((g.K - k0 + BK - 1) / BK));
    if (nseg > 1) total += (int)((p.K[1] + BK - 1) / BK);
  } else if (sp.mode == SPARSE_DW) {
    total = (int)((g.K + BK - 1) / BK);
  } else {
    total = (nseg - (p.nseg > 1)) * ((b + BK - 1) / BK) + (p.nseg > 1 ? (int)((p.K[1] + BK - 1) / BK) : 0);
  }

  // Piece i of this thread: a k-major operand's neighbouring threads take the chunks of one row (its address is the thread's own),
  // an mn-major one's neighbouring rows of one chunk (the chunk is the wavefront's: its eight addresses are a wavefront-uniform
  // base plus the row)
  const int uwave = __builtin_amdgcn_readfirstlane(wave);
  auto a_row = [&](int i) { return A_KM ? (tid + i * 256) / CH : (tid + i * 256) % BM; };
  auto a_chunk = [&](int i) { return A_KM ? tid % CH : (uwave * 64 + i * 256) / BM; };
  auto b_row = [&](int i) { return B_KM ? (tid + i * 256) / CH : (tid + i * 256) % BN; };
  auto b_chunk = [&](int i) { return B_KM ? tid % CH : (uwave * 64 + i * 256) / BN; };
  auto a_mine = [&](int i) { return A_ALL || tid + i * 256 < BM * CH; };
  const TI* pa[A_PIECES];   // k-major: element chunk * 8 of this thread's row in the step at the cursor
  const TI* pb[B_PIECES];
  uint32_t ra[A_PIECES], rb[B_PIECES];  // mn-major: this thread's row
#pragma unroll
  for (int i = 0; i < A_PIECES; i++) ra[i] = (uint32_t)min(m0 + a_row(i), M - 1);  // rows past M are never stored
  auto b_global = [&](int i) -> int64_t {
    const int c = b_row(i);
    return gated ? ((c >> 5) & 1) * N + min(n0 + (c >> 6) * 32 + (c & 31), N - 1) : min(n0 + c, N - 1);
  };
#pragma unroll
  for (int i = 0; i < B_PIECES; i++) rb[i] = (uint32_t)b_global(i);
  auto start_segment = [&]() {
#pragma unroll
    for (int i = 0; i < A_PIECES; i++) pa[i] = A_KM ? g.A + (int64_t)ra[i] * g.lda + k0 + a_chunk(i) * 8 : nullptr;
#pragma unroll
    for (int i = 0; i < B_PIECES; i++) pb[i] = B_KM ? g.B + (int64_t)rb[i] * g.ldb + k0 + b_chunk(i) * 8 : nullptr;
  };
  constexpr int ALIGN = 16 / sizeof(TI) - 1;  // elements per 16 bytes, less one
  auto vectors = [&]() {  // whether the k-major pieces of this segment can be fetched 16 bytes at a time
    return (!A_KM || ((reinterpret_cast<uintptr_t>(g.A) & 15) == 0 && (g.lda & ALIGN) == 0)) &&
           (!B_KM || ((reinterpret_cast<uintptr_t>(g.B) & 15) == 0 && (g.ldb & ALIGN) == 0));
  };
  // one piece; WHOLE: all 8 elements exist and a k-major piece is aligned; else zeros past the end of the reduction
  auto fetch_piece = [&](auto whole, auto km, const TI* base, const TI* mine, int64_t ld, uint32_t row, int chunk, Piece<TI>& f) {
    if constexpr (decltype(km)::value) {
      if constexpr (decltype(whole)::value && sizeof(TI) == 4) {
        const float4 lo = *reinterpret_cast<const float4*>(mine), hi = *reinterpret_cast<const float4*>(mine + 4);
        f.v[0] = lo.x; f.v[1] = lo.y; f.v[2] = lo.z; f.v[3] = lo.w;
        f.v[4] = hi.x; f.v[5] = hi.y; f.v[6] = hi.z; f.v[7] = hi.w;
      } else if constexpr (decltype(whole)::value) {
        union { uint4 u; TI h[8]; } t;
        t.u = *reinterpret_cast<const uint4*>(mine);
#pragma unroll
        for (int e = 0; e < 8; e++) f.v[e] = t.h[e];
      } else {
#pragma unroll
        for (int e = 0; e < 8; e++) f.v[e] = k0 + chunk * 8 + e < g.K ? mine[e] : from_f32<TI>(0.f);
      }
    } else {
#pragma unroll
      for (int e = 0; e < 8; e++) {
        const int64_t k = k0 + chunk * 8 + e;
        if (decltype(whole)::value || k < g.K) f.v[e] = (base + k * ld)[row];
        else f.v[e] = from_f32<TI>(0.f);
      }
    }
  };
  using Whole = std::true_type;
  using Ragged = std::false_type;
  Piece<TI> fa[2][A_PIECES], fb[2][B_PIECES];
  // fetches the step at the cursor into register set S and moves the cursor on by BK (not into the next segment)
  auto fetch = [&](auto whole, auto S) {
    constexpr int set = decltype(S)::value;
#pragma unroll
    for (int i = 0; i < A_PIECES; i++) {
      if (a_mine(i)) fetch_piece(whole, std::integral_constant<bool, A_KM>{}, g.A, pa[i], g.lda, ra[i], a_chunk(i), fa[set][i]);
      pa[i] += BK;
    }
#pragma unroll
    for (int i = 0; i < B_PIECES; i++) {
      fetch_piece(whole, std::integral_constant<bool, B_KM>{}, g.B, pb[i], g.ldb, rb[i], b_chunk(i), fb[set][i]);
      pb[i] += BK;
    }
    k0 += BK;
  };
  auto next_segment = [&]() {
    if (k0 >= g.K && seg + 1 < nseg) {
      g = segment(++seg);
      k0 = 0;
      start_segment();
    }
  };
  // pieces of register set S -> LDS buffer `buf`
  auto stash = [&](auto S, int buf) {
    constexpr int set = decltype(S)::value;
    lt_u32x4* const ta = a_tile(buf);
    lt_u32x4* const tb = b_tile(buf);
#pragma unroll
    for (int i = 0; i < A_PIECES; i++) {
      lt_u32x4 w[PLANES];
      split_piece(fa[set][i], (uint32_t)a_row(i) << 31, w);
#pragma unroll
      for (int q = 0; q < PLANES; q++)
        if (a_mine(i)) ta[(q * CH + a_chunk(i)) * A_ROWS + a_row(i)] = w[q];
    }
#pragma unroll
    for (int i = 0; i < B_PIECES; i++) {
      lt_u32x4 w[PLANES];
      split_piece(fb[set][i], 0u, w);
#pragma unroll
      for (int q = 0; q < PLANES; q++) tb[(q * CH + b_chunk(i)) * B_ROWS + b_row(i)] = w[q];
    }
  };
  // tail (fp32): the three smallest products of planes instead of the six others
  auto multiply = [&](auto tail, int buf) {
    const lt_u32x4* const ta = a_tile(buf);
    const lt_u32x4* const tb = b_tile(buf);
#pragma unroll
    for (int kk = 0; kk < BK / 16; kk++) {
      const int chunk = kk * 2 + (lane >> 5);
      Frag a[FM][PLANES], bb[2][PLANES];
#pragma unroll
      for (int q = 0; q < PLANES; q++) {
#pragma unroll
        for (int i = 0; i < FM; i++)
          a[i][q] = __builtin_bit_cast(Frag, ta[(q * CH + chunk) * A_ROWS + wm * 32 * FM + i * 32 + (lane & 31)]);
#pragma unroll
        for (int j = 0; j < 2; j++)
          bb[j][q] = __builtin_bit_cast(Frag, tb[(q * CH + chunk) * B_ROWS + wn * 64 + j * 32 + (lane & 31)]);
      }
      if constexpr (PLANES == 1) {
#pragma unroll
        for (int i = 0; i < FM; i++)
#pragma unroll
          for (int j = 0; j < 2; j++) acc[i][j] = Op::mfma(a[i][0], bb[j][0], acc[i][j]);
      } else {
        constexpr bool TAIL = decltype(tail)::value;
        constexpr int FIRST = TAIL ? 0 : Op::FEW, LAST = TAIL ? Op::FEW : Op::PRODUCTS - 1;
#pragma unroll
        for (int t = FIRST; t < LAST; t++)
#pragma unroll
          for (int i = 0; i < FM; i++)
#pragma unroll
            for (int j = 0; j < 2; j++) rest[i][j] = Op::mfma(a[i][Op::A_PLANE[t]], bb[j][Op::B_PLANE[t]], rest[i][j]);
        if constexpr (!TAIL) {
#pragma unroll
          for (int i = 0; i < FM; i++)
#pragma unroll
            for (int j = 0; j < 2; j++) acc[i][j] = Op::mfma(a[i][0], bb[j][0], acc[i][j]);
        }
      }
    }
  };
  // a step whose successors are whole: nothing in it is conditional, so that the wait for the older fetches leaves the younger
  // ones in flight
  auto step_whole = [&](auto S) {
    constexpr int set = decltype(S)::value;
    fetch(Whole{}, S);
    multiply(std::false_type{}, set);
    stash(std::integral_constant<int, set ^ 1>{}, set ^ 1);
    __syncthreads();
  };
  auto step_ragged = [&](auto S, int t) {
    constexpr int set = decltype(S)::value;
    if (t + 2 < total) {
      fetch(Ragged{}, S);
      next_segment();
    }
    multiply(std::false_type{}, set);
    if (t + 1 < total) stash(std::integral_constant<int, set ^ 1>{}, set ^ 1);
    __builtin_amdgcn_s_waitcnt(0xf70);  // vmcnt(0): the loop above then starts with nothing unaccounted for
    __syncthreads();
  };
  using S0 = std::integral_constant<int, 0>;
  using S1 = std::integral_constant<int, 1>;
  start_segment();
  fetch(Ragged{}, S0{});
  next_segment();
  stash(S0{}, 0);
  if (total > 1) {
    fetch(Ragged{}, S1{});
    next_segment();
  }
  __syncthreads();
  if constexpr (PLANES > 1)
    if (total == 1) multiply(std::true_type{}, 0);
  for (int t = 0; t < total;) {
    if (t + 3 < total && k0 + 2 * BK <= g.K && vectors()) {
      const int s = seg;  // (the next segment has an alignment of its own)
      do {
        step_whole(S0{});
        step_whole(S1{});
        t += 2;
        next_segment();
      } while (seg == s && t + 3 < total && k0 + 2 * BK <= g.K);
      if (seg != s) continue;
    }
    if (t < total) step_ragged(S0{}, t++);
    if (t < total) step_ragged(S1{}, t++);
  }

  if constexpr (PLANES > 1) {
#pragma unroll
    for (int i = 0; i < FM; i++)
#pragma unroll
      for (int j = 0; j < 2; j++) acc[i][j] += rest[i][j];
  }

  // ---- epilogue (the loop ended with a barrier).  Accumulator register r of a 32 x 32 block is row 8 * (r / 4) + 4 * (lane / 32) + r % 4, column lane % 32; each
  //      wavefront transposes a strip of 32 rows x 64 columns at a time through LDS and takes it back 4 consecutive columns
  //      per lane.  The loop over a strip is rolled (the activations are long) and what it reads from memory (residual,
  //      pre-activations) is requested for the whole strip before the first row is worked on: with one read after another, each
  //      behind the previous row's stores, a launch of a few workgroups took 60 us.
  constexpr bool PRECISE = sizeof(TC) == 4;
  float* const stage = reinterpret_cast<float*>(smem) + wave * (32 * STAGE_LD);
  const int per_row = gated ? 8 : 16, rows_per_it = 64 / per_row;  // lanes per strip row
  const int c4 = (lane % per_row) * 4, lane_row = lane / per_row;
  const int64_t nl = n0 + (gated ? wn * 32 : wn * 64) + c4, n = n_off + nl;
  const int count = (int)max((int64_t)0, min((int64_t)4, N - nl));  // columns of this lane that exist
  float bias0[4] = {0.f, 0.f, 0.f, 0.f}, bias1[4] = {0.f, 0.f, 0.f, 0.f};
  if (epi.bias && count > 0) {
    load_few(epi.bias + n, false, count, bias0);
    if (gated) load_few(epi.bias + epi.inter + n, false, count, bias1);
  }
  // 4 elements per access: every row start and the lane's columns aligned to 4 elements
  bool vec = count == 4 && (n & 3) == 0;
  if constexpr (KIND == EPI_STORE) vec = vec && (epi.ldo & 3) == 0 && (reinterpret_cast<uintptr_t>(epi.out) & 15) == 0;
  if constexpr (KIND == EPI_ACT_FWD || KIND == EPI_ACT_BWD)
    vec = vec && (epi.ld_pre & 3) == 0 && (epi.ld_hid & 3) == 0 && (epi.inter & 3) == 0 &&
          ((reinterpret_cast<uintptr_t>(epi.pre) | reinterpret_cast<uintptr_t>(epi.hid) | reinterpret_cast<uintptr_t>(epi.dpre)) & 15) == 0;
  if constexpr (KIND == EPI_OUT)
    vec = vec && (epi.ldy & 3) == 0 && ((reinterpret_cast<uintptr_t>(epi.x) | reinterpret_cast<uintptr_t>(epi.y)) & 15) == 0;

  // element (row m of the tile's coordinates, row j of B) of fp32 operands, in fp32 arithmetic; 8 k at a time, so that their loads
  // wait for memory together, up to the 8 that hold a NaN
  auto element = [&](int64_t m, int64_t j) __attribute__((always_inline)) {
    float sum = 0.f;
    for (int s = 0; s < nseg; s++) {
      const Segment<TI> q = segment(s);
      const int64_t end = s ? q.K : min(slice_k1, q.K), step_a = A_KM ? 1 : q.lda, step_b = B_KM ? 1 : q.ldb;
      const TI* const row_a = q.A + (A_KM ? m * q.lda : m);
      const TI* const row_b = q.B + (B_KM ? j * q.ldb : j);
      for (int64_t k = s ? 0 : slice_k0; k < end && sum == sum; k += 8) {
        float x[8], y[8];
#pragma unroll
        for (int e = 0; e < 8; e++) {
          const int64_t i = min(k + e, end - 1);
          x[e] = to_f32(row_a[i * step_a]);
          y[e] = to_f32(row_b[i * step_b]);
        }
#pragma unroll
        for (int e = 0; e < 8; e++) sum = k + e < end ? fmaf(x[e], y[e], sum) : sum;
      }
    }
    return sum;
  };
  // (fp32: odd rows are negated; 0 - v and not -v, so that a sum of zeros is +0 in every row)
  auto unflipped = [&](float v, int row) { return PLANES > 1 && (row & 1) ? 0.f - v : v; };
#pragma unroll
  for (int i = 0; i < FM; i++) {
    const int64_t mrow0 = m0 + wm * 32 * FM + i * 32;
    constexpr int READS = 8;  // rows of a strip per lane (EPI_ACT_BWD, EPI_OUT: 16 lanes per row)
    float in0[READS][4], in1[READS][4];
    if constexpr (KIND == EPI_ACT_BWD || KIND == EPI_OUT) {
#pragma unroll
      for (int it = 0; it < READS; it++) {
        const int64_t m = min(mrow0 + it * 4 + lane_row, M - 1);
        if (count > 0) {
          if constexpr (KIND == EPI_ACT_BWD) {
            const TC* pre = reinterpret_cast<const TC*>(epi.pre) + m * epi.ld_pre + n;
            load_few(pre, vec, count, in0[it]);
            if (epi.gated) load_few(pre + epi.inter, vec, count, in1[it]);
          } else if (epi.x) {
            load_few(reinterpret_cast<const TX*>(epi.x) + m * epi.ldy + n, vec, count, in0[it]);
          }
        }
      }
    }
#pragma unroll
    for (int j = 0; j < 2; j++)
#pragma unroll
      for (int r = 0; r < 16; r++)
        stage[(8 * (r >> 2) + 4 * (lane >> 5) + (r & 3)) * STAGE_LD + j * 32 + (lane & 31)] = unflipped(acc[i][j][r], r);
    __builtin_amdgcn_wave_barrier();
    auto row_of = [&](int it) { return it * rows_per_it + lane_row; };
    auto staged = [&](int row, int col, float (&v)[4]) __attribute__((always_inline)) {
      const float4 t = *reinterpret_cast<const float4*>(&stage[row * STAGE_LD + col]);
      v[0] = t.x; v[1] = t.y; v[2] = t.z; v[3] = t.w;
      if constexpr (PLANES > 1) {
        const float any = (v[0] + v[1]) + (v[2] + v[3]);
        if (__builtin_expect(any != any, 0)) {
#pragma unroll 1
          for (int e = 0; e < count; e++) {
            const float o = e == 0 ? v[0] : e == 1 ? v[1] : e == 2 ? v[2] : v[3];
            if (o == o) continue;
            const float f = element(mrow0 + row, (gated ? n0 + wn * 32 + (col >= 32 ? N : 0) + (col & 31) : n0 + wn * 64 + col) + e);
#pragma unroll
            for (int q = 0; q < 4; q++) v[q] = q == e ? f : v[q];
          }
        }
      }
    };
    if constexpr (KIND == EPI_ACT_BWD || KIND == EPI_OUT) {
      lt_rolled_rows<READS>([&](int it, float (&r0)[4], float (&r1)[4]) {
        const int64_t m = mrow0 + row_of(it);
        if (m >= M || count == 0) return;
        float v[4];
        staged(row_of(it), c4, v);
        if constexpr (KIND == EPI_ACT_BWD) {
          TC* dpre = reinterpret_cast<TC*>(epi.dpre) + m * epi.ld_pre + n;
          float h[4], o[4];
#pragma unroll
          for (int e = 0; e < 4; e++) {
            float a, da;
            act_eval<PRECISE>(epi.act, r0[e], a, da);
            h[e] = epi.gated ? a * r1[e] : a;
            o[e] = epi.gated ? v[e] * r1[e] * da : v[e] * da;
            v[e] *= a;
          }
          store_few(dpre, vec, count, o);
          if (epi.gated) store_few(dpre + epi.inter, vec, count, v);
          if (epi.hid) store_few(reinterpret_cast<TC*>(epi.hid) + m * epi.ld_hid + n, vec, count, h);
        } else {
          const int64_t idx = m * epi.ldy + n;
#pragma unroll
          for (int e = 0; e < 4; e++) v[e] += bias0[e];
          if (epi.drop.p > 0.f) {
            bool keep[4];
            if ((idx & 3) == 0) {
              dropout_keep4(epi.drop, idx, keep);
            } else {
#pragma unroll
              for (int e = 0; e < 4; e++) keep[e] = dropout_keep(epi.drop, idx + e);
            }
#pragma unroll
            for (int e = 0; e < 4; e++) v[e] = keep[e] ? v[e] * epi.drop.scale : 0.f;
          }
          if (epi.x) {
#pragma unroll
            for (int e = 0; e < 4; e++) v[e] += r0[e];
          }
          store_few(reinterpret_cast<TX*>(epi.y) + idx, vec, count, v);
        }
      }, in0, in1);
    } else {
#pragma unroll 1
      for (int it = 0; it < 32 / rows_per_it; it++) {
        const int64_t m = mrow0 + row_of(it);
        if (m >= M || count == 0) continue;
        float v[4];
        staged(row_of(it), c4, v);
#pragma unroll
        for (int e = 0; e < 4; e++) v[e] += bias0[e];
        if constexpr (KIND == EPI_STORE) {
          if (epi.out_dtype == LT_F32) store_few(reinterpret_cast<float*>(epi.out) + m * epi.ldo + n, vec, count, v);
          else store_few(reinterpret_cast<bf16*>(epi.out) + m * epi.ldo + n, vec, count, v);
        } else {
          TC* pre = reinterpret_cast<TC*>(epi.pre) + m * epi.ld_pre + n;
          float h[4];
#pragma unroll
          for (int e = 0; e < 4; e++) {
            v[e] = to_f32(from_f32<TC>(v[e]));  // the activation sees the stored (rounded) pre-activation, as backward will
            h[e] = act_value<PRECISE>(epi.act, v[e]);
          }
          store_few(pre, vec, count, v);
          if (gated) {
            float vl[4];
            staged(row_of(it), 32 + c4, vl);
#pragma unroll
            for (int e = 0; e < 4; e++) {
              vl[e] = to_f32(from_f32<TC>(vl[e] + bias1[e]));
              h[e] *= vl[e];
            }
            store_few(pre + epi.inter, vec, count, vl);
          }
          store_few(reinterpret_cast<TC*>(epi.hid) + m * epi.ld_hid + n, vec, count, h);
        }
      }
    }
    __builtin_amdgcn_wave_barrier();
  }
}

template <typename T, bool A_KM, bool B_KM, int KIND, typename TX, int FM>
int launch(const GemmProblem& p, int tiles_m, int tiles_n, int groups, hipStream_t stream) {
  hipLaunchKernelGGL((gemm_generic_kernel<T, A_KM, B_KM, KIND, T, TX, FM>), dim3((unsigned)(tiles_m * tiles_n), (unsigned)groups),
                     dim3(256), 0, stream, p, tiles_m, tiles_n);
  LT_LAUNCH_CHECK();
  return LT_OK;
}

// The epilogues beside the plain store occur in one layout each: the projections' (both operands k-major) and, for EPI_ACT_BWD, the
// input gradient's (B mn-major).
template <typename T, int FM>
int launch_kind(const GemmProblem& p, int kind, int io_dtype, int tm, int tn, int groups, hipStream_t stream) {
  const bool a_km = p.sp.mode == SPARSE_NONE ? p.A[0].kmajor : p.sp.mode != SPARSE_DW;
  const bool b_km = p.sp.mode == SPARSE_NONE ? p.B[0].kmajor : p.sp.mode == SPARSE_FWD;
  for (int s = 1; s < p.nseg; s++)
    LT_REQUIRE((bool)p.A[s].kmajor == a_km && (bool)p.B[s].kmajor == b_km, LT_ERR_UNSUPPORTED, "gemm: k-segments of different layouts");
  if (kind == EPI_STORE) {
    if (a_km && b_km) return launch<T, true, true, EPI_STORE, float, FM>(p, tm, tn, groups, stream);
    if (a_km) return launch<T, true, false, EPI_STORE, float, FM>(p, tm, tn, groups, stream);
    if (b_km) return launch<T, false, true, EPI_STORE, float, FM>(p, tm, tn, groups, stream);
    return launch<T, false, false, EPI_STORE, float, FM>(p, tm, tn, groups, stream);
  }
  if (kind == EPI_ACT_FWD && a_km && b_km) return launch<T, true, true, EPI_ACT_FWD, float, FM>(p, tm, tn, groups, stream);
  if (kind == EPI_ACT_BWD && a_km && !b_km) return launch<T, true, false, EPI_ACT_BWD, float, FM>(p, tm, tn, groups, stream);
  if (kind == EPI_OUT && a_km && b_km) {
    if (io_dtype == LT_BF16) return launch<T, true, true, EPI_OUT, bf16, FM>(p, tm, tn, groups, stream);
    return launch<T, true, true, EPI_OUT, float, FM>(p, tm, tn, groups, stream);
  }
  LT_FAIL(LT_ERR_UNSUPPORTED, "gemm: epilogue %d does not occur in this operand layout", kind);
}

template <typename T>
int launch_tile(const GemmProblem& p, int kind, int io_dtype, bool half_tile, int tm, int tn, int groups, hipStream_t stream) {
  return half_tile ? launch_kind<T, 1>(p, kind, io_dtype, tm, tn, groups, stream)
                   : launch_kind<T, 2>(p, kind, io_dtype, tm, tn, groups, stream);
}

}  // namespace

int lt_launch_gemm_generic(const GemmProblem& p, int kind, int dtype, int io_dtype, hipStream_t stream) {
  LT_REQUIRE(p.M > 0 && p.N > 0 && p.nseg >= 1 && p.nseg <= 2, LT_ERR_BAD_ARG, "gemm: bad sizes M=%lld N=%lld nseg=%d",
             (long long)p.M, (long long)p.N, p.nseg);
  const bool gated = kind == EPI_ACT_FWD && p.epi.gated;
  int64_t rows = p.M, cols = p.N, groups = 1;
  const SparseWalk& sp = p.sp;
  if (sp.mode != SPARSE_NONE) {
    LT_REQUIRE(!gated, LT_ERR_UNSUPPORTED, "block-sparse gemm has no gated-activation epilogue");
    LT_REQUIRE(sp.block > 0 && sp.blocks_per_in > 0 && sp.blocks_per_out > 0, LT_ERR_BAD_ARG, "block-sparse gemm: bad layout");
    cols = sp.block;
    if (sp.mode == SPARSE_DW) {
      rows = sp.block;
      groups = p.N / sp.block * sp.blocks_per_in;  // N = in_features
    } else {
      groups = p.N / sp.block;  // N = out_features (FWD) or in_features (DX)
    }
    LT_REQUIRE(groups >= 1 && groups <= 65535, LT_ERR_UNSUPPORTED, "block-sparse gemm: %lld groups exceed the grid limit",
               (long long)groups);
  }
  double flops = lt_gemm_flops(p, kind);
  if (sp.mode == SPARSE_FWD || sp.mode == SPARSE_DX) {
    flops = 2.0 * (double)p.M * (double)p.N * ((sp.mode == SPARSE_FWD ? sp.blocks_per_out : sp.blocks_per_in) * (double)sp.block +
                                                (p.nseg > 1 ? (double)p.K[1] : 0.0));
  } else if (sp.mode == SPARSE_DW) {
    flops = 2.0 * (double)sp.tokens * (double)groups * sp.block * sp.block;
  }
  static const char* tags[4] = {"gemm_generic", "blocksparse_fwd_generic", "blocksparse_dx_generic", "blocksparse_dw_generic"};
  LtProfileScope scope(tags[sp.mode], flops, 0.0, stream);
  if (sp.mode == SPARSE_NONE && p.ksplit > 1) {
    LT_REQUIRE(kind == EPI_STORE && p.nseg == 1 && p.epi.out_dtype == LT_F32 && !p.epi.bias, LT_ERR_BAD_ARG,
               "gemm: a split reduction stores fp32 partial sums of one k-segment");
    groups = p.ksplit;
  }
  const int64_t tiles_n = (cols + (gated ? 64 : 128) - 1) / (gated ? 64 : 128);
  // 64-row tiles where there are no more rows, or where there are fewer than two 128-row ones per CU
  const bool half_tile = rows <= 64 || (rows + 127) / 128 * tiles_n * groups < 512;
  const int64_t tiles_m = (rows + (half_tile ? 63 : 127)) / (half_tile ? 64 : 128);
  LT_REQUIRE(tiles_m * tiles_n <= 0x7fffffff, LT_ERR_UNSUPPORTED, "gemm: M=%lld N=%lld exceed the grid limit", (long long)p.M,
             (long long)p.N);
  return dtype == LT_F32 ? launch_tile<float>(p, kind, io_dtype, half_tile, (int)tiles_m, (int)tiles_n, (int)groups, stream)
                         : launch_tile<bf16>(p, kind, io_dtype, half_tile, (int)tiles_m, (int)tiles_n, (int)groups, stream);
}
