// Host side of the tiled bf16 GEMMs: which problems the kernels of gemm_mfma_kernels.h take, which kernel a problem goes
// to, split reductions and their summing passes.  The kernels are instantiated per epilogue kind in gemm_mfma_kind*.hip.
#include "gemm_mfma_kernels.h"
#ifdef LT_TILE_TIMING
int& lt_tile_timing_launch_counter() { static int n = 0; return n; }
#endif

// defined in gemm_mfma_kind{0,1,2,3}.hip (KIND = EPI_STORE, EPI_ACT_FWD, EPI_ACT_BWD, EPI_OUT)
int lt_mfma_launch_dense_kind0(const GemmProblem& p, int io_dtype, hipStream_t stream);
int lt_mfma_launch_dense_kind1(const GemmProblem& p, int io_dtype, hipStream_t stream);
int lt_mfma_launch_dense_kind2(const GemmProblem& p, int io_dtype, hipStream_t stream);
int lt_mfma_launch_dense_kind3(const GemmProblem& p, int io_dtype, hipStream_t stream);
int lt_mfma_launch_sparse_kind0(const GemmProblem& p, hipStream_t stream);
int lt_mfma_launch_sparse_kind1(const GemmProblem& p, hipStream_t stream);
// 128 x 128 tile, plain store, `slices` slices of the reduction (gemm_mfma_kind0.hip)
int lt_mfma_launch_skinny(const GemmProblem& p, int slices, hipStream_t stream);


bool lt_gemm_mfma_supported(const GemmProblem& p, int kind) {
  constexpr int BM = 256, BN = 256;
  const bool gated = kind == EPI_ACT_FWD && p.epi.gated;
  if (p.M <= 0 || p.N <= 0) return false;
  const int64_t tile_n = gated ? BN / 2 : BN;
  const bool a_km = p.A[0].kmajor, b_km = p.B[0].kmajor;
  if (!a_km && b_km) return false;
  if ((kind == EPI_ACT_FWD || kind == EPI_OUT) && !(a_km && b_km)) return false;
  if (kind == EPI_ACT_BWD && !(a_km && !b_km)) return false;
  // Tiles that stick out past N (and past M for an mn-major A) are the copy-based kernel's: it copies the last row or the
  // last 8 columns again and its epilogue skips what is outside, 8 columns at a time.
  if (p.N % tile_n != 0 || (!a_km && p.M % BM != 0)) {
    if (p.N % 8 != 0 || (!a_km && p.M % 8 != 0) || !dma_selected(p, kind)) return false;
  }
  if ((int64_t)((p.M + BM - 1) / BM) * ((p.N + tile_n - 1) / tile_n) > 0x7fffffff) return false;
  // the epilogue moves 8 columns at a time
  const EpiParams& e = p.epi;
  if (e.bias && !lt_aligned(e.bias, 16)) return false;
  if (kind == EPI_STORE && (e.ldo % 8 != 0 || !lt_aligned(e.out, 16))) return false;
  if ((kind == EPI_ACT_FWD || kind == EPI_ACT_BWD) &&
      (e.ld_pre % 8 != 0 || e.ld_hid % 8 != 0 || e.inter % 8 != 0 || !lt_aligned(e.pre, 16) ||
       (e.hid && !lt_aligned(e.hid, 16)) || (e.dpre && !lt_aligned(e.dpre, 16))))
    return false;
  if (kind == EPI_OUT && (e.ldy % 8 != 0 || !lt_aligned(e.y, 16) || (e.x && !lt_aligned(e.x, 16)))) return false;
  for (int s = 0; s < p.nseg; s++) {
    if ((bool)p.A[s].kmajor != a_km || (bool)p.B[s].kmajor != b_km) return false;
    if (p.K[s] <= 0) return false;
    if ((a_km || b_km) && p.K[s] % 8 != 0) return false;
    if (p.A[s].ld % 8 != 0 || p.B[s].ld % 8 != 0) return false;
    if (!lt_aligned(p.A[s].ptr, 16) || !lt_aligned(p.B[s].ptr, 16)) return false;
  }
  return true;
}

bool lt_sparse_mfma_supported(const GemmProblem& p, int kind);

namespace {
int64_t mid_tiles(int64_t M, int64_t N) { return ((M + 127) / 128) * ((N + 127) / 128); }

// An unfused product's reduction over `stages` stages, split into the number of slices with the least estimated time; returns it in
// us.  A round of `tiles` * slices workgroups takes stage_us(workgroups) per stage; a slice costs a write and a read of its fp32
// partial result at 5 TB/s, the sum a launch.
template <typename F> double best_slices(int64_t M, int64_t N, int64_t tiles, int64_t stages, int64_t max_workgroups, F&& stage_us, int& slices) {
  double best_us = 1e30;
  slices = 1;
  for (int s = 1; s <= 16 && (s == 1 || (tiles * s <= max_workgroups && stages / s >= 4)); s++) {
    const double us = (double)((stages + s - 1) / s) * stage_us(tiles * s) + (s > 1 ? s * (double)M * N * 8.0 / 5e6 + 4.0 : 0.0);
    if (us < best_us * 0.97) {
      best_us = us;
      slices = s;
    }
  }
  return best_us;
}
// 128 x 128 tiles: 64 k take a workgroup 0.45 us alone on its CU, two of them 0.95 us (measured on [128 - 4096, 2048] over 8192: 53 - 69
// us for up to 256 workgroups, 125 for 512).  The main loop that copies between the matrix instructions takes 44 - 68 and 130 there; the
// estimates, and those of mid_selected, are still the older loop's, which leave a product to the other kernel a little too soon.
double mid_best(int64_t M, int64_t N, int64_t K, int& slices, double one = 0.45, double two = 0.95) {
  return best_slices(M, N, mid_tiles(M, N), (K + 63) / 64, 512, [=](int64_t w) { return w <= 256 ? one : two; }, slices);
}
int mid_slices(int64_t M, int64_t N, int64_t K) {
  int slices;
  mid_best(M, N, K, slices);
  return slices;
}
int splitk_slices(int64_t M, int64_t N, int64_t K);
// More 128 x 128 tiles than run at once (512): by the rounds that both kinds of tile take.  A last round that fills part of the chip costs 256 x
// 256 tiles most of a whole one, one that leaves the CUs a single 128 x 128 tile half of a whole one; and the two workgroups of a CU work
// through their epilogues beside each other's products, which is worth the more the shorter the reduction.
// Activation epilogues, whole rounds of 128 x 128 tiles against half as many of 256 x 256, us: over 512 69, 80; over 1024 104, 103; over 2048 348,
// 321; a gated forward epilogue, which 256 x 256 tiles read back whole, 10 % worse.  419 products, T 560 - 70000, widths 128 - 28672, reductions
// 64 - 4096: where the estimate takes these tiles they are 0.39 - 1.06 of the other's time, 24 % below it on average.  256 x 256 and 128 x 128
// tiles, us: [3333, 6400] over 1600, SiLU 115, 98, its input gradient 128, 110; [5500, 3072] over 768 84, 58; [2500, 8192] over 2048 148, 108;
// [4096, 2048] over 512 46.6, 40.0.
// A single round of 256 x 256 tiles that leaves CUs idle has the caches to itself, and over a long reduction nothing is left to work beside:
// forward [2203, 5176] over 4096 107, 119; [563, 14776] over 3584 111, 119; [1100, 8192] over 3072 85, 91 (over 2048 65, 63); backward [2203, 5176]
// over 4096 121, 136 (over 3584 [889, 10048] 114, 105).
// Unfused products and down-projections have less of an epilogue to work beside: two whole rounds against one 57, 53 over 1024, 94, 79 over 2048,
// 172, 145 over 4096.  They change where the large tiles' second round is nearly empty: [5500, 2880] over 2880 148, 113, its input gradient 137, 110;
// over 11520 494, 397; [10000, 1600] over 1600 100, 85; a down-projection, whose dropout and residual are some work, also where it is half
// full ([11376, 2080] over 784 90, 81) or one of several ([31229, 3616] over 848 410, 371), where an unfused product keeps the large tiles: input
// gradient [19957, 1392] over 1104 102, 117; [16748, 3408] over 1048 151, 168; [11462, 2832] over 1424 145, 161.  T 2000 - 40000, widths 512 - 4096,
// reductions 768 - 16384, of the other's time: 102 down-projections 0.54 - 1.04, 13 % below it on average, 41 input gradients 0.69 - 1.00, 14 %.
bool mid_rounds_shorter(int64_t M, int64_t columns, int64_t K, int kind, bool gated_forward) {
  const double large = (double)((M + 255) / 256 * ((columns + 255) / 256)) / 256, small = (double)mid_tiles(M, columns) / 512;
  auto whole = [](double r) { return (double)(int64_t)r; };
  const double lf = large - whole(large), sf = small - whole(small);
  const double large_rounds = lf == 0.0 ? large : large < 1.0 ? 0.65 + 0.35 * lf : whole(large) + std::min(1.0, 0.58 + std::max(0.0, lf - 0.4) * 1.1);
  const double small_rounds = sf == 0.0 ? small : whole(small) + (sf <= 0.5 ? 0.5 : std::min(1.0, 0.82 + (sf - 0.5) * 0.7));
  const bool fused = kind == EPI_ACT_FWD || kind == EPI_ACT_BWD;
  if (!fused && (large < 1.0 || K < 768)) return false;  // (shorter reductions: not measured)
  if (fused && large < 1.0 && K > (kind == EPI_ACT_BWD ? 3584 : 2048)) return false;
  const double ratio = fused ? 0.92 + 0.16 * std::min(1.0, std::max(0.0, ((double)K - 512) / 1536)) + (gated_forward ? 0.1 : 0.0)
                             : (kind == EPI_OUT ? 1.0 : 1.16) + 0.26 * std::min(1.0, std::max(0.0, ((double)K - 768) / 1600));
  return ratio * small_rounds / 2 < 0.96 * large_rounds;
}
// 128 x 128 tiles where they all run at once, two workgroups per CU; 256 x 256 ones then fill half of the chip at most.  [1024, 8192]
// over 2048 (512 of them): 37 us against 47.  Where the product is unfused, the 256 x 256
// kernel can split its reduction into as many slices as `room` (bytes of workspace) holds, and the estimates are compared:
//   k-major A: 64 k take 0.58 us (two workgroups on a CU 1.04) against 1.45, and a start and an end of 15 us.  Down-projection of hidden
//     4096 over 16384, T 1025 and 1790: 260 and 269 us against 209 and 238 in two slices; its input gradient, T 1024 and 1200: 170 and
//     271 against 141 and 172; T 2048 (128 tiles of 256 x 256, unsplit): 271 against 374.  A tenth is left to the 128 x 128 tiles,
//     within which either was the faster one.
//   weight gradients (both operands mn-major): 64 k of a 256 x 256 tile take 1.2 us, and its start and end 5 us more.
bool mid_selected(const GemmProblem& p, int kind, size_t room = 0) {
  const int64_t columns = kind == EPI_ACT_FWD && p.epi.gated ? 2 * p.N : p.N;
  if (!lt_gemm_mid_supported(p, kind)) return false;
  if (mid_tiles(p.M, columns) > 512)
    return p.A[0].kmajor && mid_rounds_shorter(p.M, columns, p.K[0], kind, kind == EPI_ACT_FWD && p.epi.gated);
  const int64_t tiles = ((p.M + 255) / 256) * ((p.N + 255) / 256), stages = (p.K[0] + 63) / 64;
  const double partial_us = (double)p.M * p.N * 4.0 / 5e6;  // a pass over one slice's partial sums
  int slices;
  int64_t s = splitk_slices(p.M, p.N, p.K[0]);
  if (p.A[0].kmajor) {
    s = std::min<int64_t>(s, (int64_t)(room / ((size_t)p.M * (size_t)p.N * sizeof(float))));
    if (s <= 1) return true;
    const double us = (double)((stages + s - 1) / s) * 1.45 + 15.0 + s * partial_us + 4.0;
    return mid_best(p.M, p.N, p.K[0], slices, 0.58, 1.04) < 1.1 * us;
  }
  const double us = (double)((tiles * s + 255) / 256) * ((double)(stages + s - 1) / s * 1.2 + 5.0) + (s > 1 ? 2 * s * partial_us + 4.0 : 0.0);
  return mid_best(p.M, p.N, p.K[0], slices) < us;
}
}  // namespace

size_t lt_gemm_mid_splitk_workspace(int64_t M, int64_t N, int64_t K) {
  const int slices = mid_tiles(M, N) <= 512 ? mid_slices(M, N, K) : 1;
  return slices > 1 ? lt_align_up((size_t)slices * (size_t)M * (size_t)N * sizeof(float), 256) : 0;
}

int lt_gemm_colsum_rows(const GemmProblem& p, int dtype, int io_dtype) {
  if (dtype != LT_BF16 || p.epi.ld_pre % 8 != 0) return 0;
  if (mid_selected(p, EPI_ACT_BWD)) return 64;
  if (p.sp.mode == SPARSE_NONE)
    return lt_gemm_mfma_supported(p, EPI_ACT_BWD) && dma_selected(p, EPI_ACT_BWD) ? 128 : 0;
  return p.sp.mode == SPARSE_DX && lt_sparse_mfma_supported(p, EPI_ACT_BWD) ? 64 : 0;
}

static const char* mfma_tag(const GemmProblem& p, int kind, bool mid) {
  static const char* names[2][3][4] = {
      {{"gemm_bf16_nt_store", "gemm_bf16_nt_act_fwd", "gemm_bf16_nt_act_bwd", "gemm_bf16_nt_out"},
       {"gemm_bf16_nn_store", "gemm_bf16_nn_act_fwd", "gemm_bf16_nn_act_bwd", "gemm_bf16_nn_out"},
       {"gemm_bf16_tn_store", "gemm_bf16_tn_act_fwd", "gemm_bf16_tn_act_bwd", "gemm_bf16_tn_out"}},
      {{"gemm_mid_nt_store", "gemm_mid_nt_act_fwd", "gemm_mid_nt_act_bwd", "gemm_mid_nt_out"},
       {"gemm_mid_nn_store", "gemm_mid_nn_act_fwd", "gemm_mid_nn_act_bwd", "gemm_mid_nn_out"},
       {"gemm_mid_tn_store", "gemm_mid_tn_act_fwd", "gemm_mid_tn_act_bwd", "gemm_mid_tn_out"}}};
  const int layout = p.A[0].kmajor ? (p.B[0].kmajor ? 0 : 1) : 2;
  return names[mid][layout][kind];
}

double lt_gemm_flops(const GemmProblem& p, int kind) {
  const double n = (kind == EPI_ACT_FWD && p.epi.gated) ? 2.0 * p.N : (double)p.N;
  double k = (double)p.K[0] + (p.nseg > 1 ? (double)p.K[1] : 0.0);
  return 2.0 * (double)p.M * n * k;
}

int lt_launch_gemm_mfma(const GemmProblem& p, int kind, int io_dtype, hipStream_t stream) {
  LT_REQUIRE(lt_gemm_mfma_supported(p, kind), LT_ERR_UNSUPPORTED, "tiled bf16 gemm does not take this problem");
  const bool mid = mid_selected(p, kind);
  LtProfileScope scope(mfma_tag(p, kind, mid), lt_gemm_flops(p, kind), 0.0, stream);
  if (mid) return lt_launch_gemm_mid(p, kind, io_dtype, stream);
  switch (kind) {
    case EPI_STORE: return lt_mfma_launch_dense_kind0(p, io_dtype, stream);
    case EPI_ACT_FWD: return lt_mfma_launch_dense_kind1(p, io_dtype, stream);
    case EPI_ACT_BWD: return lt_mfma_launch_dense_kind2(p, io_dtype, stream);
    case EPI_OUT: return lt_mfma_launch_dense_kind3(p, io_dtype, stream);
  }
  LT_FAIL(LT_ERR_BAD_ARG, "unknown epilogue kind %d", kind);
}

namespace {
constexpr int SKINNY_MAX_SLICES = 16;
}  // namespace

// partial sums of up to SKINNY_MAX_SLICES slices of a [tokens, lowrank] (or equally large) fp32 result
size_t lt_gemm_skinny_workspace(int64_t tokens, int64_t lowrank) {
  return lt_align_up((size_t)SKINNY_MAX_SLICES * (size_t)tokens * (size_t)lowrank * sizeof(float), 256);
}

namespace {
// slices of the reduction for an [M, N] result on 256 x 256 tiles: enough workgroups for the 256 CUs, each slice at least
// 16 k-steps long
int splitk_slices(int64_t M, int64_t N, int64_t K) {
  const int64_t tiles = ((M + 255) / 256) * ((N + 255) / 256);
  if (tiles >= 128) return 1;
  const int64_t by_k = K / (16 * DK);
  return (int)std::max<int64_t>(1, std::min<int64_t>(std::min<int64_t>(256 / tiles, by_k), 8));
}
}  // namespace

size_t lt_gemm_splitk_workspace(int64_t M, int64_t N, int64_t K) {
  const int slices = splitk_slices(M, N, K);
  return slices > 1 ? lt_align_up((size_t)slices * (size_t)M * (size_t)N * sizeof(float), 256) : 0;
}

namespace {
// Slices of an any-shape product's reduction: the number with the least estimated time.  A CU holds three 128 x 128 workgroups
// (four of the 64 x 128 ones a small grid runs on), in fp32, which has twice the accumulators, one less; with w of them resident a
// k-step of 16 takes about 0.35 + 0.6 w us (0.42 + 0.32 w), measured in fp32 on 4096^3 and 321 x 7168 x 1792; a slice costs a write and
// a read of its fp32 partial result at 5 TB/s.  Counting the one less in fp32 changes nothing (training step, T 4096, hidden 768: 1266 us
// and 1277), so the rule is the same for both.
int generic_splitk_slices(int64_t M, int64_t N, int64_t K) {
  const int64_t tiles = ((M + 127) / 128) * ((N + 127) / 128), half_tiles = ((M + 63) / 64) * ((N + 127) / 128);
  if (tiles >= 3072) return 1;
  int best = 1;
  double best_us = 1e30;
  for (int s = 1; s <= 16 && (s == 1 || K / s >= 128); s++) {
    const bool half = M <= 64 || tiles * s < 512;
    const int64_t workgroups = (half ? half_tiles : tiles) * s, slots = half ? 1024 : 768;
    auto step_us = [&](int64_t resident) { return half ? 0.42 + 0.32 * resident : 0.35 + 0.6 * resident; };
    const int64_t full = workgroups / slots, rest = workgroups % slots;
    const double steps = (double)((K + 16 * s - 1) / (16 * s));
    double us = steps * (full * step_us(slots / 256) + (rest ? step_us((rest + 255) / 256) : 0.0));
    if (s > 1) us += (double)s * M * N * 8.0 / 5e6 + 4.0;
    if (us < best_us * 0.97) {
      best_us = us;
      best = s;
    }
  }
  return best;
}
}  // namespace

size_t lt_gemm_generic_splitk_workspace(int64_t M, int64_t N, int64_t K) {
  const int slices = generic_splitk_slices(M, N, K);
  return slices > 1 ? lt_align_up((size_t)slices * (size_t)M * (size_t)N * sizeof(float), 256) : 0;
}

int lt_launch_gemm_skinny(const GemmProblem& p, int dtype, int io_dtype, void* workspace, size_t workspace_bytes,
                          hipStream_t stream, ColReduceQueue* queue, bool may_wait) {
  if (lt_gemm_stream_supported(p, EPI_STORE, dtype, io_dtype)) return lt_launch_gemm_stream(p, EPI_STORE, dtype, io_dtype, stream);
  if (lt_gemm_thin_selected(p, dtype, workspace != nullptr)) return lt_launch_gemm_thin(p, stream);
  const bool a_km = p.A[0].kmajor, b_km = p.B[0].kmajor;
  const EpiParams& e = p.epi;
  if (e.bias) may_wait = false;
  const size_t slice = (size_t)p.M * (size_t)p.N * sizeof(float);
  if (dtype == LT_BF16 && e.ldo == p.N && mid_selected(p, EPI_STORE, workspace ? workspace_bytes : 0)) {
    const int slices = (int)std::min<size_t>((size_t)mid_slices(p.M, p.N, p.K[0]), workspace ? workspace_bytes / slice : 0);
    if (slices <= 1) return lt_launch_gemm(p, EPI_STORE, dtype, io_dtype, stream);
    GemmProblem q = p;
    q.ksplit = slices;
    q.split_stride = p.M * p.N;
    q.epi = EpiParams{};
    float* partial;
    LT_TRY(lt_place_partials(workspace, slices * slice, 1, may_wait, queue, &partial, stream));
    q.epi.out = partial;
    q.epi.ldo = p.N;
    q.epi.out_dtype = LT_F32;
    LT_TRY(lt_launch_gemm(q, EPI_STORE, dtype, io_dtype, stream));
    return lt_splitk_reduce(partial, slices, p.M * p.N, p.M * p.N, (int)p.N, e.bias, e.out_dtype, e.out, stream, queue);
  }
  bool ok = dtype == LT_BF16 && p.nseg == 1 && p.sp.mode == SPARSE_NONE && p.M > 0 && p.N > 0 && p.N % 128 == 0 &&
            !(!a_km && b_km) && (a_km || p.M % 128 == 0) && ((!a_km && !b_km) || p.K[0] % 8 == 0) && p.K[0] > 0 &&
            p.A[0].ld % 8 == 0 && p.B[0].ld % 8 == 0 && lt_aligned(p.A[0].ptr, 16) && lt_aligned(p.B[0].ptr, 16) &&
            e.ldo == p.N && lt_aligned(e.out, 16) && (!e.bias || lt_aligned(e.bias, 16));
  const int64_t tiles = ((p.M + 127) / 128) * (p.N / 128);
  // a result only 128 wide (or, for an mn-major A, 128 tall) would leave half of every 256 x 256 tile empty: the 128 x 128
  // tile below takes it when it can
  const bool half_tiles = ok && (p.N == 128 || (!a_km && p.M == 128));
  if (!half_tiles && dtype == LT_BF16 && p.sp.mode == SPARSE_NONE && lt_gemm_mfma_supported(p, EPI_STORE)) {
    // 256 x 256 tiles fit: the copy-based kernel, its reduction split when the tiles alone leave CUs idle
    const int slices = p.nseg == 1 ? splitk_slices(p.M, p.N, p.K[0]) : 1;
    if (slices > 1 && workspace && workspace_bytes >= slices * slice && dma_selected(p, EPI_STORE) && e.ldo == p.N) {
      GemmProblem q = p;
      q.ksplit = slices;
      q.variant = 2;
      q.split_stride = p.M * p.N;
      float* partial;
      LT_TRY(lt_place_partials(workspace, slices * slice, 1, may_wait, queue, &partial, stream));
      q.epi.out = partial;
      q.epi.ldo = p.N;
      q.epi.out_dtype = LT_F32;
      q.epi.bias = nullptr;
      LT_TRY(lt_launch_gemm(q, EPI_STORE, dtype, io_dtype, stream));
      return lt_splitk_reduce(partial, slices, p.M * p.N, p.M * p.N, (int)p.N, e.bias, e.out_dtype, e.out, stream, queue);
    }
    if (((p.M + 255) / 256) * ((p.N + 255) / 256) >= 64 || slices == 1) ok = false;
  }
  if (!ok) {
    // any-shape kernel: split the reduction when the tiles alone leave most workgroup slots empty
    const bool tiled = dtype == LT_BF16 && lt_gemm_mfma_supported(p, EPI_STORE);
    const int slices = (!tiled && p.nseg == 1 && p.sp.mode == SPARSE_NONE && e.ldo == p.N && (p.N & 3) == 0 &&
                        lt_aligned(e.out, 16) && (!e.bias || lt_aligned(e.bias, 16)))
                           ? generic_splitk_slices(p.M, p.N, p.K[0]) : 1;
    if (slices > 1 && workspace && workspace_bytes >= slices * slice) {
      GemmProblem q = p;
      q.ksplit = slices;
      q.split_stride = p.M * p.N;
      float* partial;
      LT_TRY(lt_place_partials(workspace, slices * slice, 1, may_wait, queue, &partial, stream));
      q.epi.out = partial;
      q.epi.out_dtype = LT_F32;
      q.epi.bias = nullptr;
      LT_TRY(lt_launch_gemm_generic(q, EPI_STORE, dtype, io_dtype, stream));
      return lt_splitk_reduce(partial, slices, p.M * p.N, p.M * p.N, (int)p.N, e.bias, e.out_dtype, e.out, stream, queue);
    }
    return lt_launch_gemm(p, EPI_STORE, dtype, io_dtype, stream);
  }
  const int kt_total = (int)((p.K[0] + BK - 1) / BK);
  int slices = 1;
  if (workspace && tiles < 192) {
    // two workgroups per CU (64 KiB of LDS each): the slices are short and bound by load latency
    // (one workgroup per CU where a slice's fp32 partial result is as large as the operand tile it read: with twice the
    // slices the partial sums cost more than the second workgroup hides -- measured on [4096, 128] results)
    const int64_t workgroups = tiles <= 64 ? 256 : 512;
    slices = (int)std::min<int64_t>(std::min<int64_t>(workgroups / tiles, kt_total / 4), SKINNY_MAX_SLICES);
    const int64_t fit = (int64_t)(workspace_bytes / slice);
    slices = (int)std::max<int64_t>(1, std::min<int64_t>(slices, fit));
  }
  GemmProblem q = p;
  float* partial = nullptr;
  if (slices > 1) {
    q.ksplit = slices;
    q.split_stride = p.M * p.N;
    LT_TRY(lt_place_partials(workspace, slices * slice, 1, may_wait, queue, &partial, stream));
    q.epi.out = partial;
    q.epi.out_dtype = LT_F32;
    q.epi.bias = nullptr;
  }
  {
    LtProfileScope scope("gemm_bf16_skinny", lt_gemm_flops(p, EPI_STORE), 0.0, stream);
    const int status = lt_mfma_launch_skinny(q, slices, stream);
    if (status != LT_OK || slices == 1) return status;
  }
  return lt_splitk_reduce(partial, slices, p.M * p.N, p.M * p.N, (int)p.N, e.bias, e.out_dtype, e.out, stream, queue);
}

// Which of the products share a launch.  Low-rank gradients are a few tiles each, in as many slices as there are CUs: a launch of 9 - 16 us
// that is mostly its start and its end.  With the same number of slices for all of a subset, their workgroups are equally long and at
// most 256, one per CU, so that the launch takes as long as its longest slice; the estimate is mid_best's, and a launch costs 5 us more.
// Launches one by one, together: qkv, rank 16, T 16384 (108 + 18 tiles, 2 slices) 63 + 16 us, 67; PixelFly of hidden 1024, rank 64, T 4000
// (8 + 32, 6) 9 + 11, 13.5; (64 + 8, 3) 16 + 8, 17.5.  108 layers, T 64 - 20000, widths 64 - 6144, ranks 8 - 136: where the estimate puts products
// together, all take 0.46 - 0.96 of the launches one by one with their sums, the older loop's stage time notwithstanding.
int lt_launch_gemm_gradients(const GemmProblem* problems, int n, int dtype, int io_dtype, void* workspace, size_t workspace_bytes,
                             hipStream_t stream, ColReduceQueue* queue) {
  LT_REQUIRE(n <= LT_MID_GROUP_MAX, LT_ERR_BAD_ARG, "gradients: %d of them", n);
  unsigned group = 0;
  int slices = 1;
  double gain = 0.0;
  for (unsigned subset = 3; dtype == LT_BF16 && workspace && subset < 1u << n; subset++) {
    int64_t tiles = 0;
    size_t elements = 0;
    double alone = 0.0;
    int members = 0;
    bool ok = true;
    for (int j = 0; ok && j < n; j++) {
      if (!(subset >> j & 1)) continue;
      const GemmProblem& p = problems[j];
      ok = !p.A[0].kmajor && !p.B[0].kmajor && p.K[0] == problems[0].K[0] && p.epi.ldo == p.N && !p.epi.bias &&
           mid_selected(p, EPI_STORE, workspace_bytes);
      if (!ok) break;
      int s;
      alone += mid_best(p.M, p.N, p.K[0], s) + 5.0;
      tiles += mid_tiles(p.M, p.N);
      elements += (size_t)p.M * (size_t)p.N;
      members++;
    }
    if (!ok || members < 2 || tiles > 256) continue;
    const int64_t stages = (problems[0].K[0] + 63) / 64;
    const int most = (int)std::max<int64_t>(1, std::min<int64_t>(std::min<int64_t>(256 / tiles, stages / 4), SKINNY_MAX_SLICES));
    for (int s = 1; s <= most; s++) {
      if (s > 1 && s * elements * sizeof(float) + LT_MID_GROUP_MAX * 256 > workspace_bytes) break;
      const double us = (double)((stages + s - 1) / s) * 0.45 + (s > 1 ? s * (double)elements * 8.0 / 5e6 + 4.0 : 0.0) + 5.0;
      if (alone - us > gain) {
        gain = alone - us;
        group = subset;
        slices = s;
      }
    }
  }
  GemmProblem together[LT_MID_GROUP_MAX];
  ColReduceQueue* sums = queue;
  char* place = nullptr;
  int members = 0;
  if (slices > 1) {
    size_t bytes = 0;
    int results = 0;
    for (int j = 0; j < n; j++)
      if (group >> j & 1) {
        bytes += lt_align_up(slices * (size_t)problems[j].M * (size_t)problems[j].N * sizeof(float), 256);
        results++;
      }
    float* partial;
    LT_TRY(lt_place_partials(workspace, bytes, results, true, sums, &partial, stream));
    place = (char*)partial;
  }
  for (int j = 0; j < n; j++) {
    if (!(group >> j & 1)) continue;
    GemmProblem& q = together[members++] = problems[j];
    if (slices > 1) {
      q.ksplit = slices;
      q.split_stride = q.M * q.N;
      q.epi.out = place;
      q.epi.out_dtype = LT_F32;
      place += lt_align_up(slices * (size_t)q.M * (size_t)q.N * sizeof(float), 256);
    }
  }
  if (members) LT_TRY(lt_launch_gemm_mid_group(together, members, stream));
  members = 0;
  for (int j = 0; j < n; j++) {  // (sums that do not wait, before their place is used again)
    if (!(group >> j & 1)) continue;
    const GemmProblem& p = problems[j];
    if (slices > 1)
      LT_TRY(lt_splitk_reduce((const float*)together[members].epi.out, slices, p.M * p.N, p.M * p.N, (int)p.N, nullptr, p.epi.out_dtype,
                              p.epi.out, stream, sums));
    members++;
  }
  for (int j = 0; j < n; j++)
    if (!(group >> j & 1)) LT_TRY(lt_launch_gemm_skinny(problems[j], dtype, io_dtype, workspace, workspace_bytes, stream, queue, true));
  return LT_OK;
}

namespace {
// sum of the split-k slices of an [M, N] result, 8 columns per thread, through the EPI_OUT epilogue (bias, dropout, residual)
template <typename TX>
__global__ __launch_bounds__(256) void splitk_reduce_out_kernel(const float* __restrict__ partial, int slices, int64_t stride,
                                                                 int64_t M, int64_t N, EpiParams e) {
  const int64_t i = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) * 8;
  if (i >= M * N) return;
  float v[8];
  load8(partial + i, v);
  for (int s = 1; s < slices; s++) {
    float w[8];
    load8(partial + (int64_t)s * stride + i, w);
#pragma unroll
    for (int k = 0; k < 8; k++) v[k] += w[k];
  }
  epi_out8<TX>(e, i / N, i % N, v);
}
}  // namespace

size_t lt_gemm_out_splitk_workspace(int dtype, int64_t M, int64_t N, int64_t K, size_t cap_bytes) {
  size_t full = lt_gemm_generic_splitk_workspace(M, N, K);
  if (dtype == LT_BF16) full = std::max({full, lt_gemm_splitk_workspace(M, N, K), lt_gemm_mid_splitk_workspace(M, N, K)});
  const size_t slice = (size_t)M * (size_t)N * sizeof(float);
  if (full == 0 || cap_bytes < 2 * slice) return 0;
  return std::min(full, lt_align_up(cap_bytes / slice * slice, 256));
}

int lt_launch_gemm_out(const GemmProblem& p, int dtype, int io_dtype, void* workspace, size_t workspace_bytes,
                       hipStream_t stream) {
  const EpiParams& e = p.epi;
  if (lt_gemm_stream_supported(p, EPI_OUT, dtype, io_dtype)) return lt_launch_gemm_stream(p, EPI_OUT, dtype, io_dtype, stream);
  if (p.nseg == 1 && p.sp.mode == SPARSE_NONE && workspace && lt_aligned(workspace, 16) && p.M > 0 && p.N > 0 &&
      p.N % 8 == 0 && e.ldy % 8 == 0 && lt_aligned(e.y, 16) && (!e.x || lt_aligned(e.x, 16)) &&
      (!e.bias || lt_aligned(e.bias, 16))) {
    GemmProblem q = p;
    q.epi = EpiParams{};
    q.epi.out = workspace;
    q.epi.ldo = p.N;
    q.epi.out_dtype = LT_F32;
    const size_t slice = (size_t)p.M * (size_t)p.N * sizeof(float);
    // the tiled kernel where it takes the problem, else the any-shape kernel
    const bool tiled = dtype == LT_BF16 && lt_gemm_mfma_supported(q, EPI_STORE) && dma_selected(q, EPI_STORE);
    const bool tiled_unsplit = dtype == LT_BF16 && lt_gemm_mfma_supported(p, EPI_OUT);
    const bool mid = dtype == LT_BF16 && mid_selected(q, EPI_STORE, workspace_bytes);
    const int wanted = mid ? mid_slices(p.M, p.N, p.K[0])
                       : tiled ? splitk_slices(p.M, p.N, p.K[0]) : tiled_unsplit ? 1 : generic_splitk_slices(p.M, p.N, p.K[0]);
    const int slices = (int)std::min<size_t>((size_t)wanted, workspace_bytes / slice);
    if (slices > 1) {
      q.ksplit = slices;
      q.split_stride = p.M * p.N;
      if (tiled && !mid) q.variant = 2;
      if (tiled) LT_TRY(lt_launch_gemm(q, EPI_STORE, dtype, io_dtype, stream));
      else LT_TRY(lt_launch_gemm_generic(q, EPI_STORE, dtype, io_dtype, stream));
      LtProfileScope scope("splitk_reduce_out", 0.0,
                           (double)p.M * p.N * (4.0 * slices + (e.x ? 2 : 1) * lt_dtype_size(io_dtype)), stream);
      const dim3 grid((unsigned)((p.M * p.N / 8 + 255) / 256)), block(256);
      if (io_dtype == LT_BF16)
        hipLaunchKernelGGL((splitk_reduce_out_kernel<bf16>), grid, block, 0, stream, (const float*)workspace, slices, p.M * p.N, p.M, p.N, e);
      else
        hipLaunchKernelGGL((splitk_reduce_out_kernel<float>), grid, block, 0, stream, (const float*)workspace, slices, p.M * p.N, p.M, p.N, e);
      LT_LAUNCH_CHECK();
      return LT_OK;
    }
  }
  return lt_launch_gemm(p, EPI_OUT, dtype, io_dtype, stream);
}

// block-sparse walk on the matrix cores: 64 x 64 blocks, bf16, 16-byte aligned operands
bool lt_sparse_mfma_supported(const GemmProblem& p, int kind) {
  const SparseWalk& sp = p.sp;
  const EpiParams& e = p.epi;
  if (sp.mode == SPARSE_NONE || sp.block != 64 || p.M <= 0) return false;
  // gated forward epilogue: p.N counts the gate columns; the walk pairs gate block j with linear block j + N / 64
  if (kind == EPI_ACT_FWD && e.gated && (sp.mode != SPARSE_FWD || p.N % 64 != 0 || e.inter != p.N)) return false;
  if (sp.ld_act % 8 != 0 || !lt_aligned(sp.act, 16)) return false;
  if (sp.mode == SPARSE_DW) {
    if (kind != EPI_STORE || sp.ld_act2 % 8 != 0 || !lt_aligned(sp.act2, 16) || !lt_aligned(e.out, 16)) return false;
    return true;
  }
  if (!lt_aligned(sp.weight, 16)) return false;
  // the walk addresses a tile's rows with 32-bit byte offsets, products of a row number and a pitch of at most 24 bits (2^32 / 257)
  if (257 * sp.ld_act * 2 + 1024 >= (int64_t)1 << 32) return false;
  if (p.nseg > 1) {
    if (257 * p.A[1].ld * 2 + 1024 >= (int64_t)1 << 32 || 257 * p.B[1].ld * 2 + 1024 >= (int64_t)1 << 32) return false;
    if (p.K[1] <= 0 || p.K[1] % 8 != 0 || p.A[1].ld % 8 != 0 || p.B[1].ld % 8 != 0 || !lt_aligned(p.A[1].ptr, 16) ||
        !lt_aligned(p.B[1].ptr, 16))
      return false;
  }
  if (e.bias && !lt_aligned(e.bias, 16)) return false;
  if (kind == EPI_STORE && (e.ldo % 8 != 0 || !lt_aligned(e.out, 16))) return false;
  if ((kind == EPI_ACT_FWD || kind == EPI_ACT_BWD) &&
      (e.ld_pre % 8 != 0 || e.ld_hid % 8 != 0 || e.inter % 8 != 0 || !lt_aligned(e.pre, 16) ||
       (e.hid && !lt_aligned(e.hid, 16)) || (e.dpre && !lt_aligned(e.dpre, 16))))
    return false;
  if (kind == EPI_OUT && (e.ldy % 8 != 0 || !lt_aligned(e.y, 16) || (e.x && !lt_aligned(e.x, 16)))) return false;
  return true;
}

bool lt_sparse_forward_grouped(const GemmProblem& p, int kind) {
  const SparseWalk& sp = p.sp;
  if (sp.mode != SPARSE_FWD || (kind != EPI_STORE && kind != EPI_ACT_FWD) || (kind == EPI_ACT_FWD && p.epi.gated)) return false;
  if (!lt_sparse_mfma_supported(p, kind)) return false;
  if (sp.out_group < 4 || sp.out_group % 4 != 0 || sp.out_stride > 1 || p.N % 256 != 0) return false;
  // the list travels in one register: at most 64 entries, input block and flat position in 16 bits each
  if (sp.blocks_per_out > 64 || sp.ld_act / 64 * sp.blocks_per_in > 65535) return false;
  if (p.nseg > 1 && p.K[1] % 64 != 0) return false;  // (this form copies whole k-blocks only)
  // 32-bit byte offsets inside a tile
  if (257 * sp.ld_act * 2 + 1024 >= (int64_t)1 << 32) return false;
  if (p.nseg > 1 && (257 * p.A[1].ld * 2 + 1024 >= (int64_t)1 << 32 || 257 * p.B[1].ld * 2 + 1024 >= (int64_t)1 << 32)) return false;
  return true;
}

bool lt_sparse_dw_out_grouped(const GemmProblem& p) {
  const SparseWalk& sp = p.sp;
  const int64_t out_features = sp.ld_act;
  if (sp.out_stride > 1 && (int64_t)sp.out_group * sp.out_stride * 64 != out_features) return false;  // runs must tile the blocks
  return sp.mode == SPARSE_DW && sp.out_group >= 4 && sp.out_group % 4 == 0 && sp.forward_indices && out_features % 256 == 0 &&
         sp.tokens > 0 && 33 * sp.ld_act * 2 + 1024 < (int64_t)1 << 32 && 33 * sp.ld_act2 * 2 + 1024 < (int64_t)1 << 32;
}

bool lt_sparse_dw_in_grouped(const GemmProblem& p) {
  const SparseWalk& sp = p.sp;
  const int64_t in_features = p.N;
  if (sp.mode != SPARSE_DW || !lt_sparse_mfma_supported(p, EPI_STORE) || lt_sparse_dw_out_grouped(p)) return false;
  if (sp.in_group < 4 || sp.in_group % 4 != 0 || !sp.backward_indices || in_features % 256 != 0) return false;
  if (sp.in_stride > 1 && (int64_t)sp.in_group * sp.in_stride * 64 != in_features) return false;  // runs must tile the blocks
  return sp.tokens > 0 && 33 * sp.ld_act * 2 + 1024 < (int64_t)1 << 32 && 33 * sp.ld_act2 * 2 + 1024 < (int64_t)1 << 32;
}

namespace {
// Slices of the token reduction of a grouped weight gradient with `tiles` tiles: enough workgroups for the 256 CUs, each slice at
// least 32 k-steps long.  Measured: hidden 1024, tiled butterfly, T 4000: 64 tiles of the up-projection whole 80 us, in three slices
// 51 and their sum 7.
int dw_slices(int64_t tiles, int64_t tokens) {
  if (tiles >= 192) return 1;
  return (int)std::max<int64_t>(1, std::min<int64_t>(std::min<int64_t>(256 / tiles, tokens / (32 * DK)), 8));
}
int64_t dw_tiles(int64_t features, int per_block) { return (int64_t)((per_block + 3) / 4) * (features / 256); }
}  // namespace

int lt_sparse_dw_slices(const GemmProblem& p) {
  const SparseWalk& sp = p.sp;
  if (sp.mode != SPARSE_DW || !lt_sparse_mfma_supported(p, EPI_STORE)) return 0;
  if (lt_sparse_dw_out_grouped(p)) return dw_slices(dw_tiles(sp.ld_act, sp.blocks_per_out), sp.tokens);
  return lt_sparse_dw_in_grouped(p) ? dw_slices(dw_tiles(p.N, sp.blocks_per_in), sp.tokens) : 0;
}

size_t lt_sparse_dw_split_workspace(int64_t in_features, int64_t out_features, int blocks_per_in, int blocks_per_out, int in_group,
                                    int out_group, int64_t tokens) {
  // (an upper bound that needs no more than the layer's shape: both forms, whichever of them the index tables allow)
  int slices = 1;
  if (out_group >= 4 && out_features % 256 == 0) slices = dw_slices(dw_tiles(out_features, blocks_per_out), tokens);
  if (in_group >= 4 && in_features % 256 == 0) slices = std::max(slices, dw_slices(dw_tiles(in_features, blocks_per_in), tokens));
  return slices > 1 ? lt_align_up((size_t)slices * (size_t)(in_features / 64) * blocks_per_in * 4096 * sizeof(float), 256) : 0;
}

int lt_launch_gemm_sparse(const GemmProblem& p, int kind, int dtype, int io_dtype, hipStream_t stream) {
  if (dtype != LT_BF16 || !lt_sparse_mfma_supported(p, kind)) return lt_launch_gemm_generic(p, kind, dtype, io_dtype, stream);
  const SparseWalk& sp = p.sp;
  const double steps = sp.mode == SPARSE_FWD ? sp.blocks_per_out : sp.blocks_per_in;
  double flops = 2.0 * (double)p.M * (double)p.N * (steps * 64.0 + (p.nseg > 1 ? (double)p.K[1] : 0.0));
  if (kind == EPI_ACT_FWD && p.epi.gated) flops *= 2.0;
  if (sp.mode == SPARSE_DW) flops = 2.0 * (double)sp.tokens * (double)(p.N / 64) * sp.blocks_per_in * 4096.0;
  static const char* tags[4] = {"", "blocksparse_fwd_bf16", "blocksparse_dx_bf16", "blocksparse_dw_bf16"};
  LtProfileScope scope(tags[sp.mode], flops, 0.0, stream);
  if (sp.mode != SPARSE_DW && !lt_sparse_forward_grouped(p, kind)) return lt_launch_gemm_walk(p, kind, io_dtype, stream);
  if (kind == EPI_STORE) return lt_mfma_launch_sparse_kind0(p, stream);
  if (kind == EPI_ACT_FWD) return lt_mfma_launch_sparse_kind1(p, stream);
  LT_FAIL(LT_ERR_BAD_ARG, "block-sparse product: unknown epilogue kind %d", kind);
}

int lt_launch_gemm(const GemmProblem& p, int kind, int dtype, int io_dtype, hipStream_t stream) {
  if (lt_gemm_stream_supported(p, kind, dtype, io_dtype)) return lt_launch_gemm_stream(p, kind, dtype, io_dtype, stream);
  if (dtype == LT_BF16 && lt_gemm_mfma_supported(p, kind)) return lt_launch_gemm_mfma(p, kind, io_dtype, stream);
  return lt_launch_gemm_generic(p, kind, dtype, io_dtype, stream);
}
