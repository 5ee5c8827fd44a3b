// Main loop of the copy-based kernels whose wavefronts own 64 x 64 sub-tiles: 128 x 128 tiles (gemm_mid.hip), block-sparse walks
// (gemm_walk.hip).  Needs gemm_mfma_kernels.h.
//
// A step is 64 k, four groups of four matrix instructions, STAGES steps in LDS.  What bounds it: LDS (a group of 64 x 64 reads as many cycles as
// it multiplies) and the address unit, which the four wavefronts share: handed the copies of a whole stage behind the barrier, it held
// up the LDS reads and matrix instructions that followed them, whatever the number of stages in flight.  So the copies go out a
// few per group, between the matrix instructions, and fragments are read one group ahead, across the barrier:
//     groups 0, 1, 2 of step t: LDS reads of the next group, copies left of the stage begun behind the last barrier
//     wait for this wavefront's copies of step t + 1 and its LDS reads; barrier: buffer t is free, buffer t + 1 full
//     group 3: LDS reads of group 0 of step t + 1, the first copies of stage t + STAGES, into buffer t
// Measured, all copies behind the barrier against this: weight gradient [2304, 768] over 16384 75 us, 63; [3333, 1600] over 6400 112, 106;
// input-gradient walk of 41 steps, one workgroup per CU, 61 us, 34.
#pragma once

namespace {

// COPIES copy instructions per wavefront and stage, READS LDS reads per group and wavefront.
//   copy(S, t, J0, J1)   copy instructions J0 .. J1 - 1 of step t into buffer S (steps past the end: zeros)
//   load(S, kk, f)       fragments of group kk of buffer S into register set f
//   multiply(f)          the four matrix instructions on register set f
template <int STAGES, int COPIES, int READS> struct StagedLoop {
  static_assert(STAGES >= 2, "a stage to read and a stage to fill");
  // copies sent out in the groups 3, 0, 1, 2 after a barrier: with two stages in the first two of them (the next barrier waits for them
  // all), else spread evenly
  static constexpr int first_of(int part) {
    return STAGES == 2 ? (part >= 2 ? COPIES : part * ((COPIES + 1) / 2)) : part * COPIES / 4;
  }
  template <int I> using Int = std::integral_constant<int, I>;

  // ahead of step t: everything but the groups 0 .. 2 copies of step t + STAGES - 1; leaves the fragments of group 0 in set 0
  template <typename Copy, typename Load> static __device__ __forceinline__ void start(int t, Copy&& copy, Load&& load) {
    lt_static_for<STAGES - 1>([&](auto S) __attribute__((always_inline)) { copy(S, t + (int)decltype(S)::value, Int<0>{}, Int<COPIES>{}); });
    copy(Int<STAGES - 1>{}, t + STAGES - 1, Int<first_of(0)>{}, Int<first_of(1)>{});
    wait_copies_and_barrier<(STAGES - 2) * COPIES + first_of(1)>();
    load(Int<0>{}, Int<0>{}, Int<0>{});
  }
  // one step, in buffer S
  template <typename S_, typename Copy, typename Load, typename Multiply>
  static __device__ __forceinline__ void step(S_, int t, Copy&& copy, Load&& load, Multiply&& multiply) {
    constexpr int S = S_::value;
    lt_static_for<3>([&](auto KK) __attribute__((always_inline)) {
      constexpr int kk = decltype(KK)::value, c0 = first_of(kk + 1), c1 = first_of(kk + 2);
      load(S_{}, Int<kk + 1>{}, Int<(kk + 1) & 1>{});
      if constexpr (c1 > c0) copy(Int<(S + STAGES - 1) % STAGES>{}, t + STAGES - 1, Int<c0>{}, Int<c1>{});
      multiply(Int<kk & 1>{});
      SchedInterleave3<READS, c1 - c0, 4, 4>::run();
    });
    wait_copies_and_barrier<(STAGES - 2) * COPIES>();
    load(Int<(S + 1) % STAGES>{}, Int<0>{}, Int<0>{});
    copy(Int<S>{}, t + STAGES, Int<first_of(0)>{}, Int<first_of(1)>{});
    multiply(Int<1>{});
    SchedInterleave3<READS, first_of(1), 4, 4>::run();
  }
  // steps t0 .. t0 + count - 1, t0 a multiple of STAGES
  template <typename Copy, typename Load, typename Multiply>
  static __device__ __forceinline__ void run(int t0, int count, Copy&& copy, Load&& load, Multiply&& multiply) {
    int t = t0;
    for (; t + STAGES <= t0 + count; t += STAGES)
      lt_static_for<STAGES>([&](auto S) __attribute__((always_inline)) { step(S, t + decltype(S)::value, copy, load, multiply); });
    lt_static_for<STAGES - 1>([&](auto S) __attribute__((always_inline)) {
      if (t + decltype(S)::value < t0 + count) step(S, t + decltype(S)::value, copy, load, multiply);
    });
  }
};

}  // namespace
