// Workgroup reductions of FP64 values for gfx950: DPP butterflies within a wave, one LDS exchange
// between waves, everything in a fixed order, so results are the same on every run and lane.
#pragma once
#include <hip/hip_runtime.h>

namespace mmff {

// Wave-level FP64 steps with DPP: a butterfly inside each 16-lane row
// (lane xor 1, 2, 4, 8), then the four row results are combined in a fixed order, so every
// lane gets the same value.
template <int CTRL>
__device__ __forceinline__ double dpp_d(double v) {
  // every lane reads a lane of its own row, so no lane keeps an old value
  const int lo = __builtin_amdgcn_mov_dpp(__double2loint(v), CTRL, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(v), CTRL, 0xf, 0xf, true);
  return __hiloint2double(hi, lo);
}
__device__ __forceinline__ double lane_d(double v, int lane) {
  const int lo = __builtin_amdgcn_readlane(__double2loint(v), lane);
  const int hi = __builtin_amdgcn_readlane(__double2hiint(v), lane);
  return __hiloint2double(hi, lo);
}
constexpr int DPP_QUAD_XOR1 = 0xB1, DPP_QUAD_XOR2 = 0x4E, DPP_QUAD_REV = 0x1B, DPP_ROW_HALF_MIRROR = 0x141,
              DPP_ROW_ROR8 = 0x128;
template <int CTRL>
__device__ __forceinline__ float dpp_f(float v) {
  return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), CTRL, 0xf, 0xf, true));
}

// Sums (or maxima) of K values per lane over a wave at once. At each butterfly step a lane keeps
// one of two values and sends the other to its partner, so the values left halve from step to
// step instead of each going through all steps: 69 instructions for K = 8, against 248 for
// eight separate butterflies (of 16-28 per value, a third of them DPP moves). Lane bits 0-2 end
// up selecting the value: value q is in lanes l with (l & (KP - 1)) == q. Each value's additions
// pair the same lanes in the same order as in a butterfly of its own (IEEE addition commutes), so
// the result has the same bits.
template <bool MAX>
__device__ __forceinline__ double red_op(double a, double b) {
  return MAX ? fmax(a, b) : a + b;
}
// lane l of a row receives lane l ^ X of the same row
template <int X>
__device__ __forceinline__ double row_xor(double v) {
  if constexpr (X == 1) return dpp_d<DPP_QUAD_XOR1>(v);
  if constexpr (X == 2) return dpp_d<DPP_QUAD_XOR2>(v);
  if constexpr (X == 4) return dpp_d<DPP_QUAD_REV>(dpp_d<DPP_ROW_HALF_MIRROR>(v));  // l ^ 7, then ^ 3
  return dpp_d<DPP_ROW_ROR8>(v);
}
template <int K, int X, bool MAX>
__device__ __forceinline__ void red_step(const double (&v)[K], double (&r)[(K + 1) / 2], int lane) {
  const bool up = (lane & X) != 0;
#pragma unroll
  for (int k = 0; k < K / 2; k++) {
    const double keep = up ? v[2 * k + 1] : v[2 * k], send = up ? v[2 * k] : v[2 * k + 1];
    r[k] = red_op<MAX>(keep, row_xor<X>(send));
  }
  if constexpr (K & 1) r[K / 2] = red_op<MAX>(v[K - 1], row_xor<X>(v[K - 1]));
}
// ((row 0 + row 1) + row 2) + row 3 of lane l's column, in every row
template <bool MAX>
__device__ __forceinline__ double red_rows(double v) {
  const unsigned lo = (unsigned)__double2loint(v), hi = (unsigned)__double2hiint(v);
  const auto l2 = __builtin_amdgcn_permlane32_swap(lo, lo, false, false);  // rows {0, 1} / {2, 3} in both halves
  const auto h2 = __builtin_amdgcn_permlane32_swap(hi, hi, false, false);
  const auto l01 = __builtin_amdgcn_permlane16_swap(l2[0], l2[0], false, false);
  const auto h01 = __builtin_amdgcn_permlane16_swap(h2[0], h2[0], false, false);
  const auto l23 = __builtin_amdgcn_permlane16_swap(l2[1], l2[1], false, false);
  const auto h23 = __builtin_amdgcn_permlane16_swap(h2[1], h2[1], false, false);
  const double r0 = __hiloint2double((int)h01[0], (int)l01[0]), r1 = __hiloint2double((int)h01[1], (int)l01[1]);
  const double r2 = __hiloint2double((int)h23[0], (int)l23[0]), r3 = __hiloint2double((int)h23[1], (int)l23[1]);
  return MAX ? fmax(fmax(r0, r1), fmax(r2, r3)) : ((r0 + r1) + r2) + r3;
}
// One value: its rows' results by readlane, which is shorter than the swaps when there is nothing
// to share them with
template <bool MAX>
__device__ __forceinline__ double wave_red1(double v) {
  v = red_op<MAX>(v, row_xor<1>(v));
  v = red_op<MAX>(v, row_xor<2>(v));
  v = red_op<MAX>(v, dpp_d<DPP_ROW_HALF_MIRROR>(v));
  v = red_op<MAX>(v, row_xor<8>(v));
  return red_op<MAX>(red_op<MAX>(red_op<MAX>(lane_d(v, 0), lane_d(v, 16)), lane_d(v, 32)), lane_d(v, 48));
}
// value q of v over the wave, in the lanes with (lane & 7) == q (K > 4), (lane & 3) == q (K > 2), ...
template <int K, bool MAX>
__device__ __forceinline__ double wave_red(const double (&v)[K], int lane) {
  double a[(K + 1) / 2], b[(K + 3) / 4], c[(K + 7) / 8];
  red_step<K, 1, MAX>(v, a, lane);
  red_step<(K + 1) / 2, 2, MAX>(a, b, lane);
  red_step<(K + 3) / 4, 4, MAX>(b, c, lane);
  return red_rows<MAX>(red_op<MAX>(c[0], row_xor<8>(c[0])));
}

// SLOT: LDS words per wave, a power of two that covers the values of one reduction
// EXTRA: the workgroup has more waves than NT / 64; they take part in the barriers and read the
// totals, and add nothing
template <int NT, int SLOT = 8, bool EXTRA = false>
struct Reducer {
  static constexpr int NW = NT / 64;
  double* buf;  // 2 phases * NW * SLOT doubles
  int phase;
  // K sums followed by KM maxima of v over the workgroup, at most 8 values in all: the waves'
  // results meet in LDS (lane q writes and later adds up value q, in wave order), and every
  // lane reads the totals from the lanes that hold them, as wave-uniform values.
  template <int K, int KM>
  __device__ __forceinline__ void run(double (&v)[K + KM]) {
    constexpr int KT = K + KM;
    static_assert(KT <= SLOT, "at most SLOT values per reduction");
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    if constexpr (KT == 1) {
      constexpr bool MAX = KM == 1;
      double a = wave_red1<MAX>(v[0]);
      if constexpr (NW > 1) {
        double* b = buf + phase * (NW * SLOT);
        if (lane == 0 && (!EXTRA || w < NW)) b[w * SLOT] = a;
        __syncthreads();
        a = b[0];
#pragma unroll
        for (int ww = 1; ww < NW; ww++) a = red_op<MAX>(a, b[ww * SLOT]);
        phase ^= 1;
      } else {
        __syncthreads();
      }
      v[0] = a;
      return;
    }
    double s = 0.0, x = 0.0;
    if constexpr (K > 0) {
      double t[K];
#pragma unroll
      for (int k = 0; k < K; k++) t[k] = v[k];
      s = wave_red<K, false>(t, lane);
    }
    if constexpr (KM > 0) {
      double t[KM];
#pragma unroll
      for (int k = 0; k < KM; k++) t[k] = v[K + k];
      x = wave_red<KM, true>(t, lane);
    }
    if constexpr (NW == 1) {
      __syncthreads();  // orders the wave's LDS traffic, as callers expect of a reduction
    } else {
      // sums in the words 0..K-1 of a wave's slot, maxima in K..KT-1
      double* b = buf + phase * (NW * SLOT);
      if (K > 0 && lane < K && (!EXTRA || w < NW)) b[w * SLOT + lane] = s;
      if (KM > 0 && lane < KM && (!EXTRA || w < NW)) b[w * SLOT + K + lane] = x;
      __syncthreads();
      if constexpr (K > 0) {
        const int q = lane & (SLOT - 1);
        s = b[q];
#pragma unroll
        for (int ww = 1; ww < NW; ww++) s += b[ww * SLOT + q];
      }
      if constexpr (KM > 0) {
        const int q = (K + lane) & (SLOT - 1);
        x = b[q];
#pragma unroll
        for (int ww = 1; ww < NW; ww++) x = fmax(x, b[ww * SLOT + q]);
      }
      phase ^= 1;
    }
#pragma unroll
    for (int k = 0; k < K; k++) v[k] = lane_d(s, k);
#pragma unroll
    for (int k = 0; k < KM; k++) v[K + k] = lane_d(x, k);
  }
  __device__ __forceinline__ double sum(double a) {
    double v[1] = {a};
    run<1, 0>(v);
    return v[0];
  }
  __device__ __forceinline__ double max(double a) {
    double v[1] = {a};
    run<0, 1>(v);
    return v[0];
  }
};

}  // namespace mmff
