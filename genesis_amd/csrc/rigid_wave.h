// Wavefront-wide exchanges and reductions by cross-lane moves of the vector unit (DPP row operations and the gfx950
// permlane swaps) instead of LDS permutes: a step of a butterfly is one or two moves on the register file (about 8
// cycles) instead of a round trip through the LDS unit (over 100), and the sums are chains of six such steps. With the
// last iteration's unused factor update dropped, the solve of 1,500 20-box piles went from 1,231 to 1,084 us.
#pragma once
#include <hip/hip_runtime.h>

namespace gsr {

constexpr int kWave = 64;

// LDS pointers carry their address space so every access compiles to ds_* instructions (not flat), and the compiler
// knows they never alias global memory.
#define GSR_LDS __attribute__((address_space(3)))
typedef GSR_LDS float lds_f;
typedef GSR_LDS int lds_i;
typedef GSR_LDS unsigned long long lds_u64;
typedef GSR_LDS char lds_c;

// Workgroup -> env for the one-env-per-workgroup kernels. The dispatcher deals workgroups to the 8 XCDs round-robin
// (workgroup i to XCD i % 8) and every XCD has its own L2, while the env-minor state arrays put 32 neighbouring envs
// in one 128-byte line. Within each chunk of 256 workgroups, XCD x therefore gets a run of 32 consecutive envs, so
// the waves it holds at once share their lines in its L2 instead of each XCD fetching every line. A bijection on
// [0, n): a partial last chunk is split the same way over its m workgroups.
__device__ __forceinline__ int xcd_env(int blk, int n) {
  constexpr int kRun = 32, kChunk = 8 * kRun;
  const int base = blk - blk % kChunk;
  const int m = min(kChunk, n - base);
  const int j = blk - base;
  const int q = m >> 3, r = m & 7, x = j & 7, k = j >> 3;
  return base + x * q + min(x, r) + k;
}

// DPP control words: lane i of a row of 16 reads lane i + n (shl), i - n (shr), (i + n) mod 16 (ror by 16 - n)
constexpr int kDppXor1 = 0xB1, kDppXor2 = 0x4E, kDppShl4 = 0x104, kDppShr4 = 0x114, kDppRor4 = 0x124, kDppRor8 = 0x128;

template <int kCtrl>
__device__ __forceinline__ int dpp(int v) {
  return __builtin_amdgcn_update_dpp(v, v, kCtrl, 0xf, 0xf, false);
}
template <int kCtrl>
__device__ __forceinline__ float dpp(float v) {
  return __int_as_float(dpp<kCtrl>(__float_as_int(v)));
}
template <int kCtrl>
__device__ __forceinline__ double dpp(double v) {
  return __hiloint2double(dpp<kCtrl>(__double2hiint(v)), dpp<kCtrl>(__double2loint(v)));
}
// lane i reads lane i ^ 4: banks (groups of 4 lanes) 0 and 2 of each row read 4 up, banks 1 and 3 read 4 down
__device__ __forceinline__ int dpp_xor4(int v) {
  const int up = __builtin_amdgcn_update_dpp(v, v, kDppShl4, 0xf, 0x5, false);
  return __builtin_amdgcn_update_dpp(up, v, kDppShr4, 0xf, 0xa, false);
}
__device__ __forceinline__ float dpp_xor4(float v) { return __int_as_float(dpp_xor4(__float_as_int(v))); }

// Both values a lane and its partner 16 (32) lanes away hold, in the same order on both: the butterfly's operands
template <int kDist>
__device__ __forceinline__ void swap_pair(int v, int& a, int& b) {
  static_assert(kDist == 16 || kDist == 32, "row or half swap");
  if constexpr (kDist == 32) {
    const auto r = __builtin_amdgcn_permlane32_swap((unsigned)v, (unsigned)v, false, false);
    a = (int)r[0];
    b = (int)r[1];
  } else {
    const auto r = __builtin_amdgcn_permlane16_swap((unsigned)v, (unsigned)v, false, false);
    a = (int)r[0];
    b = (int)r[1];
  }
}
template <int kDist>
__device__ __forceinline__ void swap_pair(float v, float& a, float& b) {
  int x, y;
  swap_pair<kDist>(__float_as_int(v), x, y);
  a = __int_as_float(x);
  b = __int_as_float(y);
}
template <int kDist>
__device__ __forceinline__ void swap_pair(double v, double& a, double& b) {
  int xl, yl, xh, yh;
  swap_pair<kDist>(__double2loint(v), xl, yl);
  swap_pair<kDist>(__double2hiint(v), xh, yh);
  a = __hiloint2double(xh, xl);
  b = __hiloint2double(yh, yl);
}

// Butterfly over the wavefront, distances 32, 16, 8, 4, 2, 1; every lane gets the result. After the steps 32, 16 and 8
// a value depends only on the lane's low three bits, so a rotation by 4 in the row reads the partner 4 lanes away.
template <class T, class Op>
__device__ __forceinline__ T wave_reduce(T v, Op op) {
  T a, b;
  swap_pair<32>(v, a, b);
  v = op(a, b);
  swap_pair<16>(v, a, b);
  v = op(a, b);
  v = op(v, dpp<kDppRor8>(v));
  v = op(v, dpp<kDppRor4>(v));
  v = op(v, dpp<kDppXor2>(v));
  return op(v, dpp<kDppXor1>(v));
}
// Sums over rows or dofs whose rounding steers discrete decisions (the line search's bracketing, the Newton stop
// test) are accumulated in double: the reference adds them one by one in FP32, an order a wavefront cannot follow,
// and a tree of FP32 partial sums has a different rounding error; the double sum is closer to both.
__device__ __forceinline__ double wave_sum_d(double v) {
  return wave_reduce(v, [](double a, double b) { return a + b; });
}
__device__ __forceinline__ int wave_or(int v) {
  return wave_reduce(v, [](int a, int b) { return a | b; });
}
__device__ __forceinline__ int wave_sum_i(int v) {
  return wave_reduce(v, [](int a, int b) { return a + b; });
}
__device__ __forceinline__ int wave_min_i(int v) {
  return wave_reduce(v, [](int a, int b) { return a < b ? a : b; });
}

// value of lane `l` (the same l on every lane) as a scalar
__device__ __forceinline__ int lane_value(int v, int l) { return __builtin_amdgcn_readlane(v, l); }
__device__ __forceinline__ float lane_value(float v, int l) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l));
}
__device__ __forceinline__ unsigned long long lane_value(unsigned long long v, int l) {
  const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)v, l);
  const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)(v >> 32), l);
  return ((unsigned long long)hi << 32) | lo;
}

// Sum over the aligned group of G lanes (a power of two, the same on every lane) holding this lane, on every lane of
// the group: distances G / 2, ..., 1
__device__ __forceinline__ float group_sum(float v, int G) {
  float a, b;
  if (G > 32) {
    swap_pair<32>(v, a, b);
    v = a + b;
  }
  if (G > 16) {
    swap_pair<16>(v, a, b);
    v = a + b;
  }
  if (G > 8) v += dpp<kDppRor8>(v);
  if (G > 4) v += dpp_xor4(v);
  if (G > 2) v += dpp<kDppXor2>(v);
  if (G > 1) v += dpp<kDppXor1>(v);
  return v;
}

}  // namespace gsr
