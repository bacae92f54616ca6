// mmf_brick.hpp -- flux tuples in LDS, as the brick kernels of both orders keep
// them (device side).
#pragma once

#include "mmf_device.hpp"

namespace mmf {

// A flux tuple in LDS: field k of slot s at lds[k NS + s].
constexpr int NTUP = 11;  // c[5], vel[3], p, a, H

template <int NS>
__device__ __forceinline__ void put_tup(double *lds, int slot, const Tup &t) {
#pragma unroll
  for (int k = 0; k < NF; ++k) lds[k * NS + slot] = t.c[k];
#pragma unroll
  for (int a = 0; a < 3; ++a) lds[(5 + a) * NS + slot] = t.vel[a];
  lds[8 * NS + slot] = t.p;
  lds[9 * NS + slot] = t.a;
  lds[10 * NS + slot] = t.H;
}

template <int NS>
__device__ __forceinline__ void get_tup(const double *lds, int slot, Tup &t) {
#pragma unroll
  for (int k = 0; k < NF; ++k) t.c[k] = lds[k * NS + slot];
#pragma unroll
  for (int a = 0; a < 3; ++a) t.vel[a] = lds[(5 + a) * NS + slot];
  t.p = lds[8 * NS + slot];
  t.a = lds[9 * NS + slot];
  t.H = lds[10 * NS + slot];
}

}  // namespace mmf
