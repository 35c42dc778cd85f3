// ekm_scan.h -- wavefront scans of affine maps, the building block of the
// batched tridiagonal solves with one wavefront per line (ekm_mgt.hip,
// ekm_sep.hip).
#pragma once
#include <hip/hip_runtime.h>

namespace {

// affine map x -> a*x + b; compose(outer, inner) = outer(inner(x))
template <typename T>
struct Aff {
  T a, b;
};
template <typename T>
__device__ inline Aff<T> compose(const Aff<T>& o, const Aff<T>& i) {
  return Aff<T>{o.a * i.a, o.a * i.b + o.b};
}

// Cross-lane moves of the wavefront scans.  dpp<CTRL, RM>(old, v): v of the
// lane that the DPP control CTRL names, or `old` where that lane lies outside
// the row or the row is masked out by RM (row_shr:n = 0x110+n, row_shl:n =
// 0x100+n, row_bcast:15 = 0x142, row_bcast:31 = 0x143; 64-bit values move as
// two 32-bit halves).
template <int CTRL, int RM, typename T>
__device__ inline T dpp(T old, T v) {
  if constexpr (sizeof(T) == 4) {
    return __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(old), __float_as_int(v), CTRL, RM, 0xf, false));
  } else {
    const long long o = __double_as_longlong(old), x = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_update_dpp((int)o, (int)x, CTRL, RM, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp((int)(o >> 32), (int)(x >> 32), CTRL, RM, 0xf, false);
    return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
  }
}
template <typename T>
__device__ inline T rdlane(T v, int l) {
  if constexpr (sizeof(T) == 4) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l));
  } else {
    const long long x = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_readlane((int)x, l), hi = __builtin_amdgcn_readlane((int)(x >> 32), l);
    return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
  }
}
template <int CTRL, int RM, typename T>
__device__ inline Aff<T> dpp_aff(const Aff<T>& v) {
  return Aff<T>{dpp<CTRL, RM>((T)1, v.a), dpp<CTRL, RM>((T)0, v.b)};
}

// inclusive scan over the lanes in increasing order: lane i gets
// map_i o map_{i-1} o ... o map_0 (in-row doubling steps, then the row
// prefixes carried by row_bcast:15 to rows 1 and 3 and row_bcast:31 to rows
// 2 and 3)
template <typename T>
__device__ inline Aff<T> wave_scan_up(Aff<T> v) {
  v = compose(v, dpp_aff<0x111, 0xf>(v));
  v = compose(v, dpp_aff<0x112, 0xf>(v));
  v = compose(v, dpp_aff<0x114, 0xf>(v));
  v = compose(v, dpp_aff<0x118, 0xf>(v));
  v = compose(v, dpp_aff<0x142, 0xa>(v));
  v = compose(v, dpp_aff<0x143, 0xc>(v));
  return v;
}

// inclusive scan in decreasing order: lane i gets map_i o ... o map_63
// (in-row doubling steps, then the suffix maps of the rows above, read from
// the first lane of each row)
template <typename T>
__device__ inline Aff<T> wave_scan_down(Aff<T> v) {
  v = compose(v, dpp_aff<0x101, 0xf>(v));
  v = compose(v, dpp_aff<0x102, 0xf>(v));
  v = compose(v, dpp_aff<0x104, 0xf>(v));
  v = compose(v, dpp_aff<0x108, 0xf>(v));
  const Aff<T> r1{rdlane(v.a, 16), rdlane(v.b, 16)};
  const Aff<T> r2{rdlane(v.a, 32), rdlane(v.b, 32)};
  const Aff<T> r3{rdlane(v.a, 48), rdlane(v.b, 48)};
  const Aff<T> s2 = r3, s1 = compose(r2, r3), s0 = compose(r1, s1);
  const int row = (threadIdx.x & 63) >> 4;
  const Aff<T> tail = row == 0 ? s0 : row == 1 ? s1 : row == 2 ? s2 : Aff<T>{(T)1, (T)0};
  return compose(v, tail);
}

}  // namespace
