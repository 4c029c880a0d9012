// Exchanges and reductions within a wave (64 lanes) by DPP moves and
// v_readlane, without LDS.
#pragma once

#include <hip/hip_runtime.h>

namespace sylver_amd {

// v from another lane by a DPP control; lanes without a source keep v.
template <int CTRL>
__device__ __forceinline__ int dpp(int v) {
   return __builtin_amdgcn_update_dpp(v, v, CTRL, 0xf, 0xf, false);
}
template <int CTRL>
__device__ __forceinline__ float dpp(float v) {
   return __int_as_float(dpp<CTRL>(__float_as_int(v)));
}
template <int CTRL>
__device__ __forceinline__ double dpp(double v) {
   const long long u = __double_as_longlong(v);
   const int lo = dpp<CTRL>((int)(u & 0xffffffff)), hi = dpp<CTRL>((int)(u >> 32));
   return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}

// v of lane `lane` (uniform) as a scalar.
__device__ __forceinline__ int lane_value(int v, int lane) { return __builtin_amdgcn_readlane(v, lane); }
__device__ __forceinline__ float lane_value(float v, int lane) {
   return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane));
}
__device__ __forceinline__ double lane_value(double v, int lane) {
   const long long u = __double_as_longlong(v);
   const int lo = __builtin_amdgcn_readlane((int)(u & 0xffffffff), lane);
   const int hi = __builtin_amdgcn_readlane((int)(u >> 32), lane);
   return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}

// v, the same in every active lane, as a scalar.
__device__ __forceinline__ double uniform_value(double v) {
   const long long u = __double_as_longlong(v);
   const int lo = __builtin_amdgcn_readfirstlane((int)(u & 0xffffffff));
   const int hi = __builtin_amdgcn_readfirstlane((int)(u >> 32));
   return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}

// Reduction over the wave by `op` (associative, idempotent): row scans, then
// the rows' last lanes onward; lane 63 ends with the result.
template <typename V, typename Op>
__device__ __forceinline__ V wave_reduce(V v, Op op) {
   v = op(v, dpp<0x111>(v));  // row_shr:1
   v = op(v, dpp<0x112>(v));
   v = op(v, dpp<0x114>(v));
   v = op(v, dpp<0x118>(v));
   v = op(v, dpp<0x142>(v));  // row_bcast:15
   v = op(v, dpp<0x143>(v));  // row_bcast:31
   return lane_value(v, 63);
}

}  // namespace sylver_amd
