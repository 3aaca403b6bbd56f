// Device-side helpers shared by the gfx950 kernels of the Doppler-moment path: complex
// arithmetic, the workgroup -> tile map and the column-blocked layout.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace hfx {

__device__ __forceinline__ float2 cmul(float2 a, float2 b) {
  return make_float2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}
// a * b with its rounding pinned (one product and one fused multiply-add per part): for
// products that must round alike in every inlined copy, whatever the compiler contracts
__device__ __forceinline__ float2 cmul_rn(float2 a, float2 b) {
  return make_float2(__fmaf_rn(a.x, b.x, -__fmul_rn(a.y, b.y)), __fmaf_rn(a.x, b.y, __fmul_rn(a.y, b.x)));
}
__device__ __forceinline__ float2 cmulc(float2 a, float2 b) {  // a * conj(b)
  return make_float2(a.x * b.x + a.y * b.y, a.y * b.x - a.x * b.y);
}
__device__ __forceinline__ float2 cadd(float2 a, float2 b) { return make_float2(a.x + b.x, a.y + b.y); }
__device__ __forceinline__ float2 csub(float2 a, float2 b) { return make_float2(a.x - b.x, a.y - b.y); }
// Bijective workgroup -> tile map that gives each of the 8 XCDs (workgroups are dispatched
// round-robin over them) a contiguous run of tiles, so neighbouring rows written into the
// column-blocked layout share an L2.
__device__ __forceinline__ int xcd_tile(int b, int n) {
  const int n8 = n & ~7;
  if (b >= n8) return b;
  return (b & 7) * (n8 >> 3) + (b >> 3);
}

// |v|^2 for the moment sums with its rounding pinned (one product, one fused multiply-add), so
// that every pass and build forms the sums from the same values
__device__ __forceinline__ float sq_mag(float2 v) { return __fmaf_rn(v.x, v.x, __fmul_rn(v.y, v.y)); }

// |X| for the moment sums: the hardware square root (v_sqrt_f32, within 1 ulp) instead of the
// correctly rounded sqrtf sequence, which costs about ten more VALU instructions per element in
// the column pass; the moments are sums over planes held to a relative tolerance, not bits.
__device__ __forceinline__ float mag_sqrt(float x) { return __builtin_amdgcn_sqrtf(x); }

// Column-blocked layout of an H x W plane with column blocks of C in {1, 2, 4}: element
// (y, x) sits at (x / C) * H * C + y * C + x % C.  For the wave-owned row x = lane + 64 m
// (C divides 64) that is blk_lane_offset(lane) + y * C + m * 64 * H, so a row store or load
// needs one shift-and-mask per lane instead of a division per element.
__device__ __forceinline__ long long blk_lane_offset(int lane, int H, int C) {
  const unsigned ul = (unsigned)lane, lc = (unsigned)__builtin_ctz((unsigned)C);
  return (long long)(ul >> lc) * H * C + (ul & (unsigned)(C - 1));
}

}  // namespace hfx
