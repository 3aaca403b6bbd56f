// Addresses of the band DFT along an axis (k_dft_axis_mfma): the four columns that a lane loads out
// of a contiguous [outer][n][inner] tensor.  Free of HIP headers, so that the host can walk the same
// arithmetic against the bounds of a tensor.
#pragma once

namespace hfx {

// A wave owns a tile of 64 columns; column c is (c / inner, c % inner) of (outer, inner), `cols` =
// outer * inner.  ESZ: bytes of a sample.  VEC: inner is a multiple of four and the tensor is aligned
// to four samples (at most 16 bytes): the four columns of lane rw (0 .. 15) are adjacent, one aligned
// access.  Otherwise they lie 16 apart, so that neighbouring lanes access neighbouring columns.
template <int ESZ, bool VEC> struct AxisColumns {
  static constexpr int N = VEC ? 1 : 4;  // addresses that a lane keeps
  long long off[N];                      // bytes from the tensor to sample 0 of the column(s)
  long long step;                        // bytes from sample j to j + 1

  __host__ __device__ static inline long long column(long long tile, int rw, int t) {
    return tile * 64 + (VEC ? 4 * rw + t : rw + 16 * t);
  }

  // A lane past the last column, whose results are not stored, loads the last four columns with VEC
  // and the last one without.
  __host__ __device__ inline void init(long long tile, int rw, long long cols, int n, long long inner) {
    step = inner * ESZ;
#pragma unroll
    for (int t = 0; t < N; ++t) {
      const long long own = column(tile, rw, t), last = cols - (VEC ? 4 : 1), c = own < last ? own : last;
      const long long o = c / inner, i = c - o * inner;
      off[t] = (o * n * inner + i) * ESZ;
    }
  }
};

}  // namespace hfx
