// Addresses of the band DFT along an axis (k_dft_axis_mfma): the four columns that a lane loads out
// of a contiguous [outer][n][inner] tensor.  Free of HIP headers, so that the host can walk the same
// arithmetic against the bounds of a tensor.
#pragma once

namespace hfx {

// ESZ: bytes of a sample.  VEC: inner is a multiple of four and the tensor is aligned to four
// samples (at most 16 bytes), so the four columns are one aligned access.  Column c is
// (c / inner, c % inner) of (outer, inner); `cols` = outer * inner.
template <int ESZ, bool VEC> struct AxisColumns {
  static constexpr int N = VEC ? 1 : 4;  // addresses that a lane keeps
  long long off[N];                      // bytes from the tensor to sample 0 of the column(s)
  long long step;                        // bytes from sample j to j + 1

  // Columns c0 .. c0 + 3 (c0 a multiple of four).  A lane past the last column, whose results are not
  // stored, loads the last four columns with VEC and the last one without.
  __host__ __device__ inline void init(long long c0, long long cols, int n, long long inner) {
    step = inner * ESZ;
#pragma unroll
    for (int t = 0; t < N; ++t) {
      const long long last = cols - (VEC ? 4 : 1), c = c0 + t < last ? c0 + t : last;
      const long long o = c / inner, i = c - o * inner;
      off[t] = (o * n * inner + i) * ESZ;
    }
  }
};

}  // namespace hfx
