// Optional in-path stages: the Filter2D band-pass table, the Flatfield Gaussian high-pass
// (Fourier table and the spatial separable form).
//
// Both spectral stages run on the shared 2-D FFT passes (row pass, column pass with the table
// multiplied between its forward and inverse transforms, inverse row pass); these kernels
// build their tables, in the column-blocked layout those passes read:
//   (r, c) -> (c / blk_c) * H * blk_c + r * blk_c + c % blk_c.
#include "hfx_kernels.hh"

namespace hfx {

namespace {

constexpr float kPiF = 3.14159265358979f;

__device__ __forceinline__ long long tab_index(int r, int c, int H, int W, int blk_c) {
  return blk_c > 0 ? (long long)(c / blk_c) * H * blk_c + (long long)r * blk_c + (c % blk_c)
                   : (long long)r * W + c;
}

// Cosine-tapered edge of the annulus (filter2d.cu:165-240): 1 inside radius r, a quarter
// cosine over the next s pixels, 0 beyond.  `q` is the squared distance scaled by `k2`
// (4 for the half-integer centred grid, 1 for the integer grid), so that the comparisons
// against r and r + s are exact integer tests; the taper itself is evaluated in FP32.
__device__ __forceinline__ float taper(long long q, int k2, float dist, int r, int s) {
  if (q < (long long)k2 * r * r) return 1.0f;
  const long long rs = (long long)r + s;
  if (s > 0 && q < (long long)k2 * rs * rs)
    return cosf((dist - (float)r) / (float)s * kPiF / 2);
  return 0.0f;
}

}  // namespace

// Filter2D table (filter2d.cu:165-305).
//   complex input: the annulus a(1-b) around the grid centre (W/2.0, H/2.0), stored after the
//     quadrant exchange of the four corners (DC to index 0 for even sizes), with the value
//     in both the real and the imaginary part, as the reference's table holds it;
//   real input: the annulus around DC on the integer frequency grid (|kx|, signed ky), real.
// Every table entry is the one the reference's kernels write for that frequency; the real
// input's half spectrum is extended to the full grid through |kx|.
__global__ void k_filter2d_table(float2 *out, int H, int W, int r_in, int r_out, int s_in, int s_out,
                                 int complex_mode, int blk_c) {
  const int c = blockIdx.x * blockDim.x + threadIdx.x;
  const int r = blockIdx.y;
  if (c >= W || r >= H) return;
  long long q;
  int k2;
  if (complex_mode) {
    // position before the corner exchange (only the 2*(W/2) x 2*(H/2) block moves)
    const int hw = W / 2, hh = H / 2;
    int rs = r, cs = c;
    if (r < 2 * hh && c < 2 * hw) {
      rs = r < hh ? r + hh : r - hh;
      cs = c < hw ? c + hw : c - hw;
    }
    const long long x2 = 2LL * cs - W, y2 = 2LL * rs - H;  // twice the centred coordinates
    q = x2 * x2 + y2 * y2;
    k2 = 4;
  } else {
    const long long kx = c <= W / 2 ? c : W - c;
    const long long ky = r <= H / 2 ? r : r - H;
    q = kx * kx + ky * ky;
    k2 = 1;
  }
  const float dist = (float)(sqrt((double)q) / (k2 == 4 ? 2.0 : 1.0));
  const float a = taper(q, k2, dist, r_out, s_out);
  const float b = taper(q, k2, dist, r_in, s_in);
  const float m = a * (1 - b);
  out[tab_index(r, c, H, W, blk_c)] = make_float2(m, complex_mode ? m : 0.0f);
}

void launch_filter2d_table(float2 *out, int H, int W, int r_in, int r_out, int s_in, int s_out,
                           int complex_mode, int blk_c, hipStream_t st) {
  hipLaunchKernelGGL(k_filter2d_table, dim3((W + 127) / 128, H), dim3(128), 0, st, out, H, W, r_in, r_out,
                     s_in, s_out, complex_mode, blk_c);
}

// Flatfield Gaussian high-pass in the Fourier domain (flatfield.cu:143-180):
//   gain(kx, ky) = (1 - exp(-2 pi^2 (sx^2 fx^2 + sy^2 fy^2))) * scale,
//   fx = |kx| / W, fy = signed ky / H, real; evaluated in FP32 as the reference does.
__global__ void k_flatfield_table(float2 *out, int H, int W, float sigma_y, float sigma_x, float scale,
                                  int blk_c) {
  const int c = blockIdx.x * blockDim.x + threadIdx.x;
  const int r = blockIdx.y;
  if (c >= W || r >= H) return;
  const int kx = c <= W / 2 ? c : W - c;
  const float fx = (float)kx / (float)W;
  const float fy_idx = r <= H / 2 ? (float)r : (float)(r - H);
  const float fy = fy_idx / (float)H;
  const float two_pi_squared = 19.739208802178716f;
  const float lowpass = expf(-two_pi_squared * (sigma_x * sigma_x * fx * fx + sigma_y * sigma_y * fy * fy));
  out[tab_index(r, c, H, W, blk_c)] = make_float2((1.0f - lowpass) * scale, 0.0f);
}

void launch_flatfield_table(float2 *out, int H, int W, float sigma_y, float sigma_x, float scale, int blk_c,
                            hipStream_t st) {
  hipLaunchKernelGGL(k_flatfield_table, dim3((W + 127) / 128, H), dim3(128), 0, st, out, H, W, sigma_y,
                     sigma_x, scale, blk_c);
}

// Flatfield, spatial form (flatfield.cu:189-240): background = Gaussian blur with clamp-at-
// edge indexing, horizontal along x then vertical along y, out = in - background; the taps
// are summed in ascending order with fused multiply-adds.
//
// One block owns a TY x FF_TX tile of one plane: it stages the tile and its clamped halo in LDS,
// blurs the halo rows horizontally in place (a row's threads are lanes of one wave, which has read
// its row before it writes), then blurs vertically and subtracts from the input (read again: an
// L2 hit), so each input element is read from HBM about once.
//
// Bound by VALU and LDS latency in short loops (three 1024 x 1024 images): each thread
// blurs four neighbours at once out of a register window (one 16-byte read per four taps and four
// outputs along x, one 4-byte read per tap and four outputs along y), the next step's reads are
// issued ahead, the loads of four rows are in flight together, and the one buffer lets eight
// blocks share a CU at sigma 3: 30 -> 19 us.  The sums keep their order.
constexpr int FF_TX = 64, FF_RMAX = 31, FF_NT = 256;

// The tile buffer is sized for the actual radii (dynamic LDS): a row of the tile and halo, padded to
// whole 16-byte groups with two groups beyond the last tap's window.
__host__ __device__ constexpr int ff_pitch(int rx) { return (FF_TX + 2 * rx + 12 + 3) / 4 * 4; }
__host__ __device__ constexpr size_t ff_spatial_lds_bytes(int ty, int rx, int ry) {
  return (size_t)(ty + 2 * ry + 4) * ff_pitch(rx) * sizeof(float);
}

// one tap w on four neighbouring outputs
__device__ __forceinline__ void ff_tap(float (&s)[4], float x0, float x1, float x2, float x3, float w) {
  s[0] = fmaf(x0, w, s[0]);
  s[1] = fmaf(x1, w, s[1]);
  s[2] = fmaf(x2, w, s[2]);
  s[3] = fmaf(x3, w, s[3]);
}

template <int TY>
__global__ __launch_bounds__(FF_NT) void k_flatfield_spatial(const float *__restrict__ in, float *__restrict__ out,
                                                              int H, int W, const float *__restrict__ kx, int rx,
                                                              const float *__restrict__ ky, int ry) {
  extern __shared__ float4 ff_lds[];
  __shared__ __align__(16) float wx[68], wy[68];
  const int tid = threadIdx.x;
  const int x0 = blockIdx.x * FF_TX, y0 = blockIdx.y * TY;
  const long long base = (long long)blockIdx.z * H * W;
  const int rows = TY + 2 * ry, pitch = ff_pitch(rx);
  const int fx = (2 * rx + 1) / 4, fy = (2 * ry + 1) / 4;  // whole groups of four taps
  float *buf = reinterpret_cast<float *>(ff_lds);  // [rows + 4][pitch]; the last four rows pad the window reads
  // four rows per wave and step, all their loads in flight (a loop of one load each, with a division
  // by the pitch, was the longest part of the kernel)
  for (int i = tid; i < 68; i += FF_NT) {
    wx[i] = i <= 2 * rx ? kx[i] : 0.f;
    wy[i] = i <= 2 * ry ? ky[i] : 0.f;
  }
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  unsigned xo[3];  // (the padding repeats the last pixel, unused)
#pragma unroll
  for (int c = 0; c < 3; ++c) xo[c] = (unsigned)min(max(x0 - rx + lane + 64 * c, 0), W - 1);
  for (int r = wave; r < rows; r += 16) {
    float t[4][3];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int y = min(max(y0 - ry + min(r + 4 * u, rows - 1), 0), H - 1);
      const float *src = in + base + (long long)y * W;
#pragma unroll
      for (int c = 0; c < 3; ++c)
        if (64 * c < pitch) t[u][c] = src[xo[c]];
    }
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
      for (int c = 0; c < 3; ++c)
        if (lane + 64 * c < pitch && r + 4 * u < rows) buf[(r + 4 * u) * pitch + lane + 64 * c] = t[u][c];
  }
  __syncthreads();
  for (int i = tid; i < rows * (FF_TX / 4); i += FF_NT) {
    const int rr = i / (FF_TX / 4), c = 4 * (i % (FF_TX / 4));
    float4 *row = reinterpret_cast<float4 *>(buf + rr * pitch + c);
    const float4 *taps = reinterpret_cast<const float4 *>(wx);
    float s[4] = {0.f, 0.f, 0.f, 0.f};
    // four taps on the window a b (eight values)
    auto four = [&](const float4 &a, const float4 &b, const float4 &w) {
      ff_tap(s, a.x, a.y, a.z, a.w, w.x);
      ff_tap(s, a.y, a.z, a.w, b.x, w.y);
      ff_tap(s, a.z, a.w, b.x, b.y, w.z);
      ff_tap(s, a.w, b.x, b.y, b.z, w.w);
    };
    float4 v0 = row[0], v1 = row[1];
    int g = 0;  // groups of four taps; two per turn, the window's registers trading places
    for (; g + 2 <= fx; g += 2) {
      const float4 w0 = taps[g], w1 = taps[g + 1], v2 = row[g + 2], v3 = row[g + 3];
      four(v0, v1, w0);
      four(v1, v2, w1);
      v0 = v2;
      v1 = v3;
    }
    if (g < fx) {
      four(v0, v1, taps[g]);
      v0 = v1;
      v1 = row[g + 2];
    }
    // the last one or three taps (2 rx + 1 is odd)
    const float4 w = taps[fx];
    ff_tap(s, v0.x, v0.y, v0.z, v0.w, w.x);
    if (2 * rx + 1 - 4 * fx == 3) {
      ff_tap(s, v0.y, v0.z, v0.w, v1.x, w.y);
      ff_tap(s, v0.z, v0.w, v1.x, v1.y, w.z);
    }
    __builtin_amdgcn_wave_barrier();  // in place: no lane of the row writes before all have read
    row[0] = make_float4(s[0], s[1], s[2], s[3]);
  }
  __syncthreads();
  for (int i = tid; i < (TY / 4) * FF_TX; i += FF_NT) {
    const int r4 = 4 * (i / FF_TX), cc = i % FF_TX;
    const int x = x0 + cc;
    const float *col = buf + r4 * pitch + cc;
    const float4 *taps = reinterpret_cast<const float4 *>(wy);
    float own[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) own[j] = in[base + (long long)min(y0 + r4 + j, H - 1) * W + min(x, W - 1)];
    float s[4] = {0.f, 0.f, 0.f, 0.f};
    float a0 = col[0], a1 = col[pitch], a2 = col[2 * pitch];
    col += 3 * pitch;
    for (int g = 0; g < fy; ++g, col += 4 * pitch) {
      const float4 w = taps[g];
      const float b0 = col[0], b1 = col[pitch], b2 = col[2 * pitch], b3 = col[3 * pitch];
      ff_tap(s, a0, a1, a2, b0, w.x);
      ff_tap(s, a1, a2, b0, b1, w.y);
      ff_tap(s, a2, b0, b1, b2, w.z);
      ff_tap(s, b0, b1, b2, b3, w.w);
      a0 = b1;
      a1 = b2;
      a2 = b3;
    }
    const float4 w = taps[fy];
    const float b0 = col[0];
    ff_tap(s, a0, a1, a2, b0, w.x);
    if (2 * ry + 1 - 4 * fy == 3) {
      const float b1 = col[pitch], b2 = col[2 * pitch];
      ff_tap(s, a1, a2, b0, b1, w.y);
      ff_tap(s, a2, b0, b1, b2, w.z);
    }
    if (x >= W) continue;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int y = y0 + r4 + j;
      if (y < H) out[base + (long long)y * W + x] = own[j] - s[j];
    }
  }
}

// Radii beyond the LDS tile's halo (only on one-pixel-wide or -tall planes, where the
// Fourier form is not used): the same sums as two global passes through `tmp`.
__global__ void k_flatfield_rows(const float *__restrict__ in, float *__restrict__ tmp, long long total, int H,
                                 int W, const float *__restrict__ kx, int rx) {
  const long long idx = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= total) return;
  const long long plane = (long long)H * W;
  const long long base = idx / plane * plane;
  const int local = (int)(idx - base), y = local / W, x = local - y * W;
  float s = 0.0f;
  for (int k = -rx; k <= rx; ++k) s = fmaf(in[base + (long long)y * W + min(max(x + k, 0), W - 1)], kx[k + rx], s);
  tmp[idx] = s;
}

__global__ void k_flatfield_cols(const float *__restrict__ in, const float *__restrict__ tmp,
                                 float *__restrict__ out, long long total, int H, int W,
                                 const float *__restrict__ ky, int ry) {
  const long long idx = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= total) return;
  const long long plane = (long long)H * W;
  const long long base = idx / plane * plane;
  const int local = (int)(idx - base), y = local / W, x = local - y * W;
  float b = 0.0f;
  for (int k = -ry; k <= ry; ++k) b = fmaf(tmp[base + (long long)min(max(y + k, 0), H - 1) * W + x], ky[k + ry], b);
  out[idx] = in[idx] - b;
}

bool flatfield_spatial_fused(int rx, int ry) { return rx <= FF_RMAX && ry <= FF_RMAX; }

int launch_flatfield_spatial(const float *in, float *out, float *tmp, long long planes, int H, int W,
                             const float *kx, int rx, const float *ky, int ry, hipStream_t st) {
  if (flatfield_spatial_fused(rx, ry)) {
    if (planes > 65535) return -1;
    // 32 rows per tile halve the halo's share of the horizontal blur; 16 where the radii would take
    // the tile past 64 KB, or where the image gives too few tiles for the chip
    const long long tiles = planes * ((W + FF_TX - 1) / FF_TX) * ((H + 31) / 32);
    const unsigned gx = (unsigned)((W + FF_TX - 1) / FF_TX), gz = (unsigned)planes;
    if (ff_spatial_lds_bytes(32, rx, ry) <= 65536 && tiles >= 512)
      hipLaunchKernelGGL(k_flatfield_spatial<32>, dim3(gx, (H + 31) / 32, gz), dim3(FF_NT),
                         ff_spatial_lds_bytes(32, rx, ry), st, in, out, H, W, kx, rx, ky, ry);
    else
      hipLaunchKernelGGL(k_flatfield_spatial<16>, dim3(gx, (H + 15) / 16, gz), dim3(FF_NT),
                         ff_spatial_lds_bytes(16, rx, ry), st, in, out, H, W, kx, rx, ky, ry);
  } else {
    if (!tmp) return -1;
    const long long total = planes * H * W;
    const unsigned grid = (unsigned)((total + 255) / 256);
    hipLaunchKernelGGL(k_flatfield_rows, dim3(grid), dim3(256), 0, st, in, tmp, total, H, W, kx, rx);
    hipLaunchKernelGGL(k_flatfield_cols, dim3(grid), dim3(256), 0, st, in, tmp, out, total, H, W, ky, ry);
  }
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

}  // namespace hfx
