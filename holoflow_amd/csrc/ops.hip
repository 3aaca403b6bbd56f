// Stand-alone element-wise ops backing the per-node kinds of the path (the fused
// moment path does not use them):
//   fftshift  : out[i] = in[(i + n/2) mod n] on the selected axes (fftshift.cu:110-145)
//   moments   : mean over the plane axis of |x| (complex) or x (real magnitudes), with
//               optional f_k / f_k^2 weights (mean_abs.cu:239-276, mean.cu:268-306,
//               multiply.cu:69-92 wired by graph_builder.cc:612-631)
//   convert   : uint16 -> float32 or complex64 (x + 0i) (conversion.cu:156-202)
#include <mutex>
#include <type_traits>

#include "hfx_kernels.hh"

#include "axis_columns.hh"

namespace hfx {

struct ShiftGeo {
  int ndim;
  long long shape[8];
  long long stride[8];
  long long shift[8];
  long long total;
};

__global__ void k_fftshift(const uint8_t *in, uint8_t *out, int esz, ShiftGeo g) {
  long long tid = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (tid >= g.total) return;
  long long rem = tid, src = 0;
  for (int k = 0; k < g.ndim; ++k) {
    long long idx = g.stride[k] > 0 ? rem / g.stride[k] : 0;
    rem -= idx * g.stride[k];
    long long si = idx + g.shift[k];
    if (si >= g.shape[k]) si -= g.shape[k];
    src += si * g.stride[k];
  }
  if (esz == 4) {
    reinterpret_cast<uint32_t *>(out)[tid] = reinterpret_cast<const uint32_t *>(in)[src];
  } else if (esz == 8) {
    reinterpret_cast<uint2 *>(out)[tid] = reinterpret_cast<const uint2 *>(in)[src];
  } else {
    for (int b = 0; b < esz; ++b) out[tid * esz + b] = in[src * esz + b];
  }
}

// fftshift of [batch][rows][units] with units of U bytes (the largest of 16, 8, 4 that the row, its
// half and both buffers are multiples of): no index division, one 16-byte copy per lane.  A block's
// lanes spread over units, rows and images as the sizes fill them.  1024 x 1024 F32: 5.7 us with one
// division per axis and element, 3.3 us here; 262,140 rows of 8 F32: 7.7 and 3.6 (64
// lanes along every row: 30); 65,535 images of 4 x 4: 5.9 and 3.0 (30).
template <typename V>
__global__ __launch_bounds__(256) void k_fftshift_rows(const V *__restrict__ in, V *__restrict__ out, int batch,
                                                       int rows, int units, int row_shift, int unit_shift) {
  const int u = blockIdx.x * blockDim.x + threadIdx.x, r = blockIdx.y * blockDim.y + threadIdx.y;
  const int b = blockIdx.z * blockDim.z + threadIdx.z;
  if (u >= units || r >= rows || b >= batch) return;
  const long long base = (long long)b * rows * units;
  int sr = r + row_shift, su = u + unit_shift;
  if (sr >= rows) sr -= rows;
  if (su >= units) su -= units;
  out[base + (long long)r * units + u] = in[base + (long long)sr * units + su];
}

// The shift as [batch][rows][row bytes] when at most two adjacent axes are shifted: unshifted
// trailing axes widen the element, unshifted leading axes are the batch.  False: another form.
static bool launch_fftshift_rows(const void *in, void *out, int elem_size, int ndim, const long long *shape,
                                 const int *mask, hipStream_t st) {
  long long esz = elem_size, rows = 1, batch = 1;
  int k = ndim - 1;
  while (k > 0 && !mask[k]) esz *= shape[k--];
  const long long w = shape[k];
  const long long wbytes = w * esz, half = mask[k] ? w / 2 * esz : 0;
  long long row_shift = 0;
  if (k > 0 && mask[k - 1]) {
    rows = shape[--k];
    row_shift = rows / 2;
  }
  while (--k >= 0) {
    if (mask[k]) return false;
    batch *= shape[k];
  }
  const uintptr_t align = reinterpret_cast<uintptr_t>(in) | reinterpret_cast<uintptr_t>(out) | (uintptr_t)wbytes | (uintptr_t)half;
  const int u = align % 16 == 0 ? 16 : align % 8 == 0 ? 8 : align % 4 == 0 ? 4 : 0;
  if (u == 0) return false;
  if (rows == 1) {  // only rows: the batch takes their place
    rows = batch;
    batch = 1;
  }
  const long long units = wbytes / u;
  // the lanes of a block: 64 along a row, fewer where it is shorter, then rows, then images
  unsigned bx = 64, by = 4, bz = 1;
  while (bx / 2 >= units) bx /= 2, by *= 2;
  while (by / 2 >= rows) by /= 2, bz *= 2;
  while (bz / 2 >= batch) bz /= 2, bx *= 2;
  const long long gx = (units + bx - 1) / bx, gy = (rows + by - 1) / by, gz = (batch + bz - 1) / bz;
  if (units >= (1LL << 31) || rows >= (1LL << 31) || batch >= (1LL << 31) || gy > 65535 || gz > 65535) return false;
  const dim3 grid((unsigned)gx, (unsigned)gy, (unsigned)gz), block(bx, by, bz);
  const int us = (int)(half / u);
  auto go = [&](auto v) {
    using V = decltype(v);
    hipLaunchKernelGGL(k_fftshift_rows<V>, grid, block, 0, st, reinterpret_cast<const V *>(in),
                       reinterpret_cast<V *>(out), (int)batch, (int)rows, (int)units, (int)row_shift, us);
  };
  u == 16 ? go(uint4{}) : u == 8 ? go(uint2{}) : go(uint32_t{});
  return true;
}

int launch_fftshift(const void *in, void *out, int elem_size, int ndim, const long long *shape,
                    const int *mask, hipStream_t st) {
  if (ndim < 1 || ndim > 8) return -1;
  ShiftGeo g;
  g.ndim = ndim;
  long long acc = 1;
  for (int k = ndim - 1; k >= 0; --k) {
    g.shape[k] = shape[k];
    g.stride[k] = acc;
    g.shift[k] = mask[k] ? shape[k] / 2 : 0;
    acc *= shape[k];
  }
  g.total = acc;
  if (acc == 0) return 0;
  if (!launch_fftshift_rows(in, out, elem_size, ndim, shape, mask, st))
    hipLaunchKernelGGL(k_fftshift, dim3((unsigned)((acc + 255) / 256)), dim3(256), 0, st,
                       reinterpret_cast<const uint8_t *>(in), reinterpret_cast<uint8_t *>(out), elem_size, g);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

// Mean over the plane axis of m_k(p) = |x| (complex), x or |x| (real), or its square, weighted by
// w_k when WEIGHTED; products rounded before the ascending sum.  V pixels per lane (16-byte
// loads), planes in groups of J whose loads are in flight together: three reductions of
// [15][1024^2] F32, 63 MB each in the last-level cache, 15.8 -> 12.7 us each.
template <bool CPLX, bool WEIGHTED, int V, int J>
__global__ __launch_bounds__(256) void k_weighted_mean(const float *__restrict__ in, const float *__restrict__ w,
                                                       float *__restrict__ out, long long planes, long long npix,
                                                       int power2, int absval) {
  const long long p = ((long long)blockIdx.x * 256 + threadIdx.x) * V;
  if (p >= npix) return;
  constexpr int C = CPLX ? 2 : 1, NV = V * C;
  typedef float vec __attribute__((ext_vector_type(NV)));
  float s[V];
#pragma unroll
  for (int t = 0; t < V; ++t) s[t] = 0.f;
  auto add = [&](const vec &x, long long k) {
#pragma unroll
    for (int t = 0; t < V; ++t) {
      float m;
      if constexpr (CPLX) {
        const float re = x[2 * t], im = x[2 * t + 1];
        m = re * re + im * im;
        if (!power2) m = sqrtf(m);
      } else {
        if constexpr (NV == 1)
          m = x[0];
        else
          m = x[t];
        m = power2 ? m * m : (absval ? fabsf(m) : m);
      }
      s[t] += WEIGHTED ? __fmul_rn(w[k], m) : m;
    }
  };
  const float *src = in + p * C;
  const long long step = npix * C;
  long long k = 0;
  for (; k + J <= planes; k += J) {
    vec x[J];
#pragma unroll
    for (int j = 0; j < J; ++j) x[j] = *reinterpret_cast<const vec *>(src + (k + j) * step);
#pragma unroll
    for (int j = 0; j < J; ++j) add(x[j], k + j);
  }
  if (k < planes) {  // the rest, with planes past the end loading the last one, unused
    vec x[J];
#pragma unroll
    for (int j = 0; j < J; ++j) x[j] = *reinterpret_cast<const vec *>(src + (k + j < planes ? k + j : planes - 1) * step);
#pragma unroll
    for (int j = 0; j < J; ++j)
      if (k + j < planes) add(x[j], k + j);
  }
  const float n = (float)planes;
#pragma unroll
  for (int t = 0; t < V; ++t) s[t] = s[t] / n;
  if constexpr (V == 4)
    *reinterpret_cast<float4 *>(out + p) = make_float4(s[0], s[1], s[2], s[3]);
  else if constexpr (V == 2)
    *reinterpret_cast<float2 *>(out + p) = make_float2(s[0], s[1]);
  else
    out[p] = s[0];
}

template <bool CPLX, bool WEIGHTED>
static void launch_mean(const float *in, const float *w, float *out, long long planes, long long npix, int power2,
                        int absval, hipStream_t st) {
  constexpr int V = CPLX ? 2 : 4;
  // wide loads need aligned planes, and pay only when the wider lanes still fill the chip
  const uintptr_t align = reinterpret_cast<uintptr_t>(in) % 16 + reinterpret_cast<uintptr_t>(out) % (4 * V);
  const bool wide = align == 0 && npix % V == 0 && npix / V >= 65536;
  const dim3 block(256);
  // Complex planes that stay in the 256 MiB last-level cache: two planes in flight per lane.  Eight
  // walk eight planes at once, which the cache serves worse: [15][1024^2] 25.2 against 21.9 us,
  // [30][1024^2] 46.9 and 39.7; beyond it, out of memory, eight are better ([52][2048^2] 321 and 336).
  if (CPLX && wide && planes * npix * 8 <= (256LL << 20))
    hipLaunchKernelGGL((k_weighted_mean<CPLX, WEIGHTED, V, CPLX ? 2 : 8>), dim3((unsigned)((npix / V + 255) / 256)), block, 0,
                       st, in, w, out, planes, npix, power2, absval);
  else if (wide)
    hipLaunchKernelGGL((k_weighted_mean<CPLX, WEIGHTED, V, 8>), dim3((unsigned)((npix / V + 255) / 256)), block, 0, st, in,
                       w, out, planes, npix, power2, absval);
  else
    hipLaunchKernelGGL((k_weighted_mean<CPLX, WEIGHTED, 1, 8>), dim3((unsigned)((npix + 255) / 256)), block, 0, st, in, w,
                       out, planes, npix, power2, absval);
}

int launch_weighted_mean(const void *in, int in_complex, long long planes, long long npix, const float *w, float *out,
                         int power2, int absval, hipStream_t st) {
  const float *x = reinterpret_cast<const float *>(in);
  if (in_complex)
    w ? launch_mean<true, true>(x, w, out, planes, npix, power2, absval, st)
      : launch_mean<true, false>(x, w, out, planes, npix, power2, absval, st);
  else
    w ? launch_mean<false, true>(x, w, out, planes, npix, power2, absval, st)
      : launch_mean<false, false>(x, w, out, planes, npix, power2, absval, st);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

// ---------------------------------------------------------------- Conversion (all pairs)
// dtype codes: 1 U16, 2 F32, 3 CF32, 4 U8; strategy: 0 Real, 1 Scaled, 2 Modulus,
// 3 Argument (conversion.cu:138-150, kernels :156-215).
template <int DT> __device__ __forceinline__ float conv_load_real(const void *in, long long i) {
  if constexpr (DT == 1) return (float)reinterpret_cast<const uint16_t *>(in)[i];
  if constexpr (DT == 4) return (float)reinterpret_cast<const uint8_t *>(in)[i];
  return reinterpret_cast<const float *>(in)[i];
}

__device__ __forceinline__ float conv_complex(float2 z, int strategy) {
  return strategy == 3 ? atan2f(z.y, z.x) : hypotf(z.x, z.y);
}

// elements that a lane of k_convert's wide form converts at once: 16 bytes on the wider side
constexpr int convert_width(int in, int out) { return in == 3 || out == 3 ? 2 : 4; }

template <int IN, int OUT> __device__ __forceinline__ void convert_one(const void *in, void *out, int strategy, long long i) {
  if constexpr (IN == 3) {  // CF32 -> F32: modulus (hypot) or argument (atan2)
    reinterpret_cast<float *>(out)[i] = conv_complex(reinterpret_cast<const float2 *>(in)[i], strategy);
  } else if constexpr (OUT == 3) {
    reinterpret_cast<float2 *>(out)[i] = make_float2(conv_load_real<IN>(in, i), 0.f);
  } else {
    reinterpret_cast<float *>(out)[i] = conv_load_real<IN>(in, i);
  }
}

// Bound by memory.  G > 0: V consecutive elements per lane and access and G such groups in flight,
// 16 bytes of neighbouring lanes next to each other on the wider side; G = 0 (buffers not aligned to V
// elements): one element per lane.  [64][1024^2] U16 -> F32 (403 MB): 149 us with one element per lane,
// 66-69 here; 4 M U16 -> CF32: 8.5 and 7.0 (four elements per lane, whose two stores then take every
// other 16 bytes: 9.9).
template <int IN, int OUT, int G>
__global__ __launch_bounds__(256) void k_convert(const void *__restrict__ in, void *__restrict__ out, int strategy,
                                                 long long n) {
  if constexpr (G == 0) {
    const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
    if (i < n) convert_one<IN, OUT>(in, out, strategy, i);
  } else {
    constexpr int V = convert_width(IN, OUT), NI = IN == 3 ? 2 * V : V;  // elements and their 32-bit parts
    typedef std::conditional_t<IN == 1, uint16_t, std::conditional_t<IN == 4, uint8_t, float>> E;
    typedef E vin __attribute__((ext_vector_type(NI)));
    typedef float vout __attribute__((ext_vector_type(OUT == 3 ? 2 * V : V)));
    const long long i0 = (long long)blockIdx.x * (256 * V * G) + V * threadIdx.x;
    if (i0 + 256 * V * (G - 1) + V <= n) {
      vin raw[G];
#pragma unroll
      for (int g = 0; g < G; ++g) raw[g] = *reinterpret_cast<const vin *>(reinterpret_cast<const E *>(in) + (i0 + 256 * V * g) * (NI / V));
#pragma unroll
      for (int g = 0; g < G; ++g) {
        vout y;
#pragma unroll
        for (int t = 0; t < V; ++t) {
          if constexpr (IN == 3) {
            y[t] = conv_complex(make_float2(raw[g][2 * t], raw[g][2 * t + 1]), strategy);
          } else if constexpr (OUT == 3) {
            y[2 * t] = (float)raw[g][t];
            y[2 * t + 1] = 0.f;
          } else {
            y[t] = (float)raw[g][t];
          }
        }
        *reinterpret_cast<vout *>(reinterpret_cast<float *>(out) + (i0 + 256 * V * g) * (OUT == 3 ? 2 : 1)) = y;
      }
    } else {
      for (int g = 0; g < G; ++g)
        for (int t = 0; t < V; ++t)
          if (i0 + 256 * V * g + t < n) convert_one<IN, OUT>(in, out, strategy, i0 + 256 * V * g + t);
    }
  }
}

template <int IN, int OUT> static void launch_convert_pair(const void *in, void *out, int strategy, long long n, hipStream_t st) {
  constexpr int V = convert_width(IN, OUT);
  constexpr int in_bytes = V * (IN == 1 ? 2 : IN == 4 ? 1 : IN == 3 ? 8 : 4), out_bytes = V * (OUT == 3 ? 8 : 4);
  const bool wide = reinterpret_cast<uintptr_t>(in) % in_bytes == 0 && reinterpret_cast<uintptr_t>(out) % out_bytes == 0;
  auto go = [&](auto g) {
    constexpr int G = decltype(g)::value;
    const long long per_block = 256 * (G == 0 ? 1 : V * G);
    hipLaunchKernelGGL((k_convert<IN, OUT, G>), dim3((unsigned)((n + per_block - 1) / per_block)), dim3(256), 0, st, in, out, strategy, n);
  };
  // two groups per lane only where the halved grid still fills the chip: argument of 1 M CF32 3.2 us
  // with one, 3.7 with two (and 4.1 with four); 8 M CF32 moduli 16.1 with one, 15.1 with two
  if (!wide)
    go(std::integral_constant<int, 0>{});
  else if (n < (1 << 21))
    go(std::integral_constant<int, 1>{});
  else
    go(std::integral_constant<int, 2>{});
}

// min / max of n floats: per-block partials, then one block folds them (order-free ops)
__global__ __launch_bounds__(256) void k_minmax_partial(const float *in, long long n, float2 *partial) {
  float lo = INFINITY, hi = -INFINITY;
#pragma unroll 8
  for (long long i = (long long)blockIdx.x * 256 + threadIdx.x; i < n; i += (long long)gridDim.x * 256) {
    const float v = in[i];
    lo = fminf(lo, v);
    hi = fmaxf(hi, v);
  }
  __shared__ float2 red[256];
  red[threadIdx.x] = make_float2(lo, hi);
  __syncthreads();
  for (int s = 128; s > 0; s >>= 1) {
    if (threadIdx.x < s) {
      red[threadIdx.x].x = fminf(red[threadIdx.x].x, red[threadIdx.x + s].x);
      red[threadIdx.x].y = fmaxf(red[threadIdx.x].y, red[threadIdx.x + s].y);
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) partial[blockIdx.x] = red[0];
}

__global__ __launch_bounds__(256) void k_minmax_final(float2 *partial, int nblocks) {
  float lo = INFINITY, hi = -INFINITY;
  for (int i = threadIdx.x; i < nblocks; i += 256) {
    lo = fminf(lo, partial[i].x);
    hi = fmaxf(hi, partial[i].y);
  }
  __shared__ float2 red[256];
  red[threadIdx.x] = make_float2(lo, hi);
  __syncthreads();
  for (int s = 128; s > 0; s >>= 1) {
    if (threadIdx.x < s) {
      red[threadIdx.x].x = fminf(red[threadIdx.x].x, red[threadIdx.x + s].x);
      red[threadIdx.x].y = fmaxf(red[threadIdx.x].y, red[threadIdx.x + s].y);
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) partial[nblocks] = red[0];
}

// F32 -> U8/U16 scaled to the tensor's [min, max] (conversion.cu:177-195), V elements per lane
template <typename O, int V>
__global__ __launch_bounds__(256) void k_scaled(const float *__restrict__ in, O *__restrict__ out, long long n,
                                                const float2 *__restrict__ mm) {
  const long long i = ((long long)blockIdx.x * 256 + threadIdx.x) * V;
  if (i >= n) return;
  const float lo = mm->x, hi = mm->y;
  const float top = sizeof(O) == 1 ? 255.f : 65535.f;
  const float scale = top / (hi - lo);
  auto one = [&](float x) {
    const int val = (int)((x - lo) * scale + 0.5f);
    return (O)fminf(fmaxf((float)val, 0.f), top);
  };
  if (V == 4 && i + 3 < n) {
    const float4 x = *reinterpret_cast<const float4 *>(in + i);
    typedef O vec __attribute__((ext_vector_type(4)));
    *reinterpret_cast<vec *>(out + i) = vec{one(x.x), one(x.y), one(x.z), one(x.w)};
  } else {
    for (long long j = i; j < i + V && j < n; ++j) out[j] = one(in[j]);
  }
}

template <typename O> static void launch_scaled(const float *in, O *out, long long n, const float2 *mm, hipStream_t st) {
  // (four per lane leave a small grid short of blocks: 65,536 elements 6.4 us for the whole conversion
  // with one per lane, 6.8 with four; 2 M 10.1 and 8.4)
  if (n >= (1 << 20) && reinterpret_cast<uintptr_t>(in) % 16 == 0 && reinterpret_cast<uintptr_t>(out) % (4 * sizeof(O)) == 0)
    hipLaunchKernelGGL((k_scaled<O, 4>), dim3((unsigned)((n + 1023) / 1024)), dim3(256), 0, st, in, out, n, mm);
  else
    hipLaunchKernelGGL((k_scaled<O, 1>), dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, in, out, n, mm);
}

int minmax_blocks(long long n) { return (int)((n + 255) / 256 < 1024 ? (n + 255) / 256 : 1024); }

// Library-held scratch of the allocation-free Scaled conversion: the per-block min/max
// partials of at most 1024 blocks plus the folded pair (8,200 bytes, any n).  Each GPU holds
// its own copy for the life of the process; calls on one GPU share it, so calls that overlap
// on one GPU (concurrent streams) race.  Every call writes each pair it reads first, so
// nothing needs clearing between calls.
constexpr int kConvScratchPairs = 1025;
static __device__ __align__(256) float2 scratch[kConvScratchPairs];

long long convert_static_scratch_bytes() { return (long long)sizeof(float2) * kConvScratchPairs; }

// Device address of `scratch` on the current device, looked up once per device (the host
// symbol is only a stand-in: kernels must receive this address).
int convert_static_scratch(void **ptr) {
  constexpr int kMaxDevices = 64;
  static std::mutex mu;
  static void *per_device[kMaxDevices] = {};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return -1;
  std::lock_guard<std::mutex> lock(mu);
  if (!per_device[dev]) {
    void *p = nullptr;
    if (hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) != hipSuccess || !p) return -1;
    per_device[dev] = p;
  }
  *ptr = per_device[dev];
  return 0;
}

int launch_convert(const void *in, int in_dt, void *out, int out_dt, int strategy, long long n,
                   void *scratch, hipStream_t st) {
  if (n == 0) return 0;
  if (strategy == 1) {
    const int nb = minmax_blocks(n);
    float2 *part = reinterpret_cast<float2 *>(scratch);
    hipLaunchKernelGGL(k_minmax_partial, dim3(nb), dim3(256), 0, st, reinterpret_cast<const float *>(in), n, part);
    hipLaunchKernelGGL(k_minmax_final, dim3(1), dim3(256), 0, st, part, nb);
    if (out_dt == 4)
      launch_scaled(reinterpret_cast<const float *>(in), reinterpret_cast<uint8_t *>(out), n, part + nb, st);
    else
      launch_scaled(reinterpret_cast<const float *>(in), reinterpret_cast<uint16_t *>(out), n, part + nb, st);
  } else if (in_dt == 1) {
    out_dt == 3 ? launch_convert_pair<1, 3>(in, out, strategy, n, st) : launch_convert_pair<1, 2>(in, out, strategy, n, st);
  } else if (in_dt == 4) {
    out_dt == 3 ? launch_convert_pair<4, 3>(in, out, strategy, n, st) : launch_convert_pair<4, 2>(in, out, strategy, n, st);
  } else if (in_dt == 3) {
    launch_convert_pair<3, 2>(in, out, strategy, n, st);
  } else {
    launch_convert_pair<2, 3>(in, out, strategy, n, st);
  }
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

// ---------------------------------------------------------------- SlidingAverage step
// ravg = (ravg + x / ws) - old / ws, then the old slot takes ravg (slide_avg.cu:102-125,
// 200-215: two kernels and a copy; each operation rounds to FP32 in the same order here).
__global__ void k_slide_avg(const float *x, float *old_slot, float *ravg, long long n, float ws) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  float r = ravg[i];
  r = r + x[i] / ws;
  r = r - old_slot[i] / ws;
  ravg[i] = r;
  old_slot[i] = r;
}

int launch_slide_avg(const float *x, float *old_slot, float *ravg, long long n, int ws, hipStream_t st) {
  if (n == 0) return 0;
  hipLaunchKernelGGL(k_slide_avg, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, x, old_slot, ravg, n,
                     (float)ws);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

// Gather of a strided view (holonp::Copy, copy.cu:40,117-125; the pieces of
// holonp::Concatenate).  Strides and offset in bytes, as TDesc has them.  Element t of the
// view goes to out[(t / out_block) * out_pitch + t % out_block]: one input of a
// concatenation along an inner axis lands in its column band of the output in one launch.
struct CopyGeo {
  int ndim, esz;
  long long shape[8];
  long long in_stride[8];
  long long in_offset;
  long long total;
  long long out_block, out_pitch;
};

__global__ void k_strided_copy(const uint8_t *in, uint8_t *out, CopyGeo g) {
  long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= g.total) return;
  long long rem = t, src = g.in_offset;
  for (int k = g.ndim - 1; k >= 0; --k) {
    const long long idx = rem % g.shape[k];
    rem /= g.shape[k];
    src += idx * g.in_stride[k];
  }
  const long long o = (t / g.out_block) * g.out_pitch + t % g.out_block;
  if (g.esz == 8)
    reinterpret_cast<uint2 *>(out)[o] = *reinterpret_cast<const uint2 *>(in + src);
  else if (g.esz == 4)
    reinterpret_cast<uint32_t *>(out)[o] = *reinterpret_cast<const uint32_t *>(in + src);
  else
    for (int b = 0; b < g.esz; ++b) out[o * g.esz + b] = in[src + b];
}

// Contiguous fast path: 16 bytes per lane, 4 vectors in flight per lane, grid sized to the
// device (8 blocks of 256 per CU), grid-stride over the buffer.
__global__ __launch_bounds__(256) void k_copy16(const uint4 *__restrict__ in, uint4 *__restrict__ out,
                                                long long n16) {
  const long long stride = (long long)gridDim.x * blockDim.x;
  long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  for (; i + 3 * stride < n16; i += 4 * stride) {
    const uint4 a = in[i], b = in[i + stride], c = in[i + 2 * stride], d = in[i + 3 * stride];
    out[i] = a;
    out[i + stride] = b;
    out[i + 2 * stride] = c;
    out[i + 3 * stride] = d;
  }
  for (; i < n16; i += stride) out[i] = in[i];
}

// HBM bandwidth probe (measurement only): mode 0 reads the buffer (each lane folds its
// 16-byte vectors into one word, stored only if it equals a value no data here produces, so
// the loads stay live), mode 1 writes it, mode 2 copies it.  U independent 16-byte vectors per
// lane per iteration, grid-stride over the buffer, non-temporal for NT = 1.
template <int MODE, int U, int NT>
__global__ __launch_bounds__(256) void k_hbm_probe(const uint4 *__restrict__ in, uint4 *__restrict__ out,
                                                   long long n16, unsigned *sink) {
  const long long stride = (long long)gridDim.x * 256;
  long long i = (long long)blockIdx.x * 256 + threadIdx.x;
  typedef unsigned u4v __attribute__((ext_vector_type(4)));
  unsigned acc = 0;
  const uint4 fill = make_uint4(threadIdx.x, blockIdx.x, 0x5a5a5a5au, 0xa5a5a5a5u);
  for (; i + (U - 1) * stride < n16; i += U * stride) {
    u4v v[U];
    if (MODE != 1) {
#pragma unroll
      for (int u = 0; u < U; ++u)
        v[u] = NT ? __builtin_nontemporal_load(reinterpret_cast<const u4v *>(in) + i + u * stride)
                  : reinterpret_cast<const u4v *>(in)[i + u * stride];
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (MODE == 0) {
        acc ^= v[u].x ^ v[u].y ^ v[u].z ^ v[u].w;
      } else {
        const u4v w = MODE == 1 ? u4v{fill.x, fill.y, fill.z, fill.w} : v[u];
        if (NT)
          __builtin_nontemporal_store(w, reinterpret_cast<u4v *>(out) + i + u * stride);
        else
          reinterpret_cast<u4v *>(out)[i + u * stride] = w;
      }
    }
  }
  for (; i < n16; i += stride) {
    if (MODE == 0) {
      const uint4 v = in[i];
      acc ^= v.x ^ v.y ^ v.z ^ v.w;
    } else {
      out[i] = MODE == 1 ? fill : in[i];
    }
  }
  if (MODE == 0 && acc == 0x9e3779b9u) sink[blockIdx.x & 255] = acc;
}

template <int MODE, int U>
static void launch_probe_u(int nt, unsigned blocks, const uint4 *in, uint4 *out, long long n16, unsigned *sink,
                           hipStream_t st) {
  if (nt)
    hipLaunchKernelGGL((k_hbm_probe<MODE, U, 1>), dim3(blocks), dim3(256), 0, st, in, out, n16, sink);
  else
    hipLaunchKernelGGL((k_hbm_probe<MODE, U, 0>), dim3(blocks), dim3(256), 0, st, in, out, n16, sink);
}

template <int MODE>
static int launch_probe_mode(int unroll, int nt, unsigned blocks, const uint4 *in, uint4 *out, long long n16,
                             unsigned *sink, hipStream_t st) {
  switch (unroll) {
    case 1: launch_probe_u<MODE, 1>(nt, blocks, in, out, n16, sink, st); break;
    case 2: launch_probe_u<MODE, 2>(nt, blocks, in, out, n16, sink, st); break;
    case 4: launch_probe_u<MODE, 4>(nt, blocks, in, out, n16, sink, st); break;
    case 8: launch_probe_u<MODE, 8>(nt, blocks, in, out, n16, sink, st); break;
    default: return -2;
  }
  return 0;
}

int launch_hbm_probe(int mode, const void *in, void *out, long long bytes, int blocks_per_cu, int unroll,
                     int nontemporal, unsigned *sink, hipStream_t st) {
  const int cus = device_cus();
  const long long n16 = bytes / 16;
  if (n16 <= 0) return 0;
  long long blocks = (long long)blocks_per_cu * cus;
  if (blocks > (n16 + 255) / 256) blocks = (n16 + 255) / 256;
  const uint4 *i4 = reinterpret_cast<const uint4 *>(in);
  uint4 *o4 = reinterpret_cast<uint4 *>(out);
  int rc = -2;
  switch (mode) {
    case 0: rc = launch_probe_mode<0>(unroll, nontemporal, (unsigned)blocks, i4, o4, n16, sink, st); break;
    case 1: rc = launch_probe_mode<1>(unroll, nontemporal, (unsigned)blocks, i4, o4, n16, sink, st); break;
    case 2: rc = launch_probe_mode<2>(unroll, nontemporal, (unsigned)blocks, i4, o4, n16, sink, st); break;
  }
  if (rc != 0) return rc;
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

static int launch_copy_bytes(const uint8_t *in, uint8_t *out, long long bytes, hipStream_t st) {
  const int cus = device_cus();
  const long long n16 = bytes / 16;
  if (n16 > 0) {
    long long blocks = (n16 + 255) / 256;
    if (blocks > 8LL * cus) blocks = 8LL * cus;
    hipLaunchKernelGGL(k_copy16, dim3((unsigned)blocks), dim3(256), 0, st,
                       reinterpret_cast<const uint4 *>(in), reinterpret_cast<uint4 *>(out), n16);
  }
  const long long tail = bytes - n16 * 16;
  if (tail > 0) {
    CopyGeo g{};
    g.ndim = 1;
    g.esz = 1;
    g.shape[0] = tail;
    g.in_stride[0] = 1;
    g.in_offset = n16 * 16;
    g.total = tail;
    g.out_block = tail;
    g.out_pitch = tail;
    hipLaunchKernelGGL(k_strided_copy, dim3(1), dim3(256), 0, st, in, out + n16 * 16, g);
  }
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

int launch_strided_copy(const void *in, void *out, int elem_size, int ndim, const long long *shape,
                        const long long *in_strides, long long in_offset, long long out_block,
                        long long out_pitch, hipStream_t st) {
  if (ndim < 1 || ndim > 8) return -1;
  {
    // a C-contiguous view written contiguously is a plain byte copy
    bool contiguous = out_block <= 0;
    long long expect = elem_size, total = 1;
    for (int k = ndim - 1; k >= 0; --k) {
      if (shape[k] != 1 && in_strides[k] != expect) contiguous = false;
      expect *= shape[k];
      total *= shape[k];
    }
    const uint8_t *src = reinterpret_cast<const uint8_t *>(in) + in_offset;
    if (contiguous && ((reinterpret_cast<uintptr_t>(src) | reinterpret_cast<uintptr_t>(out)) % 16) == 0)
      return total == 0 ? 0 : launch_copy_bytes(src, reinterpret_cast<uint8_t *>(out), total * elem_size, st);
  }
  CopyGeo g;
  g.ndim = ndim;
  g.esz = elem_size;
  g.in_offset = in_offset;
  g.total = 1;
  for (int k = 0; k < ndim; ++k) {
    g.shape[k] = shape[k];
    g.in_stride[k] = in_strides[k];
    g.total *= shape[k];
  }
  if (g.total == 0) return 0;
  g.out_block = out_block > 0 ? out_block : g.total;
  g.out_pitch = out_block > 0 ? out_pitch : g.total;
  hipLaunchKernelGGL(k_strided_copy, dim3((unsigned)((g.total + 255) / 256)), dim3(256), 0, st,
                     reinterpret_cast<const uint8_t *>(in), reinterpret_cast<uint8_t *>(out), g);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

// Broadcasting element-wise product (holonp::Multiply, multiply.cu:69-92): out has the
// broadcast shape; an operand's element stride is 0 on its broadcast axes.  Real operands
// are promoted to x + 0i when the output is complex.
struct MulGeo {
  int ndim;
  long long shape[8];
  long long sa[8], sb[8];  // element strides
  long long total;
  int a_complex, b_complex, out_complex;
};

__global__ void k_multiply(const void *a, const void *b, void *out, MulGeo g) {
  long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= g.total) return;
  long long rem = t, ia = 0, ib = 0;
  for (int k = g.ndim - 1; k >= 0; --k) {
    const long long idx = rem % g.shape[k];
    rem /= g.shape[k];
    ia += idx * g.sa[k];
    ib += idx * g.sb[k];
  }
  const float2 va = g.a_complex ? reinterpret_cast<const float2 *>(a)[ia]
                                : make_float2(reinterpret_cast<const float *>(a)[ia], 0.f);
  const float2 vb = g.b_complex ? reinterpret_cast<const float2 *>(b)[ib]
                                : make_float2(reinterpret_cast<const float *>(b)[ib], 0.f);
  if (g.out_complex)
    reinterpret_cast<float2 *>(out)[t] = cmul(va, vb);
  else
    reinterpret_cast<float *>(out)[t] = va.x * vb.x;
}

int launch_multiply(const void *a, int a_complex, const long long *sa, const void *b, int b_complex,
                    const long long *sb, int ndim, const long long *shape, void *out, hipStream_t st) {
  if (ndim < 1 || ndim > 8) return -1;
  MulGeo g;
  g.ndim = ndim;
  g.total = 1;
  for (int k = 0; k < ndim; ++k) {
    g.shape[k] = shape[k];
    g.sa[k] = sa[k];
    g.sb[k] = sb[k];
    g.total *= shape[k];
  }
  g.a_complex = a_complex;
  g.b_complex = b_complex;
  g.out_complex = a_complex || b_complex;
  if (g.total == 0) return 0;
  hipLaunchKernelGGL(k_multiply, dim3((unsigned)((g.total + 255) / 256)), dim3(256), 0, st, a, b, out, g);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

// Direct DFT along the middle axis of [outer][n][inner] for the stand-alone RFFT / FFT
// kinds (any axis, any length).  Twiddles are evaluated in FP64 from the exactly
// reduced integer argument (k*j mod n) and rounded to FP32; products and sums are FP32.
struct DftAxisArgs {
  const void *in;
  int dtype;  // 1 U16, 2 F32, 3 CF32
  long long outer, inner;
  int n, kb, ke;
  float scale;
  float2 *out;
};

__global__ void k_dft_axis(DftAxisArgs a) {
  long long nk = a.ke - a.kb;
  long long total = a.outer * nk * a.inner;
  long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= total) return;
  long long i = t % a.inner;
  long long k = (t / a.inner) % nk + a.kb;
  long long o = t / (a.inner * nk);
  float sr = 0.f, si = 0.f;
  for (int j = 0; j < a.n; ++j) {
    long long src = (o * a.n + j) * a.inner + i;
    float xr, xi = 0.f;
    if (a.dtype == 1)
      xr = (float)reinterpret_cast<const uint16_t *>(a.in)[src];
    else if (a.dtype == 2)
      xr = reinterpret_cast<const float *>(a.in)[src];
    else {
      float2 v = reinterpret_cast<const float2 *>(a.in)[src];
      xr = v.x;
      xi = v.y;
    }
    long long m = (k * j) % a.n;
    double s, c;
    sincospi(2.0 * (double)m / (double)a.n, &s, &c);
    float wr = (float)c, wi = (float)(-s);
    sr += xr * wr - xi * wi;
    si += xr * wi + xi * wr;
  }
  a.out[t] = make_float2(sr * a.scale, si * a.scale);
}

// Band DFT of up to DFT_SHORT points: a lane owns one column and sums directly over j, which leaves
// little but the stream (the matrix form spends 16 bins and four pairs of samples on them).  All bins
// of 1 M U16 columns at n = 1, 4 and 8: 5.4, 9.5 and 21 us, in the matrix form 20, 23.8 and 27.
// At 12 points and 12 bins the sums cost more than the matrix form (65,536 columns: 11.1 against 5.8).
constexpr int DFT_SHORT = 8;
template <int DT> __global__ __launch_bounds__(256) void k_dft_axis_short(DftAxisArgs a, long long cols) {
  __shared__ float2 tw[DFT_SHORT];
  if (threadIdx.x < a.n) {
    double s, c;
    sincospi(2.0 * (double)threadIdx.x / (double)a.n, &s, &c);
    tw[threadIdx.x] = make_float2((float)c, (float)(-s));
  }
  __syncthreads();
  const long long c = (long long)blockIdx.x * 256 + threadIdx.x;
  if (c >= cols) return;
  const long long o = c / a.inner, i = c - o * a.inner;
  float2 x[DFT_SHORT];
#pragma unroll
  for (int j = 0; j < DFT_SHORT; ++j) {
    if (j >= a.n) break;
    const long long src = (o * a.n + j) * a.inner + i;
    if constexpr (DT == 1)
      x[j] = make_float2((float)reinterpret_cast<const uint16_t *>(a.in)[src], 0.f);
    else if constexpr (DT == 2)
      x[j] = make_float2(reinterpret_cast<const float *>(a.in)[src], 0.f);
    else
      x[j] = reinterpret_cast<const float2 *>(a.in)[src];
  }
  for (int k = a.kb; k < a.ke; ++k) {
    float2 acc = make_float2(0.f, 0.f);
    int m = 0;
#pragma unroll
    for (int j = 0; j < DFT_SHORT; ++j) {
      if (j >= a.n) break;
      const float2 w = tw[m];
      if constexpr (DT == 3) {
        acc.x += x[j].x * w.x - x[j].y * w.y;
        acc.y += x[j].x * w.y + x[j].y * w.x;
      } else {
        acc.x += x[j].x * w.x;
        acc.y += x[j].x * w.y;
      }
      m += k;
      m = m >= a.n ? m - a.n : m;
    }
    a.out[(o * (a.ke - a.kb) + (k - a.kb)) * a.inner + i] = make_float2(acc.x * a.scale, acc.y * a.scale);
  }
}

// Band DFT along the middle axis on the matrix cores, n <= DFT_MAXN.  A wave owns 64 columns (an
// outer and an inner index; four per lane, AxisColumns), and the symmetry of the kernel is folded
// as in the fused path's time DFT: with s = x_p + x_{n-p}, d = x_p - x_{n-p},
//   X_k = x_0 [+ (-1)^k x_{n/2}] + sum_{p=1}^{(n-1)/2} (s cos(2 pi k p / n) - i d sin(2 pi k p / n)),
// so 16 bins and 16 columns take 2 ((n-1)/2)/4 + 1 FP32 MFMAs for real input, twice that for
// complex.  Step st covers the pairs p = 4 st + g + 1 (g = lane >> 4, the MFMA's K index).  The
// operands cos, -sin come from an LDS table of the n roots (FP64 sincospi, rounded once) through a
// running index k p mod n, one 8-byte read per 16 bins and step for four (complex: eight) MFMAs per
// operand, so any n and any bin range work without an operand matrix.
//
// Bound by memory: F32 [64][1024^2] -> 33 bins (three 16-bin tiles) moves 545 MB.  The kernel it
// replaces (direct sums on the VALU, 16 bins per pass over the input) took 570 us there.
//
// Lanes whose pair or column does not exist get zero samples, not zero weights, so that an
// infinity elsewhere in the column is not turned into a NaN.  Floating samples are halved on the way into
// the pairs and the results scaled by two more (exact), so that the pairs of samples beyond half the
// float range stay finite.
//
// DT: 1 U16, 2 F32, 3 CF32.  VEC: the four columns of a lane are adjacent in memory and aligned.
constexpr int DFT_MAXN = 4096;
typedef float f4v __attribute__((ext_vector_type(4)));

template <int DT, bool VEC> struct DftColumns {
  static constexpr int NF = DT == 3 ? 8 : 4;  // floats of four samples
  const char *in;
  AxisColumns<DT == 1 ? 2 : DT == 2 ? 4 : 8, VEC> col;
  __device__ __forceinline__ void init(const DftAxisArgs &a, long long tile, int rw, long long cols) {
    in = reinterpret_cast<const char *>(a.in);
    col.init(tile, rw, cols, a.n, a.inner);
  }
  // the raw samples j of the four columns
  struct Raw {
    uint4 q[VEC && DT == 3 ? 2 : 1];
    unsigned w[VEC ? 1 : NF];
  };
  __device__ __forceinline__ void load(Raw &r, int j) const {
    const long long off = j * col.step;
    if constexpr (VEC) {
      if constexpr (DT == 1) {
        const uint2 v = *reinterpret_cast<const uint2 *>(in + col.off[0] + off);
        r.q[0].x = v.x;
        r.q[0].y = v.y;
      } else {
        r.q[0] = *reinterpret_cast<const uint4 *>(in + col.off[0] + off);
        if constexpr (DT == 3) r.q[1] = *reinterpret_cast<const uint4 *>(in + col.off[0] + off + 16);
      }
    } else {
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        if constexpr (DT == 1) {
          r.w[t] = *reinterpret_cast<const uint16_t *>(in + col.off[t] + off);
        } else if constexpr (DT == 2) {
          r.w[t] = *reinterpret_cast<const unsigned *>(in + col.off[t] + off);
        } else {
          const uint2 v = *reinterpret_cast<const uint2 *>(in + col.off[t] + off);
          r.w[2 * t] = v.x;
          r.w[2 * t + 1] = v.y;
        }
      }
    }
  }
  // samples as floats (complex: re, im per column)
  __device__ __forceinline__ static void unpack(const Raw &r, float (&x)[NF]) {
    if constexpr (VEC && DT == 1) {
      x[0] = (float)(r.q[0].x & 0xffffu);
      x[1] = (float)(r.q[0].x >> 16);
      x[2] = (float)(r.q[0].y & 0xffffu);
      x[3] = (float)(r.q[0].y >> 16);
    } else if constexpr (VEC) {
#pragma unroll
      for (int h = 0; h < NF / 4; ++h) {
        x[4 * h] = __uint_as_float(r.q[h].x);
        x[4 * h + 1] = __uint_as_float(r.q[h].y);
        x[4 * h + 2] = __uint_as_float(r.q[h].z);
        x[4 * h + 3] = __uint_as_float(r.q[h].w);
      }
    } else {
#pragma unroll
      for (int t = 0; t < NF; ++t) x[t] = DT == 1 ? (float)r.w[t] : __uint_as_float(r.w[t]);
    }
  }
};

// NBF: 16-bin tiles from bin k0 on that a wave holds at once (the input is read once per launch)
template <int DT, bool VEC, int NBF>
__global__ __launch_bounds__(256, 2) void k_dft_axis_mfma(DftAxisArgs a, int k0, long long cols) {
  extern __shared__ float2 tw[];
  for (int m = threadIdx.x; m < a.n; m += 256) {
    double s, c;
    sincospi(2.0 * (double)m / (double)a.n, &s, &c);
    tw[m] = make_float2((float)c, (float)(-s));
  }
  __syncthreads();
  using X = DftColumns<DT, VEC>;
  constexpr int NF = X::NF;
  constexpr int K = DT == 3 ? 2 : 4;  // pair steps in flight
  constexpr float HALF = DT == 1 ? 1.f : 0.5f;
  const float scale = a.scale * (1.f / HALF);
  const int n = a.n, pairs = (n - 1) / 2, steps = (pairs + 3) / 4;
  const int lane = threadIdx.x & 63, g = lane >> 4, rw = lane & 15;
  const long long tiles = (cols + 63) / 64;
  for (long long it = (long long)blockIdx.x * 4 + (threadIdx.x >> 6); it < tiles; it += (long long)gridDim.x * 4) {
    X x;
    x.init(a, it, rw, cols);
    f4v re[NBF][4], im[NBF][4];
    int idx[NBF], inc[NBF];  // k p mod n of this lane's bin and pair, and its advance by four pairs
#pragma unroll
    for (int f = 0; f < NBF; ++f) {
      const long long k = k0 + 16 * f + rw;
      idx[f] = (int)(k * (g + 1) % n);
      inc[f] = (int)(4 * k % n);
#pragma unroll
      for (int t = 0; t < 4; ++t) re[f][t] = im[f][t] = f4v{0.f, 0.f, 0.f, 0.f};
    }
    typename X::Raw r[K][2], xe;
    auto load = [&](int st, int slot) {
      const int p = min(4 * st + g + 1, max(pairs, 1));
      x.load(r[slot][0], n > 1 ? p : 0);
      x.load(r[slot][1], n - p);
    };
    x.load(xe, g == 0 ? 0 : n / 2);
#pragma unroll
    for (int j = 0; j < K; ++j) load(j, j);
    auto step = [&](int st, int slot, bool refill) {
      float x1[NF], x2[NF];
      X::unpack(r[slot][0], x1);
      X::unpack(r[slot][1], x2);
      if (refill) load(st + K, slot);
      const bool in = 4 * st + g < pairs;
      float sm[NF], df[NF];
#pragma unroll
      for (int t = 0; t < NF; ++t) {
        const float h = HALF * x1[t];
        sm[t] = in ? fmaf(HALF, x2[t], h) : 0.f;
        df[t] = in ? fmaf(-HALF, x2[t], h) : 0.f;
      }
#pragma unroll
      for (int f = 0; f < NBF; ++f) {
        const float2 w = tw[idx[f]];
        idx[f] += inc[f];
        idx[f] = idx[f] >= n ? idx[f] - n : idx[f];
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          if constexpr (DT == 3) {
            re[f][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(w.x, sm[2 * t], re[f][t], 0, 0, 0);
            im[f][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(w.x, sm[2 * t + 1], im[f][t], 0, 0, 0);
          } else {
            re[f][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(w.x, sm[t], re[f][t], 0, 0, 0);
            im[f][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(w.y, df[t], im[f][t], 0, 0, 0);
          }
        }
        if constexpr (DT == 3) {
#pragma unroll
          for (int t = 0; t < 4; ++t) {
            re[f][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(w.y, -df[2 * t + 1], re[f][t], 0, 0, 0);
            im[f][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(w.y, df[2 * t], im[f][t], 0, 0, 0);
          }
        }
      }
    };
    int st = 0;
    for (; st + K < steps; st += K) {
#pragma unroll
      for (int j = 0; j < K; ++j) step(st + j, j, true);
    }
#pragma unroll
    for (int j = 0; j < K; ++j) step(st + j, j, false);  // steps past the last pair add zeros
    // x_0 (g = 0, weight 1) and, for even n, x_{n/2} (g = 1, weight (-1)^k)
    float xv[NF];
    X::unpack(xe, xv);
    const bool in = g == 0 || (g == 1 && n % 2 == 0);
#pragma unroll
    for (int t = 0; t < NF; ++t) xv[t] = in ? HALF * xv[t] : 0.f;
#pragma unroll
    for (int f = 0; f < NBF; ++f) {
      const float w = g == 1 && ((k0 + 16 * f + rw) & 1) ? -1.f : 1.f;
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        if constexpr (DT == 3) {
          re[f][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(w, xv[2 * t], re[f][t], 0, 0, 0);
          im[f][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(w, xv[2 * t + 1], im[f][t], 0, 0, 0);
        } else {
          re[f][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(w, xv[t], re[f][t], 0, 0, 0);
        }
      }
    }
    // lane holds bins 16 f + 4 g + r of its four columns
    const long long nk = a.ke - a.kb, c0 = x.col.column(it, rw, 0);
    if (c0 >= cols) continue;
#pragma unroll
    for (int f = 0; f < NBF; ++f) {
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int k = k0 + 16 * f + 4 * g + q;
        if (k >= a.ke) continue;
        float2 v[4];
#pragma unroll
        for (int t = 0; t < 4; ++t) v[t] = make_float2(re[f][t][q] * scale, im[f][t][q] * scale);
        if constexpr (VEC) {
          const long long o = c0 / a.inner, i = c0 - o * a.inner;
          float4 *dst = reinterpret_cast<float4 *>(a.out + (o * nk + (k - a.kb)) * a.inner + i);
          dst[0] = make_float4(v[0].x, v[0].y, v[1].x, v[1].y);
          dst[1] = make_float4(v[2].x, v[2].y, v[3].x, v[3].y);
        } else {
#pragma unroll
          for (int t = 0; t < 4; ++t) {
            const long long c = x.col.column(it, rw, t);
            if (c < cols) {
              const long long o = c / a.inner, i = c - o * a.inner;
              a.out[(o * nk + (k - a.kb)) * a.inner + i] = v[t];
            }
          }
        }
      }
    }
  }
}

template <int DT, bool VEC, int NBF> static void launch_axis_nbf(const DftAxisArgs &a, int k0, long long cols, hipStream_t st) {
  const int cus = device_cus();
  // persistent: the blocks that are resident at once (their registers allow four, three and two per
  // CU for one, two and three 16-bin tiles) walk the tiles
  const long long quads = (cols + 255) / 256, most = (long long)cus * (NBF == 1 ? 4 : NBF == 2 ? 3 : 2);
  const unsigned grid = (unsigned)(quads < most ? quads : most);
  hipLaunchKernelGGL((k_dft_axis_mfma<DT, VEC, NBF>), dim3(grid), dim3(256), (size_t)a.n * sizeof(float2), st, a, k0, cols);
}

template <int DT, bool VEC> static void launch_axis(const DftAxisArgs &a, long long cols, hipStream_t st) {
  // the bins in as few passes over the input as the registers allow (three 16-bin tiles; two where
  // a lane keeps four addresses), evenly filled
  constexpr int MOST = VEC ? 3 : 2;
  const int tiles = (a.ke - a.kb + 15) / 16, passes = (tiles + MOST - 1) / MOST, nbf = (tiles + passes - 1) / passes;
  for (int k0 = a.kb; k0 < a.ke; k0 += 16 * nbf) {
    if (nbf == 1)
      launch_axis_nbf<DT, VEC, 1>(a, k0, cols, st);
    else if (nbf == 2)
      launch_axis_nbf<DT, VEC, 2>(a, k0, cols, st);
    else
      launch_axis_nbf<DT, VEC, MOST>(a, k0, cols, st);
  }
}

int launch_dft_axis(const void *in, int dtype, long long outer, int n, long long inner, int kb,
                    int ke, float scale, float2 *out, hipStream_t st) {
  DftAxisArgs a{in, dtype, outer, inner, n, kb, ke, scale, out};
  long long total = outer * (long long)(ke - kb) * inner;
  if (total == 0) return 0;
  const long long cols = outer * inner;
  if (n <= DFT_SHORT) {
    const dim3 grid((unsigned)((cols + 255) / 256)), block(256);
    switch (dtype) {
      case 1: hipLaunchKernelGGL(k_dft_axis_short<1>, grid, block, 0, st, a, cols); break;
      case 2: hipLaunchKernelGGL(k_dft_axis_short<2>, grid, block, 0, st, a, cols); break;
      default: hipLaunchKernelGGL(k_dft_axis_short<3>, grid, block, 0, st, a, cols); break;
    }
  } else if (n <= DFT_MAXN) {
    const uintptr_t align = reinterpret_cast<uintptr_t>(in) % (dtype == 1 ? 8 : 16) + reinterpret_cast<uintptr_t>(out) % 16;
    const bool vec = inner % 4 == 0 && align == 0;  // four adjacent columns share an outer index
    switch (dtype) {
      case 1: vec ? launch_axis<1, true>(a, cols, st) : launch_axis<1, false>(a, cols, st); break;
      case 2: vec ? launch_axis<2, true>(a, cols, st) : launch_axis<2, false>(a, cols, st); break;
      default: vec ? launch_axis<3, true>(a, cols, st) : launch_axis<3, false>(a, cols, st); break;
    }
  } else {
    hipLaunchKernelGGL(k_dft_axis, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, st, a);
  }
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

}  // namespace hfx
