// Time DFT of a uint16 frame window on MFMA (see dft_core.hh), in these forms:
//
//   k_dft          : stand-alone; writes the band planes [planes][H][W] in natural layout
//                    (optionally times the Fresnel lens; negative-band conjugate planes for
//                    the two-sided FFT path).  Used for the per-stage entry point and for
//                    widths the fused kernels do not cover.
//   k_dft_fold     : the same for FP32 with 9..64 bins, with the real-input
//                    symmetry folded into the contraction (about half the MFMAs).
//   k_dft_row      : fused time DFT + forward row FFT.  A persistent workgroup walks a
//                    set of image rows; for each row its waves (64 or 128 pixels each) keep
//                    the band spectra in MFMA registers, push them through LDS into one
//                    padded row per plane, run one wave-level row FFT per plane and write
//                    the result once, column-blocked, for the column pass.  The next row's
//                    first frames are loaded while the current row is transformed.  The
//                    band planes never make an HBM round trip in natural layout.
//   k_front        : the FP32 form of k_dft_row (T = 32, 64, 128) with the waves split into producers (DFT)
//                    and consumers (row FFTs) that overlap across rows (the main path).
//
// Plane q of the output: q < nb -> bin kb+q; q >= nb (two-sided path) -> conj of computed
// bin 2*nb - q, i.e. X[T - (kb + 2*nb - q)] of a real input (fft.cu:163-194 +
// graph_builder.cc:270-287).
#include <algorithm>
#include <type_traits>

#include "dft_core.hh"
#include "hfx_kernels.hh"
#include "wfft.hh"

namespace hfx {

struct DftArgs {
  DftRing r;
  int kb, nb, nbc, both, W;
  int nwin;                // windows of the launch
  float2 *planes;          // k_dft: natural [planes][npix]; the fused kernels: blocked
  long long planes_stride; // elements from one window's planes to the next
  const void *wm_hi, *wm_lo;
  const float2 *lx, *ly;   // k_dft, k_dft_row: Fresnel lens vectors or null
  // fused kernels only
  const float2 *tw;        // W-point FFT twiddles
  int H, blk_c, n_planes, grouped;
  // the windows of one launch: one plan's consecutive windows (first frames, planes at a stride),
  // or for k_front one window each of a group of plans of one shape (the group's tables).  What a
  // single window of the stand-alone kernels needs comes first, in two 64-byte lines, and the tables
  // last: kernel arguments lie in host memory, and each further line of them that a kernel reads is
  // another round trip (load_args)
  int firsts[HFX_MAX_WIN];
  const uint16_t *rings[HFX_MAX_GROUP];
  long long ring_frames_w[HFX_MAX_GROUP];
  float2 *planes_w[HFX_MAX_GROUP];
  const float2 *lx_w[HFX_MAX_GROUP], *ly_w[HFX_MAX_GROUP];
};

// a wave-uniform value kept in a scalar register from here on (an opaque copy the compiler
// cannot rematerialise by reloading the kernel argument)
__device__ __forceinline__ int pin_sgpr(int v) {
  asm volatile("" : "+s"(v));
  return v;
}

// The band scalars every bin store tests, pinned in scalar registers at the top of a kernel:
// left to the compiler they are reloaded from the kernel arguments inside the stores'
// branches, and each reload's wait (lgkmcnt) also waits for the LDS writes in flight.
struct Band {
  int nb, nbc, kb, both, T;
};
__device__ __forceinline__ Band pinned_band(const DftArgs &a) {
  return {pin_sgpr(a.nb), pin_sgpr(a.nbc), pin_sgpr(a.kb), pin_sgpr(a.both), pin_sgpr(a.r.T)};
}

// Centring offset of computed bin `bin`: 2048 T on a DC bin, else 0.  The DC bin is bin 0, or
// bin T itself, the extra bin the two-sided path computes when its band ends at T (its
// conjugate plane is X[0]).  Added to every bin: a select instead of a branch around the
// additions (adding +0 changes no other value, only the sign of a zero).
__device__ __forceinline__ float dc_offset(int kb, int T, int bin) {
  return kb + bin == 0 || kb + bin == T ? 2048.0f * (float)T : 0.0f;
}

// value of computed bin `bin` for 4 pixels, with the centring offset restored
__device__ __forceinline__ void dft_bin_values(const Band &b, const f4 (&acc)[4], int h, int bin,
                                               float2 (&v)[4]) {
  const float dc = dc_offset(b.kb, b.T, bin);
#pragma unroll
  for (int t = 0; t < 4; ++t) v[t] = make_float2(acc[t][2 * h] + dc, acc[t][2 * h + 1]);
}

// ----------------------------------------------------------------------- stand-alone
// Band bin `bin` of the 4 pixels from p0 into its natural-layout plane (and the conjugate
// plane of the two-sided path), times the lens when there is one.
__device__ __forceinline__ void dft_store_bin(float2 *planes, long long npix, const Band &b, long long p0, int bin,
                                              const float2 (&v)[4], const float2 (&L)[4], bool lens) {
#pragma unroll
  for (int side = 0; side < 2; ++side) {
    int q;
    if (side == 0) {
      if (bin >= b.nb) continue;
      q = bin;
    } else {
      if (!b.both) continue;
      const int j = b.nb - bin;
      if (j < 0 || j >= b.nb) continue;
      q = b.nb + j;
    }
    float2 o[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      float2 c = side ? make_float2(v[t].x, -v[t].y) : v[t];
      o[t] = lens ? cmul(c, L[t]) : c;
    }
    float4 *dst = reinterpret_cast<float4 *>(planes + (long long)q * npix + p0);
    dst[0] = make_float4(o[0].x, o[0].y, o[1].x, o[1].y);
    dst[1] = make_float4(o[2].x, o[2].y, o[3].x, o[3].y);
  }
}

// All arguments that a kernel reads, asked for in one go at its start: kernel arguments lie in host
// memory, and the compiler else loads each where it is first used, one round trip after the other
// (time DFT of a 64 x 64 window, T = 32: 5.3 us so, 4.9 here; front of 256 x 512, T = 32, 7 planes 9.0 and 8.5).
template <bool FUSED = false> __device__ __forceinline__ void load_args(const DftArgs &a) {
  asm volatile("" ::"s"(a.r.ring), "s"(a.r.ring_frames), "s"(a.r.first), "s"(a.r.npix), "s"(a.r.T), "s"(a.kb), "s"(a.nb),
               "s"(a.nbc), "s"(a.both), "s"(a.W), "s"(a.nwin), "s"(a.planes), "s"(a.planes_stride), "s"(a.wm_hi),
               "s"(a.wm_lo), "s"(a.lx), "s"(a.ly));
  if constexpr (FUSED)
    asm volatile("" ::"s"(a.tw), "s"(a.H), "s"(a.blk_c), "s"(a.n_planes), "s"(a.grouped), "s"(gridDim.x));
}

// Window of item i where each window has `per` items (no division in the first window, which is all
// of a single-window launch: the integer division is some forty dependent instructions).
__device__ __forceinline__ int window_of(unsigned i, unsigned per) {
  if (i < per) return 0;
  return (int)(i / per);
}

// Ring of window w of the launch (windows of one plan share it up to the first frame).
template <bool GROUPS = false> __device__ __forceinline__ DftRing window_ring(const DftArgs &a, int w) {
  DftRing r = a.r;
  if (GROUPS && a.grouped) {
    r.ring = a.rings[w];
    r.ring_frames = a.ring_frames_w[w];
  }
  if (w != 0) r.first = a.firsts[w];  // (window 0's is in the struct's first lines)
  return r;
}

// Persistent: a block stages the operand matrix once (tens of KB, and index arithmetic per
// element) and then walks groups of four 64-pixel tiles blockIdx, blockIdx + grid, ... of all
// windows of the launch, window-major.  (Windows on the grid's y dimension: eight windows of 256^2,
// T = 64, 29.6 -> 31.0 us.)
template <int NBT, int MODE>
__global__ __launch_bounds__(256) void k_dft(DftArgs a) {
  extern __shared__ float4 lds_dyn[];
  load_args(a);
  dft_stage_matrix<NBT, MODE>(lds_dyn, a.wm_hi, a.wm_lo, a.r.T, threadIdx.x, 256);
  __syncthreads();
  const Band b = pinned_band(a);
  const unsigned quads = (unsigned)((a.r.npix + 255) / 256);  // groups of four tiles of a window
  const bool lens = a.lx != nullptr;
  for (unsigned it = blockIdx.x; it < quads * a.nwin; it += gridDim.x) {
    const unsigned w = window_of(it, quads);
    const DftRing r = window_ring(a, w);
    float2 *planes = a.planes + w * a.planes_stride;
    // an opaque per-tile copy of the lane index keeps the lane-derived LDS and load addresses of
    // the MFMA loop from being hoisted out of the tile loop (where they would hold registers)
    int lane;
    asm volatile("v_mov_b32 %0, %1" : "=v"(lane) : "v"(threadIdx.x & 63));
    // tiles past the end load clamped pixels (dft_px) and store nothing
    const long long p0w = ((long long)(it - w * quads) * 4 + (threadIdx.x >> 6)) * 64;
    uint2 pre[1][dft_pre_steps<MODE>()];
    dft_prefetch<MODE, 1>(r, p0w, lane, pre);
    f4 acc1[1][NBT][4];
    dft_tile<NBT, MODE, 1>(r, lds_dyn, p0w, lane, pre, acc1);
    auto &acc = acc1[0];

    const long long p0 = p0w + 4 * (lane & 15);
    if (p0 >= a.r.npix) continue;
    float2 L[4];
    if (lens) {
      const int y = (int)(p0 / a.W), x = (int)(p0 % a.W);  // W % 4 == 0: same row
      const float2 ly = a.ly[y];
#pragma unroll
      for (int t = 0; t < 4; ++t) L[t] = cmul(a.lx[x + t], ly);
    }
#pragma unroll
    for (int bt = 0; bt < NBT; ++bt) {
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int bin = bt * 8 + 2 * (lane >> 4) + h;
        if (bin >= b.nbc) continue;
        float2 v[4];
        dft_bin_values(b, acc[bt], h, bin, v);
        dft_store_bin(planes, a.r.npix, b, p0, bin, v, L, lens);
      }
    }
  }
}

// FP32 stand-alone time DFT with the real-input symmetry folded (dft_fold_tile): NBF tiles of
// 16 bins per wave (all of the band's tiles: every frame sample is loaded by one wave only).
// Same outputs as k_dft<NBT, 0> up to FP32 rounding, with 2 (T/8) + 1 MFMAs per
// 16 bins and 16 pixels instead of T/2.
// Persistent like k_dft.  The second launch bound (resident blocks per CU) makes the compiler
// keep the accumulators in ordinary registers instead of splitting them off into accumulation
// registers: up to two tiles fit in three waves per SIMD, three and four tiles in two.
constexpr int fold_min_blocks(int nbf) { return nbf <= 2 ? 3 : 2; }
template <int NBF, bool CUT>
__global__ __launch_bounds__(256, fold_min_blocks(NBF)) void k_dft_fold(DftArgs a) {
  extern __shared__ float4 lds_dyn[];
  float *lf = reinterpret_cast<float *>(lds_dyn);
  load_args(a);
  stage_fold_matrix_rt(lf, reinterpret_cast<const float *>(a.wm_hi), a.r.T, NBF, a.nbc, threadIdx.x, 256);
  __syncthreads();
  const Band b = pinned_band(a);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const unsigned quads = (unsigned)((a.r.npix + 255) / 256);  // groups of four tiles of a window
  const bool lens = a.lx != nullptr;
  for (unsigned it = blockIdx.x; it < quads * a.nwin; it += gridDim.x) {
    const unsigned w = window_of(it, quads);
    const DftRing r = window_ring(a, w);
    float2 *planes = a.planes + w * a.planes_stride;
    int lane;  // opaque per tile, as in k_dft
    asm volatile("v_mov_b32 %0, %1" : "=v"(lane) : "v"(threadIdx.x & 63));
    // tiles past the end load clamped pixels (dft_px) and store nothing
    const long long p0w = ((long long)(it - w * quads) * 4 + wave) * 64;
    f4 ac[NBF][4], as[NBF][4];
    dft_fold_tile<NBF, CUT>(r, lf, p0w, lane, ac, as);

    const long long p0 = p0w + 4 * (lane & 15);
    if (p0 >= a.r.npix) continue;
    float2 L[4];
    if (lens) {
      const int y = (int)(p0 / a.W), x = (int)(p0 % a.W);  // W % 4 == 0: same row
      const float2 ly = a.ly[y];
#pragma unroll
      for (int t = 0; t < 4; ++t) L[t] = cmul(a.lx[x + t], ly);
    }
#pragma unroll
    for (int f = 0; f < NBF; ++f) {
#pragma unroll
      for (int rr = 0; rr < 4; ++rr) {
        const int bin = 16 * f + 4 * (lane >> 4) + rr;
        if (bin >= b.nbc) continue;
        const float dc = dc_offset(b.kb, b.T, bin);
        float2 v[4];
#pragma unroll
        for (int t = 0; t < 4; ++t) v[t] = make_float2(ac[f][t][rr] + dc, as[f][t][rr]);
        dft_store_bin(planes, a.r.npix, b, p0, bin, v, L, lens);
      }
    }
  }
}

// ----------------------------------------------------------------------- fused with row FFT
// Planes per LDS group: the group's padded rows fill ~127 KB (15 planes at W = 1024), which
// leaves room for the pass twiddles and the operand matrix of the MFMA loop.
template <int W> constexpr int row_group() { return 130560 / (WaveFft<W>::SCR * 8); }

// Waves per row: one per 64 pixels up to 512 wide, one per 128 pixels (two MFMA tiles
// sharing every operand load) beyond, which keeps 8 waves and a 256-register budget.
template <int W> constexpr int row_tpw() { return W > 512 ? 2 : 1; }
template <int W> constexpr int row_threads() { return W / row_tpw<W>(); }

// MULTI: the planes need more than one LDS group (two-sided bands at large widths); a
// separate instantiation so the common single-group kernel carries no spill code.
template <int W, int NBT, int MODE, bool MULTI>
__global__ __launch_bounds__(row_threads<W>()) void k_dft_row(DftArgs a) {
  load_args<true>(a);
  using F = WaveFft<W>;
  constexpr int TPW = row_tpw<W>();
  constexpr int NT = row_threads<W>();
  constexpr int NW = NT / 64;
  constexpr int E = F::E;
  constexpr int GB = row_group<W>();
  __shared__ float2 scr[GB * F::SCR];  // one padded row per plane of the current group
  __shared__ __align__(16) float2 twl[F::TW];
  extern __shared__ float4 wmat[];     // operand matrix of the MFMA loop

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  dft_stage_matrix<NBT, MODE>(wmat, a.wm_hi, a.wm_lo, a.r.T, tid, NT);
  F::stage_twiddles(twl, a.tw, tid, NT);
  __syncthreads();

  const Band b = pinned_band(a);
  const long long plane_elems = (long long)a.H * W;
  const bool lens = a.lx != nullptr;
  const int G = gridDim.x;
  // rows of all windows of the launch, window-major (MULTI has no registers for the window's
  // pointers: 217 -> 296 us at 1024^2; its launcher runs one window at a time)
  const int rows = MULTI ? a.H : a.H * a.nwin;
  int row = xcd_tile(blockIdx.x, G);
  uint2 pre[TPW][dft_pre_steps<MODE>()];
  auto prefetch = [&](int i, int ln) {
    if constexpr (MULTI) {
      dft_prefetch<MODE, TPW>(a.r, (long long)i * W + wave * 64 * TPW, ln, pre);
    } else {
      const int w = window_of(i, a.H);
      dft_prefetch<MODE, TPW>(window_ring(a, w), (long long)(i - w * a.H) * W + wave * 64 * TPW, ln, pre);
    }
  };
  if (row < rows) prefetch(row, lane);

  for (; row < rows; row += G) {
    const int win = MULTI ? 0 : window_of(row, a.H), y = row - win * a.H;
    // An opaque per-row copy of the lane index keeps the many loop-invariant LDS
    // addresses of the scatter and the transforms out of registers across rows.
    int lane;
    asm volatile("v_mov_b32 %0, %1" : "=v"(lane) : "v"(tid & 63));
    f4 acc[TPW][NBT][4];
    dft_tile<NBT, MODE, TPW>(MULTI ? a.r : window_ring(a, win), wmat, (long long)y * W + wave * 64 * TPW, lane, pre, acc);
    // lens factors of the lane's pixels (1 without a lens: the product with (1, 0) is exact,
    // and cheaper than a select)
    auto lens_factors = [&](int i, float2 (&L)[4]) {
      const int x0 = (wave * TPW + i) * 64 + 4 * (lane & 15);
#pragma unroll
      for (int t = 0; t < 4; ++t) L[t] = make_float2(1.f, 0.f);
      if (lens) {
        const float2 ly = a.ly[y];
#pragma unroll
        for (int t = 0; t < 4; ++t) L[t] = cmul(a.lx[x0 + t], ly);
      }
    };
    // single group: the factors are loaded before the next row's prefetch (loaded after it,
    // their wait would also wait for the prefetch: the vector-memory counter drains in order);
    // MULTI loads them per group in the scatter, where registers are scarcer
    float2 Ls[TPW][4];
    if constexpr (!MULTI) {
#pragma unroll
      for (int i = 0; i < TPW; ++i) lens_factors(i, Ls[i]);
    }
    // the next row's first frames load while this row is scattered and transformed
    if (row + G < rows) prefetch(row + G, lane);

    // scatter planes [q0, q0+GB) from the MFMA registers into padded LDS rows
    auto scatter = [&](int q0) {
#pragma unroll
      for (int i = 0; i < TPW; ++i) {
        const int x0 = (wave * TPW + i) * 64 + 4 * (lane & 15);  // first of the lane's 4 pixels
        float2 L[4];
        if constexpr (MULTI)
          lens_factors(i, L);
        else
#pragma unroll
          for (int t = 0; t < 4; ++t) L[t] = Ls[i][t];
#pragma unroll
        for (int bt = 0; bt < NBT; ++bt) {
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            const int bin = bt * 8 + 2 * (lane >> 4) + h;
            if (bin >= b.nbc) continue;
            float2 v[4];
            dft_bin_values(b, acc[i][bt], h, bin, v);
#pragma unroll
            for (int side = 0; side < 2; ++side) {
              int q;
              if (side == 0) {
                if (bin >= b.nb) continue;
                q = bin;
              } else {
                if (!b.both) continue;
                const int j = b.nb - bin;
                if (j < 0 || j >= b.nb) continue;
                q = b.nb + j;
              }
              if (q < q0 || q >= q0 + GB) continue;
              float2 *dst = scr + (q - q0) * F::SCR;
#pragma unroll
              for (int t = 0; t < 4; ++t) {
                float2 c = side ? make_float2(v[t].x, -v[t].y) : v[t];
                dst[F::pad(x0) + t] = cmul(c, L[t]);  // x0 is a multiple of four
              }
            }
          }
        }
      }
    };
    // one wave per plane row of the group: forward row FFT, then the column-blocked store
    auto transform = [&](int q0) {
      const int q1 = min(q0 + GB, a.n_planes);
      const long long row_off = blk_lane_offset(lane, a.H, a.blk_c) + (long long)y * a.blk_c;
      for (int q = q0 + wave; q < q1; q += NW) {
        float2 *ws = scr + (q - q0) * F::SCR;
        float2 v[E];
#pragma unroll
        for (int m = 0; m < E; ++m) v[m] = lds_get(ws + F::pad(lane) + F::padc(64 * m));
        F::template run<false>(v, ws, twl, lane);
        float2 *dst = a.planes + win * a.planes_stride + (long long)q * plane_elems + row_off;
#pragma unroll
        for (int m = 0; m < E; ++m) dst[(long long)m * 64 * a.H] = v[m];
      }
    };
    if constexpr (!MULTI) {
      // every plane fits one group, so the MFMA accumulators are dead before the
      // transforms need their registers
      scatter(0);
      __syncthreads();
      transform(0);
      __syncthreads();
    } else {
      for (int q0 = 0; q0 < a.n_planes; q0 += GB) {
        scatter(q0);
        __syncthreads();
        transform(q0);
        __syncthreads();
      }
    }
  }
}

// ----------------------------------------------------------------------- pipelined front
// Same result as k_dft_row for a single LDS group of planes (up to FP32 rounding where the
// DFT is folded), with the waves split by role: W/128 producer waves (8 at W = 1024) run the
// MFMA time DFT of the block's next row into registers while the consumer waves run the row
// FFTs of the current row's planes out of LDS and store them; then the producers scatter the
// next row into LDS.  HBM loads and MFMAs of one row overlap the LDS/VALU work and the stores
// of the previous one.
// Producers own 128 pixels each (two 64-pixel MFMA tiles) and stream their frame loads
// through a register ring that runs on across rows: DftStream (interleaved cos/-sin rows, up
// to 8 bins) or DftStreamFold (9..16 bins, real-input symmetry folded).  FP32 only, for T in
// {32, 64, 128}.
// Consumer waves: a block has at most twelve waves where a producer holds the folded DFT's sums
// (three per SIMD, 168 registers; a thirteenth spills: 1024^2 batch 1690 -> 1980 us), so four, six
// and eight at 1024, 768 and 512; up to 8 bins, eight at 512 (four windows of 512^2, T = 32: 92 ->
// 87 us) and four beyond, where eight measured 3-5 % slower.
template <int W> constexpr int front_pw() { return W / 128; }
template <int W, bool FOLD, bool FEW> constexpr int front_cw() {
  return FEW ? 4 : W == 512 ? 8 : FOLD ? 12 - front_pw<W>() : 4;
}
template <int W, int NBT, bool FEW> constexpr int front_threads() { return (front_pw<W>() + front_cw<W, NBT == 2, FEW>()) * 64; }
// k_front: whether the row FFTs' waves issue first.  They are the longer half of a row at 9..16 bins
// (front alone 84.6 -> 75.5 us at 1024^2, T = 64, 15 planes; at up to 8 bins 3 % slower), but a cache
// line of the planes holds four rows, and blocks that run ahead leave it before their neighbours have
// filled it: with T = 32, where the DFT holds them back least, tall frames lose (rows x width, 15
// planes, without -> with: 1024 x 512 33.5 -> 39.7, 1024 x 768 49.1 -> 70.5, 1024^2 54.4 -> 79.8) and only
// short ones gain (512 x 768, 9 planes 24.3 -> 23.0).  Several groups of planes per row hold them back
// too: 1024^2, T = 32, 24 planes 113 -> 92.  With T = 128 the DFT is as long as the FFTs and rows shorter
// than 1024 points lose: 2048 x 512, 15 planes 109 -> 115, 1024 x 768 90 -> 94 (1024^2 121 -> 104).
constexpr bool front_fft_first(int W, bool fold, int T, bool multi, bool tall) {
  if (!fold) return false;
  if (W == 1024) return T > 32 || multi || !tall;
  if (W == 768) return T == 64 || (T == 32 && !multi && !tall);
  return T == 64 && !tall;
}
// 512-point rows of tall frames at T = 64: four consumer waves keep the blocks together (1024 rows,
// windows with 15 planes 70.3 -> 68.0 us, 30 planes 112.5 -> 108.0; batches of 2048 rows with 30 planes 2,035 ->
// 1,873; frames of 512 rows with an angular spectrum 51.0 with eight and priority, 54.1 with four).
constexpr bool front_few(int W, bool fold, int T, bool tall) { return W == 512 && fold && T == 64 && tall; }
// where frames of 1024 rows and more take a form of their own
constexpr bool front_has_tall(int W, bool fold, int T) {
  return front_few(W, fold, T, true) || front_fft_first(W, fold, T, false, true) != front_fft_first(W, fold, T, false, false);
}
// Whether the row FFTs' code of k_front starts on an odd dword.  It is 4- and 8-byte instructions without a
// loop among them, and how they fall on the instruction fetch counts: 1024^2, T = 64, 15 planes take 75 us
// wherever it lands on an odd dword and 79-86 on an even one (the whole kernel moved by 0 to 16 dwords);
// 512-point rows with T = 128 are better on an even one (1024 rows, 30 planes 85 against 89 us), several
// groups of planes with T = 32 too (1024^2, 30 planes 112 against 118), the others differ by less than
// 2 %.  The place is pinned against a 64-byte line, so that nothing ahead of it in the kernel moves it.
constexpr bool front_odd(int W, int T, bool multi) { return !(W == 512 && T == 128) && !(multi && T == 32); }
constexpr int front_ring(int T) { return T / 4 < 8 ? T / 4 : 8; }

// MULTI: the planes take several LDS groups (two-sided bands).  The producers keep a row's spectra
// and scatter one group after the other, each as soon as the consumers are done with the previous
// one; the next row's DFT overlaps the last group's row FFTs.
template <int W, int NBT, int MODE, int T, bool MULTI = false, bool TALL = false>
__global__ __launch_bounds__((front_threads<W, NBT, front_few(W, NBT == 2, T, TALL)>())) void k_front(DftArgs a) {
  constexpr bool FEW = front_few(W, NBT == 2, T, TALL);
  static_assert(MODE == 0, "the pipelined front kernel runs the FP32 time DFT");
  load_args<true>(a);
  using F = WaveFft<W>;
  constexpr int TPW = 2;
  constexpr int NPW = front_pw<W>();
  constexpr int NT = (front_threads<W, NBT, FEW>());
  constexpr int E = F::E;
  constexpr int GB = row_group<W>();
  __shared__ float2 scr[GB * F::SCR];  // one padded row per plane
  __shared__ __align__(16) float2 twl[F::TW];
  extern __shared__ float4 wmat[];     // operand matrix of the MFMA loop

  // one 16-bin tile (NBT == 2: up to 16 bins as 32 interleaved cos/-sin rows): the folded
  // contraction of DftStreamFold, half the MFMAs
  constexpr bool FOLD = NBT == 2;
  const int tid = threadIdx.x;
  const int wave = tid >> 6;
  const bool producer = wave < NPW;    // wave-uniform role
  const int rw = producer ? wave : wave - NPW;
  if constexpr (FOLD)
    stage_fold_matrix_rt(reinterpret_cast<float *>(wmat), reinterpret_cast<const float *>(a.wm_hi), T, 1, a.nbc,
                         tid, NT);
  else
    dft_stage_matrix<NBT, MODE>(wmat, a.wm_hi, a.wm_lo, a.r.T, tid, NT);
  F::stage_twiddles(twl, a.tw, tid, NT);
  __syncthreads();

  const long long plane_elems = (long long)a.H * W;
  const bool lens = a.lx != nullptr;
  const int G = gridDim.x;
  const int y0 = xcd_tile(blockIdx.x, G);
  const int rows = a.H * a.nwin;                           // rows of all windows, window-major
  const int nr = y0 < rows ? (rows - 1 - y0) / G + 1 : 0;  // of them this block's
  // LDS groups of planes, evenly filled
  const int ng = MULTI ? (a.n_planes + GB - 1) / GB : 1;
  const int gp = MULTI ? (a.n_planes + ng - 1) / ng : a.n_planes;

  f4 acc[TPW][NBT][4];        // interleaved rows (!FOLD)
  f4 fre[TPW][4], fim[TPW][4];  // Re and Im of bins 4 g + r (FOLD)
  std::conditional_t<FOLD, DftStreamFold<TPW, T, 4>, DftStream<NBT, TPW, T, front_ring(T)>> stream;
  auto px0 = [&](int y) { return (long long)y * W + rw * 64 * TPW; };
  auto win_of = [&](int i) { return window_of(y0 + i * G, a.H); };
  auto row_y = [&](int i) { return y0 + i * G - win_of(i) * a.H; };
  auto ring_of = [&](int i) { return window_ring<true>(a, win_of(i)); };

  // producers: the band spectra of row i for their 128 pixels
  auto dft_row = [&](int i, int lane) {
    // the last row's refills (never used) all read the first pixels of the window's frames:
    // every wave of every CU loads the same few KB, which stay in L2 instead of costing HBM reads
    const bool next = i + 1 < nr;
    const int j = next ? i + 1 : i;
    const long long pn = next ? px0(row_y(j)) : 0;
    if constexpr (FOLD)
      stream.row(ring_of(i), ring_of(j), wmat, px0(row_y(i)), pn, lane, fre, fim);
    else
      stream.row(ring_of(i), ring_of(j), reinterpret_cast<const float *>(wmat), px0(row_y(i)), pn, lane, acc);
  };
  const Band b = pinned_band(a);
  // producers: MFMA registers of row i -> padded LDS rows (its window's lens for Fresnel)
  auto scatter = [&](int i, int q0, int lane) {  // group of planes from q0
    const int y = row_y(i);
    const float2 *lxw = a.grouped ? a.lx_w[win_of(i)] : a.lx, *lyw = a.grouped ? a.ly_w[win_of(i)] : a.ly;
    // band bin `bin` of 4 pixels from x0 into the LDS plane rows (and its conjugate plane on
    // the two-sided path), lens applied.  The product's rounding is pinned (cmul_rn): the
    // first row is scattered by the copy of this code before the row loop, the others by the
    // copy inside it, and a window's first row may fall in either (a grouped launch), so both
    // copies must round alike.
    auto put = [&](int x0, int bin, const float2 (&v)[4], const float2 (&L)[4]) {
#pragma unroll
      for (int side = 0; side < 2; ++side) {
        int q;
        if (side == 0) {
          if (bin >= b.nb) continue;
          q = bin;
        } else {
          if (!b.both) continue;
          const int j = b.nb - bin;
          if (j < 0 || j >= b.nb) continue;
          q = b.nb + j;
        }
        if (MULTI && (q < q0 || q >= q0 + gp)) continue;
        float2 *dst = scr + (q - q0) * F::SCR;
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          float2 c = side ? make_float2(v[t].x, -v[t].y) : v[t];
          dst[F::pad(x0) + t] = cmul_rn(c, L[t]);  // x0 is a multiple of four
        }
      }
    };
#pragma unroll
    for (int i = 0; i < TPW; ++i) {
      const int x0 = (rw * TPW + i) * 64 + 4 * (lane & 15);
      // lens factors; 1 without a lens (the product with (1, 0) is exact, and cheaper than a select)
      float2 L[4] = {make_float2(1.f, 0.f), make_float2(1.f, 0.f), make_float2(1.f, 0.f), make_float2(1.f, 0.f)};
      if (lens) {
        const float2 ly = lyw[y];
#pragma unroll
        for (int t = 0; t < 4; ++t) L[t] = cmul(lxw[x0 + t], ly);
      }
      if constexpr (FOLD) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          // bins past the computed ones fail put's own tests (nbc = nb, or nb + 1 on the
          // two-sided path, whose conjugate planes use bins 1..nb)
          const int bin = 4 * (lane >> 4) + r;
          // the centring offset restored on the DC bin: a select, not a branch
          const float dc = dc_offset(b.kb, T, bin);
          float2 v[4];
#pragma unroll
          for (int t = 0; t < 4; ++t) v[t] = make_float2(fre[i][t][r] + dc, fim[i][t][r]);
          put(x0, bin, v, L);
        }
      } else {
#pragma unroll
        for (int bt = 0; bt < NBT; ++bt) {
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            const int bin = bt * 8 + 2 * (lane >> 4) + h;
            if (bin >= b.nbc) continue;
            float2 v[4];
            dft_bin_values(b, acc[i][bt], h, bin, v);
            put(x0, bin, v, L);
          }
        }
      }
    }
  };

  // consumers: one wave per plane row: forward row FFT, then the column-blocked store
  auto transform = [&](int i, int q0, int lane) {
    const int y = row_y(i);
    float2 *planes = a.grouped ? a.planes_w[win_of(i)] : a.planes + win_of(i) * a.planes_stride;
    const long long row_off = blk_lane_offset(lane, a.H, a.blk_c) + (long long)y * a.blk_c;
    const int q1 = MULTI ? min(q0 + gp, a.n_planes) : a.n_planes;
    for (int q = q0 + rw; q < q1; q += front_cw<W, FOLD, FEW>()) {
      float2 *ws = scr + (q - q0) * F::SCR;
      float2 v[E];
#pragma unroll
      for (int m = 0; m < E; ++m) v[m] = lds_get(ws + F::pad(lane) + F::padc(64 * m));
      F::template run<false>(v, ws, twl, lane);
      float2 *dst = planes + (long long)q * plane_elems + row_off;
#pragma unroll
      for (int m = 0; m < E; ++m) dst[(long long)m * 64 * a.H] = v[m];
    }
  };

  // The two roles run separate loops (wave-uniform branch) that meet at the same number of
  // workgroup barriers: 1 + 2 per row and group.  Keeping them apart keeps the producers' MFMA
  // accumulators out of the consumers' register allocation.
  if (producer) {
    const int lane0 = tid & 63;
    if (nr > 0) {
      stream.start(ring_of(0), px0(row_y(0)), lane0);
      dft_row(0, lane0);
      scatter(0, 0, lane0);
    }
    __syncthreads();
    for (int i = 0; i < nr; ++i) {
      int lane;
      asm volatile("v_mov_b32 %0, %1" : "=v"(lane) : "v"(tid & 63));
      if constexpr (MULTI) {
        for (int g = 1; g < ng; ++g) {
          __syncthreads();  // consumers are done with row i's planes below group g
          scatter(i, g * gp, lane);
          __syncthreads();
        }
      }
      if (i + 1 < nr) dft_row(i + 1, lane);
      __syncthreads();  // consumers are done with row i's planes
      if (i + 1 < nr) scatter(i + 1, 0, lane);
      __syncthreads();  // row i + 1's planes are in LDS
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the last row's unused refills land first
  } else {
    if constexpr (front_fft_first(W, FOLD, T, MULTI, TALL)) __builtin_amdgcn_s_setprio(3);
    __syncthreads();
    for (int i = 0; i < nr; ++i) {
      for (int g = 0; g < ng; ++g) {
        // the place of the row FFTs' code, pinned (front_odd)
        if constexpr (front_odd(W, T, MULTI))
          asm volatile(".p2align 6\n\ts_nop 0");
        else
          asm volatile(".p2align 6");
        // opaque lane index: keeps loop-invariant LDS addresses out of registers
        int lane;
        asm volatile("v_mov_b32 %0, %1" : "=v"(lane) : "v"(tid & 63));
        transform(i, g * gp, lane);
        __syncthreads();
        __syncthreads();
      }
    }
  }
}

// ----------------------------------------------------------------------- launch
static DftArgs make_args(const DftLaunch &L) {
  DftArgs a{};
  a.r.ring = L.ring;
  a.r.ring_frames = L.ring_frames;
  a.r.first = L.first;
  a.r.npix = L.npix;
  a.r.T = L.T;
  a.W = L.W;
  a.kb = L.kb;
  a.nb = L.nb;
  a.nbc = L.nbc;
  a.both = L.both;
  a.lx = L.lx;
  a.ly = L.ly;
  switch (L.precision) {
    case 0: a.wm_hi = L.wm_f32; break;
    case 2: a.wm_hi = L.wm_bf16; break;
    default: a.wm_hi = L.wm_f16hi; break;
  }
  a.wm_lo = L.wm_f16lo;
  a.nwin = L.nwin > 0 ? L.nwin : 1;
  a.planes = L.planes;
  a.planes_stride = L.planes_stride;
  for (int w = 0; w < a.nwin && w < HFX_MAX_WIN; ++w) a.firsts[w] = (int)(w == 0 ? L.first : L.firsts[w]);
  a.grouped = a.nwin > 1 && L.rings[0] != nullptr;
  for (int w = 0; a.grouped && w < a.nwin && w < HFX_MAX_GROUP; ++w) {
    a.rings[w] = L.rings[w];
    a.ring_frames_w[w] = L.ring_frames_w[w];
    a.planes_w[w] = L.planes_w[w];
    a.lx_w[w] = L.lx_w[w];
    a.ly_w[w] = L.ly_w[w];
  }
  return a;
}

// Grid of a persistent stand-alone DFT kernel: as many blocks as are resident at once (the
// occupancy calculator's count per CU times the CUs), at most one per group of four 64-pixel tiles.
static dim3 persistent_grid(const void *kernel, size_t lds, const DftArgs &a) {
  int per_cu = 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, 256, lds) != hipSuccess || per_cu < 1) per_cu = 1;
  return dim3((unsigned)std::min((a.r.npix + 255) / 256 * a.nwin, (long long)device_cus() * per_cu));
}

template <int NBT, int MODE> static int launch_plain(const DftArgs &a, hipStream_t st) {
  const size_t lds = dft_matrix_lds_bytes(NBT, MODE, a.r.T);
  const dim3 grid = persistent_grid(reinterpret_cast<const void *>(&k_dft<NBT, MODE>), lds, a);
  hipLaunchKernelGGL((k_dft<NBT, MODE>), grid, dim3(256), lds, st, a);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

template <int NBT> static int launch_plain_mode(const DftArgs &a, int mode, hipStream_t st) {
  switch (mode) {
    case 0: return launch_plain<NBT, 0>(a, st);
    case 1: return launch_plain<NBT, 1>(a, st);
    case 2: return launch_plain<NBT, 2>(a, st);
    case 3: return launch_plain<NBT, 3>(a, st);
  }
  return -2;
}

template <int NBF, bool CUT> static int launch_fold_cut(const DftArgs &a, hipStream_t st) {
  const size_t lds = dft_fold_lds_bytes(NBF, a.r.T);
  const dim3 grid = persistent_grid(reinterpret_cast<const void *>(&k_dft_fold<NBF, CUT>), lds, a);
  hipLaunchKernelGGL((k_dft_fold<NBF, CUT>), grid, dim3(256), lds, st, a);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

template <int NBF> static int launch_fold(const DftArgs &a, hipStream_t st) {
  return a.r.T % 32 == 0 ? launch_fold_cut<NBF, false>(a, st) : launch_fold_cut<NBF, true>(a, st);
}

int launch_time_dft(const DftLaunch &L, hipStream_t st) {
  if (L.nwin > HFX_MAX_WIN) return -6;
  const DftArgs a = make_args(L);
  // FP32 with more than one 16-row tile of interleaved rows: the folded contraction.  Its last batch
  // of steps may be cut short, so any T % 4 == 0 runs (512 x 768, T = 48, 12 bins: 29.6 us with k_dft,
  // 20.5 folded); longer windows that are no multiple of 32 stay on k_dft, whose larger operand
  // matrix sets the window lengths that such a band accepts.
  if (L.precision == 0 && (L.T % 32 == 0 || L.T <= 256) && L.nbc > 8 && L.nbc <= 64) {
    switch ((L.nbc + 15) / 16) {
      case 1: return launch_fold<1>(a, st);
      case 2: return launch_fold<2>(a, st);
      case 3: return launch_fold<3>(a, st);
      case 4: return launch_fold<4>(a, st);
    }
  }
  switch ((2 * L.nbc + 15) / 16) {
    case 1: return launch_plain_mode<1>(a, L.precision, st);
    case 2: return launch_plain_mode<2>(a, L.precision, st);
    case 3: return launch_plain_mode<3>(a, L.precision, st);
    case 4: return launch_plain_mode<4>(a, L.precision, st);
    case 5: return launch_plain_mode<5>(a, L.precision, st);
    case 6: return launch_plain_mode<6>(a, L.precision, st);
    case 7: return launch_plain_mode<7>(a, L.precision, st);
    case 8: return launch_plain_mode<8>(a, L.precision, st);
  }
  return -2;
}

bool dft_row_supported(int W, int nbc, int T) {
  return (W == 512 || W == 768 || W == 1024) && (2 * nbc + 15) / 16 <= 2 && T <= 128;
}

bool dft_front_pipelined(int W, int nbc, int T, int n_planes, int precision) {
  if (!dft_row_supported(W, nbc, T) || precision != 0 || !(T == 32 || T == 64 || T == 128)) return false;
  const int group = W == 512 ? row_group<512>() : W == 768 ? row_group<768>() : row_group<1024>();
  return n_planes <= group;
}

template <int W, int NBT, int MODE> static int launch_row(const DftArgs &a, hipStream_t st) {
  const size_t lds = dft_matrix_lds_bytes(NBT, MODE, a.r.T);
  // persistent grid: one workgroup per CU (the LDS footprint allows no more), each walking rows
  // blockIdx, blockIdx + grid, ... of the launch's windows
  const int cus = device_cus();
  const long long rows = (long long)a.H * a.nwin;
  const unsigned grid = (unsigned)(rows < cus ? rows : cus);
  const int T = a.r.T;
  // several groups need more than 8 computed bins at every width (two-sided, 16 planes or more)
  constexpr bool CAN_MULTI = NBT == 2 && W > 512;
  const bool multi = a.n_planes > row_group<W>();
  if (MODE == 0 && (CAN_MULTI || !multi) && (T == 32 || T == 64 || T == 128)) {
    const dim3 g(grid);
    auto go = [&](auto t) {
      constexpr int TT = decltype(t)::value;
      constexpr bool CAN_TALL = front_has_tall(W, NBT == 2, TT), FEW = front_few(W, NBT == 2, TT, CAN_TALL);
      if (multi)
        hipLaunchKernelGGL((k_front<W, NBT, 0, TT, CAN_MULTI>), g, dim3(front_threads<W, NBT, false>()), lds, st, a);
      else if (CAN_TALL && a.H >= 1024)
        hipLaunchKernelGGL((k_front<W, NBT, 0, TT, false, CAN_TALL>), g, dim3(front_threads<W, NBT, FEW>()), lds, st, a);
      else
        hipLaunchKernelGGL((k_front<W, NBT, 0, TT>), g, dim3(front_threads<W, NBT, false>()), lds, st, a);
    };
    if (T == 32)
      go(std::integral_constant<int, 32>{});
    else if (T == 64)
      go(std::integral_constant<int, 64>{});
    else
      go(std::integral_constant<int, 128>{});
  } else if (a.n_planes <= row_group<W>()) {
    hipLaunchKernelGGL((k_dft_row<W, NBT, MODE, false>), dim3(grid), dim3(row_threads<W>()), lds, st, a);
  } else if constexpr (CAN_MULTI) {
    for (int w = 0; w < a.nwin; ++w) {  // one window per launch
      DftArgs one = a;
      one.r.first = a.firsts[w];
      one.planes = a.planes + w * a.planes_stride;
      hipLaunchKernelGGL((k_dft_row<W, NBT, MODE, true>), dim3((unsigned)(a.H < cus ? a.H : cus)), dim3(row_threads<W>()),
                         lds, st, one);
    }
  } else {
    return -2;
  }
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

template <int W, int NBT> static int launch_row_mode(const DftArgs &a, int mode, hipStream_t st) {
  switch (mode) {
    case 0: return launch_row<W, NBT, 0>(a, st);
    case 1: return launch_row<W, NBT, 1>(a, st);
    case 2: return launch_row<W, NBT, 2>(a, st);
    case 3: return launch_row<W, NBT, 3>(a, st);
  }
  return -2;
}

template <int W> static int launch_row_w(const DftArgs &a, int nbt, int mode, hipStream_t st) {
  if (nbt == 1) return launch_row_mode<W, 1>(a, mode, st);
  if (nbt == 2) return launch_row_mode<W, 2>(a, mode, st);
  return -2;
}

int launch_time_dft_row(const DftLaunch &L, int H, int blk_c, int n_planes, const float2 *tw,
                        hipStream_t st) {
  if (!dft_row_supported(L.W, L.nbc, L.T)) return -2;
  if (L.nwin > HFX_MAX_WIN || (long long)H * (L.nwin > 1 ? L.nwin : 1) > INT32_MAX) return -6;
  // windows of several plans: only k_front reads their tables
  if (L.nwin > 1 && L.rings[0] != nullptr &&
      (L.nwin > HFX_MAX_GROUP || !dft_front_pipelined(L.W, L.nbc, L.T, n_planes, L.precision)))
    return -6;
  DftArgs a = make_args(L);
  a.H = H;
  a.blk_c = blk_c;
  a.n_planes = n_planes;
  a.tw = tw;
  const int nbt = (2 * L.nbc + 15) / 16;
  switch (L.W) {
    case 512: return launch_row_w<512>(a, nbt, L.precision, st);
    case 768: return launch_row_w<768>(a, nbt, L.precision, st);
    case 1024: return launch_row_w<1024>(a, nbt, L.precision, st);
  }
  return -2;
}

}  // namespace hfx
