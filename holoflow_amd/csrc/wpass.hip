// Row and column passes of the spatial 2-D FFT, built on the wave-level FFT (wfft.hh).
//
// Kernel kinds (compile-time, so each kernel carries only its own data path):
//   NAT_TO_BLK : natural complex or real input (optionally centred in a zero-padded grid
//                and times the Fresnel lens) -> column-blocked spectrum      (row pass)
//   BLK_TO_MOM : column-blocked input -> transform -> moment images, summing over all planes
//                (row pass inverse for the angular spectrum, column pass forward for
//                Fresnel); BLK_TO_MOM5 also makes the two band-split M0 images
//   BLK_MID    : column-blocked -> forward, times the transfer function, inverse ->
//                column-blocked in place                                      (column pass)
//   BLK_LENS   : column-blocked -> inverse, times the Fresnel lens, forward -> column-blocked in
//                place (row pass between Filter2D's spectrum and the propagation's)
//   BLK_TO_NAT : column-blocked -> transform -> natural complex (optionally times the
//                output lens), natural |X| or natural real part
//
// Column-blocked layout of one H x W plane with block width C (C | W):
//   (y, x) -> (x / C) * H * C + y * C + x % C
//
// Work split: a wave owns P = 64 / L transforms (one from 256 points on).  The moment kinds
// also split the planes over S subsets of waves, whose partial sums are added in a fixed order
// through LDS at the end, so results are deterministic.
//
// Moment epilogue (graph_builder.cc:604-647, mean_abs.cu:239-276, mean.cu:268-306):
//   a_k = |X_k| (or |X_k|^2), M0 = sum_k a_k / n, M1 = sum_k (f_k a_k) / n,
//   M2 = sum_k (f_k^2 a_k) / n, summed in ascending k within a subset with the products rounded
//   before the sum as the reference's multiply-then-mean does; stored with the optional
//   fftshift out[i] = in[(i + n/2) mod n] (fftshift.cu:110-145).
#include <algorithm>
#include <type_traits>

#include "hfx_kernels.hh"
#include "wfft.hh"

namespace hfx {

namespace {

enum Kind { NAT_TO_BLK = 0, BLK_TO_MOM = 1, BLK_MID = 2, BLK_TO_NAT = 3, BLK_TO_MOM5 = 4, BLK_LENS = 5 };
constexpr bool is_mom(int k) { return k == BLK_TO_MOM || k == BLK_TO_MOM5; }
// Transform direction each kind is compiled for: the row pass out of natural data is
// forward (it feeds the column pass), the row passes that read the blocked spectrum back
// (angular spectrum) are inverse, and every column pass is forward (BLK_MID runs forward,
// transfer function, inverse; BLK_LENS starts inverse).  The launchers reject a PassArgs::inv that disagrees.
constexpr bool row_inv(int k) { return k != NAT_TO_BLK; }

__device__ __forceinline__ float magnitude(float2 v, bool power2) {
  const float a = sq_mag(v);
  return power2 ? a : mag_sqrt(a);
}

// Running sums of one lane's E pixels: a, f a, f^2 a; with a band split, sum 0 holds the planes
// below the split and sum 3 those from it on (M0 is their sum).
template <int E, bool BAND> struct Moments {
  static constexpr int NACC = BAND ? 4 : 3;
  float s[NACC][E];
  __device__ __forceinline__ void zero() {
#pragma unroll
    for (int k = 0; k < NACC; ++k)
#pragma unroll
      for (int m = 0; m < E; ++m) s[k][m] = 0.f;
  }
  // f, f2: the plane's M1/M2 weights, read by the caller at the top of its plane iteration
  // (wave-uniform scalar loads) so that their latency is not paid after the transform
  template <bool HI> __device__ __forceinline__ void add(const float2 (&v)[E], float f, float f2, bool power2) {
#pragma unroll
    for (int m = 0; m < E; ++m) add_mag<HI>(m, magnitude(v[m], power2), f, f2);
  }
  template <bool HI> __device__ __forceinline__ void add_mag(int m, float a, float f, float f2) {
    s[HI ? 3 : 0][m] += a;
    s[1][m] += __fmul_rn(f, a);
    s[2][m] += __fmul_rn(f2, a);
  }
};

// Sums of the S plane subsets of a block, added in subset order: thread t (of the 64 * waves
// threads that hold one subset) of subset `sub` gets the elements m = sub, sub + S, ... of its
// position, so the additions and the stores after them are spread over all waves.  Two of the
// sums fit the transforms' scratch at a time.  tr: the thread whose pixels this one reads back (t,
// or with TR another mapping that suits the stores better).
template <int E, int S, int NACC, bool TR = false>
__device__ __forceinline__ void fold_subsets(const float (&s)[NACC][E], float *red, int sub, int t, int tr, int nt,
                                             float (&val)[NACC][(E + S - 1) / S]) {
  constexpr int IT = (E + S - 1) / S;
  if constexpr (S == 1 && !TR) {
#pragma unroll
    for (int k = 0; k < NACC; ++k)
#pragma unroll
      for (int m = 0; m < E; ++m) val[k][m] = s[k][m];
  } else {
#pragma unroll
    for (int k0 = 0; k0 < NACC; k0 += 2) {
      __syncthreads();  // the scratch (or the previous two sums) is free
#pragma unroll
      for (int k = k0; k < NACC && k < k0 + 2; ++k)
#pragma unroll
        for (int m = 0; m < E; ++m) red[(((k - k0) * S + sub) * E + m) * nt + t] = s[k][m];
      __syncthreads();
#pragma unroll
      for (int k = k0; k < NACC && k < k0 + 2; ++k)
#pragma unroll
        for (int it = 0; it < IT; ++it) {
          const int m = sub + it * S;
          float x = 0.f;
          if (m < E) {
            x = red[((k - k0) * S * E + m) * nt + tr];
#pragma unroll
            for (int j = 1; j < S; ++j) x += red[(((k - k0) * S + j) * E + m) * nt + tr];
          }
          val[k][it] = x;
        }
    }
  }
}

// The pointers of this block's window: win[blockIdx.z] of a grouped launch (G), else the
// pass's own plus blockIdx.z window strides (0 for a single window).  Grouped launches are
// separate instantiations: reading the pointers through the window table changes how the
// compiler schedules the loads (measured 685 -> 1270 us for the 2048-point moment row pass).
template <bool G> __device__ __forceinline__ PassWin pass_window(const PassArgs &a) {
  if constexpr (G) {
    return a.win[blockIdx.z];
  } else {
    const long long z = blockIdx.z;
    PassWin w;
    w.in = reinterpret_cast<const char *>(a.in) + z * a.win_in;
    w.out = a.out;
    w.mid_tf = a.mid_tf;
#pragma unroll
    for (int k = 0; k < 5; ++k) w.mom_out[k] = a.mom.out[k] + z * a.win_mom;
    return w;
  }
}

// offset of pixel (y, x) in a moment image (fftshift applied on store when asked)
__device__ __forceinline__ long long moment_index(const PassArgs &a, int y, int x) {
  int ys = y, xs = x;  // 0 <= y < H, 0 <= x < W
  if (a.mom.shift) {   // (y + H - H/2) mod H, without a division
    ys = y + (a.H - a.H / 2);
    if (ys >= a.H) ys -= a.H;
    xs = x + (a.W - a.W / 2);
    if (xs >= a.W) xs -= a.W;
  }
  return (long long)ys * a.W + xs;
}

template <int NACC, int IT>
__device__ __forceinline__ void store_moment(const PassArgs &a, const PassWin &pw, int y, int x,
                                             const float (&val)[NACC][IT], int it) {
  const long long o = moment_index(a, y, x);
  const float n_all = (float)a.planes;
  if constexpr (NACC == 4) {
    pw.mom_out[0][o] = (val[0][it] + val[3][it]) / n_all;
    pw.mom_out[3][o] = val[0][it] / (float)a.mom.split;
    pw.mom_out[4][o] = val[3][it] / (float)(a.planes - a.mom.split);
  } else {
    pw.mom_out[0][o] = val[0][it] / n_all;
  }
  pw.mom_out[1][o] = val[1][it] / n_all;
  pw.mom_out[2][o] = val[2][it] / n_all;
}

}  // namespace

// ------------------------------------------------------------------------- row pass
// Waves per workgroup that own rows (RW).  Each wave owns padded scratch rows in LDS and the
// workgroup shares one twiddle table, so the LDS footprint sets the occupancy: at 2048 points
// four waves (86 KB) leave one workgroup, one wave per SIMD, per CU, while eight waves in one
// workgroup (155 KB) give two waves per SIMD to hide the memory latency; at 1024 points eight
// waves (77 KB) give four per SIMD instead of three.  The moment kinds keep four: their sums
// leave no register room.  Short transforms take one wave per block, so that a small image still
// reaches many CUs.
//
// Planes over waves in the moment kinds (S waves per row).  Below 256 points eight waves sum one
// subset of the planes each, folded at the end (a 64 x 64 window's moment pass: 14.7 -> 4.6 us
// against one wave for all planes).  From 256 points on the sums run over the planes in order,
// so that they do not depend on the launch: either one wave does all planes of its row, or, with
// SPLIT, S waves transform S planes at a time, hand their magnitudes over through LDS, and each
// adds up its share of the row's elements.  That takes one row per block up to 1024 points (the
// waves of a row wait for each other only, and a few hundred rows still reach every CU), and
// eight waves per block at 2048, where a block fills the CU.
//
// Launches of few rows split: one wave per row leaves most SIMDs empty there.  The more rows, the
// more planes it takes to win back the rounds that S planes do not fill; from 1024 rows on the
// chip is full without it.  Row pass, one wave per row -> split: 256 x 512 with 1, 4, 16 planes 5.0 ->
// 4.5, 7.6 -> 5.1, 18.8 -> 10.0 us; 512 x 1024 with 1, 2, 5, 15 planes 7.9 -> 7.8, 9.8 -> 8.7, 15.7 ->
// 13.5, 34.2 -> 24.3; 512 x 2048 with 2, 5, 15 20.1 -> 15.9, 34.3 -> 31.5, 74.3 -> 65.5; 768 x 768 with 3,
// 4, 5, 6, 7, 8, 15 11.4 -> 10.9, 13.1 -> 11.6, 14.7 -> 15.9, 16.4 -> 16.4, 18.3 -> 16.8, 19.9 -> 17.8, 31.7
// -> 27.8; 1024 x 1024 with 5, 16 planes 18.5 -> 21.9, 39.6 -> 39.9.  Above 512 rows one wave per row
// stays better where the last-level cache does not hold the planes (768 x 1024 with 40, 44, 52
// planes 80.3 -> 75.6, 92.2 -> 104, 115 -> 147) and for 2048-point rows with the band split, whose
// block of eight waves holds two rows only (768 x 2048 with 9, 20 planes 55 -> 64, 101 -> 115).
constexpr bool wrow_splits(long long rows, int planes, int n, bool band) {
  if (rows <= 512) return rows <= 256 || planes >= 2;
  return rows < 1024 && (planes >= 8 || planes % 4 == 3 || planes % 4 == 0) && rows * planes * n * 8 <= 256LL << 20 &&
         !(n >= 2048 && band);
}
constexpr int wrow_subsets(int n, int kind, bool split) {
  if (!is_mom(kind)) return 1;
  return n < 256 ? 8 : !split ? 1 : n >= 2048 && kind == BLK_TO_MOM ? 2 : 4;
}
constexpr int wrow_waves(int n, int kind, bool split) {
  if (n < 256) return 1;
  if (!is_mom(kind)) return n >= 1024 ? 8 : 4;
  return !split ? 4 : n >= 2048 ? 8 / wrow_subsets(n, kind, true) : 1;
}
constexpr int wrow_threads(int n, int kind, bool split) {
  return 64 * wrow_waves(n, kind, split) * wrow_subsets(n, kind, split);
}

// IN (NAT_TO_BLK only): 1 = the input is a complex plane of the output's size with no lens, so a
// row loads from one base address with no per-element bounds checks or index products; 2 = the
// same times the lens; 3 = a complex plane centred in zeros, no lens; 0 = any input.  Rows outside the
// input plane are not computed: the column pass takes them as zeros (k_wcol, PADDED).  512 x 768
// padded to 768 x 1024, 12 planes: row pass 28.6 -> 20.8 us against transforming all rows through the
// general load, column pass 47.7 -> 44.0.
template <int N, int KIND, bool G = false, int IN = 0, bool SPLIT = false>
__global__ __launch_bounds__(wrow_threads(N, KIND, SPLIT)) void k_wrow(PassArgs a) {
  using F = WaveFft<N>;
  constexpr int E = F::E, L = F::L, P = F::P;
  constexpr int RW = wrow_waves(N, KIND, SPLIT), S = wrow_subsets(N, KIND, SPLIT);
  __shared__ __align__(16) float2 scr[RW * S * P * F::SCR];
  __shared__ __align__(16) float2 twl[F::TWL];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int rw = wave % RW, sub = wave / RW;
  const int l = lane % L, p = lane / L;
  const int y = (xcd_tile(blockIdx.x, gridDim.x) * RW + rw) * P + p + (KIND == NAT_TO_BLK ? a.off_y : 0);
  const int yend = KIND == NAT_TO_BLK ? a.off_y + a.in_h : a.H;
  const bool active = y < yend;
  const int yl = active ? y : yend - 1;  // rows past the end load the last row and store nothing
  const PassWin pw = pass_window<G>(a);
  const int C = a.blk_c;
  const long long plane_elems = (long long)a.H * a.W;
  float2 *ws = scr + (wave * P + p) * F::SCR;

  // blocked offset of element m of the lane's row, (yl, l + L m)
  const long long boff = blk_lane_offset(l, a.H, C) + (long long)yl * C;
  const long long mstep = (long long)L * a.H;
  auto blk = [&](int m) {
    if constexpr (L >= 4)
      return boff + m * mstep;  // C divides L
    else
      return blk_lane_offset(l + L * m, a.H, C) + (long long)yl * C;
  };
  auto load = [&](float2 (&v)[E], long long q) {
    if constexpr (KIND != NAT_TO_BLK) {
      const float2 *in = reinterpret_cast<const float2 *>(pw.in) + q * plane_elems;
#pragma unroll
      for (int m = 0; m < E; ++m) v[m] = in[blk(m)];
    } else if constexpr (IN == 3) {
      const float2 *row = reinterpret_cast<const float2 *>(pw.in) + (q * a.in_h + (yl - a.off_y)) * a.in_w;
#pragma unroll
      for (int m = 0; m < E; ++m) {
        const int xi = l + L * m - a.off_x;
        const float2 t = row[min(max(xi, 0), a.in_w - 1)];
        const bool in = xi >= 0 && xi < a.in_w;
        v[m] = make_float2(in ? t.x : 0.f, in ? t.y : 0.f);
      }
    } else if constexpr (IN != 0) {
      const float2 *row = reinterpret_cast<const float2 *>(pw.in) + q * plane_elems + (long long)yl * N;
#pragma unroll
      for (int m = 0; m < E; ++m) v[m] = row[l + L * m];
      if constexpr (IN == 2) {
        const float2 ly = a.pre_ly[yl];
#pragma unroll
        for (int m = 0; m < E; ++m) v[m] = cmul(v[m], cmul(a.pre_lx[l + L * m], ly));
      }
    } else {
#pragma unroll
      for (int m = 0; m < E; ++m) {
        const int x = l + L * m;
        const int yi = yl - a.off_y, xi = x - a.off_x;
        float2 t = make_float2(0.f, 0.f);
        if (xi >= 0 && xi < a.in_w) {
          const long long o = q * (long long)a.in_h * a.in_w + (long long)yi * a.in_w + xi;
          if (a.in_mode == IN_NAT_C)
            t = reinterpret_cast<const float2 *>(pw.in)[o];
          else
            t = make_float2(reinterpret_cast<const float *>(pw.in)[o], 0.f);
          if (a.pre_lx) t = cmul(t, cmul(a.pre_lx[xi], a.pre_ly[yi]));
        }
        v[m] = t;
      }
    }
  };
  // the first plane's row loads while the twiddles are staged (at 2048 points, where a block holds
  // the whole CU, loads ahead of the table measured slower: 850 against 730 us for 52 planes)
  float2 v[E];
  const int q0 = is_mom(KIND) ? (sub < a.planes ? sub : a.planes - 1) : (int)blockIdx.y;
  if constexpr (N < 2048) load(v, q0);
  F::stage_twiddles(twl, a.tw, tid, 64 * RW * S);
  __syncthreads();
  if constexpr (N >= 2048) load(v, q0);

  if constexpr (is_mom(KIND) && SPLIT) {
    static_assert(P == 1 && E % S == 0, "a wave's share of the elements");
    constexpr bool BAND = KIND == BLK_TO_MOM5;
    constexpr int ES = E / S, NACC = Moments<ES, BAND>::NACC;
    Moments<ES, BAND> acc;
    acc.zero();
    // the magnitudes of a wave's plane, in its own scratch
    float *own = reinterpret_cast<float *>(ws);
    const float *mine = reinterpret_cast<const float *>(scr + rw * F::SCR) + sub * ES * L + l;
    for (int qb = 0; qb < a.planes; qb += S) {
      float f[S], f2[S];
#pragma unroll
      for (int j = 0; j < S; ++j) {
        f[j] = a.mom.f[min(qb + j, a.planes - 1)];
        f2[j] = a.mom.f2[min(qb + j, a.planes - 1)];
      }
      F::template stage_in<row_inv(KIND)>(v, ws, l);
      load(v, min(qb + sub + S, a.planes - 1));  // as below; past the last plane: unused
      float2 o[E];
      F::template stage_out<row_inv(KIND)>(o, ws, twl, l);
      float mag[E];
#pragma unroll
      for (int m = 0; m < E; ++m) mag[m] = magnitude(o[m], a.mom.power2);
      __builtin_amdgcn_wave_barrier();
#pragma unroll
      for (int m = 0; m < E; ++m) lds_put(own + l + L * m, mag[m]);
      __syncthreads();
#pragma unroll
      for (int j = 0; j < S; ++j) {
        if (qb + j >= a.planes) break;
        const float *from = mine + j * RW * F::SCR * 2;
        if (BAND && qb + j >= a.mom.split) {
#pragma unroll
          for (int m = 0; m < ES; ++m) acc.template add_mag<BAND>(m, from[L * m], f[j], f2[j]);
        } else {
#pragma unroll
          for (int m = 0; m < ES; ++m) acc.template add_mag<false>(m, from[L * m], f[j], f2[j]);
        }
      }
      __syncthreads();
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // an unused last refill lands first
    if (!active) return;
#pragma unroll
    for (int m = 0; m < ES; ++m) store_moment<NACC, ES>(a, pw, y, l + L * (sub * ES + m), acc.s, m);
  } else if constexpr (is_mom(KIND)) {
    constexpr bool BAND = KIND == BLK_TO_MOM5;
    Moments<E, BAND> acc;
    acc.zero();
    int q = sub;
    // (the band split as two loops: fewer sums are live at a time)
    auto run_planes = [&](int end, auto hi) {
      for (; q < end; q += S) {
        const float f = a.mom.f[q], f2 = a.mom.f2[q];
        F::template stage_in<row_inv(KIND)>(v, ws, l);
        // the next plane's row is loaded once pass 1 has moved this one into the scratch, so its
        // latency overlaps the remaining passes; the load is unconditional (the last one reloads
        // the last plane, unused), which keeps it out of a branch
        load(v, q + S < a.planes ? q + S : q);
        float2 o[E];
        F::template stage_out<row_inv(KIND)>(o, ws, twl, l);
        acc.template add<decltype(hi)::value>(o, f, f2, a.mom.power2);
      }
    };
    if constexpr (BAND) {
      run_planes(a.mom.split, std::false_type{});
      run_planes(a.planes, std::true_type{});
    } else {
      run_planes(a.planes, std::false_type{});
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // an unused last refill lands first
    constexpr int IT = (E + S - 1) / S, NACC = Moments<E, BAND>::NACC;
    float val[NACC][IT];
    fold_subsets<E, S, NACC>(acc.s, reinterpret_cast<float *>(scr), sub, rw * 64 + lane, rw * 64 + lane, 64 * RW, val);
#pragma unroll
    for (int it = 0; it < IT; ++it) {
      const int m = sub + it * S;
      if (m < E && active) store_moment<NACC, IT>(a, pw, y, l + L * m, val, it);
    }
  } else {
    F::template stage_in<row_inv(KIND)>(v, ws, l);
    float2 o[E];
    F::template stage_out<row_inv(KIND)>(o, ws, twl, l);
    if constexpr (KIND == BLK_LENS) {
      const float2 ly = a.pre_ly[yl];
#pragma unroll
      for (int m = 0; m < E; ++m) o[m] = cmul(o[m], cmul(a.pre_lx[l + L * m], ly));
      F::template run<false>(o, ws, twl, l);
    }
    if (!active) return;
    if constexpr (KIND == NAT_TO_BLK || KIND == BLK_LENS) {
      float2 *dst = reinterpret_cast<float2 *>(pw.out) + q0 * plane_elems;
#pragma unroll
      for (int m = 0; m < E; ++m) dst[blk(m)] = o[m];
    } else if (a.out_mode == OUT_NAT_RE) {
      float *dst = reinterpret_cast<float *>(pw.out) + q0 * plane_elems + (long long)y * N;
#pragma unroll
      for (int m = 0; m < E; ++m) dst[l + L * m] = o[m].x;
    } else {
      float2 *dst = reinterpret_cast<float2 *>(pw.out) + q0 * plane_elems + (long long)y * N;
#pragma unroll
      for (int m = 0; m < E; ++m) dst[l + L * m] = o[m];
    }
  }
}

// ------------------------------------------------------------------------- column pass
// Waves per workgroup that own columns (WC, of P columns each) and, for the moment kinds, plane
// subsets (S).  A wave keeps its columns (E values per lane) and their moment sums in
// registers.  At 1024 rows three subsets (12 waves, 3 per SIMD) without a register prefetch
// measured faster than two subsets with the next plane prefetched; the four-sum kind (band
// split) takes two (8 waves, 256 registers each), and 2048-row columns leave room for one.
// The plane-parallel kinds take one plane per block; at 2048 rows eight waves share one twiddle
// table (155 KB of LDS, two waves per SIMD instead of one).  At 1024 rows eight waves in the
// plane-parallel kinds, or four (NARROW) where the grid is small (wcol_narrow).  Short columns as in
// the row pass.
constexpr int wcol_subsets(int n, int kind) {
  return !is_mom(kind) || n >= 2048 ? 1 : n >= 256 ? (kind == BLK_TO_MOM5 ? 2 : 3) : 8;
}
constexpr int wcol_waves(int n, int kind, bool narrow = false) {
  return n < 256 ? 1 : kind == BLK_TO_NAT || (n >= 1024 && !is_mom(kind) && !narrow) ? 8 : 4;
}
constexpr int wcol_threads(int n, int kind, bool narrow = false) {
  return 64 * wcol_waves(n, kind, narrow) * wcol_subsets(n, kind);
}
// 1024-row columns with a transfer function in `blocks4` blocks of four waves: those, while they all
// run at once (three per CU) and leave the busiest CU fewer waves than blocks of eight would.  Eight
// -> four: 768 x 1024 planes (W x H) with 3 planes (576 blocks) 19.4 -> 16.2 us, 512 wide with 5 (640)
// 19.2 -> 16.5, 128 wide with 7 (224) 13.1 -> 11.8; 512 wide with 3 (384) 12.7 -> 12.9, 768 wide with 7
// (1,344) 29.9 -> 32.8.
constexpr bool wcol_narrow(long long blocks4, int cus) {
  return blocks4 <= 3LL * cus && 4 * ((blocks4 + cus - 1) / cus) < 8 * ((blocks4 + 2 * cus - 1) / (2 * cus));
}

// LOOP (BLK_MID): 2048-row columns, where a block fills the CU, so that nothing else runs while it
// starts, loads its first columns and drains: one block per CU stays and walks the (tile, plane) items, each
// loading its next column behind the inverse transform and the stores of this one.  The waves load
// in step, since four columns share every cache line (without the barrier they drift apart and the
// pass is slower than one item per block: 1.9 ms).  52 planes of 2048^2 with the moment pass behind
// it: 1677 -> 1596 us.  At 1024 rows and below, where blocks share a CU, one item per block is
// faster (28 planes of 1024^2 with the moment pass: 169 against 176).
// PADDED (BLK_MID): only the rows [row0, row1) of the input were written; the others are zero.
// The 2048-row moment kinds, one wave per SIMD, let their LDS accesses be paired: 52 planes of 2048^2
// 630 -> 541 us, of 2048 x 512 303 -> 254 (the 2048-row transfer-function kind, two waves per SIMD, is
// 3 % slower with pairs, and the shorter lengths are even or slower).
template <int N, int KIND, bool G = false, bool PADDED = false, bool LOOP = false, bool NARROW = false>
__global__ __launch_bounds__(wcol_threads(N, KIND, NARROW)) void k_wcol(PassArgs a) {
  using F = WaveFft<N, is_mom(KIND) && N >= 2048>;
  constexpr int E = F::E, L = F::L, P = F::P;
  constexpr int S = wcol_subsets(N, KIND), WC = wcol_waves(N, KIND, NARROW);
  __shared__ __align__(16) float2 scr[WC * S * P * F::SCR];
  __shared__ __align__(16) float2 twl[F::TWL];
  const int tid = threadIdx.x, lane = tid & 63;
  // wave-uniform to the compiler too: plane indices, weights and tile offsets become scalars
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wc = wave % WC, sub = wave / WC;
  // lane -> (column p of the wave, lane l of its transform): four columns first, so that
  // consecutive lanes read consecutive elements of the blocked layout
  constexpr int Q = P < 4 ? P : 4;
  const int l = (lane / Q) % L, p = lane % Q + Q * (lane / (Q * L));

  const int C = a.blk_c;
  // column tiles in contiguous runs per XCD: the moment images are written column-wise, so
  // the 8 tiles that share an output cache line (32 floats) then share an L2 that merges
  // their 16-byte pieces before they go out
  // BLK_MID multiplies every plane's column by the same transfer-function tile, so its blocks
  // run plane-fastest (block = tile * planes + plane, in contiguous runs per XCD): the planes
  // of one tile are in flight together on one XCD and read the table tile from its L2,
  // instead of the whole table streaming from memory once per plane.
  int bt, bp, item = 0, item_end = 0;
  if constexpr (LOOP) {
    // one eighth of the items to each XCD, whose blocks walk it side by side
    const long long items = (long long)((a.W + WC * P - 1) / (WC * P)) * a.planes;
    const int xcd = blockIdx.x % 8;
    item = (int)(items * xcd / 8) + blockIdx.x / 8;
    item_end = (int)(items * (xcd + 1) / 8);
    if (item >= item_end) return;
    bt = item / a.planes;
    bp = item - bt * a.planes;
  } else if constexpr (KIND == BLK_MID) {
    const int b = xcd_tile(blockIdx.x, gridDim.x);
    bt = b / a.planes;
    bp = b - bt * a.planes;
  } else {
    bt = xcd_tile(blockIdx.x, gridDim.x);
    bp = blockIdx.y;
  }
  const int x = (bt * WC + wc) * P + p;
  const bool active = x < a.W;
  const int xl = active ? x : a.W - 1;  // columns past the end load the last one and store nothing
  const long long plane_elems = (long long)a.H * a.W;
  // element l + L m of the column: coff + m * col_step, the per-m step a wave-uniform scalar (no
  // per-element 64-bit products kept live across the transforms)
  const long long coff = blk_lane_offset(xl, a.H, C) + (long long)l * C;
  const long long col_step = (long long)L * C;
  const PassWin pw = pass_window<G>(a);
  float2 *ws = scr + (wave * P + p) * F::SCR;

  auto load = [&](float2 (&v)[E], long long q) {
    const float2 *in = reinterpret_cast<const float2 *>(pw.in) + q * plane_elems;
    if constexpr (PADDED) {
      // an element outside loads the nearest row inside, which its neighbours load anyway
      const long long c0 = blk_lane_offset(xl, a.H, C);
#pragma unroll
      for (int m = 0; m < E; ++m) {
        const int y = l + L * m;
        const float2 t = in[c0 + (long long)min(max(y, a.row0), a.row1 - 1) * C];
        const bool inside = y >= a.row0 && y < a.row1;
        v[m] = make_float2(inside ? t.x : 0.f, inside ? t.y : 0.f);
      }
    } else {
#pragma unroll
      for (int m = 0; m < E; ++m) v[m] = in[coff + m * col_step];
    }
  };
  // the first plane's column loads while the twiddles are staged (as in the row pass; the moment
  // kinds of long columns have no registers to spare for it)
  float2 v[E];
  const int q0 = is_mom(KIND) ? (sub < a.planes ? sub : a.planes - 1) : bp;
  constexpr bool EARLY = !is_mom(KIND) || N < 256;
  if constexpr (EARLY && N < 2048) load(v, q0);
  F::stage_twiddles(twl, a.tw, tid, 64 * WC * S);
  __syncthreads();
  if constexpr (EARLY && N >= 2048) load(v, q0);

  if constexpr (LOOP) {
    static_assert(KIND == BLK_MID && P == 1 && !PADDED && !G, "full columns, one per wave");
    const int nloc = gridDim.x / 8;
    const float2 *in = reinterpret_cast<const float2 *>(pw.in);
    float2 *out = reinterpret_cast<float2 *>(pw.out);
    const long long lane_off = (long long)l * C;
    // column bt * WC + wc of plane bp; C divides the tile's columns
    long long co = coff, po = (long long)bp * plane_elems;
    for (;;) {
      F::template stage_in<false>(v, ws, l);
      float2 tf[E];
#pragma unroll
      for (int m = 0; m < E; ++m) tf[m] = pw.mid_tf[co + m * col_step];
      F::template stage_out<false>(v, ws, twl, l);
#pragma unroll
      for (int m = 0; m < E; ++m) asm volatile("" : "+v"(tf[m].x), "+v"(tf[m].y));
#pragma unroll
      for (int m = 0; m < E; ++m) v[m] = cmul(v[m], tf[m]);
      F::template stage_in<true>(v, ws, l);
      // the next item's column loads behind this one's inverse transform and its stores; the last
      // one loads its own column again, unused
      __syncthreads();  // the block's waves load in step
      const bool more = item + nloc < item_end;
      item += more ? nloc : 0;
      const int nt = item / a.planes, np = item - nt * a.planes;
      const int nx = min(nt * WC + wc, a.W - 1);
      const long long nco = blk_lane_offset(nx, a.H, C) + lane_off, npo = (long long)np * plane_elems;
#pragma unroll
      for (int m = 0; m < E; ++m) v[m] = in[npo + nco + m * col_step];
      float2 o[E];
      F::template stage_out<true>(o, ws, twl, l);
#pragma unroll
      for (int m = 0; m < E; ++m) out[po + co + m * col_step] = o[m];
      if (!more) break;
      co = nco;
      po = npo;
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the unused last load lands first
  } else if constexpr (is_mom(KIND)) {
    constexpr bool BAND = KIND == BLK_TO_MOM5;
    Moments<E, BAND> acc;
    acc.zero();
    int q = sub;
    auto run_planes = [&](int end, auto hi) {
      for (; q < end; q += S) {
        const float f = a.mom.f[q], f2 = a.mom.f2[q];
        if constexpr (!EARLY) load(v, q);
        F::template run<false>(v, ws, twl, l);
        acc.template add<decltype(hi)::value>(v, f, f2, a.mom.power2);
        if (EARLY && q + S < a.planes) load(v, q + S);
      }
    };
    if constexpr (BAND) {
      run_planes(a.mom.split, std::false_type{});
      run_planes(a.planes, std::true_type{});
    } else {
      run_planes(a.planes, std::false_type{});
    }
    constexpr int IT = (E + S - 1) / S, NACC = Moments<E, BAND>::NACC;
    float val[NACC][IT];
    // One column per wave: the fold hands four neighbouring columns of a row to four neighbouring
    // lanes.  A store then touches 16 cache lines instead of 64, which had bound the pass as much
    // as its transforms (15 planes of 1024^2: 43.5 -> 32.5 us; 10 of 2048 x 1024: 90 -> 71 us).
    // Column c's lanes are rotated by 16 c so that the reads hit all banks.
    constexpr bool TR = P == 1;
    static_assert(!TR || WC == 4, "the fold pairs four columns");
    int ln;  // opaque: keeps the fold's addresses out of registers during the transforms
    asm volatile("v_mov_b32 %0, %1" : "=v"(ln) : "v"(threadIdx.x & 63));
    const int rt = wc * 64 + ln, rc = rt % 4, rl = rt / 4;
    const int t = wc * 64 + (TR ? (ln + 16 * wc) % 64 : ln);
    fold_subsets<E, S, NACC, TR>(acc.s, reinterpret_cast<float *>(scr), sub, t, TR ? rc * 64 + (rl + 16 * rc) % 64 : t,
                                 64 * WC, val);
    const int sx = TR ? bt * 4 + rc : x, sl = TR ? rl : l;
    if (sx < a.W) {
#pragma unroll
      for (int it = 0; it < IT; ++it) {
        const int m = sub + it * S;
        if (m < E) store_moment<NACC, IT>(a, pw, sl + L * m, sx, val, it);
      }
    }
  } else {
    if constexpr (KIND == BLK_MID) {
      // the table tile loads once pass 1 has moved the column into the scratch, so its latency
      // overlaps the remaining passes (held together by the empty asm: the compiler else sinks
      // each load to its product)
      F::template stage_in<false>(v, ws, l);
      float2 tf[E];
#pragma unroll
      for (int m = 0; m < E; ++m) tf[m] = pw.mid_tf[coff + m * col_step];
      F::template stage_out<false>(v, ws, twl, l);
#pragma unroll
      for (int m = 0; m < E; ++m) asm volatile("" : "+v"(tf[m].x), "+v"(tf[m].y));
#pragma unroll
      for (int m = 0; m < E; ++m) v[m] = cmul(v[m], tf[m]);
      F::template run<true>(v, ws, twl, l);
      if (!active) return;
      float2 *dst = reinterpret_cast<float2 *>(pw.out) + q0 * plane_elems;
#pragma unroll
      for (int m = 0; m < E; ++m) dst[coff + m * col_step] = v[m];
    } else {
      F::template run<false>(v, ws, twl, l);
      const bool mag = a.out_mode == OUT_NAT_MAG;
      if (!mag && a.post_lx) {
        const float2 lx = a.post_lx[xl];
#pragma unroll
        for (int m = 0; m < E; ++m) v[m] = cmul(v[m], cmul(lx, a.post_ly[l + L * m]));
      }
      if constexpr (P == 1) {
        // a wave's column lies one element per row in the natural layout: the block's eight columns
        // go through the scratch, so that eight lanes store eight neighbours of one row (64
        // single elements per store touched 64 cache lines: 15 planes of 1024^2, |X|, 95 us; 48
        // here).  Row y of column c sits rotated by R c within the column's region: the regions are
        // a multiple of all banks apart.
        constexpr int CB = WC, R = 64 / CB;
        auto rot = [](int y, int c, int r) { return y + r * c < N ? y + r * c : y + r * c - N; };
        const int tx0 = bt * CB;
        __builtin_amdgcn_wave_barrier();
        if (mag) {
          float *reg = reinterpret_cast<float *>(ws);
#pragma unroll
          for (int m = 0; m < E; ++m) reg[rot(l + L * m, wc, R)] = sqrtf(v[m].x * v[m].x + v[m].y * v[m].y);
        } else {
#pragma unroll
          for (int m = 0; m < E; ++m) ws[rot(l + L * m, wc, R / 2)] = v[m];
        }
        __syncthreads();
        const int c = tid % CB, y0 = tid / CB;
        if (tx0 + c >= a.W) return;
        const long long o = q0 * plane_elems + (long long)y0 * a.W + tx0 + c, ostep = (long long)(64 * WC / CB) * a.W;
        if (mag) {
          float *dst = reinterpret_cast<float *>(pw.out) + o;
          const float *reg = reinterpret_cast<const float *>(scr + c * F::SCR);
#pragma unroll
          for (int m = 0; m < E; ++m) dst[m * ostep] = reg[rot(y0 + 64 * m, c, R)];
        } else {
          float2 *dst = reinterpret_cast<float2 *>(pw.out) + o;
          const float2 *reg = scr + c * F::SCR;
#pragma unroll
          for (int m = 0; m < E; ++m) dst[m * ostep] = reg[rot(y0 + 64 * m, c, R / 2)];
        }
      } else {
        if (!active) return;
        const long long o = q0 * plane_elems + (long long)l * a.W + x, ostep = (long long)L * a.W;
        if (mag) {
          float *dst = reinterpret_cast<float *>(pw.out) + o;
#pragma unroll
          for (int m = 0; m < E; ++m) dst[m * ostep] = sqrtf(v[m].x * v[m].x + v[m].y * v[m].y);
        } else {
          float2 *dst = reinterpret_cast<float2 *>(pw.out) + o;
#pragma unroll
          for (int m = 0; m < E; ++m) dst[m * ostep] = v[m];
        }
      }
    }
  }
}

// ------------------------------------------------------------------------- launch
bool wave_pass_supported(int n) { return n == 256 || n == 512 || n == 768 || n == 1024 || n == 2048; }

bool row_pass_supported(int W) {
#define X(n) if (W == n) return true;
  HFX_FFT_SIZES(X)
#undef X
  return false;
}

int pick_blk_c(int W, int) {
  for (int c = 4; c > 1; c /= 2)
    if (W % c == 0) return c;
  return 1;
}

bool col_pass_supported(int H, int blk_c) { return row_pass_supported(H) && blk_c >= 1 && blk_c <= 4; }

template <int N, int KIND> static int launch_wrow_n(const PassArgs &a, hipStream_t st) {
  if ((a.inv != 0) != row_inv(KIND)) return -5;
  constexpr bool CAN_SPLIT = is_mom(KIND) && N >= 256;
  const int h = KIND == NAT_TO_BLK ? a.in_h : a.H;
  const unsigned nz = (unsigned)(a.nwin > 1 ? a.nwin : 1);
  const bool split = CAN_SPLIT && wrow_splits((long long)a.H * nz, a.planes, N, KIND == BLK_TO_MOM5);
  const int rows = (split ? wrow_waves(N, KIND, CAN_SPLIT) : wrow_waves(N, KIND, false)) * WaveFft<N>::P;
  const dim3 grid((unsigned)((h + rows - 1) / rows), is_mom(KIND) ? 1u : (unsigned)a.planes, nz);
  const dim3 block(split ? wrow_threads(N, KIND, CAN_SPLIT) : wrow_threads(N, KIND, false));
  constexpr bool CAN_GROUP = is_mom(KIND) && N >= 256;  // (wave_pass_supported)
  if (a.grouped && !CAN_GROUP) return -4;
  if constexpr (is_mom(KIND)) {
    if (a.grouped && split)
      hipLaunchKernelGGL((k_wrow<N, KIND, CAN_GROUP, 0, CAN_SPLIT>), grid, block, 0, st, a);
    else if (a.grouped)
      hipLaunchKernelGGL((k_wrow<N, KIND, CAN_GROUP>), grid, block, 0, st, a);
    else if (split)
      hipLaunchKernelGGL((k_wrow<N, KIND, false, 0, CAN_SPLIT>), grid, block, 0, st, a);
    else
      hipLaunchKernelGGL((k_wrow<N, KIND>), grid, block, 0, st, a);
  } else if constexpr (KIND == NAT_TO_BLK) {
    const bool cplx = a.in_mode == IN_NAT_C, full = a.in_h == a.H && a.in_w == a.W && a.off_x == 0 && a.off_y == 0;
    if (cplx && full && a.pre_lx == nullptr)
      hipLaunchKernelGGL((k_wrow<N, KIND, false, 1>), grid, block, 0, st, a);
    else if (cplx && full)
      hipLaunchKernelGGL((k_wrow<N, KIND, false, 2>), grid, block, 0, st, a);
    else if (cplx && a.pre_lx == nullptr)
      hipLaunchKernelGGL((k_wrow<N, KIND, false, 3>), grid, block, 0, st, a);
    else
      hipLaunchKernelGGL((k_wrow<N, KIND>), grid, block, 0, st, a);
  } else {
    hipLaunchKernelGGL((k_wrow<N, KIND>), grid, block, 0, st, a);
  }
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

template <int N, int KIND> static int launch_wcol_n(const PassArgs &a, hipStream_t st) {
  if (a.inv != 0) return -5;
  constexpr int cols = wcol_waves(N, KIND) * WaveFft<N>::P;
  const unsigned tiles = (unsigned)((a.W + cols - 1) / cols);
  // BLK_MID: one flat dimension, plane-fastest (see k_wcol); the plane-parallel others: y = plane
  const dim3 grid(KIND == BLK_MID ? tiles * (unsigned)a.planes : tiles,
                  is_mom(KIND) || KIND == BLK_MID ? 1u : (unsigned)a.planes, (unsigned)(a.nwin > 1 ? a.nwin : 1));
  const dim3 block(wcol_threads(N, KIND));
  constexpr bool CAN_LOOP = KIND == BLK_MID && N >= 2048, CAN_NARROW = KIND == BLK_MID && N == 1024;
  // LOOP from five items per block on.  One item per block -> LOOP: 512 wide with 8, 16 (four per block),
  // 20, 52 planes 49.2 -> 51.5, 98.8 -> 101, 110.2 -> 108.7, 288 -> 272 us; 2048 wide with 4 (four), 5, 12,
  // 52 97.5 -> 98.4, 115.4 -> 113.9, 276 -> 246, 1174 -> 1045.  A multiple of eight blocks: the items are
  // split over the XCDs.
  const unsigned cus = CAN_LOOP || CAN_NARROW ? (unsigned)device_cus() : 0, loop_blocks = std::max(8u, cus & ~7u);
  const bool padded = a.row1 > a.row0 && (a.row0 > 0 || a.row1 < a.H);
  constexpr bool CAN_GROUP = KIND != BLK_TO_NAT && N >= 256;  // (wave_pass_supported)
  if ((padded && KIND != BLK_MID) || (a.grouped && !CAN_GROUP)) return -4;
  if (a.grouped)
    hipLaunchKernelGGL((k_wcol<N, KIND, CAN_GROUP>), grid, block, 0, st, a);
  else if (padded)
    hipLaunchKernelGGL((k_wcol<N, KIND, false, KIND == BLK_MID>), grid, block, 0, st, a);
  else if (CAN_LOOP && a.W % cols == 0 && a.nwin <= 1 && grid.x >= 5 * loop_blocks)
    hipLaunchKernelGGL((k_wcol<N, KIND, false, false, CAN_LOOP>), dim3(loop_blocks), block, 0, st, a);
  else if (CAN_NARROW && wcol_narrow((long long)((a.W + 3) / 4) * a.planes, (int)cus))
    hipLaunchKernelGGL((k_wcol<N, KIND, false, false, false, CAN_NARROW>), dim3((unsigned)((a.W + 3) / 4) * (unsigned)a.planes),
                       dim3(wcol_threads(N, KIND, CAN_NARROW)), 0, st, a);
  else
    hipLaunchKernelGGL((k_wcol<N, KIND>), grid, block, 0, st, a);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

template <int KIND> static int wrow_dispatch(const PassArgs &a, hipStream_t st) {
#define X(s) if (a.W == s) return launch_wrow_n<s, KIND>(a, st);
  HFX_FFT_SIZES(X)
#undef X
  return -2;
}

template <int KIND> static int wcol_dispatch(const PassArgs &a, hipStream_t st) {
#define X(s) if (a.H == s) return launch_wcol_n<s, KIND>(a, st);
  HFX_FFT_SIZES(X)
#undef X
  return -2;
}

int launch_row_pass(const PassArgs &a, hipStream_t st) {
  if (a.in_mode != IN_BLK) {
    if (a.out_mode != OUT_BLK) return -4;
    return wrow_dispatch<NAT_TO_BLK>(a, st);
  }
  if (a.out_mode == OUT_MOMENTS)
    return a.mom.split > 0 ? wrow_dispatch<BLK_TO_MOM5>(a, st) : wrow_dispatch<BLK_TO_MOM>(a, st);
  if (a.out_mode == OUT_BLK && a.pre_lx) return wrow_dispatch<BLK_LENS>(a, st);
  if ((a.out_mode == OUT_NAT_C && !a.post_lx) || a.out_mode == OUT_NAT_RE) return wrow_dispatch<BLK_TO_NAT>(a, st);
  return -4;
}

int launch_col_pass(const PassArgs &a, hipStream_t st) {
  if (a.in_mode != IN_BLK || a.W % a.blk_c != 0 || !col_pass_supported(a.H, a.blk_c)) return -3;
  if (a.mid_tf) {
    if (a.out_mode != OUT_BLK) return -4;
    return wcol_dispatch<BLK_MID>(a, st);
  }
  if (a.out_mode == OUT_MOMENTS)
    return a.mom.split > 0 ? wcol_dispatch<BLK_TO_MOM5>(a, st) : wcol_dispatch<BLK_TO_MOM>(a, st);
  if (a.out_mode == OUT_NAT_C || a.out_mode == OUT_NAT_MAG) return wcol_dispatch<BLK_TO_NAT>(a, st);
  return -4;
}

}  // namespace hfx
