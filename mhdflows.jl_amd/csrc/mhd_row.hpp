// The fused x-row kernel of a right-hand side: complex rows -> real rows -> products -> complex rows.
//
// Real rows are transformed two at a time as one complex row of the full length NX: the real rows
// A, B with half spectra X, Y have the complex row A + iB with spectrum
//   Z_k = X_k + i Y_k,  Z_{NX-k} = conj(X_k) + i conj(Y_k)      (0 <= k <= NX/2)
// and back, X_k = (Z_k + conj Z_{NX-k}) / 2, Y_k = (Z_k - conj Z_{NX-k}) / 2i.  Against packing
// the even and odd samples of one row into a half-length complex row, nothing is multiplied on
// the way in or out (the half-length form costs 10 operations a value each way), the input needs
// no exchange (Z_{NX-k} is formed from the same loaded values, read a second time in mirrored
// order through the cache), and only the kept entries of the output are unpacked.
//
// A and B are the same field (or product) of two neighbouring rows, never two fields: the rounding
// of a transform is relative to the larger of the two, and fields may differ by orders of
// magnitude (a seed magnetic field in a dynamo run).
//
// A transform of NX points belongs to TX = NX/E threads; thread t holds the positions t + j*TX
// before the first and after the last pass, whatever the radices, so the products feed the
// forward transforms from registers.  Twiddles are loaded once per work item and kept in
// registers for all its transforms.
//
// Exchanges: LDS serves 128 B a cycle from 32 banks, i.e. G = 16 (Float32) or 8 (Float64) lanes of
// a wave at a time, and slot s of a transform is in group s mod G.  Reads take consecutive
// positions.  Writes of the pass with stride Ns and radix R take Ns consecutive positions out of
// every Ns*R; C padding slots per G positions shift them apart (exch_pad).  Every exchange has
// the C that its own write needs: none for Ns >= G.  Counted over all plans this leaves 1.0
// cycles an access (1.5 in a few exchanges of the smallest lengths); one padding for all
// exchanges of a plan had 28 % of the kernel's cycles in bank conflicts (256 points).  Indexes are
// written as base + constant, which pad() keeps apart as their bits are disjoint (powers of two).
#pragma once
#include "mhd_kernels.hpp"

namespace mhd {

// Row plans, by length and plan number: E values a thread and the radices, powers of two first.
template <class T, int N, int P> struct RowPlan2;
#define MHD_ROWPLAN2_B(N_, P_, E_, ...)              \
  template <class T> struct RowPlan2<T, N_, P_> {    \
    static constexpr int E = E_;                     \
    using R = Radices<__VA_ARGS__>;                  \
  };
// plan 0: eight values a thread (twelve for lengths with a factor 3)
MHD_ROWPLAN2_B(8, 0, 8, 8)
MHD_ROWPLAN2_B(16, 0, 8, 8, 2)
MHD_ROWPLAN2_B(24, 0, 12, 2, 12)
MHD_ROWPLAN2_B(32, 0, 8, 8, 4)
MHD_ROWPLAN2_B(48, 0, 12, 4, 12)
MHD_ROWPLAN2_B(64, 0, 8, 8, 8)
MHD_ROWPLAN2_B(96, 0, 12, 4, 2, 12)
MHD_ROWPLAN2_B(128, 0, 8, 8, 8, 2)
MHD_ROWPLAN2_B(192, 0, 12, 4, 4, 12)
MHD_ROWPLAN2_B(256, 0, 8, 8, 8, 4)
MHD_ROWPLAN2_B(384, 0, 12, 4, 4, 2, 12)
MHD_ROWPLAN2_B(512, 0, 8, 8, 8, 8)
MHD_ROWPLAN2_B(768, 0, 12, 4, 4, 4, 12)
MHD_ROWPLAN2_B(1024, 0, 8, 8, 8, 8, 2)
// plan 1: four values a thread (six)
MHD_ROWPLAN2_B(8, 1, 4, 4, 2)
MHD_ROWPLAN2_B(16, 1, 4, 4, 4)
MHD_ROWPLAN2_B(24, 1, 6, 2, 2, 6)
MHD_ROWPLAN2_B(32, 1, 4, 4, 4, 2)
MHD_ROWPLAN2_B(48, 1, 6, 2, 2, 2, 6)
MHD_ROWPLAN2_B(64, 1, 4, 4, 4, 4)
MHD_ROWPLAN2_B(96, 1, 6, 2, 2, 2, 2, 6)
MHD_ROWPLAN2_B(128, 1, 4, 4, 4, 4, 2)
MHD_ROWPLAN2_B(192, 1, 6, 2, 2, 2, 2, 2, 6)
MHD_ROWPLAN2_B(256, 1, 4, 4, 4, 4, 4)
MHD_ROWPLAN2_B(384, 1, 6, 2, 2, 2, 2, 2, 2, 6)
MHD_ROWPLAN2_B(512, 1, 4, 4, 4, 4, 4, 2)
MHD_ROWPLAN2_B(768, 1, 6, 2, 2, 2, 2, 2, 2, 2, 6)
MHD_ROWPLAN2_B(1024, 1, 16, 16, 16, 4)
// The plan a row launch uses unless its variant asks for the other one.  Six fields (MHD) of four
// values a thread fit 118 VGPRs (Float32: four waves a SIMD), of eight 221 (two); up to 512 points
// the waves are worth more than the shorter sequence of passes (us a launch, plan 0 / plan 1:
// Float32 64^3 17.3 / 14.0, 256^3 197 / 174, 512x256x128 201 / 194; Float64 256^3 414 / 341), for
// longer rows the passes are (768x256x128 463 / 500, 1024x256x128 460 / 739).  Three fields (HD)
// leave both plans their waves: four values only where launches are too small to fill the chip
// (64^3 11.8 / 10.1, 192^3 47.5 / 55.2, 512x256x128 84 / 100).
inline int rowpair_plan(int nx, int phys) { return nx <= (phys == PHYS_MHD ? 512 : 96) ? 1 : 0; }
// values a thread holds, for host-side launch shapes
inline int rowpair_E(int nx, int plan) {
  if (nx % 3 == 0) return plan ? 6 : 12;
  if (nx == 1024) return plan ? 16 : 8;
  return plan ? 4 : 8;
}
#undef MHD_ROWPLAN2_B

template <class T> constexpr int lds_group() { return 128 / (int)sizeof(cx<T>); }
template <class T> constexpr int exch_pad(int Ns, int R) {
  const int G = lds_group<T>();
  const int c = Ns >= G ? 0 : (Ns * R >= G ? (Ns == 1 ? 1 : G / R) : Ns);
  return c > 4 ? 0 : c;
}
template <class T, int C> __host__ __device__ constexpr int pad(int pos) { return pos + C * (pos / lds_group<T>()); }

// Launch shape: 128 threads, LPW transforms at a time, each of two rows.
template <class T, int NX, int PLAN> struct RowPairShape {
  using P = RowPlan2<T, NX, PLAN>;
  static constexpr int E = P::E;
  static constexpr int TX = NX / E;
  static constexpr int LPW = 128 / TX;
  static constexpr int RPW = 2 * LPW;                        // rows of a work item
  static constexpr int SLOTS = pad<T, 4>(NX) + 2;            // + 2: transforms of one wave on other banks
  static constexpr int LDS_CX = LPW * SLOTS;
  static_assert(128 % TX == 0, "a workgroup holds whole transforms");
};

// Fields requested ahead of the transforms: all of them where they fit the registers
template <class T, int NIN, int E> struct RowAhead {
  static constexpr int fit = (sizeof(T) == 4 ? 24 : 12) / E > 1 ? (sizeof(T) == 4 ? 24 : 12) / E : 1;
  static constexpr int value = fit < NIN ? fit : NIN;
};

// The advective products of one point, u = v[0..2], b = v[3..5], in the order of NADV_MHD / NADV_HD:
// T_ij = b_i b_j - u_i u_j and M_aj = u_a b_j - b_a u_j, or U_ij = u_i u_j, the diagonal entries
// less the 22 entry.
template <class T, int KIND>
__device__ __forceinline__ T advective(int p, const T* v) {
  if constexpr (KIND == ROW_MHD) {
    switch (p) {
      case 0: return (v[3] * v[3] - v[0] * v[0]) - (v[5] * v[5] - v[2] * v[2]);
      case 1: return v[3] * v[4] - v[0] * v[1];
      case 2: return v[3] * v[5] - v[0] * v[2];
      case 3: return v[0] * v[4] - v[3] * v[1];
      case 4: return v[0] * v[5] - v[3] * v[2];
      case 5: return v[1] * v[5] - v[4] * v[2];
      case 6: return (v[4] * v[4] - v[1] * v[1]) - (v[5] * v[5] - v[2] * v[2]);
      default: return v[4] * v[5] - v[1] * v[2];
    }
  } else {
    switch (p) {
      case 0: return v[0] * v[0] - v[2] * v[2];
      case 1: return v[0] * v[1];
      case 2: return v[0] * v[2];
      case 3: return v[1] * v[1] - v[2] * v[2];
      default: return v[1] * v[2];
    }
  }
}

// Twiddles of every pass but the first, in registers
template <class T, int N, int E, int Ns, class Rad> struct RowTw;
template <class T, int N, int E, int Ns> struct RowTw<T, N, E, Ns, Radices<>> {
  __device__ __forceinline__ void load(int, const cx<T>*) {}
};
template <class T, int N, int E, int Ns, int R, int... Rest> struct RowTw<T, N, E, Ns, Radices<R, Rest...>> {
  static constexpr int TX = N / E, NB = E / R;
  // butterflies t + i*TX whose index modulo Ns is the same share their twiddles
  static constexpr int NT = Ns == 1 ? 0 : (TX % Ns == 0 ? 1 : NB);
  cx<T> w[NT > 0 ? NT : 1][R > 1 ? R - 1 : 1];
  RowTw<T, N, E, Ns * R, Radices<Rest...>> next;
  __device__ __forceinline__ void load(int t, const cx<T>* tab) {
    if constexpr (Ns > 1) {
#pragma unroll
      for (int i = 0; i < NT; ++i) {
        const int m1 = ((t + i * TX) % Ns) * (N / (Ns * R));
#pragma unroll
        for (int r = 1; r < R; ++r) w[i][r - 1] = tab[r * m1];
      }
    }
    next.load(t, tab);
  }
};

// One transform of direction S on x[j] = the value at position t + j*TX, in place.  row: the
// transform's LDS slots.  A sync precedes every exchange write.
template <class T, int N, int E, int S, bool WS, int Ns, class Rad> struct RowPass;
template <class T, int N, int E, int S, bool WS, int Ns> struct RowPass<T, N, E, S, WS, Ns, Radices<>> {
  template <class Tw> static __device__ __forceinline__ void run(cx<T>*, int, cx<T>*, const Tw&) {}
};
template <class T, int N, int E, int S, bool WS, int Ns, int R, int... Rest>
struct RowPass<T, N, E, S, WS, Ns, Radices<R, Rest...>> {
  template <class Tw>
  static __device__ __forceinline__ void run(cx<T>* x, int t, cx<T>* row, const Tw& tw) {
    constexpr int TX = N / E, NB = E / R;
    static_assert(E % R == 0, "radix must divide the values a thread holds");
    constexpr bool LAST = sizeof...(Rest) == 0;
    constexpr int C = exch_pad<T>(Ns, R);
    if constexpr (!LAST) xsync<WS>();
#pragma unroll
    for (int i = 0; i < NB; ++i) {
      cx<T> v[R];
#pragma unroll
      for (int r = 0; r < R; ++r) {
        v[r] = x[i + r * NB];
        if constexpr (Ns > 1)
          if (r > 0) v[r] = twmul<S>(v[r], tw.w[Tw::NT == 1 ? 0 : i][r > 0 ? r - 1 : 0]);
      }
      Bfly<T, R, S>::run(v);
      if constexpr (LAST) {
        // position b + r*Ns of butterfly b = t + i*TX, where Ns = N/R = NB*TX
#pragma unroll
        for (int r = 0; r < R; ++r) x[i + r * NB] = v[r];
      } else {
        static_assert((Ns & (Ns - 1)) == 0 && (R & (R - 1)) == 0, "padded indexes add up for powers of two");
        const int b = t + i * TX;
        cx<T>* const d = row + pad<T, C>((b / Ns) * Ns * R + b % Ns);
#pragma unroll
        for (int r = 0; r < R; ++r) d[pad<T, C>(r * Ns)] = v[r];
      }
    }
    if constexpr (!LAST) {
      xsync<WS>();
      if constexpr (TX % lds_group<T>() == 0) {
        const cx<T>* const s = row + pad<T, C>(t);
#pragma unroll
        for (int j = 0; j < E; ++j) x[j] = s[pad<T, C>(j * TX)];
      } else {
#pragma unroll
        for (int j = 0; j < E; ++j) x[j] = row[pad<T, C>(t + j * TX)];
      }
      RowPass<T, N, E, S, WS, Ns * R, Radices<Rest...>>::run(x, t, row, tw.next);
    }
  }
};

// One work item (RPW rows of one run), run by a 128-thread workgroup.  xbuf holds
// RowPairShape::LDS_CX exchange slots, red 2*128 values and stw NX twiddles.  Every early return
// is taken by the whole workgroup.
template <class T, int NX, int KIND, int PLAN>
__device__ __forceinline__ void rowpair_item(const RowArgs& a, int64_t item, const RunBuf<T>* __restrict__ runs,
                                             const cx<T>* __restrict__ twx, cx<T>* xbuf, T* red, cx<T>* stw) {
  static_assert(KIND == ROW_MHD || KIND == ROW_HD, "the fused kinds");
  using SHP = RowPairShape<T, NX, PLAN>;
  using P = typename SHP::P;
  using Rad = typename P::R;
  constexpr int E = SHP::E, TX = SHP::TX, H = E / 2;
  constexpr int NIN = KIND == ROW_MHD ? 6 : 3, NPROD = KIND == ROW_MHD ? NADV_MHD : NADV_HD;
  constexpr bool WS = TX <= 64;

  const int t = threadIdx.x;
  const int rw = t / TX, tr = t % TX;
  const Geom& G = a.g;
  const int run = (int)(item / a.blocks_per_run);
  const int64_t blk = a.blk0 + item % a.blocks_per_run;
  // Rows row0 (even) and row0 + 1, in one z-plane as ny is even.  Rows past the end load the
  // item's first rows and store nothing.
  const int64_t first = blk * SHP::RPW, row0 = first + 2 * rw;
  const bool ok = row0 < a.rows;
  const RunBuf<T>& rb = runs[run];
  if (gated_off(a.gate, rb)) return;
  const bool pruned = a.prune_out && step_pruned(rb);
  for (int i = t; i < NX; i += 128) stw[i] = twx[i];
  __syncthreads();
  cx<T>* const xrow = xbuf + rw * SHP::SLOTS;

  // The entries of the two half spectra of field f that position tr + j*TX takes: entry p for
  // p < NX/2, the mirrored entry NX - p for p >= NX/2 (j >= E/2).  AHEAD fields are requested
  // before the first transform starts, so the loads' latencies overlap.  Addresses are a uniform
  // base (the item's first row of a field) plus a 32-bit offset and a constant.
  constexpr int AHEAD = RowAhead<T, NIN, E>::value;
  const int ncols = a.in_ncols;
  cx<T> ra[NIN][E], rc[NIN][E];
  const int64_t ifs = field_stride(G, a.in_sel), irs = row_stride(G, a.in_sel);
  const int64_t ifirst = row_offset(G, a.in_sel, first);
  const gptr<const cx<T>> src = gmem<const cx<T>>(rb.buf[a.in_sel]) + (int64_t)a.in_f0 * ifs + ifirst;
  const uint32_t ioff = ok ? (uint32_t)(row_offset(G, a.in_sel, row0) - ifirst) : 0u;
  const uint32_t iup = ioff + tr, idn = ioff + (NX / 2 - tr);  // entries tr, NX/2 - tr of row0
  auto request = [&](int f0, int f1) {
#pragma unroll
    for (int f = f0; f < f1; ++f)
#pragma unroll
      for (int j = 0; j < E; ++j) ra[f][j] = rc[f][j] = cx<T>{T(0), T(0)};
#pragma unroll
    for (int j = 0; j < E; ++j) {
      const int k = j < H ? tr + j * TX : (NX / 2 - tr) - (j - H) * TX;
      if (k < ncols) {
#pragma unroll
        for (int f = f0; f < f1; ++f) {
          const gptr<const cx<T>> pa = src + (int64_t)f * ifs, pc = pa + irs;
          const uint32_t o = j < H ? iup + j * TX : idn - (j - H) * TX;
          ra[f][j] = ldst<false, T>(pa + o);
          rc[f][j] = ldst<false, T>(pc + o);
        }
      }
    }
  };
  request(0, AHEAD);
  RowTw<T, NX, E, 1, Rad> tw;
  tw.load(tr, stw);

  // z[f][j].re, .im: field f at x = tr + j*TX of the two rows
  cx<T> z[NIN][E];
  const T scale = T(G.inv_n);
#pragma unroll
  for (int f = 0; f < NIN; ++f) {
    if (f + AHEAD < NIN) request(f + AHEAD, f + AHEAD + 1);
#pragma unroll
    for (int j = 0; j < E; ++j) {
      cx<T> A = ra[f][j], B = rc[f][j];
      if ((j == 0 || j == H) && tr == 0) A.im = B.im = T(0);  // c2r ignores Im of the DC and Nyquist entries
      z[f][j] = j < H ? cx<T>{A.re - B.im, A.im + B.re} : cx<T>{A.re + B.im, B.re - A.im};
    }
    RowPass<T, NX, E, 1, WS, 1, Rad>::run(z[f], tr, xrow, tw);
#pragma unroll
    for (int j = 0; j < E; ++j) z[f][j] = z[f][j] * scale;
  }

  // A dealiased step's real fields would be overwritten by a later step of the same call before
  // anything reads them, so only the call's last step, which is full, stores them.
  if (a.write_vars && !pruned && ok) {
    const gptr<T> rbase = gmem(rb.vars) + (int64_t)a.real_out_f0 * G.nr + first * NX;
    const uint32_t o = (uint32_t)(2 * rw * NX + tr);
#pragma unroll
    for (int f = 0; f < NIN; ++f) {
      const gptr<T> va = rbase + (int64_t)f * G.nr;
#pragma unroll
      for (int j = 0; j < E; ++j) {
        va[o + j * TX] = z[f][j].re;
        va[o + NX + j * TX] = z[f][j].im;
      }
    }
  }
  if (a.want_max) {  // rows past the end repeat others
    T mu = T(0), mb = T(0);
#pragma unroll
    for (int f = 0; f < NIN; ++f)
#pragma unroll
      for (int j = 0; j < E; ++j) {
        // the largest square is the square of the largest magnitude (rounding is monotonic)
        const T s1 = fabs(z[f][j].re), s2 = fabs(z[f][j].im);
        if (f < 3) mu = nanmax(nanmax(mu, s1), s2);
        else mb = nanmax(nanmax(mb, s1), s2);
      }
    mu = mu * mu;
    mb = mb * mb;
    T* const red1 = red + 128;
    red[t] = mu;
    red1[t] = mb;
    __syncthreads();
    for (int s = 64; s > 0; s >>= 1) {
      if (t < s) {
        red[t] = nanmax(red[t], red[t + s]);
        red1[t] = nanmax(red1[t], red1[t + s]);
      }
      __syncthreads();
    }
    if (t == 0) {
      const gptr<T> part = gmem(rb.partial);
      part[2 * blk] = red[0];
      part[2 * blk + 1] = red1[0];
    }
  }

  // entries [0, kend) of every product row are stored: the kept ones of a dealiased step or all,
  // rounded up to whole lines in the work buffer (entries past NX/2 are zeros)
  const bool dst_work = a.out_sel == B_WORK;
  const int kfull = dst_work ? G.wrs : NX / 2 + 1;
  const int kend = !ok ? 0 : (pruned ? (dst_work ? G.kx_keep_w : G.kx_keep) : kfull);
  const int64_t ofs = field_stride(G, a.out_sel), ors = row_stride(G, a.out_sel);
  const int64_t ofirst = row_offset(G, a.out_sel, first);
  const gptr<cx<T>> out = gmem(rb.buf[a.out_sel]) + (int64_t)a.out_f0 * ofs + ofirst;
  const uint32_t oup = (ok ? (uint32_t)(row_offset(G, a.out_sel, row0) - ofirst) : 0u) + tr;
#pragma unroll
  for (int i = 0; i < NPROD; ++i) {
    // the two diagonal products, which share their 22 entry, one after the other
    constexpr int ORDER[2][8] = {{0, 3, 1, 2, 4, 0, 0, 0}, {0, 6, 1, 2, 7, 3, 4, 5}};
    const int p = ORDER[KIND == ROW_MHD][i];
    cx<T> w[E];
#pragma unroll
    for (int j = 0; j < E; ++j) {
      T v[NIN], u[NIN];
#pragma unroll
      for (int f = 0; f < NIN; ++f) { v[f] = z[f][j].re; u[f] = z[f][j].im; }
      w[j] = cx<T>{advective<T, KIND>(p, v), advective<T, KIND>(p, u)};
    }
    RowPass<T, NX, E, -1, WS, 1, Rad>::run(w, tr, xrow, tw);
    // mirror exchange: the value at position q >= NX/2 goes to slot NX - q
    xsync<WS>();
    {
      cx<T>* const d = xrow + (NX / 2 - tr);
#pragma unroll
      for (int j = H; j < E; ++j) d[-(j - H) * TX] = w[j];
    }
    xsync<WS>();
    // twice the product's half spectrum is stored (rhs_at halves it): no factor 1/2 here
    const gptr<cx<T>> da = out + (int64_t)p * ofs, dc = da + ors;
#pragma unroll
    for (int j = 0; j < H; ++j) {
      const int k = tr + j * TX;
      if (k < kend) {
        cx<T> Zm = xrow[k];
        if (j == 0 && tr == 0) Zm = w[0];  // entry 0 is its own mirror
        stst<false, T>(da + (oup + j * TX), cx<T>{w[j].re + Zm.re, w[j].im - Zm.im});
        stst<false, T>(dc + (oup + j * TX), cx<T>{w[j].im + Zm.im, Zm.re - w[j].re});
      }
    }
    if (NX / 2 < kend) {
      // the Nyquist entry is thread 0's value at position NX/2; zeros follow it to the line's end
      const T nr = tr == 0 ? T(2) * w[H].re : T(0), ni = tr == 0 ? T(2) * w[H].im : T(0);
      for (int k = tr; k < kend - NX / 2; k += TX) {
        stst<false, T>(da + (oup + NX / 2 + (k - tr)), cx<T>{k == tr ? nr : T(0), T(0)});
        stst<false, T>(dc + (oup + NX / 2 + (k - tr)), cx<T>{k == tr ? ni : T(0), T(0)});
      }
    }
  }
}

template <class T, int NX, int KIND, int PLAN>
__global__ void __launch_bounds__(128)
rowpair_kernel(RowArgs a, const RunBuf<T>* __restrict__ runs, const cx<T>* __restrict__ twx) {
  using SHP = RowPairShape<T, NX, PLAN>;
  __shared__ cx<T> xb[SHP::LDS_CX];
  __shared__ T red[2 * 128];
  __shared__ cx<T> stw[NX];
  const int64_t item = xcd_item(blockIdx.x, (int64_t)gridDim.x);
  if (item >= a.blocks_per_run * a.nruns) return;
  rowpair_item<T, NX, KIND, PLAN>(a, item, runs, twx, xb, red, stw);
}

}  // namespace mhd
