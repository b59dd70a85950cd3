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
// after the last inverse and before the first forward pass, whatever the radices, so the products
// feed the forward transforms from registers.  Twiddles are loaded once per work item and kept in
// registers for all its transforms.
//
// A pass of radix R has B = N/R butterflies; thread t takes b = t, t + TX, ..., and where B is no
// multiple of TX some threads sit a pass out: lengths 3 * 2^k then need few passes of radix 4 and
// 8 in place of many of radix 2, and hold three or six values a thread instead of six or twelve.
// The last inverse pass is always a full one, so the products are formed in its layout.
//
// Exchanges: LDS serves 128 B a cycle from 32 banks, i.e. G = 16 (Float32) or 8 (Float64) lanes of
// a wave at a time, and slot s of a transform is in group s mod G.  Reads take consecutive
// positions.  Writes of the pass with stride Ns and radix R take Ns consecutive positions out of
// every Ns*R; padding slots shift them apart (Exchange): C per G positions where Ns*R is a power of
// two, c per Ns*R positions otherwise, chosen for each exchange by its own writes.  One padding for
// all exchanges of a plan had 28 % of the kernel's cycles in bank conflicts (256 points).  Slots are
// written as base + constant.
#pragma once
#include "mhd_kernels.hpp"

namespace mhd {

// Row plans, by length and plan number: E values a thread, the inverse radices, and the forward ones
// (the same where they are powers of two, reversed otherwise).
template <class L, bool REV> struct ForwardOrder { using type = L; };
template <class L> struct ForwardOrder<L, true> { using type = typename RReverse<L>::type; };
template <class T, int N, int P> struct RowPlan2;
#define MHD_ROWPLAN2_B(N_, P_, E_, ...)              \
  template <class T> struct RowPlan2<T, N_, P_> {    \
    static constexpr int E = E_;                     \
    using R = Radices<__VA_ARGS__>;                  \
    using F = typename ForwardOrder<R, (N_ % 3 == 0)>::type; \
  };
// plan 0: eight values a thread (three, six or twelve for lengths with a factor 3)
MHD_ROWPLAN2_B(8, 0, 8, 8)
MHD_ROWPLAN2_B(16, 0, 8, 8, 2)
MHD_ROWPLAN2_B(24, 0, 3, 8, 3)
MHD_ROWPLAN2_B(32, 0, 8, 8, 4)
MHD_ROWPLAN2_B(48, 0, 6, 8, 6)
MHD_ROWPLAN2_B(64, 0, 8, 8, 8)
MHD_ROWPLAN2_B(96, 0, 3, 4, 8, 3)
MHD_ROWPLAN2_B(128, 0, 8, 8, 8, 2)
MHD_ROWPLAN2_B(192, 0, 6, 8, 4, 6)
MHD_ROWPLAN2_B(256, 0, 8, 8, 8, 4)
MHD_ROWPLAN2_B(384, 0, 3, 4, 4, 8, 3)
MHD_ROWPLAN2_B(512, 0, 8, 8, 8, 8)
MHD_ROWPLAN2_B(768, 0, 12, 4, 4, 4, 12)
MHD_ROWPLAN2_B(1024, 0, 8, 8, 8, 8, 2)
// plan 1: four values a thread (three or six)
MHD_ROWPLAN2_B(8, 1, 4, 4, 2)
MHD_ROWPLAN2_B(16, 1, 4, 4, 4)
MHD_ROWPLAN2_B(24, 1, 3, 4, 2, 3)
MHD_ROWPLAN2_B(32, 1, 4, 4, 4, 2)
MHD_ROWPLAN2_B(48, 1, 3, 4, 4, 3)
MHD_ROWPLAN2_B(64, 1, 4, 4, 4, 4)
MHD_ROWPLAN2_B(96, 1, 3, 4, 4, 2, 3)
MHD_ROWPLAN2_B(128, 1, 4, 4, 4, 4, 2)
MHD_ROWPLAN2_B(192, 1, 3, 4, 4, 4, 3)
MHD_ROWPLAN2_B(256, 1, 4, 4, 4, 4, 4)
MHD_ROWPLAN2_B(384, 1, 6, 8, 8, 6)
MHD_ROWPLAN2_B(512, 1, 4, 4, 4, 4, 4, 2)
MHD_ROWPLAN2_B(768, 1, 6, 4, 4, 8, 6)
MHD_ROWPLAN2_B(1024, 1, 16, 16, 16, 4)
#undef MHD_ROWPLAN2_B
// The plan a row launch uses unless its variant asks for the other one.  Six fields (MHD) of three
// or four values a thread fit 128 VGPRs (Float32: four waves a SIMD), of eight 211 (two); below 512
// points the waves are worth more than the shorter sequence of passes, at 1024 the passes are, and
// at 768 Float64 plan 1 is compiled with 144 B of scratch a lane.  RK4 steps, ms, plan
// 0 / plan 1: Float32 128x256x128 0.899 / 0.866, 192x256x128 1.214 / 1.166, 256x256x128 1.679 / 1.603,
// 384x256x128 2.607 / 2.526, 512x64x64 0.420 / 0.438, 512^3 26.19 / 26.58, 768x128x128 2.59 / 2.51,
// 768x256x256 10.48 / 10.16, 1024x128x128 3.21 / 3.49; Float64 128x256x128 1.712 / 1.638, 192x256x128
// 2.521 / 2.424, 256x256x128 3.265 / 3.131, 512x256x256 12.65 / 12.46, 768x128x128 4.83 / 8.63,
// 1024x128x128 6.42 / 12.03.  Three fields (HD) leave both plans their waves: fewer values only where
// launches are too small to fill the chip and at 384 points with their three passes (Float32
// 384x256x128 1.440 / 1.387, Float64 2.959 / 2.661); otherwise plan 0 (Float32 192x256x128 0.704 /
// 0.718, 512x128x128 0.854 / 0.905, 768x128x128 1.374 / 1.409; Float64 512x128x128 1.700 / 1.780,
// 768x128x128 2.83 / 4.74).
inline int rowpair_plan(int nx, int phys, bool f64) {
  if (phys == PHYS_MHD) return nx < 512 || nx == (f64 ? 512 : 768) ? 1 : 0;
  return nx <= 96 || nx == 384 ? 1 : 0;
}
// values a thread holds, for host-side launch shapes
inline int rowpair_E(int nx, int plan) {
  switch (nx) {
#define MHD_ROW_E(N_) case N_: return plan ? RowPlan2<float, N_, 1>::E : RowPlan2<float, N_, 0>::E;
    MHD_ROW_E(8) MHD_ROW_E(16) MHD_ROW_E(24) MHD_ROW_E(32) MHD_ROW_E(48) MHD_ROW_E(64) MHD_ROW_E(96)
    MHD_ROW_E(128) MHD_ROW_E(192) MHD_ROW_E(256) MHD_ROW_E(384) MHD_ROW_E(512) MHD_ROW_E(768) MHD_ROW_E(1024)
#undef MHD_ROW_E
  }
  return 8;
}

// Row launches next to the two plans: rowteam_kernel (on plan 1) with a wave per product, or three
// waves in all.  Three divide six fields and nine (HD: six) products without a rest; four and five
// took 22.7 and 24.4 us at 96^3 for 21.7.
constexpr int ROW_TEAM = 2, ROW_TEAM_HALF = 3;
inline bool rowteam_length(int nx) { return nx <= 256; }
// The team that a whole launch over `pairs` row pairs takes, 0 for none.  The waves of a plain
// launch each run 15 (HD: 9) transforms one after the other; with less than about two of them a SIMD
// the launch takes as long as one wave does, and teams shorten that.  us a launch, plain / a wave per
// product / three waves, by the waves of the plain launch: Float32 32^3 (64) 12.0 / 8.0 / 9.0, 48^3
// (288) 12.9 / 9.4 / 10.2, 64^3 (512) 14.1 / 10.7 / 11.2, 128x64x64 (1024) 17.8 / 16.6 / 14.9,
// 256x64x64 (2048) 21.4 / 26.9 / 22.0, 96^3 (2304) 23.1 / 29.7 / 21.7, 192x96x64 (3072) 25.6 / 37.5 /
// 26.5; Float64 32^3 13.8 / 9.0 / 9.9, 48^3 14.8 / 12.8 / 11.6, 64^3 16.6 / 15.2 / 13.8, 96^3 37.1 / 47.6 /
// 31.1, 128x96x64 (1536) 25.1 / 37.8 / 28.2, an RK4 step of 192x64x64 (2048) 383 plain / 396 three waves.
// Without a magnetic field: Float32 32^3 9.5 / 7.0 / 7.4, 64^3 10.4 / 8.6 / 8.7, 128x96x64 16.0 / 14.1 /
// 13.3, 128^3 (4096) 21.1 / 27.1 / 22.2; Float64 64^3 11.9 / 10.2 / 10.1, 128x96x64 20.2 / 22.5 / 18.9.
inline int rowpair_team(int nx, int phys, bool f64, int64_t pairs) {
  if (!rowteam_length(nx)) return 0;
  const int64_t waves = pairs * (nx / rowpair_E(nx, 1)) / 64;
  if (waves < (f64 && phys == PHYS_MHD ? 192 : 768)) return ROW_TEAM;
  const bool early = nx % 3 ? f64 || phys == PHYS_MHD : f64 && phys == PHYS_MHD && nx > 96;
  return waves < (early ? 1280 : 2560) ? ROW_TEAM_HALF : 0;
}
// The plan of a grid of `pairs` row pairs: plan 1 where one run is a team.  It does not depend on the
// number of runs, so a run ends with the same bits alone and beside others.
inline int rowpair_grid_plan(int nx, int phys, bool f64, int64_t pairs) {
  return rowpair_team(nx, phys, f64, pairs) ? 1 : rowpair_plan(nx, phys, f64);
}
// The launch of `nruns` runs of such a grid: a team (then one run is one too) or the grid's plan.
inline int rowpair_choice(int nx, int phys, bool f64, int64_t pairs, int nruns) {
  const int team = rowpair_team(nx, phys, f64, pairs * nruns);
  return team ? team : rowpair_grid_plan(nx, phys, f64, pairs);
}

template <class T> constexpr int lds_group() { return 128 / (int)sizeof(cx<T>); }
template <class T, int C> __host__ __device__ constexpr int pad(int pos) { return pos + C * (pos / lds_group<T>()); }

// The exchange after the pass (Ns, R): slot of a written position base + r*Ns with
// base = (b / Ns) * Ns*R + b % Ns, and of a read position b + r*B.
template <class T, int Ns, int R> struct Exchange {
  static constexpr int G = lds_group<T>(), NR = Ns * R;
  static constexpr bool POW2 = (NR & (NR - 1)) == 0;
  static constexpr int c2() {
    const int c = Ns >= G ? 0 : (NR >= G ? (Ns == 1 ? 1 : G / R) : Ns);
    return c > 4 ? 0 : c;
  }
  // lanes in the way of each other, summed over a wave's groups, with c padding slots per NR
  static constexpr int conflicts(int c) {
    int sum = 0;
    for (int l0 = 0; l0 < 64; l0 += G) {
      int worst = 0;
      for (int s = 0; s < G; ++s) {
        int n = 0;
        for (int l = l0; l < l0 + G; ++l) n += ((l / Ns) * (NR + c) + l % Ns) % G == s ? 1 : 0;
        worst = n > worst ? n : worst;
      }
      sum += worst;
    }
    return sum;
  }
  static constexpr int block_c() {
    int best = 0;
    for (int c = 1; c < G && c <= NR / 3; ++c) best = conflicts(c) < conflicts(best) ? c : best;
    return best;
  }
  static constexpr int C = POW2 ? c2() : block_c();
  static __device__ __forceinline__ int write_base(int b) {
    if constexpr (POW2) return pad<T, C>((b / Ns) * NR + b % Ns);
    else return (b / Ns) * (NR + C) + b % Ns;
  }
  static constexpr int write_step(int r) { return POW2 ? pad<T, C>(r * Ns) : r * Ns; }
  // slots for N positions
  static constexpr int slots(int N) { return POW2 ? pad<T, C>(N) : N + C * (N / NR); }
  // read slot of b + r*B as base(b) + step(r*B); valid where separable<B>()
  template <int B> static constexpr bool separable() { return POW2 ? B % G == 0 : B % NR == 0; }
  static __device__ __forceinline__ int read_slot(int pos) { return POW2 ? pad<T, C>(pos) : pos + C * (pos / NR); }
  static constexpr int read_step(int pos) { return POW2 ? pad<T, C>(pos) : pos + C * (pos / NR); }
};
// LDS slots a transform needs: the most of any exchange, and N/2 + 1 for the mirror exchange
template <class T, int N, int Ns, class Rad> struct ExchangeSlots;
template <class T, int N, int Ns, int R0> struct ExchangeSlots<T, N, Ns, Radices<R0>> {
  static constexpr int value = N / 2 + 1;
};
template <class T, int N, int Ns, int R, int R2, int... Rest> struct ExchangeSlots<T, N, Ns, Radices<R, R2, Rest...>> {
  static constexpr int a = Exchange<T, Ns, R>::slots(N), b = ExchangeSlots<T, N, Ns * R, Radices<R2, Rest...>>::value;
  static constexpr int value = a > b ? a : b;
};
// values a thread holds during the passes: the most of any pass
template <int N, int TX, class Rad> struct PassValues;
template <int N, int TX> struct PassValues<N, TX, Radices<>> { static constexpr int value = 0; };
template <int N, int TX, int R, int... Rest> struct PassValues<N, TX, Radices<R, Rest...>> {
  static constexpr int a = (N / R + TX - 1) / TX * R, b = PassValues<N, TX, Radices<Rest...>>::value;
  static constexpr int value = a > b ? a : b;
};

// Launch shape: 128 threads, LPW transforms at a time, each of two rows.
template <class T, int NX, int PLAN> struct RowPairShape {
  using P = RowPlan2<T, NX, PLAN>;
  static constexpr int E = P::E;
  static constexpr int TX = NX / E;
  static constexpr int LPW = 128 / TX;
  static constexpr int RPW = 2 * LPW;                        // rows of a work item
  static constexpr int EM = PassValues<NX, TX, typename P::R>::value;
  static constexpr int SI = ExchangeSlots<T, NX, 1, typename P::R>::value, SF = ExchangeSlots<T, NX, 1, typename P::F>::value;
  static constexpr int SLOTS = (SI > SF ? SI : SF) + 2;      // + 2: transforms of one wave on other banks
  static constexpr int LDS_CX = LPW * SLOTS;
  static_assert(128 % TX == 0, "a workgroup holds whole transforms");
  // layouts of the half spectra: of the first inverse and the last forward pass
  static constexpr int R0 = RFirst<typename P::R>::value, B0 = NX / R0, N0 = (B0 + TX - 1) / TX, E0 = N0 * R0;
  static constexpr int RF = RLast<typename P::F>::value, BF = NX / RF, NF = (BF + TX - 1) / TX;
  static_assert(R0 % 2 == 0 && RF % 2 == 0, "a pass's upper half of positions mirrors the lower");
  static_assert(NX / RLast<typename P::R>::value % TX == 0 && NX / RFirst<typename P::F>::value % TX == 0 && E <= EM,
                "the products' layout is full");
};

// Fields requested ahead of the transforms: all of them where they fit the registers
template <class T, int NIN, int E> struct RowAhead {
  static constexpr int fit = (sizeof(T) == 4 ? 24 : 12) / E > 1 ? (sizeof(T) == 4 ? 24 : 12) / E : 1;
  static constexpr int value = fit < NIN ? fit : NIN;
};

// The advective products of one point, u = v[0..2], b = v[3..5], in the order of nprod:
// T_ij = b_i b_j - u_i u_j and M_ij = u_i b_j - b_i u_j, or U_ij = u_i u_j.
//
// What is fused and what is rounded is spelled out, so that every launch that forms a product gives
// the same bits.
template <class T>
__device__ __forceinline__ T diff2(T a, T b, T c, T d) { return fma(a, b, -(c * d)); }  // a b - c d
template <class T>
__device__ __forceinline__ T mul_rounded(T a, T b) {
#pragma clang fp contract(off)
  return a * b;
}
// the indexes i, j of product p
__host__ __device__ constexpr int advective_i(int p) { return p < 3 || p == 6 || p == 7 ? 0 : (p == 5 ? 2 : 1); }
__host__ __device__ constexpr int advective_j(int p) { return p == 0 ? 0 : (p == 1 || p == 3 || p == 6 ? 1 : 2); }
template <class T, int KIND>
__device__ __forceinline__ T advective(int p, const T* v) {
  const int i = advective_i(p), j = advective_j(p);
  if constexpr (KIND == ROW_MHD) {
    if (p < 6) return diff2(v[3 + i], v[3 + j], v[i], v[j]);
    return diff2(v[i], v[3 + j], v[3 + i], v[j]);
  } else {
    return mul_rounded(v[i], v[j]);
  }
}

// a w, or a conj(w) for the inverse direction
template <int S, class T> __device__ __forceinline__ cx<T> row_twmul(cx<T> a, cx<T> w) {
  if (S < 0) return {diff2(a.re, w.re, a.im, w.im), fma(a.re, w.im, a.im * w.re)};
  return {fma(a.re, w.re, a.im * w.im), diff2(a.im, w.re, a.re, w.im)};
}

// Twiddles of every pass but the first, in registers
template <class T, int N, int TX, int Ns, class Rad> struct RowTw;
template <class T, int N, int TX, int Ns> struct RowTw<T, N, TX, Ns, Radices<>> {
  __device__ __forceinline__ void load(int, const cx<T>*) {}
};
template <class T, int N, int TX, int Ns, int R, int... Rest> struct RowTw<T, N, TX, Ns, Radices<R, Rest...>> {
  static constexpr int NB = (N / R + TX - 1) / TX;
  // butterflies t + i*TX whose index modulo Ns is the same share their twiddles
  static constexpr int NT = Ns == 1 ? 0 : (TX % Ns == 0 ? 1 : NB);
  cx<T> w[NT > 0 ? NT : 1][R > 1 ? R - 1 : 1];
  RowTw<T, N, TX, Ns * R, Radices<Rest...>> next;
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

// One transform of direction S, in place: before a pass of radix R, x[i + r*NB] is the value at
// position b + r*B, b = t + i*TX; after the last pass x[i + r*NB] is the value at b + r*B of that
// pass.  row: the transform's LDS slots.  A sync precedes every exchange write.
template <class T, int N, int TX, int S, bool WS, int Ns, class Rad> struct RowPass;
template <class T, int N, int TX, int S, bool WS, int Ns> struct RowPass<T, N, TX, S, WS, Ns, Radices<>> {
  template <class Tw> static __device__ __forceinline__ void run(cx<T>*, int, cx<T>*, const Tw&) {}
};
template <class T, int N, int TX, int S, bool WS, int Ns, int R, int... Rest>
struct RowPass<T, N, TX, S, WS, Ns, Radices<R, Rest...>> {
  template <class Tw>
  static __device__ __forceinline__ void run(cx<T>* x, int t, cx<T>* row, const Tw& tw) {
    constexpr int B = N / R, NB = (B + TX - 1) / TX;
    constexpr bool LAST = sizeof...(Rest) == 0;
    using X = Exchange<T, Ns, R>;
    if constexpr (!LAST) xsync<WS>();
#pragma unroll
    for (int i = 0; i < NB; ++i) {
      const int b = t + i * TX;
      if ((i + 1) * TX <= B || b < B) {
        cx<T> v[R];
#pragma unroll
        for (int r = 0; r < R; ++r) {
          v[r] = x[i + r * NB];
          if constexpr (Ns > 1)
            if (r > 0) v[r] = row_twmul<S>(v[r], tw.w[Tw::NT == 1 ? 0 : i][r > 0 ? r - 1 : 0]);
        }
        Bfly<T, R, S>::run(v);
        if constexpr (LAST) {
#pragma unroll
          for (int r = 0; r < R; ++r) x[i + r * NB] = v[r];
        } else {
          cx<T>* const d = row + X::write_base(b);
#pragma unroll
          for (int r = 0; r < R; ++r) d[X::write_step(r)] = v[r];
        }
      }
    }
    if constexpr (!LAST) {
      xsync<WS>();
      constexpr int R2 = RFirst<Radices<Rest...>>::value, B2 = N / R2, NB2 = (B2 + TX - 1) / TX;
#pragma unroll
      for (int i = 0; i < NB2; ++i) {
        const int b = t + i * TX;
        if ((i + 1) * TX <= B2 || b < B2) {
          if constexpr (X::template separable<B2>()) {
            const cx<T>* const s = row + X::read_slot(b);
#pragma unroll
            for (int r = 0; r < R2; ++r) x[i + r * NB2] = s[X::read_step(r * B2)];
          } else {
#pragma unroll
            for (int r = 0; r < R2; ++r) x[i + r * NB2] = row[X::read_slot(b + r * B2)];
          }
        }
      }
      RowPass<T, N, TX, S, WS, Ns * R, Radices<Rest...>>::run(x, t, row, tw.next);
    }
  }
};

// The packed row of a pair of rows from their half-spectrum entries A, B of element e
template <class T, int NX, class SHP>
__device__ __forceinline__ cx<T> row_pack(cx<T> A, cx<T> B, int e, int tr) {
  const int i = e % SHP::N0, r = e / SHP::N0;
  // c2r ignores Im of the DC and Nyquist entries
  if (i == 0 && (r == 0 || r == SHP::R0 / 2) && tr == 0) A.im = B.im = T(0);
  return r < SHP::R0 / 2 ? cx<T>{A.re - B.im, A.im + B.re} : cx<T>{A.re + B.im, B.re - A.im};
}

// Store the half spectra of the two real rows whose packed transform is w (last forward pass's
// layout): entries [0, kend) of each, at da + o and dc + o with o = oup + k - tr.
template <class T, int NX, class SHP>
__device__ __forceinline__ void row_store(const cx<T>* w, int tr, cx<T>* xrow, gptr<cx<T>> da, gptr<cx<T>> dc,
                                          uint32_t oup, int kend) {
  constexpr int TX = SHP::TX, RF = SHP::RF, BF = SHP::BF, NF = SHP::NF;
  // mirror exchange: the value at position q = b + r*BF >= NX/2 goes to slot NX - q
  xsync<(SHP::TX <= 64)>();
#pragma unroll
  for (int r = RF / 2; r < RF; ++r)
#pragma unroll
    for (int ii = 0; ii < NF; ++ii) {
      const int b = tr + ii * TX;
      if ((ii + 1) * TX <= BF || b < BF) xrow[(RF - r) * BF - b] = w[ii + r * NF];
    }
  xsync<(SHP::TX <= 64)>();
  // twice the product's half spectrum is stored (rhs_at halves it): no factor 1/2 here
#pragma unroll
  for (int r = 0; r < RF / 2; ++r)
#pragma unroll
    for (int ii = 0; ii < NF; ++ii) {
      const int b = tr + ii * TX, k = b + r * BF;
      if (k < kend && ((ii + 1) * TX <= BF || b < BF)) {
        const cx<T> Z = w[ii + r * NF];
        cx<T> Zm = xrow[k];
        if (ii == 0 && r == 0 && tr == 0) Zm = Z;  // entry 0 is its own mirror
        const uint32_t o = oup + (ii * TX + r * BF);
        stst<false, T>(da + o, cx<T>{Z.re + Zm.re, Z.im - Zm.im});
        stst<false, T>(dc + o, cx<T>{Z.im + Zm.im, Zm.re - Z.re});
      }
    }
  if (NX / 2 < kend) {
    // the Nyquist entry is thread 0's value at position NX/2; zeros follow it to the line's end
    const cx<T> nq = w[RF / 2 * NF];
    const T nr = tr == 0 ? T(2) * nq.re : T(0), ni = tr == 0 ? T(2) * nq.im : T(0);
    for (int k = tr; k < kend - NX / 2; k += TX) {
      stst<false, T>(da + (oup + NX / 2 + (k - tr)), cx<T>{k == tr ? nr : T(0), T(0)});
      stst<false, T>(dc + (oup + NX / 2 + (k - tr)), cx<T>{k == tr ? ni : T(0), T(0)});
    }
  }
}

// One work item (RPW rows of one run), run by a 128-thread workgroup.  xbuf holds
// RowPairShape::LDS_CX exchange slots, red 2*128 values and stw NX twiddles.  Every early return
// is taken by the whole workgroup.
template <class T, int NX, int KIND, int PLAN>
__device__ __forceinline__ void rowpair_item(const RowArgs& a, int64_t item, const RunBuf<T>* __restrict__ runs,
                                             const cx<T>* __restrict__ twx, cx<T>* xbuf, T* red, cx<T>* stw) {
  static_assert(KIND == ROW_MHD || KIND == ROW_HD, "the fused kinds");
  using SHP = RowPairShape<T, NX, PLAN>;
  using P = typename SHP::P;
  using Inv = typename P::R;
  using Fwd = typename P::F;
  constexpr int E = SHP::E, TX = SHP::TX, EM = SHP::EM;
  constexpr int NIN = KIND == ROW_MHD ? 6 : 3, NPROD = KIND == ROW_MHD ? 9 : 6;
  constexpr bool WS = TX <= 64;
  constexpr int R0 = SHP::R0, B0 = SHP::B0, N0 = SHP::N0, E0 = SHP::E0;

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

  // The entries of the two half spectra of field f that position p = b + r*B0 takes: entry p for
  // p < NX/2 (r < R0/2), the mirrored entry NX - p otherwise.  AHEAD fields are requested before
  // the first transform starts, so the loads' latencies overlap.  Addresses are a uniform base (the
  // item's first row of a field) plus a 32-bit offset and a constant.
  constexpr int AHEAD = RowAhead<T, NIN, E0>::value;
  const int ncols = a.in_ncols;
  cx<T> ra[NIN][E0], rc[NIN][E0];
  const int64_t ifs = field_stride(G, a.in_sel), irs = row_stride(G, a.in_sel);
  const int64_t ifirst = row_offset(G, a.in_sel, first);
  const gptr<const cx<T>> src = gmem<const cx<T>>(rb.buf[a.in_sel]) + (int64_t)a.in_f0 * ifs + ifirst;
  const uint32_t ioff = ok ? (uint32_t)(row_offset(G, a.in_sel, row0) - ifirst) : 0u;
  const uint32_t iup = ioff + tr, idn = ioff + (NX / 2 - tr);  // entries tr, NX/2 - tr of row0
  auto request = [&](int f0, int f1) {
#pragma unroll
    for (int f = f0; f < f1; ++f)
#pragma unroll
      for (int e = 0; e < E0; ++e) ra[f][e] = rc[f][e] = cx<T>{T(0), T(0)};
#pragma unroll
    for (int r = 0; r < R0; ++r)
#pragma unroll
      for (int i = 0; i < N0; ++i) {
        const int b = tr + i * TX;
        // entry up + b (r < R0/2) or down - b
        const int up = r * B0, down = (R0 - r) * B0;
        const int k = r < R0 / 2 ? up + b : down - b;
        if (k < ncols && ((i + 1) * TX <= B0 || b < B0)) {
          const uint32_t o = r < R0 / 2 ? iup + (up + i * TX) : idn - (NX / 2 - down + i * TX);
#pragma unroll
          for (int f = f0; f < f1; ++f) {
            const gptr<const cx<T>> pa = src + (int64_t)f * ifs, pc = pa + irs;
            ra[f][i + r * N0] = ldst<false, T>(pa + o);
            rc[f][i + r * N0] = ldst<false, T>(pc + o);
          }
        }
      }
  };
  request(0, AHEAD);

  // z[f][e].re, .im: field f of the two rows at x = tr + e*TX
  cx<T> z[NIN][E];
  const T scale = T(G.inv_n);
  RowTw<T, NX, TX, 1, Inv> twi;
  twi.load(tr, stw);
#pragma unroll
  for (int f = 0; f < NIN; ++f) {
    if (f + AHEAD < NIN) request(f + AHEAD, f + AHEAD + 1);
    cx<T> x[EM];
#pragma unroll
    for (int e = 0; e < E0; ++e) x[e] = row_pack<T, NX, SHP>(ra[f][e], rc[f][e], e, tr);
    RowPass<T, NX, TX, 1, WS, 1, Inv>::run(x, tr, xrow, twi);
#pragma unroll
    for (int e = 0; e < E; ++e) z[f][e] = x[e] * scale;
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
  RowTw<T, NX, TX, 1, Fwd> twf;
  if constexpr (std::is_same<Inv, Fwd>::value) twf = twi;
  else twf.load(tr, stw);
#pragma unroll
  for (int p = 0; p < NPROD; ++p) {
    cx<T> w[EM];
#pragma unroll
    for (int j = 0; j < E; ++j) {
      T v[NIN], u[NIN];
#pragma unroll
      for (int f = 0; f < NIN; ++f) { v[f] = z[f][j].re; u[f] = z[f][j].im; }
      w[j] = cx<T>{advective<T, KIND>(p, v), advective<T, KIND>(p, u)};
    }
    RowPass<T, NX, TX, -1, WS, 1, Fwd>::run(w, tr, xrow, twf);
    const gptr<cx<T>> da = out + (int64_t)p * ofs;
    row_store<T, NX, SHP>(w, tr, xrow, da, da + ors, oup, kend);
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

// ---------------------------------------------------------------------------
// The same launch for grids too small to fill the chip: a row pair's transforms side by side.
// ---------------------------------------------------------------------------
// Bound by latency: rowpair_kernel's waves there are fewer than SIMDs, and each runs its transforms
// one after the other.  Here a workgroup of NT waves takes 64 / TX row pairs; wave q transforms the
// fields q, q + NT, ... of all of them, leaves the real values in LDS, and after one barrier forms,
// transforms and stores the products q, q + NT, ...  Field and product numbers are a wave's, so
// nothing diverges.  A product reads four (HD: two) fields back from LDS, which costs more LDS
// traffic and address arithmetic than the registers of rowpair_kernel: full chips take that one.
// The results are rowpair_kernel's with plan 1, bit for bit.
template <class T, int NX, int KIND, int NT> struct RowTeamShape {
  using SHP = RowPairShape<T, NX, 1>;
  static constexpr int TX = SHP::TX;
  static constexpr int LPT = 64 / TX;                        // row pairs of a work item
  static constexpr int NIN = KIND == ROW_MHD ? 6 : 3;
  static constexpr int THREADS = 64 * NT;
  static constexpr int LDS_CX = NT * LPT * SHP::SLOTS + NIN * LPT * NX;
  static_assert(TX <= 64, "a wave holds whole transforms");
};

template <class T, int NX, int KIND, int NT>
__global__ void __launch_bounds__(64 * NT)
rowteam_kernel(RowArgs a, const RunBuf<T>* __restrict__ runs, const cx<T>* __restrict__ twx) {
  using TS = RowTeamShape<T, NX, KIND, NT>;
  using SHP = typename TS::SHP;
  using Inv = typename SHP::P::R;
  using Fwd = typename SHP::P::F;
  constexpr int E = SHP::E, TX = SHP::TX, EM = SHP::EM, LPT = TS::LPT;
  constexpr int R0 = SHP::R0, B0 = SHP::B0, N0 = SHP::N0, E0 = SHP::E0;
  constexpr int NIN = TS::NIN, NPROD = KIND == ROW_MHD ? 9 : 6;
  constexpr int NFT = (NIN + NT - 1) / NT;  // fields a wave transforms, at most
  __shared__ cx<T> lds[TS::LDS_CX];
  __shared__ T red[2 * NT];
  __shared__ cx<T> stw[NX];
  const int64_t item = xcd_item(blockIdx.x, (int64_t)gridDim.x);
  if (item >= a.blocks_per_run * a.nruns) return;

  const int t = threadIdx.x, team = __builtin_amdgcn_readfirstlane(t / 64);
  const int lane = t % 64, rw = lane / TX, tr = lane % TX;
  const Geom& G = a.g;
  const int run = (int)(item / a.blocks_per_run);
  const int64_t blk = a.blk0 + item % a.blocks_per_run;
  // rows as in rowpair_item
  const int64_t first = blk * (2 * LPT), row0 = first + 2 * rw;
  const bool ok = row0 < a.rows;
  const RunBuf<T>& rb = runs[run];
  if (gated_off(a.gate, rb)) return;
  const bool pruned = a.prune_out && step_pruned(rb);
  cx<T>* const xrow = lds + (team * LPT + rw) * SHP::SLOTS;
  cx<T>* const zs = lds + NT * LPT * SHP::SLOTS + rw * NX + tr;  // field f's values at zs[f * LPT * NX + e * TX]

  const int ncols = a.in_ncols;
  cx<T> ra[NFT][E0], rc[NFT][E0];
  const int64_t ifs = field_stride(G, a.in_sel), irs = row_stride(G, a.in_sel);
  const int64_t ifirst = row_offset(G, a.in_sel, first);
  const gptr<const cx<T>> src = gmem<const cx<T>>(rb.buf[a.in_sel]) + (int64_t)a.in_f0 * ifs + ifirst;
  const uint32_t ioff = ok ? (uint32_t)(row_offset(G, a.in_sel, row0) - ifirst) : 0u;
  const uint32_t iup = ioff + tr, idn = ioff + (NX / 2 - tr);  // entries tr, NX/2 - tr of row0
#pragma unroll
  for (int q = 0; q < NFT; ++q) {
    const int f = team + q * NT;
    const gptr<const cx<T>> pa = src + (int64_t)f * ifs, pc = pa + irs;
#pragma unroll
    for (int r = 0; r < R0; ++r)
#pragma unroll
      for (int i = 0; i < N0; ++i) {
        const int b = tr + i * TX, up = r * B0, down = (R0 - r) * B0;
        const int k = r < R0 / 2 ? up + b : down - b;
        cx<T> A{T(0), T(0)}, B{T(0), T(0)};
        if (f < NIN && k < ncols && ((i + 1) * TX <= B0 || b < B0)) {
          const uint32_t o = r < R0 / 2 ? iup + (up + i * TX) : idn - (NX / 2 - down + i * TX);
          A = ldst<false, T>(pa + o);
          B = ldst<false, T>(pc + o);
        }
        ra[q][i + r * N0] = A;
        rc[q][i + r * N0] = B;
      }
  }
  for (int i = t; i < NX; i += TS::THREADS) stw[i] = twx[i];
  __syncthreads();

  const T scale = T(G.inv_n);
  const bool put_vars = a.write_vars && !pruned && ok;
  T mu = T(0), mb = T(0);
  {
    RowTw<T, NX, TX, 1, Inv> tw;
    tw.load(tr, stw);
#pragma unroll
    for (int q = 0; q < NFT; ++q) {
      const int f = team + q * NT;
      if (f >= NIN) break;
      cx<T> x[EM];
#pragma unroll
      for (int e = 0; e < E0; ++e) x[e] = row_pack<T, NX, SHP>(ra[q][e], rc[q][e], e, tr);
      RowPass<T, NX, TX, 1, true, 1, Inv>::run(x, tr, xrow, tw);
#pragma unroll
      for (int e = 0; e < E; ++e) {
        x[e] = x[e] * scale;
        zs[f * (LPT * NX) + e * TX] = x[e];
      }
      if (put_vars) {
        const gptr<T> va = gmem(rb.vars) + (int64_t)(a.real_out_f0 + f) * G.nr + first * NX;
        const uint32_t o = (uint32_t)(2 * rw * NX + tr);
#pragma unroll
        for (int e = 0; e < E; ++e) {
          va[o + e * TX] = x[e].re;
          va[o + NX + e * TX] = x[e].im;
        }
      }
      if (a.want_max) {
        T m = T(0);
#pragma unroll
        for (int e = 0; e < E; ++e) m = nanmax(nanmax(m, fabs(x[e].re)), fabs(x[e].im));
        if (f < 3) mu = nanmax(mu, m);
        else mb = nanmax(mb, m);
      }
    }
  }
  if (a.want_max) {
#pragma unroll
    for (int s = 32; s > 0; s >>= 1) {
      mu = nanmax(mu, __shfl_xor(mu, s));
      mb = nanmax(mb, __shfl_xor(mb, s));
    }
    if (lane == 0) {
      red[2 * team] = mu * mu;
      red[2 * team + 1] = mb * mb;
    }
  }
  __syncthreads();
  if (a.want_max && t == 0) {
    T m0 = red[0], m1 = red[1];
    for (int q = 1; q < NT; ++q) {
      m0 = nanmax(m0, red[2 * q]);
      m1 = nanmax(m1, red[2 * q + 1]);
    }
    const gptr<T> part = gmem(rb.partial);
    part[2 * blk] = m0;
    part[2 * blk + 1] = m1;
  }

  const bool dst_work = a.out_sel == B_WORK;
  const int kfull = dst_work ? G.wrs : NX / 2 + 1;
  const int kend = !ok ? 0 : (pruned ? (dst_work ? G.kx_keep_w : G.kx_keep) : kfull);
  const int64_t ofs = field_stride(G, a.out_sel), ors = row_stride(G, a.out_sel);
  const int64_t ofirst = row_offset(G, a.out_sel, first);
  const gptr<cx<T>> out = gmem(rb.buf[a.out_sel]) + (int64_t)a.out_f0 * ofs + ofirst;
  const uint32_t oup = (ok ? (uint32_t)(row_offset(G, a.out_sel, row0) - ofirst) : 0u) + tr;
  RowTw<T, NX, TX, 1, Fwd> tw;
  tw.load(tr, stw);
  for (int p = team; p < NPROD; p += NT) {
    const cx<T>* const zi = zs + advective_i(p) * (LPT * NX);
    const cx<T>* const zj = zs + advective_j(p) * (LPT * NX);
    cx<T> w[EM];
#pragma unroll
    for (int e = 0; e < E; ++e) {
      const cx<T> ui = zi[e * TX], uj = zj[e * TX];
      if constexpr (KIND == ROW_MHD) {
        const cx<T> bi = zi[3 * LPT * NX + e * TX], bj = zj[3 * LPT * NX + e * TX];
        if (p < 6) w[e] = cx<T>{diff2(bi.re, bj.re, ui.re, uj.re), diff2(bi.im, bj.im, ui.im, uj.im)};
        else w[e] = cx<T>{diff2(ui.re, bj.re, bi.re, uj.re), diff2(ui.im, bj.im, bi.im, uj.im)};
      } else {
        w[e] = cx<T>{mul_rounded(ui.re, uj.re), mul_rounded(ui.im, uj.im)};
      }
    }
    RowPass<T, NX, TX, -1, true, 1, Fwd>::run(w, tr, xrow, tw);
    const gptr<cx<T>> da = out + (int64_t)p * ofs;
    row_store<T, NX, SHP>(w, tr, xrow, da, da + ors, oup, kend);
  }
}

}  // namespace mhd
