// Runs the kernels of Runge-Kutta steps on the host, with every buffer of a run at the end (or at the
// start) of pages whose neighbours cannot be touched: an access past a buffer ends the program and
// names the kernel.  Also checks that the launches meant to give the same bits do: the two access
// forms of the spectral kernel, and the row kernel against its teams.
//
// kernel_bounds <float|double>: prints "ok" and returns 0 if nothing was out of bounds.
#include <signal.h>
#include <sys/mman.h>
#include <ucontext.h>
#include <unistd.h>

#include <cstdio>
#include <cstdlib>
#include <functional>
#include <random>
#include <string>
#include <vector>

#include "mhd_kernels.hpp"
#include "mhd_row.hpp"

dim3 threadIdx, blockIdx, blockDim, gridDim;

using namespace mhd;

// ---- fibers -------------------------------------------------------------------
namespace {
constexpr size_t STACK = 256 << 10;
struct Fiber {
  ucontext_t ctx;
  std::vector<char> stack;
  int state = 0;  // 0 running, 1 at a block barrier, 2 at a wave barrier, 3 done
  double val = 0;
};
std::vector<Fiber> fibers;
ucontext_t sched;
int cur = 0, nlive = 0;
std::function<void()> body;
std::string what;

void entry() {
  body();
  fibers[cur].state = 3;
  swapcontext(&fibers[cur].ctx, &sched);
}
void yield(int state) {
  const int me = cur;
  fibers[me].state = state;
  swapcontext(&fibers[me].ctx, &sched);
}

[[noreturn]] void die(const std::string& m) {
  fprintf(stderr, "%s: %s\n", what.c_str(), m.c_str());
  exit(1);
}

// one workgroup of n threads
void run_block(int n) {
  if ((int)fibers.size() < n) fibers.resize(n);
  for (int i = 0; i < n; ++i) {
    Fiber& f = fibers[i];
    if (f.stack.empty()) f.stack.resize(STACK);
    getcontext(&f.ctx);
    f.ctx.uc_stack.ss_sp = f.stack.data();
    f.ctx.uc_stack.ss_size = STACK;
    f.ctx.uc_link = nullptr;
    f.state = 0;
    makecontext(&f.ctx, entry, 0);
  }
  for (;;) {
    for (int i = 0; i < n; ++i) {
      if (fibers[i].state != 0) continue;
      cur = i;
      threadIdx.x = (unsigned)i;
      swapcontext(&sched, &fibers[i].ctx);
    }
    // release each wave that stands whole at a wave barrier, else the block at its barrier
    bool moved = false, done = true;
    for (int w = 0; w < n; w += 64) {
      int waiting = 0, over = 0;
      const int e = w + 64 < n ? w + 64 : n;
      for (int i = w; i < e; ++i) {
        waiting += fibers[i].state == 2;
        over += fibers[i].state == 3;
      }
      done = done && over == e - w;
      if (!waiting) continue;
      if (waiting != e - w) die("a wave's lanes part at a wave barrier");
      for (int i = w; i < e; ++i) fibers[i].state = 0;
      moved = true;
    }
    if (done) return;
    if (moved) continue;
    for (int i = 0; i < n; ++i)
      if (fibers[i].state != 1) die("a thread left before a block barrier");
    for (int i = 0; i < n; ++i) fibers[i].state = 0;
  }
}

// kernels without barriers: one thread after the other
template <class F> void run_plain(dim3 grid, int threads, F&& f) {
  for (blockIdx.z = 0; blockIdx.z < grid.z; ++blockIdx.z)
    for (blockIdx.y = 0; blockIdx.y < grid.y; ++blockIdx.y)
      for (blockIdx.x = 0; blockIdx.x < grid.x; ++blockIdx.x)
        for (int t = 0; t < threads; ++t) {
          threadIdx.x = (unsigned)t;
          f();
        }
  blockIdx = dim3(0, 0, 0);
}
template <class F> void run_fibers(unsigned nb, int threads, F&& f) {
  body = f;
  gridDim = dim3(nb);
  for (unsigned b = 0; b < nb; ++b) {
    blockIdx = dim3(b, 0, 0);
    run_block(threads);
  }
}
}  // namespace

void host_block_barrier() { yield(1); }
void host_wave_barrier() { yield(2); }
double host_wave_xor(double v, int mask) {
  fibers[cur].val = v;
  const int me = cur;
  yield(2);
  const double r = fibers[me ^ mask].val;
  yield(2);
  return r;
}

// ---- guarded buffers ----------------------------------------------------------
namespace {
bool at_end = true;
const size_t PAGE = 4096;
template <class U> U* guarded(size_t n) {
  const size_t bytes = n * sizeof(U), pages = (bytes + PAGE - 1) / PAGE;
  char* p = (char*)mmap(nullptr, (pages + 2) * PAGE, PROT_NONE, MAP_PRIVATE | MAP_ANONYMOUS, -1, 0);
  if (p == MAP_FAILED || mprotect(p + PAGE, pages * PAGE, PROT_READ | PROT_WRITE)) die("mmap");
  return (U*)(p + PAGE + (at_end ? pages * PAGE - bytes : 0));
}
void on_fault(int) {
  const char m[] = ": access outside a buffer\n";
  (void)!write(2, what.c_str(), what.size());
  (void)!write(2, m, sizeof(m) - 1);
  _exit(2);
}

template <class T> std::vector<cx<T>> table(int n, int cnt) {
  std::vector<cx<T>> h(cnt);
  for (int m = 0; m < cnt; ++m) h[m] = {(T)cos(2 * M_PI * m / n), (T)-sin(2 * M_PI * m / n)};
  return h;
}
template <class T> cx<T>* guarded_table(int n, int cnt) {
  const auto h = table<T>(n, cnt);
  cx<T>* d = guarded<cx<T>>(cnt);
  memcpy(d, h.data(), cnt * sizeof(cx<T>));
  return d;
}

// ---- one run ------------------------------------------------------------------
template <class T, int NX, int NY, int NZ, int PHYS> struct Run {
  static constexpr int NF = PHYS == PHYS_MHD ? 6 : 3, KIND = PHYS == PHYS_MHD ? ROW_MHD : ROW_HD;
  static constexpr int S = 128 / (int)sizeof(cx<T>);
  Geom g;
  RunBuf<T>* rb;
  cx<T>*twx, *twy, *twz;
  int np = nprod(PHYS);

  Run() {
    g = make_geom(NX, NY, NZ, 2 * M_PI, 2 * M_PI, 2 * M_PI, (int)sizeof(cx<T>));
    rb = guarded<RunBuf<T>>(1);
    memset((void*)rb, 0, sizeof(*rb));
    for (int b : {B_SOL, B_STIN, B_ACC}) rb->buf[b] = guarded<cx<T>>((size_t)g.nc * NF);
    rb->buf[B_WORK] = guarded<cx<T>>((size_t)g.wnc * np);
    rb->vars = guarded<T>((size_t)g.nr * NF);
    rb->partial = guarded<T>(2 * (size_t)blocks(rows_per_block(2)));  // the most of any launch
    rb->plane = guarded<cx<T>>((size_t)NF * NY * NZ);
    rb->clk = guarded<RunClock>(1);
    rb->nu = rb->eta = 1e-3;
    rb->nnu = 2;
    rb->clk->dt = 1e-3;
    rb->clk->target = INT64_MAX;
    rb->clk->use_cfl = 1;
    rb->clk->cfl_coef = 0.3;
    rb->clk->dl = 2 * M_PI / NX;
    rb->clk->t_diff = 1.0;
    rb->clk->maxu2 = rb->clk->maxb2 = 1.0;
    twx = guarded_table<T>(NX, NX);
    twy = guarded_table<T>(NY, NY);
    twz = guarded_table<T>(NZ, NZ);
    std::mt19937_64 rng(3);
    std::normal_distribution<double> nd;
    for (int64_t i = 0; i < g.nc * NF; ++i) rb->buf[B_SOL][i] = {(T)nd(rng), (T)nd(rng)};
    for (int64_t i = 0; i < g.wnc * np; ++i) rb->buf[B_WORK][i] = {(T)nd(rng), (T)nd(rng)};
  }

  template <int DIR, int N> void colpass(const char* name, int axis, int src, int nfields, bool prune, bool plane, bool cfl) {
    what = name;
    ColArgs a{};
    a.g = g;
    a.axis = axis;
    a.nfields = nfields;
    a.src = src;
    a.dst = B_WORK;
    a.ncols = prune ? g.kx_keep : g.nkr;
    const int scols = a.ncols >= g.nkr ? g.wrs : g.kx_keep_w;
    a.nstrips = ((a.ncols > scols ? a.ncols : scols) + S - 1) / S;
    a.nother = a.other_lo_end = axis == 1 ? NZ : NY;
    if (axis == 2 && prune) {
      a.nother = nkept_y(g);
      a.other_lo_end = g.ly_lo_end;
      a.other_gap = g.ly_hi_begin - g.ly_lo_end;
    }
    if (prune) {
      a.mask_lo = axis == 1 ? g.ly_lo_end : g.mz_lo_end;
      a.mask_hi = axis == 1 ? g.ly_hi_begin : g.mz_hi_begin;
    }
    a.nruns = 1;
    a.nitems = (int64_t)nfields * a.nother * a.nstrips;
    a.gate = 1;
    a.plane_out = plane;
    a.prune_out = DIR < 0;
    a.cfl = cfl ? 2 : 0;
    run_fibers((unsigned)((a.nitems + 7) / 8 * 8), S * (N / Plan<N>::E),
               [&] { colpass_kernel<T, N, S, DIR>(a, rb, axis == 1 ? twy : twz); });
  }

  // launch: 0, 1 the plans; 2, 3 the teams
  static int rows_per_block(int launch) {
    if (launch >= 2) return 2 * (64 / (NX / RowPlan2<T, NX, 1>::E));
    return launch ? RowPairShape<T, NX, 1>::RPW : RowPairShape<T, NX, 0>::RPW;
  }
  static int blocks(int rpb) { return (NY * NZ + rpb - 1) / rpb; }
  int rows(int launch, bool last) {
    what = "row launch " + std::to_string(launch);
    RowArgs r{};
    r.g = g;
    r.nruns = 1;
    r.rows = (int64_t)NY * NZ;
    r.blocks_per_run = blocks(rows_per_block(launch));
    r.in_sel = r.out_sel = B_WORK;
    r.in_ncols = g.kx_keep;
    r.write_vars = r.want_max = last;
    r.gate = r.prune_out = 1;
    const unsigned nb = (unsigned)((r.blocks_per_run + 7) / 8 * 8);
    constexpr int FULL = PHYS == PHYS_MHD ? 9 : 6, HALF = 3;
    if (launch == 0) run_fibers(nb, 128, [&] { rowpair_kernel<T, NX, KIND, 0>(r, rb, twx); });
    else if (launch == 1) run_fibers(nb, 128, [&] { rowpair_kernel<T, NX, KIND, 1>(r, rb, twx); });
    else if (launch == 2) run_fibers(nb, 64 * FULL, [&] { rowteam_kernel<T, NX, KIND, FULL>(r, rb, twx); });
    else run_fibers(nb, 64 * HALF, [&] { rowteam_kernel<T, NX, KIND, HALF>(r, rb, twx); });
    return (int)r.blocks_per_run;
  }

  template <bool NT> void spectral(int stepper, int stage) {
    what = "spectral stage " + std::to_string(stage) + (NT ? "" : " plain");
    static const double A[5] = {0.0, -0.4, -1.2, -1.7, -1.5}, B[5] = {0.15, 0.4, 0.8, 0.7, 0.15};
    SpecArgs s{};
    s.g = g;
    s.nruns = 1;
    s.mode = stepper;
    s.stage = stage;
    s.in_sel = stepper == SP_RK4 && stage > 0 ? B_STIN : B_SOL;
    s.mask_input = s.add_force = 1;
    s.self_sel = -1;
    s.f_hi = NF;
    s.prod_sel = B_WORK;
    s.nitems = g.nc;
    s.planes = 2;
    s.gate = 1;
    s.ca = A[stage];
    s.cb = B[stage];
    blockDim = dim3(256);
    run_plain(dim3((unsigned)((g.ny * g.nkr + 255) / 256), NZ, 1), 256,
              [&] { spectral_kernel<T, PHYS, 2, 0, NT>(s, rb); });
  }

  template <bool NT> void step(int stepper, int launch, bool pruned) {
    rb->clk->prune_until = pruned ? rb->clk->step + 2 : 0;
    const int stages = stepper == SP_RK4 ? 4 : 5;
    for (int st = 0; st < stages; ++st) {
      const bool last = st == stages - 1;
      colpass<1, NZ>("inverse z", 2, stepper == SP_RK4 && st > 0 ? B_STIN : B_SOL, NF, true, true, st == 0);
      colpass<1, NY>("inverse y", 1, B_WORK, NF, true, false, false);
      const int blocks = rows(launch, last);
      colpass<-1, NY>("forward y", 1, B_WORK, np, false, false, false);
      colpass<-1, NZ>("forward z", 2, B_WORK, np, false, false, false);
      spectral<NT>(stepper, st);
      if (last) {
        what = "maxima";
        blockDim = dim3(256);
        run_fibers(1, 256, [&] { reduce_max_kernel<T>(rb, blocks, 1); });
      }
    }
  }
};

template <class T> bool same(const std::vector<cx<T>>& a, const std::vector<cx<T>>& b) {
  return a.size() == b.size() && memcmp(a.data(), b.data(), a.size() * sizeof(cx<T>)) == 0;
}

// a dealiased and a full step with every row launch
template <class T, int NX, int NY, int NZ, int PHYS> void steps(int stepper) {
  std::vector<cx<T>> ref;
  for (int launch : {1, 2, 3, 0}) {
    Run<T, NX, NY, NZ, PHYS> r;
    for (bool pruned : {true, false}) r.template step<true>(stepper, launch, pruned);
    const std::vector<cx<T>> sol(r.rb->buf[B_SOL], r.rb->buf[B_SOL] + r.g.nc * r.NF);
    what = "row launch " + std::to_string(launch);
    if (launch == 1) ref = sol;
    else if (launch > 1 && !same(ref, sol)) die("other bits");
  }
}

// every stage of the spectral kernel in both access forms, on whatever the buffers hold
template <class T, int N, int PHYS, bool NT> std::vector<cx<T>> stages(int stepper) {
  Run<T, N, N, N, PHYS> r;
  for (bool pruned : {true, false}) {
    r.rb->clk->prune_until = pruned ? r.rb->clk->step + 2 : 0;
    for (int st = 0; st < (stepper == SP_RK4 ? 4 : 5); ++st) r.template spectral<NT>(stepper, st);
  }
  return std::vector<cx<T>>(r.rb->buf[B_SOL], r.rb->buf[B_SOL] + r.g.nc * r.NF);
}
template <class T, int N, int PHYS> void spectral_forms(int stepper) {
  const auto a = stages<T, N, PHYS, true>(stepper), b = stages<T, N, PHYS, false>(stepper);
  what = "spectral forms";
  if (!same(a, b)) die("other bits");
}

template <class T> void all() {
  spectral_forms<T, 64, PHYS_MHD>(SP_RK4);
  spectral_forms<T, 64, PHYS_MHD>(SP_LSRK54);
  spectral_forms<T, 24, PHYS_HD>(SP_RK4);
  steps<T, 16, 8, 24, PHYS_MHD>(SP_RK4);
  steps<T, 64, 8, 8, PHYS_MHD>(SP_RK4);
  steps<T, 48, 8, 8, PHYS_HD>(SP_LSRK54);
}
}  // namespace

int main(int argc, char** argv) {
  signal(SIGSEGV, on_fault);
  signal(SIGBUS, on_fault);
  if (argc != 2) return 1;
  for (bool end : {true, false}) {
    at_end = end;
    if (std::string(argv[1]) == "float") all<float>();
    else all<double>();
  }
  printf("ok\n");
  return 0;
}
