// Multi-shift CG, spectral bounds and the overlap operator (see msolve.hpp).
#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstdlib>
#include <random>
#include <stdexcept>

#include "msolve.hpp"
#include "stencil.hpp"

namespace qed3 {
namespace {

// fields y_k with coefficients a_k for k_combine
struct ShiftSet {
  Spin<double>* x[kMaxShifts];
  double a[kMaxShifts];
  int n;
};

struct FinStore {
  double2* out;
  __device__ bool skip() const { return false; }
  __device__ void operator()(double2 t) const { *out = t; }
};

__device__ __forceinline__ void axpy_(Spin<double>& y, double a, const Spin<double>& x) {
  y.a.x += a * x.a.x;
  y.a.y += a * x.a.y;
  y.b.x += a * x.b.x;
  y.b.y += a * x.b.y;
}
__device__ __forceinline__ double nrm2(const Spin<double>& v) {
  return v.a.x * v.a.x + v.a.y * v.a.y + v.b.x * v.b.x + v.b.y * v.b.y;
}

// partials of (|w|^2, |p|^2)
__global__ __launch_bounds__(256) void k_pair_norms(const Spin<double>* __restrict__ w,
                                                    const Spin<double>* __restrict__ p, size_t n,
                                                    double2* partials) {
  double2 acc = {0.0, 0.0};
  for (size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += size_t(gridDim.x) * blockDim.x) {
    acc.x += nrm2(w[i]);
    acc.y += nrm2(p[i]);
  }
  store_partial(acc, partials, blockIdx.x);
}

// ---- device-driven multi-shift CG: every scalar recursion runs in one-block finalisers, so a
// chunk of iterations is one graph replay and the host polls once per chunk.  An iteration is
//   w = D p with |w|^2, |p|^2;  alpha, zeta_i, alpha_i
//   r -= alpha (D^dag w + s0 p) with |r|^2;  beta, beta_i, convergence
//   x_i += alpha_i p_i, p_i = zeta_i r + beta_i p_i (one read of p_i), p = r + beta p
// so neither norm nor update has a pass of its own and D^dag w is never stored.  The smallest
// shift s0 is the one CG runs on (zeta = 1): its p_i is p.  On a small lattice the launches are
// the cost: five an iteration instead of seven, and the scalars' recursions one lane a shift
// instead of one thread for all (finalisers 4.8 -> 2.9 us with ten shifts); overlap operator at
// simplicial n=16, Lt=16, degree 21: 7.4 -> 4.9 ms.
struct MSScalars {
  double rho, bn2, alpha, beta, a_prev, b_prev, s0, tol2;
  double shift[kMaxShifts], z[kMaxShifts], zo[kMaxShifts], zn[kMaxShifts], ai[kMaxShifts], bi[kMaxShifts];
  int active[kMaxShifts];  // still iterating
  int now[kMaxShifts];     // active in the current iteration (what the update pass works on)
  int iters[kMaxShifts];
  Spin<double>* x[kMaxShifts];  // the caller's solutions (not in the captured arguments)
  int ns, it, maxiter;
  int done;  // 0 running, 1 every shift converged, 3 iteration cap, 4 breakdown
  int update;  // the update pass of the current iteration is due
};

struct ShiftPtrs {
  Spin<double>* p[kMaxShifts];
  int n, base;  // base: the smallest shift, whose p_i is p
};

struct ShiftVals {
  double s[kMaxShifts];
  Spin<double>* x[kMaxShifts];
};

// r = p = p_i = b, x_i = 0, partial |b|^2
__global__ __launch_bounds__(256) void k_ms_init(const Spin<double>* __restrict__ b, Spin<double>* r, Spin<double>* p,
                                                 ShiftPtrs S, ShiftVals X, size_t n, double2* partials) {
  double2 acc = {0.0, 0.0};
  Spin<double> z;
  z.a = {0.0, 0.0};
  z.b = {0.0, 0.0};
  for (size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += size_t(gridDim.x) * blockDim.x) {
    const Spin<double> v = b[i];
    acc.x += nrm2(v);
    r[i] = v;
    p[i] = v;
    for (int k = 0; k < S.n; k++) {
      X.x[k][i] = z;
      if (k != S.base) S.p[k][i] = v;
    }
  }
  store_partial(acc, partials, blockIdx.x);
}

struct FinMSStart {
  MSScalars* sc;
  ShiftVals X;
  int ns, maxiter;
  double s0, tol2;
  __device__ bool skip() const { return false; }
  __device__ void operator()(double2 t) const {
    const double b2 = t.x;
    sc->rho = sc->bn2 = b2;
    sc->alpha = sc->beta = 0.0;
    sc->a_prev = 1.0;
    sc->b_prev = 0.0;
    sc->s0 = s0;
    sc->tol2 = tol2;
    sc->ns = ns;
    sc->it = 0;
    sc->maxiter = maxiter;
    sc->update = 0;
    for (int i = 0; i < ns; i++) {
      sc->shift[i] = X.s[i];
      sc->x[i] = X.x[i];
      sc->z[i] = sc->zo[i] = sc->zn[i] = 1.0;
      sc->active[i] = b2 > 0 ? 1 : 0;
      sc->iters[i] = 0;
    }
    sc->done = (b2 > 0 && maxiter > 0) ? 0 : (b2 > 0 ? 3 : 1);
  }
};

// w = D p, partials of (|w|^2, |p|^2)
struct EpiMSD {
  static constexpr bool kReduce = true;
  static constexpr bool kOwnFinaliser = true;
  Spin<double>* w;
  const Spin<double>* p;
  const MSScalars* sc;
  __device__ bool skip() const { return sc->done != 0; }
  __device__ void begin() {}
  __device__ void operator()(size_t i, const Spin<double>& v, double2& acc) const {
    st(w + i, v);
    acc.x += nrm2(v);
    acc.y += nrm2(ld(p + i));
  }
};

// r -= alpha (D^dag w + s0 p), partials of |r|^2
struct EpiMSDdag {
  static constexpr bool kReduce = true;
  static constexpr bool kOwnFinaliser = true;
  Spin<double>* r;
  const Spin<double>* p;
  const MSScalars* sc;
  double alpha, as0;
  __device__ bool skip() const { return sc->done != 0; }
  __device__ void begin() {
    alpha = sc->alpha;
    as0 = sc->alpha * sc->s0;
  }
  __device__ void operator()(size_t i, const Spin<double>& q, double2& acc) const {
    Spin<double> rr = ld(r + i);
    axpy_(rr, -alpha, q);
    axpy_(rr, -as0, ld(p + i));
    st(r + i, rr);
    acc.x += nrm2(rr);
  }
};

// The iteration's two finalisers, one lane a shift (ns <= 32, in the first wave).  BETA = false:
// alpha = rho / <p, (A + s0) p>, zeta_i and alpha_i of every active shift (Jegerlehner).
// BETA = true: beta, beta_i, then the shifts' zeta history, iteration counts and convergence
// (|zeta_i| |r| <= tol |b|), the iteration cap.
template <bool BETA>
__global__ __launch_bounds__(256) void k_ms_scalars(const double2* __restrict__ partials, unsigned n, MSScalars* sc) {
  static_assert(kMaxShifts <= 64, "one lane of the first wave per shift");
  if (sc->done != 0) {  // uniform
    if (!BETA && threadIdx.x == 0) sc->update = 0;
    return;
  }
  __shared__ double2 tot_;
  const int i = threadIdx.x;
  const bool mine = i < sc->ns;
  double z = 0, zo = 0, zn = 0, sh = 0;
  int act = 0;
  if (mine) {  // in flight with the partials
    z = sc->z[i];
    zo = sc->zo[i];
    zn = sc->zn[i];
    sh = sc->shift[i];
    act = sc->active[i];
  }
  double2 s = {0.0, 0.0};
  for (unsigned k = threadIdx.x; k < n; k += blockDim.x) {
    const double2 v = partials[k];
    s.x += v.x;
    s.y += v.y;
  }
  s = block_sum2(s);
  if (threadIdx.x == 0) tot_ = s;
  __syncthreads();
  if (threadIdx.x >= 64) return;
  const double2 t = tot_;
  if constexpr (!BETA) {
    const double pq = t.x + sc->s0 * t.y, ap = sc->a_prev, bp = sc->b_prev;
    const bool ok = pq > 0.0 && pq < 1e300;
    const double alpha = sc->rho / pq;
    if (mine && ok) {
      sc->now[i] = act;
      if (act) {
        const double ds = sh - sc->s0;
        const double zx = z * zo * ap / (alpha * bp * (zo - z) + zo * ap * (1.0 + ds * alpha));
        sc->zn[i] = zx;
        sc->ai[i] = alpha * zx / z;
      }
    }
    if (i == 0) {
      sc->update = 0;
      if (ok)
        sc->alpha = alpha;
      else
        sc->done = 4;
    }
  } else {
    const double rho_new = t.x, beta = rho_new / sc->rho;
    const double stop = sqrt(sc->tol2 * sc->bn2), rn = sqrt(rho_new), alpha = sc->alpha;
    const int it = sc->it + 1, cap = sc->maxiter;
    bool on = false;
    if (mine && act) {
      sc->bi[i] = beta * (zn / z) * (zn / z);
      sc->zo[i] = z;
      sc->z[i] = zn;
      sc->iters[i] = it;
      on = !(fabs(zn) * rn <= stop);
      if (!on) sc->active[i] = 0;
    }
    const bool any = __ballot(on) != 0;
    if (i == 0) {
      sc->beta = beta;
      sc->it = it;
      sc->a_prev = alpha;
      sc->b_prev = beta;
      sc->rho = rho_new;
      sc->update = 1;
      if (!any)
        sc->done = 1;
      else if (it >= cap)
        sc->done = 3;
    }
  }
}

// x_i += alpha_i p_i, p_i = zeta_i r + beta_i p_i for the shifts active in this iteration, and
// p = r + beta p.  Runs once more after the iteration that ended the solve.  Rows of blocks
// (blockIdx.y) share the shifts out, row 0 taking the base; one row where the points alone fill
// the GPU, since every row reads r again.
__global__ __launch_bounds__(256) void k_ms_update(const Spin<double>* __restrict__ r, Spin<double>* p, ShiftPtrs S,
                                                   size_t n, const MSScalars* sc) {
  if (sc->update == 0) return;
  const double beta = sc->beta;
  for (size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += size_t(gridDim.x) * blockDim.x) {
    const Spin<double> rr = r[i];
    if (blockIdx.y == 0) {
      const Spin<double> pp = p[i];
      if (sc->now[S.base]) {  // uniform
        Spin<double> xv = sc->x[S.base][i];
        axpy_(xv, sc->ai[S.base], pp);
        sc->x[S.base][i] = xv;
      }
      Spin<double> v = rr;
      axpy_(v, beta, pp);
      p[i] = v;
    }
    for (int k = blockIdx.y; k < S.n; k += gridDim.y) {
      if (k == S.base || !sc->now[k]) continue;  // uniform
      const double a = sc->zn[k], bb = sc->bi[k];
      const Spin<double> pk = S.p[k][i];
      Spin<double> xv = sc->x[k][i];
      axpy_(xv, sc->ai[k], pk);
      sc->x[k][i] = xv;
      Spin<double> o;
      o.a = {a * rr.a.x + bb * pk.a.x, a * rr.a.y + bb * pk.a.y};
      o.b = {a * rr.b.x + bb * pk.b.x, a * rr.b.y + bb * pk.b.y};
      S.p[k][i] = o;
    }
  }
}

// |b - D^dag w - s x|^2 into *out, w = D x
struct EpiShiftResid {
  static constexpr bool kReduce = true;
  const Spin<double>* b;
  const Spin<double>* x;
  double s;
  double2* out;
  __device__ bool skip() const { return false; }
  __device__ void begin() {}
  __device__ void operator()(size_t i, const Spin<double>& q, double2& acc) const {
    Spin<double> v = ld(b + i);
    axpy_(v, -1.0, q);
    axpy_(v, -s, ld(x + i));
    acc.x += nrm2(v);
  }
  __device__ void operator()(double2 t) const { *out = t; }
};

// out = c0 in + c1 (v + sum_k a_k y_k)   (y_k in S.x, a_k in S.a)
__global__ __launch_bounds__(256) void k_combine(Spin<double>* out, const Spin<double>* __restrict__ in,
                                                 double c0, const Spin<double>* __restrict__ v,
                                                 double c1, ShiftSet S, size_t n) {
  for (size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += size_t(gridDim.x) * blockDim.x) {
    Spin<double> s = v[i];
    for (int k = 0; k < S.n; k++) axpy_(s, S.a[k], S.x[k][i]);
    Spin<double> o;
    if (in) {
      o = in[i];
      o.a = {c0 * o.a.x, c0 * o.a.y};
      o.b = {c0 * o.b.x, c0 * o.b.y};
    } else {
      o.a = {0.0, 0.0};
      o.b = {0.0, 0.0};
    }
    axpy_(o, c1, s);
    out[i] = o;
  }
}

// res = b - u - s x; partial |res|^2
__global__ __launch_bounds__(256) void k_shift_resid(const Spin<double>* __restrict__ b,
                                                     const Spin<double>* __restrict__ u,
                                                     const Spin<double>* __restrict__ x, double s,
                                                     size_t n, double2* partials) {
  double2 acc = {0.0, 0.0};
  for (size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += size_t(gridDim.x) * blockDim.x) {
    Spin<double> v = b[i];
    axpy_(v, -1.0, u[i]);
    axpy_(v, -s, x[i]);
    acc.x += nrm2(v);
  }
  store_partial(acc, partials, blockIdx.x);
}

// v = w / |w| with the given scale; partial <v_old, w> is done by Dirac::dot
__global__ __launch_bounds__(256) void k_scale(Spin<double>* v, const Spin<double>* __restrict__ w,
                                               double s, size_t n) {
  for (size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += size_t(gridDim.x) * blockDim.x) {
    Spin<double> o = w[i];
    o.a = {s * o.a.x, s * o.a.y};
    o.b = {s * o.b.x, s * o.b.y};
    v[i] = o;
  }
}

template <typename T>
T* dnew(size_t n, hipStream_t st) {
  T* p = nullptr;
  QED3_HIP(hipMallocAsync((void**)&p, std::max<size_t>(n, 1) * sizeof(T), st));
  return p;
}

struct Reducer {
  double2* partials;
  double2* out;
  double2* host;
  unsigned nb;
  hipStream_t st;
  double2 get() {
    hipLaunchKernelGGL(k_finalize<FinStore>, dim3(1), dim3(256), 0, st, partials, nb, FinStore{out});
    QED3_HIP(hipMemcpyAsync(host, out, sizeof(double2), hipMemcpyDeviceToHost, st));
    QED3_HIP(hipStreamSynchronize(st));
    return *host;
  }
};

}  // namespace

// Work memory that stays with the context from one solve to the next; more is given back at the end
// (dual n=128, Lt=64 with ten shifts takes 8 GB), which costs 0.2 to 0.6 ms a solve (dual n=64, Lt=32:
// one shift 28.4 -> 28.6 ms, ten 90.1 -> 90.7).
constexpr size_t kKeptWork = size_t(256) << 20;

std::vector<CGResult> multishift_cg(Dirac& D, const std::vector<double>& shifts,
                                    const std::vector<Spin<double>*>& x, const Spin<double>* b,
                                    const CGOptions& o) {
  const auto t0 = std::chrono::steady_clock::now();
  const int ns = int(shifts.size());
  if (ns < 1 || ns > kMaxShifts || int(x.size()) != ns)
    throw std::invalid_argument("multishift_cg: 1..32 shifts, one solution vector each");
  for (double s : shifts)
    if (!(s >= 0) || !std::isfinite(s)) throw std::invalid_argument("multishift_cg: shifts must be >= 0");
  const size_t n = D.points();
  hipStream_t st = D.stream();
  const unsigned nb = unsigned(std::min<size_t>((n + 255) / 256, 4096));
  // work memory: r, p, w, the p_i of every shift but the base (the smallest), the residual
  // norms and the scalars, each region 256-byte aligned
  const size_t f = (n * sizeof(Spin<double>) + 255) / 256 * 256;
  const size_t norms = (size_t(kMaxShifts) * sizeof(double2) + 255) / 256 * 256;
  const size_t work = (ns + 2) * f + norms + sizeof(MSScalars);
  unsigned char* base = static_cast<unsigned char*>(D.scratch(14, work));
  auto field = [&](int k) { return reinterpret_cast<Spin<double>*>(base + size_t(k) * f); };
  Spin<double>*r = field(0), *p = field(1), *w = field(2);
  double2* out = reinterpret_cast<double2*>(base + (ns + 2) * f);
  MSScalars* sc = reinterpret_cast<MSScalars*>(base + (ns + 2) * f + norms);
  // read-back: the norms, then the scalars
  unsigned char* host = static_cast<unsigned char*>(D.host_block(norms + sizeof(MSScalars)));
  const double2* hout = reinterpret_cast<const double2*>(host);
  MSScalars* hs = reinterpret_cast<MSScalars*>(host + norms);
  ShiftPtrs S{};
  ShiftVals X{};
  S.n = ns;
  S.base = int(std::min_element(shifts.begin(), shifts.end()) - shifts.begin());
  for (int i = 0, k = 3; i < ns; i++) {
    S.p[i] = i == S.base ? p : field(k++);
    X.s[i] = shifts[i];
    X.x[i] = x[i];
  }
  const GridReduce gr = D.reducer();
  hipLaunchKernelGGL(k_ms_init, dim3(nb), dim3(256), 0, st, b, r, p, S, X, n, gr.partials);
  hipLaunchKernelGGL(k_finalize<FinMSStart>, dim3(1), dim3(256), 0, st, gr.partials, nb,
                     FinMSStart{sc, X, ns, o.maxiter, shifts[S.base], o.tol * o.tol});
  QED3_HIP(hipGetLastError());
  const DiracView<double> v64 = D.view<double>();
  const int nn = D.tables().max_nn;
  const HaloView hvf = D.halo_for<double>(false), hvt = D.halo_for<double>(true);
  // the norms take one partial a block: more slices a thread where the set shape's grid has more
  // blocks than the reduction scratch
  auto fit = [&](StencilTile t) {
    const size_t nxr = size_t((D.V() + t.block - 1) / t.block + 7) / 8 * 8;
    while (t.ts < D.Lt() && nxr * size_t((D.Lt() + t.ts - 1) / t.ts) > kReduceCapacity) t.ts *= 2;
    return t;
  };
  const StencilTile tf = fit(D.tile<double>(false)), tt = fit(D.tile<double>(true));
  // rows of the update pass: up to 2,048 blocks over the points and the shifts
  const unsigned rows = std::max(1u, std::min(unsigned(ns), 2048u / nb));
  auto one_iter = [&] {
    const unsigned n1 = launch_stencil<double, false>(v64, nn, p, EpiMSD{w, p, sc}, tf, gr, st, hvf);
    hipLaunchKernelGGL(k_ms_scalars<false>, dim3(1), dim3(256), 0, st, gr.partials, n1, sc);
    const unsigned n2 = launch_stencil<double, true>(v64, nn, w, EpiMSDdag{r, p, sc, 0.0, 0.0}, tt, gr, st, hvt);
    hipLaunchKernelGGL(k_ms_scalars<true>, dim3(1), dim3(256), 0, st, gr.partials, n2, sc);
    hipLaunchKernelGGL(k_ms_update, dim3(nb, rows), dim3(256), 0, st, r, p, S, n, sc);
  };
  // chunks of iterations replayed as one kept graph (the caller's x_i are read from the
  // scalars); the kernels of iterations after the end exit at once
  const int chunk = n > (1u << 20) ? 8 : 16;
  hipGraphExec_t exec = nullptr;
  if (std::getenv("QED3_NO_GRAPH") == nullptr) {
    GraphKey key;
    key.add(v64).add(hvf).add(hvt).add(tf).add(tt).add(base).add(gr.partials).add(n).add(nn).add(ns).add(S.base);
    GraphSlot& g = D.graph_slot(3);
    if (!g.exec || g.key != key.words)
      g.capture(st, key.words, [&] {
        for (int c = 0; c < chunk; c++) one_iter();
      });
    exec = g.exec;
  }
  for (int c = 0; c <= o.maxiter / chunk + 1; c++) {
    if (exec)
      QED3_HIP(hipGraphLaunch(exec, st));
    else
      for (int k = 0; k < chunk; k++) one_iter();
    QED3_HIP(hipGetLastError());
    QED3_HIP(hipMemcpyAsync(hs, sc, sizeof(MSScalars), hipMemcpyDeviceToHost, st));
    QED3_HIP(hipStreamSynchronize(st));
    if (hs->done != 0) break;
  }
  // FP64 true residual per shift
  for (int i = 0; i < ns; i++) {
    launch_stencil<double, false>(v64, nn, x[i], EpiStore<double>{w}, tf, gr, st, hvf);
    launch_stencil<double, true>(v64, nn, w, EpiShiftResid{b, x[i], shifts[i], out + i}, tt, gr, st, hvt);
  }
  QED3_HIP(hipGetLastError());
  QED3_HIP(hipMemcpyAsync(host, out, ns * sizeof(double2), hipMemcpyDeviceToHost, st));
  QED3_HIP(hipStreamSynchronize(st));
  const double sec = std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
  std::vector<CGResult> res(ns);
  for (int i = 0; i < ns; i++) {
    res[i].iterations = hs->iters[i];
    res[i].true_resid = hs->bn2 > 0 ? std::sqrt(hout[i].x / hs->bn2) : 0.0;
    res[i].status = res[i].true_resid <= o.tol * 1.0000001 ? 0 : 3;
    res[i].seconds = sec;
  }
  if (work > kKeptWork) D.release_scratch(14);
  return res;
}

void spectral_bounds(Dirac& D, double tol, int maxiter, double* mu_min, double* mu_max) {
  const size_t n = D.points();
  hipStream_t st = D.stream();
  const unsigned nb = unsigned(std::min<size_t>((n + 255) / 256, 4096));
  Spin<double>* v = dnew<Spin<double>>(n, st);
  Spin<double>* w = dnew<Spin<double>>(n, st);
  Spin<double>* t = dnew<Spin<double>>(n, st);
  double2* partials = dnew<double2>(nb, st);
  double2* out = dnew<double2>(1, st);
  double2* host = nullptr;
  QED3_HIP(hipHostMalloc((void**)&host, sizeof(double2), hipHostMallocDefault));
  Reducer red{partials, out, host, nb, st};
  // seeded start vector with every component nonzero
  std::vector<Spin<double>> h(n);
  std::mt19937_64 g(12345);
  std::normal_distribution<double> nd;
  for (auto& s : h) s = Spin<double>{{nd(g), nd(g)}, {nd(g), nd(g)}};
  QED3_HIP(hipMemcpyAsync(v, h.data(), n * sizeof(Spin<double>), hipMemcpyHostToDevice, st));
  auto normalize = [&](Spin<double>* dst, const Spin<double>* src) {
    hipLaunchKernelGGL(k_pair_norms, dim3(nb), dim3(256), 0, st, src, src, n, partials);
    const double nn = red.get().x;
    hipLaunchKernelGGL(k_scale, dim3(nb), dim3(256), 0, st, dst, src, 1.0 / std::sqrt(nn), n);
  };
  auto rayleigh = [&](const Spin<double>* a, const Spin<double>* c) {
    double re, im;
    D.dot(a, c, &re, &im);
    return re;
  };
  normalize(v, v);
  double mu = 0, mu_old = -1;
  for (int it = 0; it < maxiter; it++) {
    D.apply<double>(false, t, v, false);
    D.apply<double>(true, w, t, false);
    mu = rayleigh(v, w);
    normalize(v, w);
    if (std::abs(mu - mu_old) <= tol * std::abs(mu)) break;
    mu_old = mu;
  }
  *mu_max = mu;
  QED3_HIP(hipMemcpyAsync(v, h.data(), n * sizeof(Spin<double>), hipMemcpyHostToDevice, st));
  normalize(v, v);
  CGOptions o;
  o.tol = std::min(1e-12, tol * 1e-2);
  o.mixed = false;
  double nu = 0, nu_old = -1;
  for (int it = 0; it < maxiter; it++) {
    const CGResult r = cg_solve(D, w, v, o);
    if (r.status != 0) throw std::runtime_error("spectral_bounds: inner CG did not converge");
    nu = rayleigh(v, w);  // <v, A^{-1} v> -> 1/mu_min
    normalize(v, w);
    if (std::abs(nu - nu_old) <= tol * std::abs(nu)) break;
    nu_old = nu;
  }
  *mu_min = 1.0 / nu;
  for (void* ptr : {(void*)v, (void*)w, (void*)t, (void*)partials, (void*)out}) (void)hipFreeAsync(ptr, st);
  QED3_HIP(hipStreamSynchronize(st));
  (void)hipHostFree(host);
}

Overlap::Overlap(Dirac& D, int n, double lambda_min, double lambda_max, double tol)
    : D_(D), z_(n, lambda_min / lambda_max), lmax_(lambda_max), tol_(tol) {
  if (!(lambda_min > 0 && lambda_max > lambda_min)) throw std::invalid_argument("need 0 < lambda_min < lambda_max");
  if (z_.size - 1 > kMaxShifts) throw std::invalid_argument("Zolotarev degree too large (at most 65)");
  const size_t bytes = D.points() * sizeof(Spin<double>);
  sol_.resize(z_.size - 1);
  for (auto& p : sol_) QED3_HIP(hipMalloc(&p, bytes));
  QED3_HIP(hipMalloc(&y_, bytes));
  QED3_HIP(hipMalloc(&t_, bytes));
}

Overlap::~Overlap() {
  for (auto* p : sol_) (void)hipFree(p);
  for (auto* p : ysol_) (void)hipFree(p);
  (void)hipFree(y_);
  (void)hipFree(t_);
}

void Overlap::apply(bool dag, Spin<double>* out, const Spin<double>* in) {
  const size_t n = D_.points();
  hipStream_t st = D_.stream();
  const unsigned nb = unsigned(std::min<size_t>((n + 255) / 256, 4096));
  // (D^dag D / lmax^2 + sigma_m)^{-1} v = lmax^2 (D^dag D + lmax^2 sigma_m)^{-1} v
  std::vector<double> sh = z_.shifts();
  for (double& s : sh) s *= lmax_ * lmax_;
  const Spin<double>* rhs = in;
  if (dag) {  // y = D^dag psi / lmax
    D_.apply<double>(true, t_, in, false);
    hipLaunchKernelGGL(k_scale, dim3(nb), dim3(256), 0, st, y_, t_, 1.0 / lmax_, n);
    rhs = y_;
  }
  CGOptions o;
  o.tol = tol_;
  o.mixed = false;
  const std::vector<CGResult> r = multishift_cg(D_, sh, sol_, rhs, o);
  iters_ = r.empty() ? 0 : r[0].iterations;
  for (const auto& ri : r)
    if (ri.status != 0) throw std::runtime_error("overlap: shifted solve did not converge");
  ShiftSet S;
  S.n = int(sol_.size());
  for (int m = 0; m < S.n; m++) {
    S.x[m] = sol_[m];
    S.a[m] = z_.A[m + 1] * lmax_ * lmax_;
  }
  if (!dag) {
    // t = psi + sum A_m Z_m ; out = psi + (C/lmax) D t
    hipLaunchKernelGGL(k_combine, dim3(nb), dim3(256), 0, st, t_, static_cast<const Spin<double>*>(nullptr),
                       0.0, in, 1.0, S, n);
    D_.apply<double>(false, y_, t_, false);
    ShiftSet none;
    none.n = 0;
    hipLaunchKernelGGL(k_combine, dim3(nb), dim3(256), 0, st, out, in, 1.0, y_, z_.C / lmax_, none, n);
  } else {
    // out = psi + C (y + sum A_m Y_m)
    hipLaunchKernelGGL(k_combine, dim3(nb), dim3(256), 0, st, out, in, 1.0, y_, z_.C, S, n);
  }
  QED3_HIP(hipGetLastError());
  QED3_HIP(hipStreamSynchronize(st));
}

void Overlap::force(const Spin<double>* eta, double* fs, double* ft) {
  const size_t n = D_.points();
  hipStream_t st = D_.stream();
  const unsigned nb = unsigned(std::min<size_t>((n + 255) / 256, 4096));
  const int ns = int(sol_.size());
  if (ysol_.empty()) {
    ysol_.resize(ns);
    for (auto& p : ysol_) QED3_HIP(hipMalloc(&p, n * sizeof(Spin<double>)));
  }
  // R_m v = lmax^2 (D^dag D + lmax^2 sigma_m)^{-1} v: the solver's x_m are Z_m / lmax^2, Y_m / lmax^2
  std::vector<double> sh = z_.shifts();
  for (double& s : sh) s *= lmax_ * lmax_;
  D_.apply<double>(true, t_, eta, false);
  hipLaunchKernelGGL(k_scale, dim3(nb), dim3(256), 0, st, y_, t_, 1.0 / lmax_, n);  // D^dag eta / lmax
  CGOptions o;
  o.tol = tol_;
  o.mixed = false;
  auto check = [](const std::vector<CGResult>& r) {
    for (const auto& ri : r)
      if (ri.status != 0) throw std::runtime_error("overlap force: shifted solve did not converge");
  };
  check(multishift_cg(D_, sh, sol_, eta, o));
  check(multishift_cg(D_, sh, ysol_, y_, o));
  const double l2 = lmax_ * lmax_, c0 = -2.0 * z_.C / lmax_;
  // Z_0 = eta + sum_m A_m lmax^2 x_m into t_, then f = c0 Re <eta, dD Z_0>
  ShiftSet S;
  S.n = ns;
  for (int m = 0; m < ns; m++) {
    S.x[m] = sol_[m];
    S.a[m] = z_.A[m + 1] * l2;
  }
  hipLaunchKernelGGL(k_combine, dim3(nb), dim3(256), 0, st, t_, static_cast<const Spin<double>*>(nullptr), 0.0,
                     eta, 1.0, S, n);
  D_.force_bilinear(eta, t_, nullptr, nullptr, c0, true, fs, ft);
  // pole terms: c0 (-A_m) lmax^3 [Re <D xZ_m, dD xY_m> + Re <D xY_m, dD xZ_m>]
  for (int m = 0; m < ns; m++) {
    D_.apply<double>(false, t_, sol_[m], false);
    D_.apply<double>(false, y_, ysol_[m], false);
    D_.force_bilinear(t_, ysol_[m], y_, sol_[m], -c0 * z_.A[m + 1] * l2 * lmax_, false, fs, ft);
  }
  QED3_HIP(hipGetLastError());
  QED3_HIP(hipStreamSynchronize(st));
}

void Overlap::apply_dhd(Spin<double>* out, const Spin<double>* in, Spin<double>* tmp) {
  const size_t n = D_.points();
  const unsigned nb = unsigned(std::min<size_t>((n + 255) / 256, 4096));
  apply(false, out, in);
  apply(true, tmp, in);
  ShiftSet none;
  none.n = 0;
  hipLaunchKernelGGL(k_combine, dim3(nb), dim3(256), 0, D_.stream(), out, out, 1.0, tmp, 1.0, none, n);
  QED3_HIP(hipGetLastError());
}

CGResult Overlap::solve_dhd(Spin<double>* x, const Spin<double>* b, double tol, int maxiter) {
  if (!(tol > 0) || maxiter < 0) throw std::invalid_argument("solve_dhd: tol > 0, maxiter >= 0");
  const auto t0 = std::chrono::steady_clock::now();
  const size_t n = D_.points();
  hipStream_t st = D_.stream();
  const unsigned nb = unsigned(std::min<size_t>((n + 255) / 256, 4096));
  Spin<double>* r = dnew<Spin<double>>(n, st);
  Spin<double>* p = dnew<Spin<double>>(n, st);
  Spin<double>* q = dnew<Spin<double>>(n, st);
  Spin<double>* tmp = dnew<Spin<double>>(n, st);
  double2* partials = dnew<double2>(nb, st);
  double2* out = dnew<double2>(1, st);
  double2* host = nullptr;
  QED3_HIP(hipHostMalloc((void**)&host, sizeof(double2), hipHostMallocDefault));
  Reducer red{partials, out, host, nb, st};
  const size_t bytes = n * sizeof(Spin<double>);
  ShiftSet none;
  none.n = 0;
  QED3_HIP(hipMemsetAsync(x, 0, bytes, st));
  QED3_HIP(hipMemcpyAsync(r, b, bytes, hipMemcpyDeviceToDevice, st));
  QED3_HIP(hipMemcpyAsync(p, b, bytes, hipMemcpyDeviceToDevice, st));
  hipLaunchKernelGGL(k_pair_norms, dim3(nb), dim3(256), 0, st, b, b, n, partials);
  const double bn2 = red.get().x;
  double rr = bn2;
  CGResult res;
  int it = 0;
  while (bn2 > 0 && rr > tol * tol * bn2 && it < maxiter) {
    apply_dhd(q, p, tmp);
    double pq, im;
    D_.dot(p, q, &pq, &im);
    if (!(pq > 0) || !std::isfinite(pq)) {
      res.status = 4;
      break;
    }
    const double alpha = rr / pq;
    hipLaunchKernelGGL(k_combine, dim3(nb), dim3(256), 0, st, x, x, 1.0, p, alpha, none, n);
    hipLaunchKernelGGL(k_combine, dim3(nb), dim3(256), 0, st, r, r, 1.0, q, -alpha, none, n);
    hipLaunchKernelGGL(k_pair_norms, dim3(nb), dim3(256), 0, st, r, r, n, partials);
    const double rr_new = red.get().x;
    hipLaunchKernelGGL(k_combine, dim3(nb), dim3(256), 0, st, p, r, 1.0, p, rr_new / rr, none, n);
    rr = rr_new;
    it++;
  }
  // true residual |b - A x| / |b|
  apply_dhd(q, x, tmp);
  hipLaunchKernelGGL(k_shift_resid, dim3(nb), dim3(256), 0, st, b, q, x, 0.0, n, partials);
  const double tr = red.get().x;
  res.iterations = it;
  res.true_resid = bn2 > 0 ? std::sqrt(tr / bn2) : 0.0;
  if (res.status == 0 && !(rr <= tol * tol * bn2)) res.status = 3;
  for (void* ptr : {(void*)r, (void*)p, (void*)q, (void*)tmp, (void*)partials, (void*)out}) (void)hipFreeAsync(ptr, st);
  QED3_HIP(hipStreamSynchronize(st));
  (void)hipHostFree(host);
  res.seconds = std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
  return res;
}

void Overlap::refresh_bounds(double tol, int maxiter) {
  double mu_min = 0, mu_max = 0;
  spectral_bounds(D_, tol, maxiter, &mu_min, &mu_max);
  const double lmin = std::sqrt((1.0 - 100.0 * tol) * mu_min), lmax = std::sqrt((1.0 + 100.0 * tol) * mu_max);
  if (!(lmin > 0 && lmax > lmin)) throw std::runtime_error("overlap: bad spectral bounds");
  z_.set(lmin / lmax);
  lmax_ = lmax;
}

}  // namespace qed3
