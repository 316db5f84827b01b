// Device side of the time-exact Horner preconditioner (horner.hpp): one layer
// g_out = T^{-1}(c v + S_th g_in) (or its adjoint form) per launch.
//
// Under T the spin-up row's recurrence runs forward in time and the spin-down row's backward
// (the other way round under T^dagger).  Two forms:
//   FP32 fields in any gauge (the checked apply and the training gradient): a transport pass
//     y = c v + S_th g over all points, then the two rows' recurrences; with many sites, both
//     together, a thread a column;
//   binary16 fields in the temporal gauge (the solver): the parallel-in-time layer below.
#pragma once
#include <type_traits>

#include "horner.hpp"
#include "stencil.hpp"

namespace qed3 {
namespace hk {

// binary16 complex arithmetic on (re, im) pairs: x y and acc + x y, in packed FMAs
__device__ __forceinline__ half2_t cmul16(half2_t x, half2_t y) {
  const half2_t ys = {-y.y, y.x};
  return __builtin_elementwise_fma(x.yy, ys, x.xx * y);
}
__device__ __forceinline__ half2_t cfma16(half2_t x, half2_t y, half2_t acc) {
  const half2_t ys = {-y.y, y.x};
  return __builtin_elementwise_fma(x.yy, ys, __builtin_elementwise_fma(x.xx, y, acc));
}

// element idx of base through a 32-bit byte offset (idx * sizeof(T) < 2^32), so that the
// access takes a uniform base from scalar registers and a 32-bit vector offset
template <class T>
__device__ __forceinline__ const T& at32(const T* base, unsigned idx) {
  return *reinterpret_cast<const T*>(reinterpret_cast<const char*>(base) + idx * unsigned(sizeof(T)));
}
template <class T>
__device__ __forceinline__ T* ptr32(T* base, unsigned idx) {
  return reinterpret_cast<T*>(reinterpret_cast<char*>(base) + idx * unsigned(sizeof(T)));
}
template <class T>
__device__ __forceinline__ const T* cptr32(const T* base, unsigned idx) {
  return reinterpret_cast<const T*>(reinterpret_cast<const char*>(base) + idx * unsigned(sizeof(T)));
}

// Loads through a buffer resource (base, nbytes): byte offset voff (per thread) + soff (a
// scalar register: uniform across the wave); loads beyond nbytes return zeros.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t buf_rsrc(const void* base, unsigned nbytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), short(0), int(nbytes), 0x00020000);
}
__device__ __forceinline__ SpinH bload_h(const void* base, unsigned nbytes, unsigned voff, unsigned soff) {
  return __builtin_bit_cast(SpinH, __builtin_amdgcn_raw_buffer_load_b64(buf_rsrc(base, nbytes), voff, soff, 0));
}
__device__ __forceinline__ unsigned bload_w(const void* base, unsigned nbytes, unsigned voff, unsigned soff) {
  return __builtin_bit_cast(unsigned, __builtin_amdgcn_raw_buffer_load_b32(buf_rsrc(base, nbytes), voff, soff, 0));
}
// e^{i theta} of a 10-bit angle (theta = 2 pi a / 1024) as a binary16 pair; the hardware sine
// and cosine take revolutions
__device__ __forceinline__ half2_t angle_pair10(unsigned a) {
  const float rev = float(a) * (1.0f / 1024.0f);
  return half2_t{(_Float16)__builtin_amdgcn_cosf(rev), (_Float16)__builtin_amdgcn_sinf(rev)};
}

// component a of a point as FP32 complex
__device__ __forceinline__ float2 comp(const Spin<float>& v, int a) { return a == 0 ? v.a : v.b; }
__device__ __forceinline__ float2 comp(const SpinH& v, int a) {
  return a == 0 ? float2{float(v.v.x), float(v.v.y)} : float2{float(v.v.z), float(v.v.w)};
}
__device__ __forceinline__ half2_t comp16(const SpinH& v, int a) {
  return a == 0 ? half2_t{v.v.x, v.v.y} : half2_t{v.v.z, v.v.w};
}
__device__ __forceinline__ Spin<float> to_f(const Spin<float>& v) { return v; }
__device__ __forceinline__ Spin<float> to_f(const SpinH& v) { return from_half(v); }
// a point from its two components, stored (binary16 stores are non-temporal: written once,
// read by the next kernel)
__device__ __forceinline__ void put(Spin<float>* p, float2 c0, float2 c1) {
  Spin<float> v;
  v.a = c0;
  v.b = c1;
  *p = v;
}
__device__ __forceinline__ void put(SpinH* p, float2 c0, float2 c1) {
  Spin<float> v;
  v.a = c0;
  v.b = c1;
  sth_nt(p, to_half(v));
}
// the value a load of what put() stored would return
__device__ __forceinline__ Spin<float> stored(const Spin<float>*, float2 c0, float2 c1) {
  Spin<float> v;
  v.a = c0;
  v.b = c1;
  return v;
}
__device__ __forceinline__ Spin<float> stored(const SpinH*, float2 c0, float2 c1) {
  Spin<float> v;
  v.a = c0;
  v.b = c1;
  return from_half(to_half(v));
}

// Injection sources: the point i as stored.
template <typename F>
struct SrcF {
  const F* p;
  __device__ SrcF bind() const { return *this; }
  __device__ F raw(size_t i) const { return p[i]; }
  __device__ F bat(unsigned nbytes, unsigned voff, unsigned soff) const { return bload_h(p, nbytes, voff, soff); }
  __device__ float2 scale(float2 c) const { return c; }
};
// binary16 field whose stored values still owe the factor *f (parallel-in-time layer only):
// the layer folds it into its injection coefficient
struct SrcFS {
  const SpinH* p;
  const double* f;
  struct Bound {
    const SpinH* p;
    float f;
    __device__ SpinH bat(unsigned nbytes, unsigned voff, unsigned soff) const { return bload_h(p, nbytes, voff, soff); }
    __device__ float2 scale(float2 c) const { return {c.x * f, c.y * f}; }
  };
  __device__ Bound bind() const { return {p, float(*f)}; }
};

// Injection with a side field (parallel-in-time layer only): the layer also accumulates
// |v|^2 and Re<o, v> over its points (v the injection as stored, o the side field) into the
// reduction of its epilogue, which must have kReduce.
struct SrcDots {
  static constexpr bool kDots = true;
  const SpinH* p;
  const SpinH* o;
  __device__ SrcDots bind() const { return *this; }
  __device__ SpinH raw(size_t i) const { return p[i]; }
  __device__ SpinH bat(unsigned nbytes, unsigned voff, unsigned soff) const { return bload_h(p, nbytes, voff, soff); }
  __device__ SpinH bside(unsigned nbytes, unsigned voff, unsigned soff) const {
    return bload_h(o, nbytes, voff, soff);
  }
  __device__ float2 scale(float2 c) const { return c; }
};
template <class S, class = void>
struct SrcHasDots : std::false_type {};
template <class S>
struct SrcHasDots<S, std::void_t<decltype(S::kDots)>> : std::bool_constant<S::kDots> {};

struct EpiNone {
  static constexpr bool kReduce = false;
  __device__ bool skip() const { return false; }
  __device__ void operator()(size_t, const Spin<float>&, double2&) const {}
  __device__ void operator()(double2) const {}
};

// ---- layers on FP32 fields -------------------------------------------------------------
// The transport pass: y(s, x) = c_j v - sum_j u_j (m_same g_a + m_flip g_abar)(nb_j) for both spin
// rows, a thread per site and tile of ts slices (the hop rows stay in registers).  It carries the
// layer's gathers and has no order in time, so every point can be in flight: walking a site's
// column with one thread, transports and recurrences together (the form before), left the GPU at
// 80 blocks on dual n=32, Lt=32 and took 48 us a layer; this pass and the recurrences' take 9 + 9.
// The roundings are spelled out (and contraction off), so that the FP32 results do not depend on
// the code around them.
constexpr int kTransportSlices = 4;
__device__ __forceinline__ float2 cmul_coef(float2 h, float2 g) {  // h g
#pragma clang fp contract(off)
  return {__builtin_fmaf(g.x, h.x, -(g.y * h.y)), __builtin_fmaf(g.y, h.x, g.x * h.y)};
}
__device__ __forceinline__ float2 cmul_phase(float2 u, float2 c) {  // u c
#pragma clang fp contract(off)
  return {__builtin_fmaf(u.x, c.x, -(u.y * c.y)), __builtin_fmaf(u.x, c.y, u.y * c.x)};
}
// sum_j u_j (m_same g_a + m_flip g_abar)(nb_j), lk < 0: the link is stored the other way round
template <int NS, class G>
__device__ __forceinline__ float2 transport_row(const float4 (&hr)[NS], const float2 (&u)[NS], const int (&lk)[NS], const G& g,
                                                int a) {
#pragma clang fp contract(off)
  float2 t = {0.f, 0.f};
#pragma unroll
  for (int j = 0; j < NS; j++) {
    float2 uj = u[j];
    if (lk[j] < 0) uj.y = -uj.y;
    const Spin<float> gj = g(j);
    const float2 cm = cadd<float>(cmul_coef({hr[j].x, hr[j].y}, comp(gj, a)),
                                  cmul_coef({hr[j].z, hr[j].w}, comp(gj, 1 - a)));
    t = cadd<float>(t, cmul_phase(uj, cm));
  }
  return t;
}
template <int NS, bool ADJ>
__global__ __launch_bounds__(256) void k_horner_transport(HornerView hv, DiracView<float> d,
                                                          const Spin<float>* __restrict__ v,
                                                          const Spin<float>* __restrict__ gin, Spin<float>* __restrict__ y,
                                                          float2 cj, TileMap tm) {
#pragma clang fp contract(off)
  int xr, st;
  tile_of(tm, blockIdx.x, xr, st);
  const int V = hv.V;
  const int x = xr < tm.nxr ? xr * int(blockDim.x) + int(threadIdx.x) : V;
  if (x >= V) return;
  constexpr int rF = ADJ ? 1 : 0, rB = 1 - rF;
  int nb[NS], lk[NS];
  float4 hrF[NS], hrB[NS];
  const size_t mF = size_t((ADJ ? 2 : 0) + rF) * NS * V, mB = size_t((ADJ ? 2 : 0) + rB) * NS * V;
#pragma unroll
  for (int j = 0; j < NS; j++) {
    nb[j] = d.nbr[size_t(j) * V + x];
    lk[j] = d.lnk[size_t(j) * V + x];
    hrF[j] = hv.hrow[mF + size_t(j) * V + x];
    hrB[j] = hv.hrow[mB + size_t(j) * V + x];
  }
  const int s1 = min(hv.Lt, (st + 1) * kTransportSlices);
  for (int s = st * kTransportSlices; s < s1; s++) {
    const size_t sV = size_t(s) * V;
    const float2* uS = d.uS + size_t(s) * d.E;
    float2 u[NS];
    Spin<float> g[NS];
#pragma unroll
    for (int j = 0; j < NS; j++) {
      u[j] = uS[lk[j] >= 0 ? lk[j] : ~lk[j]];
      g[j] = gin[sV + nb[j]];
    }
    auto near = [&](int j) { return g[j]; };
    const Spin<float> vv = v[sV + x];
    float2 yF = cmul_phase(cj, comp(vv, rF)), yB = cmul_phase(cj, comp(vv, rB));
    const float2 tF = transport_row<NS>(hrF, u, lk, near, rF), tB = transport_row<NS>(hrB, u, lk, near, rB);
    yF.x -= tF.x;
    yF.y -= tF.y;
    yB.x -= tB.x;
    yB.y -= tB.y;
    if constexpr (rF == 0)
      put(y + sV + x, yF, yB);
    else
      put(y + sV + x, yB, yF);
  }
}

// One row's recurrence, state = (y + kappa_t u^t state) / c_x, walked forward (FWD) or backward in
// time.  A link's phase times v, conjugated for the forward walk:
template <bool FWD>
__device__ __forceinline__ float2 recur_hop(float2 u, float2 v) {
#pragma clang fp contract(off)
  if constexpr (FWD)
    return {__builtin_fmaf(u.y, v.y, u.x * v.x), __builtin_fmaf(u.x, v.y, -(u.y * v.x))};
  else
    return {__builtin_fmaf(u.x, v.x, -(u.y * v.y)), __builtin_fmaf(v.x, u.y, v.y * u.x)};
}
// S holds the time wrap (the link from Lt-1 to 0, which T leaves out): a recurrence starts from
// bc kappa_t w g(the far end of its walk), w the wrap link's phase
template <bool FWD>
__device__ __forceinline__ float2 recur_wrap(float bc, float kt, float2 w, float2 g) {
#pragma clang fp contract(off)
  float2 t = recur_hop<FWD>(w, g);
  if constexpr (FWD) t.x = __builtin_fmaf(w.x, g.x, w.y * g.y);
  return {bc * kt * t.x, bc * kt * t.y};
}
// y of a first layer (no input field)
__device__ __forceinline__ float2 first_y(float2 cj, float2 v) {
#pragma clang fp contract(off)
  return {__builtin_fmaf(cj.x, v.x, -(cj.y * v.y)), __builtin_fmaf(cj.y, v.x, cj.x * v.y)};
}
// the state after one slice; at a walk's start (wrap) st is the wrap term, already weighted (0 in a
// first layer), else the state before, across the link of phase u
template <bool FWD, bool FIRST>
__device__ __forceinline__ float2 recur_step(float2 y, float2 u, float2 st, bool wrap, float kt, float invc) {
#pragma clang fp contract(off)
  if (!wrap) {
    const float2 t = recur_hop<FWD>(u, st);
    if constexpr (FWD && FIRST) {
      y = {__builtin_fmaf(kt, t.x, y.x), __builtin_fmaf(kt, t.y, y.y)};
    } else {
      const float2 w = {kt * t.x, kt * t.y};
      y = {y.x + w.x, y.y + w.y};
    }
  } else {
    y = {y.x + st.x, y.y + st.y};
  }
  return {invc * y.x, invc * y.y};
}

// The recurrences, one thread per site and spin row, each value written over its y.  The chain is
// arithmetic only: the loads of the next kRecurDepth slices are issued while this group's are worked
// through.  FIRST (no input field): y = c_j v formed here, without a transport pass or a wrap term.
constexpr int kRecurDepth = 8;
template <bool FWD, bool FIRST>
__device__ __forceinline__ void horner_recur_walk(const HornerView& hv, const DiracView<float>& d, const Spin<float>* in,
                                                  const Spin<float>* __restrict__ gin, Spin<float>* out, float2 cj,
                                                  int x, int row) {
  const int V = hv.V, Lt = hv.Lt;
  const float invc = hv.invc[x], kt = hv.kt[x];
  auto at = [&](int k) { return size_t(FWD ? k : Lt - 1 - k) * V + x; };
  // component `row` of the point, as two floats
  auto half = [&](const Spin<float>* p, size_t i) { return reinterpret_cast<const float2*>(p)[2 * i + row]; };
  float2 st = {0.f, 0.f};
  if constexpr (!FIRST) st = recur_wrap<FWD>(d.bc, kt, d.uT[size_t(Lt - 1) * V + x], half(gin, at(Lt - 1)));
  struct Group {
    float2 y[kRecurDepth], u[kRecurDepth];
  };
  auto load = [&](int k0, Group& G) {
#pragma unroll
    for (int j = 0; j < kRecurDepth; j++) {
      const int k = min(k0 + j, Lt - 1);
      G.y[j] = half(in, at(k));
      G.u[j] = d.uT[at(FWD ? max(k - 1, 0) : k)];  // the link the walk crosses to reach slice at(k)
    }
  };
  Group cur, nxt;
  load(0, cur);
  for (int k0 = 0; k0 < Lt; k0 += kRecurDepth) {
    if (k0 + kRecurDepth < Lt) load(k0 + kRecurDepth, nxt);
#pragma unroll
    for (int j = 0; j < kRecurDepth; j++) {
      const int k = k0 + j;
      if (k < Lt) {
        const float2 y = FIRST ? first_y(cj, cur.y[j]) : cur.y[j];
        st = recur_step<FWD, FIRST>(y, cur.u[j], st, k == 0, kt, invc);
        reinterpret_cast<float2*>(out)[2 * at(k) + row] = st;
      }
    }
    cur = nxt;
  }
}

template <bool ADJ, bool FIRST>
__global__ __launch_bounds__(256) void k_horner_recur(HornerView hv, DiracView<float> d, const Spin<float>* in,
                                                      const Spin<float>* __restrict__ gin, Spin<float>* out,
                                                      float2 cj) {
  const int nxb = (hv.V + 255) / 256;
  const int row = int(blockIdx.x) / nxb;
  const int x = (int(blockIdx.x) - row * nxb) * 256 + int(threadIdx.x);
  if (x >= hv.V) return;
  if (row == (ADJ ? 1 : 0))  // uniform: the row that runs forward in time
    horner_recur_walk<true, FIRST>(hv, d, in, gin, out, cj, x, row);
  else
    horner_recur_walk<false, FIRST>(hv, d, in, gin, out, cj, x, row);
}

// The layer with one thread a column: a block owns a range of sites.  Pass 1, forward in time: per
// slice the block stages g_in of its range and halo in LDS (two tiles in turn, one barrier a slice),
// every thread forms both rows' transports, steps the forward row and stores its state beside the
// other row's y.  Pass 2, backward in time: every thread reads its own column back and steps the
// other row.  Both passes move whole points, 120 B a point on three slots; the transport pass and the
// recurrences by rows move 150 (half points, both rows' lines fetched twice), but over all points at
// once.  So this form where the columns fill the GPU; the roundings are the same.
template <int NS, bool ADJ, bool FIRST>
__global__ __launch_bounds__(256) void k_horner_column(HornerView hv, DiracView<float> d, HaloView halo,
                                                       const Spin<float>* __restrict__ v,
                                                       const Spin<float>* __restrict__ gin,
                                                       Spin<float>* __restrict__ gout, float2 cj, TileMap tm) {
#pragma clang fp contract(off)
  extern __shared__ unsigned char column_raw[];
  float4* tile = reinterpret_cast<float4*>(column_raw);  // [2][R + hmax], points
  int xr, st_;
  tile_of(tm, blockIdx.x, xr, st_);
  if (xr >= tm.nxr) return;  // uniform
  const int V = hv.V, Lt = hv.Lt, R = blockDim.x;
  const int x = xr * R + int(threadIdx.x);
  const bool act = x < V;
  constexpr int rF = ADJ ? 1 : 0, rB = 1 - rF;
  const int h0 = FIRST ? 0 : halo.halo_off[xr], nh = FIRST ? 0 : halo.halo_off[xr + 1] - h0;
  const int hid0 = int(threadIdx.x) < nh ? halo.halo[h0 + threadIdx.x] : -1;
  const int hid1 = int(threadIdx.x) + R < nh ? halo.halo[h0 + threadIdx.x + R] : -1;
  int nb[NS], lk[NS];
  float4 hrF[NS], hrB[NS];
  float invc = 0.f, kt = 0.f;
  float2 stF = {0.f, 0.f}, stB = {0.f, 0.f};
  if (act) {
    invc = hv.invc[x];
    kt = hv.kt[x];
    if constexpr (!FIRST) {
      const size_t mF = size_t((ADJ ? 2 : 0) + rF) * NS * V, mB = size_t((ADJ ? 2 : 0) + rB) * NS * V;
#pragma unroll
      for (int j = 0; j < NS; j++) {
        nb[j] = halo.nbl[size_t(j) * V + x];
        lk[j] = d.lnk[size_t(j) * V + x];
        hrF[j] = hv.hrow[mF + size_t(j) * V + x];
        hrB[j] = hv.hrow[mB + size_t(j) * V + x];
      }
      const size_t end = size_t(Lt - 1) * V + x;
      const float2 w = d.uT[end];
      stF = recur_wrap<true>(d.bc, kt, w, comp(gin[end], rF));
      stB = recur_wrap<false>(d.bc, kt, w, comp(gin[x], rB));
    }
  }
  struct Loads {
    Spin<float> v, gc, gh0, gh1;
    float2 u[NS], ut;  // ut: the temporal link s-1 -> s
  };
  auto load = [&](int s, Loads& L) {
    const size_t sV = size_t(s) * V;
    if (act) {
      L.v = v[sV + x];
      if (s > 0) L.ut = d.uT[sV - V + x];
      if constexpr (!FIRST) {
        const float2* uS = d.uS + size_t(s) * d.E;
#pragma unroll
        for (int j = 0; j < NS; j++) L.u[j] = uS[lk[j] >= 0 ? lk[j] : ~lk[j]];
        L.gc = gin[sV + x];
      }
    }
    if constexpr (!FIRST) {
      if (hid0 >= 0) L.gh0 = gin[sV + hid0];
      if (hid1 >= 0) L.gh1 = gin[sV + hid1];
    }
  };
  Loads cur, nxt;
  load(0, cur);
  for (int s = 0; s < Lt; s++) {
    if (s + 1 < Lt) load(s + 1, nxt);  // a slice ahead: in flight during this slice's work
    float4* tb = tile + (s & 1) * (R + halo.hmax);
    if constexpr (!FIRST) {
      auto quad = [](const Spin<float>& p) { return float4{p.a.x, p.a.y, p.b.x, p.b.y}; };
      if (act) tb[threadIdx.x] = quad(cur.gc);
      if (hid0 >= 0) tb[R + threadIdx.x] = quad(cur.gh0);
      if (hid1 >= 0) tb[2 * R + threadIdx.x] = quad(cur.gh1);
      for (int k = int(threadIdx.x) + 2 * R; k < nh; k += R) tb[R + k] = quad(gin[size_t(s) * V + halo.halo[h0 + k]]);
      __syncthreads();
    }
    if (act) {
      float2 yF, yB;
      if constexpr (FIRST) {
        yF = first_y(cj, comp(cur.v, rF));
        yB = first_y(cj, comp(cur.v, rB));
      } else {
        auto near = [&](int j) {
          const float4 p = tb[nb[j]];
          return Spin<float>{{p.x, p.y}, {p.z, p.w}};
        };
        yF = cmul_phase(cj, comp(cur.v, rF));
        yB = cmul_phase(cj, comp(cur.v, rB));
        const float2 tF = transport_row<NS>(hrF, cur.u, lk, near, rF), tB = transport_row<NS>(hrB, cur.u, lk, near, rB);
        yF.x -= tF.x;
        yF.y -= tF.y;
        yB.x -= tB.x;
        yB.y -= tB.y;
      }
      stF = recur_step<true, FIRST>(yF, cur.ut, stF, s == 0, kt, invc);
      if constexpr (rF == 0)
        put(gout + size_t(s) * V + x, stF, yB);
      else
        put(gout + size_t(s) * V + x, yB, stF);
    }
    cur = nxt;
  }
  if (!act) return;
  Spin<float> t = gout[size_t(Lt - 1) * V + x], tn = t;
  float2 u{};
  for (int s = Lt - 1; s >= 0; s--) {
    const size_t i = size_t(s) * V + x;
    if (s > 0) tn = gout[i - V];
    if (s < Lt - 1) u = d.uT[i];  // the link s -> s+1
    const float2 gF = comp(t, rF);
    stB = recur_step<false, FIRST>(comp(t, rB), u, stB, s == Lt - 1, kt, invc);
    if constexpr (rF == 0)
      put(gout + i, gF, stB);
    else
      put(gout + i, stB, gF);
    t = tn;
  }
}

// One layer of K (ADJ: of K^dagger) on FP32 fields: gout = T^{-1}(c_j v + S_th gin).  By columns from
// kColumnSites sites on, where a thread a column is more than a wave per SIMD; halo: of ranges of 256
// sites, needed there (horner_halo).  Application of four layers by rows / by columns in us, sites in
// thousands: dual n=60, Lt=64 (72) 567 / 669; simplicial n=90, Lt=64 (81) 744 / 757; dual n=64, Lt=32
// (82) 281 / 298; dual n=66, Lt=20 (87) 207 / 188; simplicial n=96, Lt=32 (92) 417 / 371; dual n=68,
// Lt=64 (92) 702 / 744; simplicial n=128, Lt=64 (164) 1539 / 1172; dual n=128, Lt=64 (328) 2664 / 2175,
// a training step there 6312 / 5353.
constexpr int kColumnSites = 88000;
inline HaloView horner_halo(Dirac& D) { return D.V() >= kColumnSites ? D.halo(256) : HaloView{}; }
template <bool ADJ, bool FIRST>
inline void launch_horner_layer(const HornerView& hv, const DiracView<float>& tables, const HaloView& halo,
                                const Spin<float>* v, const Spin<float>* gin, Spin<float>* gout, float2 cj,
                                hipStream_t st) {
  TileMap tm;
  tm.nxr = (hv.V + 255) / 256;
  tm.nxr_pad = (tm.nxr + 7) / 8 * 8;
  tm.remap = 1;
  if (hv.V >= kColumnSites) {
    tm.nst = 1;
    const dim3 grid{unsigned(tm.nxr_pad)};
    const size_t smem = FIRST ? 0 : size_t(2) * (256 + halo.hmax) * sizeof(Spin<float>);
    if (hv.nslot == 6)
      hipLaunchKernelGGL((k_horner_column<6, ADJ, FIRST>), grid, dim3(256), smem, st, hv, tables, halo, v, gin, gout, cj,
                         tm);
    else
      hipLaunchKernelGGL((k_horner_column<3, ADJ, FIRST>), grid, dim3(256), smem, st, hv, tables, halo, v, gin, gout, cj,
                         tm);
    return;
  }
  if constexpr (!FIRST) {
    tm.nst = (hv.Lt + kTransportSlices - 1) / kTransportSlices;
    const dim3 grid(unsigned(tm.nxr_pad) * unsigned(tm.nst));
    if (hv.nslot == 6)
      hipLaunchKernelGGL((k_horner_transport<6, ADJ>), grid, dim3(256), 0, st, hv, tables, v, gin, gout, cj, tm);
    else
      hipLaunchKernelGGL((k_horner_transport<3, ADJ>), grid, dim3(256), 0, st, hv, tables, v, gin, gout, cj, tm);
  }
  hipLaunchKernelGGL((k_horner_recur<ADJ, FIRST>), dim3(2 * unsigned((hv.V + 255) / 256)), dim3(256), 0, st, hv, tables,
                     FIRST ? v : gout, gin, gout, cj);
}

// ---- parallel-in-time layer (the solver's path: binary16 fields, temporal gauge) ------
// In the temporal gauge every temporal link inside a column is 1, so both recurrences have
// the constant real coefficient a = kappa_t / c_x:
//   forward  st(s) = a st(s-1) + y(s) / c_x,   backward  st(s) = a st(s+1) + y(s) / c_x,
// with the wrap term (bc kappa_t w g_in at the column's far end) added to y at the first
// (forward) or last (backward) slice.  A linear recurrence splits over time chunks: lane k
// of a site owns slices [kT, kT + T) and runs both recurrences over its chunk from a zero
// start, holding its chunk in registers; the chunks' end values are exchanged in LDS and
// every lane adds carry a^m to its values (m the distance from its chunk's start, for the
// backward row from its end), with carry_k = E_{k-1} + a^T carry_{k-1} (forward) and
// carry_k = E_{k+1} + a^{len_{k+1}} carry_{k+1} (backward), E the lanes' end values.  So a
// layer reads its input and injection once and writes its output once, and a site's time
// column runs on C = ceil(Lt / T) threads (C * S <= kTcBlock, S sites per block; the threads
// of a lane are consecutive, so a wave reads and writes consecutive sites of one slice).  Per
// step the block stages the C slices its lanes are at, for its S sites and their halo (halo
// tables of ranges of S sites).  The spatial link phases come per site as the view's uSite10:
// the slots' angles (orientation applied) at 10 bits, three to a 32-bit word, so a thread
// reads one word per slice on the trivalent lattice (a wave's loads consecutive).  The rounding
// (at most pi/1024 rad) is of the order of the binary16 arithmetic's and only enters the
// preconditioner.  With six slots the kernel is bound by VALU issue, so each block looks the
// 1,024 binary16 (cos, sin) pairs up in a 4 KB LDS table it fills once (a sine and a cosine,
// quarter rate, and their conversions per slot and slice before), and the transports are chains
// of packed FMAs into the rows' accumulators, 12 a slot instead of 16 packed operations: 25-29%
// fewer vector instructions, learned solves of simplicial n=64, Lt=32: 2604 -> 2496 us, n=48,
// Lt=45: 2530 -> 2392, n=128, Lt=64: 13300 -> 12780; with three slots 1-3% less up to n=64, and no
// change at n=128, Lt=64, where the layer moves 5.4 TB/s.
constexpr int kTcDepth = 2;    // steps whose loads are in flight ahead of the one computed
// most threads per block (S sites x C lanes) with T slices per lane: the short chunks leave the
// registers for twice the lanes
constexpr int tc_block(int T) { return T == 16 ? 256 : 512; }

// LDS written by threads of a wave and read back by other threads of the same wave: the wave
// executes its LDS instructions in order, so only the compiler must keep them in order
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// FUSE (K^dagger's last layer only): the kernel then also applies the first layer of K to
// the output it has just stored, from the same registers: gout2 = T^{-1}(cj2 gout) with
// gout as stored (binary16), which saves K's first launch and its read of gout.
// WS (S = the wave size): a lane is one wave, which stages its tile (its sites and their
// whole halo) and alone reads it, so the per-step staging needs no block barrier.
template <int NS, bool ADJ, bool FIRST, int T, class Src, class Epi, bool FUSE = false, bool UL = false,
          bool H2 = false, bool WS = false>
__global__ __launch_bounds__(tc_block(T), (NS == 3 ? 4 : 2)) void k_horner_layer_tc(HornerView hv, DiracView<float, phasepair_t> d,
                                                         HaloView halo, Src src, const SpinH* __restrict__ gin,
                                                         SpinH* __restrict__ gout, float2 cj, TileMap tm, Epi epi,
                                                         GridReduce gr, int C, SpinH* __restrict__ gout2,
                                                         float2 cj2) {
  static_assert(!FUSE || ADJ, "K's first layer fuses into a layer of K^dagger");
  static_assert(!WS || UL, "wave-synchronous staging needs one wave per lane");
  constexpr bool kDots = SrcHasDots<Src>::value;
  static_assert(!kDots || Epi::kReduce, "the injection's products need the epilogue's reduction");
  if (epi.skip()) return;  // uniform
  extern __shared__ float4 hk_tile_raw[];
  const int S = int(blockDim.x) / C;
  // a wave: consecutive sites of one lane (UL: S a multiple of the wave size, so the lane, its
  // slices and their offsets are wave-uniform and live in scalar registers)
  int lane = int(threadIdx.x) / S;
  if constexpr (UL) lane = __builtin_amdgcn_readfirstlane(lane);
  const int sl = int(threadIdx.x) - lane * S;
  SpinH* tile = reinterpret_cast<SpinH*>(hk_tile_raw);         // [2][C][S + hmax]
  const int row = S + halo.hmax;
  float2* carry = reinterpret_cast<float2*>(tile + (FIRST ? 0 : 2 * C * row));  // [2][blockDim]
  HopRow16* hqs = reinterpret_cast<HopRow16*>(carry + 2 * blockDim.x);  // [S][2 rows][NS], the sites' hop rows
  half2_t* phase_tab = reinterpret_cast<half2_t*>(hqs + (FIRST ? 0 : S * 2 * NS));  // [1024] e^{i theta}
  int xr, st_;
  tile_of(tm, blockIdx.x, xr, st_);
  (void)st_;
  const int V = hv.V, Lt = hv.Lt;
  const bool live = xr < tm.nxr;
  const int x0 = xr * S;
  const int x = live ? x0 + sl : V;
  const bool act = x < V;
  const unsigned xc = act ? unsigned(x) : 0u;  // idle threads load site 0 and discard it
  const int s0 = lane * T;
  const int lenU = max(0, min(T, Lt - s0));  // slices of this lane
  const int len = act ? lenU : 0;            // ... that this thread stores
  // slices this thread computes: UL computes them on idle threads too (discarded), so that the
  // step loop branches on the wave-uniform count
  const int lenC = UL ? lenU : len;
  constexpr int rF = ADJ ? 1 : 0, rB = 1 - rF;
  // halo of this block's range: lane c stages slice cT + j of it, its S threads share it
  const int h0 = (live && !FIRST) ? halo.halo_off[xr] : 0;
  const int nh = (live && !FIRST) ? halo.halo_off[xr + 1] - h0 : 0;
  const int hid0 = (sl < nh) ? halo.halo[h0 + sl] : -1;
  const int hid1 = (sl + S < nh) ? halo.halo[h0 + sl + S] : -1;
  const unsigned hc0 = hid0 >= 0 ? unsigned(hid0) : xc, hc1 = hid1 >= 0 ? unsigned(hid1) : xc;
  // neighbour slots in the tile
  int nb[NS];
#pragma unroll
  for (int j = 0; j < NS; j++) nb[j] = 0;
  float invc = 0.f, kt = 0.f;
  if (act) {
    if constexpr (!FIRST) {
#pragma unroll
      for (int j = 0; j < NS; j++) nb[j] = halo.nbl[j * V + x];
      // the site's hop rows go to LDS once (lane 0), read per step by all its lanes
      if (lane == 0) {
        const size_t mF = size_t((ADJ ? 2 : 0) + rF) * NS * V, mB = size_t((ADJ ? 2 : 0) + rB) * NS * V;
#pragma unroll
        for (int j = 0; j < NS; j++) {
          hqs[(sl * 2 + 0) * NS + j] = hv.hrow16[mF + size_t(j) * V + x];
          hqs[(sl * 2 + 1) * NS + j] = hv.hrow16[mB + size_t(j) * V + x];
        }
      }
    }
    invc = hv.invc[x];
    kt = hv.kt[x];
  }
  const HopRow16* hqF = hqs + (sl * 2 + 0) * NS;
  const HopRow16* hqB = hqs + (sl * 2 + 1) * NS;
  const float a = invc * kt;
  const auto in = src.bind();
  const float2 cjs = in.scale(cj);  // the injection's coefficient with what its values owe
  // the wrap terms, weighted: the forward row's on the first slice of lane 0, the backward
  // row's on the last slice of the last lane
  float2 wF = {0.f, 0.f}, wB = {0.f, 0.f};
  if constexpr (!FIRST) {
    if (act && s0 == 0) {
      const float2 w = ldu(d.uPoly + x);
      const float2 g = comp(gin[size_t(Lt - 1) * V + x], rF);
      const float2 t = cmul<float>({w.x, -w.y}, g);
      wF = {d.bc * kt * t.x, d.bc * kt * t.y};
    }
    if (act && len > 0 && s0 + len == Lt) {
      const float2 w = ldu(d.uPoly + x);
      const float2 g = comp(gin[x], rB);
      const float2 t = cmul<float>(w, g);
      wB = {d.bc * kt * t.x, d.bc * kt * t.y};
    }
  }
  constexpr int NW = (NS + 2) / 3;  // packed angle words per site and slice
  struct Loads {
    SpinH v, gc, gh0, gh1;
    SpinH o;  // kDots: the side field
    unsigned u[NW];  // the slots' link angles, packed
  };
  // slice s0 + j of this lane (own point, links, kDots: the side field) and slice c T + j of
  // the halo share.  Every thread issues the same loads at every step (lanes past the column's
  // end re-read its last slice, idle threads site 0; the values are not used), so that the
  // loads of the next kTcDepth steps stay in flight while this one computes; 32-bit offsets
  // (checked at launch).
  // buffer loads: the slice's byte offset in the scalar offset when it is wave-uniform (UL),
  // the thread's site or link in the vector offset
  const unsigned fbytes = unsigned(V) * unsigned(Lt) * unsigned(sizeof(SpinH));
  constexpr unsigned usz = sizeof(unsigned);
  const unsigned ubytes = unsigned(V) * unsigned(NW) * unsigned(Lt) * usz;
  const unsigned vx = xc * unsigned(sizeof(SpinH)), vh0 = hc0 * unsigned(sizeof(SpinH)),
                 vh1 = hc1 * unsigned(sizeof(SpinH)), vxu = xc * usz;
  auto load = [&](int j, Loads& Ld) {
    const unsigned s = unsigned(min(s0 + j, Lt - 1));
    const unsigned oG = s * unsigned(V) * unsigned(sizeof(SpinH));  // the slice's field offset
    const unsigned oU = s * unsigned(NW * V) * usz;  // ... and phases
    const unsigned sG = UL ? oG : 0u, sU = UL ? oU : 0u, vG = UL ? 0u : oG, vU = UL ? 0u : oU;
    Ld.v = in.bat(fbytes, vG + vx, sG);
    if constexpr (kDots) Ld.o = in.bside(fbytes, vG + vx, sG);
    if constexpr (!FIRST) {
#pragma unroll
      for (int w = 0; w < NW; w++) Ld.u[w] = bload_w(d.uSite10, ubytes, vU + vxu, sU + unsigned(w * V) * usz);
      Ld.gc = bload_h(gin, fbytes, vG + vx, sG);
      Ld.gh0 = bload_h(gin, fbytes, vG + vh0, sG);
      if constexpr (H2) Ld.gh1 = bload_h(gin, fbytes, vG + vh1, sG);
    }
  };
  // both rows' transports sum_q u_q (s_q g_r + f_q g_(1-r)) of the staged neighbours
  auto transport = [&](const Loads& Ld, const SpinH* tb, float2& tF, float2& tB) {
    half2_t aF = {(_Float16)0.f, (_Float16)0.f}, aB = aF;
#pragma unroll
    for (int q = 0; q < NS; q++) {
      const half2_t u = phase_tab[(Ld.u[q / 3] >> (10 * (q % 3))) & 1023u];
      const SpinH g = tb[nb[q]];
      const half2_t gF = comp16(g, rF), gB = comp16(g, rB);
      aF = cfma16(u, cfma16(hqF[q].f, gB, cmul16(hqF[q].s, gF)), aF);
      aB = cfma16(u, cfma16(hqB[q].f, gF, cmul16(hqB[q].s, gB)), aB);
    }
    tF = {float(aF.x), float(aF.y)};
    tB = {float(aB.x), float(aB.y)};
  };
  if constexpr (!FIRST)
    for (unsigned k = threadIdx.x; k < 1024u; k += blockDim.x) phase_tab[k] = angle_pair10(k);
  float2 zF[T];   // forward row: the chunk's states (FP32)
  half2_t zB[T];  // backward row: its recurrence inputs, then its states (binary16)
  float2 prevF = {0.f, 0.f};
  float2 dots = {0.f, 0.f};  // kDots: this thread's |v|^2 and Re<o, v> over its chunk
  constexpr int NB = kTcDepth + 1;  // load buffers: this step's and the next kTcDepth steps'
  Loads lb[NB];
#pragma unroll
  for (int j = 0; j < kTcDepth && j < T; j++) load(j, lb[j]);
  if constexpr (WS && !FIRST) __syncthreads();  // the hop rows lane 0 staged, before any lane reads them
#pragma unroll
  for (int j = 0; j < T; j++) {
    if (j + kTcDepth < T) load(j + kTcDepth, lb[(j + kTcDepth) % NB]);
    const Loads& cur = lb[j % NB];
    SpinH* tb = tile + ((j & 1) * C + lane) * row;
    if constexpr (!FIRST) {
      if (j < lenC) tb[sl] = cur.gc;
      if (live && s0 + j < Lt) {
        if (hid0 >= 0) tb[S + sl] = cur.gh0;
        if constexpr (H2) {  // a halo longer than the block's range
          if (hid1 >= 0) tb[2 * S + sl] = cur.gh1;
          for (int q = sl + 2 * S; q < nh; q += S) tb[S + q] = gin[size_t(s0 + j) * V + halo.halo[h0 + q]];
        }
      }
      if constexpr (WS)
        wave_sync();
      else
        __syncthreads();
    }
    if (j < lenC) {
      if constexpr (kDots) {
        if (act) {
          const Spin<float> v = from_half(cur.v), o = from_half(cur.o);
          dots.x += v.a.x * v.a.x + v.a.y * v.a.y + v.b.x * v.b.x + v.b.y * v.b.y;
          dots.y += o.a.x * v.a.x + o.a.y * v.a.y + o.b.x * v.b.x + o.b.y * v.b.y;
        }
      }
      float2 yF = cmul<float>(cjs, comp(cur.v, rF)), yB = cmul<float>(cjs, comp(cur.v, rB));
      if constexpr (!FIRST) {
        float2 tF, tB;
        transport(cur, tb, tF, tB);
        yF.x -= tF.x;
        yF.y -= tF.y;
        yB.x -= tB.x;
        yB.y -= tB.y;
      }
      if (j == 0) {
        yF.x += wF.x;
        yF.y += wF.y;
      }
      if (j == lenC - 1) {
        yB.x += wB.x;
        yB.y += wB.y;
      }
      prevF = {a * prevF.x + invc * yF.x, a * prevF.y + invc * yF.y};
      zF[j] = prevF;
      zB[j] = half2_t{(_Float16)yB.x, (_Float16)yB.y};
    }
  }
  // local backward recurrence over the chunk held in registers
  float2 nextB = {0.f, 0.f};
#pragma unroll
  for (int j = T - 1; j >= 0; j--) {
    if (j < lenC) {
      nextB = {a * nextB.x + invc * float(zB[j].x), a * nextB.y + invc * float(zB[j].y)};
      zB[j] = half2_t{(_Float16)nextB.x, (_Float16)nextB.y};
    }
  }
  // carries across the lanes of each site
  float aT = 1.f;
#pragma unroll
  for (int j = 0; j < T; j++) aT *= a;
  carry[threadIdx.x] = prevF;                       // forward end value (0 for an empty lane)
  carry[blockDim.x + threadIdx.x] = nextB;          // backward end value
  __syncthreads();
  float2 cF = {0.f, 0.f}, cB = {0.f, 0.f};
  for (int c = 0; c < lane; c++) {
    const float2 e = carry[c * S + sl];
    cF = {aT * cF.x + e.x, aT * cF.y + e.y};
  }
  for (int c = C - 1; c > lane; c--) {
    const int lc = max(0, min(T, Lt - c * T));
    float ac = 1.f;
    for (int q = 0; q < lc; q++) ac *= a;
    const float2 e = carry[blockDim.x + c * S + sl];
    cB = {ac * cB.x + e.x, ac * cB.y + e.y};
  }
  // add the carries and store
  double2 acc = {double(dots.x), double(dots.y)};
  float pF = a;
#pragma unroll
  for (int j = 0; j < T; j++) {
    if (j < lenC) {
      zF[j].x += pF * cF.x;
      zF[j].y += pF * cF.y;
      pF *= a;
    }
  }
  // backward row: add a^(len - j) carry while storing, last slice first
  float pB = a;
#pragma unroll
  for (int j = T - 1; j >= 0; j--) {
    if (j < lenC) {
      const float2 b = {float(zB[j].x) + pB * cB.x, float(zB[j].y) + pB * cB.y};
      pB *= a;
      if (act) {
        const unsigned i = unsigned(s0 + j) * unsigned(V) + unsigned(x);
        if constexpr (rF == 0) {
          put(ptr32(gout, i), zF[j], b);
          epi(size_t(i), stored(gout, zF[j], b), acc);
        } else {
          put(ptr32(gout, i), b, zF[j]);
          epi(size_t(i), stored(gout, b, zF[j]), acc);
        }
      }
      if constexpr (FUSE) zB[j] = half2_t{(_Float16)b.x, (_Float16)b.y};  // row rB as stored
    }
  }
  if constexpr (Epi::kReduce) store_partial(acc, gr.partials, blockIdx.x);
  if constexpr (FUSE) {
    // K's first layer on the stored output (rows: ADJ's forward row rF = 1 is K's backward
    // row, ADJ's rB = 0 K's forward row): forward over cj2 out_0, backward over cj2 out_1
    float2 p0 = {0.f, 0.f};
#pragma unroll
    for (int j = 0; j < T; j++) {
      if (j < lenC) {
        const float2 h0 = {float(zB[j].x), float(zB[j].y)};
        const float2 h1 = {float((_Float16)zF[j].x), float((_Float16)zF[j].y)};
        const float2 y0 = cmul<float>(cj2, h0), y1 = cmul<float>(cj2, h1);
        p0 = {a * p0.x + invc * y0.x, a * p0.y + invc * y0.y};
        zF[j] = p0;
        zB[j] = half2_t{(_Float16)y1.x, (_Float16)y1.y};
      }
    }
    float2 p1 = {0.f, 0.f};
#pragma unroll
    for (int j = T - 1; j >= 0; j--) {
      if (j < lenC) {
        p1 = {a * p1.x + invc * float(zB[j].x), a * p1.y + invc * float(zB[j].y)};
        zB[j] = half2_t{(_Float16)p1.x, (_Float16)p1.y};
      }
    }
    __syncthreads();  // every lane has read the first exchange
    carry[threadIdx.x] = p0;
    carry[blockDim.x + threadIdx.x] = p1;
    __syncthreads();
    float2 c0 = {0.f, 0.f}, c1 = {0.f, 0.f};
    for (int c = 0; c < lane; c++) {
      const float2 e = carry[c * S + sl];
      c0 = {aT * c0.x + e.x, aT * c0.y + e.y};
    }
    for (int c = C - 1; c > lane; c--) {
      const int lc = max(0, min(T, Lt - c * T));
      float ac = 1.f;
      for (int q = 0; q < lc; q++) ac *= a;
      const float2 e = carry[blockDim.x + c * S + sl];
      c1 = {ac * c1.x + e.x, ac * c1.y + e.y};
    }
    float q0 = a;
#pragma unroll
    for (int j = 0; j < T; j++) {
      if (j < lenC) {
        zF[j].x += q0 * c0.x;
        zF[j].y += q0 * c0.y;
        q0 *= a;
      }
    }
    float q1 = a;
#pragma unroll
    for (int j = T - 1; j >= 0; j--) {
      if (j < lenC) {
        const float2 b = {float(zB[j].x) + q1 * c1.x, float(zB[j].y) + q1 * c1.y};
        q1 *= a;
        if (act) put(ptr32(gout2, unsigned(s0 + j) * unsigned(V) + unsigned(x)), zF[j], b);
      }
    }
  }
}

// Shape of the parallel-in-time layer: T slices per lane, C = ceil(Lt / T) lanes per site, S
// sites per block.  Up to 64 slices a lane is one wave (S = 64), which stages its own tile
// without block barriers; longer columns split a block of 256 threads over more lanes (C a
// power of two, at most 64) and synchronise per step.
constexpr long kTcSimds = 1024;
struct TcShape {
  int T, C, S;
};
inline int tc_sites(int Lt) {
  if (Lt <= 64) return 64;
  int c = 8;
  while (c * 16 < Lt) c <<= 1;
  if (c > 64) throw std::invalid_argument("time extent too long for the parallel-in-time layer");
  return 256 / c;
}
// A lane's steps are a serial chain of loads, so the fewer waves there are the shorter its
// chunk should be; the longer one spends less on carries and on the wrap terms once the GPU is
// full.  Learned solves, T = 4 / 8 / 16 in us (waves with T = 8): simplicial n=16, Lt=16: 1001 /
// 1135 / 1484 (82); dual n=24, Lt=20: 1347 / 1436 / 1755 (540); simplicial n=64, Lt=32: 2742 /
// 2605 / 2871 (2,564); dual n=64, Lt=32: 4064 / 3808 / 3957 (5,120); simplicial n=128, Lt=64:
// - / 13242 / 13102 (20,488).  So: 4 while chunks of 8 would leave some of the 1,024 SIMDs
// without a wave, 16 from ten waves a SIMD on; and 16 where more lanes' tiles would not fit in
// LDS (halos of several times the range, as of randomly numbered tables).
constexpr size_t kTcLds = 64 * 1024;
inline size_t tc_smem(int C, int S, int nslot, bool first, int hmax) {
  return (first ? 0 : size_t(2) * C * (S + hmax) * sizeof(SpinH) + size_t(S) * 2 * nslot * sizeof(HopRow16) +
                          1024 * sizeof(half2_t)) +
         size_t(2) * C * S * sizeof(float2);
}
inline TcShape tc_shape(int V, int Lt, int nslot, bool first, int hmax) {
  const int S = tc_sites(Lt);
  if (S != 64) return {16, 256 / S, S};
  auto lanes = [&](int T) { return (Lt + T - 1) / T; };
  auto waves = [&](int T) { return long((V + S - 1) / S) * lanes(T); };
  int T = waves(16) > 10 * kTcSimds ? 16 : (waves(8) <= kTcSimds && lanes(4) * S <= tc_block(4) ? 4 : 8);
  if (tc_smem(lanes(T), S, nslot, first, hmax) > kTcLds) T = 16;
  return {T, lanes(T), S};
}

// gout2 != nullptr (ADJ only): also K's first layer with coefficient cj2 into gout2 (FUSE).
template <bool ADJ, bool FIRST, class Src, class Epi>
void launch_horner_layer_tc(const HornerView& hv, const DiracView<float, phasepair_t>& tables,
                                   const HaloView& halo, const Src& src, const SpinH* gin, SpinH* gout, float2 cj,
                                   const Epi& epi, GridReduce gr, hipStream_t st, const hipEvent_t* bracket = nullptr,
                                   SpinH* gout2 = nullptr, float2 cj2 = {0.f, 0.f}) {
  if (gout2 && !ADJ) throw std::logic_error("only a K^dagger layer carries K's first layer");
  if (gout2 && (gout2 == gout || gout2 == gin)) throw std::logic_error("fused output aliases an operand");
  const TcShape sh = tc_shape(hv.V, hv.Lt, hv.nslot, FIRST, FIRST ? 0 : halo.hmax);
  const int C = sh.C, S = sh.S;
  if (!tables.uPoly || !tables.uSite10)
    throw std::logic_error("parallel-in-time layer needs the temporal gauge");
  if (!FIRST && !halo.nbl) throw std::logic_error("parallel-in-time layer launched without halo tables");
  TileMap tm;
  tm.nxr = (hv.V + S - 1) / S;
  tm.nxr_pad = (tm.nxr + 7) / 8 * 8;
  tm.nst = 1;
  tm.remap = 1;
  const unsigned nblk = unsigned(tm.nxr_pad);
  if (Epi::kReduce && nblk > kReduceCapacity) throw std::invalid_argument("layer grid exceeds the reduction scratch");
  const size_t smem = tc_smem(C, S, hv.nslot, FIRST, FIRST ? 0 : halo.hmax);
  if (smem > kTcLds) throw std::invalid_argument("parallel-in-time layer: halo too large for LDS");
  if (size_t(hv.V) * size_t(hv.Lt) * sizeof(SpinH) > 0xffffffffull ||
      size_t(hv.V) * size_t((hv.nslot + 2) / 3) * size_t(hv.Lt) * sizeof(unsigned) > 0xffffffffull)
    throw std::invalid_argument("parallel-in-time layer: fields beyond 32-bit offsets");
  if (bracket) QED3_HIP(hipEventRecord(bracket[0], st));
  auto go = [&](auto fuse, auto t, auto ws, auto h2) {
    constexpr bool F = decltype(fuse)::value && ADJ;
    constexpr bool U = decltype(ws)::value;
    constexpr bool H = decltype(h2)::value && !FIRST;
    constexpr bool W = U && !FIRST;
    constexpr int T = decltype(t)::value;
    if (hv.nslot == 6)
      hipLaunchKernelGGL((k_horner_layer_tc<6, ADJ, FIRST, T, Src, Epi, F, U, H, W>), dim3(nblk), dim3(C * S), smem, st,
                         hv, tables, halo, src, gin, gout, cj, tm, epi, gr, C, gout2, cj2);
    else
      hipLaunchKernelGGL((k_horner_layer_tc<3, ADJ, FIRST, T, Src, Epi, F, U, H, W>), dim3(nblk), dim3(C * S), smem, st,
                         hv, tables, halo, src, gin, gout, cj, tm, epi, gr, C, gout2, cj2);
  };
  // wave-uniform and wave-synchronous where a lane is one wave (S = 64); the second halo load
  // only where some block's halo is longer than its range
  const bool h2 = !FIRST && halo.hmax > S;
  auto go2 = [&](auto fuse, auto t, auto ws) {
    if (h2)
      go(fuse, t, ws, std::true_type{});
    else
      go(fuse, t, ws, std::false_type{});
  };
  auto go3 = [&](auto fuse) {
    if (S != 64)
      go2(fuse, std::integral_constant<int, 16>{}, std::false_type{});
    else if (sh.T == 16)
      go2(fuse, std::integral_constant<int, 16>{}, std::true_type{});
    else if (sh.T == 8)
      go2(fuse, std::integral_constant<int, 8>{}, std::true_type{});
    else
      go2(fuse, std::integral_constant<int, 4>{}, std::true_type{});
  };
  if (gout2)
    go3(std::true_type{});
  else
    go3(std::false_type{});
  if (bracket) QED3_HIP(hipEventRecord(bracket[1], st));
  if constexpr (Epi::kReduce)
    hipLaunchKernelGGL((k_finalize<Epi>), dim3(1), dim3(256), 0, st, gr.partials, nblk, epi);
}

}  // namespace hk
}  // namespace qed3
