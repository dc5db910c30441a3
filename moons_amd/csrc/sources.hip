// sources.hip -- the explicit source terms of a time step, a launch (or two) a
// term group instead of one for every interpolation, derivative and product.
//
// What bounds them: as sequences of whole-field passes the sources of an MHD
// step were about 180 launches, each 4-6 us at 64^3 for its start alone and
// 10-13 us at 128^3, where each reads and writes one to three fields of 17 MB
// through temporaries.  Here a thread forms one output element from the fields
// themselves: the temporaries stay in registers, neighbours come from the
// caches, and HBM carries each input and output about once.
//
// Every element keeps the operand order and the roundings of the passes it
// replaces (interpO2_SF, del, multiply, add in the reference's order,
// code/handwritten/ops/ops_advect.f90:71-127,186-200, ops_interp.f90,
// code/handwritten/stencils/stencils.f90), so the results are the same bits.
#include <type_traits>

#include "common.hpp"

namespace moons {

constexpr int kSrc = 256;

// A field: values and shape.
struct FView {
  double *p;
  int s[3];
};
static FView fview(const moons_field_s *f) {
  FView v{nullptr, {1, 1, 1}};
  if (f) v = FView{f->d, {f->s[0], f->s[1], f->s[2]}};
  return v;
}
struct FView3 {
  FView f[3];
};
static FView3 fview3(moons_field_s *const f[3]) { return FView3{{fview(f[0]), fview(f[1]), fview(f[2])}}; }

template <int E>
__device__ __forceinline__ size_t fstride(const FView &f) {
  return E == 0 ? (size_t)1 : (E == 1 ? (size_t)f.s[0] : (size_t)f.s[0] * f.s[1]);
}
struct Pos {
  int q[3];
};
template <int E>
__device__ __forceinline__ Pos at(Pos a, int o) {
  a.q[E] = o;
  return a;
}
__device__ __forceinline__ size_t off(const FView &f, const Pos &a) {
  return (size_t)a.q[0] + (size_t)f.s[0] * ((size_t)a.q[1] + (size_t)f.s[1] * a.q[2]);
}
// The thread's element of a field (memory order, XCD-contiguous blocks, so that
// the neighbouring planes it reads share an L2); false beyond the field.
__device__ __forceinline__ bool my_element(const int (&s)[3], Pos &a, size_t &o) {
  const unsigned t = (unsigned)xcd_remap((int)blockIdx.x, (int)gridDim.x) * kSrc + threadIdx.x;
  const unsigned n01 = (unsigned)s[0] * s[1];
  if (t >= n01 * s[2]) return false;
  a.q[2] = t / n01;
  const unsigned r = t - a.q[2] * n01;
  a.q[1] = r / s[0];
  a.q[0] = r - a.q[1] * s[0];
  o = t;
  return true;
}

// Whether an element lies on a ghost plane of a face in mask (bit f).
__device__ __forceinline__ bool on_ghost(int mask, const int (&s)[3], const Pos &a) {
  bool g = false;
#pragma unroll
  for (int d = 0; d < 3; ++d)
    g = g || (((mask >> (2 * d)) & 1) && a.q[d] == 0) || (((mask >> (2 * d + 1)) & 1) && a.q[d] == s[d] - 1);
  return g;
}

// interpO2_SF, C -> N, at node o of direction E: theta weights inside,
// extrapolated at the two end nodes.  val(m): the input at cell m of the pencil
// of sC cells.  Without branches, so that loads of several terms overlap.
template <typename V>
__device__ __forceinline__ double c2n(int o, int sC, const DirCoefDev &c, V val) {
  const int p = min(max(o, 1), sC - 1);
  const double hi = val(p), lo = val(p - 1);
  const double n = hi * c.theta_D[p - 1] + lo * c.theta_U[p - 1];
  if (o == 0) return 2.0 * lo - n;
  if (o == sC) return 2.0 * hi - n;
  return n;
}

// A staggered derivative's two products at output o (C2N: CC -> N, else N -> CC);
// sin: entries of the input pencil.  written: whether the pass writes o.
template <bool C2N>
struct Stag {
  int i;
  bool written, zero_end;
  double D, U;
  __device__ __forceinline__ Stag(int o, int sin, const DirCoefDev &c) {
    const int nd = C2N ? sin + 1 : sin - 1;
    zero_end = o == 0 || o == nd - 1;
    i = min(max(C2N ? o - 1 : o, 0), sin - 2);
    written = C2N ? !zero_end : true;
    D = (C2N ? c.cc2n_D : c.n2cc_D)[i];
    U = (C2N ? c.cc2n_U : c.n2cc_U)[i];
  }
  __device__ __forceinline__ double set(double f0, double f1) const {
    const double x0 = f0 * D, x1 = f1 * U;
    return written ? x0 + x1 : 0.0;
  }
  __device__ __forceinline__ double add(double acc, double f0, double f1) const {
    const double x0 = f0 * D, x1 = f1 * U, cur = zero_end ? 0.0 : acc;
    return written ? cur + x0 + x1 : cur;
  }
  __device__ __forceinline__ double sub(double acc, double f0, double f1) const {
    const double x0 = f0 * D, x1 = f1 * U, cur = zero_end ? 0.0 : acc;
    return written ? cur - (x0 + x1) : cur;
  }
};

// A collocated derivative along a pencil of s entries at o (N: on the nodes,
// else on the cell centres): assigned (first) or added to acc; 0 at the ends.
template <bool N, typename V>
__device__ __forceinline__ double del_col(bool first, double acc, int o, int s, const double *L, const double *D,
                                          const double *U, V val) {
  const bool end = o == 0 || o == s - 1;
  const int q = min(max(o - 1, 0), s - 3);
  const int b = min(max(N ? (o == 1 ? 2 : (o == s - 2 ? s - 3 : o)) : o, 1), s - 2);
  const double m = val(b - 1), c = val(b), p = val(b + 1), l = L[q], d = D[q], u = U[q];
  double r;
  if (!N && o == 1) {
    const double t1 = 0.5 * (m + c) * l * 1.0, t2 = m * l * 0.0;
    r = first ? t1 + t2 + c * d + p * u : acc + t1 + t2 + c * d + p * u;
  } else if (!N && o == s - 2) {
    const double t3 = 0.5 * (c + p) * u * 1.0, t4 = p * u * 0.0;
    r = first ? m * l + c * d + t3 + t4 : acc + m * l + c * d + t3 + t4;
  } else {
    r = first ? m * l + c * d + p * u : acc + m * l + c * d + p * u;
  }
  return end ? 0.0 : r;
}

// ------------------------------------------------- faces -> edges (U_E, U_E x B)
// The two off-diagonal interpolants of an edge direction D: components l < h
// other than D, the face component interpolated along the third direction.
struct EdgeArgs {
  FView3 in;          // face components
  double *out[3][2];  // the interpolants of l and h (null: not kept)
  const double *U[3][2]; // U_l, U_h on the edges (CROSS)
  FView3 E;           // the edges' shapes; values: U x B (CROSS)
};

template <int D, bool CROSS>
__device__ __forceinline__ void edge_block(const EdgeArgs &A, const MeshDev &M) {
  constexpr int L = D == 0 ? 1 : 0, H = D == 2 ? 1 : 2;
  Pos a;
  size_t o;
  if (!my_element(A.E.f[D].s, a, o)) return;
  const FView &fl = A.in.f[L], &fh = A.in.f[H];
  double ul = 0.0, uh = 0.0;
  if (CROSS) {
    ul = A.U[D][0][o];
    uh = A.U[D][1][o];
  }
  const double *__restrict__ pl = fl.p;
  const double *__restrict__ ph = fh.p;
  const double bl = c2n(a.q[H], fl.s[H], M.c[H], [&](int m) { return pl[off(fl, at<H>(a, m))]; });
  const double bh = c2n(a.q[L], fh.s[L], M.c[L], [&](int m) { return ph[off(fh, at<L>(a, m))]; });
  if (A.out[D][0]) {
    A.out[D][0][o] = bl;
    A.out[D][1][o] = bh;
  }
  if (CROSS) {
    const double v = ul * bh - uh * bl;
    A.E.f[D].p[o] = D == 1 ? -v : v;
  }
}
// Six interpolations and three cross products in one launch, 5.7 us at
// 50 x 39 x 45 cells; with the curl's launch (six passes, now 4.0 us) advect_B
// takes 9.7 us where the 15 passes took 59.
template <bool CROSS>
__global__ void __launch_bounds__(kSrc) k_edge(EdgeArgs A, MeshDev M) {
  if (blockIdx.y == 0) edge_block<0, CROSS>(A, M);
  else if (blockIdx.y == 1) edge_block<1, CROSS>(A, M);
  else edge_block<2, CROSS>(A, M);
}

// ---------------------------------------------------------------- curl
// Component D of curl_SF at element a: the derivative of component D+2 along
// D+1 less that of component D+1 along D+2.  FACES: edges -> faces (N -> CC),
// else faces -> edges (CC -> N).  val(c, at): component c's value.
template <int D, bool FACES, typename V>
__device__ __forceinline__ double curl_at(const FView3 &in, const Pos &a, const MeshDev &M, V val) {
  constexpr int C0 = (D + 2) % 3, E0 = (D + 1) % 3, C1 = (D + 1) % 3, E1 = (D + 2) % 3;
  const Stag<!FACES> s0(a.q[E0], in.f[C0].s[E0], M.c[E0]), s1(a.q[E1], in.f[C1].s[E1], M.c[E1]);
  const size_t o0 = off(in.f[C0], at<E0>(a, s0.i)), o1 = off(in.f[C1], at<E1>(a, s1.i));
  const double a0 = val(C0, o0), a1 = val(C0, o0 + fstride<E0>(in.f[C0]));
  const double b0 = val(C1, o1), b1 = val(C1, o1 + fstride<E1>(in.f[C1]));
  return s1.sub(s0.set(a0, a1), b0, b1);
}

// out = curl(in) (SCALE: times scale)
template <int D, bool FACES, bool SCALE>
__device__ __forceinline__ void curl_block(const FView3 &out, const FView3 &in, const MeshDev &M, double scale) {
  Pos a;
  size_t o;
  if (!my_element(out.f[D].s, a, o)) return;
  const double v = curl_at<D, FACES>(in, a, M, [&](int c, size_t q) { return in.f[c].p[q]; });
  out.f[D].p[o] = SCALE ? v * scale : v;
}
template <bool FACES, bool SCALE>
__global__ void __launch_bounds__(kSrc) k_curl3(FView3 out, FView3 in, MeshDev M, double scale) {
  if (blockIdx.y == 0) curl_block<0, FACES, SCALE>(out, in, M, scale);
  else if (blockIdx.y == 1) curl_block<1, FACES, SCALE>(out, in, M, scale);
  else curl_block<2, FACES, SCALE>(out, in, M, scale);
}

// ---------------------------------------------------------------- induction
// FB = curl(U x B) - 0 curl(J sig) (beta = 1 - alpha = 0, as O2 time marching
// has it), the AB2 right-hand side of B*, and B* = B:
//   FB' = (0 + adv * 1) + c2 * (-0);  rhs = ((FB' 1.5 + FB (-0.5)) + 0) dt, 0 on Dirichlet walls, + B
struct IndArgs {
  FView3 E, J, sig, FB, B, rhs, Bstar;
  int wall[3];
  double dt;
};
__device__ __forceinline__ double ab2_element(double F, double Fold, bool has_L, double dt, int wall, int pd, int sd,
                                              double X) {
  double v = F * 1.5;
  v = v + Fold * (-0.5);
  if (has_L) v = v + 0.0;
  v = v * dt;
  if (((wall & 1) && pd == 1) || ((wall & 2) && pd == sd - 2)) v = 0.0;
  return v + X;
}
template <int D>
__device__ __forceinline__ void ind_block(const IndArgs &A, const MeshDev &M) {
  Pos a;
  size_t o;
  const FView &fb = A.FB.f[D];
  if (!my_element(fb.s, a, o)) return;
  const double old = fb.p[o], B = A.B.f[D].p[o];
  const double adv = curl_at<D, true>(A.E, a, M, [&](int c, size_t q) { return A.E.f[c].p[q]; });
  const double cj = curl_at<D, true>(A.J, a, M, [&](int c, size_t q) { return A.J.f[c].p[q] * A.sig.f[c].p[q]; });
  double F = 0.0 + adv * 1.0;
  F = F + cj * (-0.0);
  fb.p[o] = F;
  A.rhs.f[D].p[o] = ab2_element(F, old, true, A.dt, A.wall[D], a.q[D], fb.s[D], B);
  A.Bstar.f[D].p[o] = B;
}
// 30 passes of 3-6 us at 64^3, now 18 us.
__global__ void __launch_bounds__(kSrc) k_ind_source(IndArgs A, MeshDev M) {
  if (blockIdx.y == 0) ind_block<0>(A, M);
  else if (blockIdx.y == 1) ind_block<1>(A, M);
  else ind_block<2>(A, M);
}

// Btot = B0 + B * 1
__global__ void __launch_bounds__(kSrc) k_btot(FView3 out, FView3 B0, FView3 B) {
  const int d = blockIdx.y;
  const size_t n = (size_t)out.f[d].s[0] * out.f[d].s[1] * out.f[d].s[2];
  const size_t t = (size_t)blockIdx.x * kSrc + threadIdx.x;
  if (t < n) out.f[d].p[t] = B0.f[d].p[t] + B.f[d].p[t] * 1.0;
}

// Face component C at the centre of face direction D: face -> cell (half sums
// along C) -> face (theta weights along D).
template <int C, int D>
__device__ __forceinline__ double face2face_at(const FView &f, const Pos &a, const MeshDev &M) {
  const double *__restrict__ p = f.p;
  const size_t st = fstride<C>(f);
  return c2n(a.q[D], f.s[D], M.c[D], [&](int m) {
    const size_t o = off(f, at<D>(a, m));
    return 0.5 * (p[o] + p[o + st]);
  });
}

// JxB = (edge2Face(J) x face2Face(Btot)) N
template <int D>
__device__ __forceinline__ void jxb_block(const FView3 &out, const FView3 &J, const FView3 &Bt, const MeshDev &M,
                                          double N) {
  constexpr int L = D == 0 ? 1 : 0, H = D == 2 ? 1 : 2;
  Pos a;
  size_t o;
  if (!my_element(out.f[D].s, a, o)) return;
  const size_t ol = off(J.f[L], a), oh = off(J.f[H], a);
  const double jl = 0.5 * (J.f[L].p[ol] + J.f[L].p[ol + fstride<H>(J.f[L])]);
  const double jh = 0.5 * (J.f[H].p[oh] + J.f[H].p[oh + fstride<L>(J.f[H])]);
  const double bl = face2face_at<L, D>(Bt.f[L], a, M), bh = face2face_at<H, D>(Bt.f[H], a, M);
  const double v = jl * bh - jh * bl;
  out.f[D].p[o] = (D == 1 ? -v : v) * N;
}
// 24 passes of 3-6 us at 64^3, now 9.3 us.
__global__ void __launch_bounds__(kSrc) k_jxb(FView3 out, FView3 J, FView3 Bt, MeshDev M, double N) {
  if (blockIdx.y == 0) jxb_block<0>(out, J, Bt, M, N);
  else if (blockIdx.y == 1) jxb_block<1>(out, J, Bt, M, N);
  else jxb_block<2>(out, J, Bt, M, N);
}

// ---------------------------------------------------------------- momentum
// F = -u.grad(u) + ce lap(u) + J x B + buoyancy + gravity, the AB2 right-hand
// side and (implicit diffusion) U* = U.  jx: J x B on the fluid faces (null:
// none); J x B, buoyancy and gravity count as 0 on the ghost planes.
struct MomArgs {
  FView3 U, F, Fnm1, rhs, Ustar, UE0, UE1, jx, g;
  FView T;
  int wall[3], has_L, buoy, grav, copy_U;
  double ce, dt, buoy_scale, grav_scale;
};
template <int D>
__device__ __forceinline__ void mom_block(const MomArgs &A, const MeshDev &M) {
  Pos a;
  size_t o;
  const FView &u = A.U.f[D];
  if (!my_element(u.s, a, o)) return;
  const double *__restrict__ up = u.p;
  const size_t fd = fstride<D>(u);
  const double old = A.F.f[D].p[o], U = up[o];
  // u_d d/dx_d u_d: the cell-centred component's derivative back on the faces
  double T;
  {
    const Stag<true> s(a.q[D], u.s[D] - 1, M.c[D]);
    const size_t q = off(u, at<D>(a, s.i));
    const double f0 = up[q], f1 = up[q + fd], f2 = up[q + 2 * fd];
    T = s.set(0.5 * (f0 + f1), 0.5 * (f1 + f2)) * U;
  }
  // u_v d/dx_v u_d for the other two directions v, from u_d on the edges
  auto cross = [&](auto v_, const FView &e) {
    constexpr int V = decltype(v_)::value;
    const Stag<false> s(a.q[V], e.s[V], M.c[V]);
    const size_t q = off(e, at<V>(a, s.i));
    const double d = s.set(e.p[q], e.p[q + fstride<V>(e)]);
    const double p = d * face2face_at<V, D>(A.U.f[V], a, M);
    T = T + p;
  };
  constexpr int V0 = D == 0 ? 1 : 0, V1 = D == 2 ? 1 : 2;
  cross(std::integral_constant<int, V0>{}, A.UE0.f[D]);
  cross(std::integral_constant<int, V1>{}, A.UE1.f[D]);
  double F = 0.0 + T * -1.0;
  // the collocated Laplacian
  double lap = 0.0;
  auto dir = [&](auto e_) {
    constexpr int E = decltype(e_)::value;
    const DirCoefDev &c = M.c[E];
    constexpr bool N = E == D;
    const size_t st = fstride<E>(u), q = off(u, at<E>(a, 0));
    lap = del_col<N>(E == 0, lap, a.q[E], u.s[E], N ? c.colN_L[1] : c.colCC_L[1], N ? c.colN_D[1] : c.colCC_D[1],
                     N ? c.colN_U[1] : c.colCC_U[1], [&](int m) { return up[q + m * st]; });
  };
  dir(std::integral_constant<int, 0>{});
  dir(std::integral_constant<int, 1>{});
  dir(std::integral_constant<int, 2>{});
  F = F + lap * A.ce;
  const bool zero = on_ghost(63, u.s, a);
  if (A.jx.f[D].p) F = F + (zero ? 0.0 : A.jx.f[D].p[o]) * 1.0;
  if (A.buoy) {
    const double *__restrict__ g = A.g.f[D].p;
    const double v = c2n(a.q[D], A.T.s[D], M.c[D], [&](int m) {
      const size_t q = off(A.T, at<D>(a, m));
      return A.T.p[q] * g[q];
    });
    F = F + (zero ? 0.0 : v) * A.buoy_scale;
  }
  if (A.grav) {
    const FView &g = A.g.f[D];
    const double v = c2n(a.q[D], g.s[D], M.c[D], [&](int m) { return g.p[off(g, at<D>(a, m))]; });
    F = F + (zero ? 0.0 : v) * A.grav_scale;
  }
  A.F.f[D].p[o] = F;
  A.Fnm1.f[D].p[o] = old;
  A.rhs.f[D].p[o] = ab2_element(F, old, A.has_L, A.dt, A.wall[D], a.q[D], u.s[D], U);
  if (A.copy_U) A.Ustar.f[D].p[o] = U;
}
// About 80 passes, of 3-6 us at 64^3 and 10-13 us at 128^3; now 26 and 231 us.
__global__ void __launch_bounds__(kSrc) k_mom_source(MomArgs A, MeshDev M) {
  if (blockIdx.y == 0) mom_block<0>(A, M);
  else if (blockIdx.y == 1) mom_block<1>(A, M);
  else mom_block<2>(A, M);
}

// ---------------------------------------------------------------- energy
// U_CC = face2CellCenter(U), and (q not null) q = Ux^2 + Uy^2 + Uz^2
__global__ void __launch_bounds__(kSrc) k_ucc(FView3 UCC, FView3 U, double *q) {
  Pos a;
  size_t o;
  if (!my_element(UCC.f[0].s, a, o)) return;
  double v[3];
  const size_t st[3] = {1, (size_t)U.f[1].s[0], (size_t)U.f[2].s[0] * U.f[2].s[1]};
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    const double *p = U.f[d].p + off(U.f[d], a);
    v[d] = 0.5 * (p[0] + p[st[d]]);
    UCC.f[d].p[o] = v[d];
  }
  if (q) {
    const double x = v[0] * v[0], y = v[1] * v[1], z = v[2] * v[2];
    const double xy = x + y;
    q[o] = xy + z;
  }
}

// lapUniformCoeff_SF or (n = 1) one first derivative, collocated on the cells
template <int E>
__device__ __forceinline__ double col_cc(bool first, double acc, int n, const FView &f, const Pos &a, const MeshDev &M) {
  const DirCoefDev &c = M.c[E];
  const double *__restrict__ p = f.p + off(f, at<E>(a, 0));
  const size_t st = fstride<E>(f);
  return del_col<false>(first, acc, a.q[E], f.s[E], c.colCC_L[n - 1], c.colCC_D[n - 1], c.colCC_U[n - 1],
                        [&](int m) { return p[m * st]; });
}
__device__ __forceinline__ double lap_cc(const FView &f, const Pos &a, const MeshDev &M) {
  double v = col_cc<0>(true, 0.0, 2, f, a, M);
  v = col_cc<1>(false, v, 2, f, a, M);
  return col_cc<2>(false, v, 2, f, a, M);
}

// The energy equation's sources (add_all_energy_sources), Fnm1 = F first.
struct NrgArgs {
  FView3 U, UCC, J;
  FView T, F, Fnm1, L, q, sig, qv;
  int advection, diffusion, diffusion_in_L, KE, viscous, joule, volumetric;
  double c_adv, c_diff, c_KE, c_visc, c_joule, c_vol;
};
// (cellCenter2Face(T) U) at the two faces of a cell along D, and their derivative
template <int D>
__device__ __forceinline__ double flux_div(bool first, double acc, const NrgArgs &A, const Pos &a, const MeshDev &M) {
  const FView &u = A.U.f[D];
  const double *__restrict__ tp = A.T.p + off(A.T, at<D>(a, 0));
  const size_t st = fstride<D>(A.T);
  const double *up = u.p + off(u, a);
  const int o = a.q[D];
  auto T = [&](int m) { return tp[m * st]; };
  const double f0 = c2n(o, A.T.s[D], M.c[D], T) * up[0], f1 = c2n(o + 1, A.T.s[D], M.c[D], T) * up[fstride<D>(u)];
  const Stag<false> s(o, u.s[D], M.c[D]);
  return first ? s.set(f0, f1) : s.add(acc, f0, f1);
}
// Edge component d at the cell centre: along the third direction first, then
// along d + 1.
template <int D>
__device__ __forceinline__ double edge2cc(const FView &J, const Pos &a) {
  constexpr int FD = (D + 1) % 3, OD = 3 - D - FD;
  const double *p = J.p + off(J, a);
  const size_t so = fstride<OD>(J), sf = fstride<FD>(J);
  const double lo = 0.5 * (p[0] + p[so]), hi = 0.5 * (p[sf] + p[sf + so]);
  return 0.5 * (lo + hi);
}
// About 85 passes with every source on, 5-12 us each at 120 x 100 x 110; now
// this and k_ucc, 99 + 19 us.
__global__ void __launch_bounds__(kSrc) k_nrg_source(NrgArgs A, MeshDev M) {
  Pos a;
  size_t o;
  if (!my_element(A.T.s, a, o)) return;
  A.Fnm1.p[o] = A.F.p[o];
  double F = 0.0;
  if (A.advection) {
    // div of the fluxes counts as 0 on the ghost cells
    double v = flux_div<0>(true, 0.0, A, a, M);
    v = flux_div<1>(false, v, A, a, M);
    v = flux_div<2>(false, v, A, a, M);
    if (on_ghost(63, A.T.s, a)) v = 0.0;
    F = F + v * A.c_adv;
  }
  if (A.diffusion) {
    const double w = lap_cc(A.T, a, M) * A.c_diff;
    if (A.diffusion_in_L) A.L.p[o] = 0.0 + w;
    else F = F + w;
  } else if (A.diffusion_in_L) {
    A.L.p[o] = 0.0;
  }
  if (A.KE) F = F + lap_cc(A.q, a, M) * A.c_KE;
  if (A.viscous) {
    // G[c][e] = d U_c / d x_e, squares summed over c, then e
    double acc = 0.0;
    auto dir = [&](auto e_) {
      constexpr int E = decltype(e_)::value;
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        const double g = col_cc<E>(true, 0.0, 1, A.UCC.f[c], a, M);
        const double sq = g * g;
        acc = E == 0 && c == 0 ? sq : acc + sq;
      }
    };
    dir(std::integral_constant<int, 0>{});
    dir(std::integral_constant<int, 1>{});
    dir(std::integral_constant<int, 2>{});
    F = F + acc * A.c_visc;
  }
  if (A.joule) {
    const double x = edge2cc<0>(A.J.f[0], a), y = edge2cc<1>(A.J.f[1], a), z = edge2cc<2>(A.J.f[2], a);
    double acc = x * x;
    acc = acc + y * y;
    acc = acc + z * z;
    acc = acc * A.sig.p[o];
    F = F + acc * A.c_joule;
  }
  if (A.volumetric) F = F + A.qv.p[o] * A.c_vol;
  A.F.p[o] = F;
}

// ---------------------------------------------------------------- projection
// divU = div(u) (N -> CC along each direction), 0 on the ghost planes of the
// faces in zero, times scale (scaled != 0)
__global__ void __launch_bounds__(kSrc) k_div(FView out, FView3 u, MeshDev M, int zero, int scaled, double scale) {
  Pos a;
  size_t o;
  if (!my_element(out.s, a, o)) return;
  double v;
  {
    const Stag<false> s(a.q[0], u.f[0].s[0], M.c[0]);
    const size_t q = off(u.f[0], a);
    v = s.set(u.f[0].p[q], u.f[0].p[q + 1]);
  }
  {
    const Stag<false> s(a.q[1], u.f[1].s[1], M.c[1]);
    const size_t q = off(u.f[1], a);
    v = s.add(v, u.f[1].p[q], u.f[1].p[q + u.f[1].s[0]]);
  }
  {
    const Stag<false> s(a.q[2], u.f[2].s[2], M.c[2]);
    const size_t q = off(u.f[2], a);
    v = s.add(v, u.f[2].p[q], u.f[2].p[q + (size_t)u.f[2].s[0] * u.f[2].s[1]]);
  }
  if (on_ghost(zero, out.s, a)) v = 0.0;
  out.p[o] = scaled ? v * scale : v;
}

// g = grad(phi) inv; X = X* - g
template <int D>
__device__ __forceinline__ void project_block(const FView3 &X, const FView3 &Xs, const FView3 &g, const FView &phi,
                                              const MeshDev &M, double inv) {
  Pos a;
  size_t o;
  if (!my_element(g.f[D].s, a, o)) return;
  const Stag<true> s(a.q[D], phi.s[D], M.c[D]);
  const size_t q = off(phi, at<D>(a, s.i));
  const double v = s.set(phi.p[q], phi.p[q + fstride<D>(phi)]) * inv, x = Xs.f[D].p[o];
  g.f[D].p[o] = v;
  X.f[D].p[o] = x - v;
}
__global__ void __launch_bounds__(kSrc) k_project(FView3 X, FView3 Xs, FView3 g, FView phi, MeshDev M, double inv) {
  if (blockIdx.y == 0) project_block<0>(X, Xs, g, phi, M, inv);
  else if (blockIdx.y == 1) project_block<1>(X, Xs, g, phi, M, inv);
  else project_block<2>(X, Xs, g, phi, M, inv);
}

// ---------------------------------------------------------------- launchers
static dim3 grid3(moons_field_s *const f[3]) {
  size_t n = 0;
  for (int d = 0; d < 3; ++d) n = f[d]->n > n ? f[d]->n : n;
  return dim3((unsigned)((n + kSrc - 1) / kSrc), 3);
}
// elements are numbered in 32 bits
static int below_2_31(moons_field_s *const f[3]) {
  for (int d = 0; d < 3; ++d)
    if (f[d]->n >= ((size_t)1 << 31)) return fail(MOONS_ERR_ARG, "fields of 2^31 or more elements are not supported");
  return MOONS_OK;
}
static bool on_mesh(const moons_field_s *f, const moons_mesh_s *m, int dl) {
  return f->m == m && f->dl == dl && f->n < ((size_t)1 << 31);
}
static const int kEdge[3] = {MOONS_DL_EDGE_X, MOONS_DL_EDGE_Y, MOONS_DL_EDGE_Z};

bool edges_fit(moons_field_s *const E[3], moons_field_s *const U_E[6], moons_field_s *const B[3],
               moons_field_s *const tmp[6]) {
  const moons_mesh_s *m = B[0]->m;
  // tmp of edge d: l and h
  static const int kTmp[3][2] = {{2, 4}, {0, 5}, {1, 3}};
  for (int d = 0; d < 3; ++d) {
    if (!on_mesh(B[d], m, 1 << d) || !on_mesh(E[d], m, kEdge[d])) return false;
    const moons_field_s *f[5] = {E[d], U_E[2 * d], U_E[2 * d + 1], tmp[kTmp[d][0]], tmp[kTmp[d][1]]};
    for (int q = 1; q < 5; ++q) {
      if (!on_mesh(f[q], m, kEdge[d])) return false;
      for (int r = 0; r < q; ++r)
        if (f[q]->d == f[r]->d && (q >= 3 || r == 0)) return false; // an operand that is also a result
    }
  }
  return !current_gate();
}

int launch_edge_cross(moons_field_s *const E[3], moons_field_s *const U_E[6], moons_field_s *const B[3],
                      moons_field_s *const tmp[6]) {
  static const int kTmp[3][2] = {{2, 4}, {0, 5}, {1, 3}};
  EdgeArgs A{};
  A.in = fview3(B);
  A.E = fview3(E);
  for (int d = 0; d < 3; ++d)
    for (int q = 0; q < 2; ++q) {
      A.out[d][q] = tmp ? tmp[kTmp[d][q]]->d : nullptr;
      A.U[d][q] = U_E[2 * d + q]->d;
    }
  hipLaunchKernelGGL(k_edge<true>, grid3(E), dim3(kSrc), 0, stream(), A, B[0]->m->dev);
  MOONS_LAUNCH_CHECK();
  return MOONS_OK;
}

int launch_face2edge(moons_field_s *const UE[6], moons_field_s *const U[3]) {
  EdgeArgs A{};
  A.in = fview3(U);
  moons_field_s *e[3] = {UE[0], UE[2], UE[4]};
  if (int st = below_2_31(e)) return st;
  A.E = fview3(e);
  for (int d = 0; d < 3; ++d)
    for (int q = 0; q < 2; ++q) A.out[d][q] = UE[2 * d + q]->d;
  hipLaunchKernelGGL(k_edge<false>, grid3(e), dim3(kSrc), 0, stream(), A, U[0]->m->dev);
  MOONS_LAUNCH_CHECK();
  return MOONS_OK;
}

bool curl3_fits(moons_field_s *const out[3], moons_field_s *const in[3]) {
  const moons_mesh_s *m = in[0]->m;
  const bool faces = out[0]->dl == 1;
  for (int d = 0; d < 3; ++d)
    if (!on_mesh(out[d], m, faces ? 1 << d : kEdge[d]) || !on_mesh(in[d], m, faces ? kEdge[d] : 1 << d)) return false;
  return !current_gate();
}

int launch_curl3(moons_field_s *const out[3], moons_field_s *const in[3], bool scaled, double scale) {
  const bool faces = out[0]->dl == 1;
  const FView3 o = fview3(out), i = fview3(in);
  const MeshDev &M = in[0]->m->dev;
  if (faces) {
    if (scaled) hipLaunchKernelGGL((k_curl3<true, true>), grid3(out), dim3(kSrc), 0, stream(), o, i, M, scale);
    else hipLaunchKernelGGL((k_curl3<true, false>), grid3(out), dim3(kSrc), 0, stream(), o, i, M, scale);
  } else {
    if (scaled) hipLaunchKernelGGL((k_curl3<false, true>), grid3(out), dim3(kSrc), 0, stream(), o, i, M, scale);
    else hipLaunchKernelGGL((k_curl3<false, false>), grid3(out), dim3(kSrc), 0, stream(), o, i, M, scale);
  }
  MOONS_LAUNCH_CHECK();
  return MOONS_OK;
}

int launch_ind_source(moons_field_s *const E[3], moons_field_s *const J[3], moons_field_s *const sig[3],
                      moons_field_s *const FB[3], moons_field_s *const B[3], moons_field_s *const rhs[3],
                      moons_field_s *const Bstar[3], const int wall[3], double dt) {
  if (int st = below_2_31(FB)) return st;
  IndArgs A{fview3(E), fview3(J), fview3(sig), fview3(FB), fview3(B), fview3(rhs), fview3(Bstar),
            {wall[0], wall[1], wall[2]}, dt};
  hipLaunchKernelGGL(k_ind_source, grid3(FB), dim3(kSrc), 0, stream(), A, FB[0]->m->dev);
  MOONS_LAUNCH_CHECK();
  return MOONS_OK;
}

int launch_btot(moons_field_s *const out[3], moons_field_s *const B0[3], moons_field_s *const B[3]) {
  hipLaunchKernelGGL(k_btot, grid3(out), dim3(kSrc), 0, stream(), fview3(out), fview3(B0), fview3(B));
  MOONS_LAUNCH_CHECK();
  return MOONS_OK;
}

int launch_jxb(moons_field_s *const out[3], moons_field_s *const J[3], moons_field_s *const Bt[3], double N) {
  if (int st = below_2_31(out)) return st;
  hipLaunchKernelGGL(k_jxb, grid3(out), dim3(kSrc), 0, stream(), fview3(out), fview3(J), fview3(Bt), out[0]->m->dev, N);
  MOONS_LAUNCH_CHECK();
  return MOONS_OK;
}

int launch_nrg_source(const NrgSource &S) {
  // (volumetric heating reads its own element alone; elements are numbered in 32 bits)
  const bool stencils = S.advection || S.diffusion || S.KE || S.viscous || S.joule;
  if (S.T->n >= (size_t)1 << (stencils ? 31 : 32))
    return fail(MOONS_ERR_ARG, "fields of 2^31 or more elements are not supported");
  NrgArgs A{};
  const dim3 grid((unsigned)((S.T->n + kSrc - 1) / kSrc));
  const MeshDev &M = S.T->m->dev;
  if (S.KE || S.viscous) {
    A.UCC = fview3(S.UCC);
    hipLaunchKernelGGL(k_ucc, grid, dim3(kSrc), 0, stream(), A.UCC, fview3(S.U), S.KE ? S.q->d : nullptr);
    MOONS_LAUNCH_CHECK();
  }
  if (S.advection) A.U = fview3(S.U);
  if (S.joule) {
    A.J = fview3(S.J);
    A.sig = fview(S.sig);
  }
  A.T = fview(S.T);
  A.F = fview(S.F);
  A.Fnm1 = fview(S.Fnm1);
  A.L = fview(S.L);
  A.q = fview(S.q);
  A.qv = fview(S.qv);
  A.advection = S.advection;
  A.diffusion = S.diffusion;
  A.diffusion_in_L = S.diffusion_in_L;
  A.KE = S.KE;
  A.viscous = S.viscous;
  A.joule = S.joule;
  A.volumetric = S.volumetric;
  A.c_adv = S.c_adv;
  A.c_diff = S.c_diff;
  A.c_KE = S.c_KE;
  A.c_visc = S.c_visc;
  A.c_joule = S.c_joule;
  A.c_vol = S.c_vol;
  hipLaunchKernelGGL(k_nrg_source, grid, dim3(kSrc), 0, stream(), A, M);
  MOONS_LAUNCH_CHECK();
  return MOONS_OK;
}

bool div_fits(const moons_field_s *divU, moons_field_s *const u[3]) {
  if (divU->dl != MOONS_DL_CC || divU->n >= ((size_t)1 << 31) || current_gate()) return false;
  for (int d = 0; d < 3; ++d)
    if (!on_mesh(u[d], divU->m, 1 << d)) return false;
  return true;
}

int launch_div(moons_field_s *divU, moons_field_s *const u[3], bool scaled, double scale) {
  int zero = 0;
  for (int f = 0; f < 6; ++f)
    if (!(divU->has_bcs && divU->bct[f] == MOONS_BC_PERIODIC)) zero |= 1 << f;
  hipLaunchKernelGGL(k_div, dim3((unsigned)((divU->n + kSrc - 1) / kSrc)), dim3(kSrc), 0, stream(), fview(divU),
                     fview3(u), divU->m->dev, zero, scaled ? 1 : 0, scale);
  MOONS_LAUNCH_CHECK();
  return MOONS_OK;
}

// (X may be X*: each element reads its own entry alone)
bool project_fits(moons_field_s *const X[3], moons_field_s *const Xstar[3], moons_field_s *const g[3],
                  const moons_field_s *phi) {
  if (phi->dl != MOONS_DL_CC || phi->n >= ((size_t)1 << 31) || current_gate()) return false;
  for (int d = 0; d < 3; ++d)
    if (!on_mesh(g[d], phi->m, 1 << d) || !on_mesh(X[d], phi->m, 1 << d) || !on_mesh(Xstar[d], phi->m, 1 << d) ||
        g[d]->d == X[d]->d || g[d]->d == Xstar[d]->d)
      return false;
  return true;
}

int launch_project(moons_field_s *const X[3], moons_field_s *const Xstar[3], moons_field_s *const g[3],
                   const moons_field_s *phi, double inv) {
  hipLaunchKernelGGL(k_project, grid3(g), dim3(kSrc), 0, stream(), fview3(X), fview3(Xstar), fview3(g), fview(phi),
                     phi->m->dev, inv);
  MOONS_LAUNCH_CHECK();
  return MOONS_OK;
}

int launch_mom_source(const MomSource &S) {
  if (int st = below_2_31(S.U)) return st;
  MomArgs A{};
  A.U = fview3(S.U);
  A.F = fview3(S.F);
  A.Fnm1 = fview3(S.Fnm1);
  A.rhs = fview3(S.rhs);
  A.copy_U = S.Ustar != nullptr;
  if (S.Ustar) A.Ustar = fview3(S.Ustar);
  // u_d on the edges along the third direction of (d, v): its derivative along
  // v lies on the d faces; v the lower (UE0) and the higher (UE1) of the others
  static const int kUE[3][2] = {{4, 2}, {5, 0}, {3, 1}};
  for (int d = 0; d < 3; ++d) {
    A.UE0.f[d] = fview(S.UE[kUE[d][0]]);
    A.UE1.f[d] = fview(S.UE[kUE[d][1]]);
    A.wall[d] = S.wall[d];
  }
  if (S.jx) A.jx = fview3(S.jx);
  A.has_L = S.Ustar != nullptr;
  A.buoy = S.T != nullptr;
  A.grav = S.grav;
  if (S.T) A.T = fview(S.T);
  if (S.T || S.grav)
    for (int d = 0; d < 3; ++d) A.g.f[d] = fview(S.g[d]);
  A.ce = S.ce;
  A.dt = S.dt;
  A.buoy_scale = S.buoy_scale;
  A.grav_scale = S.grav_scale;
  hipLaunchKernelGGL(k_mom_source, grid3(S.U), dim3(kSrc), 0, stream(), A, S.U[0]->m->dev);
  MOONS_LAUNCH_CHECK();
  return MOONS_OK;
}

} // namespace moons
