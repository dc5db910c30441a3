// vfpcg.hip -- FP64 Jacobi-PCG for the face-centred vector solves: the
// momentum implicit diffusion (mom_diffusion, A = I + c lap_centered_VF) and
// the induction implicit diffusion (ind_diffusion, A = I + c curl(k curl)).
//
// Restates solve_PCG_VF (code/handwritten/solvers/PCG/PCG_solver_algorithm.f90:109-179),
// modify_RHS_VF (PCG_aux.f90:56-79), the operators (matrix_free_operators.f90:120-146,
// 176-202) and prec_mom_VF / prec_ind_VF (preconditioners.f90:86-129).
//
// One iteration, all on the three components at once (one grid row each):
//   apply_BCs_implicit(p)   one launch
//   k_vf_mom_op | k_vf_curl twice   Ax = vol A p with the wall rules
//   k_vf_dot       partials of (p,Ax)
//   k_vf_update    alpha; x += a p, r -= a Ax, partials (r,r), (Minv r, r)
//   k_vf_pupdate   exit test, beta; p = b p + Minv r
// A kernel that needs a dot product sums the previous kernel's partials in its
// prologue, every block in the same order; block 0 publishes the scalars in a
// device control block, so the loop needs no host round trip.  The order of
// every sum is one for all kernels (dot_map), so that it does not depend on how
// the work around it is split.  With a launch for each dot product, for its
// scalar and for z = Minv r (14 launches an iteration), a 128^3 iteration took
// 270-285 us, of which the operators, a thread an element with its 1D
// coefficients loaded each time, were 100 us.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <type_traits>
#include <vector>

#include "cc_stencil.hpp"

namespace moons {

struct VF3 {
  double *p[3];
  int s[3][3];
  size_t n[3];
};

struct VfCtrl {
  int iter, done, exit_loop, iter_max, n_skip, pad_;
  double tol_rel, tol_abs;
  double rho[2]; // rho of the last iteration, indexed by its parity
  double alpha, beta, res0, res, pq, rr, rz;
};

static VF3 vf3(moons_field_s *const f[3]) {
  VF3 v;
  for (int d = 0; d < 3; ++d) {
    v.p[d] = f[d]->d;
    for (int e = 0; e < 3; ++e) v.s[d][e] = f[d]->s[e];
    v.n[d] = f[d]->n;
  }
  return v;
}

// ------------------------------------------------------------------ kernels
// The operators' blocks: 256 columns of kVZ planes over every element of a
// component (ghosts included), the columns numbered through the plane (rows of
// 131 elements in tiles of 64 would leave a third of the waves nearly empty);
// blocks are numbered XCD-contiguously, so that neighbouring planes share an L2.
constexpr int kVZ = 8; // 2, 4, 8 planes: 65, 53, 50 us for k_vf_mom_op at 128^3, the curls equal within 2 us

struct VfGrid {
  int nt; // column tiles a plane
};

struct VfCol {
  int i, j, k0, nk; // the thread's column of a tile (clamped inside); nk 0: outside the component
};
__device__ __forceinline__ VfCol vf_col(const VfGrid &g, const int (&s)[3]) {
  const int b = xcd_remap((int)blockIdx.x, (int)gridDim.x);
  const int q = (b % g.nt) * kNT + (int)threadIdx.x, n = s[0] * s[1], qc = min(q, n - 1);
  VfCol c;
  c.j = qc / s[0];
  c.i = qc - c.j * s[0];
  c.k0 = b / g.nt * kVZ;
  c.nk = q < n ? max(0, min(kVZ, s[2] - c.k0)) : 0;
  return c;
}

// The staggered 1D stencils of the three directions (cc2n: CC -> N, n2cc: N -> CC).
struct StagCoefs {
  const double *cc2n_D[3], *cc2n_U[3], *n2cc_D[3], *n2cc_U[3];
};

// The wall-plane rules of the operator's output in the PCG loop
// (multiply_wall_Neumann 0.5, assign_wall_Dirichlet 0, assign_wall_Periodic_single
// 0 on the boundary-normal planes 1 and s-2 of each component),
// then the product with the cell volume: applied by the operator kernels to
// each element they write when `on` is set.
struct WallVol {
  int on;
  const double *vol[3];
  int lo[3], hi[3]; // 0 none, 1 Dirichlet (set 0), 2 Neumann (times 0.5)
  int per[3];       // periodic pair: plane s-2 set to 0
};

__device__ __forceinline__ double wall_rule(const WallVol &W, int d, int pd, int sd, double v) {
  if (pd == 1) {
    if (W.lo[d] == 1) v = 0.0;
    else if (W.lo[d] == 2) v = v * 0.5;
  }
  if (pd == sd - 2) {
    if (W.hi[d] == 1) v = 0.0;
    else if (W.hi[d] == 2) v = v * 0.5;
    if (W.per[d]) v = 0.0;
  }
  return v;
}

// Whether an interior element counts in the dot products: not on the Dirichlet
// wall-node planes (dot_product_VF: multiply, assign_wall_Dirichlet, sum pad 1;
// code/handwritten/ops/ops_aux.f90:199-207).
// excl: bit 2d = exclude plane 1 of component d, bit 2d+1 = plane s-2.
__device__ __forceinline__ bool in_dot(int excl, int d, int sd, int pd) {
  return !((((excl >> (2 * d)) & 1) && pd == 1) || (((excl >> (2 * d + 1)) & 1) && pd == sd - 2));
}

// The interior (pad 1) elements of a component in the order in which every dot
// product adds them: thread t of the grid row takes elements t, t + threads, ...
// of the interior in memory order.  visit(o, p): element o at position p along d.
template <typename F>
__device__ __forceinline__ void dot_map(const int (&s)[3], int d, F visit) {
  const int n0 = s[0] - 2, n01 = n0 * (s[1] - 2);
  const int ni = n01 * (s[2] - 2); // fields of the VF solver stay below 2^31 elements (checked at creation)
#pragma unroll 4
  for (int t = blockIdx.x * kNT + threadIdx.x; t < ni; t += gridDim.x * kNT) {
    const int k = 1 + t / n01;
    const int r = t - (k - 1) * n01;
    const int j = 1 + r / n0;
    const int i = 1 + (r - (j - 1) * n0);
    visit((size_t)i + (size_t)s[0] * ((size_t)j + (size_t)s[1] * k), i, j, k);
  }
}
// The other elements (the ghost planes), each once, over the same threads.
template <typename F>
__device__ __forceinline__ void ghost_map(const int (&s)[3], F visit) {
  const int pz = s[0] * s[1], py = s[0] * (s[2] - 2), px = (s[1] - 2) * (s[2] - 2);
  for (int t = blockIdx.x * kNT + threadIdx.x; t < 2 * (pz + py + px); t += gridDim.x * kNT) {
    int q = t, i, j, k;
    if (q < 2 * pz) {
      k = q < pz ? 0 : s[2] - 1;
      q -= q < pz ? 0 : pz;
      i = q % s[0];
      j = q / s[0];
    } else if ((q -= 2 * pz) < 2 * py) {
      j = q < py ? 0 : s[1] - 1;
      q -= q < py ? 0 : py;
      i = q % s[0];
      k = 1 + q / s[0];
    } else {
      q -= 2 * py;
      i = q < px ? 0 : s[0] - 1;
      q -= q < px ? 0 : px;
      j = 1 + q % (s[1] - 2);
      k = 1 + q / (s[1] - 2);
    }
    visit((size_t)i + (size_t)s[0] * ((size_t)j + (size_t)s[1] * k), i, j, k);
  }
}

// V dot products from the block sums of the last kernel, part[(v 3 + d) nb + b]:
// each component's blocks by a strided sum a thread and the block tree, the
// components added x, y, z (sum(temp%x) + sum(temp%y) + sum(temp%z)).
template <int V>
__device__ __forceinline__ void dot_totals(const double *part, int nb, double (&tot)[V]) {
  constexpr int NW = kNT / kWave;
  __shared__ double sh[3 * V][NW];
  double v[3 * V];
#pragma unroll
  for (int c = 0; c < 3 * V; ++c) v[c] = 0.0;
  for (int q = threadIdx.x; q < nb; q += kNT)
#pragma unroll
    for (int c = 0; c < 3 * V; ++c) v[c] += part[(size_t)c * nb + q];
#pragma unroll
  for (int c = 0; c < 3 * V; ++c) {
#pragma unroll
    for (int o = kWave / 2; o > 0; o >>= 1) v[c] += __shfl_down(v[c], o, kWave);
    if ((threadIdx.x & (kWave - 1)) == 0) sh[c][threadIdx.x / kWave] = v[c];
  }
  __syncthreads();
#pragma unroll
  for (int u = 0; u < V; ++u) {
    tot[u] = 0.0;
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      double s = 0.0;
#pragma unroll
      for (int w = 0; w < NW; ++w) s += sh[3 * u + d][w];
      tot[u] = tot[u] + s;
    }
  }
}

// The block's sum of one dot product's terms into part[(v 3 + d) nb + b].
__device__ __forceinline__ void put_dot(double acc, int v, double *part, double *sh) {
  const double s = block_sum<kNT>(acc, sh);
  if (threadIdx.x == 0) part[((size_t)v * 3 + blockIdx.y) * gridDim.x + blockIdx.x] = s;
}

// Partials of (a, b)
__global__ void __launch_bounds__(kNT) k_vf_dot(VF3 a, VF3 b, int excl, double *part, const int *done) {
  if (*done) return;
  __shared__ double sh[kNT / kWave];
  const int d = blockIdx.y;
  const int s[3] = {a.s[d][0], a.s[d][1], a.s[d][2]};
  const double *__restrict__ ad = a.p[d];
  const double *__restrict__ bd = b.p[d];
  double acc = 0.0;
  dot_map(s, d, [&](size_t o, int i, int j, int k) {
    const double t = ad[o] * bd[o];
    if (in_dot(excl, d, s[d], d == 0 ? i : (d == 1 ? j : k))) acc += t;
  });
  put_dot(acc, 0, part, sh);
}

// The staggered derivative out and back along one direction at position o of a
// pencil of se values (two del passes through a temporary), as coefficients:
// value = tA c0 + tB c1 with tA = f[o-1] a0 + f[o] a1 and tB = f[o] b0 + f[o+1] b1.
// along_n: the data are node-located along the direction (N -> CC -> N), else
// CC -> N -> CC.  A temporary's end entries are 0 (okA, okB); an entry the
// second pass does not write keeps the sum so far (written), which starts at
// zero at the pencil's ends (zero_end).  tB of position o is tA of o + 1.
struct Stag2 {
  double a0, a1, b0, b1, c0, c1;
  bool okA, okB, written, zero_end;
};
__device__ __forceinline__ Stag2 stag2(bool along_n, int o, int se, const double *cD, const double *cU,
                                       const double *nD, const double *nU) {
  Stag2 r;
  r.zero_end = o == 0 || o == se - 1;
  if (along_n) {
    const int q = min(max(o, 1), se - 2);
    r.written = !r.zero_end;
    r.okA = r.okB = true;
    r.a0 = nD[q - 1]; r.a1 = nU[q - 1]; r.b0 = nD[q]; r.b1 = nU[q]; r.c0 = cD[q - 1]; r.c1 = cU[q - 1];
  } else {
    const int qa = max(o - 1, 0), qb = min(o, se - 2);
    r.written = true;
    r.okA = o >= 1;
    r.okB = o <= se - 2;
    r.a0 = cD[qa]; r.a1 = cU[qa]; r.b0 = cD[qb]; r.b1 = cU[qb]; r.c0 = nD[o]; r.c1 = nU[o];
  }
  return r;
}

// One direction's term added to the sum of the earlier ones (first: assigned).
__device__ __forceinline__ double stag2_add(const Stag2 &S, bool first, double acc, double tA, double tB) {
  const double x0 = tA * S.c0, x1 = tB * S.c1;
  const double cur = first || S.zero_end ? 0.0 : acc;
  if (!S.written) return cur;
  return first ? x0 + x1 : cur + x0 + x1;
}

// Ax = x + c lap(x) for the three face components: mom_diffusion
// (code/handwritten/solvers/matrix_free_operators.f90:176-202) over
// lap_centered_SF_given_both (code/handwritten/ops/ops_discrete.f90:112-122),
// with the rounding of its sequence of passes.  A thread marches a column: the
// x and y coefficients stay in registers, the z coefficients of the tile in LDS
// (loaded plane by plane, uniform in the block, they were a chain of scalar
// loads: 93 us at 128^3), the z neighbours and the z-face derivative come from
// the plane before.  103 us at 128^3 (14.9 at 64^3) with a thread an element
// and 32 loads each, now 50 (10.4).
__global__ void __launch_bounds__(kNT) k_vf_mom_op(VF3 Ax, VF3 x, StagCoefs C, double c, WallVol W, VfGrid g,
                                                  const int *gate) {
  if (gate && *gate) return;
  // [0], [1]: a0, a1 of plane k0 + u (its b0, b1 are the next plane's); [2], [3]: c0, c1
  __shared__ double sz[4][kVZ + 1];
  const int d = blockIdx.y;
  const int s[3] = {x.s[d][0], x.s[d][1], x.s[d][2]};
  const size_t sx = s[0], sxy = (size_t)s[0] * s[1];
  const double *__restrict__ xp = x.p[d];
  double *__restrict__ op = Ax.p[d];
  const double *__restrict__ vp = W.on ? W.vol[d] : nullptr;
  const bool zn = d == 2;
  const VfCol t = vf_col(g, s);
  const int i = t.i, j = t.j;
  // neighbours outside the pencil are not used; their loads go to the element itself
  const int im = i > 0 ? -1 : 0, ip = i < s[0] - 1 ? 1 : 0;
  const long jm = j > 0 ? -(long)sx : 0, jp = j < s[1] - 1 ? (long)sx : 0;
  const double *col = xp + i + j * sx;
  double zc[kVZ + 2], nb[kVZ][4], vol[kVZ];
#pragma unroll
  for (int u = 0; u < kVZ + 2; ++u) zc[u] = col[(size_t)min(max(t.k0 - 1 + u, 0), s[2] - 1) * sxy];
#pragma unroll
  for (int u = 0; u < kVZ; ++u) {
    const double *q = col + (size_t)min(t.k0 + u, s[2] - 1) * sxy;
    nb[u][0] = q[im];
    nb[u][1] = q[ip];
    nb[u][2] = q[jm];
    nb[u][3] = q[jp];
    vol[u] = W.on ? vp[q - xp] : 0.0;
  }
  const Stag2 X = stag2(d == 0, i, s[0], C.cc2n_D[0], C.cc2n_U[0], C.n2cc_D[0], C.n2cc_U[0]);
  const Stag2 Y = stag2(d == 1, j, s[1], C.cc2n_D[1], C.cc2n_U[1], C.n2cc_D[1], C.n2cc_U[1]);
  if (threadIdx.x <= kVZ) {
    const int u = threadIdx.x, o = t.k0 + u, qa = min(max(o - 1, 0), s[2] - 2);
    sz[0][u] = zn ? C.n2cc_D[2][qa] : C.cc2n_D[2][qa];
    sz[1][u] = zn ? C.n2cc_U[2][qa] : C.cc2n_U[2][qa];
    const int qc = zn ? min(max(o - 1, 0), s[2] - 3) : min(o, s[2] - 1);
    sz[2][u] = zn ? C.cc2n_D[2][qc] : C.n2cc_D[2][qc];
    sz[3][u] = zn ? C.cc2n_U[2][qc] : C.n2cc_U[2][qc];
  }
  __syncthreads();
  double tz = zn || t.k0 >= 1 ? zc[0] * sz[0][0] + zc[1] * sz[1][0] : 0.0;
#pragma unroll
  for (int u = 0; u < kVZ; ++u) {
    const int k = t.k0 + u;
    const double f = zc[u + 1];
    double acc = stag2_add(X, true, 0.0, X.okA ? nb[u][0] * X.a0 + f * X.a1 : 0.0,
                           X.okB ? f * X.b0 + nb[u][1] * X.b1 : 0.0);
    acc = stag2_add(Y, false, acc, Y.okA ? nb[u][2] * Y.a0 + f * Y.a1 : 0.0,
                    Y.okB ? f * Y.b0 + nb[u][3] * Y.b1 : 0.0);
    const bool end = k == 0 || k == s[2] - 1;
    const double tB = zn || k <= s[2] - 2 ? f * sz[0][u + 1] + zc[u + 2] * sz[1][u + 1] : 0.0;
    const double cur = end ? 0.0 : acc;
    acc = zn && end ? cur : cur + tz * sz[2][u] + tB * sz[3][u];
    tz = tB;
    const double w = acc * c;
    double res = w + f;
    if (W.on) res = wall_rule(W, d, d == 0 ? i : (d == 1 ? j : k), s[d], res) * vol[u];
    vol[u] = res;
  }
#pragma unroll
  for (int u = 0; u < kVZ; ++u)
    if (u < t.nk) op[i + j * sx + (size_t)(t.k0 + u) * sxy] = vol[u];
}

// out_d = curl(in)_d, then (FACES = false, faces -> edges) out_d = curl * aux_d or
// (FACES, edges -> faces) out_d = curl * c + aux_d (multiply then add, as
// ind_diffusion_explicit) with the wall rules and the volume: curl_SF component d
// (code/handwritten/ops/ops_discrete.f90:184-202) assigns the derivative of
// in[(d+2)%3] along (d+1)%3 and subtracts that of in[(d+1)%3] along (d+2)%3,
// both staggered (faces -> edges CC -> N, edges -> faces N -> CC), with the
// rounding and the zeroed end entries of the two del passes.  A thread marches
// a column as in k_vf_mom_op.
// 48 (faces -> edges) + 53 us at 128^3, bound by HBM as with a thread an element
// (48 + 50), whose edges -> faces pass left the wall rules and the volume to a pass of their own.
template <int D, bool FACES>
__device__ __forceinline__ void vf_curl_block(const VF3 &out, const VF3 &in, const StagCoefs &C, const VF3 &aux, double c,
                                              const WallVol &W, const VfGrid &g) {
  const int s[3] = {out.s[D][0], out.s[D][1], out.s[D][2]};
  const size_t sx = s[0], sxy = (size_t)s[0] * s[1];
  const double *__restrict__ ap = aux.p[D];
  const double *__restrict__ vp = FACES && W.on ? W.vol[D] : nullptr;
  double *__restrict__ op = out.p[D];
  constexpr int C0 = (D + 2) % 3, E0 = (D + 1) % 3, C1 = (D + 1) % 3, E1 = (D + 2) % 3;
  const VfCol t = vf_col(g, s);
  if (t.nk == 0) return;
  const int i = t.i, j = t.j;
  // derivative of component CI along E at this column: values lo and hi of each plane
  double lo[2][kVZ], hi[2][kVZ], av[kVZ], vol[kVZ];
  auto gather = [&](auto ci_, auto e_, double (&vl)[kVZ], double (&vh)[kVZ]) {
    constexpr int ci = decltype(ci_)::value, e = decltype(e_)::value;
    const int *si = in.s[ci];
    const size_t ix = si[0], ixy = (size_t)si[0] * si[1];
    const double *__restrict__ p = in.p[ci];
#pragma unroll
    for (int u = 0; u < kVZ; ++u) {
      const int k = min(t.k0 + u, s[2] - 1);
      int q[3] = {i, j, k};
      // inputs o - 1, o (CC -> N) or o, o + 1 (N -> CC); ends that are not written load a clamped position
      const int o = q[e], i0 = FACES ? min(o, si[e] - 2) : min(max(o - 1, 0), si[e] - 2);
      q[e] = i0;
      const size_t at = (size_t)q[0] + (size_t)q[1] * ix + (size_t)q[2] * ixy;
      vl[u] = p[at];
      vh[u] = p[at + (e == 0 ? 1 : (e == 1 ? ix : ixy))];
    }
  };
  gather(std::integral_constant<int, C0>{}, std::integral_constant<int, E0>{}, lo[0], hi[0]);
  gather(std::integral_constant<int, C1>{}, std::integral_constant<int, E1>{}, lo[1], hi[1]);
#pragma unroll
  for (int u = 0; u < kVZ; ++u) {
    const size_t at = i + j * sx + (size_t)min(t.k0 + u, s[2] - 1) * sxy;
    av[u] = ap[at];
    vol[u] = FACES && W.on ? vp[at] : 0.0;
  }
#pragma unroll
  for (int u = 0; u < kVZ; ++u)
    if (u < t.nk) {
      const int k = t.k0 + u;
      double v = 0.0;
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        const int e = q == 0 ? E0 : E1, ci = q == 0 ? C0 : C1;
        const int o = e == 0 ? i : (e == 1 ? j : k);
        const int sin = in.s[ci][e], m = o - (FACES ? 0 : 1);
        const bool written = m >= 0 && m <= sin - 2, zero_end = o == 0 || o == s[e] - 1;
        // (a per-lane index, so that the planes' coefficient loads are in flight
        // together; uniform ones would be a chain of scalar loads)
        int mc = min(max(m, 0), sin - 2);
        asm volatile("" : "+v"(mc));
        const double x0 = lo[q][u] * (FACES ? C.n2cc_D[e][mc] : C.cc2n_D[e][mc]);
        const double x1 = hi[q][u] * (FACES ? C.n2cc_U[e][mc] : C.cc2n_U[e][mc]);
        if (q == 0) {
          v = written ? x0 + x1 : 0.0;
        } else {
          const double cur = zero_end ? 0.0 : v;
          v = written ? cur - (x0 + x1) : cur;
        }
      }
      double res;
      if (!FACES) {
        res = v * av[u];
      } else {
        const double w = v * c;
        res = w + av[u];
        if (W.on) res = wall_rule(W, D, D == 0 ? i : (D == 1 ? j : k), s[D], res) * vol[u];
      }
      vol[u] = res;
    }
#pragma unroll
  for (int u = 0; u < kVZ; ++u) // (the stores last, as in k_vf_mom_op)
    if (u < t.nk) op[i + j * sx + (size_t)(t.k0 + u) * sxy] = vol[u];
}

template <bool FACES>
__global__ void __launch_bounds__(kNT) k_vf_curl(VF3 out, VF3 in, StagCoefs C, VF3 aux, double c, WallVol W, VfGrid g,
                                                const int *gate) {
  if (gate && *gate) return;
  if (blockIdx.y == 0) vf_curl_block<0, FACES>(out, in, C, aux, c, W, g);
  else if (blockIdx.y == 1) vf_curl_block<1, FACES>(out, in, C, aux, c, W, g);
  else vf_curl_block<2, FACES>(out, in, C, aux, c, W, g);
}

// modify_RHS_VF and the set-up: r = vol ((b - A x_BC) - A x) with the wall
// rules, p = z = Minv r, partials of (r,r), (r,z).  has_bc = 0: x_BC is zero
// everywhere, and so is A x_BC.  A x_BC counts as 0 on the ghost planes of the
// faces in ghosts[d] (bit f: face f).
struct GhostMask {
  int m[3];
};
__global__ void __launch_bounds__(kNT) k_vf_rhs(VF3 r, VF3 p, VF3 b, VF3 Abc, VF3 Ax, VF3 M, WallVol W, GhostMask gm,
                                               int has_bc, int excl, double *part) {
  __shared__ double sh[kNT / kWave];
  const int d = blockIdx.y;
  const int s[3] = {r.s[d][0], r.s[d][1], r.s[d][2]};
  const int m = gm.m[d];
  double a_rr = 0.0, a_rz = 0.0;
  auto element = [&](size_t o, int i, int j, int k, bool dot) {
    const bool ghost = ((m & 1) && i == 0) || ((m & 2) && i == s[0] - 1) || ((m & 4) && j == 0) ||
                       ((m & 8) && j == s[1] - 1) || ((m & 16) && k == 0) || ((m & 32) && k == s[2] - 1);
    double v = b.p[d][o];
    if (has_bc) v = v - (ghost ? 0.0 : Abc.p[d][o]);
    v = v - Ax.p[d][o];
    v = v * W.vol[d][o];
    const int pd = d == 0 ? i : (d == 1 ? j : k);
    v = wall_rule(W, d, pd, s[d], v);
    r.p[d][o] = v;
    const double z = M.p[d][o] * v;
    p.p[d][o] = z;
    if (dot && in_dot(excl, d, s[d], pd)) {
      a_rr += v * v;
      a_rz += v * z;
    }
  };
  dot_map(s, d, [&](size_t o, int i, int j, int k) { element(o, i, j, k, true); });
  ghost_map(s, [&](size_t o, int i, int j, int k) { element(o, i, j, k, false); });
  put_dot(a_rr, 0, part, sh);
  put_dot(a_rz, 1, part, sh);
}

// Set-up exit test (PCG_solver_algorithm.f90:130-140), one block.
__global__ void __launch_bounds__(kNT) k_vf_init(VfCtrl *ctrl, const double *part, int nb) {
  double two[2];
  dot_totals<2>(part, nb, two);
  if (threadIdx.x != 0) return;
  ctrl->res0 = sqrt(two[0]);
  ctrl->rho[0] = two[1];
  const double res = sqrt(fabs(two[1]));
  ctrl->res = res;
  const bool e1 = res / ctrl->res0 < ctrl->tol_rel, e2 = res < ctrl->tol_abs, e3 = 0 >= ctrl->iter_max;
  ctrl->exit_loop = (e1 ? 1 : 0) | (e2 ? 2 : 0) | (e3 ? 4 : 0);
  ctrl->iter = e2 ? 1 : 0;
  ctrl->done = e2 ? 1 : 0;
}

// alpha = rho/(p,Ax); x = x + p*alpha; r = r + Ax*(-alpha); partials (r,r), (Minv r, r).
// One pass where x and r, z = Minv r and the two dot products were four kernels
// (48 + 26 + 2 x 18 us at 128^3, now 76: seven arrays of 50 MB, beyond the
// last-level cache, at 4.6 TB/s).
__global__ void __launch_bounds__(kNT) k_vf_update(VF3 x, VF3 p, VF3 r, VF3 Ax, VF3 M, VfCtrl *ctrl,
                                                  const double *partA, double *partB, int excl, int it) {
  if (ctrl->done) return;
  __shared__ double sh[kNT / kWave];
  const int d = blockIdx.y;
  const int s[3] = {r.s[d][0], r.s[d][1], r.s[d][2]};
  double *__restrict__ xd = x.p[d];
  double *__restrict__ rd = r.p[d];
  const double *__restrict__ pd = p.p[d];
  const double *__restrict__ ad = Ax.p[d];
  const double *__restrict__ md = M.p[d];
  double pq[1];
  dot_totals<1>(partA, gridDim.x, pq);
  const double alpha = ctrl->rho[(it - 1) & 1] / pq[0], malpha = -alpha;
  if (blockIdx.x == 0 && d == 0 && threadIdx.x == 0) {
    ctrl->pq = pq[0];
    ctrl->alpha = alpha;
  }
  double a_rr = 0.0, a_rz = 0.0;
  dot_map(s, d, [&](size_t o, int i, int j, int k) {
    xd[o] = xd[o] + pd[o] * alpha;
    const double rn = rd[o] + ad[o] * malpha;
    rd[o] = rn;
    const double z = md[o] * rn;
    if (in_dot(excl, d, s[d], d == 0 ? i : (d == 1 ? j : k))) {
      a_rr += rn * rn;
      a_rz += z * rn;
    }
  });
  ghost_map(s, [&](size_t o, int, int, int) {
    xd[o] = xd[o] + pd[o] * alpha;
    rd[o] = rd[o] + ad[o] * malpha;
  });
  put_dot(a_rr, 0, partB, sh);
  put_dot(a_rz, 1, partB, sh);
}

// Exit test of iteration `it`, then p = p*beta + Minv r.  Block 0 publishes.
__global__ void __launch_bounds__(kNT) k_vf_pupdate(VF3 p, VF3 r, VF3 M, VfCtrl *ctrl, const double *partB, int nb,
                                                   int it) {
  if (ctrl->done) return;
  const int d = blockIdx.y;
  double *__restrict__ pd = p.p[d];
  const double *__restrict__ rd = r.p[d];
  const double *__restrict__ md = M.p[d];
  double two[2];
  dot_totals<2>(partB, nb, two);
  const double rr = two[0], rz = two[1], rho_old = ctrl->rho[(it - 1) & 1];
  const double beta = rz / rho_old;
  const double res = sqrt(fabs(rr));
  const bool check = it % ctrl->n_skip == 0, last = it >= ctrl->iter_max;
  const bool e1 = check && res / ctrl->res0 < ctrl->tol_rel, e2 = check && res < ctrl->tol_abs;
  if (blockIdx.x == 0 && d == 0 && threadIdx.x == 0) {
    ctrl->iter = it;
    ctrl->rr = rr;
    if (check) {
      ctrl->res = res;
      ctrl->exit_loop = (e1 ? 1 : 0) | (e2 ? 2 : 0) | (last ? 4 : 0);
    } else if (last) {
      ctrl->exit_loop |= 4;
    }
    ctrl->rz = rz;
    ctrl->beta = beta;
    ctrl->rho[it & 1] = rz;
    if (e1 || e2 || last) ctrl->done = 1;
  }
  if (e1 || e2 || last) return;
  const unsigned n = (unsigned)p.n[d], step = gridDim.x * kNT;
#pragma unroll 4
  for (unsigned t = blockIdx.x * kNT + threadIdx.x; t < n; t += step) {
    const double z = md[t] * rd[t];
    pd[t] = pd[t] * beta + z;
  }
}

// x_BC's cells: zero, three components in one launch
__global__ void __launch_bounds__(kNT) k_vf_zero(VF3 v) {
  const int d = blockIdx.y;
  const size_t t = (size_t)blockIdx.x * kNT + threadIdx.x;
  if (t < v.n[d]) v.p[d][t] = 0.0;
}

// zero the ghost planes (0 and s - 1) normal to each component, but for periodic faces (mask bit 2d + side)
__global__ void __launch_bounds__(kNT) k_vf_zero_planes(VF3 v, int mask) {
  const int d = blockIdx.y, side = blockIdx.z;
  if (!((mask >> (2 * d + side)) & 1)) return;
  const int *s = v.s[d];
  const int a = (d + 1) % 3, b = (d + 2) % 3;
  const int t = blockIdx.x * kNT + threadIdx.x;
  if (t >= s[a] * s[b]) return;
  int q[3];
  q[d] = side ? s[d] - 1 : 0;
  q[a] = t % s[a];
  q[b] = t / s[a];
  v.p[d][(size_t)q[0] + (size_t)s[0] * ((size_t)q[1] + (size_t)s[1] * q[2])] = 0.0;
}

} // namespace moons

using namespace moons;

struct moons_pcgvf_s {
  moons_mesh_s *m = nullptr;
  int kind = 0;
  double c = 0.0;
  int iter_max = 1000, n_skip = 1;
  double tol_rel = 1e-6, tol_abs = 1e-13;
  moons_field_s bcs[3];                     // locations and BCs of x (no storage)
  moons_field_s *r[3] = {}, *p[3] = {}, *Ax[3] = {}, *Abc[3] = {}, *xbc[3] = {}, *vol[3] = {}, *Minv[3] = {};
  moons_field_s *k[3] = {};                 // sigmaInv on edges (induction)
  moons_field_s *E[3] = {};                 // edge work (induction)
  double *part = nullptr;                   // block sums: of (p,Ax) (3 nb), then of (r,r) and (z,r) (6 nb)
  VfGrid g{};
  int ng = 0;                               // blocks a component of the operators
  int nb = 0;                               // and of the kernels with dot products
  int excl = 0;
  VfCtrl *ctrl = nullptr, *host = nullptr, *host_init = nullptr; // pinned: read-backs, initial block
  bool minv_ready = false;
  hipEvent_t ev0 = nullptr, ev1 = nullptr;
};

static void vf_free(moons_pcgvf_s *S) {
  moons_field_s **all[] = {S->r, S->p, S->Ax, S->Abc, S->xbc, S->vol, S->Minv, S->k, S->E};
  for (auto arr : all)
    for (int d = 0; d < 3; ++d)
      if (arr[d]) moons_field_destroy(arr[d]);
  if (S->part) (void)hipFree(S->part);
  if (S->ctrl) (void)hipFree(S->ctrl);
  if (S->host) (void)hipHostFree(S->host);
  if (S->host_init) (void)hipHostFree(S->host_init);
  if (S->ev0) (void)hipEventDestroy(S->ev0);
  if (S->ev1) (void)hipEventDestroy(S->ev1);
  delete S;
}

// Fields of the solver carry x's BCs (p is x's copy in the reference).
static void copy_bcs(moons_field_s *dst, const moons_field_s &src) { copy_bcs_of(dst, &src); }

// Minv of prec_mom_VF / prec_ind_VF computed on the host in the reference's
// operation order (laplacian_diagonal / curl_curl_diagonal, *c, +1, *vol, 1/x,
// ghosts zeroed), then uploaded.
static int vf_minv(moons_pcgvf_s *S) {
  const HostCoords *C = S->m->hc;
  std::vector<double> sig[3];
  int ss[3][3];
  const int edl[3] = {MOONS_DL_EDGE_X, MOONS_DL_EDGE_Y, MOONS_DL_EDGE_Z};
  if (S->kind == 2) {
    for (int d = 0; d < 3; ++d) {
      sig[d].resize(S->k[d]->n);
      int st = moons_field_download(S->k[d], sig[d].data(), S->k[d]->n);
      if (st) return st;
      for (int e = 0; e < 3; ++e) ss[d][e] = ((edl[d] >> e) & 1) ? C[e].sn : C[e].sc;
    }
  }
  for (int d = 0; d < 3; ++d) {
    const int dl = 1 << d;
    int s[3];
    for (int e = 0; e < 3; ++e) s[e] = ((dl >> e) & 1) ? C[e].sn : C[e].sc;
    const size_t n = (size_t)s[0] * s[1] * s[2];
    std::vector<double> M(n, 0.0);
    auto I3 = [&](const int *sh, int i, int j, int k) { return (size_t)i + (size_t)sh[0] * ((size_t)j + (size_t)sh[1] * k); };
    const int p0 = (dl >> 0) & 1, p1 = (dl >> 1) & 1, p2 = (dl >> 2) & 1;
    for (int k = 1; k < s[2] - 1; ++k)
      for (int j = 1; j < s[1] - 1; ++j)
        for (int i = 1; i < s[0] - 1; ++i) {
          double dg;
          if (S->kind == 1) {
            dg = C[0].n2cc_D[i] * C[0].cc2n_U[i - 1] + C[0].n2cc_U[i - p0] * C[0].cc2n_D[i - p0] +
                 C[1].n2cc_D[j] * C[1].cc2n_U[j - 1] + C[1].n2cc_U[j - p1] * C[1].cc2n_D[j - p1] +
                 C[2].n2cc_D[k] * C[2].cc2n_U[k - 1] + C[2].n2cc_U[k - p2] * C[2].cc2n_D[k - p2];
          } else if (d == 0) {
            dg = -C[1].n2cc_D[j] * sig[2][I3(ss[2], i, j, k)] * C[1].cc2n_U[j - 1] -
                 C[1].n2cc_U[j] * sig[2][I3(ss[2], i, j + 1, k)] * C[1].cc2n_D[j] -
                 C[2].n2cc_D[k] * sig[1][I3(ss[1], i, j, k)] * C[2].cc2n_U[k - 1] -
                 C[2].n2cc_U[k] * sig[1][I3(ss[1], i, j, k + 1)] * C[2].cc2n_D[k];
          } else if (d == 1) {
            dg = -C[0].n2cc_D[i] * sig[2][I3(ss[2], i, j, k)] * C[0].cc2n_U[i - 1] -
                 C[0].n2cc_U[i] * sig[2][I3(ss[2], i + 1, j, k)] * C[0].cc2n_D[i] -
                 C[2].n2cc_D[k] * sig[0][I3(ss[0], i, j, k)] * C[2].cc2n_U[k - 1] -
                 C[2].n2cc_U[k] * sig[0][I3(ss[0], i, j, k + 1)] * C[2].cc2n_D[k];
          } else {
            dg = -C[0].n2cc_D[i] * sig[1][I3(ss[1], i, j, k)] * C[0].cc2n_U[i - 1] -
                 C[0].n2cc_U[i] * sig[1][I3(ss[1], i + 1, j, k)] * C[0].cc2n_D[i] -
                 C[1].n2cc_D[j] * sig[0][I3(ss[0], i, j, k)] * C[1].cc2n_U[j - 1] -
                 C[1].n2cc_U[j] * sig[0][I3(ss[0], i, j + 1, k)] * C[1].cc2n_D[j];
          }
          const double *dh0 = p0 ? C[0].dhc.data() : C[0].dhn.data();
          const double *dh1 = p1 ? C[1].dhc.data() : C[1].dhn.data();
          const double *dh2 = p2 ? C[2].dhc.data() : C[2].dhn.data();
          const double vol = dh0[i - p0] * dh1[j - p1] * dh2[k - p2];
          double v = dg * S->c;
          v = v + 1.0;
          v = v * vol;
          M[I3(s, i, j, k)] = 1.0 / v;
        }
    int st = moons_field_upload(S->Minv[d], M.data(), n);
    if (st) return st;
  }
  return MOONS_OK;
}

static inline size_t vmax(moons_field_s *const f[3]) { return std::max(f[0]->n, std::max(f[1]->n, f[2]->n)); }

// Wall planes of the boundary-normal component: multiply_wall_Neumann(0.5),
// assign_wall_Dirichlet(0), assign_wall_Periodic_single(0)
// (code/handwritten/block_field/block_field_extend.f90:273-377).
static WallVol vf_walls(const moons_pcgvf_s *S) {
  WallVol W{};
  W.on = 1;
  for (int d = 0; d < 3; ++d) {
    const moons_field_s &b = S->bcs[d];
    W.vol[d] = S->vol[d]->d;
    auto rule = [](int t) { return t == MOONS_BC_DIRICHLET ? 1 : (t == MOONS_BC_NEUMANN ? 2 : 0); };
    W.lo[d] = rule(b.bct[2 * d]);
    W.hi[d] = rule(b.bct[2 * d + 1]);
    W.per[d] = b.bct[2 * d] == MOONS_BC_PERIODIC && b.bct[2 * d + 1] == MOONS_BC_PERIODIC && b.s[d] > 4;
  }
  return W;
}

// Ax = A x (implicit BCs on x first when implicit_); loop: with the wall-plane
// rules and the volume product.
static int vf_op(moons_pcgvf_s *S, moons_field_s *Ax[3], moons_field_s *x[3], bool implicit_, bool loop = false) {
  int st;
  if (implicit_ && (st = launch_apply_bcs3(x, true))) return st;
  StagCoefs C;
  for (int e = 0; e < 3; ++e) {
    const DirCoefDev &cd = S->m->dev.c[e];
    C.cc2n_D[e] = cd.cc2n_D; C.cc2n_U[e] = cd.cc2n_U;
    C.n2cc_D[e] = cd.n2cc_D; C.n2cc_U[e] = cd.n2cc_U;
  }
  const WallVol W = loop ? vf_walls(S) : WallVol{};
  const int *gate = current_gate();
  const dim3 grid(S->ng, 3), blk(kNT);
  if (S->kind == 1) {
    hipLaunchKernelGGL(k_vf_mom_op, grid, blk, 0, stream(), vf3(Ax), vf3(x), C, S->c, W, S->g, gate);
  } else {
    // E = k curl(x), then Ax = x + c curl(E)
    hipLaunchKernelGGL(k_vf_curl<false>, grid, blk, 0, stream(), vf3(S->E), vf3(x), C, vf3(S->k), 0.0, WallVol{}, S->g,
                       gate);
    hipLaunchKernelGGL(k_vf_curl<true>, grid, blk, 0, stream(), vf3(Ax), vf3(S->E), C, vf3(x), S->c, W, S->g, gate);
  }
  MOONS_LAUNCH_CHECK();
  return MOONS_OK;
}

extern "C" {

int moons_pcg_vf_create(moons_mesh_t m, int op, moons_field_t x[3], moons_field_t k[3], moons_pcgvf_t *out) {
  if (!stream()) return fail(MOONS_ERR_STATE, "moons_init has not been called");
  if (!m || !x || !out) return fail(MOONS_ERR_ARG, "moons_pcg_vf_create: null argument");
  if (op != MOONS_OP_MOM_DIFFUSION && op != MOONS_OP_IND_DIFFUSION)
    return fail(MOONS_ERR_ARG, "moons_pcg_vf_create: operator must be mom_diffusion or ind_diffusion");
  for (int d = 0; d < 3; ++d)
    if (!x[d] || x[d]->dl != (1 << d) || x[d]->m != m)
      return fail(MOONS_ERR_ARG, "moons_pcg_vf_create: x must be the three face components on this mesh");
  for (int d = 0; d < 3; ++d)
    if (x[d]->n >= ((size_t)1 << 31))
      return fail(MOONS_ERR_ARG, "moons_pcg_vf_create: fields of 2^31 or more elements are not supported");
  if (op == MOONS_OP_IND_DIFFUSION) {
    const int edl[3] = {MOONS_DL_EDGE_X, MOONS_DL_EDGE_Y, MOONS_DL_EDGE_Z};
    if (!k) return fail(MOONS_ERR_ARG, "moons_pcg_vf_create: ind_diffusion needs sigmaInv on edges");
    for (int d = 0; d < 3; ++d)
      if (!k[d] || k[d]->dl != edl[d]) return fail(MOONS_ERR_ARG, "moons_pcg_vf_create: k must be on edges x,y,z");
  }
  moons_pcgvf_s *S = new moons_pcgvf_s();
  S->m = m;
  S->kind = op;
  int st = MOONS_OK;
  for (int d = 0; d < 3 && !st; ++d) {
    S->bcs[d] = *x[d];
    S->bcs[d].d = nullptr;
    moons_field_s **vecs[] = {S->r, S->p, S->Ax, S->Abc, S->xbc, S->vol, S->Minv};
    for (auto v : vecs)
      if (!st) st = moons_field_create(m, 1 << d, &v[d]);
    if (!st) {
      copy_bcs(S->p[d], *x[d]);
      copy_bcs(S->xbc[d], *x[d]);
      copy_bcs(S->Ax[d], *x[d]);
      st = moons_volume(S->vol[d]);
    }
  }
  if (!st && op == MOONS_OP_IND_DIFFUSION) {
    const int edl[3] = {MOONS_DL_EDGE_X, MOONS_DL_EDGE_Y, MOONS_DL_EDGE_Z};
    for (int d = 0; d < 3 && !st; ++d) {
      st = moons_field_create(m, edl[d], &S->k[d]);
      if (!st) st = moons_field_copy(S->k[d], k[d]);
      if (!st) st = moons_field_create(m, edl[d], &S->E[d]);
    }
  }
  if (st) {
    vf_free(S);
    return st;
  }
  {
    // tiles over the largest plane of any component or edge field (node counts)
    S->g.nt = (m->hc[0].sn * m->hc[1].sn + kNT - 1) / kNT;
    S->ng = S->g.nt * ((m->hc[2].sn + kVZ - 1) / kVZ);
    S->nb = (int)std::min<size_t>(1024, (vmax(S->r) + kNT - 1) / kNT);
  }
  for (int d = 0; d < 3; ++d)
    for (int side = 0; side < 2; ++side)
      if (x[d]->has_bcs && x[d]->bct[2 * d + side] == MOONS_BC_DIRICHLET) S->excl |= 1 << (2 * d + side);
  bool ok = hipMalloc(&S->part, 9 * (size_t)S->nb * sizeof(double)) == hipSuccess &&
            hipMalloc(&S->ctrl, sizeof(VfCtrl)) == hipSuccess &&
            hipHostMalloc(&S->host, sizeof(VfCtrl), hipHostMallocDefault) == hipSuccess &&
            hipHostMalloc(&S->host_init, sizeof(VfCtrl), hipHostMallocDefault) == hipSuccess &&
            hipEventCreate(&S->ev0) == hipSuccess && hipEventCreate(&S->ev1) == hipSuccess;
  if (!ok) {
    vf_free(S);
    return fail(MOONS_ERR_HIP, "moons_pcg_vf_create: allocation failed");
  }
  (void)hipMemsetAsync(S->ctrl, 0, sizeof(VfCtrl), stream());
  std::memset(S->host_init, 0xff, sizeof(VfCtrl));
  *out = S;
  return MOONS_OK;
}

int moons_pcg_vf_destroy(moons_pcgvf_t S) {
  if (!S) return MOONS_OK;
  if (stream()) (void)hipStreamSynchronize(stream());
  vf_free(S);
  return MOONS_OK;
}

int moons_pcg_vf_set_isp(moons_pcgvf_t S, int iter_max, double tol_rel, double tol_abs, int n_skip_check_res) {
  if (!S || iter_max < 1 || n_skip_check_res < 1) return fail(MOONS_ERR_ARG, "moons_pcg_vf_set_isp: bad argument");
  S->iter_max = iter_max;
  S->tol_rel = tol_rel;
  S->tol_abs = tol_abs;
  S->n_skip = n_skip_check_res;
  return MOONS_OK;
}

int moons_pcg_vf_update_mfp(moons_pcgvf_t S, double coeff_implicit_time_split, int update_preconditioner) {
  if (!S) return fail(MOONS_ERR_ARG, "moons_pcg_vf_update_mfp: null solver");
  const bool changed = S->c != coeff_implicit_time_split;
  S->c = coeff_implicit_time_split;
  // Minv depends on c and the mesh only: rebuilding it for an unchanged c
  // would reproduce the same array
  if (update_preconditioner && (changed || !S->minv_ready)) {
    if (sync_free()) return fail(MOONS_ERR_STATE, "moons_pcg_vf_update_mfp: a new coefficient cannot be set inside a graph");
    const int st = vf_minv(S);
    if (st) return st;
    S->minv_ready = true;
  }
  return MOONS_OK;
}

int moons_pcg_vf_solve(moons_pcgvf_t S, moons_field_t x[3], moons_field_t b[3], moons_pcg_info *info) {
  if (!S || !x || !b) return fail(MOONS_ERR_ARG, "moons_pcg_vf_solve: null argument");
  for (int d = 0; d < 3; ++d)
    if (!x[d] || !b[d] || x[d]->dl != (1 << d) || b[d]->dl != (1 << d) || x[d]->m != S->m || b[d]->m != S->m)
      return fail(MOONS_ERR_ARG, "moons_pcg_vf_solve: x and b must be face components on the solver's mesh");
  VfCtrl h;
  std::memset(&h, 0, sizeof(VfCtrl));
  h.iter_max = S->iter_max;
  h.n_skip = S->n_skip;
  h.tol_rel = S->tol_rel;
  h.tol_abs = S->tol_abs;
  if (std::memcmp(&h, S->host_init, sizeof(VfCtrl)) != 0) {
    if (!sync_free()) MOONS_HIP(hipStreamSynchronize(stream()));
    *S->host_init = h;
  }
  MOONS_HIP(hipMemcpyAsync(S->ctrl, S->host_init, sizeof(VfCtrl), hipMemcpyHostToDevice, stream()));
  const bool nosync = sync_free();
  if (!nosync) MOONS_HIP(hipEventRecord(S->ev0, stream()));
  // the solve's x carries its own BCs; keep a copy with x's BCs for the implicit application
  moons_field_s xs[3];
  moons_field_s *xp[3];
  for (int d = 0; d < 3; ++d) {
    xs[d] = *x[d];
    xp[d] = &xs[d];
  }
  int st;
  const int *done = &S->ctrl->done;
  double *partA = S->part, *partB = S->part + 3 * (size_t)S->nb;
  const dim3 grid(S->nb, 3), blk(kNT);
  set_gate(done);
  // ---- modify_RHS_VF and the set-up.  x_BC is zero inside with ghosts from
  // the BC values; with no value set it is zero everywhere and A x_BC with it.
  bool has_bc = false;
  GhostMask gm{};
  int planes = 0;
  for (int d = 0; d < 3; ++d)
    for (int f = 0; f < 6; ++f) {
      const bool per = S->xbc[d]->has_bcs && S->xbc[d]->bct[f] == MOONS_BC_PERIODIC;
      has_bc = has_bc || (S->xbc[d]->has_bcs && S->xbc[d]->bval[f] != 0.0);
      if (!per) gm.m[d] |= 1 << f;
      if (f / 2 == d && S->xbc[d]->bct[f] != MOONS_BC_PERIODIC) planes |= 1 << f;
    }
  if (has_bc) {
    hipLaunchKernelGGL(k_vf_zero, dim3((unsigned)((vmax(S->xbc) + kNT - 1) / kNT), 3), blk, 0, stream(), vf3(S->xbc));
    if ((st = launch_apply_bcs3(S->xbc, false))) goto out;
    const int *n = S->m->dev.sn;
    const int pmax = std::max(n[0] * n[1], std::max(n[1] * n[2], n[0] * n[2]));
    hipLaunchKernelGGL(k_vf_zero_planes, dim3((pmax + kNT - 1) / kNT, 3, 2), blk, 0, stream(), vf3(S->xbc), planes);
    if ((st = vf_op(S, S->Abc, S->xbc, false))) goto out;
  }
  if ((st = vf_op(S, S->Ax, xp, true))) goto out;
  hipLaunchKernelGGL(k_vf_rhs, grid, blk, 0, stream(), vf3(S->r), vf3(S->p), vf3(b), vf3(S->Abc), vf3(S->Ax),
                     vf3(S->Minv), vf_walls(S), gm, has_bc ? 1 : 0, S->excl, partB);
  hipLaunchKernelGGL(k_vf_init, dim3(1), blk, 0, stream(), S->ctrl, partB, S->nb);
  {
    int launched = 0;
    for (;;) {
      if (nosync) {
        if (launched >= S->iter_max) break;
      } else {
        MOONS_HIP(hipMemcpyAsync(S->host, S->ctrl, sizeof(VfCtrl), hipMemcpyDeviceToHost, stream()));
        MOONS_HIP(hipStreamSynchronize(stream()));
        if (S->host->done || launched >= S->iter_max) break;
      }
      // the first chunk covers a preset solve (a few iterations) without a read-back in between
      int chunk = nosync ? S->iter_max : std::min(launched == 0 ? 5 : std::max(2, std::min(16, launched / 4)), S->iter_max - launched);
      for (int c = 0; c < chunk; ++c) {
        const int it = launched + c + 1;
        if ((st = vf_op(S, S->Ax, S->p, true, true))) goto out; // with the wall rules and vol
        hipLaunchKernelGGL(k_vf_dot, grid, blk, 0, stream(), vf3(S->p), vf3(S->Ax), S->excl, partA, done);
        hipLaunchKernelGGL(k_vf_update, grid, blk, 0, stream(), vf3(xp), vf3(S->p), vf3(S->r), vf3(S->Ax), vf3(S->Minv),
                           S->ctrl, partA, partB, S->excl, it);
        hipLaunchKernelGGL(k_vf_pupdate, grid, blk, 0, stream(), vf3(S->p), vf3(S->r), vf3(S->Minv), S->ctrl, partB,
                           S->nb, it);
        MOONS_LAUNCH_CHECK();
      }
      launched += chunk;
    }
  }
  set_gate(nullptr);
  // apply_BCs(x) after the last update (PCG_solver_algorithm.f90:149,170)
  if ((st = launch_apply_bcs3(x, false))) return st;
  if (nosync) {
    if (info) {
      info->iterations = -1;
      info->exit_loop = 0;
      info->res_norm0 = info->res_norm = info->ms = 0.0;
    }
    return MOONS_OK;
  }
  MOONS_HIP(hipEventRecord(S->ev1, stream()));
  MOONS_HIP(hipMemcpyAsync(S->host, S->ctrl, sizeof(VfCtrl), hipMemcpyDeviceToHost, stream()));
  MOONS_HIP(hipStreamSynchronize(stream()));
  if (std::isnan(S->host->res) || std::isnan(S->host->res0))
    return fail(MOONS_ERR_NAN, "Error: NaN in PCG residual (check_nans, PCG_solver_algorithm.f90:223-248)");
  if (info) {
    info->iterations = S->host->iter;
    info->exit_loop = S->host->exit_loop;
    info->res_norm0 = S->host->res0;
    info->res_norm = S->host->res;
    float ms = 0.f;
    (void)hipEventElapsedTime(&ms, S->ev0, S->ev1);
    info->ms = ms;
  }
  return MOONS_OK;
out:
  set_gate(nullptr);
  return st;
}

} // extern "C"
