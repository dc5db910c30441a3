// pcg_resident.hpp -- the Jacobi-PCG loop of a small or medium grid as ONE
// kernel that stays resident: every block owns a box of cells and keeps its
// x, r, p, q and Minv in registers (p in LDS as well, for the x and y
// neighbours), so an iteration moves only box surfaces and two block sums.
//
// Included by pcg.hip, after the operator helpers.
//
// What bounds it: the launch-per-kernel loop reads or writes 88 B per cell and
// iteration and pays three kernel starts.  Here an iteration is two all-reduces
// over the blocks (about 2.8 and 3.6 us at 256 blocks, 1.4 us each at 16), the
// halo's loads and the arithmetic of the block's cells.  Measured, us an
// iteration before -> now: 16^3 17.0 -> 4.6, 32^3 19.2 -> 5.7, 64^3 18.5 -> 9.0,
// 96^3 32.3 -> 11.9, 128^3 48.9 -> 16.4.
//
// Box: whole x rows (n0), `by` rows, CPT planes; a thread owns one (i, j)
// column of CPT cells, so its z neighbours are its own registers, and the x
// and y stencil coefficients stay in registers for the whole solve.
//
// Exchange without a third synchronisation: the neighbours' p is not sent.
// After the r update each block publishes its surface r (before the (r,r),
// (r,z) sum, which orders it), and each block forms p = p beta + Minv r of the
// halo cells itself, with the owner's operands and order, so the same bits.
//
// All-reduce: every block stores its sum in its slot (an 8-byte agent-scope
// atomic, the surface stores complete before it) and thread t of every block
// polls slot t, so one hop; the sums are then added in slot order, the same in
// every block.  A slot holds kSlotEmpty until its sum arrives (a NaN result is
// stored in the canonical pattern).  Slots alternate between two sets by
// iteration parity; a block empties its slot of one sum after the next sum has
// completed (then every block has read it), and the emptying store completes
// before the block's next publication, after which alone the slot is polled
// again.  Counters with an agent-scope fence cost 33 us a round at 256 blocks
// (the fence writes back and invalidates the whole L2), so all shared data go
// through agent-scope atomics and there is no fence.
//
// Residency: the grid never exceeds the number of CUs, one block a CU, and it
// runs on the library's one stream only (never in a captured graph, whose
// replays may share the GPU with each other: there the kernels at the end of
// this file do the same sums a launch at a time).  Should blocks nevertheless not
// all be resident, every wait is bounded: a block that gives up sets `abort`,
// the others see it while they wait, every block returns, x is untouched (the
// result goes to a buffer that k_pcg_take copies only from a complete run),
// and the host solves again with the launch-per-kernel loop, and with it only
// from then on.
#pragma once

namespace moons {

constexpr unsigned long long kSlotEmpty = ~0ull;
constexpr int kResMaxBlocks = 256;
// slots: (1 + 2 sums) x 2 sets x blocks, then the abort word
constexpr size_t kResSlotWords = (size_t)6 * kResMaxBlocks + 1;

struct ResPlan {
  int cpt = 0;    // planes a block (0: not eligible)
  int by, gy, gz; // rows a block, blocks along y and z
  size_t lds;     // dynamic LDS bytes
  int nb() const { return gy * gz; }
};

__device__ __forceinline__ void agent_store(unsigned long long *p, unsigned long long v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ unsigned long long agent_load(const unsigned long long *p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void agent_store(double *p, double v) {
  agent_store(reinterpret_cast<unsigned long long *>(p), (unsigned long long)__double_as_longlong(v));
}
__device__ __forceinline__ double agent_load(const double *p) {
  return __longlong_as_double((long long)agent_load(reinterpret_cast<const unsigned long long *>(p)));
}

template <int CTRL, int ROWS>
__device__ __forceinline__ double dpp_add(double v) {
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, ROWS, 0xf, false);
  const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, ROWS, 0xf, false);
  return v + __hiloint2double(hi, lo);
}
// Sum over the wave in a fixed order, in lane 63 (row shifts by 1, 2, 4, 8,
// then the rows joined): no LDS round trips.  Every lane must be active.
__device__ __forceinline__ double wave_sum63(double v) {
  v = dpp_add<0x111, 0xf>(v);
  v = dpp_add<0x112, 0xf>(v);
  v = dpp_add<0x114, 0xf>(v);
  v = dpp_add<0x118, 0xf>(v);
  v = dpp_add<0x142, 0xa>(v);
  return dpp_add<0x143, 0xc>(v);
}

template <int NT>
struct ResShared {
  double part[2][NT / kWave], all[2][NT / kWave];
  int bad;
};

// The block's sums of v[0..V) (as left in sh.part by every wave), for thread t < V.
template <int NT>
__device__ __forceinline__ double block_total(const ResShared<NT> &sh, int q) {
  double s = 0.0;
#pragma unroll
  for (int u = 0; u < NT / kWave; ++u) s += sh.part[q][u];
  return s;
}
template <int NT, int V>
__device__ __forceinline__ void wave_totals(double (&v)[V], double (&to)[2][NT / kWave]) {
#pragma unroll
  for (int q = 0; q < V; ++q) v[q] = wave_sum63(v[q]);
  if ((threadIdx.x & (kWave - 1)) == kWave - 1) {
#pragma unroll
    for (int q = 0; q < V; ++q) to[q][threadIdx.x / kWave] = v[q];
  }
}
// The sums over nb blocks' values from the waves' sums in sh.all.
template <int NT, int V>
__device__ __forceinline__ void grid_totals(double (&v)[V], const ResShared<NT> &sh, int nb) {
  const int nw = (nb + kWave - 1) / kWave;
#pragma unroll
  for (int q = 0; q < V; ++q) {
    double s = 0.0;
    for (int u = 0; u < nw; ++u) s += sh.all[q][u];
    v[q] = s;
  }
}

// Sums v[0..V) over all blocks (slot set S of V x nb words); false when the
// wait was given up, the same in every thread.  Stores issued before the call
// have completed when the block's slot is published.
template <int NT, int V>
__device__ __forceinline__ bool all_reduce(double (&v)[V], unsigned long long *S, int nb, ResShared<NT> &sh,
                                           unsigned long long *abort_, int spins) {
  const int t = threadIdx.x, w = t / kWave;
  wave_totals<NT, V>(v, sh.part);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  if (t < V) {
    const double s = block_total<NT>(sh, t);
    unsigned long long bits = (unsigned long long)__double_as_longlong(s);
    if (s != s) bits = 0x7ff8000000000000ull;
    agent_store(S + (size_t)t * nb + blockIdx.x, bits);
  }
  if (w * kWave < nb) {
    double a[V];
#pragma unroll
    for (int q = 0; q < V; ++q) a[q] = 0.0;
    if (t < nb) {
      unsigned long long b[V];
      for (int n = 1;; ++n) {
        bool there = true;
#pragma unroll
        for (int q = 0; q < V; ++q) b[q] = agent_load(S + (size_t)q * nb + t);
#pragma unroll
        for (int q = 0; q < V; ++q) there = there && b[q] != kSlotEmpty;
        if (there) break;
        if (n >= spins || ((n & 255) == 0 && agent_load(abort_) != 0)) {
          sh.bad = 1;
          break;
        }
      }
#pragma unroll
      for (int q = 0; q < V; ++q) a[q] = __longlong_as_double((long long)b[q]);
    }
    wave_totals<NT, V>(a, sh.all);
  }
  __syncthreads();
  if (sh.bad) {
    if (t == 0) agent_store(abort_, 1ull);
    return false;
  }
  grid_totals<NT, V>(v, sh, nb);
  return true;
}

// A value the compiler must take as new: keeps addresses formed from it inside
// the iteration, where they cost an addition, instead of in registers across
// the loop, where they would push the cells' vectors into scratch memory.
template <typename T>
__device__ __forceinline__ T opaque(T v) {
  asm volatile("" : "+v"(v));
  return v;
}

__device__ __forceinline__ int opaque_s(int v) { // the same for a value all lanes share
  asm volatile("" : "+s"(v));
  return v;
}

// How a thread reads the neighbour of its boundary cell: the value at an LDS
// offset times a factor (the implicit BC rules: -v, v, or the Robin factor
// times v, all of the cell itself; the far cell when periodic).  A face
// without BCs holds zero ghosts: the zero column 0 of the tile.  Inside, the
// neighbour itself times 1, which is exact.
struct NbRule {
  int off;
  double fac;
};
__device__ __forceinline__ NbRule nb_rule(int type, double rob, int inside, int far, int zero) {
  if (type == MOONS_BC_PERIODIC) return NbRule{far, 1.0};
  if (type == MOONS_BC_NONE) return NbRule{zero, 1.0};
  if (type == MOONS_BC_DIRICHLET || type == MOONS_BC_ANTISYMMETRIC) return NbRule{0, -1.0};
  if (type == MOONS_BC_ROBIN) return NbRule{0, rob};
  return NbRule{0, 1.0};
}
// the factor of a z ghost on the cell's own value (0 ghosts: 0, of a face without BCs)
__device__ __forceinline__ double z_factor(int type, double rob) {
  if (type == MOONS_BC_NONE) return 0.0;
  if (type == MOONS_BC_DIRICHLET || type == MOONS_BC_ANTISYMMETRIC) return -1.0;
  return type == MOONS_BC_ROBIN ? rob : 1.0;
}

// x_out = the solution after the loop started by k_pcg_rhs and k_pcg_init.
// r: its surface cells are overwritten.  Block 0 publishes the control block.
template <int NT, int CPT, bool NRG>
__global__ void __launch_bounds__(NT) k_pcg_resident(const double *__restrict__ x, double *r,
                                                    const double *__restrict__ p, double *__restrict__ x_out, CCGeom G,
                                                    int by, int gy, PcgCtrl *ctrl, unsigned long long *slots,
                                                    int spins, NrgK K) {
  const PcgCtrl C = *ctrl; // the tolerances and the set-up's rho and res
  if (C.done) return;
  extern __shared__ double sp[]; // p, (k, j, i) with one ring of halo in j and i; then Minv of the y halo
  __shared__ ResShared<NT> sh;
  __shared__ double sz[CPT + 1][8]; // cD, cU of the face below plane u; nD, nU, dh, lA, lB of the plane
  // Minv of the cells: kept, or with 16 planes a thread (x, r, p and q alone
  // are 128 registers) divided out anew in each iteration, with the same bits
  constexpr bool kKeep = CPT < 16;
  const int t = threadIdx.x, nb = gridDim.x;
  const int n0 = G.n0, n1 = G.n1, n2 = G.n2;
  const size_t sx = G.s0, sxy = (size_t)G.s0 * G.s1;
  const int L = xcd_remap(blockIdx.x, nb);
  const int j0 = 1 + (L % gy) * by, k0 = 1 + (L / gy) * CPT;
  const int nj = min(by, n1 + 1 - j0), nk = min(CPT, n2 + 1 - k0);
  const int W = n0 + 2, PL = (by + 2) * W;
  double *smv = sp + (size_t)CPT * PL;
  const int jj = t / n0, ii = t - jj * n0;
  const bool active = jj < nj;
  const int i = 1 + ii, j = j0 + (active ? jj : 0);
  const double dxy = G.c[0].dh[i] * G.c[1].dh[j];
  const double axy = G.c[0].lA[i] + G.c[0].lB[i] + G.c[1].lA[j] + G.c[1].lB[j];
  const St6<double> SX = st6(G.c[0], i), SY = st6(G.c[1], j);
  const size_t oij = (size_t)i + (size_t)j * sx, base = oij + (size_t)k0 * sxy;

  // halo cells: real ones (a neighbour's, or the far side's when periodic)
  const bool per_y = G.bct[2] == MOONS_BC_PERIODIC, per_z = G.bct[4] == MOONS_BC_PERIODIC;
  const bool ylo = j0 > 1 || per_y, yhi = j0 + nj <= n1 || per_y;
  const bool zlo = k0 > 1 || per_z, zhi = k0 + nk <= n2 || per_z;
  const int jlo = j0 > 1 ? j0 - 1 : n1, jhi = j0 + nj <= n1 ? j0 + nj : 1;
  const int klo = k0 > 1 ? k0 - 1 : n2, khi = k0 + nk <= n2 ? k0 + nk : 1;
  const int lrow = active ? (jj + 1) * W + i : W + 1; // the thread's first cell in LDS
  const NbRule xm = i > 1 ? NbRule{-1, 1.0} : nb_rule(G.bct[0], G.robc[0], -1, n0 - 1, -i);
  const NbRule xp = i < n0 ? NbRule{1, 1.0} : nb_rule(G.bct[1], G.robc[1], 1, 1 - n0, -i);
  const NbRule ym = j > 1 || per_y ? NbRule{-W, 1.0} : nb_rule(G.bct[2], G.robc[2], -W, -W, -i);
  const NbRule yp = j < n1 || per_y ? NbRule{W, 1.0} : nb_rule(G.bct[3], G.robc[3], W, W, -i);
  const double fzlo = z_factor(G.bct[4], G.robc[4]), fzhi = z_factor(G.bct[5], G.robc[5]);

  for (int q = t; q < CPT * PL; q += NT) sp[q] = 0.0;
  if (t == 0) sh.bad = 0;
  if (t <= nk) {
    sz[t][0] = G.c[2].cD[k0 - 1 + t];
    sz[t][1] = G.c[2].cU[k0 - 1 + t];
    if (t < nk) {
      sz[t][2] = G.c[2].nD[k0 + t];
      sz[t][3] = G.c[2].nU[k0 + t];
      sz[t][4] = G.c[2].dh[k0 + t];
      sz[t][5] = G.c[2].lA[k0 + t];
      sz[t][6] = G.c[2].lB[k0 + t];
    }
  }
  __syncthreads();

  double xv[CPT], rv[CPT], pv[CPT], mv[kKeep ? CPT : 1];
#pragma unroll
  for (int u = 0; u < CPT; ++u) {
    xv[u] = rv[u] = pv[u] = 0.0;
    if (kKeep) mv[u] = 0.0;
    if (active && u < nk) {
      const size_t o = base + (size_t)u * sxy;
      xv[u] = x[o];
      rv[u] = r[o];
      pv[u] = p[o];
      if (kKeep) mv[u] = minv_at<double>(G, dxy, axy, k0 + u);
      sp[lrow + u * PL] = pv[u];
    }
  }
  double mzlo = 0.0, mzhi = 0.0, pzlo = 0.0, pzhi = 0.0;
  if (active && zlo) {
    mzlo = minv_at<double>(G, dxy, axy, klo);
    pzlo = p[oij + (size_t)klo * sxy];
  }
  if (active && zhi) {
    mzhi = minv_at<double>(G, dxy, axy, khi);
    pzhi = p[oij + (size_t)khi * sxy];
  }
  // y halo rows: row q (side, plane) of 2 nk, cell h of n0, over the block's threads
  const int hq0 = t / n0, hi0 = t - hq0 * n0, dq = NT / n0, di = NT - dq * n0;
  auto next_halo = [&](int &q, int &h) {
    q += dq;
    h += di;
    if (h >= n0) {
      h -= n0;
      ++q;
    }
  };
  for (int q = hq0, h = hi0; q < 2 * nk; next_halo(q, h)) {
    const bool hiside = q >= nk;
    const int u = hiside ? q - nk : q;
    if (hiside ? yhi : ylo) {
      const int jr = hiside ? jhi : jlo, ir = h + 1, kr = k0 + u;
      const double dxyr = G.c[0].dh[ir] * G.c[1].dh[jr];
      const double axyr = G.c[0].lA[ir] + G.c[0].lB[ir] + G.c[1].lA[jr] + G.c[1].lB[jr];
      smv[q * n0 + h] = minv_at<double>(G, dxyr, axyr, kr);
      sp[u * PL + (hiside ? nj + 1 : 0) * W + ir] = p[(size_t)ir + (size_t)jr * sx + (size_t)kr * sxy];
    }
  }
  // z ghosts from the cells next to them
  auto last_plane = [&]() {
    double last = pv[0];
#pragma unroll
    for (int u = 1; u < CPT; ++u) {
      const double v = pv[u];
      last = u == nk - 1 ? v : last;
    }
    return last;
  };
  if (!zlo) pzlo = pv[0] * fzlo;
  if (!zhi) pzhi = last_plane() * fzhi;
  __syncthreads();

  double rho = C.rho[0], res = C.res, rr = 0.0, alpha = 0.0, beta = 0.0, pq = 0.0, rz = 0.0;
  int exit_loop = C.exit_loop;
  unsigned long long *s1 = slots, *s2 = slots + 2 * kResMaxBlocks, *abort_ = slots + 6 * kResMaxBlocks;
  int it = 1;
  for (;; ++it) {
    const int par = it & 1;
    // q = vol A p, (p, q); the z-face gradient is shared by the two cells of the face
    double qv[CPT], acc[1] = {0.0};
#pragma unroll
    for (int u = 0; u < CPT; ++u) qv[u] = 0.0;
    const int nk_ = opaque_s(nk);
    if (active) {
      int at = opaque(lrow);
      double gz = pzlo * sz[0][0] + pv[0] * sz[0][1];
      const double *kx = nullptr, *ky = nullptr, *kz = nullptr;
      if (NRG) {
        kx = opaque(K.k[0] + (size_t)i + (size_t)(G.s0 + 1) * ((size_t)j + (size_t)G.s1 * k0));
        ky = opaque(K.k[1] + (size_t)i + sx * ((size_t)j + (size_t)(G.s1 + 1) * k0));
        kz = opaque(K.k[2] + base);
        gz = gz * kz[0];
      }
#pragma unroll
      for (int u = 0; u < CPT; ++u) {
        if (u < nk_) {
          const double *row = sp + at;
          const double c = pv[u], up = pv[u + 1 < CPT ? u + 1 : u], end = pzhi;
          const double zp = u + 1 < CPT && u + 1 < nk_ ? up : end;
          double gxm = (row[xm.off] * xm.fac) * SX.cDm + c * SX.cUm, gxp = c * SX.cD + (row[xp.off] * xp.fac) * SX.cU;
          double gym = (row[ym.off] * ym.fac) * SY.cDm + c * SY.cUm, gyp = c * SY.cD + (row[yp.off] * yp.fac) * SY.cU;
          double gzp = c * sz[u + 1][0] + zp * sz[u + 1][1];
          if (NRG) {
            kz += sxy;
            gxm = gxm * kx[0];
            gxp = gxp * kx[1];
            gym = gym * ky[0];
            gyp = gyp * ky[sx];
            gzp = gzp * kz[0];
            kx += (size_t)(G.s0 + 1) * G.s1;
            ky += sx * (size_t)(G.s1 + 1);
          }
          double v = gxm * SX.nD + gxp * SX.nU;
          v = v + gym * SY.nD + gyp * SY.nU;
          v = v + gz * sz[u][2] + gzp * sz[u][3];
          if (NRG) {
            v = v * K.c;
            v = v + c;
          }
          gz = gzp;
          qv[u] = v * (dxy * sz[u][4]);
          acc[0] += c * qv[u];
        }
        at += PL;
        // at most four planes' operands in flight: more would not fit the registers
        if ((u & 3) == 3) __builtin_amdgcn_sched_barrier(0);
      }
    }
    if (!all_reduce<NT, 1>(acc, s1 + par * kResMaxBlocks, nb, sh, abort_, spins)) return;
    // the other sum of the last iteration has been read by every block: empty its slots
    if (t < 2 && it > 1) agent_store(s2 + (par ^ 1) * 2 * kResMaxBlocks + (size_t)t * nb + blockIdx.x, kSlotEmpty);
    pq = acc[0];
    alpha = rho / pq;
    const double malpha = -alpha;
    double two[2] = {0.0, 0.0};
    if (active) {
      const bool edge = jj == 0 || jj == nj - 1;
      double *ro = opaque(r + base);
      const int nk_ = opaque_s(nk), top = nk_ - 1;
#pragma unroll
      for (int u = 0; u < CPT; ++u) {
        if (u < nk_) {
          xv[u] = xv[u] + pv[u] * alpha;
          const double rn = rv[u] + qv[u] * malpha;
          rv[u] = rn;
          if (edge || u == 0 || u == top) agent_store(ro, rn);
          two[0] += rn * rn;
          const double m = kKeep ? mv[kKeep ? u : 0] : 1.0 / ((axy + sz[u][5] + sz[u][6]) * (dxy * sz[u][4]));
          qv[u] = m * rn; // z: q is not needed any more
          two[1] += qv[u] * rn;
        }
        ro += sxy;
      }
    }
    if (!all_reduce<NT, 2>(two, s2 + par * 2 * kResMaxBlocks, nb, sh, abort_, spins)) return;
    if (t == 0) agent_store(s1 + par * kResMaxBlocks + blockIdx.x, kSlotEmpty);
    rr = two[0];
    rz = two[1];
    const ExitDecision e = exit_decision(&C, it, rr);
    beta = rz / rho;
    rho = rz;
    if (e.checked) {
      res = e.res;
      exit_loop = e.flags;
    } else if (e.stop) {
      exit_loop |= e.flags;
    }
    if (e.stop) break;
    // p = p beta + Minv r, own cells and halo; the halo's r loads first
    constexpr int HB = CPT >= 8 ? 8 : 4;
    double rh[HB], rlo = 0.0, rhi = 0.0;
    int q = opaque(hq0), h = opaque(hi0);
    {
      const double *rij = opaque(r + oij);
      if (active && zlo) rlo = agent_load(rij + (size_t)klo * sxy);
      if (active && zhi) rhi = agent_load(rij + (size_t)khi * sxy);
    }
    auto halo_load = [&](int qb, int hb) {
#pragma unroll
      for (int m = 0; m < HB; ++m) {
        const bool hiside = qb >= nk;
        rh[m] = 0.0;
        if (qb < 2 * nk && (hiside ? yhi : ylo))
          rh[m] = agent_load(r + (size_t)(hb + 1) + (size_t)(hiside ? jhi : jlo) * sx +
                             (size_t)(k0 + (hiside ? qb - nk : qb)) * sxy);
        next_halo(qb, hb);
      }
    };
    auto halo_update = [&]() {
#pragma unroll
      for (int m = 0; m < HB; ++m) {
        const bool hiside = q >= nk;
        if (q < 2 * nk && (hiside ? yhi : ylo)) {
          double *at = sp + (hiside ? q - nk : q) * PL + (hiside ? nj + 1 : 0) * W + h + 1;
          const double z = smv[q * n0 + h] * rh[m];
          *at = *at * beta + z;
        }
        next_halo(q, h);
      }
    };
    halo_load(q, h);
    {
      int at = opaque(lrow);
      const int nk_ = opaque_s(nk);
#pragma unroll
      for (int u = 0; u < CPT; ++u) {
        pv[u] = pv[u] * beta + qv[u];
        if (active && u < nk_) sp[at] = pv[u];
        at += PL;
      }
    }
    halo_update();
    while (q < 2 * nk) {
      halo_load(q, h);
      halo_update();
    }
    if (zlo) {
      const double z = mzlo * rlo;
      pzlo = pzlo * beta + z;
    }
    if (zhi) {
      const double z = mzhi * rhi;
      pzhi = pzhi * beta + z;
    }
    if (!zlo) pzlo = pv[0] * fzlo;
    if (!zhi) pzhi = last_plane() * fzhi;
    __syncthreads();
  }
  if (active) {
#pragma unroll
    for (int u = 0; u < CPT; ++u)
      if (u < nk) x_out[base + (size_t)u * sxy] = xv[u];
  }
  if (blockIdx.x == 0 && t == 0) {
    ctrl->iter = it;
    ctrl->rr = rr;
    ctrl->res = res;
    ctrl->exit_loop = exit_loop;
    ctrl->pq = pq;
    ctrl->alpha = alpha;
    ctrl->rz = rz;
    ctrl->beta = beta;
    ctrl->rho[it & 1] = rho;
    ctrl->done = kResDone;
  }
}

// ---- the same loop a kernel at a time, for a captured graph: the resident
// loop's boxes, arithmetic and orders of summation, so that a replay equals
// the eager solve bit for bit.  p's face ghosts are kept in memory here.
struct Box {
  int i, j, k0, nk; // the thread's column; nk 0: none
};
__device__ __forceinline__ Box box_of(const CCGeom &G, int by, int gy, int cpt) {
  const int L = xcd_remap(blockIdx.x, gridDim.x), t = threadIdx.x, jj = t / G.n0, j0 = 1 + (L % gy) * by;
  Box b;
  b.i = 1 + t - jj * G.n0;
  b.j = j0 + jj;
  b.k0 = 1 + (L / gy) * cpt;
  b.nk = jj < min(by, G.n1 + 1 - j0) ? min(cpt, G.n2 + 1 - b.k0) : 0;
  return b;
}
// sums of the last kernel's V x nb block sums, the same in every block
template <int NT, int V>
__device__ __forceinline__ void box_sums(double (&v)[V], const double *part, int nb, ResShared<NT> &sh) {
  const int t = threadIdx.x;
#pragma unroll
  for (int q = 0; q < V; ++q) v[q] = t < nb ? part[(size_t)q * nb + t] : 0.0;
  wave_totals<NT, V>(v, sh.all);
  __syncthreads();
  grid_totals<NT, V>(v, sh, nb);
}
template <int NT, int V>
__device__ __forceinline__ void box_put(double (&v)[V], double *part, int nb, ResShared<NT> &sh) {
  wave_totals<NT, V>(v, sh.part);
  __syncthreads();
  if (threadIdx.x < V) part[(size_t)threadIdx.x * nb + blockIdx.x] = block_total<NT>(sh, threadIdx.x);
}

template <int NT, bool NRG>
__global__ void __launch_bounds__(NT) k_box_matvec(const double *__restrict__ p, double *__restrict__ q, CCGeom G, int by,
                                                  int gy, int cpt, const PcgCtrl *ctrl, double *part, NrgK K) {
  if (ctrl->done) return;
  __shared__ ResShared<NT> sh;
  const Box b = box_of(G, by, gy, cpt);
  const size_t sx = G.s0, sxy = (size_t)G.s0 * G.s1;
  double acc[1] = {0.0};
  if (b.nk > 0) {
    const double dxy = G.c[0].dh[b.i] * G.c[1].dh[b.j];
    const St6<double> SX = st6(G.c[0], b.i), SY = st6(G.c[1], b.j);
#pragma unroll 4
    for (int u = 0; u < b.nk; ++u) {
      const int k = b.k0 + u;
      const size_t o = (size_t)b.i + (size_t)b.j * sx + (size_t)k * sxy;
      const double c = p[o];
      const double v = NRG ? nrg7(K, G, c, p[o - 1], p[o + 1], p[o - sx], p[o + sx], p[o - sxy], p[o + sxy], b.i, b.j, k)
                           : lap7s(c, p[o - 1], p[o + 1], p[o - sx], p[o + sx], p[o - sxy], p[o + sxy], SX, SY,
                                   st6(G.c[2], k));
      const double qv = v * (dxy * G.c[2].dh[k]);
      q[o] = qv;
      acc[0] += c * qv;
    }
  }
  box_put<NT, 1>(acc, part, gridDim.x, sh);
}

template <int NT>
__global__ void __launch_bounds__(NT) k_box_update(double *__restrict__ x, const double *__restrict__ p,
                                                  double *__restrict__ r, const double *__restrict__ q, CCGeom G, int by,
                                                  int gy, int cpt, PcgCtrl *ctrl, const double *part1, double *part2,
                                                  int it) {
  if (ctrl->done) return;
  __shared__ ResShared<NT> sh;
  const Box b = box_of(G, by, gy, cpt);
  double pq[1];
  box_sums<NT, 1>(pq, part1, gridDim.x, sh);
  const double alpha = ctrl->rho[(it - 1) & 1] / pq[0], malpha = -alpha;
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    ctrl->pq = pq[0];
    ctrl->alpha = alpha;
  }
  double two[2] = {0.0, 0.0};
  if (b.nk > 0) {
    const size_t sx = G.s0, sxy = (size_t)G.s0 * G.s1;
    const double dxy = G.c[0].dh[b.i] * G.c[1].dh[b.j];
    const double axy = G.c[0].lA[b.i] + G.c[0].lB[b.i] + G.c[1].lA[b.j] + G.c[1].lB[b.j];
#pragma unroll 4
    for (int u = 0; u < b.nk; ++u) {
      const size_t o = (size_t)b.i + (size_t)b.j * sx + (size_t)(b.k0 + u) * sxy;
      x[o] = x[o] + p[o] * alpha;
      const double rn = r[o] + q[o] * malpha;
      r[o] = rn;
      two[0] += rn * rn;
      const double z = minv_at<double>(G, dxy, axy, b.k0 + u) * rn;
      two[1] += z * rn;
    }
  }
  box_put<NT, 2>(two, part2, gridDim.x, sh);
}

template <int NT>
__global__ void __launch_bounds__(NT) k_box_pupdate(double *__restrict__ p, const double *__restrict__ r, CCGeom G,
                                                   int by, int gy, int cpt, PcgCtrl *ctrl, const double *part2, int it) {
  if (ctrl->done) return;
  __shared__ ResShared<NT> sh;
  const Box b = box_of(G, by, gy, cpt);
  double two[2];
  box_sums<NT, 2>(two, part2, gridDim.x, sh);
  const double rr = two[0], rz = two[1];
  const ExitDecision e = exit_decision(ctrl, it, rr);
  const double beta = rz / ctrl->rho[(it - 1) & 1];
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    publish_exit(ctrl, it, rr, e);
    ctrl->rz = rz;
    ctrl->beta = beta;
    ctrl->rho[it & 1] = rz;
  }
  if (e.stop || b.nk == 0) return;
  const size_t sx = G.s0, sxy = (size_t)G.s0 * G.s1;
  const double dxy = G.c[0].dh[b.i] * G.c[1].dh[b.j];
  const double axy = G.c[0].lA[b.i] + G.c[0].lB[b.i] + G.c[1].lA[b.j] + G.c[1].lB[b.j];
  const bool edge_ij = b.i == 1 || b.i == G.n0 || b.j == 1 || b.j == G.n1;
#pragma unroll 4
  for (int u = 0; u < b.nk; ++u) {
    const int k = b.k0 + u;
    const size_t o = (size_t)b.i + (size_t)b.j * sx + (size_t)k * sxy;
    const double z = minv_at<double>(G, dxy, axy, k) * r[o];
    const double pn = p[o] * beta + z;
    p[o] = pn;
    if (edge_ij || k == 1 || k == G.n2) fill_ghosts_implicit(p, G, b.i, b.j, k, pn);
  }
}

// x = the resident loop's result, unless it was given up or the set-up's exit test ended the solve.
__global__ void __launch_bounds__(kNT) k_pcg_take(double *__restrict__ x, const double *__restrict__ x_out, CCGeom G,
                                                 PcgCtrl *ctrl, const unsigned long long *slots) {
  const bool given_up = slots[6 * kResMaxBlocks] != 0;
  if (given_up && blockIdx.x == 0 && threadIdx.x == 0) ctrl->given_up = 1;
  if (given_up || ctrl->done != kResDone) return;
  const TileIdx t = tile_of(G);
  if (!t.active) return;
  const size_t sx = G.s0, sxy = (size_t)G.s0 * G.s1;
  for (int k = t.k0; k < t.k1; ++k) {
    const size_t o = (size_t)t.i + (size_t)t.j * sx + (size_t)k * sxy;
    x[o] = x_out[o];
  }
}

// The box of the resident loop: among the plane counts whose blocks fit the
// CUs and whose LDS fits, the least time an iteration by a model of its two
// parts, fitted to measured iterations (18x15x17 to 128^3, within 10%): the
// two all-reduces with the halo's loads by the number of blocks (4.5 us to 16
// blocks, then 1.3 us a doubling to 64, 0.7 us above) and the cells' work by
// the planes a thread (4 planes 0.8 us, 8 2.4 us, 16 6.5 us).  E.g. 32^3 takes
// 16 blocks of 4 planes (5.8 us; 64 blocks of 1 plane 7.3 us), 64^3 128 of 4
// (9.0; 64 of 8 10.1), 128^3 256 of 16 (16.4 us).  The launch-per-kernel loop
// takes 16-19 us up to 64^3, 32 us at 96^3, 49 us at 128^3, so every grid that
// fits a box takes the resident one; the other is kept by larger grids, by rows
// of more than kResNT cells, and by grids near 128^3 whose rows leave much of a
// block idle (129 x 128 x 128 and 130 x 120 x 120 need more than 256 blocks).
constexpr int kResNT = 512;
inline ResPlan resident_plan(int n0, int n1, int n2, int cus) {
  ResPlan best;
  double least = 1e300;
  if (n0 > kResNT) return best;
  const int cpts[5] = {1, 2, 4, 8, 16};
  const double work[5] = {0.1, 0.2, 0.8, 2.4, 6.5};
  for (int c = 0; c < 5; ++c) {
    ResPlan P;
    P.cpt = cpts[c];
    P.by = std::min(kResNT / n0, n1);
    P.gy = (n1 + P.by - 1) / P.by;
    P.by = (n1 + P.gy - 1) / P.gy; // rows evenly over the blocks
    P.gy = (n1 + P.by - 1) / P.by;
    P.gz = (n2 + P.cpt - 1) / P.cpt;
    P.lds = ((size_t)P.cpt * (P.by + 2) * (n0 + 2) + (size_t)2 * P.cpt * n0) * sizeof(double);
    if ((long long)P.gy * P.gz > std::min(cus, kResMaxBlocks) || P.lds > 156 * 1024) continue;
    const double doublings = std::log2(std::max(1.0, P.nb() / 16.0));
    const double time = 4.5 + 1.3 * std::min(doublings, 2.0) + 0.7 * std::max(0.0, doublings - 2.0) + work[c];
    if (time < least) {
      least = time;
      best = P;
    }
  }
  return best;
}

} // namespace moons
