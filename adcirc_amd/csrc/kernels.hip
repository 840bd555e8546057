// Device kernels of the 2DDI per-timestep hot path for gfx950 (CDNA4).
//
// Parity design: every per-node sum the reference forms by scattering element
// contributions in ascending element order (GWCE matrix, GWCE load vector,
// momentum load vectors, TotalArea) is formed node by node over the node's
// incident elements in ascending element id (here and in patch.hip), which is the
// same order, so the result is bit-identical.  Inner products use one fixed
// blocked tree (reduce.h), identical on every launch shape.  Built with
// -ffp-contract=off so no multiply-add is fused.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "kernels.h"
#include "reduce.h"

namespace adcgpu {

// ------------------------------------------------------------ time levels
__global__ __launch_bounds__(256) void k_init_h(int np, const double* __restrict__ dp, const double* __restrict__ eta2,
                         double ifnlfa, double* __restrict__ h1, double* __restrict__ h2) {
  int i = xcd_tile(blockIdx.x, gridDim.x) * blockDim.x + threadIdx.x;
  if (i >= np) return;
  double h = dp[i] + ifnlfa * eta2[i];
  h2[i] = h;
  h1[i] = h;
}

// applyTidePotentialForcing's constituent sum (src/timestep.F:1527-1557): TIP2
// starts at zero and takes each constituent's term in order; the
// self-attraction term of NTIP = 2 is absent (its amplitudes are zero for
// NTIP = 1, src/read_input.F:6460, and adding a zero to this sum changes no bit).
__global__ __launch_bounds__(256) void k_tide_pot(int np, TipPrm p, const double* __restrict__ ln,
                                                  const double* __restrict__ slam,
                                                  double* __restrict__ tip2) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= np) return;
  double v = 0.0;
  for (int j = 0; j < p.ntif; ++j) {
    const double argtp = p.argt[j] + p.na[j] * slam[i];
    v = v + p.tpmul[j] * ln[(size_t)p.na[j] * np + i] * cos(argtp);
  }
  tip2[i] = v;
}

__device__ __forceinline__ void friction_node(int i, const FricPrm& f, double* __restrict__ tk) {
  tk[i] = friction(f, i, f.uu1[i], f.vv1[i], f.dp[i], f.eta2[i]);
}

__global__ __launch_bounds__(256) void k_friction(int np, FricPrm f, double* __restrict__ tk) {
  int i = xcd_tile(blockIdx.x, gridDim.x) * blockDim.x + threadIdx.x;
  if (i >= np) return;
  friction_node(i, f, tk);
}

// Holland (1980) vortex forcing on the device (synthetic storms for the
// resident benchmark run).  Same formulas as the oracle's host version; device
// exp/pow/sqrt differ from host libm by a few ulp.
__device__ __forceinline__ void holland_node(int i, const double* __restrict__ x,
                                             const double* __restrict__ y, const HollandPrm& p,
                                             double* __restrict__ wsx, double* __restrict__ wsy,
                                             double* __restrict__ pr) {
  const double t = p.t;
  const double pc = p.v[0] * 100.0, pn = p.v[1] * 100.0, rmax = p.v[2], B = p.v[3];
  const double xc = p.v[4] + p.v[6] * t, yc = p.v[5] + p.v[7] * t, f = p.v[8];
  const double rampd = p.v[9], rhoa = p.v[10], wfac = p.v[11];
  const double beta = p.v[12] * 3.141592653589793 / 180.0;
  const double rho0 = 1000.0, g = 9.80665;
  const double ramp = rampd > 0.0 ? tanh((2.0 * t / 86400.0) / rampd) : 1.0;
  const double dpr = pn - pc, cb = cos(beta), sb = sin(beta);
  double dx = x[i] - xc, dy = y[i] - yc;
  double r = __builtin_sqrt(dx * dx + dy * dy);
  if (r < 1.0) r = 1.0;
  double a = pow(rmax / r, B);
  double e = exp(-a);
  double pp = pc + dpr * e;
  double rf2 = 0.5 * r * f;
  double vg = __builtin_sqrt(B / rhoa * a * dpr * e + rf2 * rf2) - rf2;
  double w = wfac * vg;
  double tx = -dy / r, ty = dx / r, rx = dx / r, ry = dy / r;
  double wx = w * (cb * tx - sb * rx), wy = w * (cb * ty - sb * ry);
  double wm = __builtin_sqrt(wx * wx + wy * wy);
  double cd = 0.001 * (0.75 + 0.067 * wm);
  if (cd > 0.0035) cd = 0.0035;
  double sc = ramp * cd * (rhoa / rho0) * wm;
  wsx[i] = sc * wx;
  wsy[i] = sc * wy;
  pr[i] = (pn + ramp * (pp - pn)) / (rho0 * g);
}

__global__ __launch_bounds__(256) void k_holland(int np, const double* __restrict__ x, const double* __restrict__ y,
                          HollandPrm p, double* __restrict__ wsx, double* __restrict__ wsy,
                          double* __restrict__ pr) {
  int i = xcd_tile(blockIdx.x, gridDim.x) * blockDim.x + threadIdx.x;
  if (i >= np) return;
  holland_node(i, x, y, p, wsx, wsy, pr);
}

// --------------------------------------------------------------- GWCE
// EP chunk partials: sum COEF(i,1)^2 (src/gwce.F:646-650) in the fixed blocked
// tree (thread t of chunk c adds rows c 2048 + t + 512 r, r = 0..3, in order;
// then the chunk tree).  The matrix is rebuilt when NCChange > 0 and NCChange is
// then cleared (src/gwce.F:427-428): this pass, between the kernel that tests it
// and those that set it, clears it and leaves F_REBUILT for the node pass.
__device__ __forceinline__ void lhs_ep_block(const DevMesh& m, const DevState& s, int* flags,
                                             double* __restrict__ ep_part, int bid, int nch) {
  __shared__ double lds[8];
  const int chunk = xcd_tile(bid, nch);
  const int base = chunk * RED_CHUNK + threadIdx.x;
  double d[RED_PER_THREAD];
#pragma unroll
  for (int r = 0; r < RED_PER_THREAD; ++r) {
    const int i = base + RED_THREADS * r;
    d[r] = i < m.np ? s.coef[i] : 0.0;
  }
  double acc = 0.0;
#pragma unroll
  for (int r = 0; r < RED_PER_THREAD; ++r) acc = acc + d[r] * d[r];
  const double tot = chunk_tree(acc, lds);
  if (threadIdx.x == 0) ep_part[chunk] = tot;
  if (bid == 0 && threadIdx.x == 0) {
    const int ncc = flags[F_NCCHANGE];
    flags[F_REBUILT] = ncc > 0 ? 1 : 0;
    if (ncc > 0) flags[F_NREBUILD] += 1;
    flags[F_NCCHANGE] = 0;
  }
}

__global__ __launch_bounds__(RED_THREADS) void k_lhs_ep(DevMesh m, DevState s, int* flags,
                                                        double* __restrict__ ep_part) {
  lhs_ep_block(m, s, flags, ep_part, blockIdx.x, gridDim.x);
}
__global__ __launch_bounds__(RED_THREADS) void k_lhs_ep_batch(const MemberArgs* __restrict__ a) {
  const MemberArgs& x = a[blockIdx.y];
  if ((int)blockIdx.x >= x.nch) return;
  lhs_ep_block(x.m, x.s, x.pre.flags, x.ep_part, blockIdx.x, x.nch);
}

// The off-diagonals of a solve whose unscaling was deferred, scaled and
// unscaled as scal and unscal do (src/itpackv.F:2394-2400, 2460-2479).
__global__ __launch_bounds__(256) void k_coef_restore(DevMesh m, DevState s,
                                                      const double* __restrict__ w) {
  const int i = xcd_tile(blockIdx.x, gridDim.x) * blockDim.x + threadIdx.x;
  if (i >= m.np) return;
  const int np = m.np, nn = m.nneigh[i];
  const double wi = w[i], ri = 1.0 / wi;
  for (int j = 1; j < nn; ++j) {
    const size_t q = (size_t)j * np + i;
    const double wj = w[m.col[q]];
    s.coef[q] = (s.coef[q] * wi * wj) * ri * (1.0 / wj);
  }
}

// QFORCE of flow-boundary entry K: for a specified (or zero) flux, codes up
// to 29, (QN2 - QN0)/DT2 + Tau0Var*QN1 (src/gwce.F:1741, 1783); for outward
// radiation (30) the value k_flux_shift formed at the step's start.
__device__ __forceinline__ double qforce(const DevMesh& m, const DevState& s, int K) {
  if (m.lbcodei[K] == 30) return s.qrad[K];
  const double q = (s.qn2[K] - s.qn0[K]) / (m.dt * 2.0) + m.tau0[m.nbv[K]] * s.qn1[K];
  // river radiation (52) past the flux-settling steps (src/gwce.F:1767-1775)
  return m.lbcodei[K] == 52 ? q - s.qrad[K] : q;
}

// The specified-flux line integrals a node receives (src/gwce.F:1777-1832):
// for each boundary edge NBV(J-1)-NBV(J) it lies on, in edge order,
// NCI*NCJ*BNDLEN2O3(J-1)/4 * (2 QFORCE(own) + QFORCE(other)) added to its
// GWCE_LV.  The edges whose terms are exactly +0 (zero length) are left out.
__device__ __forceinline__ double flux_terms(const DevMesh& m, const DevState& s, int k, double acc) {
  for (int p = m.fb_ptr[k]; p < m.fb_ptr[k + 1]; ++p) {
    const int e = m.fb_ent[p];
    const int J = e >> 1;
    const int ni = m.nbv[J - 1], nj = m.nbv[J];
    const double qi = qforce(m, s, J - 1), qj = qforce(m, s, J);
    const double w = (double)(s.nodecode[ni] * s.nodecode[nj]) * m.bndlen[J - 1] / 4.0;
    acc = acc + ((e & 1) ? w * (2.0 * qj + qi) : w * (2.0 * qi + qj));
  }
  return acc;
}

// The shift of the normal flux to the previous time levels and the step's
// new QN2 (src/timestep.F:605-612, then 861-903): next == null leaves QN2
// zero, as the reference's shift does.  An outward-radiating entry (30) takes
// QN1 from the last velocities and depth (src/timestep.F:929-940) and its
// QFORCE, -sqrt(G H1) ETAS/DT - Tau0Var QN1 with H1 the depth the GWCE will
// hold (the last step's H2) and ETAS the last increment (src/gwce.F:1750-1754,
// 1785-1789), is formed here, before the assembly rewrites ETAS.
__global__ __launch_bounds__(256) void k_flux_shift(DevMesh m, DevState s,
                                                    const double* __restrict__ next, int nvel) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= nvel) return;
  s.qn0[k] = s.qn1[k];
  double q1 = s.qn2[k];
  s.qn2[k] = next ? next[k] : 0.0;
  if (m.lbcodei[k] == 30) {
    const int b = m.nbv[k];
    const double un1 = s.uu1[b] * m.csii[k] + s.vv1[b] * m.siii[k];
    q1 = s.h2[b] * un1;
    const double celerity = __builtin_sqrt(m.g * s.h2[b]);
    s.qrad[k] = -celerity * s.etas[b] / m.dt - m.tau0[b] * q1;
  } else if (m.lbcodei[k] == 52) {
    // Celerity*(ETAS/DT + Tau0Var*(ETA1 - ElevDisc)): ETA2 now is the GWCE's ETA1
    const int b = m.nbv[k];
    const double celerity = __builtin_sqrt(m.g * s.h2[b]);
    s.qrad[k] = celerity * (s.etas[b] / m.dt + m.tau0[b] * (s.eta2[b] - s.elevdisc[k]));
  }
  s.qn1[k] = q1;
}

// Node pass of the GWCE: the boundary terms of GWCE_LV, the time-level shift of
// ETA and the elevation boundary conditions (src/gwce.F:1613-1631, 1638-1651,
// 1846-1855), and after a rebuild the elevation-boundary rows of the matrix
// (src/gwce.F:700-743): a boundary row becomes EP on the diagonal with its
// off-diagonals and OBCCOEF entries zeroed; an entry that couples another row to
// a boundary node moves to OBCCOEF.  `eta1` already points at the previous
// ETA2; `eta2` is rewritten.  EP = sqrt(sum of squared diagonals / NP) from the
// chunk partials, by every block that has a row that takes it (a boundary row,
// or a zero diagonal).
template <bool LUMPED>
__device__ __forceinline__ void rhs_node_block(const DevMesh& m, DevState s,
                                               const double* __restrict__ eta_bc, int nch,
                                               const double* __restrict__ ep_part,
                                               double* __restrict__ scal, const JcgPre& pre,
                                               const HollandPrm& hol, int met, int bid, int nb) {
  __shared__ double lds[4];
  __shared__ double ep_s;
  const int i = xcd_tile(bid, nb) * blockDim.x + threadIdx.x;
  if (i < pre.barrier_words) pre.barrier[i] = 0u;
  if (i < pre.part_words) pre.part[i] = JCG_EMPTY;
  if (i == 0) pre.barrier[JCG_ADMIT_WORD] = pre.admit0;
  const bool rebuilt = pre.flags[F_REBUILT] != 0;
  const bool in = i < m.np;
  // the step's forcing beside: arithmetic, where the rest of the pass waits for
  // memory (a pass of its own took 23 us at 1M nodes, 5 at 20,000)
  if (met && in) holland_node(i, m.x, m.y, hol, s.wsx2, s.wsy2, s.pr2);
  const int bi = in ? m.bnd_index[i] : -1;
  double dg = in ? s.coef[i] : 1.0;
  const bool take_ep = dg == 0.0 || bi >= 0;
  double ep = 0.0;
  // block 0 also keeps EP for the steps without a rebuild
  if (__syncthreads_or(take_ep || (rebuilt && bid == 0))) {
    if (rebuilt) {
      double acc = 0.0;
      for (int c = threadIdx.x; c < nch; c += RED_XTHREADS) acc = acc + ep_part[c];
      const double tot = block_tree(acc, lds);
      if (threadIdx.x == 0) {
        ep_s = __builtin_sqrt(tot / (double)m.np);
        if (bid == 0) scal[S_EP] = ep_s;
      }
      __syncthreads();
      ep = ep_s;
    } else {
      ep = scal[S_EP];
    }
  }
  if (!in) return;
  const int o0 = m.obcg_ptr[i], o1 = LUMPED ? o0 : m.obcg_ptr[i + 1];
  double rhs, u;
  if (bi >= 0) {
    if (rebuilt) {
      dg = ep;
      s.coef[i] = ep;
      const int nn = m.nneigh[i];
      for (int j = 1; j < nn; ++j) s.coef[(size_t)j * m.np + i] = 0.0;
      for (int p = o0; p < o1; ++p) s.obc[m.obcg[p]] = 0.0;
    }
    const double e2 = eta_bc[bi];
    const double es = e2 - s.eta1[i];
    if (pre.keep_prev) pre.etas_prev[i] = s.etas[i];
    s.eta2[i] = e2;
    u = es;
    // lumped: the boundary row's own COEFD (src/gwce.F:1856-1862)
    rhs = es * (double)s.nodecode[i] * (LUMPED ? dg : ep);
  } else {
    double acc = s.gwce_lv[i];
    if (bi < -1) acc = flux_terms(m, s, -2 - bi, acc);
    for (int p = o0; p < o1; ++p) {
      const int slot = m.obcg[p];
      if (rebuilt) {  // a lumped LHS has no boundary columns
        const size_t z = m.obcg_q[p];
        s.obc[slot] = s.coef[z];
        s.coef[z] = 0.0;
      }
      const int I = slot / m.mnei;
      const int b = m.nbd[I];
      const double es = eta_bc[I] - s.eta1[b];
      acc = acc - es * s.obc[slot];
    }
    rhs = acc;
    u = s.etas[i];
    const double u_ref = u;
    if (pre.warm == 1) {
      // the increment extrapolated from the last two: ETA2 extrapolated to
      // second order instead of the first order the previous increment gives
      u = 2.0 * u - pre.etas_prev[i];
    }
    if (pre.keep_prev) pre.etas_prev[i] = u_ref;
    s.eta2[i] = 0.0;
  }
  // a zero diagonal (a dry row) becomes EP (src/gwce.F:737-741); then the
  // first scaling pass of JCG (src/itpackv.F:2374-2393): w = 1/sqrt(diag),
  // u and rhs scaled in place
  if (dg == 0.0) {
    dg = ep;
    s.coef[i] = dg;
  }
  if (LUMPED) {
    // explicit solve (src/gwce.F:2009-2022); no JCG follows
    if (dg < 0.0) atomicOr(&pre.flags[F_ERROR], ERR_DIAG);
    if (i == 0) {
      pre.flags[F_NUMITR] = 0;
      pre.flags[F_IER] = 0;
    }
    s.gwce_lv[i] = rhs;
    const double rdiag = dg == 0.0 ? 0.0 : 1.0 / dg;
    const double es = rhs * rdiag;
    s.etas[i] = es;
    s.eta2[i] = (double)s.nodecode[i] * (es + 0.0) + s.eta1[i];
    return;
  }
  if (!(dg > 0.0)) atomicOr(&pre.flags[F_ERROR], ERR_DIAG);
  const double sq = __builtin_sqrt(dg);
  const double w = 1.0 / sq;
  s.etas[i] = u * sq;
  // the learned start (zero correction on boundary and dry rows), scaled
  if (pre.warm == 2) pre.ml_u[i] = (u + pre.ml_corr[i]) * sq;
  pre.w[i] = w;
  s.gwce_lv[i] = rhs * w;
}

template <bool LUMPED>
__global__ __launch_bounds__(256) void k_rhs_node(DevMesh m, DevState s,
                                                  const double* __restrict__ eta_bc, int nch,
                                                  const double* __restrict__ ep_part,
                                                  double* __restrict__ scal, JcgPre pre,
                                                  HollandPrm hol, int met) {
  rhs_node_block<LUMPED>(m, s, eta_bc, nch, ep_part, scal, pre, hol, met, blockIdx.x, gridDim.x);
}
__global__ __launch_bounds__(256) void k_rhs_node_batch(const MemberArgs* __restrict__ a, int step,
                                                        int it, int met) {
  const MemberArgs& x = a[blockIdx.y];
  const int nb = (x.m.np + 255) / 256;
  if ((int)blockIdx.x >= nb) return;
  HollandPrm hol = x.hol;
  hol.t = it * x.dt;
  rhs_node_block<false>(x.m, x.s, x.eta_bc + (size_t)step * x.m.neta, x.nch, x.ep_part, x.scal, x.pre,
                        hol, met, blockIdx.x, nb);
}
template __global__ void k_rhs_node<false>(DevMesh, DevState, const double*, int, const double*, double*, JcgPre, HollandPrm, int);
template __global__ void k_rhs_node<true>(DevMesh, DevState, const double*, int, const double*, double*, JcgPre, HollandPrm, int);

// ---------------------------------------------------------------- wet/dry
// Values that another block of the launch reads: written through, and read past
// the caches.
__device__ __forceinline__ void wd_put(double* p, double v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void wd_put(int* p, int v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void wd_put(unsigned long long* p, unsigned long long v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <class T>
__device__ __forceinline__ T wd_get(const T* p) {
  return __hip_atomic_load(const_cast<T*>(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// The candidate indices of candidate element e's predecessors, or -1.
__device__ __forceinline__ int2 wd_pred_index(const WdWork& w, int e) {
  const int2 p = w.pred[e];
  return make_int2(p.x >= 0 ? w.lc[p.x].y : -1, p.y >= 0 ? w.lc[p.y].y : -1);
}

// Ordered W1 friction updates, values: M_k = max(m0_k, M of k's predecessors)
// in candidate order, then each node takes the M of its last candidate.  TK
// values are finite, so max is exact and order-free, and M_k is the maximum of
// m0 over k and all of its ancestors in the predecessor graph (edges run from
// lower to higher candidate index).
//
// Block closure.  Candidates are cut into blocks of WD_BLOCK.  Inside a block,
// M_k splits into the maximum over k's ancestors inside the block (cv) and the
// set of earlier-block candidates those ancestors name as predecessors (cE,
// bits into the block's table of external names xtab).  Pointer doubling
// forms both: each candidate keeps a frontier of at most two ancestors not
// yet folded in; a round replaces frontier members by their own frontiers
// (folding in their values and name sets) whenever the result still has at
// most two members.  After every such step ancestors(k) = folded(k) plus
// ancestors(frontier(k)), and the lowest candidate with a non-empty frontier
// can always expand it, so the rounds end; along a wetting front, where
// candidates chain through shared nodes, they take about log2 of the chain
// length.  A block naming more than WD_XMAX external candidates sets
// F_WDSERIAL, and every value is formed serially instead.
__device__ __forceinline__ void wd_add(int* u, int& nu, int f) {
  if (f == 0xffff) return;
  for (int i = 0; i < nu; ++i)
    if (u[i] == f) return;
  u[nu++] = f;
}

__device__ __forceinline__ void wd_close(const DevMesh& m, const DevState& s, const WdWork& w,
                                         int* flags, double* wc_lds, int bid, int nb) {
  double* sv = wc_lds;                                                       // [2][WD_BLOCK]
  unsigned long long* sE = reinterpret_cast<unsigned long long*>(sv + 2 * WD_BLOCK);  // [2][WD_XW][WD_BLOCK]
  int* sF = reinterpret_cast<int*>(sE + 2 * WD_XW * WD_BLOCK);               // [2][WD_BLOCK]
  int* hkey = sF + 2 * WD_BLOCK;                                             // [WD_HASH]
  int* hidx = hkey + WD_HASH;                                                // [WD_HASH]
  __shared__ int xn;
  const int n = flags[F_NCAND];
  const int nblk = (n + WD_BLOCK - 1) / WD_BLOCK;
  const int l = threadIdx.x;
  for (int b = bid; b < nblk; b += nb) {
    const int base = b * WD_BLOCK, k = base + l;
    for (int i = l; i < WD_HASH; i += WD_BLOCK) hkey[i] = -1;
    if (l == 0) xn = 0;
    __syncthreads();
    int qq[2] = {-1, -1}, wn[2] = {-1, -1};
    double v = 0.0;
    if (k < n) {
      const int e = w.cid[k];
      const int2 q = wd_pred_index(w, e), x = w.wnode[e];
      v = w.m0[e];
      qq[0] = q.x;
      qq[1] = q.y;
      wn[0] = x.x;
      wn[1] = x.y;
    }
    // the block's external names: one hash slot per distinct candidate
    int slot[2] = {-1, -1};
    bool won[2] = {false, false};
    bool ovf = false;
    for (int j = 0; j < 2; ++j) {
      const int x = qq[j];
      if (x < 0 || x >= base) continue;
      int h = (int)(((unsigned)x * 2654435761u) >> 23);  // 9 bits: WD_HASH slots
      for (int probes = 0; probes < WD_HASH; ++probes) {
        const int old = atomicCAS(&hkey[h], -1, x);
        if (old == -1 || old == x) {
          won[j] = old == -1;
          slot[j] = h;
          break;
        }
        h = (h + 1) & (WD_HASH - 1);
      }
      if (slot[j] < 0) ovf = true;
    }
    __syncthreads();
    for (int j = 0; j < 2; ++j)
      if (won[j]) {
        const int i = atomicAdd(&xn, 1);
        hidx[slot[j]] = i;
        if (i < WD_XMAX) wd_put(&w.xtab[b * WD_XMAX + i], qq[j]);
      }
    __syncthreads();
    unsigned long long E[WD_XW] = {};
    int f0 = 0xffff, f1 = 0xffff;
    for (int j = 0; j < 2; ++j) {
      const int x = qq[j];
      if (x < 0) continue;
      if (x >= base) {
        const int li = x - base;
        if (f0 == 0xffff) f0 = li;
        else if (li != f0) f1 = li;
      } else if (slot[j] >= 0) {
        const int i = hidx[slot[j]];
        if (i < WD_XMAX) E[i >> 6] |= 1ull << (i & 63);
        else ovf = true;
      }
    }
    if (__syncthreads_or(ovf)) {
      if (l == 0) atomicOr(&flags[F_WDSERIAL], 1);
      continue;
    }
    if (l == 0) wd_put(&w.xcnt[b], xn);
    int cur = 0;
    sv[l] = v;
#pragma unroll
    for (int i = 0; i < WD_XW; ++i) sE[i * WD_BLOCK + l] = E[i];
    sF[l] = f0 | (f1 << 16);
    __syncthreads();
    while (true) {
      const int nx = cur ^ 1;
      const double* cv_ = sv + cur * WD_BLOCK;
      const unsigned long long* cE_ = sE + cur * WD_XW * WD_BLOCK;
      const int* cF_ = sF + cur * WD_BLOCK;
      int F = cF_[l];
      const int a = F & 0xffff, c = (F >> 16) & 0xffff;
      // members to fold in this round: bit 0 = a, bit 1 = c
      int fold = 0;
      if (a != 0xffff) {
        const int Fa = cF_[a];
        const int Fc = c != 0xffff ? cF_[c] : -1;
        int u[4], nu = 0;
        wd_add(u, nu, Fa & 0xffff);
        wd_add(u, nu, (Fa >> 16) & 0xffff);
        if (c != 0xffff) {
          wd_add(u, nu, Fc & 0xffff);
          wd_add(u, nu, (Fc >> 16) & 0xffff);
        }
        if (nu <= 2) {
          fold = c != 0xffff ? 3 : 1;
          F = (nu > 0 ? u[0] : 0xffff) | ((nu > 1 ? u[1] : 0xffff) << 16);
        } else {
          // expand one member alone
          int ua[3], na = 0;
          wd_add(ua, na, c);
          wd_add(ua, na, Fa & 0xffff);
          wd_add(ua, na, (Fa >> 16) & 0xffff);
          if (na <= 2) {
            fold = 1;
            F = (na > 0 ? ua[0] : 0xffff) | ((na > 1 ? ua[1] : 0xffff) << 16);
          } else if (c != 0xffff) {
            int uc[3], nc = 0;
            wd_add(uc, nc, a);
            wd_add(uc, nc, Fc & 0xffff);
            wd_add(uc, nc, (Fc >> 16) & 0xffff);
            if (nc <= 2) {
              fold = 2;
              F = (nc > 0 ? uc[0] : 0xffff) | ((nc > 1 ? uc[1] : 0xffff) << 16);
            }
          }
        }
      }
      if (fold & 1) {
        v = fmax(v, cv_[a]);
#pragma unroll
        for (int i = 0; i < WD_XW; ++i) E[i] |= cE_[i * WD_BLOCK + a];
      }
      if (fold & 2) {
        v = fmax(v, cv_[c]);
#pragma unroll
        for (int i = 0; i < WD_XW; ++i) E[i] |= cE_[i * WD_BLOCK + c];
      }
      sv[nx * WD_BLOCK + l] = v;
#pragma unroll
      for (int i = 0; i < WD_XW; ++i) sE[(nx * WD_XW + i) * WD_BLOCK + l] = E[i];
      sF[nx * WD_BLOCK + l] = F;
      cur = nx;
      if (!__syncthreads_or((F & 0xffff) != 0xffff)) break;
    }
    if (nblk == 1) {  // no candidates outside the block: the values are final
      for (int j = 0; j < 2; ++j)
        if (wn[j] >= 0) s.tk[wn[j]] = v;
    } else if (k < n) {
      wd_put(&w.cv[k], v);
#pragma unroll
      for (int i = 0; i < WD_XW; ++i) wd_put(&w.cE[(size_t)k * WD_XW + i], E[i]);
    }
  }
}

// Serial form of the ordered updates (blocks with too many external names):
// the candidates pass through LDS in chunks of WD_CHUNK; one lane forms M
// along the chunk (the previous candidate's M in a register, the last WD_RING
// values in an LDS ring, older ones read back from w.M) and the block writes
// the chunk's TK values.  `lds` holds WD_SERIAL_LDS bytes.
__device__ void wd_serial(const WdWork& w, int n, double* __restrict__ tk, double* lds) {
  double* ring = lds;                                             // [WD_RING]
  double* cm0 = ring + WD_RING;                                   // [WD_CHUNK]
  int2* cpred = reinterpret_cast<int2*>(cm0 + WD_CHUNK);          // [WD_CHUNK]
  int2* cwn = cpred + WD_CHUNK;                                   // [WD_CHUNK]
  const int t = threadIdx.x;
  double mprev = 0.0;  // M of the previous candidate (lane 0)
  for (int base = 0; base < n; base += WD_CHUNK) {
    const int cn = min(WD_CHUNK, n - base);
    for (int i = t; i < cn; i += blockDim.x) {
      const int e = w.cid[base + i];
      cm0[i] = w.m0[e];
      cpred[i] = wd_pred_index(w, e);
      cwn[i] = w.wnode[e];
    }
    __syncthreads();
    if (t == 0) {
      for (int i = 0; i < cn; ++i) {
        const int k = base + i;
        double v = cm0[i];
        const int2 q = cpred[i];
        if (q.x >= 0)
          v = fmax(v, q.x == k - 1 ? mprev
                                   : (q.x >= k - WD_RING ? ring[q.x & (WD_RING - 1)] : w.M[q.x]));
        if (q.y >= 0)
          v = fmax(v, q.y == k - 1 ? mprev
                                   : (q.y >= k - WD_RING ? ring[q.y & (WD_RING - 1)] : w.M[q.y]));
        ring[k & (WD_RING - 1)] = v;
        w.M[k] = v;
        mprev = v;
      }
    }
    __syncthreads();
    for (int i = t; i < cn; i += blockDim.x) {
      const double v = ring[(base + i) & (WD_RING - 1)];
      const int2 x = cwn[i];
      if (x.x >= 0) tk[x.x] = v;
      if (x.y >= 0) tk[x.y] = v;
    }
    __syncthreads();
  }
}

// Values of the external names, block after block: name i of block c is an
// earlier candidate x of block b < c, so its value is max(cv[x], values of
// the names of block b set in cE[x]), all known by then.  One block, one lane
// per name; LDS of WD_LINK_LDS bytes (the name values of up to WD_LINK_BLOCKS
// blocks; beyond that they are kept in w.xval).  Then each candidate's M_k,
// written as TK of the nodes it is the last candidate of.
__device__ __forceinline__ void wd_link(const WdWork& w, int n, double* __restrict__ tk,
                                        double* lk_lds) {
  const int nblk = (n + WD_BLOCK - 1) / WD_BLOCK;
  double* X = nblk <= WD_LINK_BLOCKS ? lk_lds : w.xval;
  const int t = threadIdx.x;
  auto value = [&](int x) {
    double v = wd_get(&w.cv[x]);
    unsigned long long E[WD_XW];
#pragma unroll
    for (int i = 0; i < WD_XW; ++i) E[i] = wd_get(&w.cE[(size_t)x * WD_XW + i]);
    const double* Xb = X + (x / WD_BLOCK) * WD_XMAX;
#pragma unroll
    for (int i = 0; i < WD_XW; ++i)
      while (E[i]) {
        v = fmax(v, Xb[64 * i + __ffsll((long long)E[i]) - 1]);
        E[i] &= E[i] - 1;
      }
    return v;
  };
  for (int c = 1; c < nblk; ++c) {
    if (t < wd_get(&w.xcnt[c])) X[c * WD_XMAX + t] = value(wd_get(&w.xtab[c * WD_XMAX + t]));
    __syncthreads();
  }
  for (int k = t; k < n; k += blockDim.x) {
    const int2 x = w.wnode[w.cid[k]];
    const double v = value(k);
    if (x.x >= 0) tk[x.x] = v;
    if (x.y >= 0) tk[x.y] = v;
  }
}

// The ordered friction updates of the step's candidates (linked and listed by the
// pass before): block closure by as many blocks as have candidates; the block
// that ends last joins the blocks' values and writes TK, so that no block waits
// for another.  Dynamic LDS: WD_CHAIN_LDS bytes.
__device__ __forceinline__ void wd_chain_block(const DevMesh& m, const DevState& s, const WdWork& w,
                                               int* flags, int bid, int nb) {
  extern __shared__ double ch_lds[];
  __shared__ int last;
  const int n = flags[F_NCAND];
  const int nblk = (n + WD_BLOCK - 1) / WD_BLOCK;
  const int active = min(nblk, nb);
  if (bid >= active) return;
  wd_close(m, s, w, flags, ch_lds, bid, nb);
  if (nblk > 1) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this wave's values are written
    __syncthreads();
    if (threadIdx.x == 0) last = atomicAdd(&flags[F_WDDONE], 1) == active - 1;
    __syncthreads();
    if (!last) return;
    if (wd_get(&flags[F_WDSERIAL]))
      wd_serial(w, n, s.tk, ch_lds);
    else
      wd_link(w, n, s.tk, ch_lds);
    if (threadIdx.x == 0) flags[F_WDDONE] = 0;
  }
  // the candidate marks are clear between steps (every block has followed its
  // links by now)
  __syncthreads();
  for (int k = threadIdx.x; k < n; k += blockDim.x) {
    const int e = w.cid[k];
    w.mask[e >> 6] = 0ull;
    w.bcnt[e >> 8] = 0;
    w.lc[e] = make_int2(-1, -1);
  }
}

__global__ __launch_bounds__(WD_BLOCK) void k_wd_chain(DevMesh m, DevState s, WdWork w, int* flags) {
  wd_chain_block(m, s, w, flags, blockIdx.x, gridDim.x);
}
__global__ __launch_bounds__(WD_BLOCK) void k_wd_chain_batch(const MemberArgs* __restrict__ a) {
  const MemberArgs& x = a[blockIdx.y];
  if ((int)blockIdx.x >= x.nchain) return;
  wd_chain_block(x.m, x.s, x.wd, x.pre.flags, blockIdx.x, x.nchain);
}

// computeAlpha: ALPHAL of element e.
__device__ __forceinline__ double wd_alpha(const DevMesh& m, const DevState& s, int e, int* flags,
                                           double slim) {
  const int n1 = m.nm[3 * e], n2 = m.nm[3 * e + 1], n3 = m.nm[3 * e + 2];
  double al = 1.0;
  const int ncele = s.nodecode[n1] * s.nodecode[n2] * s.nodecode[n3] * s.noff[e];
  if (ncele == 1)
    al = compute_alpha(s.eta2[n1], s.eta2[n2], s.eta2[n3], m.dp[n1], m.dp[n2], m.dp[n3], slim,
                       [&](double fx[3], double fy[3]) {
                         for (int k = 0; k < 3; ++k) {
                           fx[k] = m.fdx[3 * e + k];
                           fy[k] = m.fdy[3 * e + k];
                         }
                         return m.areas[e];
                       });
  s.alphal[e] = al;
  // the passes that read ALPHAL take 1 unless this is set
  if (al != 1.0) atomicOr(&flags[F_ALPHA], 1);
  return al;
}

__global__ __launch_bounds__(256) void k_wd_alpha(DevMesh m, DevState s, int* flags, double slim) {
  int e = xcd_tile(blockIdx.x, gridDim.x) * blockDim.x + threadIdx.x;
  if (e >= m.ne) return;
  wd_alpha(m, s, e, flags, slim);
}

__global__ __launch_bounds__(256) void k_h2(int np, const double* __restrict__ dp, const double* __restrict__ eta2,
                     double ifnlfa, double* __restrict__ h2) {
  int i = xcd_tile(blockIdx.x, gridDim.x) * blockDim.x + threadIdx.x;
  if (i >= np) return;
  h2[i] = dp[i] + ifnlfa * eta2[i];
}

__global__ __launch_bounds__(256) void k_fill_u32(unsigned* p, unsigned v, int n) {
  int i = xcd_tile(blockIdx.x, gridDim.x) * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}

__global__ __launch_bounds__(256) void k_fill_i32(int* p, int v, int n) {
  int i = xcd_tile(blockIdx.x, gridDim.x) * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}

__global__ void k_run_clear(int* flags) {
  if (threadIdx.x == 0)
    flags[F_ITSUM] = flags[F_NREBUILD] = flags[F_NITMAX] = flags[F_MLUSED] = 0;
}

// TotalArea / MJU at cold start (src/mesh.F:3360-3400), node gather.
__global__ __launch_bounds__(256) void k_total_area(DevMesh m, DevState s) {
  int i = xcd_tile(blockIdx.x, gridDim.x) * blockDim.x + threadIdx.x;
  if (i >= m.np) return;
  int mju = 0;
  double ta = 0.0;
  for (int p = m.inc_ptr[i]; p < m.inc_ptr[i + 1]; ++p) {
    const int e = m.inc[p] / 3;
    const int ncele = s.nodecode[m.nm[3 * e]] * s.nodecode[m.nm[3 * e + 1]] *
                      s.nodecode[m.nm[3 * e + 2]] * s.noff[e];
    mju += ncele;
    ta = ta + (double)ncele * m.areas[e] / 2.0;
  }
  if (mju == 0) mju = 1;
  s.mju[i] = mju;
  s.totalarea[i] = ta;
}

}  // namespace adcgpu
