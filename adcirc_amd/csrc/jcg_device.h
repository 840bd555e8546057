// The scalar part of ITPACK's jcg shared by the solver kernels: its state, the
// adaptive eigenvalue estimate (chgcon, zbrent, determ), the stopping test
// (pstop) and the recurrence parameters (parcon).
#pragma once
#include <hip/hip_runtime.h>

#include "kernels.h"

namespace adcgpu {

// Element access through a 32-bit byte offset from a uniform base: the
// addresses then take the scalar-base + 32-bit-offset form of the vector
// memory instructions instead of one 64-bit VGPR pair per row.  Arrays here
// stay below 4 GiB (checked on the host).
template <class T>
__device__ __forceinline__ T& at(T* base, unsigned i) {
  return *reinterpret_cast<T*>(reinterpret_cast<char*>(base) + i * (unsigned)sizeof(T));
}
template <class T>
__device__ __forceinline__ const T& at(const T* base, unsigned i) {
  return *reinterpret_cast<const T*>(reinterpret_cast<const char*>(base) + i * (unsigned)sizeof(T));
}

// Agent-scope load of a value another block wrote (coherent across XCDs).
__device__ __forceinline__ double ld_agent(const double* p) {
  return __hip_atomic_load(const_cast<double*>(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

struct ItLocal {
  int in, adapt, halt, q1, maxfn, nsig, itmax, stop;
  double zeta, cme, gamma, rho, delnnm, delsnm, udnm, stptst, gamold, rhoold, cmold;
  double c1, c2, c3, c4, tz;
};

// determ (src/itpackv.F:1029-1068): the backward three-term recurrence with
// the two running values kept in registers (same operations, same order).
// The recurrence is a chain of one multiply and one add per row; the rows'
// values come from LDS four at a time, the next four loaded while these are
// used, so that the chain and not the LDS latency sets the pace.
__device__ __forceinline__ double jcg_determ(int n, const double* tri1, const double* tri2,
                                             double x) {
  double a2 = tri1[n - 1] - x;                            // wk2(n)
  double a1 = (tri1[n - 2] - x) * a2 + tri2[n - 1];       // wk2(n-1)
  double p[4], q[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const int r = n - 3 - k > 0 ? n - 3 - k : 0;
    p[k] = tri1[r];
    q[k] = tri2[r + 1];
  }
  for (int l = n - 3; l >= 0; l -= 4) {
    double pc[4], qc[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      pc[k] = p[k];
      qc[k] = q[k];
      const int r = l - 4 - k > 0 ? l - 4 - k : 0;
      p[k] = tri1[r];
      q[k] = tri2[r + 1];
    }
#pragma unroll
    for (int k = 0; k < 4; ++k)
      if (l - k >= 0) {
        const double w = (pc[k] - x) * a1 + qc[k] * a2;  // wk2(l-k)
        a2 = a1;
        a1 = w;
      }
  }
  return a1;
}

// The tridiagonal's values for the evaluations of one zbrent call.  REG: up to
// JCG_TRI_REG rows in registers, last row first (from LDS, whose latency exceeds
// the recurrence's, an evaluation takes twice as long); for kernels with
// registers to spare.
constexpr int JCG_TRI_REG = 20;
template <bool REG>
struct JcgTri {
  int n;
  const double *tri1, *tri2;
  double p[REG ? JCG_TRI_REG : 1], q[REG ? JCG_TRI_REG : 1];  // tri1, tri2 of row n-1-k
  __device__ __forceinline__ JcgTri(int n_, const double* t1, const double* t2)
      : n(n_), tri1(t1), tri2(t2) {
    if (REG) {
#pragma unroll
      for (int k = 0; k < (REG ? JCG_TRI_REG : 1); ++k) {
        const int r = n - 1 - k > 0 ? n - 1 - k : 0;
        p[k] = tri1[r];
        q[k] = tri2[r];
      }
    }
  }
  template <int K>
  __device__ __forceinline__ double rows(double a1, double a2, double x) const {
    if constexpr (K < JCG_TRI_REG) {
      if (K < n) return rows<K + 1>((p[K] - x) * a1 + q[K - 1] * a2, a1, x);
    }
    return a1;
  }
  // determ: the same operations in the same order from either place
  __device__ __forceinline__ double operator()(double x) const {
    if constexpr (REG) {
      if (n <= JCG_TRI_REG) {
        const double a2 = p[0] - x;
        return rows<2>((p[1] - x) * a2 + q[0], a2, x);
      }
    }
    return jcg_determ(n, tri1, tri2, x);
  }
};

// A condition that holds in all lanes or in none, as a scalar branch.
__device__ __forceinline__ bool in_wave(bool c) { return __ballot(c) != 0ull; }

// zbrent (src/itpackv.F:2521-2781) with eps = 0; returns ier, result in *pb.
// Called by a whole wave, whose lanes all follow the same path; lanes 0 and 1
// evaluate the two ends of the interval at once.  The three quotients of the
// interpolation are formed side by side, whether the step takes them or not:
// the call is one chain of latencies.
template <bool REG>
__device__ __forceinline__ int jcg_zbrent(int n, const double* tri1, const double* tri2, double t, int maxfn,
                          double a, double* pb) {
  double b = 1.0, c = 0, d = 0, e = 0, p, qq, r, ss, fa, fb, fc = 0, tol, rm, rone, temp;
  int ic = 2;
  const double eps = 0.0;
  const JcgTri<REG> determ(n, tri1, tri2);
  {
    const double f = determ((threadIdx.x & 63) == 1 ? b : a);
    fa = __shfl(f, 0, 64);
    fb = __shfl(f, 1, 64);
  }
  if (in_wave((fa > 0.0 && fb > 0.0) || (fa < 0.0 && fb < 0.0))) {
    *pb = b;
    return 502;
  }
  bool reset = true;
  while (true) {
    if (reset) {
      c = a; fc = fa; d = b - c; e = d;
    }
    if (in_wave(!(fabs(fc) >= fabs(fb)))) {
      a = b; b = c; c = a; fa = fb; fb = fc; fc = fa;
    }
    tol = t * fmax(fabs(b), 0.1);
    rm = (c - b) * 0.5;
    if (in_wave(fabs(fb) <= eps || fabs(c - b) <= tol)) { *pb = b; return 0; }
    if (ic >= maxfn) { *pb = b; return 501; }
    bool bisect = in_wave((fabs(e) < tol) || (fabs(fa) <= fabs(fb)));
    if (!bisect) {
      ss = fb / fa;
      const double q3 = fa / fc, r3 = fb / fc;
      if (in_wave(a == c)) {
        p = (c - b) * ss;
        qq = 1.0 - ss;
      } else {
        qq = q3;
        r = r3;
        rone = r - 1.0;
        p = ss * ((c - b) * qq * (qq - r) - (b - a) * rone);
        qq = (qq - 1.0) * rone * (ss - 1.0);
      }
      if (p > 0.0) qq = -qq;
      if (p < 0.0) p = -p;
      ss = e;
      e = d;
      const double step = p / qq;
      if (in_wave(p + p >= 3.0 * rm * qq || p + p >= fabs(ss * qq))) {
        bisect = true;
      } else {
        d = step;
      }
    }
    if (bisect) { e = rm; d = e; }
    a = b;
    fa = fb;
    temp = d;
    if (fabs(temp) <= 0.5 * tol) temp = copysign(0.5 * tol, rm);
    b = b + temp;
    fb = determ(b);
    ic = ic + 1;
    reset = !in_wave(fb == 0.0 || fc == 0.0 || (fb > 0.0 && fc < 0.0) || (fb < 0.0 && fc > 0.0));
  }
}

// chgcon(ibmth=1) (src/itpackv.F:893-1027); tri1/tri2 are the two columns.
// Called by one whole wave with its own copy of the state in L (the lanes
// hold the same values); tri1, tri2 are in LDS and read by that wave only.
template <bool REG>
__device__ __forceinline__ void jcg_chgcon(ItLocal& L, double* tri1, double* tri2) {
  const int ip = L.in;
  double start = L.cme, end1;
  if (ip == 0) {
    end1 = 0.0;
    L.cmold = 0.0;
  } else if (ip == 1) {
    end1 = 1.0 - 1.0 / L.gamma;
    tri1[0] = end1;
    tri2[0] = 0.0;
  } else {
    if (fabs(start - L.cmold) <= L.zeta * start) {
      L.adapt = 0;
      return;
    }
    L.cmold = start;
    tri1[ip - 1] = 1.0 - 1.0 / L.gamma;
    tri2[ip - 1] = (1.0 - L.rho) / (L.rho * L.rhoold * L.gamma * L.gamold);
    double b;
    int ier = jcg_zbrent<REG>(ip, tri1, tri2, L.tz, L.maxfn, start, &b);
    if (ier != 0) {
      L.adapt = 0;
      return;
    }
    end1 = b;
  }
  L.cme = end1;
}

// The eigenvalue estimate of iteration `in` (one whole wave): chgcon on the
// wave's own copy of the state, its results back to L by lane 0.
template <bool REG>
__device__ __forceinline__ void jcg_eig_wave(ItLocal& L, double* tri1, double* tri2, int in) {
  ItLocal m = L;
  m.in = in;
  if (m.adapt) jcg_chgcon<REG>(m, tri1, tri2);
  if ((threadIdx.x & 63) == 0) {
    L.in = in;
    L.adapt = m.adapt;
    L.cme = m.cme;
    L.cmold = m.cmold;
  }
}

// pstop_nrms(iflag=1) (src/itpackv.F:809-890)
__device__ __forceinline__ void jcg_pstop(ItLocal& L, double unrm, double dnrm) {
  const double con = L.cme;
  double uold, tr, tl;
  L.halt = 0;
  if (L.in < 1) {
    L.q1 = 0;
    L.udnm = 1.0;
    L.stptst = 1000.0;
  }
  if (!(L.q1 || (L.in > 5 && (L.in % 5) != 0))) {
    uold = L.udnm;
    L.udnm = unrm;
    if (L.udnm == 0.0) L.udnm = 1.0;
    if (L.in > 5 && fabs(L.udnm - uold) <= L.udnm * L.zeta) L.q1 = 1;
  }
  tr = __builtin_sqrt(L.udnm);
  tl = 1.0;
  if (con != 1.0) {
    tl = __builtin_sqrt(dnrm);
    tr = tr * (1.0 - con);
  }
  L.stptst = tl / tr;
  if (tl >= tr * L.zeta) return;
  L.halt = 1;
}

// parcon(ibmth=1) (src/itpackv.F:1774-1851)
__device__ __forceinline__ void jcg_parcon(ItLocal& L, double dtnrm, int ip) {
  const double rhoold = L.rho;
  L.gamold = L.gamma;
  L.gamma = 1.0 / (1.0 - dtnrm / L.delnnm);
  L.rho = 1.0;
  if (ip != 0) L.rho = 1.0 / (1.0 - L.gamma * L.delnnm / (L.gamold * L.delsnm * rhoold));
  L.delsnm = L.delnnm;
  L.rhoold = rhoold;
  L.c1 = L.rho * L.gamma;
  L.c2 = L.rho;
  L.c3 = 1.0 - L.rho;
  L.c4 = L.rho * (1.0 - L.gamma);
}


// The solve's scalar state at the start of a launch: ITPACK's SAVEd values
// from the last solve, the rest cleared (thread 0).
__device__ __forceinline__ void jcg_init_state(ItLocal& L, const JcgArgs& a) {
  L.in = 0;
  L.adapt = 1;
  L.halt = 0;
  L.q1 = a.saved[0] != 0.0;
  L.gamold = a.saved[1];
  L.rhoold = a.saved[2];
  L.cmold = a.saved[3];
  L.itmax = a.itmax;
  L.zeta = a.zeta;
  L.cme = 0.0;
  L.gamma = 0.0;
  L.rho = 0.0;
  L.delnnm = 0.0;
  L.delsnm = 0.0;
  L.udnm = 0.0;
  L.stptst = 0.0;
  L.maxfn = a.maxfn;
  L.tz = a.tz;
  L.stop = 0;
}

// The solve's outcome and SAVEd state (block 0, thread 0).
__device__ __forceinline__ void jcg_finish(const ItLocal& L, const JcgArgs& a, bool halted) {
  const int in_final = halted ? L.in : a.itmax;
  a.flags[F_NUMITR] = in_final;
  a.flags[F_IER] = halted ? 0 : 13;
  a.saved[0] = L.q1 ? 1.0 : 0.0;
  a.saved[1] = L.gamold;
  a.saved[2] = L.rhoold;
  a.saved[3] = L.cmold;
  a.saved[4] = L.cme;
  a.saved[5] = L.stptst;
  a.flags[F_ITSUM] += in_final;
  if (!halted) a.flags[F_NITMAX] += 1;
}

}  // namespace adcgpu
