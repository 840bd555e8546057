// ITPACK jcg (src/itpackv.F:63-456) with the matrix on the chip and one
// exchange between blocks per iteration: the solver of every context whose
// matrix bandwidth lets a block keep the rows it references in LDS.
//
// What bounds it: the exchanges' latency.  A solve of 15 iterations needs the
// matrix once (12 bytes per entry) but, with the entries read again by every
// iteration, spent 13 us of each 29 us iteration at 1M rows on them, and the
// rest on three waits in a row (grid barrier, partials, neighbours).  So:
//
// - Rows.  A block of 512 threads owns CPB 2048-row chunks; thread t holds
//   rows t + 512 r of each.  Two waves per SIMD leave 256 VGPRs a thread: the
//   scaled entries of the first W off-diagonal slots of its rows and their
//   16-bit LDS positions (8 rows x 6 slots or 4 x 8: 15-20 VGPRs a row), u, the
//   previous u and d, and N d.  The few entries past W are kept in LDS.  d of
//   the block's rows and of all rows they reference is in LDS.
// - Partials.  Each chunk's three inner-product values go straight to a slot
//   of their own; every block polls all of them, a value being its own arrival
//   flag (a slot holds JCG_EMPTY until it is written).  Barrier and reduction
//   are one trip instead of three (two counter levels, generation word,
//   partials).  A slot is written in iterations in, in+4, ..; its owner marks
//   it empty in iteration in+3.  By then every row block has read it (all have
//   published in+2, hence passed the wait of in+1), and so has the eigenvalue
//   block, whose estimate of in+1 (or in+2) was needed to pass the wait of in+2; and nobody
//   waits on the slot of in+4 before all have published in+3.
// - Neighbours.  N d is published before the partials, so a block that has
//   seen all partials can read its neighbours' N d and form their new d by
//   itself (the owner's operations on the owner's values): the update needs no
//   wait of its own.  Two buffers suffice: in+2 is written after all have
//   published in+1, hence read in.
// - The eigenvalue estimate (chgcon) runs in a block of its own: a serial chain, a
//   root search of some nine evaluations, 3.6 to 7 us with the tridiagonal in LDS.
//   With one chunk per block that is longer than a row block's own 4.7 us, and
//   only the stopping test takes the result: such blocks test iteration `in` while
//   they wait for the partials of in+1 (LATE).  By then u has moved on by one
//   update, and the iterate before is still held.  With two chunks per block
//   (14 us an iteration) the half iteration done past the halt costs more than
//   the wait (20 steps at 999,151 rows: 15.58 ms late, 15.10 at once).  The
//   tridiagonal is kept in registers during a search.
//   The estimates have four slots: that of in is read in in or in+1, and its slot
//   is marked empty in in+3, when all have published in+2, hence passed the wait
//   of in+1.
//
// The sums' trees, the rows' operations and the scalar recurrences are those
// of k_jcg; results are the same bits.
// Measured (MI355X, FP64, about 15 iterations; us per launch, k_jcg before):
// 5,151 rows 102 (248), 20,646 rows 110 (257), 250,244 rows 121 (276),
// 999,151 rows 244 (447); with every test at once 128, 133, 146, 251.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "jcg_device.h"
#include "kernels.h"
#include "reduce.h"

namespace adcgpu {

// One bounded wait (an object per wait, so that the bound is each wait's own and
// nothing of it is kept in registers between waits): every 64th unsuccessful poll
// looks at the error flag and at the clock; a wait that runs out sets the flag, so
// every block drains.
//
// An ordinary launch (JcgArgs::admit) may find part of the chip taken by blocks
// that wait for it in turn.  Each block counts itself in when it starts; a wait
// that lasts admit_ticks while some block has not started gives the launch up: the
// abort bit is set (by an exchange on the count, so never once all have
// started), every block leaves, and nothing but scratch has been written: no block
// gets past the second iteration's waits before all have started.  k_jcg_mem,
// enqueued behind, then solves the system with two blocks.
struct BoundedWait {
  const JcgArgs& a;
  int* err;
  unsigned blocks;
  long long t0 = 0;
  unsigned polls = 0;
  __device__ BoundedWait(const JcgArgs& a, int nblocks)
      : a(a), err(a.flags + F_ERROR), blocks((unsigned)nblocks) {}
  __device__ __forceinline__ bool more() {
    if ((++polls & 63u) != 0) return true;
    if (__hip_atomic_load(err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) & ERR_BARRIER)
      return false;
    const long long t = wall_clock64();
    if (t0 == 0) t0 = t;
    if (a.admit) {
      unsigned v = __hip_atomic_load(a.admit, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if (v & JCG_ABORT) return false;
      if (v != blocks) {
        if (t - t0 <= a.admit_ticks) return true;
        return !__hip_atomic_compare_exchange_strong(a.admit, &v, v | JCG_ABORT, __ATOMIC_RELAXED,
                                                     __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
    }
    if (t - t0 <= a.barrier_ticks) return true;
    atomicOr(err, ERR_BARRIER);
    return false;
  }
};

__device__ __forceinline__ bool is_empty(double v) {
  return (unsigned long long)__double_as_longlong(v) == JCG_EMPTY;
}
__device__ __forceinline__ void put_bits(double* p, unsigned long long b) {
  __hip_atomic_store(reinterpret_cast<unsigned long long*>(p), b, __ATOMIC_RELAXED,
                     __HIP_MEMORY_SCOPE_AGENT);
}
// Publishes v (a NaN that would read as empty as another NaN).
__device__ __forceinline__ void publish(double* p, double v) {
  put_bits(p, is_empty(v) ? 0x7ff8000000000000ull
                          : (unsigned long long)__double_as_longlong(v));
}
// A row's value for the blocks that reference the row (written through to
// memory; the vectors are padded to whole tiles).
__device__ __forceinline__ void publish_vec(double* v, int i, double x) {
  __hip_atomic_store(&at(v, (unsigned)i), x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// All of this wave's stores have reached memory (they are written through).
__device__ __forceinline__ void stores_done() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

// The cross-chunk sums of slot `part` into lds (sum4 of each four): thread
// t < 256 waits for chunks t and t + 256 and adds them in that order, then the
// butterfly.  t: the thread's index.  A thread whose wait failed sets *failed.
// lds: 12 doubles.
__device__ __forceinline__ void poll_partials(int t, const double* part, int nch, double* lds,
                                              int* failed, const JcgArgs& args, int nblocks) {
  if (t < RED_XTHREADS) {
    BoundedWait w(args, nblocks);
    double r0 = 0.0, r1 = 0.0, r2 = 0.0;
    if (t < nch) {
      const double* p = part + 4 * t;
      const bool two = t + RED_XTHREADS < nch;
      const double* q = two ? p + 4 * RED_XTHREADS : p;
      double a0, a1, a2, b0, b1, b2;
      for (;;) {
        a0 = ld_agent(p);
        a1 = ld_agent(p + 1);
        a2 = ld_agent(p + 2);
        b0 = ld_agent(q);
        b1 = ld_agent(q + 1);
        b2 = ld_agent(q + 2);
        if (!(is_empty(a0) || is_empty(a1) || is_empty(a2) || is_empty(b0) || is_empty(b1) ||
              is_empty(b2)))
          break;
        if (!w.more()) {
          *failed = 1;
          break;
        }
      }
      r0 = 0.0 + a0;
      r1 = 0.0 + a1;
      r2 = 0.0 + a2;
      if (two) {
        r0 = r0 + b0;
        r1 = r1 + b1;
        r2 = r2 + b2;
      }
    }
    r0 = wave_sum(r0);
    r1 = wave_sum(r1);
    r2 = wave_sum(r2);
    if ((t & 63) == 0) {
      lds[t >> 6] = r0;
      lds[4 + (t >> 6)] = r1;
      lds[8 + (t >> 6)] = r2;
    }
  }
}
__device__ __forceinline__ double sum4(const double* v) { return (v[0] + v[1]) + (v[2] + v[3]); }

// Whether iteration `in` forms u.u, by the state after the test of in-1.
__device__ __forceinline__ bool reg_need_u(const ItLocal& L, int in) {
  return !(L.q1 || (in > 5 && (in % 5) != 0));
}

// The LDS that the eigenvalue block and the row blocks share the use of.
struct RegShared {
  ItLocal L;
  double lds[12];
  double dn, uu;          // d.d and u.u of the last iteration, not tested yet
  double gamold, rhoold;  // as they were before its parcon
  int failed, ovn;
};

// The eigenvalue block: the adaptive estimate of each iteration beside the row
// blocks' products.  Its cycle sets the pace of most solves, so its first wave
// does only what the next estimate hangs on: the state is in its registers, the
// same in every lane, and the stopping test, which only tells the block when to
// leave, is made by another wave beside the next estimate (14,300 cycles an
// iteration with the test before it).
template <bool DUAL>
__device__ __forceinline__ void jcg_reg_eig(const JcgArgs& a, RegShared& sh, int nblocks) {
  __shared__ double tri1[JCG_MAX_ITMAX], tri2[JCG_MAX_ITMAX];
  __shared__ double cmes[2];
  const int t = threadIdx.x;
  const int nch = (a.n + RED_CHUNK - 1) / RED_CHUNK;
  auto slot = [&](int k) { return a.part + (size_t)k * 4 * (nch + 1); };
  ItLocal m = sh.L;  // the first wave's: the estimate and the recurrence; the second's: the test
  double dn = 0.0, uu = 0.0;
  for (int in = 0; in <= a.itmax; ++in) {
    if (t < 64) {
      if (t < 2) put_bits(slot((in + 1) & 3) + 4 * nch + t, JCG_EMPTY);
      m.in = in;
      if (in_wave(m.adapt != 0)) jcg_chgcon<true>(m, tri1, tri2);
      stores_done();
      if (t < 2) publish(slot(in & 3) + 4 * nch + t, t == 0 ? m.cme : m.cmold);
      if (t == 0) cmes[in & 1] = m.cme;
    } else if (t == 64 && in > 0) {
      m.in = in - 1;
      m.cme = cmes[(in - 1) & 1];
      jcg_pstop(m, reg_need_u(m, in - 1) ? uu : 1.0, dn);
      sh.L.halt = m.halt;
    }
    __syncthreads();
    // (row blocks that have stopped may publish no more partials)
    if (sh.L.halt) break;
    poll_partials(t, slot(in & 3), nch, sh.lds, &sh.failed, a, nblocks);
    __syncthreads();
    if (sh.failed) return;
    if (t < 64) {
      m.delnnm = sum4(sh.lds);
      jcg_parcon(m, sum4(sh.lds + 4), in);
    } else if (t == 64) {
      dn = sum4(sh.lds);
      uu = sum4(sh.lds + 8);
    }
  }
}

// An estimate into the block's state (one thread of a row block).
__device__ __forceinline__ bool reg_pair(RegShared& sh, const double* pair, const JcgArgs& a,
                                         int nblocks) {
  BoundedWait w(a, nblocks);
  double c0, c1;
  for (;;) {
    c0 = ld_agent(pair);
    c1 = ld_agent(pair + 1);
    if (!(is_empty(c0) || is_empty(c1))) break;
    if (!w.more()) {
      sh.failed = 1;
      return false;
    }
  }
  sh.L.cme = c0;
  sh.L.cmold = c1;
  return true;
}
// The stopping test of the iteration before (LATE): touches what parcon does not.
__device__ __forceinline__ void reg_test(RegShared& sh, const double* pair, int in,
                                         const JcgArgs& a, int nblocks) {
  if (!reg_pair(sh, pair, a, nblocks)) return;
  sh.L.in = in;
  jcg_pstop(sh.L, reg_need_u(sh.L, in) ? sh.uu : 1.0, sh.dn);
}

// `bid` and `nblocks`: this block's index among the blocks that solve this
// system, and their number (row blocks and the eigenvalue block).
template <bool DUAL, int CPB>
__device__ __forceinline__ void jcg_solve_reg(const JcgArgs& a, int bid, int nblocks) {
  constexpr int R = RED_PER_THREAD * CPB;                   // rows per thread
  constexpr int W = CPB == 1 ? JCG_REG_W1 : JCG_REG_W2;     // entries per row in registers
  constexpr int TILE = CPB * RED_CHUNK;
  constexpr int K = CPB == 1 ? 6 : 10;  // neighbouring rows per thread read ahead
  constexpr bool LATE = CPB == 1;       // the stopping test one iteration late
  __shared__ RegShared sh;
  __shared__ double wsum[CPB][24];
  extern __shared__ double dsh[];
  const int np = a.n;
  const int t = threadIdx.x;
  const int nch = (np + RED_CHUNK - 1) / RED_CHUNK;
  const int nrb = nblocks - 1;
  // a bound of zero allows no wait at all (the host forces the error path
  // this way): the solve is left before anything is written
  if (a.barrier_ticks <= 0) {
    if (t == 0) atomicOr(a.flags + F_ERROR, ERR_BARRIER);
    return;
  }
  if (t == 0) {
    jcg_init_state(sh.L, a);
    sh.failed = 0;
    sh.ovn = 0;
    // (a launch given up before this block started is left at once)
    if (a.admit && (atomicAdd(a.admit, 1u) & JCG_ABORT)) sh.failed = 1;
  }
  if (bid == nrb) {  // the last block: no rows
    __syncthreads();
    if (sh.failed) return;
    jcg_reg_eig<DUAL>(a, sh, nblocks);
    return;
  }
  const int lane = t & 63, wave = t >> 6;
  const int tile = xcd_tile(bid, nrb);
  const int c0 = tile * CPB;  // first chunk
  const int t0 = tile * TILE, t1 = t0 + TILE < np ? t0 + TILE : np;
  // the window: rows lo .. hi-1, all that the block's rows reference
  int lo = t0, hi = t1;
  for (int c = c0; c < c0 + CPB && c < nch; ++c) {
    lo = a.hrange[2 * c] < lo ? a.hrange[2 * c] : lo;
    hi = a.hrange[2 * c + 1] > hi ? a.hrange[2 * c + 1] : hi;
  }
  // (rows of the last tile past the system's end are kept as rows of zeros)
  const int nlo = t0 - lo, nh = nlo + (hi - t1), win = nh + TILE;
  // dynamic LDS: the window's d and a zero (read by empty slots), the entries
  // past W, then the neighbouring rows' previous d as far as it goes
  double* const ovc = dsh + win + 1;
  unsigned short* const ovp = reinterpret_cast<unsigned short*>(ovc + a.ovf);
  double* const hprev = ovc + a.ovf + (a.ovf + 3) / 4;
  const int hcap = a.lds_doubles - (int)(hprev - dsh);
  double* const hmem = a.hprev + (size_t)tile * a.hmem;
  auto slot = [&](int k) { return a.part + (size_t)k * 4 * (nch + 1); };
  if (t == 0) dsh[win] = 0.0;

  double sc[R][W];            // scaled off-diagonals
  unsigned ps[R][W / 2];      // their window positions, two to a word
  int ovb = 0;                // entries past W of these rows: first index in ovc,
  unsigned ovn[(R + 3) / 4];  // and one count byte per row
#pragma unroll
  for (int k = 0; k < (R + 3) / 4; ++k) ovn[k] = 0;
  double uc[R], up[R], dp[R], nd[R];
  int tl = t;  // this thread's first row within the tile
#define OFS(q) (tl + ((q) >> 2) * RED_CHUNK + RED_THREADS * ((q) & 3))
#define ROW(q) (t0 + OFS(q))
#define OWN(q) dsh[nlo + OFS(q)]
#define NOV(q) ((int)((ovn[(q) >> 2] >> (8 * ((q) & 3))) & 255u))
#define POS(q, j) (((j) & 1) ? ps[q][(j) >> 1] >> 16 : ps[q][(j) >> 1] & 0xffffu)
  // Values that the compiler would keep expanded across the iterations (window
  // addresses, row offsets) are made opaque at each use: recomputing them is a
  // few integer instructions, keeping them spilled registers.
  auto opaque = [&]() {
    asm volatile("" : "+v"(tl));
#pragma unroll
    for (int q = 0; q < R; ++q)
#pragma unroll
      for (int j = 0; j < W / 2; ++j) asm volatile("" : "+v"(ps[q][j]));
  };

  // ---- scal (src/itpackv.F:2374-2400): the diagonal part was done by the
  // pass before; the off-diagonals here, w of the window in LDS
  auto stage = [&](const double* v) {
    for (int k = t; k < win; k += RED_THREADS)
      dsh[k] = lo + k < np ? at(v, (unsigned)(lo + k)) : 0.0;
  };
  stage(a.w);
  __syncthreads();
  if (sh.failed) return;
#pragma unroll
  for (int q = 0; q < R; ++q) {
    const int i = ROW(q);
    const int nn = i < np ? at(a.nneigh, (unsigned)i) : 1;
    const double wi = OWN(q);
    // chunk-relative positions to window positions
    const int adj = t0 + (q >> 2) * RED_CHUNK - a.hrows - lo;
#pragma unroll
    for (int j = 0; j < W; ++j) {
      unsigned pos = (unsigned)win;
      double v = 0.0;
      if (j + 1 < nn) {
        const unsigned wd = at(a.lcol, (unsigned)((j >> 1) * np + i));
        pos = (unsigned)((int)((j & 1) ? wd >> 16 : wd & 0xffffu) + adj);
        v = at(a.coef, (unsigned)((j + 1) * np + i)) * wi * dsh[pos];
      }
      sc[q][j] = v;
      ps[q][j >> 1] = (j & 1) ? ps[q][j >> 1] | (pos << 16) : pos;
    }
    if (nn > W + 1) ovn[q >> 2] |= (unsigned)(nn - 1 - W) << (8 * (q & 3));
    if (q & 1) __builtin_amdgcn_sched_barrier(0);
  }
  {
    int m = 0;
#pragma unroll
    for (int q = 0; q < R; ++q) m += NOV(q);
    if (m > 0) {
      ovb = atomicAdd(&sh.ovn, m);
      int o = ovb;
#pragma unroll 1
      for (int q = 0; q < R; ++q) {
        const int i = ROW(q), n = NOV(q);
        const int adj = t0 + (q >> 2) * RED_CHUNK - a.hrows - lo;
        for (int k = 0; k < n; ++k, ++o) {
          const int j = W + k;
          const unsigned wd = at(a.lcol, (unsigned)((j >> 1) * np + i));
          const int pos = (int)((j & 1) ? wd >> 16 : wd & 0xffffu) + adj;
          ovc[o] = at(a.coef, (unsigned)((j + 1) * np + i)) * OWN(q) * dsh[pos];
          ovp[o] = (unsigned short)pos;
        }
      }
    }
  }
  __syncthreads();

  // v[q] less N times the vector in the window, for all rows (the rows' slots
  // in order; an empty slot adds 0 * 0)
  auto product = [&](double* v) {
#pragma unroll
    for (int q = 0; q < R; ++q) {
#pragma unroll
      for (int j = 0; j < W; ++j) v[q] = v[q] - sc[q][j] * dsh[POS(q, j)];
      if (q & 1) __builtin_amdgcn_sched_barrier(0);  // two rows' gathers in flight
    }
    if ((R > 4 ? ovn[0] | ovn[(R - 1) >> 2] : ovn[0]) != 0) {
      int o = ovb;
#pragma unroll
      for (int q = 0; q < R; ++q)
        for (int n = NOV(q); n > 0; --n, ++o) v[q] = v[q] - ovc[o] * dsh[ovp[o]];
    }
  };
  auto chunk_value = [&](const double* v) {
    return ((v[0] + v[1]) + (v[2] + v[3])) + ((v[4] + v[5]) + (v[6] + v[7]));
  };

  // ---- d0 = rhs - N u - u (src/itpackv.F:346-353), published
  // (nd holds it until the window is staged)
  auto start = [&](const double* u, double* to, int k) {
    stage(u);
#pragma unroll
    for (int q = 0; q < R; ++q) nd[q] = ROW(q) < np ? at(a.rhs, (unsigned)ROW(q)) : 0.0;
    __syncthreads();
    product(nd);
#pragma unroll
    for (int g = 0; g < CPB; ++g) {
      double s = 0.0;
#pragma unroll
      for (int q = g * RED_PER_THREAD; q < (g + 1) * RED_PER_THREAD; ++q) {
        nd[q] = nd[q] - OWN(q);
        publish_vec(to, ROW(q), nd[q]);
        s = s + nd[q] * nd[q];
      }
      if (DUAL) {  // |d0|^2 of the chunk, in the inner-product tree
        s = wave_sum(s);
        if (lane == 0) wsum[g][8 * k + wave] = s;
      }
    }
  };
  if (DUAL) {
    start(a.u2, a.d, 1);
    __syncthreads();
  }
  start(a.u, a.ndv, 0);
#pragma unroll
  for (int q = 0; q < R; ++q) {
    uc[q] = OWN(q);
    up[q] = dp[q] = 0.0;
  }
  stores_done();
  __syncthreads();
  if (t < 3 * CPB) {
    const int g = t / 3, k = t % 3, c = c0 + g;
    if (c < nch) publish(slot(3) + 4 * c + k, DUAL && k < 2 ? chunk_value(wsum[g] + 8 * k) : 0.0);
  }
  const double* dv = a.ndv;
  int flip = 0;  // N d of even iterations goes to a.ndv: a.d holds the start
  if (DUAL) {
    poll_partials(t, slot(3), nch, sh.lds, &sh.failed, a, nblocks);
    __syncthreads();
    if (sh.failed) return;
    // the start with the smaller initial pseudo-residual
    const double r0 = sum4(sh.lds), r1 = sum4(sh.lds + 4);
    if (t == 0 && bid == 0) {
      a.saved[10] = r0;
      a.saved[11] = r1;
      if (r1 < r0) a.flags[F_MLUSED] += 1;
    }
    if (r1 < r0) {
      dv = a.d;
      flip = 1;
#pragma unroll
      for (int q = 0; q < R; ++q) {
        const int i = ROW(q);
        uc[q] = i < np ? at(a.u2, (unsigned)i) : 0.0;
        nd[q] = ld_agent(&at(a.d, (unsigned)i));
      }
    }
    __syncthreads();  // sh.lds is read before it is written again
  } else {
    // the chunks the window's rows belong to (this block reads nobody else's)
    const int ca = lo / RED_CHUNK, cb = (hi - 1) / RED_CHUNK;
    for (int c = ca + t; c <= cb; c += RED_THREADS) {
      const double* p = slot(3) + 4 * c;
      BoundedWait wait(a, nblocks);
      while (is_empty(ld_agent(p)))
        if (!wait.more()) {
          sh.failed = 1;
          break;
        }
    }
    __syncthreads();
    if (sh.failed) return;
  }
  // the window's d, the neighbouring rows' previous d
#pragma unroll
  for (int q = 0; q < R; ++q) OWN(q) = nd[q];
  for (int k = t; k < nh; k += RED_THREADS) {
    const int x = k < nlo ? k : k + TILE;
    dsh[x] = ld_agent(&at(dv, (unsigned)(lo + x)));
    if (k < hcap) hprev[k] = 0.0;
    else hmem[k - hcap] = 0.0;
  }
  __syncthreads();

  // ---- iterations
  for (int in = 0; in <= a.itmax; ++in) {
    opaque();
    // u.u is formed where the test will take it (LATE: q1 is the last call's at
    // first, cleared by the first test, then at most one test old, and only ever
    // set)
    const bool need_u = (LATE && in == 1) || reg_need_u(sh.L, in);
    double* const pv = ((in ^ flip) & 1) ? a.ndv : a.d;
    if (in >= 2 && tl < 3 * CPB && c0 + tl / 3 < nch)
      put_bits(slot((in + 1) & 3) + 4 * (c0 + tl / 3) + tl % 3, JCG_EMPTY);
    // N d, published for the neighbours; the rows' partials
#pragma unroll
    for (int q = 0; q < R; ++q) nd[q] = 0.0;
    product(nd);
#pragma unroll
    for (int g = 0; g < CPB; ++g) {
      double add = 0.0, adt = 0.0, auu = 0.0;
#pragma unroll
      for (int q = g * RED_PER_THREAD; q < (g + 1) * RED_PER_THREAD; ++q) {
        publish_vec(pv, ROW(q), nd[q]);
        const double dc = OWN(q);
        add = add + dc * dc;
        adt = adt + dc * nd[q];
      }
      if (need_u) {
#pragma unroll
        for (int q = g * RED_PER_THREAD; q < (g + 1) * RED_PER_THREAD; ++q)
          auu = auu + uc[q] * uc[q];
      }
      const double x0 = wave_sum(add), x1 = wave_sum(adt), x2 = need_u ? wave_sum(auu) : 0.0;
      if (lane == 0) {
        wsum[g][wave] = x0;
        wsum[g][8 + wave] = x1;
        wsum[g][16 + wave] = x2;
      }
    }
    stores_done();
    __syncthreads();
    if (tl < 3 * CPB) {
      const int g = tl / 3, k = tl % 3, c = c0 + g;
      if (c < nch) publish(slot(in & 3) + 4 * c + k, chunk_value(wsum[g] + 8 * k));
    }
    if (t == RED_XTHREADS) {
      if (!LATE) reg_pair(sh, slot(in & 3) + 4 * nch, a, nblocks);
      else if (in > 0) reg_test(sh, slot((in - 1) & 3) + 4 * nch, in - 1, a, nblocks);
    }
    poll_partials(tl, slot(in & 3), nch, sh.lds, &sh.failed, a, nblocks);
    __syncthreads();
    if (sh.failed) return;
    if (LATE && sh.L.halt) break;
    // the neighbours' N d on its way while thread 0 forms the scalars
    double x[K];
#pragma unroll
    for (int m = 0; m < K; ++m) {
      const int k = tl + m * RED_THREADS;
      if (k < nh) x[m] = ld_agent(&at(pv, (unsigned)(lo + (k < nlo ? k : k + TILE))));
    }
    if (t == 0) {
      sh.L.delnnm = sum4(sh.lds);
      if (LATE) {
        sh.gamold = sh.L.gamold;
        sh.rhoold = sh.L.rhoold;
        sh.dn = sh.L.delnnm;
        sh.uu = sum4(sh.lds + 8);
      } else {
        sh.L.in = in;
        jcg_pstop(sh.L, need_u ? sum4(sh.lds + 8) : 1.0, sh.L.delnnm);
      }
      if (LATE || !sh.L.halt) jcg_parcon(sh.L, sum4(sh.lds + 4), in);
    }
    __syncthreads();
    if (!LATE && sh.L.halt) break;
    const double k1 = sh.L.c1, k2 = sh.L.c2, k3 = sh.L.c3, k4 = sh.L.c4;
#pragma unroll
    for (int q = 0; q < R; ++q) {
      const double dc = OWN(q);
      const double un = k1 * dc + k2 * uc[q] + k3 * up[q];
      const double dn = k1 * nd[q] + k4 * dc + k3 * dp[q];
      up[q] = uc[q];
      uc[q] = un;
      dp[q] = dc;
      OWN(q) = dn;
    }
    // the neighbouring rows: the owner's update on the owner's values
    for (int b = 0; b * K * RED_THREADS < nh; ++b) {
      const int kb = tl + b * K * RED_THREADS;
      if (b > 0) {
#pragma unroll
        for (int m = 0; m < K; ++m) {
          const int k = kb + m * RED_THREADS;
          if (k < nh) x[m] = ld_agent(&at(pv, (unsigned)(lo + (k < nlo ? k : k + TILE))));
        }
      }
#pragma unroll
      for (int m = 0; m < K; ++m) {
        const int k = kb + m * RED_THREADS;
        if (k < nh) {
          const int y = k < nlo ? k : k + TILE;
          const double dc = dsh[y];
          if (k < hcap) {
            dsh[y] = k1 * x[m] + k4 * dc + k3 * hprev[k];
            hprev[k] = dc;
          } else {
            dsh[y] = k1 * x[m] + k4 * dc + k3 * hmem[k - hcap];
            hmem[k - hcap] = dc;
          }
        }
      }
    }
    __syncthreads();
  }
  // ITMAX iterations done: the test of the last one
  if (LATE && !sh.L.halt) {
    if (t == RED_XTHREADS) reg_test(sh, slot(a.itmax & 3) + 4 * nch, a.itmax, a, nblocks);
    __syncthreads();
    if (sh.failed) return;
  }
  // the result is the iterate of the last iteration index: the one before the
  // last update, unless the test halted before that update
  const bool halted = sh.L.halt != 0;
  if (LATE && t == 0 && halted) {
    sh.L.gamold = sh.gamold;
    sh.L.rhoold = sh.rhoold;
  }

  opaque();
  int o = ovb;
  // ---- unscal (src/itpackv.F:2424-2479), ETAS and ETA2 (src/gwce.F:2006-2008)
  if (!a.defer_unscal) {
    // the off-diagonals too: w of the window in LDS again
    __syncthreads();
    stage(a.w);
    __syncthreads();
  }
#pragma unroll
  for (int q = 0; q < R; ++q) {
    const int i = ROW(q);
    if (i < np) {
      const double wi = at(a.w, (unsigned)i);
      const double u = (!LATE && halted ? uc[q] : up[q]) * wi;
      const double ri = 1.0 / wi;
      at(a.coef, (unsigned)i) = ri * ri;
      at(a.rhs, (unsigned)i) = at(a.rhs, (unsigned)i) * ri;
      at(a.u, (unsigned)i) = u;
      if (a.eta2)
        at(a.eta2, (unsigned)i) =
            (double)at(a.nodecode, (unsigned)i) * (u + 0.0) + at(a.eta1, (unsigned)i);
      if (!a.defer_unscal) {
        const int nn = at(a.nneigh, (unsigned)i);
#pragma unroll
        for (int j = 0; j < W; ++j)
          if (j + 1 < nn)
            at(a.coef, (unsigned)((j + 1) * np + i)) = sc[q][j] * ri * (1.0 / dsh[POS(q, j)]);
        for (int j = W; j < nn - 1; ++j, ++o)
          at(a.coef, (unsigned)((j + 1) * np + i)) = ovc[o] * ri * (1.0 / dsh[ovp[o]]);
      }
    }
    if (q & 1) __builtin_amdgcn_sched_barrier(0);
  }
#undef OFS
#undef ROW
#undef OWN
#undef NOV
#undef POS
  if (bid == 0 && t == 0) jcg_finish(sh.L, a, halted);
}

template <bool DUAL, int CPB>
__global__ __launch_bounds__(RED_THREADS) void k_jcg_reg(JcgArgs a) {
  jcg_solve_reg<DUAL, CPB>(a, (int)blockIdx.x, (int)gridDim.x);
}

// Several systems in one cooperative launch, as k_jcg_batch.
template <bool DUAL, int CPB>
__global__ __launch_bounds__(RED_THREADS) void k_jcg_reg_batch(const JcgArgs* __restrict__ args,
                                                               const int* __restrict__ first,
                                                               int nsys) {
  const int b = blockIdx.x;
  int m = 0;
  while (m + 1 < nsys && first[m + 1] <= b) ++m;
  jcg_solve_reg<DUAL, CPB>(args[m], b - first[m], first[m + 1] - first[m]);
}

#define ADCGPU_INST(D, C)                       \
  template __global__ void k_jcg_reg<D, C>(JcgArgs); \
  template __global__ void k_jcg_reg_batch<D, C>(const JcgArgs*, const int*, int);
ADCGPU_INST(false, 1)
ADCGPU_INST(false, 2)
ADCGPU_INST(true, 1)
ADCGPU_INST(true, 2)
#undef ADCGPU_INST

}  // namespace adcgpu
