// Device-side data layout shared by the kernels and the host driver.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace adcgpu {

// fixed blocked reduction: 2048-row chunks of 512 threads x 4 rows; chunk
// values combined by 256 threads
constexpr int RED_THREADS = 512;
constexpr int RED_PER_THREAD = 4;
constexpr int RED_CHUNK = RED_THREADS * RED_PER_THREAD;
constexpr int RED_XTHREADS = 256;

// persistent JCG launch: one block per chunk plus one eigenvalue block
constexpr int JCG_CPB = 2;                      // 2048-row chunks per block
constexpr int JCG_BLOCK = RED_THREADS * JCG_CPB;  // threads per block
constexpr int JCG_BAR_GROUP = 16;        // blocks per first-level barrier counter
constexpr int JCG_BAR_STRIDE = 64;       // words between barrier counters (256 B)
constexpr int JCG_BAR_WORDS = 10240;     // barrier words: (groups + 2) * JCG_BAR_STRIDE
                                          // + blocks * JCG_HALO_STRIDE
constexpr int JCG_ADMIT_WORD = JCG_BAR_WORDS;  // admission word of an ordinary launch:
constexpr unsigned JCG_ABORT = 0x80000000u;      // blocks started, or given up
constexpr int JCG_HALO_STRIDE = 16;      // words between per-tile halo flags (64 B)
constexpr int JCG_HALO_MAX = 2;          // widest halo (tiles each side) waited on by flags
constexpr int JCG_MAX_ITMAX = 256;       // tridiagonal history length (itmax)
// k_jcg_reg: 2048-row chunks per 512-thread block, matrix entries per row in
// registers (by chunks per block), LDS it may use in all
constexpr int JCG_REG_W1 = 8, JCG_REG_W2 = 6;
constexpr int JCG_REG_LDS_BYTES = 152 * 1024;
// an empty partial slot: a quiet NaN no computation produces
constexpr unsigned long long JCG_EMPTY = 0xfff8badc0ffee000ull;
__host__ __device__ constexpr int jcg_part_doubles(int nch) { return 4 * 4 * (nch + 1); }
// dynamic LDS for the staged pseudo-residual of a k_jcg block (JcgArgs.hrows),
// at most: the block's rows and 5,632 rows each side
constexpr int JCG_STAGE_MAX_BYTES = 120 * 1024;
static_assert(JCG_STAGE_MAX_BYTES / 8 <= 65536, "staged positions are 16-bit");
// patches: a block's threads, and at most so many elements (one per thread),
// window nodes, and own nodes.  About 10 x 10 nodes have 235 elements: one per
// thread, and a fifth more element evaluations than the mesh has elements.
constexpr int PATCH_THREADS = 256, PATCH_ELEMS = 256, PATCH_WIN = 192, PATCH_NODES = 96;
static_assert(PATCH_NODES <= PATCH_THREADS / 2 && PATCH_WIN <= PATCH_THREADS, "patch shape");
constexpr int PATCH_GWCE_FIELDS = 18, PATCH_MOM_FIELDS = 13;
constexpr int patch_lds_bytes(int fields, int terms, int wmax) {
  return 8 * (fields * wmax > terms ? fields * wmax : terms);
}
constexpr int PATCH_GWCE_TERMS = 9 * PATCH_ELEMS + 1, PATCH_MOM_TERMS = 6 * PATCH_ELEMS;
constexpr int LHS_MAXW = 32;         // widest COEF row (MNEI) that a context takes
// ordered wetting updates: candidates are closed in blocks of WD_BLOCK, each
// block naming at most WD_XMAX earlier candidates it depends on
constexpr int WD_BLOCK = 1024;
constexpr int WD_XMAX = 256;                 // four 64-bit mask words per candidate
constexpr int WD_XW = WD_XMAX / 64;
constexpr int WD_HASH = 2 * WD_XMAX;         // LDS hash slots for a block's external names
constexpr int WD_INC_MAX = 12;               // incidence lists a wetting candidate scans at once
constexpr int WD_CLOSE_LDS = 2 * WD_BLOCK * (8 + 8 * WD_XW + 4) + 2 * WD_HASH * 4;
constexpr int WD_LINK_BLOCKS = 64;           // blocks whose link values fit the LDS of k_wd_chain
// serial fallback of k_wd_chain: candidates staged through LDS in chunks, the
// running maxima of the most recent WD_RING candidates kept in an LDS ring
constexpr int WD_CHUNK = 2048;
constexpr int WD_RING = 8192;   // power of two
constexpr int WD_SERIAL_LDS = WD_RING * 8 + WD_CHUNK * (8 + 8 + 8);
constexpr int WD_LINK_LDS = WD_LINK_BLOCKS * WD_XMAX * 8 > WD_SERIAL_LDS
                                ? WD_LINK_BLOCKS * WD_XMAX * 8 : WD_SERIAL_LDS;
constexpr int WD_CHAIN_LDS = WD_LINK_LDS > WD_CLOSE_LDS ? WD_LINK_LDS : WD_CLOSE_LDS;
constexpr int WD_TILES = 1024;        // 256-element tiles a block lists
constexpr int WD_CHAIN_BLOCKS = 32;  // blocks of k_wd_chain at most

// device flag slots
enum { F_NCCHANGE = 0, F_NUMITR = 2, F_IER, F_ERROR, F_NCAND, F_ITSUM, F_NREBUILD, F_WDSERIAL,
       F_ERRSTEP,  // first step that raised ERR_ELEV or ERR_NONFINITE (0: none)
       F_NITMAX,   // solves that reached ITMAX (ier = 13)
       F_ALPHA,    // some element's ALPHAL differs from 1 (otherwise the passes
                   // that use it do not read it)
       F_MLUSED,   // solves that started from the learned guess
       F_REBUILT,  // this step's GWCE matrix was rebuilt (k_lhs_ep)
       F_ALPHA0,   // F_ALPHA as the last step left it
       F_WDDONE,   // k_wd_chain's blocks that have ended
       F_COUNT = 16 };
enum { ERR_DIAG = 1, ERR_BARRIER = 4, ERR_ELEV = 8, ERR_NONFINITE = 16,
       ERR_INPUT = 32 };  // a system the drop-in refuses (k_na_compact): not solved
// device scalar slots
enum { S_EP = 0, S_COUNT = 8 };

struct DevMesh {
  int np, ne, mnei, neta;
  double dt, g, a00, b00, c00;
  const int* nm;        // [ne*3] 0-based
  const double* fdx;    // [ne*3]
  const double* fdy;    // [ne*3]
  const double* areas;  // [ne]
  const double* x;
  const double* y;
  const double* dp;
  const double* tau0;
  const double* evm;
  const double* corif;
  const int* inc_ptr;   // [np+1] node -> incident (element, local) codes 3e+k
  const int* inc;       //        sorted by element id
  const int* slot;      // [ne*3] position p of code 3e+k in inc (inc[slot[c]] == c)
  const int* slot_cols; // [ne*3] per slot p: CSR_POSITION slots ja | jb << 16 (0-based)
  const int* nneigh;    // [np]
  const int* col;       // [mnei*np] column-major, 0-based (slot 0 = self)
  const int* bnd_index; // [np] elevation-boundary index, -1, or -2-k for the
                        //      k-th node that takes specified-flux edge terms
  const int* nbd;       // [neta] 0-based
  const int* obcg_ptr;  // [np+1] node -> boundary-column slots, (I,J) order
  const int* obcg;
  const int* obcg_q;    //        and the COEF position j*np+i of each
  const int* vbc_ptr;   // [np+1] node -> flow-boundary entries in ME2GW order
  const int* vbc;
  const int* lbcodei;
  const double* csii;
  const double* siii;
  // specified normal flux boundaries (null without): per flux node k its
  // edge terms fb_ent[fb_ptr[k] .. fb_ptr[k+1]) in the reference's edge
  // order, each 2*J + r for the edge NBV(J-1)-NBV(J) (0-based J >= 1) with
  // r = 0 when the node is NBV(J-1), 1 when it is NBV(J)
  const int* fb_ptr;
  const int* fb_ent;
  const int* nbv;       // [nvel] 0-based
  const double* bndlen; // [nvel] BNDLEN2O3
};

struct DevState {
  double *eta1, *eta2, *etas, *uu1, *vv1, *uu2, *vv2, *qx1, *qy1, *qx2, *qy2;
  double *h1, *h2, *tk, *etamax, *totalarea, *wsx1, *wsy1, *wsx2, *wsy2, *pr1, *pr2;
  double *gwce_lv, *alphal, *coef, *obc, *fric;
  int *nodecode, *nnodecode, *noff, *mju;
  int *etamax_it;  // step of the last ETAMAX rise (0: never)
  double *umax;    // peak depth-averaged speed at wet nodes
  int *umax_it;    // step of the last UMAX rise (0: never)
  unsigned char* ncele;  // [nq] NCEle of each patch element (DevPatch) for the next GWCE
  double *tip1, *tip2;   // tidal potential at time levels s and s+1 (null: none)
  double *qn0, *qn1, *qn2;  // normal flux per flow-boundary entry at three time
                            // levels (null: no flux boundaries)
  double* qrad;             // per entry: the step's QFORCE of an outward-radiating
                            // entry (LBCODEI 30), or the radiation part of a
                            // river-radiation entry's (52), formed at the step's start
  double* elevdisc;         // per entry: river radiation's reference elevation
};

__global__ void k_flux_shift(DevMesh m, DevState s, const double* next, int nvel);

// The tidal potential of one step (src/timestep.F:1527-1557, NTIP = 1), per
// constituent: its species, ARGT (the phase at the step, reduced by whole
// periods) and TPMUL = RampTip*ETRF*TPK*FFT, formed on the host.
constexpr int TIP_MAX = 32;
struct TipPrm {
  int ntif;
  int na[TIP_MAX];
  double argt[TIP_MAX], tpmul[TIP_MAX];
};

// Patches (patch.h): per patch its own nodes, the elements at them and all nodes
// of those elements (the window), each list padded to its longest length.
struct DevPatch {
  int n, nq;            // patches; element slots over all patches, n PATCH_ELEMS
  int wmax;             // the largest window
  const int* win;       // [n][PATCH_WIN] window nodes: the patch's own, ascending, then the
                        //   others; -1: none
  const int* el;        // [nq] elements, ascending
  const ushort4* lv;    // [nq] window positions of an element's vertices; w: 1 if the first
                        //   is the patch's own (each element in exactly one patch), 2: none
  const ushort2* cspan; // [n][PATCH_NODES] per own node the span of its codes; y < x: none
  const unsigned short* code;  // [n][3 PATCH_ELEMS] k PATCH_ELEMS + element for vertex k of
                        //   the patch's element, in ascending element order per node
  const unsigned* pair; // [n][mnei-1][PATCH_NODES] per own node and column j >= 1 the two
                        //   codes of the edge terms it sums (3 PATCH_ELEMS: no term), low half
                        //   first; ~0: no such column; null when some edge has more than
                        //   two elements
  const double* geo;    // [7][nq] FDXE, FDYE, AREAS; null: formed from the coordinates
};

// FDXE, FDYE and AREAS of an element from its vertices' coordinates, as a
// reader of the grid forms them (src/mesh.F): the operations of prep.py's tables.
__host__ __device__ __forceinline__ void elem_geometry(double X1, double X2, double X3, double Y1,
                                                       double Y2, double Y3, double& fx1,
                                                       double& fx2, double& fx3, double& fy1,
                                                       double& fy2, double& fy3, double& area) {
  fx1 = -(Y3 - Y2);
  fx2 = -(Y1 - Y3);
  fx3 = -(Y2 - Y1);
  fy1 = X3 - X2;
  fy2 = X1 - X3;
  fy3 = X2 - X1;
  area = fy2 * fx1 + fy1 * (Y1 - Y3);
}

// Compensated (Kahan 1965) summation in FP32: the node sums of FP32
// element contributions in the mixed-precision path.  The result carries the
// compensation into FP64.
struct Kahan32 {
  float s = 0.0f, c = 0.0f;
  __device__ __forceinline__ void add(float x) {
    const float y = x - c;
    const float t = s + y;
    c = (t - s) - y;
    s = t;
  }
  __device__ __forceinline__ double value() const { return (double)s - (double)c; }
};

struct RhsPrm {
  double ifnlfa, ifnlct, ifnlcat;
  double ondiag, offdiag;  // (1+ILump)*2 and 1-ILump (src/gwce.F:419-420)
  int fric;                // TK formed by the pass itself
  int nws;
};

struct MomPrm {
  double ifnlct;
  int nws;
  int it;            // this step, recorded where ETAMAX rises
  double errorelev;  // ErrorElev: |ETA2| above it at a wet node stops the run
  int* flags;        // run-time error flags (ERR_ELEV, ERR_NONFINITE, F_ERRSTEP)
  int form_h2;       // without wet/dry: H2 = DP + IFNLFA*ETA2 formed by the pass
  double ifnlfa;
};

// Hybrid bottom friction (NOLIBF = 2): IFHYBF and fort.15's HBREAK, FTHETA,
// FGAMMA; `on` is 0 for the other friction laws.
struct Hybrid {
  double on, hbreak, ftheta, fgamma;
};

// IFHYBF*(1 + (HBREAK/H)**FTHETA)**(FGAMMA/FTHETA) (src/nodalattr.F:2406-2410,
// src/wetdry.F:415-418, 447-451): the depth factor of the hybrid law, zero
// without it.  The device's pow differs from the C library's in the last bit
// for some arguments.
__device__ __forceinline__ double hybrid_term(const Hybrid& h, double H) {
  return h.on != 0.0 ? h.on * pow(1.0 + pow(h.hbreak / H, h.ftheta), h.fgamma / h.ftheta) : 0.0;
}

struct WdPrm {
  double h0, habsmin, hoff, velmin, iflinbf, ifnlbf, tkmax;
  Hybrid hyb;
};

// Wetting candidates of one step (src/wetdry.F:368-475 and its two twins).
// Candidate k is the k-th candidate element in element order; every array is
// sized for the worst case of one candidate per element.
struct WdWork {
  unsigned long long* mask;  // [4 ceil(ne/256)] bit e%64 of word e/64: element e is a
                             // candidate (clear between steps)
  int* bcnt;                 // [ceil(ne/256)] candidates per 256-element tile (clear between steps)
  int* cid;                  // [ne] candidate k: its element
  double* tkc;               // [ne] TK_TMP(NM123) of candidate element e
  int2* lc;                  // [ne] candidate element: local vertex of NM123 | local vertex of
                             // the partner << 2, and its candidate index; -1 otherwise
  double* m0;                // [ne] candidate element: TK_TMP and the entry TK of nodes it opens
  int2* pred;                // [ne] candidate element: the previous one on NM123 / partner, or -1
  int2* wnode;               // [ne] candidate element: NM123 / partner if it is the node's last, or -1
  double* M;                 // [ne] candidate k: TK of both nodes after k (serial fallback)
  // block closure (wd_close): candidate k's value is
  // max(cv[k], X values of the bits of cE[k]), the X values being those of the
  // earlier candidates xtab[b*WD_XMAX + i] of its block b = k / WD_BLOCK
  double* cv;                // [ne] maximum over k's ancestors inside its block
  unsigned long long* cE;    // [ne*WD_XW] external names reached inside the block
  int* xtab;                 // [nblk*WD_XMAX] block b's external names (candidate indices)
  int* xcnt;                 // [nblk] number of external names of block b
  double* xval;              // [nblk*WD_XMAX] final value of each external name
};

struct HollandPrm {
  double v[13];
  double t;
};

struct FricPrm {
  const double *uu1, *vv1, *dp, *eta2, *fric;
  double ifnlfa, iflinbf, ifnlbf, tkmax;
  Hybrid hyb;
};

// Apply2DBottomFriction (src/nodalattr.F:2400-2411), and the TKM = (TK, TK, 0)
// of Apply2DInternalWaveDrag without wave drag; TKM is represented by TK alone.
__device__ __forceinline__ double friction(const FricPrm& f, int i, double u, double v, double dp,
                                           double eta2) {
  const double uv1 = __builtin_sqrt(u * u + v * v);
  const double h1 = dp + f.ifnlfa * eta2;
  const double hyb = hybrid_term(f.hyb, h1);
  const double a = f.fric[i] * (f.iflinbf + (uv1 / h1) * (f.ifnlbf + hyb));
  return fmin(a, f.tkmax);
}

// computeAlpha (src/wetdry.F:1561-1652): ALPHAL of a wet element from ETA2 and DP
// of its vertices.  `geometry` leaves FDXE and FDYE and returns AREAS; it is called
// where some vertex is shallow only.
template <class Geometry>
__device__ __forceinline__ double compute_alpha(double e1, double e2, double e3, double d1,
                                                double d2, double d3, double slim,
                                                const Geometry& geometry) {
  double al = 1.0;
  const double hn1 = e1 + d1, hn2 = e2 + d2, hn3 = e3 + d3;
  if ((hn1 <= 5.0e-1) || (hn2 <= 5.0e-1) || (hn3 <= 5.0e-1)) {
    double fx[3], fy[3];
    const double area = geometry(fx, fy);
    const double DPDXA = d1 * fx[0] + d2 * fx[1] + d3 * fx[2];
    const double DPDYA = d1 * fy[0] + d2 * fy[1] + d3 * fy[2];
    const double DETADXA = e1 * fx[0] + e2 * fx[1] + e3 * fx[2];
    const double DETADYA = e1 * fy[0] + e2 * fy[1] + e3 * fy[2];
    const double DPM = __builtin_sqrt(DPDXA * DPDXA + DPDYA * DPDYA) / area;
    if (DPM > 1e-5) {
      const double DDTMP = DETADXA * (-DPDXA) + DETADYA * (-DPDYA);
      if (fabs(DDTMP) > 1e-12)
        al = slim * (__builtin_sqrt(DPDXA * DPDXA + DPDYA * DPDYA) / ((1.0 / area) * (DDTMP)));
    } else {
      const double DETAM = __builtin_sqrt(DETADXA * DETADXA + DETADYA * DETADYA) / area;
      if (fabs(DETAM) > 1e-12) al = slim / DETAM;
    }
    if (al <= 0.0) al = 1.0;
    if (al >= 1.0) al = 1.0;
  }
  return al;
}

struct JcgArgs {
  int n, itmax, maxfn;
  double zeta, tz;
  double* coef;       // [mnei*n] unscaled in/out (diag in slot 0)
  double* cs;         // [mnei*n] scaled off-diagonals
  const int* col;
  const int* nneigh;
  double* rhs;        // scaled in place, restored on exit
  double* u;          // initial guess in (scaled in place), ETAS out
  double* d;          // pseudo-residual of the current iteration
  double* w;          // 1/sqrt(diag)
  double* part;       // chunk partials (d.d, d.Nd, u.u): [2][nch*4] by iteration parity;
                      // k_jcg_reg: [4][(nch+1)*4] slots (jcg_part_doubles)
  double* saved;      // [12] ITPACK SAVE state q1, gamold, rhoold, cmold, cme,
                      // stptst; [6..9] = cme, cmold of the running iteration, by parity
  int prescaled;      // rows already scaled (w, u, rhs) by k_rhs_node
  int defer_unscal;   // leave the off-diagonals unscaled (k_gwce scales and
                      // unscales them if they are needed again)
  unsigned* barrier;  // [JCG_BAR_WORDS] grid barrier counters, then per-tile halo flags
  int hrows;          // >= 0: the pseudo-residual of the tile's rows and of hrows
                      // rows each side (at least the matrix bandwidth) is kept
                      // in LDS for the products (dynamic shared memory of
                      // 8 (JCG_CPB RED_CHUNK + 2 hrows) bytes); -1: gathered
                      // from memory
  const int* hrange;  // staged: per 2048-row chunk, the first and one past the last
                      // row its rows reference (within hrows of the chunk)
  const unsigned* lcol;  // staged: [(mnei/2)][n] per row, off-diagonal slots 2p+1
                         // and 2p+2 as positions counted from row (chunk's first
                         // row - hrows), 16 bits each (low half first)
  int halo;           // row tiles each side whose pseudo-residual a tile's rows read;
                      // -1: wait for all tiles (a grid barrier) after each update
  long long barrier_ticks;  // longest grid-barrier wait, in wall-clock ticks
  unsigned* admit;          // an ordinary launch of k_jcg_reg: the admission word
                            // (JCG_ABORT); null: a cooperative launch
  long long admit_ticks;    // the longest wait for blocks that have not started
  int* given;               // k_jcg_mem behind it: set (host memory) when it does the work
  int* flags;
  double* eta2;       // optional: ETA2 = NODECODE*(ETAS+0)+ETA1
  const double* eta1;
  const int* nodecode;
  double* uo;         // k_jcg_mem: [n] the previous u
  double* dpv;        //             [n] the previous d
  double* ndv;        //             [n] N d
  int lds_doubles;    // k_jcg_reg: doubles of dynamic LDS of a block
  int ovf;            //            of which for entries past the register slots
                      //            (coefficient and 16-bit position of each)
  int hmem;           //            neighbouring rows of a block whose previous d
  double* hprev;      //            does not fit the LDS: [row blocks][hmem]
  const double* u2;   // k_jcg<true>: the second (learned) start, scaled like u
  double* d2;         //              and its initial pseudo-residual
};

__global__ void k_init_h(int np, const double* dp, const double* eta2, double ifnlfa, double* h1,
                         double* h2);
// TIP2 = sum over constituents of TPMUL*L_N(NA, i)*cos(ARGT + NA*SLAM(i)); ln is
// [3][np] (long-period, diurnal, semidiurnal species)
__global__ void k_tide_pot(int np, TipPrm p, const double* ln, const double* slam, double* tip2);
__global__ void k_friction(int np, FricPrm f, double* tk);
__global__ void k_holland(int np, const double* x, const double* y, HollandPrm p, double* wsx,
                          double* wsy, double* pr);
// LUMPED: the lumped GWCE (ILump = 1), whose LHS is the diagonal COEFD only
// (kept in COEF's diagonal column) and whose solve is explicit.  CT: the type of
// the element terms (float: the mixed path).
template <bool LUMPED, typename CT>
__global__ void k_gwce(DevMesh m, DevState s, DevPatch pp, RhsPrm q, FricPrm f, const int* flags,
                       const double* restore_w);
// bad[0]: some edge has more than two elements, bad[1]: the coordinates do not
// give the geometry (both set, never cleared)
__global__ void k_patch_check(DevMesh m, DevPatch pp, unsigned* pair, int* bad);
__global__ void k_patch_geo(DevMesh m, DevPatch pp, double* geo);
__global__ void k_ncele(DevMesh m, DevState s, DevPatch pp);
__global__ void k_lhs_ep(DevMesh m, DevState s, int* flags, double* ep_part);
__global__ void k_coef_restore(DevMesh m, DevState s, const double* w);
// Jacobi scaling of the GWCE rows ahead of k_jcg (its first scaling pass)
struct JcgPre {
  double* w;          // 1/sqrt(diag)
  unsigned* barrier;  // grid barrier words of the coming k_jcg launch, cleared here
  int barrier_words;
  unsigned long long* part;  // k_jcg_reg's partial slots, marked empty here
  int part_words;
  int* flags;
  unsigned admit0;    // the admission word's first value (0, or JCG_ABORT: give up)
  double* etas_prev;  // the previous step's ETAS (kept when keep_prev != 0)
  int warm;           // 1: start JCG from 2*ETAS - ETAS_prev instead of ETAS;
                      // 2: also form the learned start ETAS + ml_corr into ml_u
  int keep_prev;      // record this step's starting ETAS in etas_prev
  const double* ml_corr;  // warm == 2: the network's correction per node
  double* ml_u;           // warm == 2: the learned start, scaled
};
// One member of a batch: what the passes of a step take.  `s` is the state after
// the GWCE's time-level rotation (k_gwce runs before it: ETA1 and ETA2, H1 and H2
// change places there).  What changes with the step is passed beside it.
struct MemberArgs {
  DevMesh m;
  DevState s;
  DevPatch pp;
  RhsPrm rq;
  FricPrm f;
  WdPrm wq;
  WdWork wd;
  MomPrm mq;
  JcgPre pre;
  HollandPrm hol;
  const double* restore_w;
  const double* eta_bc;  // the run's table, or the one row of a member without boundary
  double* ep_part;
  double* scal;
  double ifnlfa, dt;
  int nch, nlist, nchain;
};
// The passes for all members in one launch each: member blockIdx.y, whose blocks
// past its own number leave at once.
template <typename CT>
__global__ void k_gwce_batch(const MemberArgs* a);
__global__ void k_lhs_ep_batch(const MemberArgs* a);
__global__ void k_rhs_node_batch(const MemberArgs* a, int step, int it, int met);
__global__ void k_wd_elem_batch(const MemberArgs* a);
__global__ void k_wd_d2_batch(const MemberArgs* a);
__global__ void k_wd_chain_batch(const MemberArgs* a);
template <typename CT>
__global__ void k_mom_batch(const MemberArgs* a, int it);
template <bool LUMPED>
__global__ void k_rhs_node(DevMesh m, DevState s, const double* eta_bc, int nch,
                           const double* ep_part, double* scal, JcgPre pre, HollandPrm hol,
                           int met);
// DUAL: start from the better (smaller initial pseudo-residual) of a.u and a.u2;
// STAGED: the products read the pseudo-residual from LDS (a.hrows >= 0).
// Instantiated for all four combinations.
template <bool DUAL, bool STAGED>
__global__ void k_jcg(JcgArgs a);
// nsys systems in one launch: blocks first[m] .. first[m+1]-1 solve args[m]
template <bool DUAL, bool STAGED>
__global__ void k_jcg_batch(const JcgArgs* args, const int* first, int nsys);
// the matrix in registers, one exchange per iteration (jcg_reg.hip): CPB
// 2048-row chunks per 512-thread block
template <bool DUAL, int CPB>
__global__ void k_jcg_reg(JcgArgs a);
template <bool DUAL, int CPB>
__global__ void k_jcg_reg_batch(const JcgArgs* args, const int* first, int nsys);
// more row tiles than blocks: the iterates in memory (a.uo, a.dpv, a.ndv)
__global__ void k_jcg_mem(JcgArgs a);
__global__ void k_wd_elem(DevMesh m, DevState s, DevPatch pp, WdPrm q, WdWork w, int* flags);
// the first ceil(ceil(NE/256) / WD_TILES) blocks list the candidates, then one per patch
__global__ void k_wd_d2(DevMesh m, DevState s, DevPatch pp, WdPrm q, WdWork w, int* flags,
                        double ifnlfa);
__global__ void k_wd_chain(DevMesh m, DevState s, WdWork w, int* flags);
__global__ void k_wd_alpha(DevMesh m, DevState s, int* flags, double slim);
__global__ void k_h2(int np, const double* dp, const double* eta2, double ifnlfa, double* h2);
template <bool ALPHA, typename CT>
__global__ void k_mom(DevMesh m, DevState s, DevPatch pp, MomPrm q);
// The drop-in's system: the caller's ELLPACK arrays (n rows, maxnz columns)
// compacted to the solver's layout, and the solved rows back.  `check` holds the
// smallest row*4 + kind of a row that is refused; ERR_INPUT is set with it.
enum { NA_NODIAG = 0, NA_BADCOL = 1, NA_ZERODIAG = 2, NA_NEGDIAG = 3 };
constexpr int NA_OK = 0x7fffffff;
__global__ void k_na_compact(int n, int maxnz, const double* in_coef, const int* in_jcoef,
                             double* coef, int* col, int* nneigh, int* check, int* flags);
__global__ void k_na_scatter(int n, int maxnz, double* in_coef, const int* in_jcoef,
                             const double* coef, const int* flags);
__global__ void k_na_clear(int* flags, int* check, unsigned* bar, int bar_words);
__global__ void k_fill_u32(unsigned* p, unsigned v, int n);
__global__ void k_fill_i32(int* p, int v, int n);
__global__ void k_run_clear(int* flags);  // the counters of a run
__global__ void k_total_area(DevMesh m, DevState s);

}  // namespace adcgpu
