// The GWCE and momentum passes over patches (patch.h): element terms and their
// node sums in one pass.
//
// What bounds them: memory traffic and the latency of a block's three dependent
// rounds of loads.  Formed element by element, every nodal field is gathered
// some six times through L1 (51 gathers per element for the GWCE) and the
// contributions make a trip through memory (three values per element written,
// then read per node).  A block instead reads the fields of its patch's window
// once into LDS, coalesced runs of a mesh numbered with any locality, forms the
// terms of all elements at its nodes from there (one element per thread, about a
// fifth of them formed by a second patch too), and sums them in LDS.  Geometry
// and NCEle are kept in patch order, so their reads are contiguous.  What a
// block's loads do not depend on is asked for first (the lists start at fixed
// offsets, a node's update is read with the window), and four blocks of 256
// threads share a CU at different stages: half as many of 512 threads took 6%
// longer.
//
// us at 999,151 nodes (wet/dry, storm), before and after: k_gwce 154, the passes
// it replaces (element terms 102, matrix 76, friction 8, a launch each for the
// matrix's other cases 11) 197; k_mom 104 to 110, before 106 + 54.  At 20,646 nodes
// 9.1 (23.5) and 7.3 (12.3), where a launch costs 5.  At 1M k_gwce moves 270 MB in
// and 81 out past the L2 (232 and 72 counted once), 2.3 TB/s, k_mom 294 and 62,
// 3.25 TB/s; a copy reaches 5, the window's runs being some 16 nodes long.
//
// Every sum keeps the reference's order: a node's contributions are listed in
// ascending element order.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "kernels.h"
#include "reduce.h"

namespace adcgpu {

#define W(f, v) sh[(f) * ws + (v)]

// The gradient sum f1*D1 + f2*D2 + f3*D3 of FP64 nodal values in FP32: with
// D1 + D2 + D3 = 0 (the shape-function derivatives of a triangle) it is
// (f2 - f1) D2 + (f3 - f1) D3, and the differences are taken in FP64 before
// rounding, so a field's mean (an elevation of metres, a pressure head of ten
// metres) costs no FP32 digits of its variation.
__device__ __forceinline__ float grad32(double f1, double f2, double f3, float d2, float d3) {
  return (float)(f2 - f1) * d2 + (float)(f3 - f1) * d3;
}

// A patch element's FDXE, FDYE and AREAS: formed from its vertices' coordinates
// in the window (the first two fields) where that gives the mesh's values bit
// for bit, as the host has checked, else read in patch order.  Six subtractions
// and two products replace 56 bytes per element, a quarter of either pass's
// traffic.
template <typename T>
struct ElemGeo {
  T x1, x2, x3, y1, y2, y3, a;
  __device__ __forceinline__ ElemGeo() {}
  template <typename S>
  __device__ __forceinline__ explicit ElemGeo(const ElemGeo<S>& g)
      : x1((T)g.x1), x2((T)g.x2), x3((T)g.x3), y1((T)g.y1), y2((T)g.y2), y3((T)g.y3), a((T)g.a) {}
  __device__ __forceinline__ void load(const double* g, int nq, int k) {
    x1 = g[k]; x2 = g[(size_t)nq + k]; x3 = g[2 * (size_t)nq + k];
    y1 = g[3 * (size_t)nq + k]; y2 = g[4 * (size_t)nq + k]; y3 = g[5 * (size_t)nq + k];
    a = g[6 * (size_t)nq + k];
  }
  __device__ __forceinline__ void form(const double* sh, int ws, int n1, int n2, int n3) {
    elem_geometry(W(0, n1), W(0, n2), W(0, n3), W(1, n1), W(1, n2), W(1, n3), x1, x2, x3, y1, y2,
                  y3, a);
  }
};

// fields of the GWCE window
enum { RF_X, RF_Y, RF_E0, RF_E1, RF_ES, RF_U, RF_V, RF_QX, RF_QY, RF_H, RF_EVM, RF_T0, RF_PR, RF_WX, RF_WY,
       RF_TK, RF_COR, RF_DP, RF_COUNT };
static_assert(RF_COUNT == PATCH_GWCE_FIELDS, "LDS of k_gwce");

// Element contributions Temp_LV_A1..3 (src/gwce.F:1000-1615).  Terms the
// reference multiplies by identically zero quantities in this configuration
// (sponge layer, dispersion, baroclinic, water level offset) are omitted; they
// only add signed zeros.
template <bool LUMPED>
__device__ __forceinline__ void rhs_terms(const double* sh, int ws, int n1, int n2, int n3,
                                          const DevMesh& m, const RhsPrm& q,
                                          const ElemGeo<double>& g, double al, double R[3]) {
  const double FDX1 = g.x1, FDX2 = g.x2, FDX3 = g.x3, FDY1 = g.y1, FDY2 = g.y2, FDY3 = g.y3;
  const double AreaIE2 = g.a;
  const double DT = m.dt, G = m.g, A00 = m.a00, B00 = m.b00, C00 = m.c00;
  const double E0N1 = W(RF_E0, n1), E0N2 = W(RF_E0, n2), E0N3 = W(RF_E0, n3);
  const double E1N1 = W(RF_E1, n1), E1N2 = W(RF_E1, n2), E1N3 = W(RF_E1, n3);
  const double E1N1SQ = E1N1 * E1N1, E1N2SQ = E1N2 * E1N2, E1N3SQ = E1N3 * E1N3;
  const double ESN1 = W(RF_ES, n1), ESN2 = W(RF_ES, n2), ESN3 = W(RF_ES, n3);
  const double U1N1 = W(RF_U, n1), U1N2 = W(RF_U, n2), U1N3 = W(RF_U, n3);
  const double V1N1 = W(RF_V, n1), V1N2 = W(RF_V, n2), V1N3 = W(RF_V, n3);
  const double QX1N1 = W(RF_QX, n1), QX1N2 = W(RF_QX, n2), QX1N3 = W(RF_QX, n3);
  const double QY1N1 = W(RF_QY, n1), QY1N2 = W(RF_QY, n2), QY1N3 = W(RF_QY, n3);
  const double H1N1 = W(RF_H, n1), H1N2 = W(RF_H, n2), H1N3 = W(RF_H, n3);
  const double EVMN1 = W(RF_EVM, n1), EVMN2 = W(RF_EVM, n2), EVMN3 = W(RF_EVM, n3);
  const double T0N1 = W(RF_T0, n1), T0N2 = W(RF_T0, n2), T0N3 = W(RF_T0, n3);
  // the pressure head less the tidal potential at time level s
  // (src/gwce.F:1181-1185) was formed per node
  const double PR1N1 = W(RF_PR, n1), PR1N2 = W(RF_PR, n2), PR1N3 = W(RF_PR, n3);
  const double WSXAvg = (1.0 * W(RF_WX, n1) + 1.0 * W(RF_WX, n2) + 1.0 * W(RF_WX, n3)) / 3.0;
  const double WSYAvg = (1.0 * W(RF_WY, n1) + 1.0 * W(RF_WY, n2) + 1.0 * W(RF_WY, n3)) / 3.0;
  // TKM(1)=TKM(2)=TK, TKM(3)=0
  const double tk1 = W(RF_TK, n1), tk2 = W(RF_TK, n2), tk3 = W(RF_TK, n3);
  const double BSXN1 = tk1 * QX1N1 + 0.0 * QY1N1, BSYN1 = 0.0 * QX1N1 + tk1 * QY1N1;
  const double BSXN2 = tk2 * QX1N2 + 0.0 * QY1N2, BSYN2 = 0.0 * QX1N2 + tk2 * QY1N2;
  const double BSXN3 = tk3 * QX1N3 + 0.0 * QY1N3, BSYN3 = 0.0 * QX1N3 + tk3 * QY1N3;
  const double AreaIE = AreaIE2 / 2.0;
  const double AreaIE4 = 2.0 * AreaIE2;
  const double E0XGrad2A = LUMPED ? 0.0 : E0N1 * FDX1 + E0N2 * FDX2 + E0N3 * FDX3;
  const double E0YGrad2A = LUMPED ? 0.0 : E0N1 * FDY1 + E0N2 * FDY2 + E0N3 * FDY3;
  const double E1XGrad2A = E1N1 * FDX1 + E1N2 * FDX2 + E1N3 * FDX3;
  const double E1YGrad2A = E1N1 * FDY1 + E1N2 * FDY2 + E1N3 * FDY3;
  const double Tau0XGrad2A = 1.0 * (T0N1 * FDX1 + T0N2 * FDX2 + T0N3 * FDX3);
  const double Tau0YGrad2A = 1.0 * (T0N1 * FDY1 + T0N2 * FDY2 + T0N3 * FDY3);
  const double EVMXGrad = (EVMN1 * FDX1 + EVMN2 * FDX2 + EVMN3 * FDX3) / AreaIE2;
  const double EVMYGrad = (EVMN1 * FDY1 + EVMN2 * FDY2 + EVMN3 * FDY3) / AreaIE2;
  const double EVMAvgODT = ((EVMN1 + EVMN2 + EVMN3) / 3.0) / DT;
  const double MX = (EVMXGrad * (QX1N1 * FDX1 + QX1N2 * FDX2 + QX1N3 * FDX3) +
                     EVMYGrad * (QY1N1 * FDX1 + QY1N2 * FDX2 + QY1N3 * FDX3) -
                     EVMAvgODT * (ESN1 * FDX1 + ESN2 * FDX2 + ESN3 * FDX3)) / AreaIE2;
  const double MY = (EVMXGrad * (QX1N1 * FDY1 + QX1N2 * FDY2 + QX1N3 * FDY3) +
                     EVMYGrad * (QY1N1 * FDY1 + QY1N2 * FDY2 + QY1N3 * FDY3) -
                     EVMAvgODT * (ESN1 * FDY1 + ESN2 * FDY2 + ESN3 * FDY3)) / AreaIE2;
  const double CorifAvg = (W(RF_COR, n1) + W(RF_COR, n2) + W(RF_COR, n3)) / 3.0;
  const double Tau0Avg = (T0N1 + T0N2 + T0N3) / 3.0;
  const double Tau0QXAvg = (T0N1 * QX1N1 + T0N2 * QX1N2 + T0N3 * QX1N3) / 3.0;
  const double Tau0QYAvg = (T0N1 * QY1N1 + T0N2 * QY1N2 + T0N3 * QY1N3) / 3.0;
  const double U1Avg = (U1N1 + U1N2 + U1N3) / 3.0;
  const double V1Avg = (V1N1 + V1N2 + V1N3) / 3.0;
  const double QX1Avg = (QX1N1 + QX1N2 + QX1N3) / 3.0;
  const double QY1Avg = (QY1N1 + QY1N2 + QY1N3) / 3.0;
  const double ESAvg = (ESN1 + ESN2 + ESN3) / 3.0;
  const double DPAvg = (W(RF_DP, n1) + W(RF_DP, n2) + W(RF_DP, n3)) / 3.0;
  const double GDP = al * G * DPAvg * 1.0 / AreaIE4;   // both time levels (IFNL_HDP = 0)
  const double HAvg = (H1N1 + H1N2 + H1N3) / 3.0;
  const double GHAvgOAreaIE2 = (al * G * HAvg) / AreaIE2;
  const double BSXAvg = (BSXN1 + BSXN2 + BSXN3) / 3.0;
  const double BSYAvg = (BSYN1 + BSYN2 + BSYN3) / 3.0;
  const double MsFacR = AreaIE * (1.0 / DT - Tau0Avg / 2.0) / DT / 12.0;
  const double GOAreaIE4 = al * G / AreaIE4;
  const double Tau0SpaVar = (QX1Avg * Tau0XGrad2A + QY1Avg * Tau0YGrad2A) / 6.0;
  const double A00pB00 = A00 + B00;
  double JXAvg = CorifAvg * QY1Avg -
                 q.ifnlfa * GOAreaIE4 * 1.0 * (E1N1SQ * FDX1 + E1N2SQ * FDX2 + E1N3SQ * FDX3) -
                 GHAvgOAreaIE2 * (PR1N1 * FDX1 + PR1N2 * FDX2 + PR1N3 * FDX3) +
                 WSXAvg - BSXAvg + MX + Tau0QXAvg;
  double JYAvg = -CorifAvg * QX1Avg -
                 q.ifnlfa * GOAreaIE4 * 1.0 * (E1N1SQ * FDY1 + E1N2SQ * FDY2 + E1N3SQ * FDY3) -
                 GHAvgOAreaIE2 * (PR1N1 * FDY1 + PR1N2 * FDY2 + PR1N3 * FDY3) +
                 WSYAvg - BSYAvg + MY + Tau0QYAvg;
  JXAvg = JXAvg -
          q.ifnlct * (QX1Avg * (U1N1 * FDX1 + U1N2 * FDX2 + U1N3 * FDX3) +
                      QY1Avg * (U1N1 * FDY1 + U1N2 * FDY2 + U1N3 * FDY3)) / AreaIE2 +
          q.ifnlcat * U1Avg * ESAvg / DT;
  JYAvg = JYAvg -
          q.ifnlct * (QX1Avg * (V1N1 * FDX1 + V1N2 * FDX2 + V1N3 * FDX3) +
                      QY1Avg * (V1N1 * FDY1 + V1N2 * FDY2 + V1N3 * FDY3)) / AreaIE2 +
          q.ifnlcat * V1Avg * ESAvg / DT;
  const double A1 = (q.ondiag * ESN1 * 1.0 + q.offdiag * (ESN2 * 1.0 + ESN3 * 1.0)) * MsFacR -
                    GDP * (C00 * (1.0 * FDX1 * E0XGrad2A + 1.0 * FDY1 * E0YGrad2A)) -
                    GDP * (A00pB00 * (1.0 * FDX1 * E1XGrad2A + 1.0 * FDY1 * E1YGrad2A)) +
                    (1.0 * JXAvg * FDX1 + 1.0 * JYAvg * FDY1) * 0.5 + Tau0SpaVar;
  const double A2 = (q.ondiag * ESN2 * 1.0 + q.offdiag * (ESN1 * 1.0 + ESN3 * 1.0)) * MsFacR -
                    GDP * (C00 * (1.0 * FDX2 * E0XGrad2A + 1.0 * FDY2 * E0YGrad2A)) -
                    GDP * (A00pB00 * (1.0 * FDX2 * E1XGrad2A + 1.0 * FDY2 * E1YGrad2A)) +
                    (1.0 * JXAvg * FDX2 + 1.0 * JYAvg * FDY2) * 0.5 + Tau0SpaVar;
  const double A3 = (q.ondiag * ESN3 * 1.0 + q.offdiag * (ESN1 * 1.0 + ESN2 * 1.0)) * MsFacR -
                    GDP * (C00 * (1.0 * FDX3 * E0XGrad2A + 1.0 * FDY3 * E0YGrad2A)) -
                    GDP * (A00pB00 * (1.0 * FDX3 * E1XGrad2A + 1.0 * FDY3 * E1YGrad2A)) +
                    (1.0 * JXAvg * FDX3 + 1.0 * JYAvg * FDY3) * 0.5 + Tau0SpaVar;
  R[0] = A1;
  R[1] = A2;
  R[2] = A3;
}

// The same in FP32 (the mixed-precision path): FP32 arithmetic and geometry,
// gradients formed from FP64 differences (grad32).
template <bool LUMPED>
__device__ __forceinline__ void rhs_terms(const double* sh, int ws, int n1, int n2, int n3,
                                          const DevMesh& m, const RhsPrm& q,
                                          const ElemGeo<float>& g, double al64, double R[3]) {
  const float FDX1 = g.x1, FDX2 = g.x2, FDX3 = g.x3, FDY1 = g.y1, FDY2 = g.y2, FDY3 = g.y3;
  const float AreaIE2 = g.a;
  const float DT = (float)m.dt, G = (float)m.g, A00 = (float)m.a00, B00 = (float)m.b00,
              C00 = (float)m.c00;
  const float AreaIE = AreaIE2 / 2.0f;
  const float AreaIE4 = 2.0f * AreaIE2;
  const double e0a = W(RF_E0, n1), e0b = W(RF_E0, n2), e0c = W(RF_E0, n3);
  const double e1a = W(RF_E1, n1), e1b = W(RF_E1, n2), e1c = W(RF_E1, n3);
  const float ESN1 = (float)W(RF_ES, n1), ESN2 = (float)W(RF_ES, n2), ESN3 = (float)W(RF_ES, n3);
  const double ua = W(RF_U, n1), ub = W(RF_U, n2), uc = W(RF_U, n3);
  const double va = W(RF_V, n1), vb = W(RF_V, n2), vc = W(RF_V, n3);
  const double qxa = W(RF_QX, n1), qxb = W(RF_QX, n2), qxc = W(RF_QX, n3);
  const double qya = W(RF_QY, n1), qyb = W(RF_QY, n2), qyc = W(RF_QY, n3);
  const float H1N1 = (float)W(RF_H, n1), H1N2 = (float)W(RF_H, n2), H1N3 = (float)W(RF_H, n3);
  const double eva = W(RF_EVM, n1), evb = W(RF_EVM, n2), evc = W(RF_EVM, n3);
  const double t0a = W(RF_T0, n1), t0b = W(RF_T0, n2), t0c = W(RF_T0, n3);
  const double pa = W(RF_PR, n1), pb = W(RF_PR, n2), pc = W(RF_PR, n3);
  const float PR1X = grad32(pa, pb, pc, FDX2, FDX3), PR1Y = grad32(pa, pb, pc, FDY2, FDY3);
  const float WSXAvg =
      ((float)W(RF_WX, n1) + (float)W(RF_WX, n2) + (float)W(RF_WX, n3)) / 3.0f;
  const float WSYAvg =
      ((float)W(RF_WY, n1) + (float)W(RF_WY, n2) + (float)W(RF_WY, n3)) / 3.0f;
  const float U1N1 = (float)ua, U1N2 = (float)ub, U1N3 = (float)uc;
  const float V1N1 = (float)va, V1N2 = (float)vb, V1N3 = (float)vc;
  const float QX1N1 = (float)qxa, QX1N2 = (float)qxb, QX1N3 = (float)qxc;
  const float QY1N1 = (float)qya, QY1N2 = (float)qyb, QY1N3 = (float)qyc;
  const float T0N1 = (float)t0a, T0N2 = (float)t0b, T0N3 = (float)t0c;
  const float tk1 = (float)W(RF_TK, n1), tk2 = (float)W(RF_TK, n2), tk3 = (float)W(RF_TK, n3);
  const float BSXAvg = (tk1 * QX1N1 + tk2 * QX1N2 + tk3 * QX1N3) / 3.0f;
  const float BSYAvg = (tk1 * QY1N1 + tk2 * QY1N2 + tk3 * QY1N3) / 3.0f;
  const float E0XGrad2A = LUMPED ? 0.0f : grad32(e0a, e0b, e0c, FDX2, FDX3);
  const float E0YGrad2A = LUMPED ? 0.0f : grad32(e0a, e0b, e0c, FDY2, FDY3);
  const float E1XGrad2A = grad32(e1a, e1b, e1c, FDX2, FDX3);
  const float E1YGrad2A = grad32(e1a, e1b, e1c, FDY2, FDY3);
  const float E1SQX = grad32(e1a * e1a, e1b * e1b, e1c * e1c, FDX2, FDX3);
  const float E1SQY = grad32(e1a * e1a, e1b * e1b, e1c * e1c, FDY2, FDY3);
  const float Tau0XGrad2A = grad32(t0a, t0b, t0c, FDX2, FDX3);
  const float Tau0YGrad2A = grad32(t0a, t0b, t0c, FDY2, FDY3);
  const float EVMXGrad = grad32(eva, evb, evc, FDX2, FDX3) / AreaIE2;
  const float EVMYGrad = grad32(eva, evb, evc, FDY2, FDY3) / AreaIE2;
  const float EVMAvgODT = (((float)eva + (float)evb + (float)evc) / 3.0f) / DT;
  const float ESX = ESN1 * FDX1 + ESN2 * FDX2 + ESN3 * FDX3;
  const float ESY = ESN1 * FDY1 + ESN2 * FDY2 + ESN3 * FDY3;
  const float MX = (EVMXGrad * grad32(qxa, qxb, qxc, FDX2, FDX3) +
                    EVMYGrad * grad32(qya, qyb, qyc, FDX2, FDX3) - EVMAvgODT * ESX) / AreaIE2;
  const float MY = (EVMXGrad * grad32(qxa, qxb, qxc, FDY2, FDY3) +
                    EVMYGrad * grad32(qya, qyb, qyc, FDY2, FDY3) - EVMAvgODT * ESY) / AreaIE2;
  const float CorifAvg = ((float)W(RF_COR, n1) + (float)W(RF_COR, n2) + (float)W(RF_COR, n3)) / 3.0f;
  const float Tau0Avg = (T0N1 + T0N2 + T0N3) / 3.0f;
  const float Tau0QXAvg = (T0N1 * QX1N1 + T0N2 * QX1N2 + T0N3 * QX1N3) / 3.0f;
  const float Tau0QYAvg = (T0N1 * QY1N1 + T0N2 * QY1N2 + T0N3 * QY1N3) / 3.0f;
  const float U1Avg = (U1N1 + U1N2 + U1N3) / 3.0f;
  const float V1Avg = (V1N1 + V1N2 + V1N3) / 3.0f;
  const float QX1Avg = (QX1N1 + QX1N2 + QX1N3) / 3.0f;
  const float QY1Avg = (QY1N1 + QY1N2 + QY1N3) / 3.0f;
  const float ESAvg = (ESN1 + ESN2 + ESN3) / 3.0f;
  const float DPAvg = (float)((W(RF_DP, n1) + W(RF_DP, n2) + W(RF_DP, n3)) / 3.0);
  const float al = (float)al64;
  const float GDP = al * G * DPAvg / AreaIE4;
  const float HAvg = (H1N1 + H1N2 + H1N3) / 3.0f;
  const float GHAvgOAreaIE2 = (al * G * HAvg) / AreaIE2;
  const float MsFacR = AreaIE * (1.0f / DT - Tau0Avg / 2.0f) / DT / 12.0f;
  const float GOAreaIE4 = al * G / AreaIE4;
  const float Tau0SpaVar = (QX1Avg * Tau0XGrad2A + QY1Avg * Tau0YGrad2A) / 6.0f;
  const float A00pB00 = A00 + B00;
  const float fnlfa = (float)q.ifnlfa, fnlct = (float)q.ifnlct, fnlcat = (float)q.ifnlcat;
  float JXAvg = CorifAvg * QY1Avg - fnlfa * GOAreaIE4 * E1SQX - GHAvgOAreaIE2 * PR1X + WSXAvg -
                BSXAvg + MX + Tau0QXAvg;
  float JYAvg = -CorifAvg * QX1Avg - fnlfa * GOAreaIE4 * E1SQY - GHAvgOAreaIE2 * PR1Y + WSYAvg -
                BSYAvg + MY + Tau0QYAvg;
  JXAvg = JXAvg -
          fnlct * (QX1Avg * grad32(ua, ub, uc, FDX2, FDX3) +
                   QY1Avg * grad32(ua, ub, uc, FDY2, FDY3)) / AreaIE2 +
          fnlcat * U1Avg * ESAvg / DT;
  JYAvg = JYAvg -
          fnlct * (QX1Avg * grad32(va, vb, vc, FDX2, FDX3) +
                   QY1Avg * grad32(va, vb, vc, FDY2, FDY3)) / AreaIE2 +
          fnlcat * V1Avg * ESAvg / DT;
  const float ond = (float)q.ondiag, offd = (float)q.offdiag;
  const float FX[3] = {FDX1, FDX2, FDX3}, FY[3] = {FDY1, FDY2, FDY3};
  const float ES[3] = {ESN1, ESN2, ESN3};
  float Rk[3];
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    const float others = ES[(k + 1) % 3] + ES[(k + 2) % 3];
    Rk[k] = (ond * ES[k] + offd * others) * MsFacR -
            GDP * (C00 * (FX[k] * E0XGrad2A + FY[k] * E0YGrad2A)) -
            GDP * (A00pB00 * (FX[k] * E1XGrad2A + FY[k] * E1YGrad2A)) +
            (JXAvg * FX[k] + JYAvg * FY[k]) * 0.5f + Tau0SpaVar;
  }
  for (int k = 0; k < 3; ++k) R[k] = (double)Rk[k];
}

// The GWCE matrix terms of an element before the NCEle factor (src/gwce.F:
// 456-592): the diagonal terms MsOn + GA*(FDXk*FDXk + FDYk*FDYk) of its three
// vertices, and the off-diagonal ones of its edges 0-1, 0-2, 1-2 (the same bits
// for both rows of an edge: products commute).  The lumped LHS has the diagonal
// MsFacLOnDiag*SPM with OnDiag = 4 only (src/gwce.F:596-635).
template <bool LUMPED>
__device__ __forceinline__ void lhs_terms(const double* sh, int ws, int n1, int n2, int n3,
                                          const DevMesh& m, const ElemGeo<double>& g, double al,
                                          double td[3], double to[3]) {
  const double dt = m.dt;
  const double area2 = g.a;
  const double area = area2 * 0.5;
  const double t0avg = (W(RF_T0, n1) + W(RF_T0, n2) + W(RF_T0, n3)) / 3.0;
  if (LUMPED) {
    const double mson = (4.0 * area * (1.0 / dt + t0avg / 2.0)) / dt / 12.0;
    td[0] = td[1] = td[2] = mson * 1.0;
    to[0] = to[1] = to[2] = 0.0;
    return;
  }
  const double fx[3] = {g.x1, g.x2, g.x3}, fy[3] = {g.y1, g.y2, g.y3};
  const double area4 = area2 * 2.0;
  const double dpavg = (W(RF_DP, n1) + W(RF_DP, n2) + W(RF_DP, n3)) / 3.0;
  const double ga = al * m.a00 * m.g * dpavg * 1.0 / area4;
  const double mson = (2.0 * area * (1.0 / dt + t0avg / 2.0)) / dt / 12.0;
  const double msoff = (1.0 * area * (1.0 / dt + t0avg / 2.0)) / dt / 12.0;
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    td[k] = mson * 1.0 + ga * (1.0 * fx[k] * fx[k] + 1.0 * fy[k] * fy[k]);
    const int a = k == 2 ? 1 : 0, b = k == 0 ? 1 : 2;
    to[k] = msoff * 1.0 + ga * (1.0 * fx[a] * fx[b] + 1.0 * fy[a] * fy[b]);
  }
}

// The GWCE's element terms and node sums: GWCE_LV (the sums only: boundary
// terms and scaling are k_rhs_node's), and COEF when NCChange is set
// (src/gwce.F:427-428).  With q.fric TK is formed here first
// (Apply2DBottomFriction, src/nodalattr.F:2400-2411).  Without a rebuild and with
// `restore_w`, the off-diagonals are scaled and unscaled as scal and unscal do
// (src/itpackv.F:2394-2400, 2460-2479): the previous solve left them as they were
// before its scaling.
template <bool LUMPED, typename CT>
__device__ __forceinline__ void gwce_block(const DevMesh& m, const DevState& s, const DevPatch& pp,
                                           const RhsPrm& q, const FricPrm& f, const int* flags,
                                           const double* __restrict__ restore_w, int bid) {
  extern __shared__ double sh[];
  __shared__ __attribute__((aligned(4))) unsigned short code[3 * PATCH_ELEMS];
  __shared__ int win_own[PATCH_NODES];
  const int patch = xcd_tile(bid, pp.n);
  const int t = threadIdx.x, ws = pp.wmax, np = m.np;
  // what does not hang on another load first: the block's lists
  const int i = t < PATCH_WIN ? pp.win[patch * PATCH_WIN + t] : -1;
  const int ke = patch * PATCH_ELEMS + t;
  const ushort4 lv = pp.lv[ke];
  const double nce = (double)s.ncele[ke];
  // the two halves of the block share a node's row; the lower one also sums
  const int o = t & (PATCH_THREADS / 2 - 1), half = t / (PATCH_THREADS / 2);
  const bool own = o < PATCH_NODES;
  const ushort2 c = own ? pp.cspan[patch * PATCH_NODES + o] : make_ushort2(1, 0);
  const bool rebuild = flags[F_NCCHANGE] != 0, alpha = flags[F_ALPHA] != 0;
  constexpr int PRE = 5;  // columns of a row read ahead per half: up to 10
  unsigned pr2[PRE];
  const unsigned* const prow =
      pp.pair ? pp.pair + (size_t)patch * (m.mnei - 1) * PATCH_NODES + o : nullptr;
#pragma unroll
  for (int k = 0; k < PRE; ++k) {
    const int j = 1 + half + 2 * k;
    pr2[k] = !LUMPED && rebuild && prow && own && j < m.mnei ? prow[(j - 1) * PATCH_NODES] : ~0u;
  }
  for (int k = t; k < 3 * PATCH_ELEMS / 2; k += PATCH_THREADS)
    reinterpret_cast<unsigned*>(code)[k] =
        reinterpret_cast<const unsigned*>(pp.code)[patch * (3 * PATCH_ELEMS / 2) + k];
  ElemGeo<double> g;
  if (pp.geo) g.load(pp.geo, pp.nq, ke);
  if (i >= 0) {
    const double e1 = s.eta2[i], u = s.uu1[i], v = s.vv1[i], dp = m.dp[i];
    W(RF_X, t) = m.x[i];
    W(RF_Y, t) = m.y[i];
    W(RF_E0, t) = s.eta1[i];
    W(RF_E1, t) = e1;
    W(RF_ES, t) = s.etas[i];
    W(RF_U, t) = u;
    W(RF_V, t) = v;
    W(RF_QX, t) = s.qx1[i];
    W(RF_QY, t) = s.qy1[i];
    W(RF_H, t) = s.h2[i];
    W(RF_EVM, t) = m.evm[i];
    W(RF_T0, t) = m.tau0[i];
    double pr = 0.0, wx = 0.0, wy = 0.0;
    if (q.nws) {
      pr = s.pr1[i];
      wx = s.wsx1[i];
      wy = s.wsy1[i];
    }
    if (s.tip1) pr = pr - s.tip1[i];
    W(RF_PR, t) = pr;
    W(RF_WX, t) = wx;
    W(RF_WY, t) = wy;
    W(RF_COR, t) = m.corif[i];
    W(RF_DP, t) = dp;
    double tk;
    if (q.fric) {
      tk = friction(f, i, u, v, dp, e1);
      if (t < PATCH_NODES && c.y >= c.x) s.tk[i] = tk;
    } else {
      tk = s.tk[i];
    }
    W(RF_TK, t) = tk;
  }
  if (t < PATCH_NODES) win_own[t] = c.y >= c.x ? i : -1;
  __syncthreads();
  // a dry element's contributions are its (finite) terms x 0: zeros, and a
  // node sum that starts at +0 never holds -0, so a zero of either sign
  // leaves it unchanged: the terms are skipped
  double R[3] = {0.0, 0.0, 0.0}, td[3] = {0.0, 0.0, 0.0}, to[3] = {0.0, 0.0, 0.0};
  if (lv.w != 2 && nce != 0.0) {
    const double al = alpha ? s.alphal[pp.el[ke]] : 1.0;
    if (!pp.geo) g.form(sh, ws, lv.x, lv.y, lv.z);
    const ElemGeo<CT> gc(g);
    rhs_terms<LUMPED>(sh, ws, lv.x, lv.y, lv.z, m, q, gc, al, R);
    if (rebuild) lhs_terms<LUMPED>(sh, ws, lv.x, lv.y, lv.z, m, g, al, td, to);
  }
  __syncthreads();  // the window's LDS is free
  double* const cr = sh;                    // [3][PATCH_ELEMS] contributions
  double* const cd = cr + 3 * PATCH_ELEMS;  // [3][PATCH_ELEMS] diagonal terms
  double* const co = cd + 3 * PATCH_ELEMS;  // [3][PATCH_ELEMS] edge terms, then a zero
#pragma unroll
  for (int k = 0; k < 3; ++k) cr[k * PATCH_ELEMS + t] = sizeof(CT) == 4 ? (double)((float)R[k] * (float)nce) : R[k] * nce;
  if (rebuild) {
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      // the mixed path takes FP32 terms and sums them in FP64
      cd[k * PATCH_ELEMS + t] = (double)(CT)td[k] * nce;
      co[k * PATCH_ELEMS + t] = (double)(CT)to[k] * nce;
    }
    if (t == 0) co[3 * PATCH_ELEMS] = 0.0;
  }
  __syncthreads();
  const int r = own ? win_own[o] : -1;
  if (r < 0) return;
  if (half == 0) {
    double acc = 0.0;
    if (sizeof(CT) == 4) {
      Kahan32 k;  // FP32 contributions: compensated sum
      for (int p = c.x; p < c.y; ++p) k.add((float)cr[code[p]]);
      acc = k.value();
    } else {
      for (int p = c.x; p < c.y; ++p) acc = acc + cr[code[p]];
    }
    s.gwce_lv[r] = acc;
    if (rebuild) {
      double diag = 0.0;
      for (int p = c.x; p < c.y; ++p) diag = diag + cd[code[p]];
      s.coef[r] = diag;
    }
  }
  if (LUMPED) {
    // COEFD only; the off-diagonal columns are zero
    const int nn = m.nneigh[r];
    if (rebuild)
      for (int j = 1 + half; j < nn; j += 2) s.coef[(size_t)j * np + r] = 0.0;
    return;
  }
  if (!rebuild) {
    if (restore_w) {
      const int nn = m.nneigh[r];
      const double wi = restore_w[r], ri = 1.0 / wi;
      for (int j = 1 + half; j < nn; j += 2) {
        const size_t z = (size_t)j * np + r;
        const double wj = restore_w[m.col[z]];
        s.coef[z] = (s.coef[z] * wi * wj) * ri * (1.0 / wj);
      }
    }
    return;
  }
  // COEF(i, j): the terms of the (at most two) elements that hold the edge, in
  // ascending element order
  if (prow) {
#pragma unroll
    for (int k = 0; k < PRE; ++k)
      if (pr2[k] != ~0u)
        s.coef[(size_t)(1 + half + 2 * k) * np + r] =
            (0.0 + co[pr2[k] & 0xffffu]) + co[pr2[k] >> 16];
    for (int j = 1 + half + 2 * PRE; j < m.mnei; j += 2) {
      const unsigned x = prow[(j - 1) * PATCH_NODES];
      if (x == ~0u) break;
      s.coef[(size_t)j * np + r] = (0.0 + co[x & 0xffffu]) + co[x >> 16];
    }
  } else if (half == 0) {
    // some edge has more than two elements: column by column in slot order
    const int nn = m.nneigh[r];
    for (int j = 1; j < nn; ++j) {
      double v = 0.0;
      for (int p = c.x; p < c.y; ++p) {
        const int jab = m.slot_cols[m.inc_ptr[r] + p - c.x];
        const int k = code[p] / PATCH_ELEMS, le = code[p] % PATCH_ELEMS;
        if ((jab & 0xffff) == j) v = v + co[(k == 2 ? 1 : 0) * PATCH_ELEMS + le];
        if ((jab >> 16) == j) v = v + co[(k == 0 ? 1 : 2) * PATCH_ELEMS + le];
      }
      s.coef[(size_t)j * np + r] = v;
    }
  }
}

template <bool LUMPED, typename CT>
__global__ __launch_bounds__(PATCH_THREADS, 3) void k_gwce(DevMesh m, DevState s, DevPatch pp, RhsPrm q,
                                                           FricPrm f, const int* flags,
                                                           const double* __restrict__ restore_w) {
  gwce_block<LUMPED, CT>(m, s, pp, q, f, flags, restore_w, blockIdx.x);
}
template <typename CT>
__global__ __launch_bounds__(PATCH_THREADS, 3) void k_gwce_batch(const MemberArgs* __restrict__ a) {
  const MemberArgs& x = a[blockIdx.y];
  if ((int)blockIdx.x >= x.pp.n) return;
  DevState s = x.s;  // before the time levels change places
  s.eta1 = x.s.eta2;
  s.eta2 = x.s.eta1;
  s.h1 = x.s.h2;
  s.h2 = x.s.h1;
  gwce_block<false, CT>(x.m, s, x.pp, x.rq, x.f, x.pre.flags, x.restore_w, blockIdx.x);
}
template __global__ void k_gwce_batch<double>(const MemberArgs*);
template __global__ void k_gwce_batch<float>(const MemberArgs*);
template __global__ void k_gwce<false, double>(DevMesh, DevState, DevPatch, RhsPrm, FricPrm, const int*, const double*);
template __global__ void k_gwce<true, double>(DevMesh, DevState, DevPatch, RhsPrm, FricPrm, const int*, const double*);
template __global__ void k_gwce<false, float>(DevMesh, DevState, DevPatch, RhsPrm, FricPrm, const int*, const double*);
template __global__ void k_gwce<true, float>(DevMesh, DevState, DevPatch, RhsPrm, FricPrm, const int*, const double*);

// Once per context.  `pair`: per own node and column, the codes of the edge terms
// it sums in ascending element order: a slot with vertex k adds edge (k, its
// lower other vertex) to column ja and the other edge to jb.
__global__ __launch_bounds__(256) void k_patch_check(DevMesh m, DevPatch pp,
                                                     unsigned* __restrict__ pair,
                                                     int* __restrict__ bad) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k < m.ne) {
    const size_t e = k;
    const int n1 = m.nm[3 * e], n2 = m.nm[3 * e + 1], n3 = m.nm[3 * e + 2];
    double g[7];
    elem_geometry(m.x[n1], m.x[n2], m.x[n3], m.y[n1], m.y[n2], m.y[n3], g[0], g[1], g[2], g[3], g[4],
                  g[5], g[6]);
    bool same = __double_as_longlong(g[6]) == __double_as_longlong(m.areas[e]);
    for (int j = 0; j < 3; ++j)
      same = same && __double_as_longlong(g[j]) == __double_as_longlong(m.fdx[3 * e + j]) &&
             __double_as_longlong(g[3 + j]) == __double_as_longlong(m.fdy[3 * e + j]);
    if (!same) atomicOr(&bad[1], 1);
  }
  if (!pair || k >= pp.n * PATCH_NODES) return;
  const int p = k / PATCH_NODES, o = k % PATCH_NODES;
  const ushort2 c = pp.cspan[k];
  unsigned* const row = pair + (size_t)p * (m.mnei - 1) * PATCH_NODES + o;
  const unsigned none = 3 * PATCH_ELEMS;
  const int i = c.y >= c.x ? pp.win[p * PATCH_WIN + o] : -1;
  const int nn = i >= 0 ? m.nneigh[i] : 1;
  for (int j = 1; j < m.mnei; ++j)
    row[(j - 1) * PATCH_NODES] = j < nn ? none | (none << 16) : ~0u;
  for (int q = c.x; q < c.y; ++q) {
    const int code = pp.code[p * 3 * PATCH_ELEMS + q];
    const int v = code / PATCH_ELEMS, le = code % PATCH_ELEMS;
    const int jab = m.slot_cols[m.inc_ptr[i] + q - c.x];
    for (int w = 0; w < 2; ++w) {
      unsigned* const x = row + ((w ? jab >> 16 : jab & 0xffff) - 1) * PATCH_NODES;
      const unsigned edge = (w ? (v == 0 ? 1 : 2) : (v == 2 ? 1 : 0)) * PATCH_ELEMS + le;
      if ((*x & 0xffffu) == none) *x = (*x & 0xffff0000u) | edge;
      else if ((*x >> 16) == none) *x = (*x & 0xffffu) | (edge << 16);
      else atomicOr(&bad[0], 1);
    }
  }
}

// Geometry in patch order (once per context).
__global__ __launch_bounds__(256) void k_patch_geo(DevMesh m, DevPatch pp, double* __restrict__ geo) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= pp.nq) return;
  const size_t e = pp.el[k], nq = pp.nq;
  for (int j = 0; j < 3; ++j) {
    geo[j * nq + k] = m.fdx[3 * e + j];
    geo[(3 + j) * nq + k] = m.fdy[3 * e + j];
  }
  geo[6 * nq + k] = m.areas[e];
}

// NCEle of every patch element from the current NODECODE and NOFF.
__global__ __launch_bounds__(256) void k_ncele(DevMesh m, DevState s, DevPatch pp) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= pp.nq) return;
  const size_t e = pp.el[k];
  s.ncele[k] = (unsigned char)(s.nodecode[m.nm[3 * e]] * s.nodecode[m.nm[3 * e + 1]] *
                               s.nodecode[m.nm[3 * e + 2]] * s.noff[e]);
}

// ---------------------------------------------------------------- wet/dry
// D1 (src/wetdry.F:234-285) of a node: its NODECODE, and ETA2 clipped.
__device__ __forceinline__ int wd_dry(int nc, double dp, const WdPrm& q, double& eta2) {
  if (nc == 1) {
    const double htot = dp + eta2;
    if (htot <= q.h0) {
      if (htot < q.habsmin) eta2 = q.habsmin - dp;
      nc = 0;
    }
  }
  return nc;
}

// D1, W1 candidates (src/wetdry.F:332-818) and DE1 (src/wetdry.F:1110-1233).
// NNODECODE of a node is its D1 code, or 1 if a candidate element, one whose
// steady-flow velocity exceeds VELMIN, wets it: all elements of the patch's own
// nodes are here.  ETA2 and NODECODE are left to the next pass, as other patches
// read them here.  The candidates' friction updates depend on element order:
// each leaves its TK_TMP value and local vertices at its element and sets its
// bit in the candidate mask.
__device__ __forceinline__ void wd_elem_block(const DevMesh& m, const DevState& s, const DevPatch& pp,
                                              const WdPrm& q, const WdWork& w, int* flags, int bid) {
  __shared__ double se[PATCH_WIN], sp[PATCH_WIN];
  __shared__ unsigned char sc[PATCH_WIN], sn[PATCH_WIN];
  const int patch = xcd_tile(bid, pp.n);
  const int t = threadIdx.x;
  const int i = t < PATCH_WIN ? pp.win[patch * PATCH_WIN + t] : -1;
  const int ke = patch * PATCH_ELEMS + t;
  const ushort4 lv = pp.lv[ke];
  const int e = pp.el[ke];
  const ushort2 c = t < PATCH_NODES ? pp.cspan[patch * PATCH_NODES + t] : make_ushort2(1, 0);
  const int old = s.noff[e];
  // this step's ALPHAL pass sets F_ALPHA again where needed; it rewrites ALPHAL
  // while the last pass (or the host) left some value other than 1
  if (bid == 0 && t == 0) {
    flags[F_ALPHA0] = flags[F_ALPHA];
    flags[F_ALPHA] = 0;
  }
  if (i >= 0) {
    double e2 = s.eta2[i];
    const double dp = m.dp[i];
    const int nc = wd_dry(s.nodecode[i], dp, q, e2);
    se[t] = e2;
    sp[t] = dp;
    sc[t] = (unsigned char)nc;
    sn[t] = (unsigned char)nc;
  }
  __syncthreads();
  if (lv.w != 2) {
    const int n[3] = {lv.x, lv.y, lv.z};
    int noff = 1;
    const double e1 = se[n[0]], e2 = se[n[1]], e3 = se[n[2]];
    const double h1 = sp[n[0]] + e1, h2 = sp[n[1]] + e2, h3 = sp[n[2]] + e3;
    const int c0 = sc[n[0]], c1 = sc[n[1]], c2 = sc[n[2]];
    if (c0 + c1 + c2 == 2) {
      int a = -1, b = -1, c = -1;
      if (c0 == 1 && c1 == 1) { a = 0; b = 1; c = 2; }
      else if (c1 == 1 && c2 == 1) { a = 1; b = 2; c = 0; }
      else if (c2 == 1 && c0 == 1) { a = 2; b = 0; c = 1; }
      const double ht[3] = {h1, h2, h3};
      if (a >= 0 && ht[a] >= q.hoff && ht[b] >= q.hoff) {
        const double et[3] = {e1, e2, e3};
        int l123 = a;
        if (et[b] > et[a]) l123 = b;
        const int nm123 = m.nm[3 * (size_t)e + l123], nc = m.nm[3 * (size_t)e + c];
        const double dy = m.y[nc] - m.y[nm123], dx = m.x[nc] - m.x[nm123];
        const double deldist = __builtin_sqrt(dy * dy + dx * dx);
        double deleta = et[l123] - et[c];
        if (deleta < 0.0) deleta = 0.0;
        const double H1 = et[l123] + sp[n[l123]];
        const double fr = s.fric[nm123];
        const double hyb = hybrid_term(q.hyb, H1);
        const double tkwet = fmax(fr * (q.iflinbf + (q.velmin / H1) * (q.ifnlbf + hyb)), 0.0001);
        const double vel = m.g * (deleta / deldist) / tkwet;
        if (vel > q.velmin) {
          sn[n[c]] = 1;
          if (lv.w == 1) {
            w.tkc[e] = fmin(fr * (q.iflinbf + (1.0 * vel / H1) * (q.ifnlbf + hyb)), q.tkmax);
            w.lc[e].x = l123 | ((l123 == b ? a : b) << 2);
            atomicOr(&w.mask[e >> 6], 1ull << (e & 63));
            atomicAdd(&w.bcnt[e >> 8], 1);
          }
        }
      }
    }
    const double HOFF = q.hoff;
    if ((e1 >= e2) && (e2 > e3)) if ((h1 < HOFF) || (h2 < HOFF)) noff = 0;
    if ((e2 >= e3) && (e3 > e1)) if ((h2 < HOFF) || (h3 < HOFF)) noff = 0;
    if ((e3 >= e1) && (e1 > e2)) if ((h3 < HOFF) || (h1 < HOFF)) noff = 0;
    if ((e1 >= e3) && (e3 > e2)) if ((h1 < HOFF) || (h3 < HOFF)) noff = 0;
    if ((e2 >= e1) && (e1 > e3)) if ((h2 < HOFF) || (h1 < HOFF)) noff = 0;
    if ((e3 >= e2) && (e2 > e1)) if ((h3 < HOFF) || (h2 < HOFF)) noff = 0;
    // NOFF changes count toward NCCHANGE (src/wetdry.F:1428-1430)
    if (lv.w == 1 && noff != old) {
      s.noff[e] = noff;
      atomicOr(&flags[F_NCCHANGE], 1);
    }
  }
  __syncthreads();
  if (c.y >= c.x) s.nnodecode[i] = sn[t];
}

__global__ __launch_bounds__(PATCH_THREADS) void k_wd_elem(DevMesh m, DevState s, DevPatch pp, WdPrm q,
                                                           WdWork w, int* flags) {
  wd_elem_block(m, s, pp, q, w, flags, blockIdx.x);
}
__global__ __launch_bounds__(PATCH_THREADS) void k_wd_elem_batch(const MemberArgs* __restrict__ a) {
  const MemberArgs& x = a[blockIdx.y];
  if ((int)blockIdx.x >= x.pp.n) return;
  wd_elem_block(x.m, x.s, x.pp, x.wq, x.wd, x.pre.flags, blockIdx.x);
}

// Does candidate code 3*e2+k2 (element e2, local vertex k2; lc = w.lc[e2].x)
// update the TK of that vertex, i.e. is e2 a candidate and the vertex one of its
// two wet nodes?
__device__ __forceinline__ bool wd_touches(int lc, int k2) {
  return lc >= 0 && (k2 == (lc & 3) || k2 == ((lc >> 2) & 3));
}

// Ordered W1 friction updates (src/wetdry.F:447-472), links of candidate element
// e.  The reference visits the candidates in ascending element order; candidate
// k sets TK(NM123) = MAX(TK_TMP, TK(NM123)), gives the partner the larger of the
// two and takes it back if the partner was larger, so afterwards both of its
// nodes hold M_k = max(TK_TMP_k, their values before k).  A node's value before k
// is M_j of the nearest earlier candidate j on that node, or its value on entry.
// The node incidence lists are sorted by element, so j and "k is the node's last
// candidate" are found in the node's list.  Entry values fold into m0.  Done
// here, by the elements' patches: by the few blocks of the ordered updates, the
// scattered reads alone took 30 us at 4,000 candidates.
__device__ __forceinline__ void wd_pred(const DevMesh& m, const DevState& s, const WdWork& w, int e,
                                        int lc) {
  double v = w.tkc[e];
#pragma unroll 1
  for (int j = 0; j < 2; ++j) {
    const int l = (lc >> (2 * j)) & 3;
    const int x = m.nm[3 * (size_t)e + l];
    const int me = m.slot[3 * (size_t)e + l];
    const int p0 = m.inc_ptr[x], p1 = m.inc_ptr[x + 1];
    const double tk = s.tk[x];
    int pe = -1;
    bool last = true;
    if (p1 - p0 <= WD_INC_MAX) {
      // the node's whole list at once: its codes, then their marks
      int code[WD_INC_MAX], c[WD_INC_MAX];
#pragma unroll
      for (int q = 0; q < WD_INC_MAX; ++q) code[q] = p0 + q < p1 ? m.inc[p0 + q] : -1;
#pragma unroll
      for (int q = 0; q < WD_INC_MAX; ++q) c[q] = code[q] >= 0 ? w.lc[code[q] / 3].x : -1;
#pragma unroll
      for (int q = 0; q < WD_INC_MAX; ++q)
        if (wd_touches(c[q], code[q] % 3)) {
          if (p0 + q < me) pe = code[q] / 3;  // the nearest earlier one is the last seen
          if (p0 + q > me) last = false;
        }
    } else {
      for (int q = me - 1; q >= p0; --q)
        if (wd_touches(w.lc[m.inc[q] / 3].x, m.inc[q] % 3)) {
          pe = m.inc[q] / 3;
          break;
        }
      for (int q = me + 1; q < p1; ++q)
        if (wd_touches(w.lc[m.inc[q] / 3].x, m.inc[q] % 3)) {
          last = false;
          break;
        }
    }
    if (pe < 0) v = fmax(v, tk);
    (&w.pred[e].x)[j] = pe;
    (&w.wnode[e].x)[j] = last ? x : -1;
  }
  w.m0[e] = v;
}

// The candidates of tiles [WD_TILES r, WD_TILES (r+1)) in ascending element order
// (w.cid, and their indices in w.lc); the last block also leaves their number.
// Each block adds up the earlier tiles' counts itself.  A thread follows every
// 256th tile, so that a front's candidates, which lie in consecutive tiles, are
// spread over the block.
__device__ __forceinline__ void wd_list(const DevMesh& m, const WdWork& w, int r, int nr, int* flags) {
  __shared__ unsigned short cnt[WD_TILES];
  __shared__ int ofs[WD_TILES];
  __shared__ int wtot[PATCH_THREADS / 64], wbef[PATCH_THREADS / 64];
  constexpr int PER = WD_TILES / PATCH_THREADS;
  const int t = threadIdx.x;
  const int nb = (m.ne + 255) / 256, b0 = WD_TILES * r;
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    const int b = b0 + t + PATCH_THREADS * j;
    cnt[t + PATCH_THREADS * j] = (unsigned short)(b < nb ? w.bcnt[b] : 0);
  }
  int bef = 0;
#pragma unroll 8
  for (int b = t; b < b0; b += PATCH_THREADS) bef += w.bcnt[b];
  __syncthreads();
  int sum = 0;
#pragma unroll
  for (int j = 0; j < PER; ++j) sum += cnt[PER * t + j];
  int incl = sum;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const int v = __shfl_up(incl, off, 64), u = __shfl_xor(bef, off, 64);
    if ((t & 63) >= off) incl += v;
    bef += u;
  }
  if ((t & 63) == 63) {
    wtot[t >> 6] = incl;
    wbef[t >> 6] = bef;
  }
  __syncthreads();
  int k = incl - sum, all = 0;
  for (int q = 0; q < PATCH_THREADS / 64; ++q) {
    if (q < (t >> 6)) k += wtot[q];
    k += wbef[q];
    all += wtot[q] + wbef[q];
  }
  if (t == 0) {
    if (r == 0) flags[F_WDSERIAL] = 0;
    if (r == nr - 1) flags[F_NCAND] = all;
  }
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    ofs[PER * t + j] = k;
    k += cnt[PER * t + j];
  }
  __syncthreads();
  ulonglong2 mk[PER][2];
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    const int x = t + PATCH_THREADS * j;
    if (cnt[x] == 0) continue;
    const ulonglong2* p = reinterpret_cast<const ulonglong2*>(w.mask) + 2 * (size_t)(b0 + x);
    mk[j][0] = p[0];
    mk[j][1] = p[1];
  }
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    const int x = t + PATCH_THREADS * j;
    if (cnt[x] == 0) continue;
    int at = ofs[x];
#pragma unroll
    for (int q = 0; q < 4; ++q)
      for (unsigned long long y = q & 1 ? mk[j][q / 2].y : mk[j][q / 2].x; y; y &= y - 1) {
        const int e = 256 * (b0 + x) + 64 * q + __ffsll((long long)y) - 1;
        w.cid[at] = e;
        w.lc[e].y = at++;
      }
  }
}

// D2: MJU, TotalArea, landlocked nodes, NODECODE update, NCCHANGE, and
// H2 = DP + IFNLFA*ETA2 (src/wetdry.F:1361-1430, src/timestep.F:1097-1099), and
// D1's ETA2; and the candidates' links and list.  MJU counts the wet elements of a node: AREAS > 0, so NCEle = 1
// exactly when an element's term is non-zero.
__device__ __forceinline__ void wd_d2_block(const DevMesh& m, const DevState& s, const DevPatch& pp,
                                            const WdPrm& q, const WdWork& w, int* flags, double ifnlfa,
                                            int bid, int nlist) {
  __shared__ double sa[PATCH_ELEMS];
  __shared__ unsigned char sn[PATCH_WIN];
  __shared__ __attribute__((aligned(4))) unsigned short code[3 * PATCH_ELEMS];
  if (bid < nlist) {
    wd_list(m, w, bid, nlist, flags);
    return;
  }
  const int patch = xcd_tile(bid - nlist, pp.n);
  const int t = threadIdx.x;
  const int i = t < PATCH_WIN ? pp.win[patch * PATCH_WIN + t] : -1;
  const int ke = patch * PATCH_ELEMS + t;
  const ushort4 lv = pp.lv[ke];
  const int e = pp.el[ke];
  const ushort2 c = t < PATCH_NODES ? pp.cspan[patch * PATCH_NODES + t] : make_ushort2(1, 0);
  const bool own = c.y >= c.x;
  for (int k = t; k < 3 * PATCH_ELEMS / 2; k += PATCH_THREADS)
    reinterpret_cast<unsigned*>(code)[k] =
        reinterpret_cast<const unsigned*>(pp.code)[patch * (3 * PATCH_ELEMS / 2) + k];
  const int noff = s.noff[e];
  const double area = m.areas[e];
  const int lc = lv.w == 1 ? w.lc[e].x : -1;
  int nn = 0, old = 0;
  double e2 = 0.0, dp = 0.0;
  if (i >= 0) {
    nn = s.nnodecode[i];
    if (own) {
      old = s.nodecode[i];
      e2 = s.eta2[i];
      dp = m.dp[i];
    }
    sn[t] = (unsigned char)nn;
  }
  __syncthreads();
  if (lv.w != 2) {
    const int ncele = sn[lv.x] * sn[lv.y] * sn[lv.z] * noff;
    sa[t] = (double)ncele * area / 2.0;
  }
  __syncthreads();
  if (lc >= 0) wd_pred(m, s, w, e, lc);
  if (!own) return;
  int mju = 0;
  double ta = 0.0;
  for (int p = c.x; p < c.y; ++p) {
    const double a = sa[code[p] % PATCH_ELEMS];
    mju += a != 0.0 ? 1 : 0;
    ta = ta + a;
  }
  const double was = e2;
  const int nc = wd_dry(old, dp, q, e2);  // D1
  if (nn == 1 && mju == 0) nn = 0;
  if (mju == 0) mju = 1;
  s.mju[i] = mju;
  s.totalarea[i] = ta;
  if (nn != old) s.nodecode[i] = nn;
  if (nn != nc || nc != old) atomicOr(&flags[F_NCCHANGE], 1);
  if (e2 != was) s.eta2[i] = e2;
  s.h2[i] = dp + ifnlfa * e2;
}

__global__ __launch_bounds__(PATCH_THREADS) void k_wd_d2(DevMesh m, DevState s, DevPatch pp, WdPrm q,
                                                         WdWork w, int* flags, double ifnlfa) {
  wd_d2_block(m, s, pp, q, w, flags, ifnlfa, blockIdx.x, (int)gridDim.x - pp.n);
}
__global__ __launch_bounds__(PATCH_THREADS) void k_wd_d2_batch(const MemberArgs* __restrict__ a) {
  const MemberArgs& x = a[blockIdx.y];
  if ((int)blockIdx.x >= x.pp.n + x.nlist) return;
  wd_d2_block(x.m, x.s, x.pp, x.wq, x.wd, x.pre.flags, x.ifnlfa, blockIdx.x, x.nlist);
}

// --------------------------------------------------------------- momentum
enum { MF_X, MF_Y, MF_U, MF_V, MF_H1, MF_EVM, MF_E1, MF_E2, MF_DP, MF_P1, MF_P2, MF_T1, MF_T2, MF_COUNT };
static_assert(MF_COUNT == PATCH_MOM_FIELDS, "LDS of k_mom");

// computeAlpha of a wet element of the patch.
__device__ __forceinline__ double alpha_terms(const double* sh, int ws, int n1, int n2, int n3,
                                              const ElemGeo<double>& g, double slim) {
  return compute_alpha(W(MF_E2, n1), W(MF_E2, n2), W(MF_E2, n3), W(MF_DP, n1), W(MF_DP, n2),
                       W(MF_DP, n3), slim, [&](double fx[3], double fy[3]) {
                         fx[0] = g.x1; fx[1] = g.x2; fx[2] = g.x3;
                         fy[0] = g.y1; fy[1] = g.y2; fy[2] = g.y3;
                         return g.a;
                       });
}

// Element loop of Mom_Eqs_New_NC (src/momentum.F:298-699): advection,
// barotropic pressure gradient, IBPV lateral stress; contributions x NCEle.
__device__ __forceinline__ void mom_terms(const double* sh, int ws, int n1, int n2, int n3,
                                          const DevMesh& m, const DevState& s, const MomPrm& q,
                                          const ElemGeo<double>& g, int ncele, double al,
                                          double tx[3], double ty[3]) {
  const double FDX1 = g.x1, FDX2 = g.x2, FDX3 = g.x3, FDY1 = g.y1, FDY2 = g.y2, FDY3 = g.y3;
  const double AreaIE2 = g.a;
  const double THIRD = 1.0 / 3.0, DT = m.dt, GO2 = m.g / 2.0;
  const double U1N1 = W(MF_U, n1), U1N2 = W(MF_U, n2), U1N3 = W(MF_U, n3);
  const double V1N1 = W(MF_V, n1), V1N2 = W(MF_V, n2), V1N3 = W(MF_V, n3);
  const double H1N1 = W(MF_H1, n1), H1N2 = W(MF_H1, n2), H1N3 = W(MF_H1, n3);
  const double AreaIE = 0.5 * AreaIE2;
  const double U1Avg = THIRD * (U1N1 + U1N2 + U1N3);
  const double V1Avg = THIRD * (V1N1 + V1N2 + V1N3);
  const double DU1DXA = (U1N1 * FDX1 + U1N2 * FDX2 + U1N3 * FDX3) * 0.5;
  const double DU1DYA = (U1N1 * FDY1 + U1N2 * FDY2 + U1N3 * FDY3) * 0.5;
  const double DV1DXA = (V1N1 * FDX1 + V1N2 * FDX2 + V1N3 * FDX3) * 0.5;
  const double DV1DYA = (V1N1 * FDY1 + V1N2 * FDY2 + V1N3 * FDY3) * 0.5;
  const double EVMEle = THIRD * (W(MF_EVM, n1) + W(MF_EVM, n2) + W(MF_EVM, n3));
  double B1N1 = al * W(MF_E1, n1), B2N1 = al * W(MF_E2, n1);
  double B1N2 = al * W(MF_E1, n2), B2N2 = al * W(MF_E2, n2);
  double B1N3 = al * W(MF_E1, n3), B2N3 = al * W(MF_E2, n3);
  if (q.nws) {
    B1N1 = B1N1 + W(MF_P1, n1); B2N1 = B2N1 + W(MF_P2, n1);
    B1N2 = B1N2 + W(MF_P1, n2); B2N2 = B2N2 + W(MF_P2, n2);
    B1N3 = B1N3 + W(MF_P1, n3); B2N3 = B2N3 + W(MF_P2, n3);
  }
  if (s.tip1) {  // src/momentum.F:443-450
    B1N1 = B1N1 - W(MF_T1, n1); B2N1 = B2N1 - W(MF_T2, n1);
    B1N2 = B1N2 - W(MF_T1, n2); B2N2 = B2N2 - W(MF_T2, n2);
    B1N3 = B1N3 - W(MF_T1, n3); B2N3 = B2N3 - W(MF_T2, n3);
  }
  const double DBTPDX1A = B1N1 * FDX1 + B1N2 * FDX2 + B1N3 * FDX3;
  const double DBTPDX2A = B2N1 * FDX1 + B2N2 * FDX2 + B2N3 * FDX3;
  const double DBTPDY1A = B1N1 * FDY1 + B1N2 * FDY2 + B1N3 * FDY3;
  const double DBTPDY2A = B2N1 * FDY1 + B2N2 * FDY2 + B2N3 * FDY3;
  const double DBTPDXA = 0.5 * (1.0 * DBTPDX1A + 1.0 * DBTPDX2A);
  const double DBTPDYA = 0.5 * (1.0 * DBTPDY1A + 1.0 * DBTPDY2A);
  const double UDU = U1Avg * DU1DXA, VDU = V1Avg * DU1DYA;
  const double UDV = U1Avg * DV1DXA, VDV = V1Avg * DV1DYA;
  const double DU1DX = DU1DXA / AreaIE, DU1DY = DU1DYA / AreaIE;
  const double DV1DX = DV1DXA / AreaIE, DV1DY = DV1DYA / AreaIE;
  const double NCDT = (double)ncele * DT;
  const double advx = -q.ifnlct * (UDU + VDU) - GO2 * DBTPDXA - 0.0;
  const double advy = -q.ifnlct * (UDV + VDV) - GO2 * DBTPDYA - 0.0;
  const double Hs[3] = {H1N1, H1N2, H1N3};
  const double FX[3] = {FDX1, FDX2, FDX3}, FY[3] = {FDY1, FDY2, FDY3};
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    const double eh = EVMEle * Hs[k];
    const double lxx = eh * DU1DX, lxy = eh * DU1DY, lyx = eh * DV1DX, lyy = eh * DV1DY;
    // TANPHI = 0: the AreaIE*TANPHI*(...) terms are signed zeros
    tx[k] = NCDT * (advx - (1.5 * (lxx * FX[k] + lxy * FY[k]) - AreaIE * 0.0 * (lxy + lyx)) / Hs[k]);
    ty[k] = NCDT * (advy - (1.5 * (lyx * FX[k] + lyy * FY[k]) + AreaIE * 0.0 * (lxx - lyy)) / Hs[k]);
  }
}

// The same in FP32 (the mixed-precision path), gradients from FP64
// differences (grad32), FP32 contributions.
__device__ __forceinline__ void mom_terms(const double* sh, int ws, int n1, int n2, int n3,
                                          const DevMesh& m, const DevState& s, const MomPrm& q,
                                          const ElemGeo<float>& g, int ncele, double al64,
                                          float tx[3], float ty[3]) {
  const float FDX1 = g.x1, FDX2 = g.x2, FDX3 = g.x3, FDY1 = g.y1, FDY2 = g.y2, FDY3 = g.y3;
  const float AreaIE2 = g.a;
  const float THIRD = 1.0f / 3.0f, DT = (float)m.dt, GO2 = (float)(m.g / 2.0);
  const double ua = W(MF_U, n1), ub = W(MF_U, n2), uc = W(MF_U, n3);
  const double va = W(MF_V, n1), vb = W(MF_V, n2), vc = W(MF_V, n3);
  const float AreaIE = 0.5f * AreaIE2;
  const float U1Avg = THIRD * ((float)ua + (float)ub + (float)uc);
  const float V1Avg = THIRD * ((float)va + (float)vb + (float)vc);
  const float DU1DXA = grad32(ua, ub, uc, FDX2, FDX3) * 0.5f;
  const float DU1DYA = grad32(ua, ub, uc, FDY2, FDY3) * 0.5f;
  const float DV1DXA = grad32(va, vb, vc, FDX2, FDX3) * 0.5f;
  const float DV1DYA = grad32(va, vb, vc, FDY2, FDY3) * 0.5f;
  const float EVMEle = THIRD * ((float)W(MF_EVM, n1) + (float)W(MF_EVM, n2) + (float)W(MF_EVM, n3));
  double b1a = al64 * W(MF_E1, n1), b2a = al64 * W(MF_E2, n1);
  double b1b = al64 * W(MF_E1, n2), b2b = al64 * W(MF_E2, n2);
  double b1c = al64 * W(MF_E1, n3), b2c = al64 * W(MF_E2, n3);
  if (q.nws) {
    b1a = b1a + W(MF_P1, n1); b2a = b2a + W(MF_P2, n1);
    b1b = b1b + W(MF_P1, n2); b2b = b2b + W(MF_P2, n2);
    b1c = b1c + W(MF_P1, n3); b2c = b2c + W(MF_P2, n3);
  }
  if (s.tip1) {
    b1a = b1a - W(MF_T1, n1); b2a = b2a - W(MF_T2, n1);
    b1b = b1b - W(MF_T1, n2); b2b = b2b - W(MF_T2, n2);
    b1c = b1c - W(MF_T1, n3); b2c = b2c - W(MF_T2, n3);
  }
  const float DBTPDXA = 0.5f * (grad32(b1a, b1b, b1c, FDX2, FDX3) +
                                grad32(b2a, b2b, b2c, FDX2, FDX3));
  const float DBTPDYA = 0.5f * (grad32(b1a, b1b, b1c, FDY2, FDY3) +
                                grad32(b2a, b2b, b2c, FDY2, FDY3));
  const float fnlct = (float)q.ifnlct;
  const float advx = -fnlct * (U1Avg * DU1DXA + V1Avg * DU1DYA) - GO2 * DBTPDXA;
  const float advy = -fnlct * (U1Avg * DV1DXA + V1Avg * DV1DYA) - GO2 * DBTPDYA;
  const float DU1DX = DU1DXA / AreaIE, DU1DY = DU1DYA / AreaIE;
  const float DV1DX = DV1DXA / AreaIE, DV1DY = DV1DYA / AreaIE;
  const float NCDT = (float)ncele * DT;
  const float Hs[3] = {(float)W(MF_H1, n1), (float)W(MF_H1, n2), (float)W(MF_H1, n3)};
  const float FX[3] = {FDX1, FDX2, FDX3}, FY[3] = {FDY1, FDY2, FDY3};
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    const float eh = EVMEle * Hs[k];
    const float lxx = eh * DU1DX, lxy = eh * DU1DY, lyx = eh * DV1DX, lyy = eh * DV1DY;
    tx[k] = NCDT * (advx - (1.5f * (lxx * FX[k] + lxy * FY[k])) / Hs[k]);
    ty[k] = NCDT * (advy - (1.5f * (lyx * FX[k] + lyy * FY[k])) / Hs[k]);
  }
}

// A node's fields in the momentum pass.
struct MomNode {
  double u1, v1, h1, e2, ta, tk, cor, h2, wx1, wy1, wx2, wy2, emax, umax;
  int nci, bc0, bc1;
  __device__ __forceinline__ void load(const DevMesh& m, const DevState& s, const MomPrm& q, int i) {
    ta = s.totalarea[i];
    tk = s.tk[i];
    cor = m.corif[i];
    h2 = s.h2[i];
    wx1 = wy1 = wx2 = wy2 = 0.0;
    if (q.nws) {
      wx1 = s.wsx1[i];
      wy1 = s.wsy1[i];
      wx2 = s.wsx2[i];
      wy2 = s.wsy2[i];
    }
    emax = s.etamax[i];
    umax = s.umax[i];
    bc0 = m.vbc_ptr[i];
    bc1 = m.vbc_ptr[i + 1];
  }
};

// Nodal part of Mom_Eqs_New_NC (src/momentum.F:713-1182) from the summed
// contributions: /TotalArea, wind, friction/Coriolis 2x2, land-boundary
// constraints, solve, fluxes; then the peak-surge maximum
// (src/write_output.F:6357-6366).
__device__ __forceinline__ void mom_node(const DevMesh& m, const DevState& s, const MomPrm& q,
                                         const MomNode& n, int i, double mx, double my) {
  const double DTO2 = m.dt / 2.0;
  const int nci = n.nci;
  const double ta = n.ta;
  if (ta != 0.0) {
    mx = mx / ta;
    my = my / ta;
  }
  double WSX = 0.0, WSY = 0.0;
  if (q.nws) {
    WSX = DTO2 * 1.0 * (n.wx1 / n.h1 + n.wx2 / n.h2);
    WSY = DTO2 * 1.0 * (n.wy1 / n.h1 + n.wy2 / n.h2);
  }
  const double tk = n.tk;
  const double VXX = DTO2 * (tk + 0.0), VYY = DTO2 * (tk + 0.0);
  const double corifa = n.cor + q.ifnlct * 0.0 * n.u1;
  const double VXY = DTO2 * (0.0 - corifa), VYX = DTO2 * (0.0 + corifa);
  const double u1 = n.u1, v1 = n.v1;
  const double dnci = (double)nci;
  mx = dnci * (mx + WSX + (1.0 - VXX) * u1 - VXY * v1);
  my = dnci * (my + WSY + (1.0 - VYY) * v1 - VYX * u1);
  double A0 = 1.0 + VXX * dnci, A1 = 1.0 + VYY * dnci, A2 = VXY * dnci, A3 = VYX * dnci;
  // land boundary constraints in ME2GW order (src/momentum.F:810-870).  The
  // isotropy test of :816 is ABS(NORM2(TKM) - SQRT(2)*TK) < EPSILON with
  // TKM = (TK, TK, 0): flang's scaled NORM2 gives |TK|*SQRT(2) exactly, so
  // the first branch is taken unless TK is negative (a node whose total
  // depth went negative) and not tiny.
  const double n2tkm = fabs(tk) * __builtin_sqrt(2.0);
  const bool isotropic = fabs(n2tkm - __builtin_sqrt(2.0) * tk) < 2.220446049250313e-16;
  for (int p = n.bc0; p < n.bc1; ++p) {
    const int I = m.vbc[p];
    const int code = m.lbcodei[I];
    const double CS = m.csii[I], SI = m.siii[I];
    const double veln = -(s.qn2 ? s.qn2[I] : 0.0) / n.h2;
    if (code >= 0 && code <= 9) {
      if (isotropic) {
        mx = (SI * mx - CS * my - veln * A2) * dnci;
        my = veln * A0 * dnci;
        A2 = -CS * A0;
        A3 = -A2;
        A0 = SI * A0;
        A1 = A0;
      } else {
        mx = (SI * mx - CS * my) * dnci;
        my = veln * dnci;
        A0 = A0 * SI - A3 * CS;
        A2 = A2 * SI - A1 * CS;
        A3 = CS;
        A1 = SI;
      }
    } else if (code >= 10 && code <= 19) {
      mx = 0.0 * dnci;
      my = veln * dnci;
      A0 = SI;
      A2 = -CS;
      A3 = CS;
      A1 = SI;
    }
  }
  const double ddu = A0 * A1 - A2 * A3;
  const double u2 = (mx * A1 - my * A2) / ddu;
  const double v2 = (my * A0 - mx * A3) / ddu;
  s.uu2[i] = u2;
  s.vv2[i] = v2;
  const double h2 = n.h2;
  s.qx2[i] = u2 * h2;
  s.qy2[i] = v2 * h2;
  const double e2 = n.e2;
  // run-time checks of the reference: ErrorElev over the wet nodes
  // (src/timestep.F:1242-1251, 1381-1395) and a NaN velocity anywhere
  // (src/timestep.F:1413-1471; an infinite one counts too).  The first step
  // that raises either is kept.
  const bool elev_bad = nci == 1 && fabs(e2) > q.errorelev;
  const bool vel_bad = !(fabs(u2) <= 1.7976931348623157e308 && fabs(v2) <= 1.7976931348623157e308);
  if (elev_bad || vel_bad) {
    atomicOr(&q.flags[F_ERROR], (elev_bad ? ERR_ELEV : 0) | (vel_bad ? ERR_NONFINITE : 0));
    atomicCAS(&q.flags[F_ERRSTEP], 0, q.it > 0 ? q.it : 1);
  }
  // peak surge and its step (src/write_output.F:6357-6364; the host turns
  // the step into ETAMAX_Time = IT*DTDP + STATIM*86400)
  if (nci == 1 && e2 > n.emax) {
    s.etamax[i] = e2;
    s.etamax_it[i] = q.it;
  }
  // peak speed and its step (src/write_output.F:6367-6376)
  if (nci == 1) {
    const double ut = __builtin_sqrt(u2 * u2 + v2 * v2);
    if (ut > n.umax) {
      s.umax[i] = ut;
      s.umax_it[i] = q.it;
    }
  }
}

// Momentum: element contributions, node sums and the nodal update.  With ALPHA
// the element's wet/dry ALPHAL is formed here first (nothing reads it between
// the wet/dry pass and this one).
template <bool ALPHA, typename CT>
__device__ __forceinline__ void mom_block(const DevMesh& m, const DevState& s, const DevPatch& pp,
                                          const MomPrm& q, int bid) {
  extern __shared__ double sh[];
  __shared__ __attribute__((aligned(4))) unsigned short code[3 * PATCH_ELEMS];
  __shared__ unsigned char wet[PATCH_WIN];
  const int patch = xcd_tile(bid, pp.n);
  const int t = threadIdx.x, ws = pp.wmax;
  const int i = t < PATCH_WIN ? pp.win[patch * PATCH_WIN + t] : -1;
  const int ke = patch * PATCH_ELEMS + t;
  const ushort4 lv = pp.lv[ke];
  const int e = pp.el[ke];
  const ushort2 c = t < PATCH_NODES ? pp.cspan[patch * PATCH_NODES + t] : make_ushort2(1, 0);
  for (int k = t; k < 3 * PATCH_ELEMS / 2; k += PATCH_THREADS)
    reinterpret_cast<unsigned*>(code)[k] =
        reinterpret_cast<const unsigned*>(pp.code)[patch * (3 * PATCH_ELEMS / 2) + k];
  ElemGeo<double> g;
  if (pp.geo) g.load(pp.geo, pp.nq, ke);
  const int noff = s.noff[e];
  // the thread's window node; for an own node also what its update reads, ahead
  // of the element terms
  MomNode nd;
  const bool own = c.y >= c.x;
  if (i >= 0) {
    nd.u1 = s.uu1[i];
    nd.v1 = s.vv1[i];
    nd.h1 = s.h1[i];
    nd.e2 = s.eta2[i];
    nd.nci = s.nodecode[i];
    if (own) {
      nd.load(m, s, q, i);
      if (q.form_h2) s.h2[i] = nd.h2 = m.dp[i] + q.ifnlfa * nd.e2;
    }
    W(MF_X, t) = m.x[i];
    W(MF_Y, t) = m.y[i];
    W(MF_EVM, t) = m.evm[i];
    W(MF_E1, t) = s.eta1[i];
    if (ALPHA) W(MF_DP, t) = m.dp[i];
    if (q.nws) {
      W(MF_P1, t) = s.pr1[i];
      W(MF_P2, t) = s.pr2[i];
    }
    if (s.tip1) {
      W(MF_T1, t) = s.tip1[i];
      W(MF_T2, t) = s.tip2[i];
    }
    W(MF_U, t) = nd.u1;
    W(MF_V, t) = nd.v1;
    W(MF_H1, t) = nd.h1;
    W(MF_E2, t) = nd.e2;
    wet[t] = (unsigned char)nd.nci;
  }
  // ALPHAL is 1 everywhere unless the last pass, the one before or the host
  // left another value; only then is the field read or rewritten
  const bool stored = q.flags[ALPHA ? F_ALPHA0 : F_ALPHA] != 0;
  __syncthreads();
  // dry element: every contribution is NCEle*DT x (...) = 0 (see k_gwce)
  CT tx[3] = {0, 0, 0}, ty[3] = {0, 0, 0};
  if (lv.w != 2) {
    const int ncele = wet[lv.x] * wet[lv.y] * wet[lv.z] * noff;
    // the flags are final for this step: NCEle as the next GWCE pass sees it
    s.ncele[ke] = (unsigned char)ncele;
    double al = 1.0;
    if (ncele != 0 && !pp.geo) g.form(sh, ws, lv.x, lv.y, lv.z);
    if (ALPHA) {
      if (ncele == 1) al = alpha_terms(sh, ws, lv.x, lv.y, lv.z, g, 1.0e9);
      if ((stored || al != 1.0) && lv.w == 1) s.alphal[e] = al;
      if (al != 1.0) atomicOr(&q.flags[F_ALPHA], 1);
    } else if (stored) {
      al = s.alphal[e];
    }
    if (ncele != 0) {
      const ElemGeo<CT> gc(g);
      mom_terms(sh, ws, lv.x, lv.y, lv.z, m, s, q, gc, ncele, al, tx, ty);
    }
  }
  __syncthreads();  // the window's LDS is free
  CT* const cx = reinterpret_cast<CT*>(sh);  // [3][PATCH_ELEMS]
  CT* const cy = cx + 3 * PATCH_ELEMS;
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    cx[k * PATCH_ELEMS + t] = tx[k];
    cy[k * PATCH_ELEMS + t] = ty[k];
  }
  __syncthreads();
  if (!own) return;
  double mx = 0.0, my = 0.0;
  if (sizeof(CT) == 4) {
    Kahan32 kx, ky;  // FP32 contributions: compensated sums
    for (int p = c.x; p < c.y; ++p) {
      kx.add((float)cx[code[p]]);
      ky.add((float)cy[code[p]]);
    }
    mx = kx.value();
    my = ky.value();
  } else {
    for (int p = c.x; p < c.y; ++p) {
      mx = mx + cx[code[p]];
      my = my + cy[code[p]];
    }
  }
  mom_node(m, s, q, nd, i, mx, my);
}

template <bool ALPHA, typename CT>
__global__ __launch_bounds__(PATCH_THREADS, 5) void k_mom(DevMesh m, DevState s, DevPatch pp, MomPrm q) {
  mom_block<ALPHA, CT>(m, s, pp, q, blockIdx.x);
}
template <typename CT>
__global__ __launch_bounds__(PATCH_THREADS, 5) void k_mom_batch(const MemberArgs* __restrict__ a, int it) {
  const MemberArgs& x = a[blockIdx.y];
  if ((int)blockIdx.x >= x.pp.n) return;
  MomPrm q = x.mq;
  q.it = it;
  mom_block<true, CT>(x.m, x.s, x.pp, q, blockIdx.x);
}
template __global__ void k_mom_batch<double>(const MemberArgs*, int);
template __global__ void k_mom_batch<float>(const MemberArgs*, int);
template __global__ void k_mom<false, double>(DevMesh, DevState, DevPatch, MomPrm);
template __global__ void k_mom<true, double>(DevMesh, DevState, DevPatch, MomPrm);
template __global__ void k_mom<false, float>(DevMesh, DevState, DevPatch, MomPrm);
template __global__ void k_mom<true, float>(DevMesh, DevState, DevPatch, MomPrm);
#undef W

}  // namespace adcgpu
