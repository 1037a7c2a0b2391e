// CDNA4 (gfx950) kernels for the vertically implicit part of FElib's HEVI
// scheme (FDS/scale_atm_dyn_dgm_nonhydro3d_rhot_hevi.F90:772-965 and
// FDS/scale_atm_dyn_dgm_nonhydro3d_rhot_hevi_common_2.F90:111-1328).
//
// One Newton iteration is four launches:
//   1. hevi_rhs_uv   (element, one thread per node): the damping coefficient
//      alph at every vertical face node from q^n, the horizontal-momentum
//      face jumps of the iterate, their lift, MOMX_t / MOMY_t and the uv rhs;
//   2. hevi_solve_uv (64/8 lines per wavefront at p = 7, a lane per node):
//      assembles the N x N blocks of construct_matbnd_uv level by level,
//      block-Thomas elimination with the pivoted LU of solve_NnodeN_uv, back
//      substitution, MOMX, MOMY += increment;
//   3. hevi_rhs3     (element): vertical fluxes of DDENS, MOMZ, DRHOT, their
//      face jumps, Dz and lift, VFilterPM1 buoyancy, the var3 rhs and the
//      linearisation coefficients POT, WT, DPDRHOT;
//   4. hevi_solve3   (eight lines per wavefront at p = 7, a lane per node):
//      the 3N x 3N blocks of construct_matbnd, block-Thomas with the LU of
//      solve_NnodeN_var3, DDENS, MOMZ, DRHOT += increment.
// A line is the column of one horizontal node (ij) of one horizontal element
// through all NeZ elements; everything the implicit operator couples lies on
// it.  A block's columns stay in registers of their lanes, multipliers travel
// by cross-lane moves, and the levels' solutions wait in a scratch area for the
// block back substitution.  Every entry sees the same operations in the same
// order as the reference's serial loops, so results are bit for bit those of
// the CPU restatement.
#include <algorithm>
#include <cfloat>
#include <cmath>
#include <mutex>
#include <type_traits>

#include "fedg_device.h"
#include "fedg_hevi.h"
#include "fedg_mlp.h"


namespace fedg {
namespace {

struct HeviArgs {
  DevMesh m;
  Consts c;
  const double* qs[5];     // stage state q* (VID order), (Np,NeA)
  const double* q0[5];     // var0 = q^n
  double* pv[5];           // Newton iterate, (Np,Ne), written by the solves
  const double* pin[5];    // the iterate as read: pv, or q^n for a variable no solve has updated yet
  const double* DENS_hyd;
  const double* PRES_hyd;
  const double* RHOT_hyd;  // PRES00/Rdry (PRES_hyd/PRES00)^(CVdry/CPdry) per node, or null: formed in the kernels
  int alph_ready;          // alph holds the damping coefficients of q0 (a residual kernel formed them)
  const double* Rtot;
  const double* CVtot;
  const double* CPtot;
  double* alph;            // (2*Nfp, Ne): z- then z+ face nodes
  double* b3;              // (3, Np*Ne): DENS, MOMZ, RHOT rhs
  double* buv;             // (2, Np*Ne)
  double* coef;            // (3, Np*Ne): POT, WT, DPDRHOT
  double* T[5];            // implicit-operator tendencies (VID order)
  int* flagged;            // groups of lines whose pivots leave the diagonal: their number, then the groups
  double* lines;           // scratch of the line solves: the level solutions of every wavefront in flight
  double impl_fac;
  int want_b;              // form the rhs (Newton) or only the operator (impl_fac = 0)
  int NeZ;
  int finish;              // FINISH_*: what the line solves store
  double* qst[5];          // StoreImplicit: the stage state as written (qs), and its copies
  double* var0[5];
  double* varTmp[5];
};
// What the solve of DENS, MOMZ and RHOT stores: the iterate; or, in the last
// iteration of a fixed number, what hevi_tend_store_kernel would form from it.
// The solve is bound by its arithmetic, so the stores hide behind it; MOMX and
// MOMY, whose solve is not (143 -> 206 us with them) and whose iterate the others'
// residual reads, stay with the kernel.  60 x 16 x 8 elements at p = 7, a stage:
// solve 776 -> 808 us, the kernel behind it 104 -> 42 us; drop-in solve of
// 240 x 16 x 8 elements 4848 -> 4683 us.
enum { FINISH_NONE = 0, FINISH_TEND = 1, FINISH_STORE = 2, FINISH_STORE_COPY = 3 };

// a node's value P of the iterate, qs = q* there
__device__ __forceinline__ void finish_node(const HeviArgs& a, int v, uint32_t o, double P, double qs) {
  const double T = (P - qs) / a.impl_fac;
  stg_nt(a.T[v], o, T);
  if (a.finish == FINISH_TEND) return;
  if (a.finish == FINISH_STORE_COPY) {
    stg_nt(a.var0[v], o, qs);
    stg_nt(a.varTmp[v], o, qs);
  }
  stg(a.qst[v], o, qs + a.impl_fac * T);
}

__device__ __forceinline__ double gsqrtv(const HeviArgs& a, int ke, int p, int N1) {
  const int ke2d = a.m.EMap3Dto2D[ke];
  const int ij = p % (N1 * N1);
  return ldg(a.m.Gsqrt, (uint32_t)a.m.Np * ke + p) / ldg(a.m.GsqrtH, (uint32_t)ij + (uint32_t)a.m.Nfp * ke2d);
}

// vertical neighbour node of the face node (bottom: f = 0, top: f = 1); self at the column ends
__device__ __forceinline__ uint32_t vz_nbr(const HeviArgs& a, int ke, int f, int ij, int N1) {
  const int Ne2D = a.m.Ne2D;
  const int kz = ke / Ne2D;
  const uint32_t Np = a.m.Np, Nfp = a.m.Nfp;
  if (f == 0) {
    if (kz > 0) return Np * (ke - Ne2D) + ij + Nfp * (N1 - 1);
    return Np * ke + ij;
  }
  if (kz < a.NeZ - 1) return Np * (ke + Ne2D) + ij;
  return Np * ke + ij + Nfp * (N1 - 1);
}

// ---------------------------------------------------------------------------
// 1. vi_cal_del_flux_dyn_uv (:1015-1158) + eval_Ax_uv (:482-586)
// FLAT (the flat-terrain uniform box the context detected): the metric
// arrays hold Gsqrt = GsqrtH = 1, G13 = G23 = 0, G11 = G22 = 1, G12 = 0,
// nz = -1 / +1 on the bottom / top faces, E33 and Fscale constant and a
// tensor-product Lift, so those values are taken from the context's
// constants instead of loaded; every operation is kept, so the results are
// the same bits.  The outputs (and, in hevi_rhs3_body, the coefficients) and
// the stage state q* are streamed with the non-temporal hint, so that the
// iterate lines the vertical neighbours gather stay cached.
template <int N1, bool FLAT>
__device__ __forceinline__ void hevi_rhs_uv_body(const HeviArgs& a) {
  constexpr int Np = N1 * N1 * N1, Nfp = N1 * N1;
  __shared__ double sdf[2][2][Nfp];  // face (bottom, top), var (MOMX, MOMY), node
  __shared__ double sPow[640];        // the pow tables (the same values as the global ones)
  const int p = threadIdx.x;
  const int ke = blockIdx.x;
  const int ij = p % Nfp, k = p / Nfp;
  const DevMesh& m = a.m;
  const Consts& c = a.c;
  const uint32_t o = (uint32_t)Np * ke + p;
  if (a.flagged && ke == 0 && p == 0) a.flagged[0] = 0;  // for the line solve that follows
  const double gamm = c.CPdry / c.CVdry, rgamm = c.CVdry / c.CPdry;
  const double PRES0ovRdry = c.PRES00 / c.Rdry, rP0 = 1.0 / c.PRES00;
  if (!a.alph_ready) {
    pow_tables_to(sPow, p, Np);
    __syncthreads();
  }
  if (k == 0 || k == N1 - 1) {
    for (int f = 0; f < 2; ++f) {
      if ((f == 0) != (k == 0)) continue;
      const int fp = (4 + f) * Nfp + ij;  // reference face-node index
      const uint32_t gfp = (uint32_t)fp + (uint32_t)(6 * Nfp) * ke;
      const uint32_t iM = o, iP = vz_nbr(a, ke, f, ij, N1);
      const uint32_t ia = (uint32_t)(f * Nfp + ij) + (uint32_t)(2 * Nfp) * ke;
      double al;
      if (a.alph_ready) {
        al = ldg(a.alph, ia);
      } else {
        const double nz = FLAT ? (f == 0 ? -1.0 : 1.0) : ldg(m.nz, gfp);
        const int ke2d = FLAT ? 0 : m.EMap3Dto2D[ke];
        const double G11_ = FLAT ? 1.0 : ldg(m.G11, (uint32_t)ij + (uint32_t)Nfp * ke2d);
        const double G12_ = FLAT ? 0.0 : ldg(m.G12, (uint32_t)ij + (uint32_t)Nfp * ke2d);
        const double G22_ = FLAT ? 1.0 : ldg(m.G22, (uint32_t)ij + (uint32_t)Nfp * ke2d);
        double wt0[2], pres0[2], rdens0[2], Gnn[2];
        const uint32_t ix[2] = {iM, iP};
        for (int s = 0; s < 2; ++s) {
          const uint32_t n = ix[s];
          const int ken = n / Np;
          const double gam = 1.0;
          const double rgam2 = 1.0 / (gam * gam);
          const double RGsqrtV = 1.0 / (FLAT ? 1.0 : gsqrtv(a, ken, n - (uint32_t)Np * ken, N1));
          const double MOMX0 = ldg(a.q0[VU], n), MOMY0 = ldg(a.q0[VV], n), DRHOT0 = ldg(a.q0[VT], n);
          const double Rt = ldg(a.Rtot, n), CPovCV = ldg(a.CPtot, n) / ldg(a.CVtot, n);
          const double g13 = FLAT ? 0.0 : ldg(m.G13, n), g23 = FLAT ? 0.0 : ldg(m.G23, n);
          rdens0[s] = 1.0 / (ldg(a.DENS_hyd, n) + ldg(a.q0[VD], n));
          wt0[s] = (ldg(a.q0[VW], n) * RGsqrtV + g13 * MOMX0 + g23 * MOMY0) * rdens0[s];
          const double rhot_hyd = a.RHOT_hyd ? ldg(a.RHOT_hyd, n)
                                             : PRES0ovRdry * fedg_pow_tab(ldg(a.PRES_hyd, n) / c.PRES00, rgamm, sPow);
          pres0[s] = c.PRES00 * fedg_pow_tab(Rt * rP0 * (rhot_hyd + DRHOT0), CPovCV, sPow);
          const double Gxz = rgam2 * (G11_ * g13 + G12_ * g23);
          const double Gyz = rgam2 * (G12_ * g13 + G22_ * g23);
          Gnn[s] = (1.0 * (RGsqrtV * RGsqrtV) + g13 * Gxz + g23 * Gyz) * fabs(nz);
        }
        const double sM = fabs(wt0[0]) + sqrt(Gnn[0] * gamm * pres0[0] * rdens0[0]);
        const double sP = fabs(wt0[1]) + sqrt(Gnn[1] * gamm * pres0[1] * rdens0[1]);
        al = (nz * nz) * (sM > sP ? sM : sP);
        stg(a.alph, ia, al);
      }
      const double tmp1 = -0.5 * (FLAT ? m.fF[4 + f] : ldg(m.Fscale, gfp)) * al;
      sdf[f][0][ij] = tmp1 * (ldg(a.pin[VU], iP) - ldg(a.pin[VU], iM));
      sdf[f][1][ij] = tmp1 * (ldg(a.pin[VV], iP) - ldg(a.pin[VV], iM));
    }
  }
  __syncthreads();
  // Lift of the vertical-face jumps (the lateral faces carry none)
  const double L4 = FLAT ? m.liftT[k + N1 * 4] : ldg(m.Lift, (uint32_t)(p + 4 * Np));
  const double L5 = FLAT ? m.liftT[k + N1 * 5] : ldg(m.Lift, (uint32_t)(p + 5 * Np));
  const double LDx = L4 * sdf[0][0][ij] + L5 * sdf[1][0][ij];
  const double LDy = L4 * sdf[0][1][ij] + L5 * sdf[1][1][ij];
  const double RGsqrtV = 1.0 / (FLAT ? 1.0 : gsqrtv(a, ke, p, N1));
  const double Tx = -LDx * RGsqrtV, Ty = -LDy * RGsqrtV;
  if (a.want_b) {
    const uint32_t n = (uint32_t)Np * m.Ne;
    stg_nt(a.buv, o, a.impl_fac * Tx - ldg(a.pin[VU], o) + ldg_nt(a.qs[VU], o));
    stg_nt(a.buv, o + n, a.impl_fac * Ty - ldg(a.pin[VV], o) + ldg_nt(a.qs[VV], o));
  } else {
    stg_nt(a.T[VU], o, Tx);
    stg_nt(a.T[VV], o, Ty);
  }
}

// ---------------------------------------------------------------------------
// 3. vi_cal_del_flux_dyn (:1161-1328) + eval_Ax (:111-326)
template <int N1, bool FLAT>
__device__ __forceinline__ void hevi_rhs3_body(const HeviArgs& a) {
  constexpr int Np = N1 * N1 * N1, Nfp = N1 * N1;
  __shared__ double sF[3][Np];      // DENS, MOMZ, RHOT vertical fluxes
  __shared__ double sRho[Np];
  __shared__ double sdf[2][3][Nfp];  // face (bottom, top), var (DENS, MOMZ, RHOT), node
  __shared__ double sD[N1 * N1];
  __shared__ double sI[N1 * N1];
  __shared__ double sPow[640];  // the pow tables (the same values as the global ones)
  const int p = threadIdx.x;
  const int ke = blockIdx.x;
  const int ij = p % Nfp, k = p / Nfp;
  const DevMesh& m = a.m;
  const Consts& c = a.c;
  const uint32_t o = (uint32_t)Np * ke + p;
  const int kz = ke / m.Ne2D;
  const double rgamm = c.CVdry / c.CPdry;
  const double PRES0ovRdry = c.PRES00 / c.Rdry, rP0 = 1.0 / c.PRES00, P0ovR = c.PRES00 / c.Rdry;
  if (p < N1 * N1) {
    sD[p] = m.D1D[p];
    sI[p] = m.Itr[p];
  }
  pow_tables_to(sPow, p, Np);
  __syncthreads();
  // vertical face jumps of the iterate
  if (k == 0 || k == N1 - 1) {
    for (int f = 0; f < 2; ++f) {
      if ((f == 0) != (k == 0)) continue;
      const int fp = (4 + f) * Nfp + ij;
      const uint32_t gfp = (uint32_t)fp + (uint32_t)(6 * Nfp) * ke;
      const uint32_t iM = o, iP = vz_nbr(a, ke, f, ij, N1);
      const uint32_t ix[2] = {iM, iP};
      double DD[2], MZ[2], MW[2], DT[2], pott[2], dpres[2], GV[2];
      for (int s = 0; s < 2; ++s) {
        const uint32_t n = ix[s];
        const int ken = n / Np;
        GV[s] = FLAT ? 1.0 : gsqrtv(a, ken, n - (uint32_t)Np * ken, N1);
        DD[s] = ldg(a.pin[VD], n);
        MZ[s] = ldg(a.pin[VW], n);
        DT[s] = ldg(a.pin[VT], n);
        const double dens = ldg(a.DENS_hyd, n) + DD[s];
        const double PH = ldg(a.PRES_hyd, n);
        const double rhot_hyd = a.RHOT_hyd ? ldg(a.RHOT_hyd, n) : PRES0ovRdry * fedg_pow_tab(PH / c.PRES00, rgamm, sPow);
        pott[s] = (rhot_hyd + DT[s]) / dens;
        dpres[s] = c.PRES00 * fedg_pow_tab(ldg(a.Rtot, n) * rP0 * dens * pott[s], ldg(a.CPtot, n) / ldg(a.CVtot, n), sPow);
        dpres[s] = dpres[s] - PH;
        const double g13 = FLAT ? 0.0 : ldg(m.G13, n), g23 = FLAT ? 0.0 : ldg(m.G23, n);
        MW[s] = MZ[s] + GV[s] * g13 * ldg(a.pin[VU], n) + GV[s] * g23 * ldg(a.pin[VV], n);
      }
      if ((kz == 0 || kz == a.NeZ - 1) && iM == iP) {
        const double g13 = FLAT ? 0.0 : ldg(m.G13, iM), g23 = FLAT ? 0.0 : ldg(m.G23, iM);
        MZ[1] = -MZ[0] - 2.0 * GV[0] * (g13 * ldg(a.pin[VU], iM) + g23 * ldg(a.pin[VV], iM));
        MW[1] = -MW[0];
      }
      const double nz = FLAT ? (f == 0 ? -1.0 : 1.0) : ldg(m.nz, gfp);
      const double al = ldg(a.alph, (uint32_t)(f * Nfp + ij) + (uint32_t)(2 * Nfp) * ke);
      const double tmp1 = 0.5 * (FLAT ? m.fF[4 + f] : ldg(m.Fscale, gfp));
      sdf[f][0][ij] = tmp1 * (+(MW[1] - MW[0]) * nz - al * (DD[1] - DD[0]));
      sdf[f][1][ij] = tmp1 * (+(dpres[1] - dpres[0]) * nz - al * (MZ[1] - MZ[0]));
      sdf[f][2][ij] = tmp1 * (+(pott[1] * MW[1] - pott[0] * MW[0]) * nz - al * (DT[1] - DT[0]));
    }
  }
  // vertical fluxes of the node
  const double GV = FLAT ? 1.0 : gsqrtv(a, ke, p, N1);
  const double PVD = ldg(a.pin[VD], o), PVW = ldg(a.pin[VW], o), PVT = ldg(a.pin[VT], o);
  const double G13o = FLAT ? 0.0 : ldg(m.G13, o), G23o = FLAT ? 0.0 : ldg(m.G23, o);
  const double FD = PVW + GV * G13o * ldg(a.pin[VU], o) + GV * G23o * ldg(a.pin[VV], o);
  const double PH = ldg(a.PRES_hyd, o), DH = ldg(a.DENS_hyd, o);
  const double RHOT = (a.RHOT_hyd ? ldg(a.RHOT_hyd, o) : P0ovR * fedg_pow_tab(PH / c.PRES00, rgamm, sPow)) + PVT;
  const double pt_ = RHOT / (PVD + DH);
  const double Rt = ldg(a.Rtot, o), CPt = ldg(a.CPtot, o), CVt = ldg(a.CVtot, o);
  const double FW = c.PRES00 * fedg_pow_tab(Rt * rP0 * RHOT, CPt / CVt, sPow) - PH;
  sF[0][p] = FD;
  sF[1][p] = FW;
  sF[2][p] = pt_ * FD;
  sRho[p] = PVD;
  __syncthreads();
  // Dz (matvec_dirZ), VFilterPM1 and the lift of the vertical-face jumps
  double dz[3];
#pragma unroll
  for (int v = 0; v < 3; ++v) {
    double s = sF[v][ij] * sD[k];
#pragma unroll
    for (int l = 1; l < N1; ++l) s = s + sF[v][ij + Nfp * l] * sD[k + N1 * l];
    dz[v] = s;
  }
  double drho = sRho[ij] * sI[N1 * k];
#pragma unroll
  for (int l = 1; l < N1; ++l) drho = drho + sRho[ij + Nfp * l] * sI[l + N1 * k];
  const double L4 = FLAT ? m.liftT[k + N1 * 4] : ldg(m.Lift, (uint32_t)(p + 4 * Np));
  const double L5 = FLAT ? m.liftT[k + N1 * 5] : ldg(m.Lift, (uint32_t)(p + 5 * Np));
  const double E33 = FLAT ? m.fE[2] : ldg(m.E33, o);
  const double RGsqrtV = 1.0 / GV;
  const double TD = -(E33 * dz[0] + (L4 * sdf[0][0][ij] + L5 * sdf[1][0][ij])) * RGsqrtV;
  const double TT = -(E33 * dz[2] + (L4 * sdf[0][2][ij] + L5 * sdf[1][2][ij])) * RGsqrtV;
  const double TW = -(E33 * dz[1] + (L4 * sdf[0][1][ij] + L5 * sdf[1][1][ij])) * RGsqrtV - c.GRAV * drho;
  if (a.want_b) {
    const uint32_t n = (uint32_t)Np * m.Ne;
    const double dens = DH + PVD;
    stg_nt(a.coef, o, RHOT / dens);
    stg_nt(a.coef, o + n, FD / dens);
    const double CPovCV = CPt / CVt;
    stg_nt(a.coef, o + 2 * n, CPovCV * c.PRES00 * fedg_pow_tab(Rt / c.PRES00 * RHOT, CPovCV, sPow) / RHOT);
    stg_nt(a.b3, o, a.impl_fac * TD - PVD + ldg_nt(a.qs[VD], o));
    stg_nt(a.b3, o + n, a.impl_fac * TW - PVW + ldg_nt(a.qs[VW], o));
    stg_nt(a.b3, o + 2 * n, a.impl_fac * TT - PVT + ldg_nt(a.qs[VT], o));
  } else {
    stg_nt(a.T[VD], o, TD);
    stg_nt(a.T[VW], o, TW);
    stg_nt(a.T[VT], o, TT);
  }
}

// ---------------------------------------------------------------------------
// Line solves: block Thomas over the levels of a vertical line, each level's
// n x n block (n = NS N, unknown j = NS node + variable) by the pivoted LU of
// solve_NnodeN_var3 / _uv (FDS/scale_atm_dyn_dgm_hevi_common_linalgebra.F90:
// 2142-2445).
//
// A line owns a segment of SEG lanes (4 for N <= 4, else 8): lane c holds the
// NS columns of node c, A[s][i] = entry (row i, column NS c + s), and lanes
// 0..3 hold up to four right-hand sides in B[i]; 64 / SEG lines share a
// wavefront.  With whole columns in a lane's registers
//  - the pivot search, the reciprocal and the scaled column are lane-local;
//    only the multipliers l(i) travel, from a lane known at compile time
//    (DPP broadcasts: no LDS traffic in the elimination);
//  - one broadcast l(i) updates row i of all NS columns and the right-hand
//    sides of every line of the wavefront;
//  - rows are exchanged in the registers, only when a line's pivot is not on
//    the diagonal (rare for the diagonally dominant blocks of the usual steps).
// Bound: FP64 VALU issue (about 5,500 instructions per level of eight p = 7
// lines, 11 per multiplier: product, two moves, four multiply-subtract pairs;
// VALU busy 0.84 of the time).  A block needs 2 n (NS + 1) VGPRs (192 at
// p = 7), so two wavefronts share a SIMD and nothing else may stay in
// registers across the LU: a spilled address waits, in the one order vector
// memory completes in, for the stores before it (with 40 spilled registers
// 3.5 ms, with 300 6.9 ms).  The levels' solutions (b and the coupling
// columns) go to a scratch area of the wavefront's own, whose traffic hides
// behind the arithmetic, and a level's operands are loaded during the level
// before.
// Measured on the 240 x 16 x 8 p = 7 channel, per solve: 12.6 ms in the layout
// before (one row per lane, two lines per wavefront, the pivot row through LDS
// permutes) -> 3.2 ms; uv 0.745 -> 0.555 ms; 12 x 6 x 6 p = 3: 56 -> 37 us, uv
// 17.1 -> 12.7 us.
// The operations every entry sees -- pivot choice (first largest), reciprocal
// of the pivot, scaling of the column, rank-1 update, forward substitution,
// back substitution in ascending column order -- are those of the reference's
// serial loops, so results are bit for bit the CPU restatement's.

template <int I, int E, class F>
__device__ __forceinline__ void static_for(F&& f) {
  if constexpr (I < E) {
    f(std::integral_constant<int, I>{});
    static_for<I + 1, E>(f);
  }
}

// the value of lane C of the caller's SEG-lane segment, in two steps: for 8
// lanes row_newbcast of lane C to the 16-lane row, then of lane C + 8 to its
// upper half (banks 2 and 3); for 4 lanes quad_perm [C, C, C, C]
template <int SEG, int C>
__device__ __forceinline__ double bcast_1(double v) {
  if constexpr (SEG == 4) {
    constexpr int q = C * 0x55;
    return __hiloint2double(__builtin_amdgcn_mov_dpp(__double2hiint(v), q, 0xF, 0xF, true),
                            __builtin_amdgcn_mov_dpp(__double2loint(v), q, 0xF, 0xF, true));
  } else {
    return __longlong_as_double(__builtin_amdgcn_mov_dpp(__double_as_longlong(v), 0x150 + C, 0xF, 0xF, true));
  }
}
template <int SEG, int C>
__device__ __forceinline__ double bcast_2(double r, double v) {
  if constexpr (SEG == 4) return r;
  else
    return __longlong_as_double(__builtin_amdgcn_update_dpp(__double_as_longlong(r), __double_as_longlong(v),
                                                            0x158 + C, 0xF, 0xC, false));
}
template <int SEG, int C>
__device__ __forceinline__ double bcast(double v) {
  return bcast_2<SEG, C>(bcast_1<SEG, C>(v), v);
}
// the values are formed here, in this order (no instruction)
template <int M>
__device__ __forceinline__ void pin(double* x) {
  if constexpr (M == 1) asm volatile("" : "+v"(x[0]));
  if constexpr (M == 2) asm volatile("" : "+v"(x[0]), "+v"(x[1]));
  if constexpr (M == 3) asm volatile("" : "+v"(x[0]), "+v"(x[1]), "+v"(x[2]));
  if constexpr (M == 4) asm volatile("" : "+v"(x[0]), "+v"(x[1]), "+v"(x[2]), "+v"(x[3]));
}
template <int SEG, int C>
__device__ __forceinline__ int bcast_i(int v) {
  if constexpr (SEG == 4) {
    return __builtin_amdgcn_mov_dpp(v, C * 0x55, 0xF, 0xF, true);
  } else {
    const int r = __builtin_amdgcn_mov_dpp(v, 0x150 + C, 0xF, 0xF, true);
    return __builtin_amdgcn_update_dpp(r, v, 0x158 + C, 0xF, 0xC, false);
  }
}

// LDS of one wavefront: writes by some lanes are read by others of the same
// wavefront, whose LDS operations complete in order; only the compiler has to
// keep the order.
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// exchanges two register pairs where they are: through a third, or (HALVES)
// half by half without one, which is slower but lets the n = 24 solve with row
// exchanges spill 24 registers where it spills 55
template <bool HALVES>
__device__ __forceinline__ void swap_in_place(double& x, double& y) {
  if constexpr (HALVES) {
    int x0 = __double2loint(x), x1 = __double2hiint(x), y0 = __double2loint(y), y1 = __double2hiint(y);
    asm("v_swap_b32 %0, %1" : "+v"(x0), "+v"(y0));
    asm("v_swap_b32 %0, %1" : "+v"(x1), "+v"(y1));
    x = __hiloint2double(x1, x0);
    y = __hiloint2double(y1, y0);
  } else {
    double t;
    asm("v_mov_b64 %2, %0\n\tv_mov_b64 %0, %1\n\tv_mov_b64 %1, %2" : "+v"(x), "+v"(y), "=&v"(t));
  }
}

// max(|a|, |b|); a NaN is passed over unless both are
__device__ __forceinline__ double max_abs(double a, double b) {
  double r;
  asm("v_max_f64 %0, |%1|, |%2|" : "=v"(r) : "v"(a), "v"(b));
  return r;
}

// row i of the block is complete here (no instruction)
template <int NS, int n>
__device__ __forceinline__ void keep_order(double (&A)[NS][n], double (&B)[n], int i) {
  if constexpr (NS == 1) asm volatile("" : "+v"(A[0][i]), "+v"(B[i]));
  else asm volatile("" : "+v"(A[0][i]), "+v"(A[1][i]), "+v"(A[2][i]), "+v"(B[i]));
}

// LU of every segment's block, applied to the right-hand sides as it goes,
// then back substitution: B becomes the solution (lanes 0..3).
// PIVOT false: no rows are exchanged; false is returned when a line's pivot
// was not on the diagonal (its result is then to be discarded), so that the
// path is one stretch of code without a branch, whose registers hold the
// blocks.  PIVOT true: rows are exchanged in the registers (the branches make
// the allocator spill at n >= 21).
// ahead() is called in the back substitution once registers have come free:
// the next level's loads, whose latency the rest of it covers.
template <int NS, int N, int SEG, bool PIVOT, class F>
__device__ __forceinline__ bool lu_solve_cols(double (&A)[NS][NS * N], double (&B)[NS * N], int c, F&& ahead) {
  constexpr int n = NS * N;
  double inv = 1.0 / A[0][0];
  unsigned long long off = 0;
  static_for<0, n>([&](auto K) __attribute__((always_inline)) {
    constexpr int k = decltype(K)::value, ck = k / NS, sk = k % NS;
    if constexpr (k < n - 1) {
      // the largest entry below the diagonal, by halves: one chain of five
      // instead of a compare and a mask per entry
      constexpr int m = n - 1 - k;
      double top[m];
#pragma unroll
      for (int i = 0; i < m; ++i) top[i] = A[sk][k + 1 + i];
#pragma unroll
      for (int d = 1; d < m; d *= 2)
#pragma unroll
        for (int i = 0; i + d < m; i += 2 * d) top[i] = max_abs(top[i], top[i + d]);
      const double big = fabs(top[0]);
      const bool larger = big > fabs(A[sk][k]);
      const unsigned long long here = __ballot(larger & (c == ck));
      if constexpr (!PIVOT) {
        off |= here;
        asm volatile("" : "+s"(off));  // compared now: the column's old entries are not kept for later
      } else if (here) {
        // the first largest entry of a column with a larger one (NaN entries
        // are passed over, a NaN on the diagonal stays, as in the reference's
        // running comparison)
        int p = k;
#pragma unroll
        for (int i = n - 1; i > k; --i) p = fabs(A[sk][i]) == big ? i : p;
        p = larger ? p : k;
        p = bcast_i<SEG, ck>(p);
#pragma unroll
        for (int i = k + 1; i < n; ++i) {
          if (p == i) {
#pragma unroll
            for (int s = 0; s < NS; ++s) swap_in_place<(n > 21)>(A[s][i], A[s][k]);
            swap_in_place<(n > 21)>(B[i], B[k]);
          }
        }
        inv = 1.0 / A[sk][k];
      }
    }
    const double inv_k = inv;
    // Rows in chunks of CH, the multipliers one chunk ahead: each step of a
    // chunk's broadcasts lies more than the two instructions a DPP operand
    // needs behind the step before it, and no more multipliers are held than
    // the registers take.
    constexpr int CH = 3;
    auto multipliers = [&](auto I0, double* l) __attribute__((always_inline)) {
      constexpr int i0 = decltype(I0)::value, M = n - i0 < CH ? n - i0 : CH;
      if constexpr (M > 0) {
        double x[M];
#pragma unroll
        for (int r = 0; r < M; ++r) x[r] = A[sk][i0 + r] * inv_k;
        pin<M>(x);
#pragma unroll
        for (int r = 0; r < M; ++r) l[r] = bcast_1<SEG, ck>(x[r]);
        pin<M>(l);
#pragma unroll
        for (int r = 0; r < M; ++r) l[r] = bcast_2<SEG, ck>(l[r], x[r]);
        pin<M>(l);
      }
    };
    double l[CH] = {}, lnext[CH] = {};
    multipliers(std::integral_constant<int, k + 1>{}, l);
    static_for<0, (n - 1 - k + CH - 1) / CH>([&](auto Q) __attribute__((always_inline)) {
      constexpr int i0 = k + 1 + decltype(Q)::value * CH, M = n - i0 < CH ? n - i0 : CH;
      __builtin_amdgcn_sched_barrier(0);
      multipliers(std::integral_constant<int, i0 + CH>{}, lnext);
#pragma unroll
      for (int r = 0; r < M; ++r) {
        const int i = i0 + r;
#pragma unroll
        for (int s = 0; s < NS; ++s)
          if (NS * (N - 1) + s > k) A[s][i] = A[s][i] - l[r] * A[s][k];  // some lane's column is still ahead
        B[i] = B[i] - B[k] * l[r];
        keep_order(A, B, i);
        if (i == k + 1) inv = 1.0 / A[(k + 1) % NS][i];
      }
#pragma unroll
      for (int r = 0; r < CH; ++r) l[r] = lnext[r];
    });
    // the reciprocal of the pivot on the diagonal of U
    A[sk][k] = (c == ck) ? inv_k : A[sk][k];
  });
  static_for<0, n>([&](auto I) __attribute__((always_inline)) {
    constexpr int i = n - 1 - decltype(I)::value;
    // row i's broadcasts start no earlier than row i + 2 is done (all of them
    // hoisted to the top would not fit the registers)
    if constexpr (i + 2 < n) {
#pragma unroll
      for (int s = 0; s < NS; ++s) asm volatile("" : "+v"(A[s][i]), "+v"(B[i + 2]));
    }
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (i == n - 1 - n / 3) {
      ahead();
      __builtin_amdgcn_sched_barrier(0);
    }
    double t = B[i];
    const double d = bcast<SEG, i / NS>(A[i % NS][i]);
    constexpr int CB = 4;
    static_for<0, (n - 1 - i + CB - 1) / CB>([&](auto Q) __attribute__((always_inline)) {
      constexpr int j0 = i + 1 + decltype(Q)::value * CB, M = n - j0 < CB ? n - j0 : CB;
      double x[M];
      static_for<0, M>([&](auto R) __attribute__((always_inline)) {
        constexpr int j = j0 + decltype(R)::value;
        x[j - j0] = bcast_1<SEG, j / NS>(A[j % NS][i]);
      });
      pin<M>(x);
      static_for<0, M>([&](auto R) __attribute__((always_inline)) {
        constexpr int j = j0 + decltype(R)::value;
        x[j - j0] = bcast_2<SEG, j / NS>(x[j - j0], A[j % NS][i]) * B[j];
      });
      pin<M>(x);
#pragma unroll
      for (int r = 0; r < M; ++r) t = t - x[r];
    });
    B[i] = t * d;
  });
  return off == 0;
}

template <int N1>
struct LineSeg {
  static constexpr int SEG = N1 <= 4 ? 4 : 8;
  static constexpr int LPW = 64 / SEG;  // lines per wavefront
  static constexpr int WPB = 2;         // wavefronts per workgroup: adjacent lines share 128-byte memory lines
};

// What lane c loads of a line's level kz for its node (ij, c): the metric
// and, for the bottom (f = 0) and top (f = 1) face, Lift, Fscale, the damping
// coefficients of both sides and nz.
struct LineNode {
  double G, GH, Lift[2], Fs[2], am[2], ap[2], nz[2];
};
// em: EMap3Dto2D of the level's element, loaded a level earlier
template <int N>
__device__ __forceinline__ void load_node(const HeviArgs& a, int ke2D, int ij, int kz, int pv, int em, bool with_nz,
                                          LineNode& L) {
  constexpr int Nfp = N * N, Np = N * N * N;
  const DevMesh& m = a.m;
  const int NeZ = a.NeZ, ke = ke2D + kz * m.Ne2D;
  L.G = ldg(m.Gsqrt, (uint32_t)(Np * ke + ij + Nfp * pv));
  L.GH = ldg(m.GsqrtH, (uint32_t)(ij + Nfp * em));
#pragma unroll
  for (int f = 0; f < 2; ++f) {
    const bool bc = f == 0 ? kz == 0 : kz == NeZ - 1;
    const int ke2 = bc ? ke : (f == 0 ? ke - m.Ne2D : ke + m.Ne2D), f2 = bc ? f : 1 - f;
    const uint32_t gfp = (uint32_t)((4 + f) * Nfp + ij) + (uint32_t)(6 * Nfp) * ke;
    L.Lift[f] = ldg(m.Lift, (uint32_t)(ij + Nfp * pv + (4 + f) * Np));
    L.Fs[f] = ldg(m.Fscale, gfp);
    L.am[f] = ldg(a.alph, (uint32_t)(f * Nfp + ij) + (uint32_t)(2 * Nfp) * ke);
    L.ap[f] = ldg(a.alph, (uint32_t)(f2 * Nfp + ij) + (uint32_t)(2 * Nfp) * ke2);
    L.nz[f] = with_nz ? ldg(m.nz, gfp) : 0.0;
  }
}
// A copy of x the compiler knows nothing about: what is derived from it is
// formed where it is used, not kept in registers (or spilled) across the LU.
__device__ __forceinline__ int opaque(int x) {
  asm volatile("" : "+v"(x));
  return x;
}
// t1 = 0.5 impl_fac / GsqrtV Lift Fscale alph, t2 = ... nz of face f; both
// doubled at a closed boundary (the form the boundary terms take)
__device__ __forceinline__ double2 face_terms(const HeviArgs& a, const LineNode& L, int f, int kz) {
  const bool bc = f == 0 ? kz == 0 : kz == a.NeZ - 1;
  const double fac = 0.5 * a.impl_fac / (L.G / L.GH) * L.Lift[f] * L.Fs[f];
  double2 t{fac * (L.am[f] > L.ap[f] ? L.am[f] : L.ap[f]), fac * L.nz[f]};
  if (bc) {
    t.x = 2.0 * t.x;
    t.y = 2.0 * t.y;
  }
  return t;
}

// ---------------------------------------------------------------------------
// 2. construct_matbnd_uv (:905-1011) + solve_uv (:589-689)
template <int N1>
__global__ void __launch_bounds__(64 * LineSeg<N1>::WPB) hevi_solve_uv_kernel(const HeviArgs a) {
  constexpr int N = N1, Nfp = N1 * N1, Np = N1 * N1 * N1;
  constexpr int SEG = LineSeg<N1>::SEG, LPW = LineSeg<N1>::LPW, WPB = LineSeg<N1>::WPB;
  __shared__ double sT[WPB][LPW][2][SEG];  // face terms of the rows
  __shared__ double sB[WPB][LPW][2][SEG];  // right-hand sides
  __shared__ double sG[WPB][LPW][4];       // top-node solution of the level below
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63, sg = lane / SEG, c = lane % SEG;
  const DevMesh& m = a.m;
  const int nline = m.Ne2D * Nfp, ngroup = (nline + LPW - 1) / LPW;
  const int NeZ = a.NeZ;
  const uint32_t nn = (uint32_t)Np * m.Ne;
  const int slot = blockIdx.x * WPB + w;
  double* scr = a.lines + (size_t)slot * NeZ * N * (4 * LPW);  // [level][row][line][b1, b2, G, -]
  const int pv = c < N ? c : N - 1;
  double(*T)[SEG] = sT[w][sg];
  double(*Bs)[SEG] = sB[w][sg];
  double* G = sG[w][sg];
  for (int g = slot; g < ngroup; g += gridDim.x * WPB) {
    const bool lv = g * LPW + sg < nline;
    const int line = lv ? g * LPW + sg : nline - 1;
    const int ke2D = line / Nfp, ij = line % Nfp;
    double B[N];
    LineNode L;
    double b0, b1;
    int em = m.EMap3Dto2D[ke2D];
    auto load = [&](int kz) __attribute__((always_inline)) {
      const uint32_t q = (uint32_t)Np * (ke2D + kz * m.Ne2D) + ij + Nfp * pv;
      load_node<N>(a, ke2D, ij, kz, pv, em, false, L);
      em = m.EMap3Dto2D[ke2D + (kz + 1 < NeZ ? kz + 1 : kz) * m.Ne2D];
      b0 = ldg(a.buv, q);
      b1 = ldg(a.buv, q + nn);
    };
    load(0);
    __builtin_amdgcn_s_waitcnt(0x0F70);  // as in the var3 solve below
    for (int kz = 0; kz < NeZ; ++kz) {
      T[0][c] = face_terms(a, L, 0, kz).x;
      T[1][c] = face_terms(a, L, 1, kz).x;
      Bs[0][c] = b0;
      Bs[1][c] = b1;
      if (kz > 0 && c < 3) G[c] = B[N - 1];
      wave_sync();
      double A[1][N];
#pragma unroll
      for (int i = 0; i < N; ++i) A[0][i] = (i == c) ? 1.0 : 0.0;
      if (c == 0 && kz > 0) {
        const double g2 = G[2];
#pragma unroll
        for (int i = 0; i < N; ++i) A[0][i] = A[0][i] + T[0][i];
#pragma unroll
        for (int i = 0; i < N; ++i) A[0][i] = A[0][i] - (-T[0][i]) * g2;
      }
      if (c == N - 1 && kz < NeZ - 1) {
#pragma unroll
        for (int i = 0; i < N; ++i) A[0][i] = A[0][i] + T[1][i];
      }
#pragma unroll
      for (int i = 0; i < N; ++i) B[i] = 0.0;
      if (c < 2) {
#pragma unroll
        for (int i = 0; i < N; ++i) B[i] = Bs[c][i];
        if (kz > 0) {
          const double gb = G[c];
#pragma unroll
          for (int i = 0; i < N; ++i) B[i] = B[i] - (-T[0][i]) * gb;
        }
      } else if (c == 2 && kz < NeZ - 1) {
#pragma unroll
        for (int i = 0; i < N; ++i) B[i] = -T[1][i];
      }
      wave_sync();
      (void)lu_solve_cols<1, N, SEG, true>(A, B, c, [&]() __attribute__((always_inline)) {
        load(kz + 1 < NeZ ? kz + 1 : kz);
      });
      if (c < 4) {
        double* x = scr + (size_t)kz * N * (4 * LPW) + sg * 4 + c;
#pragma unroll
        for (int i = 0; i < N; ++i) x[i * (4 * LPW)] = B[i];
      }
    }
    wave_sync();
    // block back substitution: lane c takes node c
    double u = 0.0, v = 0.0, x[3], y[2];
    auto back = [&](int kz) __attribute__((always_inline)) {  // loads of a level, issued one level ahead
      const double* xk = scr + (size_t)kz * N * (4 * LPW) + (size_t)pv * (4 * LPW) + sg * 4;
      const uint32_t q = (uint32_t)Np * (ke2D + kz * m.Ne2D) + ij + Nfp * pv;
#pragma unroll
      for (int r = 0; r < 3; ++r) x[r] = xk[r];
      y[0] = ldg(a.pin[VU], q);
      y[1] = ldg(a.pin[VV], q);
    };
    back(NeZ - 1);
    for (int kz = NeZ - 1; kz >= 0; --kz) {
      const double u0 = bcast<SEG, 0>(u), v0 = bcast<SEG, 0>(v);
      u = x[0];
      v = x[1];
      const double tmp = x[2], yu = y[0], yv = y[1];
      if (kz > 0) back(kz - 1);
      if (kz < NeZ - 1) {
        u = u - tmp * u0;
        v = v - tmp * v0;
      }
      if (lv && c < N) {
        const uint32_t q = (uint32_t)Np * (ke2D + kz * m.Ne2D) + ij + Nfp * pv;
        stg(a.pv[VU], q, yu + u);
        stg(a.pv[VV], q, yv + v);
      }
    }
    wave_sync();
  }
}

// ---------------------------------------------------------------------------
// 4. construct_matbnd (:693-901) + solve (:329-479).
// Unknowns of an element: (var, pv), var fastest: DENS, MOMZ, RHOT.
// A level is assembled in two steps: lane c forms, for the rows of node c,
// the columns of node 0 (the ones the level below couples to), the
// right-hand side and the coupling to the level above, and passes them
// through LDS to the lanes that hold those columns; every lane forms the
// other columns of its own node from the rows' metric factors.
// MODE: SOLVE_ALL, every line with row exchanges; SOLVE_DIAGONAL, which gives
// the groups of lines whose pivots leave the diagonal up to the list a.flagged
// (count, then group numbers), and SOLVE_FLAGGED, which solves those.  The
// exchanges' branches make the allocator spill at p = 6 (5 registers) and p = 7
// (24), none below.  Drop-in stage, pivots on the diagonal / off it in every
// block, SOLVE_ALL against the other two:
//   p = 5, 64 x 32 x 8 elements 1066 / 1260 against 1055 / 1366 us; 8 x 4 x 4
//   85 / 99 against 86 / 114 us;
//   p = 6, 64 x 32 x 8 1799 / 2058 against 1766 / 2270 us; 8 x 4 x 4 101 / 121
//   against 99 / 139 us;
//   p = 7, 64 x 32 x 8 2552 / 2980 against 2413 / 3306 us; 16 x 8 x 8 (a group per
//   SIMD) 287 / 346 against 284 / 378 us; 8 x 4 x 4 113 / 140 against 112 / 166 us.
// So SOLVE_ALL below p = 7, and there on meshes of no more groups than SIMDs,
// where the spills hide behind the latency; beyond, the usual steps, whose
// pivots stay on the diagonal, decide.
enum { SOLVE_ALL = 0, SOLVE_DIAGONAL = 1, SOLVE_FLAGGED = 2 };
template <int N1>
struct LineLds {
  static constexpr int SEG = LineSeg<N1>::SEG, NR = 3 * SEG;  // rows the segment's lanes form (3 N1 of them used)
  double E[SEG];     // E33 / GsqrtV of the rows
  double2 T[SEG];    // face terms (t1, t2) of the rows, top face
  double C[3][NR];   // columns of node 0
  double B[4][NR];   // right-hand sides: b, G1, G2, G3
  double G[4][3];    // their top-node solutions at the level below
};
template <int N1, int MODE>
__global__ void __launch_bounds__(64 * LineSeg<N1>::WPB) __attribute__((amdgpu_waves_per_eu(2)))
hevi_solve3_kernel(const HeviArgs a) {
  constexpr int N = N1, Nfp = N1 * N1, Np = N1 * N1 * N1, n3 = 3 * N1;
  constexpr int SEG = LineSeg<N1>::SEG, LPW = LineSeg<N1>::LPW, WPB = LineSeg<N1>::WPB;
  __shared__ double sD[N][N], sI[N][N];  // impl_fac D1D and impl_fac GRAV IntrpMat, by [column node][row node]
  __shared__ LineLds<N1> sL[WPB * LPW];
  const DevMesh& m = a.m;
  const int nline = m.Ne2D * Nfp;
  const int ngroup = MODE == SOLVE_FLAGGED ? a.flagged[0] : (nline + LPW - 1) / LPW;
  if (MODE == SOLVE_FLAGGED && ngroup == 0) return;
  const int NeZ = a.NeZ;
  const uint32_t nn = (uint32_t)Np * m.Ne;
  const double impl_fac = a.impl_fac;
  for (int e = threadIdx.x; e < N * N; e += 64 * WPB) {
    sD[e / N][e % N] = impl_fac * m.D1D[e];
    sI[e % N][e / N] = impl_fac * a.c.GRAV * m.Itr[e];
  }
  __syncthreads();
  const int slot = blockIdx.x * WPB + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  double* scr = a.lines + (size_t)slot * NeZ * n3 * (4 * LPW);  // [level][row][line][b, G1, G2, G3]
  const int c0 = threadIdx.x % SEG;
  for (int u = slot; u < ngroup; u += gridDim.x * WPB) {
    const int g = MODE == SOLVE_FLAGGED ? __builtin_amdgcn_readfirstlane(a.flagged[1 + u]) : u;
    double B[n3];
    bool off = false;
    // the level's data, loaded during the level before
    LineNode L;
    double b[3], cf[3], up[3], E33;  // rhs, POT / WT / DPDRHOT of the node and of the bottom node above
    double dn[3] = {0.0, 0.0, 0.0};  // and of the top node below
    int em;
    // this lane's line (lanes beyond the last one work on it and store nothing)
    auto line_of = [&](int tid) __attribute__((always_inline)) {
      const int line = g * LPW + (tid & 63) / SEG;
      return line < nline ? line : nline - 1;
    };
    auto load = [&](int kz, bool first) __attribute__((always_inline)) {
      const int tid = opaque(threadIdx.x), c = tid % SEG, pv = c < N ? c : N - 1;
      const int line = line_of(tid), ke2D = line / Nfp, ij = line % Nfp, ke = ke2D + kz * m.Ne2D;
      const uint32_t q = (uint32_t)(Np * ke + ij + Nfp * pv);
      const uint32_t qu = kz < NeZ - 1 ? (uint32_t)(Np * (ke + m.Ne2D) + ij) : q;
      if (first) em = m.EMap3Dto2D[ke];
      load_node<N>(a, ke2D, ij, kz, pv, em, true, L);
      em = m.EMap3Dto2D[kz < NeZ - 1 ? ke + m.Ne2D : ke];
      E33 = ldg(m.E33, q);
#pragma unroll
      for (int v = 0; v < 3; ++v) {
        b[v] = ldg(a.b3 + (size_t)v * nn, q);
        cf[v] = ldg(a.coef + (size_t)v * nn, q);
        up[v] = ldg(a.coef + (size_t)v * nn, qu);
      }
    };
    load(0, true);
    // vmcnt(0): the first level waits here, so that the wait at the top of a
    // later level (loads, then the stores of the level's solutions) need not
    // cover those stores
    __builtin_amdgcn_s_waitcnt(0x0F70);
    for (int kz = 0; kz < NeZ; ++kz) {
      const bool bc1 = kz == 0, bc2 = kz == NeZ - 1;
      const int tid = opaque(threadIdx.x), c = tid % SEG, pv = c < N ? c : N - 1;
      LineLds<N1>& S = sL[tid / SEG];
      const double POT = cf[0], WT = cf[1], DPD = cf[2];
      if (!bc1 && c < 4) {
#pragma unroll
        for (int v = 0; v < 3; ++v) S.G[c][v] = B[n3 - 3 + v];
      }
      wave_sync();
      {
        const double Eg = E33 / (L.G / L.GH);
        S.E[c] = Eg;
        // rows of node c, columns of node 0
        const double P0 = bcast<SEG, 0>(POT), W0 = bcast<SEG, 0>(WT), D0 = bcast<SEG, 0>(DPD);
        const double Id = (c == 0) ? 1.0 : 0.0;
        const double fdz = Eg * sD[0][pv];
        const double2 t = face_terms(a, L, 0, kz);
        double d[3][3] = {{Id, fdz, 0.0}, {sI[0][pv], Id, fdz * D0}, {-fdz * P0 * W0, fdz * P0, Id + fdz * W0}};
        d[0][1] = d[0][1] - t.y;
        d[1][1] = d[1][1] + t.x;
        d[2][0] = d[2][0] + t.y * P0 * W0;
        d[2][1] = d[2][1] - t.y * P0;
        if (!bc1) {
          d[0][0] = d[0][0] + t.x;
          d[1][2] = d[1][2] - t.y * D0;
          d[2][2] = d[2][2] + t.x;
        }
        d[2][2] = d[2][2] - t.y * W0;
        // L: coupling to the top node of the level below, eliminated with its solution
        if (!bc1) {
#pragma unroll
          for (int v = 0; v < 3; ++v) {
            const double l0 = (v == 0) ? -t.x : (v == 1 ? 0.0 : -t.y * dn[0] * dn[1]);
            const double l1 = (v == 0) ? +t.y : (v == 1 ? -t.x : +t.y * dn[0]);
            const double l2 = (v == 0) ? 0.0 : (v == 1 ? +t.y * dn[2] : -t.x + t.y * dn[1]);
#pragma unroll
            for (int s = 0; s < 3; ++s) d[v][s] = d[v][s] - l0 * S.G[1 + s][0] - l1 * S.G[1 + s][1] - l2 * S.G[1 + s][2];
            b[v] = b[v] - l0 * S.G[0][0] - l1 * S.G[0][1] - l2 * S.G[0][2];
          }
        }
        // U: coupling to the bottom node of the level above, the G columns (none at the top level)
        const double2 tu = face_terms(a, L, 1, kz);
        S.T[c] = tu;
        const double gc[3][3] = {{-tu.x, tu.y, 0.0},
                                 {0.0, -tu.x, tu.y * up[2]},
                                 {-tu.y * up[0] * up[1], tu.y * up[0], -tu.x + tu.y * up[1]}};
#pragma unroll
        for (int v = 0; v < 3; ++v) {
          S.B[0][3 * c + v] = b[v];
#pragma unroll
          for (int s = 0; s < 3; ++s) {
            S.C[s][3 * c + v] = d[v][s];
            S.B[1 + s][3 * c + v] = bc2 ? 0.0 : gc[v][s];
          }
        }
#pragma unroll
        for (int v = 0; v < 3; ++v) dn[v] = bcast<SEG, N - 1>(cf[v]);
      }
      wave_sync();
      // the other columns
      double A[3][n3];
#pragma unroll
      for (int i = 0; i < N; ++i) {
        const double Id = (i == c) ? 1.0 : 0.0;
        const double fdz = S.E[i] * sD[pv][i];
        A[0][3 * i] = Id;
        A[1][3 * i] = fdz;
        A[2][3 * i] = 0.0;
        A[0][3 * i + 1] = sI[pv][i];
        A[1][3 * i + 1] = Id;
        A[2][3 * i + 1] = fdz * DPD;
        A[0][3 * i + 2] = -fdz * POT * WT;
        A[1][3 * i + 2] = fdz * POT;
        A[2][3 * i + 2] = Id + fdz * WT;
      }
      // top-face terms on the columns of the last node
      if (c == N - 1) {
#pragma unroll
        for (int i = 0; i < N; ++i) {
          const double2 t = S.T[i];
          A[1][3 * i] = A[1][3 * i] - t.y;
          A[1][3 * i + 1] = A[1][3 * i + 1] + t.x;
          A[0][3 * i + 2] = A[0][3 * i + 2] + t.y * POT * WT;
          A[1][3 * i + 2] = A[1][3 * i + 2] - t.y * POT;
          if (!bc2) {
            A[0][3 * i] = A[0][3 * i] + t.x;
            A[2][3 * i + 1] = A[2][3 * i + 1] - t.y * DPD;
            A[2][3 * i + 2] = A[2][3 * i + 2] + t.x;
          }
          A[2][3 * i + 2] = A[2][3 * i + 2] - t.y * WT;
        }
      }
      if (c == 0) {
#pragma unroll
        for (int i = 0; i < n3; ++i) {
#pragma unroll
          for (int s = 0; s < 3; ++s) A[s][i] = S.C[s][i];
        }
      }
      {
        const double* Bc = S.B[c < 4 ? c : 0];  // lanes beyond the right-hand sides carry a copy nobody reads
#pragma unroll
        for (int i = 0; i < n3; ++i) B[i] = Bc[i];
      }
      wave_sync();
      if (!lu_solve_cols<3, N, SEG, MODE != SOLVE_DIAGONAL>(
              A, B, c0, [&]() __attribute__((always_inline)) { load(bc2 ? kz : kz + 1, false); })) {
        off = true;
        break;
      }
      {
        const int t2 = opaque(threadIdx.x), c2 = t2 % SEG;
        if (c2 < 4) {
          double* x = scr + (size_t)kz * n3 * (4 * LPW);
          const uint32_t o = (uint32_t)((t2 & 63) / SEG * 4 + c2);
#pragma unroll
          for (int i = 0; i < n3; ++i) stg(x, o + i * (4 * LPW), B[i]);
        }
      }
    }
    if (MODE == SOLVE_DIAGONAL && off) {
      if ((threadIdx.x & 63) == 0) a.flagged[1 + atomicAdd(a.flagged, 1)] = g;
      continue;
    }
    wave_sync();
    // block back substitution: lane c takes node c
    const int tid = opaque(threadIdx.x), c = tid % SEG, pv = c < N ? c : N - 1;
    const bool lv = g * LPW + (tid & 63) / SEG < nline;
    const int line = line_of(tid), ke2D = line / Nfp, ij = line % Nfp;
    double y[3] = {0.0, 0.0, 0.0}, x[3][4], p0[3], s[3] = {0.0, 0.0, 0.0};
    auto back = [&](int kz) __attribute__((always_inline)) {  // loads of a level, issued one level ahead
      const double* xk = scr + (size_t)kz * n3 * (4 * LPW);
      const uint32_t o = (uint32_t)(3 * pv * (4 * LPW) + (tid & 63) / SEG * 4);
      const uint32_t q = (uint32_t)(Np * (ke2D + kz * m.Ne2D) + ij + Nfp * pv);
#pragma unroll
      for (int v = 0; v < 3; ++v)
#pragma unroll
        for (int r = 0; r < 4; ++r) x[v][r] = ldg(xk, o + v * (4 * LPW) + r);
      p0[0] = ldg(a.pin[VD], q);
      p0[1] = ldg(a.pin[VW], q);
      p0[2] = ldg(a.pin[VT], q);
      if (a.finish) {
        s[0] = ldg_nt(a.qs[VD], q);
        s[1] = ldg_nt(a.qs[VW], q);
        s[2] = ldg_nt(a.qs[VT], q);
      }
    };
    back(NeZ - 1);
    for (int kz = NeZ - 1; kz >= 0; --kz) {
      double y0[3], z[3][4], o[3];
      const double sD = s[0], sW = s[1], sT = s[2];
#pragma unroll
      for (int v = 0; v < 3; ++v) {
        y0[v] = bcast<SEG, 0>(y[v]);
        o[v] = p0[v];
#pragma unroll
        for (int r = 0; r < 4; ++r) z[v][r] = x[v][r];
      }
      if (kz > 0) back(kz - 1);
#pragma unroll
      for (int v = 0; v < 3; ++v) {
        y[v] = z[v][0];
        if (kz < NeZ - 1) y[v] = y[v] - z[v][1] * y0[0] - z[v][2] * y0[1] - z[v][3] * y0[2];
      }
      if (lv && c < N) {
        const uint32_t q = (uint32_t)(Np * (ke2D + kz * m.Ne2D) + ij + Nfp * pv);
        if (a.finish) {
          finish_node(a, VD, q, o[0] + y[0], sD);
          finish_node(a, VW, q, o[1] + y[1], sW);
          finish_node(a, VT, q, o[2] + y[2], sT);
        } else {
          stg(a.pv[VD], q, o[0] + y[0]);
          stg(a.pv[VW], q, o[1] + y[1]);
          stg(a.pv[VT], q, o[2] + y[2]);
        }
      }
    }
    wave_sync();
  }
}

// tendency = (iterate - q*) / impl_fac (..._rhot_hevi.F90:937-947) of nv
// variables and, as finish says, the stepper's StoreImplicit on the node: var0
// and varTmp (first stage) take q, and q = q + impl_fac T (streamed:
// non-temporal loads and stores).
struct TendStore {
  int nv;
  double* T[5];
  const double* p[5];
  const double* qs[5];
  double* q[5];
  double* var0[5];
  double* varTmp[5];
  double impl_fac;
  int finish;
};
__global__ void hevi_tend_store_kernel(const TendStore a, long n) {
  const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n) return;
#pragma unroll
  for (int v = 0; v < 5; ++v) {
    if (v >= a.nv) break;
    const double q = __builtin_nontemporal_load(a.qs[v] + t);
    const double T = (__builtin_nontemporal_load(a.p[v] + t) - q) / a.impl_fac;
    __builtin_nontemporal_store(T, a.T[v] + t);
    if (a.finish == FINISH_TEND) continue;
    if (a.finish == FINISH_STORE_COPY) {
      __builtin_nontemporal_store(q, a.var0[v] + t);
      __builtin_nontemporal_store(q, a.varTmp[v] + t);
    }
    __builtin_nontemporal_store(q + a.impl_fac * T, a.q[v] + t);
  }
}

// sums of squares of the vectors x[blockIdx.y] of n[blockIdx.y] entries, 256
// per-block partial sums each (residual norms), straight into host memory
// where the workspace has it
struct SumsqArgs {
  const double* x[5];
  long n[5];
  double* partial;
};
__global__ void sumsq_kernel(const SumsqArgs a) {
  __shared__ double s[256];
  const double* const x = a.x[blockIdx.y];
  const long n = a.n[blockIdx.y];
  double* const partial = a.partial + 256 * blockIdx.y;
  double acc = 0.0;
  for (long t = (long)blockIdx.x * blockDim.x + threadIdx.x; t < n; t += (long)gridDim.x * blockDim.x)
    acc += x[t] * x[t];
  s[threadIdx.x] = acc;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) s[threadIdx.x] += s[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) partial[blockIdx.x] = s[0];
}

// ---------------------------------------------------------------------------
// Learned initial iterate: features, targets, application, per-line residual
// and fallback.  One workgroup per line, one thread per node of the line
// (L = NeZ*N1 threads); node t of a line is (kz = t / N1, pv = t % N1).
struct LineArgs {
  const double* qs[5];
  const double* q0[5];
  const double* Tex[5];
  double* pv[5];
  double inv_s[5];      // 1 / state scale
  double inv_t[5];      // 1 / tendency-feature scale
  double inv_d[5], d[5];  // increment scale
  double impl_fac, dt;
  int Np, Nfp, Ne2D, N1, L, nlines;
  long line0, stride;
};

__device__ __forceinline__ uint32_t line_node(const LineArgs& a, long line, int t) {
  const int ke2D = (int)(line / a.Nfp), ij = (int)(line % a.Nfp);
  const int kz = t / a.N1, pv = t % a.N1;
  return (uint32_t)a.Np * (ke2D + kz * a.Ne2D) + ij + a.Nfp * pv;
}

__global__ void line_features_kernel(const LineArgs a, float* X, int n_in, float* Y, int n_out) {
  const int row = blockIdx.x, t = threadIdx.x;
  const long line = (a.line0 + (long)row * a.stride) % a.nlines;
  const uint32_t n = line_node(a, line, t);
  float* x = X + (size_t)row * n_in;
#pragma unroll
  for (int v = 0; v < 5; ++v) {
    const double qs = ldg(a.qs[v], n);
    x[v * a.L + t] = (float)(qs * a.inv_s[v]);
    const double te = a.Tex[v] ? ldg(a.Tex[v], n) : 0.0;
    x[(5 + v) * a.L + t] = (float)(a.impl_fac * te * a.inv_t[v]);
    if (Y) Y[(size_t)row * n_out + v * a.L + t] = (float)((ldg(a.pv[v], n) - qs) * a.inv_d[v]);
  }
  if (t == 0) x[10 * a.L] = (float)(a.impl_fac / a.dt);
}

__global__ void line_apply_kernel(const LineArgs a, const float* Y, int n_out) {
  const int row = blockIdx.x, t = threadIdx.x;
  const long line = (a.line0 + (long)row * a.stride) % a.nlines;
  const uint32_t n = line_node(a, line, t);
#pragma unroll
  for (int v = 0; v < 5; ++v)
    stg(a.pv[v], n, ldg(a.qs[v], n) + a.d[v] * (double)Y[(size_t)row * n_out + v * a.L + t]);
}

// residual norm^2 of every line from the uv and var3 right-hand sides
__global__ void line_resid_kernel(const LineArgs a, const double* buv, const double* b3, long nn, double* r) {
  __shared__ double sh[512];
  const long line = blockIdx.x;
  const int t = threadIdx.x;
  const uint32_t n = line_node(a, line, t);
  double acc = 0.0;
  for (int c = 0; c < 2; ++c) {
    const double x = ldg(buv, n + (uint32_t)(c * nn));
    acc += x * x;
  }
  for (int c = 0; c < 3; ++c) {
    const double x = ldg(b3, n + (uint32_t)(c * nn));
    acc += x * x;
  }
  sh[t] = acc;
  __syncthreads();
  for (int w = 256; w > 0; w >>= 1) {
    if (t < w && t + w < a.L) sh[t] += sh[t + w];
    __syncthreads();
  }
  if (t == 0) r[line] = sh[0];
}

// lines whose predicted iterate has the larger residual restart from q^n;
// r_guess becomes the residual of the start the line keeps
__global__ void line_select_kernel(const LineArgs a, double* r_guess, const double* r_plain, double* flag) {
  const long line = blockIdx.x;
  const int t = threadIdx.x;
  const double rg = r_guess[line], rp = r_plain[line];
  const bool fb = !(rg <= rp);
  if (fb) {
    const uint32_t n = line_node(a, line, t);
#pragma unroll
    for (int v = 0; v < 5; ++v) stg(a.pv[v], n, ldg(a.q0[v], n));
  }
  __syncthreads();  // every thread has read r_guess[line]
  if (t == 0) {
    flag[line] = fb ? 1.0 : 0.0;
    r_guess[line] = fb ? rp : rg;
  }
}

__global__ void sum_kernel(const double* x, long n, double* partial) {
  __shared__ double s[256];
  double acc = 0.0;
  for (long t = (long)blockIdx.x * blockDim.x + threadIdx.x; t < n; t += (long)gridDim.x * blockDim.x) acc += x[t];
  s[threadIdx.x] = acc;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) s[threadIdx.x] += s[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) partial[blockIdx.x] = s[0];
}

// waits for the partial sums of nvec vectors; they are then in partial_h
int wait_partials(fedg_ctx* ctx, const double* partial, double* partial_h, int nvec) {
  if (partial_h != partial)
    FEDG_HIP_CHECK(hipMemcpyAsync(partial_h, partial, nvec * 256 * sizeof(double), hipMemcpyDeviceToHost, ctx->stream));
  FEDG_HIP_CHECK(hipStreamSynchronize(ctx->stream));
  return FEDG_OK;
}

int host_sum(fedg_ctx* ctx, const double* x, long n, double* partial, double* partial_h, double* out) {
  hipLaunchKernelGGL(sum_kernel, dim3(256), dim3(256), 0, ctx->stream, x, n, partial);
  FEDG_HIP_CHECK(hipGetLastError());
  const int rc = wait_partials(ctx, partial, partial_h, 1);
  if (rc != FEDG_OK) return rc;
  double s = 0.0;
  for (int b = 0; b < 256; ++b) s += partial_h[b];
  *out = s;
  return FEDG_OK;
}

LineArgs line_args(const DevMesh& m, const HeviArgs& a, const double* const Tex[5], const double scale[15], double dt) {
  LineArgs l{};
  for (int v = 0; v < 5; ++v) {
    l.qs[v] = a.qs[v];
    l.q0[v] = a.q0[v];
    l.Tex[v] = Tex ? Tex[v] : nullptr;
    l.pv[v] = a.pv[v];
    l.inv_s[v] = 1.0 / scale[v];
    l.inv_t[v] = 1.0 / scale[5 + v];
    l.d[v] = scale[10 + v];
    l.inv_d[v] = 1.0 / scale[10 + v];
  }
  l.impl_fac = a.impl_fac;
  l.dt = dt;
  l.Np = m.Np;
  l.Nfp = m.Nfp;
  l.Ne2D = m.Ne2D;
  l.N1 = m.n1;
  l.L = a.NeZ * m.n1;
  l.nlines = m.Ne2D * m.Nfp;
  l.line0 = 0;
  l.stride = 1;
  return l;
}

template <int N1, bool FLAT>
__global__ void __launch_bounds__(N1* N1* N1) hevi_rhs_uv_kernel(const HeviArgs a) {
  hevi_rhs_uv_body<N1, FLAT>(a);
}
template <int N1, bool FLAT>
__global__ void __launch_bounds__(N1* N1* N1) hevi_rhs3_kernel(const HeviArgs a) {
  hevi_rhs3_body<N1, FLAT>(a);
}
// p = 7 on the flat box at no more than 128 VGPRs, so that two 512-thread
// workgroups share a CU (the kernels held 135-143 VGPRs when every node formed
// the hydrostatic RHOT with two pows; with it loaded, 70-72)
__global__ void __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(4)))
hevi_rhs_uv8_flat_kernel(const HeviArgs a) {
  hevi_rhs_uv_body<8, true>(a);
}
__global__ void __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(4)))
hevi_rhs38_flat_kernel(const HeviArgs a) {
  hevi_rhs3_body<8, true>(a);
}

// the residual kernels, on the flat box without the metric loads
template <int N1>
void launch_rhs_uv(fedg_ctx* ctx, const HeviArgs& a) {
  const DevMesh& m = ctx->m;
  if (N1 == 8 && m.flat && m.lift_tensor)
    hipLaunchKernelGGL(hevi_rhs_uv8_flat_kernel, dim3(m.Ne), dim3(512), 0, ctx->stream, a);
  else if (m.flat && m.lift_tensor)
    hipLaunchKernelGGL((hevi_rhs_uv_kernel<N1, true>), dim3(m.Ne), dim3(N1 * N1 * N1), 0, ctx->stream, a);
  else
    hipLaunchKernelGGL((hevi_rhs_uv_kernel<N1, false>), dim3(m.Ne), dim3(N1 * N1 * N1), 0, ctx->stream, a);
}
template <int N1>
void launch_rhs3(fedg_ctx* ctx, const HeviArgs& a) {
  const DevMesh& m = ctx->m;
  if (N1 == 8 && m.flat && m.lift_tensor)
    hipLaunchKernelGGL(hevi_rhs38_flat_kernel, dim3(m.Ne), dim3(512), 0, ctx->stream, a);
  else if (m.flat && m.lift_tensor)
    hipLaunchKernelGGL((hevi_rhs3_kernel<N1, true>), dim3(m.Ne), dim3(N1 * N1 * N1), 0, ctx->stream, a);
  else
    hipLaunchKernelGGL((hevi_rhs3_kernel<N1, false>), dim3(m.Ne), dim3(N1 * N1 * N1), 0, ctx->stream, a);
}

// Tallest column taken, in elements, by N1.  The kernels set no limit of their
// own (a wavefront's scratch grows with NeZ); these are the limits the entry
// points have always had, and what the no-allocation entry's fixed scratch is
// sized for.
constexpr int kMaxNeZ[9] = {0, 0, 40, 53, 39, 30, 52, 43, 37};

// finish: what the solve of DENS, MOMZ and RHOT of the last iteration stores,
// where that iteration is known beforehand (no tolerance, no residual asked
// for); FINISH_NONE is left in a.finish where it stored the iterate instead
template <int N1>
int run_newton(fedg_ctx* ctx, HeviArgs& a, HeviWork* w, int max_it, double rtol, double* resid, int* it_done,
               double r0_ext, int finish) {
  const DevMesh& m = ctx->m;
  double* const partial = w->partial;
  double* const partial_h = w->partial_h;
  if (a.NeZ > kMaxNeZ[N1]) {
    set_error("HEVI: too many elements in the vertical for the line solve (NeZ)");
    return FEDG_ERR_UNSUPPORTED;
  }
  // wavefronts of the line solves: as many as the scratch holds, walking the
  // groups of lines from their own slot of it
  constexpr int WPB = LineSeg<N1>::WPB;
  const long ngroup = ((long)m.Ne2D * N1 * N1 + LineSeg<N1>::LPW - 1) / LineSeg<N1>::LPW;
  const size_t list = line_list_doubles(ngroup);
  const long nwave =
      w->lines_n <= list ? 0
                         : std::min((ngroup + WPB - 1) / WPB * WPB,
                                    (long)((w->lines_n - list) / line_scratch_per_wave(N1, a.NeZ)) / WPB * WPB);
  if (nwave < WPB || !w->lines) {
    set_error("HEVI: the line solve's scratch holds no column of this mesh");
    return FEDG_ERR_UNSUPPORTED;
  }
  const dim3 gline((unsigned)(nwave / WPB)), bline(64 * WPB);
  // usually nothing is flagged: no more workgroups than are resident
  const dim3 gflag((unsigned)std::min(nwave / WPB, (long)4 * ctx->ncu));
  a.flagged = reinterpret_cast<int*>(w->lines);
  a.lines = w->lines + list;
  const long n = (long)m.Np * m.Ne;
  // r0_ext > 0: the residual norm at q^n, the reference of the tolerance when
  // the iteration starts from a predicted iterate (which may already meet it)
  double r0 = r0_ext;
  // rounding floor of the residual: G = impl_fac T - q + q* cancels terms of
  // the size of the state, so ||G|| cannot drop much below eps ||q*||; the
  // iteration also stops at 4 eps ||q*||, and once an update has not halved
  // the residual (it has reached its floor)
  // The norms of an iteration are one launch and one wait: partial holds the
  // sums of MOMX and MOMY's residual, of the other three's, then (of the first
  // iteration) of the five variables of the stage state.  12 x 6 x 6 elements
  // at p = 3, five steps to 1e-10: 7.45 -> 3.74 ms (with the stage's exchange in one launch).
  double atol = 0.0;
  if (rtol > 0.0) {
    SumsqArgs q{};
    for (int v = 0; v < 5; ++v) {
      q.x[v] = a.qs[v];
      q.n[v] = n;
    }
    q.partial = partial + 2 * 256;
    hipLaunchKernelGGL(sumsq_kernel, dim3(256, 5), dim3(256), 0, ctx->stream, q);
    FEDG_HIP_CHECK(hipGetLastError());
  }
  double r_prev = 0.0;
  int it = 0;
  const bool track = rtol > 0.0 || resid != nullptr;
  for (; it < max_it; ++it) {
    a.finish = !track && it == max_it - 1 ? finish : FINISH_NONE;
    launch_rhs_uv<N1>(ctx, a);
    FEDG_HIP_CHECK(hipGetLastError());
    a.alph_ready = 1;  // the damping coefficients depend on q0 alone
    hipLaunchKernelGGL(hevi_solve_uv_kernel<N1>, gline, bline, 0, ctx->stream, a);
    FEDG_HIP_CHECK(hipGetLastError());
    a.pin[VU] = a.pv[VU];
    a.pin[VV] = a.pv[VV];
    launch_rhs3<N1>(ctx, a);
    FEDG_HIP_CHECK(hipGetLastError());
    if (track) {
      SumsqArgs res{{a.buv, a.b3}, {2 * n, 3 * n}, partial};
      hipLaunchKernelGGL(sumsq_kernel, dim3(256, 2), dim3(256), 0, ctx->stream, res);
      FEDG_HIP_CHECK(hipGetLastError());
      const bool first = it == 0 && rtol > 0.0;
      const int rc = wait_partials(ctx, partial, partial_h, first ? kHeviPartials : 2);
      if (rc != FEDG_OK) return rc;
      double r2 = 0.0;
      for (int b = 0; b < 2 * 256; ++b) r2 += partial_h[b];
      if (first) {
        double q2 = 0.0;
        for (int b = 2 * 256; b < kHeviPartials * 256; ++b) q2 += partial_h[b];
        atol = 4.0 * DBL_EPSILON * sqrt(q2);
      }
      const double r = sqrt(r2);
      if (resid) resid[it] = r;
      if (it == 0 && r0_ext <= 0.0) r0 = r;
      if (rtol > 0.0 && (it > 0 || r0_ext > 0.0) && (r <= rtol * r0 || r <= atol)) break;
      if (rtol > 0.0 && it > 0 && r > 0.5 * r_prev) break;
      r_prev = r;
    }
    if (N1 <= 7 || ngroup <= (long)4 * ctx->ncu) {
      hipLaunchKernelGGL((hevi_solve3_kernel<N1, SOLVE_ALL>), gline, bline, 0, ctx->stream, a);
    } else if constexpr (N1 > 7) {
      hipLaunchKernelGGL((hevi_solve3_kernel<N1, SOLVE_DIAGONAL>), gline, bline, 0, ctx->stream, a);
      FEDG_HIP_CHECK(hipGetLastError());
      hipLaunchKernelGGL((hevi_solve3_kernel<N1, SOLVE_FLAGGED>), gflag, bline, 0, ctx->stream, a);
    }
    FEDG_HIP_CHECK(hipGetLastError());
    a.pin[VD] = a.pv[VD];
    a.pin[VW] = a.pv[VW];
    a.pin[VT] = a.pv[VT];
  }
  *it_done = it;
  return FEDG_OK;
}

// Predicted Newton iterate from the network, with the per-line fallback to
// q^n; returns ||G(q^n)|| (the tolerance's reference) in *r0.
int guess_buffers(fedg_ctx* ctx, HeviWork* w, int n_in, int n_out) {
  const DevMesh& m = ctx->m;
  const long nlines = (long)m.Ne2D * m.Nfp;
  if (w->X && w->n_in == n_in && w->n_out == n_out) return FEDG_OK;
  if (w->X) (void)hipFree(w->X);
  if (w->Y) (void)hipFree(w->Y);
  if (w->r_plain) (void)hipFree(w->r_plain);
  if (w->r_guess) (void)hipFree(w->r_guess);
  if (w->flag) (void)hipFree(w->flag);
  w->X = w->Y = nullptr;
  w->r_plain = w->r_guess = w->flag = nullptr;
  w->chunk = (int)(nlines < 16384 ? nlines : 16384);
  w->n_in = n_in;
  w->n_out = n_out;
  FEDG_HIP_CHECK(hipMalloc((void**)&w->X, sizeof(float) * (size_t)w->chunk * n_in));
  FEDG_HIP_CHECK(hipMalloc((void**)&w->Y, sizeof(float) * (size_t)w->chunk * n_out));
  FEDG_HIP_CHECK(hipMalloc((void**)&w->r_plain, sizeof(double) * nlines));
  FEDG_HIP_CHECK(hipMalloc((void**)&w->r_guess, sizeof(double) * nlines));
  FEDG_HIP_CHECK(hipMalloc((void**)&w->flag, sizeof(double) * nlines));
  return FEDG_OK;
}

template <int N1>
int predict_iterate(fedg_ctx* ctx, HeviWork* w, HeviArgs& a, HeviGuess* g, double* r0) {
  const DevMesh& m = ctx->m;
  const long nlines = (long)m.Ne2D * m.Nfp;
  const int L = a.NeZ * N1;
  int n_in = 0, n_out = 0;
  mlp_dims(g->mlp, &n_in, &n_out);
  if (n_in != 10 * L + 1 || n_out != 5 * L || L > 512) {
    set_error("HEVI guess: the network's sizes do not match 10 NeZ (p+1) + 1 inputs and 5 NeZ (p+1) outputs");
    return FEDG_ERR_ARG;
  }
  const int rcb = guess_buffers(ctx, w, n_in, n_out);
  if (rcb != FEDG_OK) return rcb;
  LineArgs la = line_args(m, a, g->Tex, g->scale, g->dt);
  const long nn = (long)m.Np * m.Ne;
  // residual of every line at q^n (pv holds q^n)
  launch_rhs_uv<N1>(ctx, a);
  FEDG_HIP_CHECK(hipGetLastError());
  a.alph_ready = 1;
  launch_rhs3<N1>(ctx, a);
  FEDG_HIP_CHECK(hipGetLastError());
  hipLaunchKernelGGL(line_resid_kernel, dim3(nlines), dim3(L), 0, ctx->stream, la, a.buv, a.b3, nn, w->r_plain);
  FEDG_HIP_CHECK(hipGetLastError());
  double r2 = 0.0;
  const int rcs = host_sum(ctx, w->r_plain, nlines, w->partial, w->partial_h, &r2);
  if (rcs != FEDG_OK) return rcs;
  *r0 = sqrt(r2);
  // network prediction, chunk by chunk
  for (long l0 = 0; l0 < nlines; l0 += w->chunk) {
    const int rows = (int)((nlines - l0) < w->chunk ? (nlines - l0) : w->chunk);
    la.line0 = l0;
    la.stride = 1;
    hipLaunchKernelGGL(line_features_kernel, dim3(rows), dim3(L), 0, ctx->stream, la, w->X, n_in, (float*)nullptr,
                       n_out);
    FEDG_HIP_CHECK(hipGetLastError());
    FEDG_HIP_CHECK(hipStreamSynchronize(ctx->stream));
    const int rcf = mlp_forward(g->mlp, w->X, w->Y, rows);
    if (rcf != FEDG_OK) return rcf;
    hipLaunchKernelGGL(line_apply_kernel, dim3(rows), dim3(L), 0, ctx->stream, la, w->Y, n_out);
    FEDG_HIP_CHECK(hipGetLastError());
  }
  // residual at the prediction; lines where it is not smaller restart from q^n
  la.line0 = 0;
  launch_rhs_uv<N1>(ctx, a);
  FEDG_HIP_CHECK(hipGetLastError());
  launch_rhs3<N1>(ctx, a);
  FEDG_HIP_CHECK(hipGetLastError());
  hipLaunchKernelGGL(line_resid_kernel, dim3(nlines), dim3(L), 0, ctx->stream, la, a.buv, a.b3, nn, w->r_guess);
  FEDG_HIP_CHECK(hipGetLastError());
  hipLaunchKernelGGL(line_select_kernel, dim3(nlines), dim3(L), 0, ctx->stream, la, w->r_guess, w->r_plain, w->flag);
  FEDG_HIP_CHECK(hipGetLastError());
  double nfb = 0.0, r2s = 0.0;
  const int rcs2 = host_sum(ctx, w->flag, nlines, w->partial, w->partial_h, &nfb);
  if (rcs2 != FEDG_OK) return rcs2;
  const int rcs3 = host_sum(ctx, w->r_guess, nlines, w->partial, w->partial_h, &r2s);
  if (rcs3 != FEDG_OK) return rcs3;
  g->lines += nlines;
  g->fallbacks += (long)(nfb + 0.5);
  g->r2_plain += r2;
  g->r2_start += r2s;
  return FEDG_OK;
}

template <int N1>
int run_operator(fedg_ctx* ctx, HeviArgs& a) {
  launch_rhs_uv<N1>(ctx, a);
  FEDG_HIP_CHECK(hipGetLastError());
  launch_rhs3<N1>(ctx, a);
  FEDG_HIP_CHECK(hipGetLastError());
  return FEDG_OK;
}

}  // namespace

namespace {
// the hydrostatic RHOT the residual kernels form from PRES_hyd (the same
// expression and pow, so the same bits), once per base state
__global__ void rhot_hyd_kernel(double* out, const double* PRES_hyd, const Consts c, long n) {
  const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n) return;
  const double rgamm = c.CVdry / c.CPdry;
  const double PRES0ovRdry = c.PRES00 / c.Rdry;
  out[t] = PRES0ovRdry * fedg_pow(PRES_hyd[t] / c.PRES00, rgamm);
}
}  // namespace

int launch_rhot_hyd(fedg_ctx* ctx, double* RHOT_hyd, const double* PRES_hyd, long n) {
  if (n <= 0) return FEDG_OK;
  hipLaunchKernelGGL(rhot_hyd_kernel, dim3((n + 255) / 256), dim3(256), 0, ctx->stream, RHOT_hyd, PRES_hyd, ctx->c, n);
  FEDG_HIP_CHECK(hipGetLastError());
  return FEDG_OK;
}

int hevi_cal_vi(fedg_ctx* ctx, HeviWork* w, double* const tend[5], const double* const q[5],
                const double* const var0[5], const double* DENS_hyd, const double* PRES_hyd, const double* Rtot,
                const double* CVtot, const double* CPtot, double impl_fac, int max_it, double rtol, double* resid,
                int* it_done, HeviGuess* guess, const HeviStore* store, const double* RHOT_hyd,
                int alph_ready, int keep_iterate) {
  const DevMesh& m = ctx->m;
  if (store && !(fabs(impl_fac) > 0.0)) {
    set_error("hevi_cal_vi: the fused StoreImplicit needs impl_fac != 0");
    return FEDG_ERR_ARG;
  }
  HeviArgs a{};
  a.m = m;
  a.c = ctx->c;
  for (int v = 0; v < 5; ++v) {
    a.qs[v] = q[v];
    a.q0[v] = var0[v];
    a.pv[v] = w->pv[v];
    a.pin[v] = var0[v];
    a.T[v] = tend[v];
  }
  a.DENS_hyd = DENS_hyd;
  a.PRES_hyd = PRES_hyd;
  a.RHOT_hyd = RHOT_hyd;
  a.alph_ready = alph_ready;
  a.Rtot = Rtot;
  a.CVtot = CVtot;
  a.CPtot = CPtot;
  a.alph = w->alph;
  a.b3 = w->b3;
  a.buv = w->buv;
  a.coef = w->coef;
  a.impl_fac = impl_fac;
  a.NeZ = m.Ne / m.Ne2D;
  const long n = (long)m.Np * m.Ne;
  *it_done = 0;
  // The first Newton iterate is q^n: the kernels read it from var0 until a
  // solve has written the variable's update to pv (run_newton moves a.pin).
  // The predicted iterate and a solve of no iteration start from a copy.
  const bool implicit = fabs(impl_fac) > 0.0;
  if (implicit && ((guess && guess->mlp) || max_it < 1)) {
    for (int v = 0; v < 5; ++v) {
      FEDG_HIP_CHECK(hipMemcpyAsync(w->pv[v], var0[v], sizeof(double) * n, hipMemcpyDeviceToDevice, ctx->stream));
      a.pin[v] = w->pv[v];
    }
  }
  auto dispatch = [&](auto n1c) -> int {
    constexpr int N1 = decltype(n1c)::value;
    if (implicit) {
      a.want_b = 1;
      double r0 = 0.0;
      if (guess && guess->mlp) {
        const int rc = predict_iterate<N1>(ctx, w, a, guess, &r0);
        if (rc != FEDG_OK) return rc;
      }
      const int finish = !store ? FINISH_TEND : store->var0[0] ? FINISH_STORE_COPY : FINISH_STORE;
      if (store)
        for (int v = 0; v < 5; ++v) {
          if (store->q[v] != q[v]) {
            set_error("hevi_cal_vi: the StoreImplicit state is not the solve's stage state");
            return FEDG_ERR_ARG;
          }
          a.qst[v] = store->q[v];
          a.var0[v] = store->var0[v];
          a.varTmp[v] = store->varTmp[v];
        }
      const int rc = run_newton<N1>(ctx, a, w, max_it, rtol, resid, it_done, r0, keep_iterate ? FINISH_NONE : finish);
      if (rc != FEDG_OK) return rc;
      // the variables the solve has not finished
      TendStore ts{};
      for (int v = 0; v < 5; ++v) {
        if (a.finish && v != VU && v != VV) continue;
        const int u = ts.nv++;
        ts.T[u] = tend[v];
        ts.p[u] = w->pv[v];
        ts.qs[u] = q[v];
        ts.q[u] = a.qst[v];
        ts.var0[u] = a.var0[v];
        ts.varTmp[u] = a.varTmp[v];
      }
      ts.impl_fac = impl_fac;
      ts.finish = finish;
      const int bs = 256;
      hipLaunchKernelGGL(hevi_tend_store_kernel, dim3((n + bs - 1) / bs), dim3(bs), 0, ctx->stream, ts, n);
      FEDG_HIP_CHECK(hipGetLastError());
      return FEDG_OK;
    }
    a.want_b = 0;
    return run_operator<N1>(ctx, a);
  };
  switch (m.n1) {
    case 2: return dispatch(std::integral_constant<int, 2>{});
    case 3: return dispatch(std::integral_constant<int, 3>{});
    case 4: return dispatch(std::integral_constant<int, 4>{});
    case 5: return dispatch(std::integral_constant<int, 5>{});
    case 6: return dispatch(std::integral_constant<int, 6>{});
    case 7: return dispatch(std::integral_constant<int, 7>{});
    case 8: return dispatch(std::integral_constant<int, 8>{});
    default:
      set_error("polynomial order not built (supported: p = 1..7)");
      return FEDG_ERR_UNSUPPORTED;
  }
}

int hevi_harvest(fedg_ctx* ctx, HeviWork* w, const double* const q[5], const double* const var0[5],
                 const double* const Tex[5], const double scale[15], double impl_fac, double dt, long line0,
                 long stride, int nrows, float* X, float* Y) {
  const DevMesh& m = ctx->m;
  HeviArgs a{};
  a.m = m;
  for (int v = 0; v < 5; ++v) {
    a.qs[v] = q[v];
    a.q0[v] = var0[v];
    a.pv[v] = w->pv[v];
  }
  a.impl_fac = impl_fac;
  a.NeZ = m.Ne / m.Ne2D;
  LineArgs la = line_args(m, a, Tex, scale, dt);
  if (la.L > 512 || nrows < 1) return FEDG_ERR_ARG;
  la.line0 = line0;
  la.stride = stride;
  hipLaunchKernelGGL(line_features_kernel, dim3(nrows), dim3(la.L), 0, ctx->stream, la, X, 10 * la.L + 1, Y,
                     5 * la.L);
  FEDG_HIP_CHECK(hipGetLastError());
  return FEDG_OK;
}

// ---------------------------------------------------------------------------
// Workspace of fedg_hevi_cal_vi_noalloc: a file-scope device array in place
// of hipMalloc, for callers that may not allocate (HIP graph capture, serving
// loops).  Every device that runs the library holds its own copy until the
// process ends; every call on a device shares it and finds the previous
// call's contents (the solve writes each part before reading it: the iterate
// is read from var0 until a solve has written it, the rhs, damping and
// linearisation coefficients and the partial sums are written by their
// kernels, so nothing needs clearing).
constexpr size_t kScratchDoubles = (size_t)8 << 20;  // 64 MiB

static __device__ __align__(256) double scratch[kScratchDoubles];

// The line solves' scratch of the same calls, apart from it so that the
// meshes the workspace takes do not change: 32 MiB hold the level solutions
// of 682 wavefronts at p = 7 and NeZ = 8, and of at least 136 for every mesh
// taken (p = 2 at 53 levels; the wavefronts in flight walk the lines).
constexpr size_t kLineScratchDoubles = (size_t)4 << 20;

static __device__ __align__(256) double line_scratch[kLineScratchDoubles];

namespace {
constexpr int kScratchDevices = 64;
std::mutex scratch_mu;
double* scratch_dev[kScratchDevices];       // address of `scratch` on each device, set once
double* line_scratch_dev[kScratchDevices];  // and of `line_scratch`

// a part of the workspace rounded up to 32 doubles (256 B alignment)
size_t part(size_t n) { return (n + 31) & ~(size_t)31; }

// doubles of the workspace a solve on mesh m needs (the HeviWork layout; 256
// more stay free, so that the meshes taken are those they always were)
size_t noalloc_need(const DevMesh& m) {
  const size_t n = (size_t)m.Np * m.Ne;
  return 5 * part(n) + part((size_t)2 * m.Nfp * m.Ne) + part(3 * n) + part(2 * n) + part(3 * n) + 256;
}
}  // namespace

// Looks up the device address of `scratch` on `device`, which must be the
// current device; once per device (later calls return at once).
int noalloc_scratch_setup(int device) {
  if (device < 0 || device >= kScratchDevices) {
    set_error("device index beyond the workspace table of fedg_hevi_cal_vi_noalloc (64 devices)");
    return FEDG_ERR_UNSUPPORTED;
  }
  std::lock_guard<std::mutex> lock(scratch_mu);
  if (scratch_dev[device]) return FEDG_OK;
  void *ptr = nullptr, *lptr = nullptr;
  hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
  if (e == hipSuccess) e = hipGetSymbolAddress(&lptr, HIP_SYMBOL(line_scratch));
  if (e != hipSuccess || ptr == nullptr || lptr == nullptr) {
    set_error(std::string("hipGetSymbolAddress of the no-allocation workspace: ") + hipGetErrorString(e));
    return FEDG_ERR_HIP;
  }
  line_scratch_dev[device] = static_cast<double*>(lptr);
  scratch_dev[device] = static_cast<double*>(ptr);
  return FEDG_OK;
}

}  // namespace fedg

extern "C" int fedg_hevi_cal_vi_noalloc(fedg_ctx* ctx, double* DENS_dt, double* MOMX_dt, double* MOMY_dt,
                                        double* MOMZ_dt, double* RHOT_dt, const double* DDENS_,
                                        const double* MOMX_, const double* MOMY_, const double* MOMZ_,
                                        const double* DRHOT_, const double* DENS_hyd, const double* PRES_hyd,
                                        const double* DDENS0_, const double* MOMX0_, const double* MOMY0_,
                                        const double* MOMZ0_, const double* DRHOT0_, const double* Rtot,
                                        const double* CVtot, const double* CPtot, double impl_fac, double dt,
                                        int max_it, double rtol, double* resid, int* iterations) {
  using namespace fedg;
  (void)dt;
  if (!ctx || !DENS_dt || !MOMX_dt || !MOMY_dt || !MOMZ_dt || !RHOT_dt || !DDENS_ || !MOMX_ || !MOMY_ || !MOMZ_ ||
      !DRHOT_ || !DENS_hyd || !PRES_hyd || !DDENS0_ || !MOMX0_ || !MOMY0_ || !MOMZ0_ || !DRHOT0_ || !Rtot ||
      !CVtot || !CPtot || max_it < 1 || !std::isfinite(impl_fac))
    return FEDG_ERR_ARG;
  const DevMesh& m = ctx->m;
  if (m.Ne2D <= 0 || m.Ne % m.Ne2D != 0) {
    set_error("HEVI: the mesh is not a stack of Ne2D-element horizontal layers");
    return FEDG_ERR_UNSUPPORTED;
  }
  const size_t need = noalloc_need(m);
  if (need > kScratchDoubles) {
    set_error("fedg_hevi_cal_vi_noalloc: the mesh needs " + std::to_string(need * sizeof(double)) +
              " bytes of workspace, the fixed workspace holds " + std::to_string(kScratchDoubles * sizeof(double)) +
              " (64 MiB); use fedg_hevi_cal_vi_newton");
    return FEDG_ERR_UNSUPPORTED;
  }
  double* p = (ctx->device >= 0 && ctx->device < kScratchDevices) ? scratch_dev[ctx->device] : nullptr;
  if (p == nullptr) {
    set_error("fedg_hevi_cal_vi_noalloc: the workspace of this context's device was not set up");
    return FEDG_ERR_HIP;
  }
  const size_t n = (size_t)m.Np * m.Ne;
  HeviWork w{};
  for (int v = 0; v < 5; ++v) {
    w.pv[v] = p;
    p += part(n);
  }
  w.alph = p;
  p += part((size_t)2 * m.Nfp * m.Ne);
  w.b3 = p;
  p += part(3 * n);
  w.buv = p;
  p += part(2 * n);
  w.coef = p;
  p += part(3 * n);
  // the partial sums take the end of the line solves' scratch
  double partial_h[kHeviPartials * 256];
  w.lines = line_scratch_dev[ctx->device];
  w.lines_n = kLineScratchDoubles - kHeviPartials * 256;
  w.partial = w.lines + w.lines_n;
  w.partial_h = partial_h;
  double* tend[5] = {DENS_dt, RHOT_dt, MOMZ_dt, MOMX_dt, MOMY_dt};
  const double* q[5] = {DDENS_, DRHOT_, MOMZ_, MOMX_, MOMY_};
  const double* q0[5] = {DDENS0_, DRHOT0_, MOMZ0_, MOMX0_, MOMY0_};
  int it = 0;
  const int rc = hevi_cal_vi(ctx, &w, tend, q, q0, DENS_hyd, PRES_hyd, Rtot, CVtot, CPtot, impl_fac, max_it, rtol,
                             resid, &it, nullptr);
  if (rc != FEDG_OK) return rc;
  FEDG_HIP_CHECK(hipStreamSynchronize(ctx->stream));
  if (iterations) *iterations = it;
  return FEDG_OK;
}
