// jacobian_kernels.hpp -- explicit Jacobian blocks of the DG-SBP Euler residual.
//
// evalJacobian (src/solver/euler/evalJacobian.jl:6-72) computes, per element,
// the volume block dR_e/dq_e (calcVolumeIntegrals_nopre_diff,
// euler_funcs_diff.jl:54-104, or the split-form calcVolumeIntegralsSplitForm_diff
// :330-430) and per face the blocks jacLL/jacLR/jacRL/jacRR
// (calcFaceIntegral_nopre_diff, flux_diff.jl:6-88) and per boundary face the
// block dR_e/dq_e (calcBoundaryFlux_nopre_diff, bc_diff.jl:124-212), and
// scatters them with ADD_VALUES into a block matrix (assembleElement /
// assembleInterface / assembleBoundary, src/jacobian/jacobian.jl:822-1759).
//
// Here a workgroup owns a few elements and writes every block of their rows
// (each element's own Np x Np blocks plus those coupling it to each
// neighbour) directly into the BSR value array: each block is written by
// exactly one workgroup, no atomics and no assembly pass.  Point derivatives
// come from forward-mode dual numbers (dF/dqL, dF/dqR), the analytic
// counterpart of the reference's hand-differentiated *_diff functions.
//
// The kernel is written so that no thread runs long and few values spill (none
// outside the entropy-stable form; there 3D p=2 puts 364 to 372 bytes a lane into
// scratch memory): a face node's derivative is one thread per seeded component (dual<1>), a volume
// pair one thread per ordered pair, differentiated in the combined direction
// with respect to one state only (the flux is symmetric: the other state's
// derivative is the other ordered pair's), and the weak form's blocks are
// formed and stored a BSR row at a time, lane by value.  With one thread per
// block and per face node, all components seeded at once (dual<2 ndof>, 300 to
// 480 bytes of spills a lane) and DIM fluxes per pair and row, the assembly
// took (MI355X, FP32 blocks) 2487 us for 4,050 triangles diagonal-E p=3 split
// form and 976 us for 6,000 tets Omega p=2 Roe; it takes 109 us and 182 us (the
// stores alone, at the copy rate, 20 us and 60 us).  The row loops of the weak
// form stay rolled: unrolled, the hoisted weights spill (454 us for the tets).
#pragma once
#include "residual_kernels.hpp"

namespace pdes {

// what a workgroup holds per element
template <class Op, int VOL, int FLUX>
struct JacElem {
  static constexpr int NP = Op::NP, ND = Op::ND, DIM = Op::DIM, NF = Op::NF, NFACES = Op::NFACES;
  double q[NP][ND];
  double A[(VOL == VOL_WEAK) ? NP * DIM : 1][ND][ND];   // dF_d/dq at node j
  // split form: the IR parameter vector of every node and its derivative
  double z[(VOL == VOL_SPLIT) ? NP : 1][ND];
  double dz[(VOL == VOL_SPLIT) ? NP : 1][ND][ND];
  // partial sums of the diagonal blocks, one per thread of a column
  static constexpr int KP = 4;
  double diag[(VOL == VOL_SPLIT) ? NP : 1][(VOL == VOL_SPLIT) ? KP : 1][ND][ND];
  // dense faces: weight of slot k's flux in row i's residual, sgn B R[i][kown]
  static constexpr bool CW = VOL == VOL_WEAK && !Op::DIAGE;
  double cw[CW ? NFACES : 1][CW ? NP : 1][CW ? NF : 1];
  double qf[NFACES][NF][2][ND];         // face-node states (entropy variables for ESLF): elementL's, elementR's
  double dFo[NFACES][NF][ND][ND];       // dF_k/dq_own   (k: elementL face node numbering)
  double dFn[NFACES][NF][ND][ND];       // dF_k/dq_nbr
  ElFace rec[NFACES];
  int32_t kown[NFACES][NF];             // own face node of slot k
  int32_t knbr[NFACES][NF];             // neighbour face node of slot k
  int32_t kslot[NFACES][NF];            // slot of own face node m
  double sgn[NFACES];
  int64_t own_run[NP];                  // first own block of each row
  // first block of the neighbour's run in each row (dense faces), or the one
  // block of each face node (diagonal-E, [NFACES][NF])
  int64_t nbr_run[NFACES][Op::DIAGE ? NF : NP];
  int64_t e;
};

template <class Op, int VOL, int FLUX, int EPB>
struct JacSmem {
  static constexpr int NP = Op::NP, ND = Op::ND, DIM = Op::DIM, NF = Op::NF, NFACES = Op::NFACES;
  double Q[DIM][NP][NP];
  double interp[Op::ST][NF];
  int32_t perm[Op::ST][NFACES];
  int32_t nodepos[NP][NFACES];
  double wface[NF];
  JacElem<Op, VOL, FLUX> el[EPB];
};

// what the entropy-stable block functions read: the tables and one element
template <class Op, int VOL, int FLUX, int EPB>
struct JacView {
  const double (&interp)[Op::ST][Op::NF];
  const int32_t (&perm)[Op::ST][Op::NFACES];
  const double (&wface)[Op::NF];
  const double (&q)[Op::NP][Op::ND];
  const double (&dFo)[Op::NFACES][Op::NF][Op::ND][Op::ND];
  const double (&dFn)[Op::NFACES][Op::NF][Op::ND][Op::ND];
  const ElFace (&rec)[Op::NFACES];
  const int32_t (&kown)[Op::NFACES][Op::NF];
  const int32_t (&knbr)[Op::NFACES][Op::NF];
  const double (&sgn)[Op::NFACES];
  __device__ __forceinline__ JacView(const JacSmem<Op, VOL, FLUX, EPB>& s, const JacElem<Op, VOL, FLUX>& x)
      : interp(s.interp), perm(s.perm), wface(s.wface), q(x.q), dFo(x.dFo), dFn(x.dFn), rec(x.rec), kown(x.kown),
        knbr(x.knbr), sgn(x.sgn) {}
};

template <class BT> __device__ __forceinline__ BT to_block(double x) { return (BT)x; }

// position of block column `col` in BSR row `row` (sorted colind), -1 if absent
__device__ __forceinline__ int64_t bsr_find(const int64_t* __restrict__ rowptr, const int32_t* __restrict__ colind,
                                            int64_t row, int32_t col) {
  int64_t lo = rowptr[row], hi = rowptr[row + 1] - 1;
  while (lo <= hi) {
    int64_t mid = (lo + hi) >> 1;
    int32_t c = colind[mid];
    if (c == col) return mid;
    if (c < col) lo = mid + 1; else hi = mid - 1;
  }
  return -1;
}

// dw/dq of the IR entropy variables at state q (convertToIR_ differentiated)
template <int DIM>
__device__ __forceinline__ void ir_vars_jacobian(const PhysConst& p, const double* q, double (*W)[DIM + 2]) {
  constexpr int ND = DIM + 2;
  dual<ND> qd[ND], w[ND];
#pragma unroll
  for (int c = 0; c < ND; ++c) { qd[c] = dual<ND>(q[c]); qd[c].d[c] = 1.0; }
  to_ir_vars<DIM>(p, qd, w);
#pragma unroll
  for (int a = 0; a < ND; ++a)
#pragma unroll
    for (int c = 0; c < ND; ++c) W[a][c] = w[a].d[c];
}

// E_tu[d] = sum_k R[iL][k] R[jR][kR(k)] B[k] n_d[k] of the entropy-conservative
// face integral (calcECFaceIntegral, faceElementIntegrals.jl:58-120), with
// (iL, jR) = (t, u) when this element is elementL and (u, t) otherwise
template <class Op, class Sm>
__device__ __forceinline__ void ec_weights(const Sm& sm, const DevSBP& sbp, const DevMesh& mesh, const ElFace& r,
                                           int t, int u, double* E) {
  constexpr int DIM = Op::DIM, NF = Op::NF;
  const int o = (r.z >> 8) & 0xff, side = (r.z >> 16) & 1;
  const int iL = side == 0 ? t : u, jR = side == 0 ? u : t;
  const double* nr = mesh.nrm_face + (int64_t)r.y * NF * DIM;
#pragma unroll
  for (int d = 0; d < DIM; ++d) E[d] = 0.0;
  for (int k = 0; k < NF; ++k) {
    const int kRk = sbp.nbrperm[k * sbp.norient + o];
    const double base = sm.interp[iL][k] * sm.interp[jR][kRk] * sm.wface[k];
#pragma unroll
    for (int d = 0; d < DIM; ++d) E[d] += base * nr[k * DIM + d];
  }
}

// d/dq of F_IR(q_L, q_R) . E for the pair (own stencil node t, neighbour
// stencil node u) of face f, with respect to the own state (wrt_own) or the
// neighbour's; the sum over directions of E_d F_d is the flux in direction E
template <class Op, class Sm>
__device__ __forceinline__ void ec_pair_derivative(const Sm& sm, const DevSBP& sbp, const DevMesh& mesh,
                                                   const PhysConst& phys, const double* qin, int f, int t, int u,
                                                   bool wrt_own, double (*D)[Op::ND]) {
  constexpr int DIM = Op::DIM, NP = Op::NP, ND = Op::ND;
  const ElFace r = sm.rec[f];
  const int fN = r.z & 0xff, side = (r.z >> 16) & 1;
  const double* qn = qin + ((int64_t)r.x * NP + sm.perm[u][fN]) * ND;
  dual<ND> qo[ND], qb[ND], zo[ND], zb[ND], zL[ND], zR[ND], F[ND];
#pragma unroll
  for (int c = 0; c < ND; ++c) {
    qo[c] = dual<ND>(sm.q[sm.perm[t][f]][c]);
    qb[c] = dual<ND>(qn[c]);
    if (wrt_own) qo[c].d[c] = 1.0;
    else qb[c].d[c] = 1.0;
  }
  ir_zvars<DIM>(phys, qo, zo);
  ir_zvars<DIM>(phys, qb, zb);
#pragma unroll
  for (int c = 0; c < ND; ++c) {
    zL[c] = side == 0 ? zo[c] : zb[c];
    zR[c] = side == 0 ? zb[c] : zo[c];
  }
  double E[DIM];
  ec_weights<Op>(sm, sbp, mesh, r, t, u, E);
  ir_flux_z<DIM, 1>(phys, zL, zR, E, F);
#pragma unroll
  for (int a = 0; a < ND; ++a)
#pragma unroll
    for (int c = 0; c < ND; ++c) D[a][c] = F[a].d[c];
}

// ESLF interior face f, own block (i, j): the entropy penalty through the
// interpolated own entropy variables, sum_k sg R[si][ko] R[sj][ko] dP_k/dw_own
// times dw/dq(q_j); for i == j also the entropy-conservative pairs of node si
template <class Op, class Sm>
__device__ __forceinline__ void eslf_own_block(const Sm& sm, const DevSBP& sbp, const DevMesh& mesh,
                                               const PhysConst& phys, const double* qin, int f, int i, int j,
                                               int si, int sj, double (*B)[Op::ND]) {
  constexpr int DIM = Op::DIM, NF = Op::NF, ST = Op::ST, ND = Op::ND;
  const double sg = sm.sgn[f];
  double M[ND][ND], W[ND][ND];
#pragma unroll
  for (int a = 0; a < ND; ++a)
#pragma unroll
    for (int c = 0; c < ND; ++c) M[a][c] = 0.0;
  for (int k = 0; k < NF; ++k) {
    const int m = sm.kown[f][k];
    const double wgt = sg * sm.interp[si][m] * sm.interp[sj][m];
#pragma unroll
    for (int a = 0; a < ND; ++a)
#pragma unroll
      for (int c = 0; c < ND; ++c) M[a][c] += wgt * sm.dFo[f][k][a][c];
  }
  ir_vars_jacobian<DIM>(phys, sm.q[j], W);
#pragma unroll
  for (int a = 0; a < ND; ++a)
#pragma unroll
    for (int c = 0; c < ND; ++c) {
      double acc = 0.0;
#pragma unroll
      for (int b = 0; b < ND; ++b) acc += M[a][b] * W[b][c];
      B[a][c] += acc;
    }
  if (i != j) return;
  for (int u = 0; u < ST; ++u) {
    double D[ND][ND];
    ec_pair_derivative<Op>(sm, sbp, mesh, phys, qin, f, si, u, true, D);
#pragma unroll
    for (int a = 0; a < ND; ++a)
#pragma unroll
      for (int c = 0; c < ND; ++c) B[a][c] += sg * D[a][c];
  }
}

// ESLF interior face f, neighbour block (row node with stencil position si,
// neighbour node jn with stencil position sj on the neighbour's face)
template <class Op, class Sm>
__device__ __forceinline__ void eslf_nbr_block(const Sm& sm, const DevSBP& sbp, const DevMesh& mesh,
                                               const PhysConst& phys, const double* qin, int f, int jn,
                                               int si, int sj, double (*B)[Op::ND]) {
  constexpr int DIM = Op::DIM, NP = Op::NP, NF = Op::NF, ND = Op::ND;
  const double sg = sm.sgn[f];
  double M[ND][ND], W[ND][ND];
#pragma unroll
  for (int a = 0; a < ND; ++a)
#pragma unroll
    for (int c = 0; c < ND; ++c) M[a][c] = 0.0;
  for (int k = 0; k < NF; ++k) {
    const double wgt = sg * sm.interp[si][sm.kown[f][k]] * sm.interp[sj][sm.knbr[f][k]];
#pragma unroll
    for (int a = 0; a < ND; ++a)
#pragma unroll
      for (int c = 0; c < ND; ++c) M[a][c] += wgt * sm.dFn[f][k][a][c];
  }
  ir_vars_jacobian<DIM>(phys, qin + ((int64_t)sm.rec[f].x * NP + jn) * ND, W);
  double D[ND][ND];
  ec_pair_derivative<Op>(sm, sbp, mesh, phys, qin, f, si, sj, false, D);
#pragma unroll
  for (int a = 0; a < ND; ++a)
#pragma unroll
    for (int c = 0; c < ND; ++c) {
      double acc = 0.0;
#pragma unroll
      for (int b = 0; b < ND; ++b) acc += M[a][b] * W[b][c];
      B[a][c] += acc + sg * D[a][c];
    }
}

// own block (i, j) of an entropy-stable operator: face f's contribution
// (interior: the entropy-stable integral; boundary: the Roe flux against the
// boundary state)
template <class Op, class Sm>
__device__ __forceinline__ void es_own_face(const Sm& sm, const DevSBP& sbp, const DevMesh& mesh,
                                            const PhysConst& phys, const double* qin, int f, int i, int j, int si,
                                            int sj, double (*B)[Op::ND]) {
  constexpr int NF = Op::NF, ND = Op::ND;
  if (sm.rec[f].x >= 0) {
    eslf_own_block<Op>(sm, sbp, mesh, phys, qin, f, i, j, si, sj, B);
    return;
  }
  for (int k = 0; k < NF; ++k) {
    const int m = sm.kown[f][k];
    const double wgt = sm.sgn[f] * sm.wface[m] * sm.interp[si][m] * sm.interp[sj][m];
#pragma unroll
    for (int a = 0; a < ND; ++a)
#pragma unroll
      for (int c = 0; c < ND; ++c) B[a][c] += wgt * sm.dFo[f][k][a][c];
  }
}

// the flux at a face node as a function of one seeded component: side 0 is
// elementL's state, side 1 elementR's (qs: both states; comp of `side` seeded)
template <class Op, int FLUX>
__device__ __forceinline__ void face_derivative(const PhysConst& phys, const double (*qs)[Op::ND], int side, int comp,
                                                const double* nrm, double scale, double* dF) {
  constexpr int DIM = Op::DIM, ND = Op::ND;
  dual<1> qL[ND], qR[ND], F[ND];
#pragma unroll
  for (int c = 0; c < ND; ++c) {
    qL[c] = dual<1>(qs[0][c]);
    qL[c].d[0] = side == 0 && c == comp ? 1.0 : 0.0;
    qR[c] = dual<1>(qs[1][c]);
    qR[c].d[0] = side == 1 && c == comp ? 1.0 : 0.0;
  }
  if constexpr (FLUX == PDES_FLUX_ROE) {
    roe_flux<DIM>(phys, qL, qR, nrm, F);
  } else if constexpr (FLUX == PDES_FLUX_IRSLF) {
    irslf_flux<DIM>(phys, qL, qR, nrm, F);
  } else {
    // entropy penalty (calcEntropyPenaltyIntegral, faceElementIntegrals.jl:
    // 199-290) of the interpolated IR entropy variables
    dual<1> qa[ND], qlr[ND], dw[ND];
    ir_to_conservative<DIM>(phys, qL, qa);
    ir_to_conservative<DIM>(phys, qR, qlr);
#pragma unroll
    for (int c = 0; c < ND; ++c) {
      qa[c] = 0.5 * (qa[c] + qlr[c]);
      dw[c] = qL[c] - qR[c];
      F[c] = dual<1>(0.0);
    }
    lf_entropy_apply<DIM>(phys, qa, dw, nrm, scale, F);
  }
#pragma unroll
  for (int a = 0; a < ND; ++a) dF[a] = F[a].d[0];
}

// elements per workgroup: as many as give every thread about one row of
// values (weak form: NP ndof^2 of them) or one volume pair column, in at most
// 40 KB of LDS for the elements (with the operator's tables 42 KB: three
// workgroups of the split form a CU, and its 212 registers allow two waves a SIMD)
template <class Op, int VOL, int FLUX>
constexpr int jac_epb() {
  constexpr int per = VOL == VOL_WEAK ? Op::NP * Op::ND * Op::ND : Op::NP * JacElem<Op, VOL, FLUX>::KP;
  constexpr int fit = 40960 / (int)sizeof(JacElem<Op, VOL, FLUX>), want = 256 / per;
  constexpr int n = want < fit ? want : fit;
  return n < 1 ? 1 : n;
}

template <class Op, int VOL, int FLUX, class BT>
__global__ void __launch_bounds__(256)
euler_jacobian_kernel(DevMesh mesh, DevSBP sbp, PhysConst phys, const double* __restrict__ qin,
                      const int64_t* __restrict__ rowptr, const int32_t* __restrict__ colind,
                      BT* __restrict__ vals, int32_t* __restrict__ err,
                      const double* __restrict__ ptc_diag, const double* __restrict__ ptc_scale) {
  constexpr int DIM = Op::DIM, NP = Op::NP, NF = Op::NF, ST = Op::ST, ND = Op::ND, NFACES = Op::NFACES;
  constexpr int NB = ND * ND, T = 256, SLOTS = NFACES * NF;
  constexpr int EPB = jac_epb<Op, VOL, FLUX>();
  constexpr bool ES = FLUX == PDES_FLUX_ESLF;
  using Elem = JacElem<Op, VOL, FLUX>;
  __shared__ JacSmem<Op, VOL, FLUX, EPB> sm;
  const int tid = threadIdx.x;
  const int64_t s0 = (int64_t)blockIdx.x * EPB;
  const int nel = (int)(launch_count(mesh) - s0 < EPB ? launch_count(mesh) - s0 : EPB);
  for (int x = tid; x < DIM * NP * NP; x += T) (&sm.Q[0][0][0])[x] = sbp.Q[x];
  for (int x = tid; x < ST * NF; x += T) (&sm.interp[0][0])[x] = sbp.interp[x];
  for (int x = tid; x < ST * NFACES; x += T) (&sm.perm[0][0])[x] = sbp.perm[x];
  for (int x = tid; x < NP * NFACES; x += T) (&sm.nodepos[0][0])[x] = sbp.nodepos[x];
  for (int x = tid; x < NF; x += T) sm.wface[x] = sbp.wface[x];
  for (int t = tid; t < nel * NP * ND; t += T) {
    const int l = t / (NP * ND), x = t - l * (NP * ND);
    (&sm.el[l].q[0][0])[x] = qin[element_of(mesh, s0 + l) * NP * ND + x];
  }
  for (int t = tid; t < nel * NFACES; t += T) {
    const int l = t / NFACES, f = t - l * NFACES;
    const int64_t e = element_of(mesh, s0 + l);
    const ElFace r = mesh.elface[e * NFACES + f];
    sm.el[l].e = e;
    sm.el[l].rec[f] = r;
    sm.el[l].sgn[f] = r.x >= 0 && ((r.z >> 16) & 1) ? 1.0 : -1.0;
  }
  __syncthreads();
  for (int t = tid; t < nel * SLOTS; t += T) {
    const int l = t / SLOTS, f = (t - l * SLOTS) / NF, k = t % NF;
    Elem& el = sm.el[l];
    const ElFace r = el.rec[f];
    int ko = k, kn = k;
    if (r.x >= 0) {
      const int o = (r.z >> 8) & 0xff;
      const int kR = sbp.nbrperm[k * sbp.norient + o];
      const int side = (r.z >> 16) & 1;
      ko = side == 0 ? k : kR;
      kn = side == 0 ? kR : k;
    }
    el.kown[f][k] = ko;
    el.knbr[f][k] = kn;
    el.kslot[f][ko] = k;
    if constexpr (Op::DIAGE) {
      // slot k couples own node perm[ko][f] with neighbour node perm[kn][fN]
      int64_t pos = -1;
      if (r.x >= 0) {
        pos = bsr_find(rowptr, colind, el.e * NP + sm.perm[ko][f], (int32_t)((int64_t)r.x * NP + sm.perm[kn][r.z & 0xff]));
        if (pos < 0) err[0] = 1;
      }
      el.nbr_run[f][k] = pos;
    }
  }
  // where each row's runs of NP blocks begin: own, and per neighbour for dense faces
  constexpr int RUNS = Op::DIAGE ? 1 : 1 + NFACES;
  for (int t = tid; t < nel * NP * RUNS; t += T) {
    const int l = t / (NP * RUNS), x = t - l * (NP * RUNS), f = x / NP - 1, i = x % NP;
    Elem& el = sm.el[l];
    const int64_t ce = f < 0 ? el.e : (int64_t)el.rec[f].x;
    int64_t pos = -1;
    if (ce >= 0) {
      pos = bsr_find(rowptr, colind, el.e * NP + i, (int32_t)(ce * NP));
      if (pos < 0 || colind[pos + NP - 1] != ce * NP + NP - 1) { err[0] = 1; pos = -1; }
    }
    if (f < 0) el.own_run[i] = pos;
    else if constexpr (!Op::DIAGE) el.nbr_run[f][i] = pos;
  }
  // states at the face nodes, one thread per (slot, side, component)
  for (int t = tid; t < nel * SLOTS * 2 * ND; t += T) {
    const int l = t / (SLOTS * 2 * ND);
    int x = t - l * (SLOTS * 2 * ND);
    const int c = x % ND, sd = (x / ND) & 1;
    x /= 2 * ND;
    const int f = x / NF, k = x - f * NF;
    Elem& el = sm.el[l];
    const ElFace r = el.rec[f];
    double v = 0.0;
    if (r.x < 0) {
      if (sd == 0)
        for (int s = 0; s < ST; ++s) v += sm.interp[s][k] * el.q[sm.perm[s][f]][c];
      else
        v = mesh.qbc[((int64_t)r.y * NF + k) * ND + c];
    } else {
      const int fN = r.z & 0xff, side = (r.z >> 16) & 1, o = (r.z >> 8) & 0xff;
      const int kk = sd == 0 ? k : sbp.nbrperm[k * sbp.norient + o];
      const bool own = sd == side;
      const double* qnb = qin + (int64_t)r.x * NP * ND;
      for (int s = 0; s < ST; ++s) {
        if constexpr (ES) {
          double qs[ND], w[ND];
#pragma unroll
          for (int a = 0; a < ND; ++a) qs[a] = own ? el.q[sm.perm[s][f]][a] : qnb[sm.perm[s][fN] * ND + a];
          to_ir_vars<DIM>(phys, qs, w);
          double wc = w[0];
#pragma unroll
          for (int a = 1; a < ND; ++a) wc = a == c ? w[a] : wc;
          v += sm.interp[s][kk] * wc;
        } else {
          v += sm.interp[s][kk] * (own ? el.q[sm.perm[s][f]][c] : qnb[sm.perm[s][fN] * ND + c]);
        }
      }
    }
    el.qf[f][k][sd][c] = v;
  }
  if constexpr (VOL == VOL_WEAK) {
    for (int t = tid; t < nel * NP * DIM * ND; t += T) {
      const int l = t / (NP * DIM * ND);
      int x = t - l * (NP * DIM * ND);
      const int comp = x % ND, d = (x / ND) % DIM, j = x / (ND * DIM);
      Elem& el = sm.el[l];
      dual<1> qd[ND], F[ND];
#pragma unroll
      for (int c = 0; c < ND; ++c) { qd[c] = dual<1>(el.q[j][c]); qd[c].d[0] = c == comp ? 1.0 : 0.0; }
      double nrm[DIM];
#pragma unroll
      for (int y = 0; y < DIM; ++y) nrm[y] = metric<DIM, NP>(mesh, el.e, j)[y * DIM + d];
      euler_flux<DIM>(phys, qd, nrm, F);
#pragma unroll
      for (int r = 0; r < ND; ++r) el.A[j * DIM + d][r][comp] = F[r].d[0];
    }
  } else {
    for (int t = tid; t < nel * NP * ND; t += T) {
      const int l = t / (NP * ND), j = (t - l * (NP * ND)) / ND, comp = t % ND;
      Elem& el = sm.el[l];
      dual<1> qd[ND], z[ND];
#pragma unroll
      for (int c = 0; c < ND; ++c) { qd[c] = dual<1>(el.q[j][c]); qd[c].d[0] = c == comp ? 1.0 : 0.0; }
      ir_zvars<DIM>(phys, qd, z);
#pragma unroll
      for (int r = 0; r < ND; ++r) el.dz[j][r][comp] = z[r].d[0];
      if (comp == 0) {
#pragma unroll
        for (int r = 0; r < ND; ++r) el.z[j][r] = z[r].v;
      }
    }
  }
  __syncthreads();

  // ---- face derivatives, one thread per (slot, side, component)
  for (int t = tid; t < nel * SLOTS * 2 * ND; t += T) {
    const int l = t / (SLOTS * 2 * ND);
    int x = t - l * (SLOTS * 2 * ND);
    const int comp = x % ND, sd = (x / ND) & 1;
    x /= 2 * ND;
    const int f = x / NF, k = x - f * NF;
    Elem& el = sm.el[l];
    const ElFace r = el.rec[f];
    double dF[ND];
    if (r.x < 0) {
      if (sd == 0) face_derivative<Op, PDES_FLUX_ROE>(phys, el.qf[f][k], 0, comp, mesh.nrm_bndry + ((int64_t)r.y * NF + k) * DIM, 1.0, dF);
    } else {
      face_derivative<Op, FLUX>(phys, el.qf[f][k], sd, comp, mesh.nrm_face + ((int64_t)r.y * NF + k) * DIM,
                                sm.wface[k], dF);
    }
    const bool own = r.x < 0 ? sd == 0 : sd == ((r.z >> 16) & 1);
    if (r.x < 0 && sd == 1) {
#pragma unroll
      for (int a = 0; a < ND; ++a) dF[a] = 0.0;
    }
#pragma unroll
    for (int a = 0; a < ND; ++a) (own ? el.dFo : el.dFn)[f][k][a][comp] = dF[a];
  }
  __syncthreads();

  if constexpr (Elem::CW) {
    for (int t = tid; t < nel * NP * SLOTS; t += T) {
      const int l = t / (NP * SLOTS), x = t - l * (NP * SLOTS), i = x / SLOTS, f = (x % SLOTS) / NF, k = x % NF;
      Elem& el = sm.el[l];
      const int m = el.kown[f][k], si = sm.nodepos[i][f];
      el.cw[f][i][k] = si >= 0 ? el.sgn[f] * sm.wface[m] * sm.interp[si][m] : 0.0;
    }
    __syncthreads();
  }

  // ---- blocks of the elements' rows
  // a face's contribution to the value `ent` of the own block (i, i) of a
  // diagonal-E operator
  auto diage_face = [&](const Elem& el, int i, int ent) {
    double v = 0.0;
#pragma unroll
    for (int f = 0; f < NFACES; ++f) {
      const int si = sm.nodepos[i][f];
      if (si < 0) continue;
      v += el.sgn[f] * sm.wface[si] * (&el.dFo[f][el.kslot[f][si]][0][0])[ent];
    }
    return v;
  };
  // implicit-Euler globalization (applyEuler, globalization.jl): -M/tau_vec on the diagonal
  auto ptc_term = [&](const Elem& el, int i, int ent) {
    if (!ptc_scale || ent % (ND + 1) != 0) return 0.0;
    return ptc_diag[el.e * NP + i] * ptc_scale[mesh.el_inst ? mesh.el_inst[el.e] : 0];
  };

  if constexpr (VOL == VOL_WEAK) {
    // lane (j, ent): value ent of column j, for every row i in turn, so that a
    // row's run of NP blocks is stored by consecutive lanes
    constexpr int JE = NP * NB;
    for (int t = tid; t < nel * JE; t += T) {
      const int l = t / JE, je = t - l * JE, j = je / NB, ent = je - j * NB;
      const Elem& el = sm.el[l];
      double Aq[DIM];
#pragma unroll
      for (int d = 0; d < DIM; ++d) Aq[d] = (&el.A[j * DIM + d][0][0])[ent];
      if constexpr (Op::DIAGE) {
#pragma unroll 1
        for (int i = 0; i < NP; ++i) {
          double v = 0.0;
#pragma unroll
          for (int d = 0; d < DIM; ++d) v += sm.Q[d][j][i] * Aq[d];
          if (i == j) v = v + diage_face(el, i, ent) - ptc_term(el, i, ent);
          if (el.own_run[i] >= 0) vals[(el.own_run[i] + j) * NB + ent] = to_block<BT>(v);
        }
      } else {
        double P[NFACES][NF];
#pragma unroll
        for (int f = 0; f < NFACES; ++f) {
          const int sj = sm.nodepos[j][f];
#pragma unroll
          for (int k = 0; k < NF; ++k)
            P[f][k] = sj >= 0 ? sm.interp[sj][el.kown[f][k]] * (&el.dFo[f][k][0][0])[ent] : 0.0;
        }
#pragma unroll 1
        for (int i = 0; i < NP; ++i) {
          double v = 0.0;
#pragma unroll
          for (int d = 0; d < DIM; ++d) v += sm.Q[d][j][i] * Aq[d];
#pragma unroll
          for (int f = 0; f < NFACES; ++f) {
#pragma unroll
            for (int k = 0; k < NF; ++k) v += el.cw[f][i][k] * P[f][k];
          }
          if (i == j) v -= ptc_term(el, i, ent);
          if (el.own_run[i] >= 0) vals[(el.own_run[i] + j) * NB + ent] = to_block<BT>(v);
        }
#pragma unroll
        for (int f = 0; f < NFACES; ++f) {
          const ElFace r = el.rec[f];
          if (r.x < 0) continue;
          const int sj = sbp.nodepos[j * NFACES + (r.z & 0xff)];
#pragma unroll
          for (int k = 0; k < NF; ++k)
            P[f][k] = sj >= 0 ? sm.interp[sj][el.knbr[f][k]] * (&el.dFn[f][k][0][0])[ent] : 0.0;
#pragma unroll 1
          for (int i = 0; i < NP; ++i) {
            double v = 0.0;
#pragma unroll
            for (int k = 0; k < NF; ++k) v += el.cw[f][i][k] * P[f][k];
            if (el.nbr_run[f][i] >= 0) vals[(el.nbr_run[f][i] + j) * NB + ent] = to_block<BT>(v);
          }
        }
      }
    }
  } else {
    // split form: res_i -= sum_k 2 S_ik F*(q_i, q_k).  With D the derivative
    // with respect to q_c of the flux of the pair (c, r) in the direction
    // sum_d 2 S_d[c][r] dxidx_d, block (r, c) is +D and block (c, c) collects
    // -D.  Thread (c, part) takes the rows r = part, part + KP, ...
    constexpr int KP = Elem::KP;
    for (int t = tid; t < nel * NP * KP; t += T) {
      const int l = t / (NP * KP), x = t - l * (NP * KP), c = x / KP, part = x - c * KP;
      Elem& el = sm.el[l];
      dual<ND> zc[ND];
#pragma unroll
      for (int a = 0; a < ND; ++a) {
        zc[a].v = el.z[c][a];
#pragma unroll
        for (int b = 0; b < ND; ++b) zc[a].d[b] = el.dz[c][a][b];
      }
      double dg[ND][ND];
#pragma unroll
      for (int a = 0; a < ND; ++a)
#pragma unroll
        for (int b = 0; b < ND; ++b) dg[a][b] = 0.0;
      for (int r = part; r < NP; r += KP) {
        if (r == c) continue;
        const double* mt = metric<DIM, NP>(mesh, el.e, r > c ? r : c);
        double n[DIM], zr[ND];
#pragma unroll
        for (int y = 0; y < DIM; ++y) {
          n[y] = 0.0;
#pragma unroll
          for (int d = 0; d < DIM; ++d) n[y] += (sm.Q[d][c][r] - sm.Q[d][r][c]) * mt[y * DIM + d];
        }
#pragma unroll
        for (int a = 0; a < ND; ++a) zr[a] = el.z[r][a];
        dual<ND> F[ND];
        ir_flux_z<DIM, 1>(phys, zc, zr, n, F);
        double B[ND][ND];
#pragma unroll
        for (int a = 0; a < ND; ++a)
#pragma unroll
          for (int b = 0; b < ND; ++b) {
            dg[a][b] -= F[a].d[b];
            B[a][b] = F[a].d[b];
          }
        if constexpr (ES) {
          const JacView<Op, VOL, FLUX, EPB> vw(sm, el);
#pragma unroll
          for (int f = 0; f < NFACES; ++f) {
            const int sr = sm.nodepos[r][f], sc = sm.nodepos[c][f];
            if (sr < 0 || sc < 0) continue;
            es_own_face<Op>(vw, sbp, mesh, phys, qin, f, r, c, sr, sc, B);
          }
        }
        if (el.own_run[r] >= 0) {
          BT* dst = vals + (el.own_run[r] + c) * NB;
#pragma unroll
          for (int a = 0; a < ND; ++a)
#pragma unroll
            for (int b = 0; b < ND; ++b) dst[a * ND + b] = to_block<BT>(B[a][b]);
        }
      }
      if constexpr (ES) {
        if (part == 0) {
          const JacView<Op, VOL, FLUX, EPB> vw(sm, el);
#pragma unroll
          for (int f = 0; f < NFACES; ++f) {
            const int sc = sm.nodepos[c][f];
            if (sc >= 0) es_own_face<Op>(vw, sbp, mesh, phys, qin, f, c, c, sc, sc, dg);
          }
        }
      }
#pragma unroll
      for (int a = 0; a < ND; ++a)
#pragma unroll
        for (int b = 0; b < ND; ++b) el.diag[c][part][a][b] = dg[a][b];
    }
    __syncthreads();
    for (int t = tid; t < nel * NP * NB; t += T) {
      const int l = t / (NP * NB), c = (t - l * (NP * NB)) / NB, ent = t % NB;
      const Elem& el = sm.el[l];
      double v = 0.0;
#pragma unroll
      for (int k = 0; k < KP; ++k) v += (&el.diag[c][k][0][0])[ent];
      if constexpr (Op::DIAGE) v += diage_face(el, c, ent);
      v -= ptc_term(el, c, ent);
      if (el.own_run[c] >= 0) vals[(el.own_run[c] + c) * NB + ent] = to_block<BT>(v);
    }
    if constexpr (ES) {
      for (int t = tid; t < nel * NFACES * NP * NP; t += T) {
        const int l = t / (NFACES * NP * NP), x = t - l * (NFACES * NP * NP);
        const int f = x / (NP * NP), i = (x / NP) % NP, jn = x % NP;
        const Elem& el = sm.el[l];
        if (el.rec[f].x < 0) continue;
        const int si = sm.nodepos[i][f], sj = sbp.nodepos[jn * NFACES + (el.rec[f].z & 0xff)];
        double B[ND][ND];
#pragma unroll
        for (int a = 0; a < ND; ++a)
#pragma unroll
          for (int b = 0; b < ND; ++b) B[a][b] = 0.0;
        if (si >= 0 && sj >= 0) {
          const JacView<Op, VOL, FLUX, EPB> vw(sm, el);
          eslf_nbr_block<Op>(vw, sbp, mesh, phys, qin, f, jn, si, sj, B);
        }
        if constexpr (!Op::DIAGE) {
          if (el.nbr_run[f][i] >= 0) {
            BT* dst = vals + (el.nbr_run[f][i] + jn) * NB;
#pragma unroll
            for (int a = 0; a < ND; ++a)
#pragma unroll
              for (int b = 0; b < ND; ++b) dst[a * ND + b] = to_block<BT>(B[a][b]);
          }
        }
      }
    }
  }
  if constexpr (Op::DIAGE) {
    // the blocks across the faces
    for (int t = tid; t < nel * SLOTS * NB; t += T) {
      const int l = t / (SLOTS * NB), x = t - l * (SLOTS * NB), slot = x / NB, ent = x - slot * NB;
      const int f = slot / NF, k = slot - f * NF;
      const Elem& el = sm.el[l];
      if (el.rec[f].x < 0 || el.nbr_run[f][k] < 0) continue;
      vals[el.nbr_run[f][k] * NB + ent] =
          to_block<BT>(el.sgn[f] * sm.wface[el.kown[f][k]] * (&el.dFn[f][k][0][0])[ent]);
    }
  }
}

// y = J x (BSR, block rows of ndof, FP32 or FP64 blocks, FP64 vectors):
// one thread per output dof; the threads of a block row read the block
// rows [a][0..ND) in turn, four of them (FP64: two) in flight, with the column
// numbers a round ahead.  Bound by memory where rows are many, by the latency of
// a round where they are few.  One block at a time, its column, then x: 101.8 us
// for 3D p=2, 6,000 tets, 276 MB of blocks, now 80.1 us (3.5 TB/s; six blocks
// 81.2, eight 85.6); 800 triangles p=1 8.4 -> 5.8 us; FP64, 882 triangles p=2
// 13.0 -> 8.7 us (four blocks 12.4).
template <int ND, class BT>
__global__ void __launch_bounds__(256)
bsr_spmv_kernel(int64_t nrows, const int64_t* __restrict__ rowptr, const int32_t* __restrict__ colind,
                const BT* __restrict__ vals, const double* __restrict__ x, double* __restrict__ y,
                double alpha, const double* __restrict__ yadd, double beta,
                const int32_t* __restrict__ el_list, int np,
                const int32_t* __restrict__ el_inst, const int32_t* __restrict__ mask) {
  const int64_t tt = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t rr = tt / ND;
  const int a = (int)(tt - rr * ND);
  if (rr >= nrows) return;
  // with an element list, launch row rr is node (rr % np) of element el_list[rr / np]
  const int64_t row = el_list ? (int64_t)el_list[rr / np] * np + (rr % np) : rr;
  // packed batches: rows of instances whose mask entry is 0 are left untouched
  if (mask && !mask[el_inst[row / np]]) return;
  const int64_t t = row * ND + a;
  double acc = 0.0;
  const int64_t b0 = rowptr[row], b1 = rowptr[row + 1];
  constexpr int U = sizeof(BT) == 8 ? 2 : 4;
  if (b0 < b1) {
    int32_t col[U];
#pragma unroll
    for (int u = 0; u < U; ++u) col[u] = colind[b0 + u < b1 ? b0 + u : b1 - 1];
    for (int64_t b = b0; b < b1; b += U) {
      BT m[U][ND];
      double xc[U][ND];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int64_t p = b + u < b1 ? b + u : b1 - 1;
#pragma unroll
        for (int c = 0; c < ND; ++c) {
          m[u][c] = vals[p * (ND * ND) + a * ND + c];
          xc[u][c] = x[(int64_t)col[u] * ND + c];
        }
      }
#pragma unroll
      for (int u = 0; u < U; ++u) col[u] = colind[b + U + u < b1 ? b + U + u : b1 - 1];
#pragma unroll
      for (int u = 0; u < U; ++u)
        if (b + u < b1) {
#pragma unroll
          for (int c = 0; c < ND; ++c) acc += (double)m[u][c] * xc[u][c];
        }
    }
  }
  double v = alpha * acc;
  if (yadd) v += beta * yadd[t];
  y[t] = v;
}

}  // namespace pdes
