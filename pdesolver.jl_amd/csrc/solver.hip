// solver.hip -- preconditioners, GMRES and Newton on the device (C ABI).
//
// NewtonBDiagPC (src/NonlinearSolvers/preconditioning_types.jl:41-110,
// preconditioning.jl:7-215): each element's diagonal (Np*ndof)^2 block of the
// Jacobian is inverted (the reference factors it with getrf and applies getrs;
// an explicit inverse makes the apply one coalesced product per element).
// Setup and apply run in FP32.
// GMRES(restart) with right preconditioning replaces the PETSc KSP of
// src/linearsolvers/ls_standard.jl:321-370 (KSP options read_input.jl:560-581);
// the Arnoldi basis, Hessenberg and update stay FP64.  Orthogonalisation is
// classical Gram-Schmidt applied twice (CGS2) in four launches per step, of
// which three read the basis.
// Newton follows newtonInner (src/NonlinearSolvers/newton.jl:137-304).
#include <algorithm>
#include <chrono>
#include <cstdlib>
#include <cmath>
#include <vector>

#include <hipcub/hipcub.hpp>

#include "jacobian.hpp"
#include "krylov_kernels.hpp"

struct pdes_precond {
  int kind = 0;
  int n = 0;                 // block size Np*nd
  float* d_inv = nullptr;    // inverse of each (modified) element block, laid out by InvLayout
  bool factored = false;
  // ILU(0): elements grouped by dependency level of the forward (lower
  // neighbours first) and backward (upper neighbours first) sweeps
  bool ilu_ready = false;
  std::vector<int64_t> fptr, bptr;
  int32_t* d_fel = nullptr;
  int32_t* d_bel = nullptr;
  int32_t* d_own = nullptr;   // per node row: offset of the element's own block run within the row
  // dependency-driven sweeps: the forward sweep's result (a vector of the
  // unknowns that holds ILU_PENDING between applications) and the ticket /
  // error / poll-limit words
  double* d_y = nullptr;
  int32_t* d_sync = nullptr;
  // sweep choice: 0 by the cost model, 1 always level by level
  // (PDES_ILU_LEVELS set), 2 always dependency-driven (PDES_ILU_DEP set)
  int force = 0;
  std::vector<int32_t> h_fl, h_bl;   // forward / backward level of each element
  // the dependency-driven sweeps' sets: the elements set by set, where each
  // set starts, and each element's place in that list
  struct Sets {
    int32_t* d_order = nullptr;
    int32_t* d_start = nullptr;
    int32_t* d_place = nullptr;
    int64_t n = 0;
  } fset, bset;
  // the sets of selected instances (packed batches), their counts, the selection flags and the select's work space
  int32_t* d_fsel = nullptr;
  int32_t* d_bsel = nullptr;
  int64_t sel_nf = 0, sel_nb = 0;
  int32_t* d_inst_sel = nullptr;
  int32_t* d_nsel = nullptr;
  void* d_select_tmp = nullptr;
  size_t select_tmp_bytes = 0;
  int sel_ninst = 0;
  double blk_per_el = 0;             // neighbour blocks of an element on one side (mean)
  // the 2 x levels sweep launches of one apply, captured once per (mask,
  // matrix) into a HIP graph over fixed staging vectors and replayed
  double* d_stage_in = nullptr;
  double* d_stage_out = nullptr;
  struct Graph {
    const int32_t* mask;
    const void* vals;
    bool fp64;
    const float* inv;
    hipGraphExec_t exec;
  };
  std::vector<Graph> graphs;
};

namespace pdes {

struct GmresWork;
void gmres_release(pdes_ctx* c);

int precond_free(pdes_ctx* c) {
  gmres_release(c);
  if (!c->pc_obj) return PDES_OK;
  if (c->pc_obj->d_inv) hipFree(c->pc_obj->d_inv);
  if (c->pc_obj->d_fel) hipFree(c->pc_obj->d_fel);
  if (c->pc_obj->d_bel) hipFree(c->pc_obj->d_bel);
  if (c->pc_obj->d_own) hipFree(c->pc_obj->d_own);
  if (c->pc_obj->d_y) hipFree(c->pc_obj->d_y);
  for (auto* k : {&c->pc_obj->fset, &c->pc_obj->bset})
    for (int32_t* p : {k->d_order, k->d_start, k->d_place})
      if (p) hipFree(p);
  if (c->pc_obj->d_fsel) hipFree(c->pc_obj->d_fsel);
  if (c->pc_obj->d_bsel) hipFree(c->pc_obj->d_bsel);
  if (c->pc_obj->d_inst_sel) hipFree(c->pc_obj->d_inst_sel);
  if (c->pc_obj->d_nsel) hipFree(c->pc_obj->d_nsel);
  if (c->pc_obj->d_select_tmp) hipFree(c->pc_obj->d_select_tmp);
  if (c->pc_obj->d_sync) hipFree(c->pc_obj->d_sync);
  if (c->pc_obj->d_stage_in) hipFree(c->pc_obj->d_stage_in);
  if (c->pc_obj->d_stage_out) hipFree(c->pc_obj->d_stage_out);
  for (auto& g : c->pc_obj->graphs) hipGraphExecDestroy(g.exec);
  delete c->pc_obj;
  c->pc_obj = nullptr;
  return PDES_OK;
}

// lanes per row of the sweeps.  A wave holds 64 / lanes whole rows, so an
// element of N rows takes ilu_waves() waves; the lanes are chosen so that a
// lane's share of a row (N / lanes inverse entries and its neighbour blocks)
// leaves room for a few elements' shares in registers, and small elements fit
// one wave.  Dense faces (up to 45 neighbour blocks a row) need more lanes than
// diagonal-E ones (at most 3).  3D p=2 (50 rows): with four lanes the sweep
// spilled, 276 us for both triangles of a 10^3 cube, five take 212 us.
template <int N, bool DIAGE>
constexpr int ilu_lanes() {
  if (DIAGE) return N <= 28 ? 2 : N <= 64 ? 1 : 2;
  return N <= 12 ? 5 : N <= 20 ? 3 : N <= 24 ? 2 : N <= 40 ? 3 : N <= 50 ? 5 : 4;
}
template <int N, bool DIAGE>
constexpr int ilu_waves() {
  return (N + 64 / ilu_lanes<N, DIAGE>() - 1) / (64 / ilu_lanes<N, DIAGE>());
}

// whether the blocks of size n belong to a diagonal-E operator
constexpr bool diage_block(int n) {
  bool diage = false;
#define PDES_DIAGE_BLOCK(D_, NP_, NF_, NS_, DE_) \
  if (NP_ * (D_ + 2) == n) diage = DE_;
  PDES_FOR_EACH_SHAPE(PDES_DIAGE_BLOCK)
#undef PDES_DIAGE_BLOCK
  return diage;
}

// Where entry (r, c) of an element's inverse is stored.  Dense-face operators:
// column-major.  Diagonal-E: four of a sweep lane's columns (l, l + LPR, ...)
// together, [column / (4 LPR)][row][lane][4], so that a lane reads its share of
// a row 16 bytes at a time and a wave reads them in order: the sweeps keep a
// few elements' shares in flight, and a wave can have 63 loads outstanding,
// which 48 to 108 single entries an element would use up.
template <int N>
struct InvLayout {
  static constexpr bool VEC4 = diage_block(N);
  static constexpr int LPR = ilu_lanes<N, VEC4>();
  static constexpr int NC = (N + LPR - 1) / LPR;              // columns per lane
  static constexpr int NCP = VEC4 ? (NC + 3) / 4 * 4 : NC;    // and with the padding
  static constexpr int SIZE = VEC4 ? NCP * LPR * N : N * N;
  static __host__ __device__ constexpr int at(int r, int c) {
    return VEC4 ? (c / (4 * LPR) * (N * LPR) + r * LPR + c % LPR) * 4 + c / LPR % 4 : c * N + r;
  }
};

// ---------------------------------------------------------------------------
// block-Jacobi setup: each element's block is gathered from the BSR matrix
// (FP32) and inverted in place by Gauss-Jordan elimination with partial (row)
// pivoting; the inverse is stored so that the apply is a coalesced
// matrix-vector product (InvLayout).
//
// A chain of N pivots, so what bounds it is the latency of one step, not its
// flops.  The block lives in registers: G x G threads, thread (tr, tc) holds
// the rows tr + G i and the columns tc + G j (one wave for N <= 32, where the
// barriers cost nothing, four beyond).  A step puts the pivot column in LDS,
// every wave finds the pivot for itself (rows are never moved: a row's place
// in the interchanged matrix is tracked instead), the pivot row's threads put
// the scaled row in LDS, and all update: two barriers a step, about 0.5 us.
// With the block in LDS and its rows moved a step took eight barriers and
// 1.9 us.  One level of the ILU(0) factorization, same bits (MI355X): 48 x 48
// blocks (2D diagonal-E p=2, 37 elements) 106 -> 36 us, 50 x 50 (3D Omega
// p=2, 150 elements) 243 -> 87 us, 72 x 72 230 -> 70 us, 12 x 12 34 -> 17 us.
// ---------------------------------------------------------------------------
template <int N>
struct GjShape {
  static constexpr int G = N <= 32 ? 8 : 16;
  static constexpr int R = (N + G - 1) / G;      // rows and columns per thread
  static constexpr int THREADS = G * G;
};

// max over the 64 lanes of a wave, in every lane
__device__ __forceinline__ uint32_t wave_max_u32(uint32_t x) {
  auto step = [&](uint32_t y) { x = y > x ? y : x; };
  step((uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x111, 0xf, 0xf, false));   // row_shr:1
  step((uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x112, 0xf, 0xf, false));   // row_shr:2
  step((uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x114, 0xf, 0xf, false));   // row_shr:4
  step((uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x118, 0xf, 0xf, false));   // row_shr:8
  step((uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x142, 0xa, 0xf, false));   // row_bcast:15
  step((uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x143, 0xc, 0xf, false));   // row_bcast:31
  return (uint32_t)__builtin_amdgcn_readlane((int)x, 63);
}

template <int N>
struct GjSmem {
  static constexpr int NPAD = GjShape<N>::G * GjShape<N>::R;   // rows beyond N hold zeros
  float fcol[2][NPAD];   // pivot column, alternate steps
  float prow[2][NPAD];   // scaled pivot row
  int pos[N];            // final place of each stored row
  int row_at[N];         // its inverse
};

// Inverts the block held in a (thread (tr, tc), see above; zero beyond N) and
// stores it.  Every thread of the workgroup calls it.
template <int N>
__device__ __forceinline__ void gauss_jordan_inverse(float (&a)[GjShape<N>::R][GjShape<N>::R], GjSmem<N>& sh,
                                                     float* __restrict__ out, int32_t* __restrict__ err) {
  constexpr int G = GjShape<N>::G, R = GjShape<N>::R;
  constexpr int LR = (N + 63) / 64;              // rows per lane in the pivot search
  const int tid = threadIdx.x, lane = tid & 63;
  const int tr = tid % G, tc = tid / G;
  int pos[LR];                                   // place of rows lane + 64 u in the interchanged matrix
#pragma unroll
  for (int u = 0; u < LR; ++u) pos[u] = lane + 64 * u < N ? lane + 64 * u : -1;
  bool singular = false;
  // k = kj G + kt: the register that holds column k is known at compile time
#pragma unroll
  for (int kj = 0; kj < R; ++kj) {
    const int kt_n = N - kj * G < G ? N - kj * G : G;
    for (int kt = 0; kt < kt_n; ++kt) {
      const int k = kj * G + kt;
      float* const fcol = sh.fcol[k & 1];
      float* const prow = sh.prow[k & 1];
      if (tc == kt) {
#pragma unroll
        for (int i = 0; i < R; ++i) fcol[tr + G * i] = a[i][kj];
      }
      __syncthreads();
      // pivot: max |column k| over the rows at places >= k, lowest place on
      // ties; a NaN is never chosen.  Keys are the value's bits plus one, 0
      // for rows that do not take part.
      uint32_t key = 0;
      int kpos = N, krow = 0;
      float kval = 0.0f;
#pragma unroll
      for (int u = 0; u < LR; ++u) {
        const int r = lane + 64 * u;
        const float x = fcol[r < N ? r : 0], v = fabsf(x);
        const uint32_t q = (pos[u] >= k && v >= 0.0f) ? __float_as_uint(v) + 1u : 0u;
        const bool take = q > key || (q == key && pos[u] < kpos);
        key = take ? q : key;
        kpos = take ? pos[u] : kpos;
        krow = take ? r : krow;
        kval = take ? x : kval;
      }
      const uint32_t best = wave_max_u32(key);
      uint64_t cand = __ballot(key == best);
      int l = __builtin_ctzll(cand);
      if (best == 0) {                           // a column of NaN: the row in place k
#pragma unroll
        for (int u = 0; u < LR; ++u) {
          const uint64_t at = __ballot(pos[u] == k);
          if (at) {
            l = __builtin_ctzll(at);
            krow = lane + 64 * u;
            kpos = k;
            kval = fcol[krow < N ? krow : 0];
          }
        }
      } else if (cand & (cand - 1)) {
        int ppos = __builtin_amdgcn_readlane(kpos, l);
        for (cand &= cand - 1; cand; cand &= cand - 1) {
          const int m = __builtin_ctzll(cand);
          const int q = __builtin_amdgcn_readlane(kpos, m);
          if (q < ppos) { ppos = q; l = m; }
        }
      }
      const int p = __builtin_amdgcn_readlane(krow, l);
      const int ppos = __builtin_amdgcn_readlane(kpos, l);
      const float pivot = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(kval), l));
      singular |= best <= 1;                     // zero pivot
#pragma unroll
      for (int u = 0; u < LR; ++u)               // rows k and ppos of the interchanged matrix swap
        pos[u] = lane + 64 * u == p ? k : pos[u] == k ? ppos : pos[u];
      const float pinv = 1.0f / pivot;
      const int pt = p % G, pi = p / G;
      if (tr == pt) {
        float v[R];
#pragma unroll
        for (int j = 0; j < R; ++j) {
          v[j] = a[0][j];
#pragma unroll
          for (int i = 1; i < R; ++i) v[j] = pi == i ? a[i][j] : v[j];
          v[j] = v[j] * pinv;
        }
        v[kj] = tc == kt ? pinv : v[kj];
#pragma unroll
        for (int j = 0; j < R; ++j) prow[tc + G * j] = v[j];
      }
      __syncthreads();
      float f[R], pr[R];
#pragma unroll
      for (int i = 0; i < R; ++i) f[i] = fcol[tr + G * i];
#pragma unroll
      for (int j = 0; j < R; ++j) pr[j] = prow[tc + G * j];
#pragma unroll
      for (int i = 0; i < R; ++i) {
        a[i][kj] = tc == kt ? 0.0f : a[i][kj];
        const bool is_p = tr + G * i == p;
#pragma unroll
        for (int j = 0; j < R; ++j) {
          float x = a[i][j];
          x -= f[i] * pr[j];
          a[i][j] = is_p ? pr[j] : x;
        }
      }
    }
  }
  if (singular && tid == 0) err[0] = 1;
  // row r of the array is row pos[r] of the inverse, and column c the column
  // of the row that ended in place c
  if (tid < 64) {
#pragma unroll
    for (int u = 0; u < LR; ++u)
      if (lane + 64 * u < N) {
        sh.pos[lane + 64 * u] = pos[u];
        sh.row_at[pos[u]] = lane + 64 * u;
      }
  }
  __syncthreads();
#pragma unroll
  for (int j = 0; j < R; ++j) {
    if (tc + G * j >= N) continue;
    const int col = sh.row_at[tc + G * j];
#pragma unroll
    for (int i = 0; i < R; ++i)
      if (tr + G * i < N) out[InvLayout<N>::at(sh.pos[tr + G * i], col)] = a[i][j];
  }
}

template <int NP, int ND, class BT>
__device__ __forceinline__ void load_own_block(const BT* __restrict__ vals, const int64_t* run,
                                               float (&a)[GjShape<NP * ND>::R][GjShape<NP * ND>::R]) {
  constexpr int N = NP * ND, G = GjShape<N>::G, R = GjShape<N>::R;
  const int tr = threadIdx.x % G, tc = threadIdx.x / G;
#pragma unroll
  for (int i = 0; i < R; ++i)
#pragma unroll
    for (int j = 0; j < R; ++j) {
      const int r = tr + G * i, c = tc + G * j;
      a[i][j] = 0.0f;
      if (r < N && c < N && run[r / ND] >= 0)
        a[i][j] = (float)vals[(run[r / ND] + c / ND) * (ND * ND) + (r % ND) * ND + c % ND];
    }
}

template <int NP, int ND, class BT>
__global__ void __launch_bounds__(GjShape<NP * ND>::THREADS)
bjacobi_factor_kernel(const int32_t* __restrict__ el_list, const int64_t* __restrict__ rowptr,
                      const int32_t* __restrict__ colind, const BT* __restrict__ vals, float* __restrict__ inv,
                      int32_t* __restrict__ err) {
  constexpr int N = NP * ND;
  __shared__ GjSmem<N> sh;
  __shared__ int64_t run[NP];
  const int64_t e = el_list ? (int64_t)el_list[blockIdx.x] : (int64_t)blockIdx.x;
  for (int i = threadIdx.x; i < NP; i += blockDim.x) run[i] = bsr_find(rowptr, colind, e * NP + i, (int32_t)(e * NP));
  __syncthreads();
  float a[GjShape<N>::R][GjShape<N>::R];
  load_own_block<NP, ND>(vals, run, a);
  // The entries are values from here on, not loads whose addresses the unrolled
  // pivots may still hold: without this the kernel took 231 registers for 50 and
  // 60 unknowns (4 x 4 entries a thread) and spilled up to 516 bytes a lane for 72
  // (5 x 5), now 37 to 59.  Set-up, FP32 blocks, 32,768 triangles: Omega p=4 3256
  // -> 1106 us, diagonal-E p=3 10,400 -> 1890 us (FP64 blocks 16,190 -> 1938);
  // 16,464 tets p=2 1389 -> 512 us.  The other sizes take 22 to 85 registers
  // without it, and 108 unknowns 7% longer with it.
  if constexpr (GjShape<N>::R == 4 || GjShape<N>::R == 5) {
#pragma unroll
    for (auto& row : a)
#pragma unroll
      for (float& x : row) asm volatile("" : "+v"(x));
  }
  gauss_jordan_inverse<N>(a, sh, inv + e * InvLayout<N>::SIZE, err);
}

// block-Jacobi apply: x_e = inv_e b_e; EPB = 256 / N elements per block, thread
// (element slot, row r) forms one row of the product (consecutive rows read
// consecutive words of the inverse).
template <int NP, int ND>
__global__ void __launch_bounds__(256)
bjacobi_apply_kernel(const int32_t* __restrict__ el_list, int64_t nel, const float* __restrict__ inv,
                     const double* __restrict__ b, double* __restrict__ x, const int32_t* __restrict__ el_inst,
                     const int32_t* __restrict__ mask) {
  constexpr int N = NP * ND;
  constexpr int EPB = 256 / N;
  __shared__ float v[EPB][N];
  const int slot = threadIdx.x / N;
  const int r = threadIdx.x - slot * N;
  const int64_t s = (int64_t)blockIdx.x * EPB + slot;
  bool act = slot < EPB && s < nel;
  int64_t e = 0;
  if (act) {
    e = el_list ? (int64_t)el_list[s] : s;
    if (mask && !mask[el_inst[e]]) act = false;
  }
  if (act) v[slot][r] = (float)b[e * N + r];
  __syncthreads();
  if (!act) return;
  const float* M = inv + e * InvLayout<N>::SIZE;
  float acc = 0.0f;
#pragma unroll
  for (int cc = 0; cc < N; ++cc) acc += M[InvLayout<N>::at(r, cc)] * v[slot][cc];
  x[e * N + r] = (double)acc;
}

// ---------------------------------------------------------------------------
// Element-block ILU(0) in the natural element order.  With E the element
// blocks of the Jacobian, L/U its strictly lower/upper element blocks and
//   D'_e = A_ee - sum_{k in lower(e)} A_ek D'_k^-1 A_ke,
// the preconditioner is M = (D' + L) D'^-1 (D' + U); no fill outside the
// element-block pattern is kept (ILU(0) on element blocks).  A_ek couples only
// the face-stencil nodes of e and of its neighbour k, so the update of D'_e
// touches only the (stencil x stencil) part of the block:
//   C = S_ek [D'_k^-1]_(Rk,Rk) S_ke,  Rk / Ce = stencil nodes of the face.
// Elements are processed level by level (a level holds elements whose lower
// neighbours are all in earlier levels), each level in one launch.
// ---------------------------------------------------------------------------
//
// The products run on the threads and registers of the elimination: thread
// (tr, tc) forms the entries that it holds, from operands in LDS.  A block's
// place in its row is read off the row's layout (lower neighbours, the NP own
// blocks from own[row] on, upper neighbours) instead of searched for, and the
// three operands of a face are loaded together, the next lower face's while this
// one's products are formed (3D p=2 levels of 150 elements 88.5 -> 82.4 us; the
// rest is the products, 2 x 50^3 a face, and the elimination).
template <int NP, int ND, int NS, bool DIAGE, class BT>
__global__ void __launch_bounds__(GjShape<NP * ND>::THREADS)
ilu_factor_level_kernel(const int32_t* __restrict__ lev_el, const int64_t* __restrict__ rowptr,
                        const int32_t* __restrict__ colind, const int32_t* __restrict__ own,
                        const BT* __restrict__ vals, const pdes::ElFace* __restrict__ elface,
                        const int32_t* __restrict__ perm, const int32_t* __restrict__ nodepos,
                        float* __restrict__ inv, int32_t* __restrict__ err, const int32_t* __restrict__ el_inst,
                        const int32_t* __restrict__ inst_active) {
  constexpr int N = NP * ND;
  constexpr int M = NS * ND;
  constexpr int G = GjShape<N>::G, R = GjShape<N>::R, RM = (M + G - 1) / G;
  constexpr int T = GjShape<N>::THREADS, LM = (M * M + T - 1) / T;
  static_assert(DIAGE || NS == NP, "dense faces couple all nodes of both elements");
  __shared__ float B1[M][M + 1];
  __shared__ float B2[M][M + 1];
  __shared__ float B3[M][M + 1];
  __shared__ float B4[M][M + 1];
  __shared__ GjSmem<N> sh;
  constexpr int NFACES = ND - 1, PLACES = NS * (DIAGE ? NS : 1);
  __shared__ int Ce[NFACES][NS], Rk[NFACES][NS];
  __shared__ int64_t run[NP];
  __shared__ int64_t at_ke[NFACES][PLACES], at_ek[NFACES][PLACES];
  const int tid = threadIdx.x;
  const int tr = tid % G, tc = tid / G;
  const int64_t e = lev_el[blockIdx.x];
  if (inst_active && !inst_active[el_inst[e]]) return;
  for (int i = tid; i < NP; i += T) run[i] = rowptr[e * NP + i] + own[e * NP + i];
  __syncthreads();
  float a[R][R];
  load_own_block<NP, ND>(vals, run, a);
  // where the blocks (row, first + node) of a neighbour element begin (dense
  // faces: NP blocks in a run) or the one block (row, first + node) is
  // (diagonal-E); -1 if absent
  auto place = [&](int64_t row, bool lower, int64_t first, int node) -> int64_t {
    const int64_t p0 = rowptr[row], o = own[row];
    const int64_t b = lower ? p0 : p0 + o + NP, n = lower ? p0 + o : rowptr[row + 1];
    const int32_t want = (int32_t)(first + (DIAGE ? node : 0));
    int64_t q = -1;
    for (int64_t p = b; p < n; p += DIAGE ? 1 : NP)
      if (colind[p] == want) q = p;
    return q;
  };
  // the places of all lower faces' blocks, looked up side by side
  for (int t = tid; t < NFACES * PLACES; t += T) {
    const int f = t / PLACES, x = t - f * PLACES;
    const pdes::ElFace r = elface[e * NFACES + f];
    if (r.x < 0 || r.x >= e) continue;
    const int64_t k = r.x;
    const int fk = r.z & 0xff;
    if (x < NS) {
      Ce[f][x] = perm[x * NFACES + f];
      Rk[f][x] = perm[x * NFACES + fk];
    }
    const int s1 = DIAGE ? x / NS : x, s2 = DIAGE ? x % NS : 0;
    at_ke[f][x] = place(k * NP + perm[s1 * NFACES + fk], false, e * NP, perm[s2 * NFACES + f]);
    at_ek[f][x] = place(e * NP + perm[s1 * NFACES + f], true, k * NP, perm[s2 * NFACES + fk]);
  }
  __syncthreads();
  // B1 = [D'_k^-1](Rk,Rk), B2 = S_ke = A(k rows Rk, e cols Ce), B4 = S_ek = A(e rows Ce, k cols Rk);
  // the next lower face's are loaded while this one's products are formed
  float v1[LM], v2[LM], v4[LM];
  auto load = [&](int f) {
    const float* Ik = inv + (int64_t)elface[e * NFACES + f].x * InvLayout<N>::SIZE;
#pragma unroll
    for (int u = 0; u < LM; ++u) {
      const int t = tid + u * T;
      v1[u] = v2[u] = v4[u] = 0.0f;
      if (t < M * M) {
        const int r1 = t / M, c1 = t - r1 * M;
        const int s1 = r1 / ND, x = r1 - s1 * ND, s2 = c1 / ND, y = c1 - s2 * ND;
        v1[u] = Ik[InvLayout<N>::at(Rk[f][s2] * ND + y, Rk[f][s1] * ND + x)];   // transposed: lanes along a column
        const int at = DIAGE ? s1 * NS + s2 : s1;
        const int64_t q2 = at_ke[f][at], q4 = at_ek[f][at];
        if (q2 >= 0) v2[u] = (float)vals[(q2 + (DIAGE ? 0 : Ce[f][s2])) * (ND * ND) + x * ND + y];
        if (q4 >= 0) v4[u] = (float)vals[(q4 + (DIAGE ? 0 : Rk[f][s2])) * (ND * ND) + x * ND + y];
      }
    }
  };
  // the next face from f on with a lower neighbour (uniform over the block)
  auto lower = [&](int f) {
    while (f < NFACES) {
      const int32_t k = elface[e * NFACES + f].x;
      if (k >= 0 && k < e) break;
      ++f;
    }
    return f;
  };
  int f = lower(0);
  if (f < NFACES) load(f);
  while (f < NFACES) {
#pragma unroll
    for (int u = 0; u < LM; ++u) {
      const int t = tid + u * T;
      if (t < M * M) {
        const int r1 = t / M, c1 = t - r1 * M;
        B1[c1][r1] = v1[u];
        B2[r1][c1] = v2[u];
        B4[r1][c1] = v4[u];
      }
    }
    __syncthreads();
    const int next = lower(f + 1);
    if (next < NFACES) load(next);
    float acc[RM][RM];
#pragma unroll
    for (int i = 0; i < RM; ++i)
#pragma unroll
      for (int j = 0; j < RM; ++j) acc[i][j] = 0.0f;
#pragma unroll (M >= 40 ? 4 : 1)
    for (int l = 0; l < M; ++l) {
      float u[RM], w[RM];
#pragma unroll
      for (int i = 0; i < RM; ++i) u[i] = tr + G * i < M ? B1[tr + G * i][l] : 0.0f;
#pragma unroll
      for (int j = 0; j < RM; ++j) w[j] = tc + G * j < M ? B2[l][tc + G * j] : 0.0f;
#pragma unroll
      for (int i = 0; i < RM; ++i)
#pragma unroll
        for (int j = 0; j < RM; ++j) acc[i][j] += u[i] * w[j];
    }
#pragma unroll
    for (int i = 0; i < RM; ++i)
#pragma unroll
      for (int j = 0; j < RM; ++j)
        if (tr + G * i < M && tc + G * j < M) B3[tr + G * i][tc + G * j] = acc[i][j];
    __syncthreads();
    // D'_e -= S_ek B3 on the rows and columns of the face's stencil nodes
    int ri[R], cj[R];
#pragma unroll
    for (int i = 0; i < R; ++i) {
      const int rr = tr + G * i, cc = tc + G * i;
      const int sr = rr < N ? nodepos[(rr / ND) * NFACES + f] : -1, sc = cc < N ? nodepos[(cc / ND) * NFACES + f] : -1;
      ri[i] = sr >= 0 ? sr * ND + rr % ND : -1;
      cj[i] = sc >= 0 ? sc * ND + cc % ND : -1;
    }
    float upd[R][R];
#pragma unroll
    for (int i = 0; i < R; ++i)
#pragma unroll
      for (int j = 0; j < R; ++j) upd[i][j] = 0.0f;
#pragma unroll (M >= 40 ? 4 : 1)
    for (int l = 0; l < M; ++l) {
      float u[R], w[R];
#pragma unroll
      for (int i = 0; i < R; ++i) u[i] = ri[i] >= 0 ? B4[ri[i]][l] : 0.0f;
#pragma unroll
      for (int j = 0; j < R; ++j) w[j] = cj[j] >= 0 ? B3[l][cj[j]] : 0.0f;
#pragma unroll
      for (int i = 0; i < R; ++i)
#pragma unroll
        for (int j = 0; j < R; ++j) upd[i][j] += u[i] * w[j];
    }
#pragma unroll
    for (int i = 0; i < R; ++i)
#pragma unroll
      for (int j = 0; j < R; ++j)
        if (ri[i] >= 0 && cj[j] >= 0) a[i][j] -= upd[i][j];
    __syncthreads();
    f = next;
  }
  gauss_jordan_inverse<N>(a, sh, inv + e * InvLayout<N>::SIZE, err);
}

// The two sums of a sweep's row, in the order that every sweep kernel uses: a
// neighbour block's product first on its own, then added to the row's (short
// chains of dependent operations), and the row of the inverse over four partial
// sums.
template <int ND, class BT>
__device__ __forceinline__ double block_dot(const BT* blk, const double* x) {
  double d = (double)blk[0] * x[0];
#pragma unroll
  for (int c = 1; c < ND; ++c) d += (double)blk[c] * x[c];
  return d;
}
// sum over u < NC of m(u) * v(u); u past the row's end is skipped by `in`
template <int NC, class FM, class FV, class FI>
__device__ __forceinline__ float row_dot(FM m, FV v, FI in) {
  float y[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int u = 0; u < NC; ++u)
    if (in(u)) y[u & 3] += m(u) * v(u);
  return (y[0] + y[1]) + (y[2] + y[3]);
}

// One level of a sweep.  Forward: x_e = D'_e^-1 (b_e - sum_{k<e} A_ek x_k).
// Backward (in place on x): x_e -= D'_e^-1 sum_{k>e} A_ek x_k.  The neighbour
// products walk the element's BSR rows and keep the blocks whose column
// element is below (forward) or above (backward) e.
template <int NP, int ND, class BT>
__global__ void __launch_bounds__(256)
ilu_sweep_level_kernel(const int32_t* __restrict__ lev_el, int64_t count, const int64_t* __restrict__ rowptr,
                       const int32_t* __restrict__ colind, const int32_t* __restrict__ own,
                       const BT* __restrict__ vals, const float* __restrict__ inv,
                       const double* __restrict__ b, double* __restrict__ x, int forward,
                       const int32_t* __restrict__ el_inst, const int32_t* __restrict__ mask,
                       const int32_t* __restrict__ inst_active) {
  constexpr int N = NP * ND;
  constexpr int EPB = 256 / N;
  // entries of this row of D'_e^-1 loaded before the neighbour products, so
  // their latency overlaps with that dependent chain (all of them up to 72
  // per row, the first 32 beyond)
  constexpr int PF = N <= 72 ? N : 32;
  __shared__ float v[EPB][N];
  const int slot = threadIdx.x / N;
  const int r = threadIdx.x - slot * N;
  const int64_t s = (int64_t)blockIdx.x * EPB + slot;
  bool act = slot < EPB && s < count;
  int64_t e = 0;
  if (act) {
    e = lev_el[s];
    const int inst = el_inst ? el_inst[e] : 0;
    if ((mask && !mask[inst]) || (inst_active && !inst_active[inst])) act = false;
  }
  float mrow[PF];
  if (act) {
    const float* Mi = inv + e * InvLayout<N>::SIZE;
#pragma unroll
    for (int cc = 0; cc < PF; ++cc) mrow[cc] = Mi[InvLayout<N>::at(r, cc)];
  }
  if (act) {
    const int i = r / ND, a = r - i * ND;
    const int64_t row = e * NP + i;
    double acc = forward ? b[e * N + r] : 0.0;
    // columns are sorted: lower-element blocks precede the element's own run
    // of NP blocks (starting at own[row] within the row), upper-element
    // blocks follow it; fixed trip counts so the loads pipeline
    const int64_t p0 = rowptr[row], p1 = rowptr[row + 1];
    const int64_t q0 = forward ? p0 : p0 + own[row] + NP;
    const int64_t q1 = forward ? p0 + own[row] : p1;
    double t = 0.0;
#pragma unroll 4
    for (int64_t p = q0; p < q1; ++p)
      t += block_dot<ND>(vals + p * ND * ND + a * ND, x + (int64_t)colind[p] * ND);
    acc = forward ? acc - t : acc + t;
    v[slot][r] = (float)acc;
  }
  __syncthreads();
  if (!act) return;
  const float* Mi = inv + e * InvLayout<N>::SIZE;
  const float y = row_dot<N>([&](int u) { return u < PF ? mrow[u < PF ? u : 0] : Mi[InvLayout<N>::at(r, u)]; },
                             [&](int u) { return v[slot][u]; }, [](int) { return true; });
  if (forward) x[e * N + r] = (double)y;
  else x[e * N + r] -= (double)y;
}

// The same level with LPR lanes per row, for dense face stencils (a row has
// tens of neighbour blocks): lane l of row r takes the blocks q0 + l,
// q0 + l + LPR, ... and the columns cc = l, l + LPR, ... of D'_e^-1; the
// partial sums meet in LDS and are added in lane order, so the bits do not
// depend on the level's width or on the other instances of a batch.
template <int NP, int ND, class BT, int LPR>
__global__ void __launch_bounds__(256)
ilu_sweep_level_ml_kernel(const int32_t* __restrict__ lev_el, int64_t count, const int64_t* __restrict__ rowptr,
                          const int32_t* __restrict__ colind, const int32_t* __restrict__ own,
                          const BT* __restrict__ vals, const float* __restrict__ inv,
                          const double* __restrict__ b, double* __restrict__ x, int forward,
                          const int32_t* __restrict__ el_inst, const int32_t* __restrict__ mask,
                          const int32_t* __restrict__ inst_active) {
  constexpr int N = NP * ND;
  constexpr int TPE = N * LPR;
  static_assert(TPE <= 256, "one element's rows must fit a workgroup");
  constexpr int EPB = 256 / TPE;
  __shared__ double tp[EPB][N][LPR];
  __shared__ float yp[EPB][N][LPR];
  __shared__ float v[EPB][N];
  const int slot = threadIdx.x / TPE;
  const int t = threadIdx.x - slot * TPE;
  const int r = t / LPR, l = t - r * LPR;
  const int64_t s = (int64_t)blockIdx.x * EPB + slot;
  bool act = slot < EPB && s < count;
  int64_t e = 0;
  if (act) {
    e = lev_el[s];
    const int inst = el_inst ? el_inst[e] : 0;
    if ((mask && !mask[inst]) || (inst_active && !inst_active[inst])) act = false;
  }
  // this lane's entries of D'_e^-1 (columns l, l + LPR, ...) and the
  // right-hand side are loaded before the neighbour products, so their
  // latency overlaps with that dependent chain; diagonal-E 16 bytes at a time,
  // as InvLayout has them (a Krylov step of 45,000 triangles numbered at random,
  // p=4, 2757 us one entry at a time, 2430 us so; p=3 1485 and 1323 us)
  constexpr int NC = (N + LPR - 1) / LPR;
  constexpr bool VEC4 = InvLayout<N>::VEC4;
  float mrow[VEC4 ? InvLayout<N>::NCP : NC];
  double bval = 0.0;
  if (act) {
    const float* Mi = inv + e * InvLayout<N>::SIZE;
    if constexpr (VEC4) {
#pragma unroll
      for (int k = 0; k < InvLayout<N>::NCP; k += 4) {
        const float4 m4 = *reinterpret_cast<const float4*>(Mi + (k / 4 * (N * LPR) + r * LPR + l) * 4);
        mrow[k] = m4.x;
        mrow[k + 1] = m4.y;
        mrow[k + 2] = m4.z;
        mrow[k + 3] = m4.w;
      }
    } else {
#pragma unroll
      for (int k = 0; k < NC; ++k)
        if (l + k * LPR < N) mrow[k] = Mi[InvLayout<N>::at(r, l + k * LPR)];
    }
    if (forward && l == 0) bval = b[e * N + r];
  }
  if (act) {
    const int i = r / ND, a = r - i * ND;
    const int64_t row = e * NP + i;
    const int64_t p0 = rowptr[row], p1 = rowptr[row + 1];
    const int64_t q0 = forward ? p0 : p0 + own[row] + NP;
    const int64_t q1 = forward ? p0 + own[row] : p1;
    double acc = 0.0;
#pragma unroll 2
    for (int64_t p = q0 + l; p < q1; p += LPR)
      acc += block_dot<ND>(vals + p * ND * ND + a * ND, x + (int64_t)colind[p] * ND);
    tp[slot][r][l] = acc;
  }
  __syncthreads();
  if (act && l == 0) {
    double sum = 0.0;
#pragma unroll
    for (int k = 0; k < LPR; ++k) sum += tp[slot][r][k];
    v[slot][r] = (float)(forward ? bval - sum : sum);
  }
  __syncthreads();
  if (act) {
    yp[slot][r][l] = row_dot<NC>([&](int u) { return mrow[u]; }, [&](int u) { return v[slot][l + u * LPR]; },
                                 [&](int u) { return l + u * LPR < N; });
  }
  __syncthreads();
  if (act && l == 0) {
    float y = 0.0f;
#pragma unroll
    for (int k = 0; k < LPR; ++k) y += yp[slot][r][k];
    if (forward) x[e * N + r] = (double)y;
    else x[e * N + r] -= (double)y;
  }
}

// ---------------------------------------------------------------------------
// Dependency-driven sweeps: one launch per triangle instead of one per level.
// The elements are cut into sets that take one or two elements of a level
// each: an element joins the set of its latest-begun neighbour when it can, so
// that most of the dependences run inside a set (ilu_sets).  A workgroup takes
// one set and walks it, so a value needed by the set's next elements is handed
// on in LDS (a step takes about 0.75 us); only values from other sets go
// through memory (1.3 us and more from result to use).  An element depends on
// its own set and on sets begun before it only, and sets are handed out in that
// order by an atomic counter, so everything a workgroup waits for belongs to a
// workgroup that already runs or is done.
//
// A sweep's output holds ILU_PENDING (a signalling-NaN bit pattern, which no
// arithmetic produces: a NaN result is quiet) wherever it is not yet
// computed, so waiting for a neighbour is loading its values until none is
// pending.  Values are loaded and stored with device-scope atomics (an 8-byte
// store is seen whole or not at all), so no stale copy in another XCD's L2 is
// ever read.  The forward sweep writes y = L^-1 b into d_y and sets its
// elements' rows of x pending (after reading b: x may be b); the backward
// sweep reads its own y, writes x and sets its rows of y pending again, so
// d_y is pending between applications (each factorization sets it so).  A
// wait gives up after a bounded number of polls, sets the error word and
// carries on, so every launch ends.
//
// What bounds a step is the latency from the last value's arrival to the next
// element's first use of the result, so nothing else is done in between.  Two
// waves of a workgroup only wait: they poll the other sets' values for the
// elements ahead, in turn, and put them in a ring in LDS.  The other waves form
// G groups that take the set's elements in turn: a group loads its next
// element's matrix into registers while the others compute (a wave that loaded
// for the element after next before it computed put 20 to 60 loads and their
// addresses into every step, 1.1 us on an n x n annulus).
// Both triangles, against one workgroup per level's four elements with every
// value through memory (MI355X): 2D diagonal-E p=2 on an n x n annulus n=24 115
// -> 75 us, n=123 653 -> 417 us; 2D Omega p=2 n=48 325 -> 171 us; 2D Omega p=1
// n=200 1097 -> 539 us; 3D Omega p=2 n=10 240 -> 212 us, p=1 n=24 1920 -> 618 us.
// The lanes, the order of operations and so the bits are the level kernels'.
// ---------------------------------------------------------------------------
constexpr int ILU_WAIT_POLLS = 1 << 18;
constexpr unsigned long long ILU_PENDING = 0x7FF4DEADBEEF0001ull;
// sync words: ticket counter, error word, poll limit (0: ILU_WAIT_POLLS)
enum { ILU_SYNC_TICKET = 0, ILU_SYNC_ERR = 1, ILU_SYNC_POLLS = 2, ILU_SYNC_WORDS = 3 };

// Groups of computing waves (w waves each) in a workgroup: 8 of one wave, 5 of
// two, 3 of three, 2 of four.  More make it slower (12 one-wave groups: 93
// instead of 64 us a triangle on a 40 x 40 annulus, 2D diagonal-E p=2): the
// waiting groups poll the LDS that the computing one needs.
constexpr int ilu_groups(int w) { return 10 / w > 8 ? 8 : 10 / w > 2 ? 10 / w : 2; }
// Elements of one level that a set takes: two where there are groups enough to
// compute them side by side and load ahead (two instead of one: 2D Omega p=2 82
// -> 72 us, three: 99 us), more where the sets would otherwise outnumber the
// CUs (about one workgroup fits a CU, and the sets beyond wait for the first
// ones to end).
constexpr int ilu_set_width(int w) { return ilu_groups(w) >= 5 ? 2 : 1; }
constexpr int ILU_WIDTH_MAX = 8, ILU_CUS = 256;

__global__ void ilu_pending_fill(double* __restrict__ y, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) y[i] = __longlong_as_double((long long)ILU_PENDING);
}

__device__ __forceinline__ bool ilu_is_pending(double v) {
  return (unsigned long long)__double_as_longlong(v) == ILU_PENDING;
}

__device__ __forceinline__ double x_load(const double* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void x_store(double* p, double v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// LDS words that the waves of a workgroup signal each other with, and the
// wait that orders a wave's LDS accesses around them
__device__ __forceinline__ int lds_get(const int* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
__device__ __forceinline__ void lds_set(int* p, int v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
__device__ __forceinline__ void lds_add(int* p, int v) {
  __hip_atomic_fetch_add(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
__device__ __forceinline__ void lds_fence() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }

template <int NP, int ND, int NS, bool DIAGE, class BT>
struct IluSet {
  static constexpr int N = NP * ND, NFACES = ND - 1;
  static constexpr int LPR = ilu_lanes<N, DIAGE>(), W = ilu_waves<N, DIAGE>(), RW = (N + W - 1) / W;
  // a lane's share of a row: inverse entries and neighbour blocks
  static constexpr int NC = InvLayout<N>::NC, NCP = InvLayout<N>::NCP;
  static constexpr int MAXB = ((DIAGE ? NFACES : NFACES * NS) + LPR - 1) / LPR;
  static constexpr int G = ilu_groups(W), POLLERS = 2;
  static constexpr int RING = 2 * ((G + 1) / 2) + 2;
  static constexpr int THREADS = 64 * (G * W + POLLERS);
  // largest set: what 64 KB of LDS hold, the reach of an LDS instruction's
  // offset (beyond it every access computes its address: 12% on 3D Omega p=2)
  static constexpr int PER_ELEMENT = 8 * N + 8 * NP + 4 + 3 * 4 * NFACES + 8;
  static constexpr int FIXED = 8 * RING * NFACES * N + 4 * G * (W > 1 ? 2 : 1) * N + 64;
  static constexpr int KMAX = (65536 - FIXED) / PER_ELEMENT < 384 ? (65536 - FIXED) / PER_ELEMENT : 384;
  static constexpr int LOCAL = KMAX * N;
  double xl[LOCAL + RING * NFACES * N];   // the set's values, then a ring of other sets' values
  // right-hand sides; two a group, as its waves can be one element apart
  alignas(16) float v[G][W > 1 ? 2 : 1][N];
  int64_t q[KMAX][NP];                    // per node row: first neighbour block << 8 | blocks
  int32_t el[KMAX];
  int32_t nb[KMAX][NFACES];               // neighbour elements of the sweep's side, ascending, -1 beyond
  int32_t at[KMAX][NFACES];               // where their values are in xl
  int32_t dep[KMAX][NFACES];              // and their places in the set, KMAX for others
  int done[KMAX + 1], rows[KMAX];         // waves that have finished the element / written its rows of v
  int ready[POLLERS];                     // elements whose outside values have come, per waiting wave
  int64_t set;
};

// in: the right-hand side (forward: b; backward: y); out: the result, which
// the neighbours' values are read from (forward: y; backward: x); reset: the
// vector whose rows of this element become pending after use (forward: x;
// backward: y).  in may alias reset.
template <int NP, int ND, int NS, bool DIAGE, class BT>
__global__ void __launch_bounds__((IluSet<NP, ND, NS, DIAGE, BT>::THREADS))
ilu_sweep_dep_kernel(const int32_t* __restrict__ order, const int32_t* __restrict__ start,
                     const int32_t* __restrict__ place, const int32_t* __restrict__ sets, int64_t nsets,
                     const pdes::ElFace* __restrict__ elface, const int64_t* __restrict__ rowptr,
                     const int32_t* colind, const int32_t* __restrict__ own, const BT* vals, const float* inv,
                     const double* in, double* out, double* reset, int forward,
                     const int32_t* __restrict__ el_inst, const int32_t* __restrict__ mask,
                     const int32_t* __restrict__ inst_active, int32_t* __restrict__ sync) {
  using C = IluSet<NP, ND, NS, DIAGE, BT>;
  constexpr int N = C::N, NFACES = C::NFACES, LPR = C::LPR, W = C::W, RW = C::RW, NC = C::NC, MAXB = C::MAXB;
  static_assert(DIAGE || NS == NP, "dense faces couple all nodes of both elements");
  __shared__ C sm;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  if (tid == 0) {
    // (the counter wraps to 0 with the last of the launch's workgroups)
    const int64_t tk = atomicInc(reinterpret_cast<unsigned*>(&sync[ILU_SYNC_TICKET]), (unsigned)nsets - 1u);
    int64_t set = tk < nsets ? (sets ? (int64_t)sets[tk] : tk) : -1;
    if (set >= 0) {
      const int inst = el_inst ? el_inst[order[start[set]]] : 0;   // a set stays within an instance
      if ((mask && !mask[inst]) || (inst_active && !inst_active[inst])) set = -1;   // no element waits on it
    }
    sm.set = set;
    for (int p = 0; p < C::POLLERS; ++p) sm.ready[p] = 0;
  }
  for (int k = tid; k < C::KMAX; k += C::THREADS) sm.done[k] = sm.rows[k] = 0;
  if (tid == 0) sm.done[C::KMAX] = W;
  __syncthreads();
  if (sm.set < 0) return;   // uniform over the workgroup
  const int base = start[sm.set], K = start[sm.set + 1] - base;
  // what the walk needs to know about the set's elements
  for (int k = tid; k < K; k += C::THREADS) {
    const int e = order[base + k];
    sm.el[k] = e;
    int id[NFACES];
#pragma unroll
    for (int f = 0; f < NFACES; ++f) {
      const int n = elface[(int64_t)e * NFACES + f].x;
      id[f] = n >= 0 && (forward ? n < e : n > e) ? n : 0x7fffffff;
    }
#pragma unroll
    for (int i = 0; i < NFACES; ++i)
#pragma unroll
      for (int f = 0; f + 1 < NFACES - i; ++f)
        if (id[f + 1] < id[f]) { const int t = id[f]; id[f] = id[f + 1]; id[f + 1] = t; }
#pragma unroll
    for (int f = 0; f < NFACES; ++f) {
      const bool has = id[f] != 0x7fffffff;
      const int pl = has ? place[id[f]] - base : -1;
      const bool local = pl >= 0 && pl < K;
      sm.nb[k][f] = has ? id[f] : -1;
      sm.at[k][f] = local ? pl * N : C::LOCAL + ((k % C::RING) * NFACES + f) * N;
      sm.dep[k][f] = local ? pl : C::KMAX;
    }
  }
  for (int t = tid; t < K * NP; t += C::THREADS) {
    const int64_t row = (int64_t)order[base + t / NP] * NP + t % NP;
    const int64_t p0 = rowptr[row], o = own[row];
    const int64_t b = forward ? p0 : p0 + o + NP, n = forward ? o : rowptr[row + 1] - b;
    sm.q[t / NP][t % NP] = b << 8 | n;
  }
  __syncthreads();

  if (wave >= C::G * W) {
    // a waiting wave
    const int wp = wave - C::G * W;
    __builtin_amdgcn_s_setprio(2);
    const int max_polls = sync[ILU_SYNC_POLLS] > 0 ? sync[ILU_SYNC_POLLS] : ILU_WAIT_POLLS;
    constexpr int NL = (N + 63) / 64;
    for (int k = wp; k < K; k += C::POLLERS) {
      if (k >= C::RING)
        while (lds_get(&sm.done[k - C::RING]) < W) __builtin_amdgcn_s_sleep(1);   // its ring slot is free
      const double* from[NFACES];
      double x[NFACES][NL];
#pragma unroll
      for (int f = 0; f < NFACES; ++f) {
        const int n = sm.nb[k][f];
        from[f] = n >= 0 && sm.at[k][f] >= C::LOCAL ? out + (int64_t)n * N : nullptr;
#pragma unroll
        for (int u = 0; u < NL; ++u)
          x[f][u] = from[f] && lane + 64 * u < N ? x_load(from[f] + lane + 64 * u) : 0.0;
      }
      int polls = 0;
      while (true) {
        bool pending = false;
#pragma unroll
        for (int f = 0; f < NFACES; ++f)
#pragma unroll
          for (int u = 0; u < NL; ++u) pending |= ilu_is_pending(x[f][u]);
        if (!__any(pending)) break;
        if (++polls > max_polls) {
          __hip_atomic_store(&sync[ILU_SYNC_ERR], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          break;
        }
#pragma unroll
        for (int f = 0; f < NFACES; ++f)
#pragma unroll
          for (int u = 0; u < NL; ++u)
            if (ilu_is_pending(x[f][u])) x[f][u] = x_load(from[f] + lane + 64 * u);
      }
#pragma unroll
      for (int f = 0; f < NFACES; ++f)
        if (from[f]) {
#pragma unroll
          for (int u = 0; u < NL; ++u)
            if (lane + 64 * u < N) sm.xl[sm.at[k][f] + lane + 64 * u] = x[f][u];
        }
      lds_fence();
      if (lane == 0) lds_set(&sm.ready[wp], k + 1);
    }
    return;
  }

  // the computing waves: lane l of row r, elements g, g + G, ... of the set
  const int g = wave / W, gw = wave - g * W;
  const int lane_l = lane % LPR, first = lane - lane_l;
  const bool has_row = lane / LPR < RW && gw * RW + lane / LPR < N;
  const int lane_r = has_row ? gw * RW + lane / LPR : N - 1;
  for (int k = g; k < K; k += C::G) {
    int l = lane_l, r = lane_r;
    // FP64 blocks of dense faces from 40 rows on: the places that follow from the
    // lane and the row are formed anew for each element.  Taken out of the loop
    // they filled the registers that the blocks need: 15 to 36 of a share's values
    // went to scratch memory, which ended the loading ahead.  Both
    // triangles, same bits: 8,192 triangles Omega p=3 1037 -> 523 us, p=4 1563 ->
    // 832 us, 6,000 tets p=2 350 -> 262 us.
    if constexpr (!DIAGE && sizeof(BT) == 8 && N >= 40) asm volatile("" : "+v"(l), "+v"(r));
    const int i = r / ND, a = r - i * ND;
    // this lane's share: entries l, l + LPR, ... of its row of D'_e^-1, row a
    // of the neighbour blocks l, l + LPR, ... (a valid block where there is
    // none), the places of their values, the right-hand side
    const int64_t e = sm.el[k];
    const int64_t q = sm.q[k][i];
    const int64_t p0 = q >> 8;
    const int n = (int)(q & 255);
    float m[C::NCP];
    // (in FP64 already where the share is small)
    using KT = std::conditional_t<(MAXB <= 3), double, BT>;
    KT blk[MAXB][ND];
    int off[MAXB];
    const float* Mi = inv + e * InvLayout<N>::SIZE;
    if constexpr (InvLayout<N>::VEC4) {
#pragma unroll
      for (int u = 0; u < C::NCP; u += 4) {
        const float4 m4 = *reinterpret_cast<const float4*>(Mi + (u / 4 * (N * LPR) + r * LPR + l) * 4);
        m[u] = m4.x;
        m[u + 1] = m4.y;
        m[u + 2] = m4.z;
        m[u + 3] = m4.w;
      }
    } else {
#pragma unroll
      for (int u = 0; u < NC; ++u) m[u] = Mi[InvLayout<N>::at(r, l + u * LPR < N ? l + u * LPR : N - 1)];
    }
#pragma unroll
    for (int u = 0; u < MAXB; ++u) {
      const int p = l + u * LPR;
      // (a row without blocks on this side: its first or last own block)
      const int64_t pp = p < n ? p0 + p : forward ? p0 : p0 - 1;
#pragma unroll
      for (int c = 0; c < ND; ++c) blk[u][c] = (KT)vals[pp * (ND * ND) + a * ND + c];
      off[u] = 0;
      if constexpr (DIAGE) {
        const int col = colind[pp];
#pragma unroll
        for (int f = 0; f < NFACES; ++f) {
          const int d = col - sm.nb[k][f] * NP;
          if (sm.nb[k][f] >= 0 && d >= 0 && d < NP) off[u] = sm.at[k][f] + d * ND;
        }
      } else {
        if (p < NFACES * NP) off[u] = sm.at[k][p / NP] + (p % NP) * ND;
      }
    }
    const double bval = in[e * N + r];
    if constexpr (MAXB <= 3) {
#pragma unroll
      for (int u = 0; u < MAXB; ++u)
#pragma unroll
        for (int c = 0; c < ND; ++c) asm volatile("" : "+v"(blk[u][c]));   // converted before the wait
    }
    // its turn: the set's elements that it depends on are done and the values
    // from outside are here
    int dep[NFACES];
#pragma unroll
    for (int f = 0; f < NFACES; ++f) dep[f] = sm.dep[k][f];
    while (true) {
      int have = W;
#pragma unroll
      for (int f = 0; f < NFACES; ++f) {
        const int d = lds_get(&sm.done[dep[f]]);
        have = d < have ? d : have;
      }
      if (lds_get(&sm.ready[k % C::POLLERS]) > k && have == W) break;
    }
    __builtin_amdgcn_s_setprio(3);
    lds_fence();
    // (a few blocks' values are read together: one LDS latency for all; fewer
    // where the share leaves no registers for four)
    constexpr int BG = MAXB * ND * (int)(sizeof(BT) / 4) > 40 ? 2 : MAXB < 4 ? MAXB : 4;
    double acc = 0.0;
#pragma unroll
    for (int u0 = 0; u0 < MAXB; u0 += BG) {
      double x[BG][ND];
#pragma unroll
      for (int u = 0; u < BG; ++u)
#pragma unroll
        for (int c = 0; c < ND; ++c)
          if (u0 + u < MAXB) x[u][c] = sm.xl[off[u0 + u < MAXB ? u0 + u : 0] + c];
#pragma unroll
      for (int u = 0; u < BG; ++u)
        if (u0 + u < MAXB) {
          const double d = block_dot<ND>(blk[u0 + u < MAXB ? u0 + u : 0], x[u]);
          if (l + (u0 + u) * LPR < n) acc += d;
        }
    }
    double sum = 0.0;
    if constexpr (LPR == 1) {
      sum += acc;
    } else {
#pragma unroll
      for (int u = 0; u < LPR; ++u) sum += __shfl(acc, first + u, 64);
    }
    float* const v = sm.v[g][W > 1 ? k / C::G % 2 : 0];
    if (has_row && l == 0) v[r] = (float)(forward ? bval - sum : sum);
    if constexpr (W == 1) {
      asm volatile("" ::: "memory");   // (a wave's LDS accesses keep their order)
    } else {
      lds_fence();
      if (lane == 0) lds_add(&sm.rows[k], 1);
      while (lds_get(&sm.rows[k]) < W) {}
      lds_fence();
    }
    const float y = row_dot<NC>([&](int u) { return m[u]; }, [&](int u) { return v[l + u * LPR]; },
                                [&](int u) { return l + u * LPR < N; });
    float ys = 0.0f;
    if constexpr (LPR == 1) {
      ys += y;
    } else {
#pragma unroll
      for (int u = 0; u < LPR; ++u) ys += __shfl(y, first + u, 64);
    }
    const double xe = forward ? (double)ys : bval - (double)ys;
    if (has_row && l == 0) {
      sm.xl[k * N + r] = xe;
      x_store(out + e * N + r, xe);
    }
    lds_fence();
    if (lane == 0) lds_add(&sm.done[k], 1);
    __builtin_amdgcn_s_setprio(0);
    // (this row of `in`, which `reset` may alias, is in bval)
    if (has_row && l == 0) x_store(reset + e * N + r, __longlong_as_double((long long)ILU_PENDING));
  }
}

// least width and largest size of a set
static void ilu_set_shape(const pdes_ctx* c, int* width, int* kmax) {
  *width = *kmax = 1;
#define PDES_ILU_SET(D_, NP_, NF_, NS_, DE_)                              \
  if (c->dim == D_ && c->Np == NP_ && (c->diag_e != 0) == DE_) {          \
    using C = IluSet<NP_, D_ + 2, NS_, DE_, float>;                     \
    static_assert(sizeof(C) <= 65536, "a set's LDS");                     \
    *width = ilu_set_width(C::W);                                         \
    *kmax = C::KMAX;                                                      \
  }
  PDES_FOR_EACH_SHAPE(PDES_ILU_SET)
#undef PDES_ILU_SET
}

// The sets of one triangle (host): elements in level order (lv, els), each
// joining the set of its latest-begun neighbour of the sweep's side, else the
// set begun last, if it has room (ilu_set_shape, ILU_CUS), else beginning one.  Dependences then go to the own
// set or to sets begun before.
static void ilu_sets(const pdes_ctx* c, bool forward, const std::vector<int32_t>& lv, const std::vector<int32_t>& els,
                     std::vector<int32_t>& order, std::vector<int32_t>& start, std::vector<int32_t>& place) {
  const int nel = c->numEl, nf = c->nfaces, levels = els.empty() ? 1 : lv[els.back()] + 1;
  int width, kmax;
  ilu_set_shape(c, &width, &kmax);
  width = std::max(width, (int)std::min<int64_t>(ILU_WIDTH_MAX, ceil_div(nel, (int64_t)levels * ILU_CUS)));
  std::vector<int32_t> set(nel, -1), len, last, at_last;   // per set: elements, latest level, elements of it
  // (packed batches: a set stays within an instance, whose elements share no
  // face with the others': join the set begun last only from the same side)
  auto inst_of = [&](int e) { return c->h_inst_of.empty() ? 0 : c->h_inst_of[e]; };
  std::vector<int32_t> newest;                             // per instance: the set begun last
  for (int e : els) {
    const int in = inst_of(e);
    if ((int)newest.size() <= in) newest.resize(in + 1, -1);
    int32_t best = -1;
    for (int f = 0; f < nf; ++f) {
      const int k = c->h_elface[(size_t)e * nf + f].x;
      if (k >= 0 && (forward ? k < e : k > e)) best = std::max(best, set[k]);
    }
    auto room = [&](int32_t t) { return t >= 0 && len[t] < kmax && (last[t] < lv[e] || at_last[t] < width); };
    int32_t to = room(best) ? best : newest[in] >= best && room(newest[in]) ? newest[in] : -1;
    if (to < 0) {
      to = (int32_t)len.size();
      len.push_back(0);
      last.push_back(-1);
      at_last.push_back(0);
      newest[in] = to;
    }
    set[e] = to;
    ++len[to];
    at_last[to] = last[to] == lv[e] ? at_last[to] + 1 : 1;
    last[to] = lv[e];
  }
  start.assign(len.size() + 1, 0);
  for (size_t k = 0; k < len.size(); ++k) start[k + 1] = start[k] + len[k];
  std::vector<int32_t> pos(start.begin(), start.end() - 1);
  order.resize(nel);
  place.resize(nel);
  for (int e : els) {
    place[e] = pos[set[e]]++;
    order[place[e]] = e;
  }
}

// dependency levels of the natural-order sweeps (host, once per context)
static int ilu_structure(pdes_ctx* c, pdes_precond* p) {
  const int nel = c->numEl, nf = c->nfaces;
  std::vector<int32_t> fl(nel, 0), bl(nel, 0);
  int fmax = 0, bmax = 0;
  for (int e = 0; e < nel; ++e) {
    int lv = 0;
    for (int f = 0; f < nf; ++f) {
      const int k = c->h_elface[(size_t)e * nf + f].x;
      if (k >= 0 && k < e) lv = std::max(lv, fl[k] + 1);
    }
    fl[e] = lv;
    fmax = std::max(fmax, lv);
  }
  for (int e = nel - 1; e >= 0; --e) {
    int lv = 0;
    for (int f = 0; f < nf; ++f) {
      const int k = c->h_elface[(size_t)e * nf + f].x;
      if (k > e) lv = std::max(lv, bl[k] + 1);
    }
    bl[e] = lv;
    bmax = std::max(bmax, lv);
  }
  auto bucket = [&](const std::vector<int32_t>& lv, int nl, std::vector<int64_t>& ptr, std::vector<int32_t>& el) {
    ptr.assign(nl + 2, 0);
    for (int e = 0; e < nel; ++e) ptr[lv[e] + 1]++;
    for (int l = 0; l <= nl; ++l) ptr[l + 1] += ptr[l];
    el.assign(nel, 0);
    std::vector<int64_t> pos(ptr.begin(), ptr.end() - 1);
    for (int e = 0; e < nel; ++e) el[pos[lv[e]]++] = e;
  };
  std::vector<int32_t> fel, bel;
  bucket(fl, fmax, p->fptr, fel);
  bucket(bl, bmax, p->bptr, bel);
  // offset of the own-element block run in every row of the BSR pattern
  const pdes_jacobian* J = c->jac;
  const int64_t nrows = (int64_t)nel * c->Np;
  std::vector<int32_t> own(nrows, 0);
  for (int64_t r = 0; r < nrows; ++r) {
    const int32_t first = (int32_t)((r / c->Np) * c->Np);
    int64_t q = J->h_rowptr[r];
    while (q < J->h_rowptr[r + 1] && J->h_colind[q] < first) ++q;
    own[r] = (int32_t)(q - J->h_rowptr[r]);
  }
  if (hipMalloc((void**)&p->d_own, std::max<int64_t>(1, nrows) * sizeof(int32_t)) != hipSuccess) {
    set_error("device allocation of the ILU row offsets failed");
    return PDES_ERR_NOMEM;
  }
  PDES_HIP(hipMemcpyAsync(p->d_own, own.data(), nrows * sizeof(int32_t), hipMemcpyHostToDevice, c->stream));
  if (hipMalloc((void**)&p->d_fel, std::max(1, nel) * sizeof(int32_t)) != hipSuccess ||
      hipMalloc((void**)&p->d_bel, std::max(1, nel) * sizeof(int32_t)) != hipSuccess) {
    set_error("device allocation of the ILU level lists failed");
    return PDES_ERR_NOMEM;
  }
  PDES_HIP(hipMemcpyAsync(p->d_fel, fel.data(), nel * sizeof(int32_t), hipMemcpyHostToDevice, c->stream));
  PDES_HIP(hipMemcpyAsync(p->d_bel, bel.data(), nel * sizeof(int32_t), hipMemcpyHostToDevice, c->stream));
  // an element that meets a neighbour at two faces: level sweeps, which walk the
  // rows (the sets' kernel goes by faces).  Diagonal-E operators only: with dense
  // faces such an element's rows hold every column of the neighbour twice, which
  // the assembly refuses.
  bool twice = false;
  for (int e = 0; e < nel && !twice; ++e)
    for (int f = 0; f < nf; ++f)
      for (int g = f + 1; g < nf; ++g) {
        const int k = c->h_elface[(size_t)e * nf + f].x;
        twice = twice || (k >= 0 && k == c->h_elface[(size_t)e * nf + g].x);
      }
  for (int pass = 0; pass < 2; ++pass) {
    std::vector<int32_t> order, start, place;
    ilu_sets(c, pass == 0, pass == 0 ? fl : bl, pass == 0 ? fel : bel, order, start, place);
    pdes_precond::Sets& k = pass == 0 ? p->fset : p->bset;
    k.n = (int64_t)start.size() - 1;
    if (hipMalloc((void**)&k.d_order, std::max(1, nel) * sizeof(int32_t)) != hipSuccess ||
        hipMalloc((void**)&k.d_start, start.size() * sizeof(int32_t)) != hipSuccess ||
        hipMalloc((void**)&k.d_place, std::max(1, nel) * sizeof(int32_t)) != hipSuccess) {
      set_error("device allocation of the ILU sets failed");
      return PDES_ERR_NOMEM;
    }
    PDES_HIP(hipMemcpyAsync(k.d_order, order.data(), nel * sizeof(int32_t), hipMemcpyHostToDevice, c->stream));
    PDES_HIP(hipMemcpyAsync(k.d_start, start.data(), start.size() * sizeof(int32_t), hipMemcpyHostToDevice, c->stream));
    PDES_HIP(hipMemcpyAsync(k.d_place, place.data(), nel * sizeof(int32_t), hipMemcpyHostToDevice, c->stream));
    PDES_HIP(hipStreamSynchronize(c->stream));   // the host vectors go out of scope
  }
  p->force = twice || std::getenv("PDES_ILU_LEVELS") ? 1 : std::getenv("PDES_ILU_DEP") ? 2 : 0;
  p->h_fl = fl;
  p->h_bl = bl;
  p->blk_per_el = (double)(J->nnzb - (int64_t)nel * c->Np * c->Np) / 2.0 / std::max(1, nel);
  const int64_t ny = std::max<int64_t>(1, c->numDof);
  // d_y is set pending with each factorization (pc_setup)
  if (hipMalloc((void**)&p->d_y, ny * sizeof(double)) != hipSuccess ||
      hipMalloc((void**)&p->d_sync, ILU_SYNC_WORDS * sizeof(int32_t)) != hipSuccess) {
    set_error("device allocation of the ILU sweep vector failed");
    return PDES_ERR_NOMEM;
  }
  PDES_HIP(hipMemsetAsync(p->d_sync, 0, ILU_SYNC_WORDS * sizeof(int32_t), c->stream));
  // PDES_ILU_WAIT_POLLS: a smaller bound on the dependency waits (for tests
  // of the give-up path; the default bound is never reached by a sweep that
  // runs normally)
  const char* polls_env = std::getenv("PDES_ILU_WAIT_POLLS");
  const int32_t poll_limit = polls_env ? (int32_t)std::max(1L, std::strtol(polls_env, nullptr, 10)) : 0;
  if (poll_limit)
    PDES_HIP(hipMemcpyAsync(p->d_sync + ILU_SYNC_POLLS, &poll_limit, sizeof(int32_t), hipMemcpyHostToDevice,
                            c->stream));
  PDES_HIP(hipStreamSynchronize(c->stream));
  p->ilu_ready = true;
  return PDES_OK;
}

// Which sweeps an application runs (both give the same bits).  The sweeps level
// by level take ILU_LEVEL_US a launch and stream the blocks at ILU_LEVEL_BW; the
// dependency-driven ones take ILU_DEP_STEP_US per level of the critical path,
// ILU_DEP_EL_US per element, or stream at ILU_DEP_BW.  Measured (MI355X, one
// triangle): natural numbering, hundreds of levels: 2D diagonal-E p=2 n=300 600
// levels 3131 us level by level, 619 us dependency-driven; 3D Omega p=2 n=20 80
// levels 842 and 608 us; p=1 n=32 128 levels 919 and 617 us.  The same meshes
// numbered at random, about 10 levels: diagonal-E n=64 47 and 39 us, n=180 171
// and 218 us; 2D Omega p=1 n=48 51 and 34 us, n=200 84 and 184 us; 3D Omega p=2
// n=10 121 and 89 us, n=16 281 and 287 us.  The elements and levels are those of
// the instances being solved when the batched solver says so, else the whole
// mesh.
constexpr double ILU_LEVEL_US = 4.5, ILU_LEVEL_BW = 3.5e6;   // bytes per us
constexpr double ILU_DEP_STEP_US = 0.85, ILU_DEP_EL_US = 0.0022, ILU_DEP_BW = 2.4e6;

static bool ilu_use_dep(const pdes_ctx* c, const pdes_precond* p) {
  if (p->force) return p->force == 2;
  const int nd = c->nd, n = c->Np * nd;
  const double be = p->blk_per_el * nd * nd * (c->jac->fp64 ? 8.0 : 4.0) + (double)n * n * 4.0 + 3.0 * n * 8.0;
  const bool hint = c->ilu_hint_el >= 0;
  const double nel = hint ? (double)c->ilu_hint_el : (double)c->numEl;
  double lev = 0.0, dep = 0.0;
  for (int pass = 0; pass < 2; ++pass) {
    const double L = std::max(1, hint ? (pass ? c->ilu_hint_lb : c->ilu_hint_lf)
                                      : (int)(pass ? p->bptr.size() : p->fptr.size()) - 1);
    lev += L * ILU_LEVEL_US + nel * be / ILU_LEVEL_BW;
    dep += std::max({L * ILU_DEP_STEP_US, nel * ILU_DEP_EL_US, nel * be / ILU_DEP_BW});
  }
  return dep < lev;
}

struct SetSelected {
  const int32_t* order;
  const int32_t* start;
  const int32_t* el_inst;
  const int32_t* sel;
  __host__ __device__ bool operator()(const int32_t& set) const { return sel[el_inst[order[start[set]]]] != 0; }
};

// The batched solver's hint for the ILU(0) applications of its next Arnoldi
// steps: they touch only the elements of the instances with inst_sel[i] != 0
// (nel of them, over lf forward and lb backward levels).  When the cost model
// then picks the dependency-driven sweeps, the lists of sets are compacted to
// those instances (order kept), so a sweep dispatches only their elements.  ilu_hint_clear ends the hint.
int ilu_hint(pdes_ctx* c, const int32_t* inst_sel, int ninst, int64_t nel, int lf, int lb) {
  pdes_precond* p = c->pc_obj;
  c->ilu_hint_el = nel;
  c->ilu_hint_lf = lf;
  c->ilu_hint_lb = lb;
  c->ilu_sel = false;
  if (!p || p->kind != PDES_PC_ILU0 || !c->d_el_inst || !ilu_use_dep(c, p)) return PDES_OK;
  const int64_t nf = p->fset.n, nb = p->bset.n;
  hipcub::CountingInputIterator<int32_t> ids(0);
  if (!p->d_fsel) {
    if (hipMalloc((void**)&p->d_fsel, std::max<int64_t>(1, nf) * sizeof(int32_t)) != hipSuccess ||
        hipMalloc((void**)&p->d_bsel, std::max<int64_t>(1, nb) * sizeof(int32_t)) != hipSuccess ||
        hipMalloc((void**)&p->d_nsel, 2 * sizeof(int32_t)) != hipSuccess) {
      set_error("device allocation of the ILU selection lists failed");
      return PDES_ERR_NOMEM;
    }
    size_t bytes = 0;
    PDES_HIP(hipcub::DeviceSelect::If(nullptr, bytes, ids, p->d_fsel, p->d_nsel, (int)std::max(nf, nb),
                                      SetSelected{p->fset.d_order, p->fset.d_start, c->d_el_inst, nullptr}, c->stream));
    if (hipMalloc(&p->d_select_tmp, std::max<size_t>(bytes, 16)) != hipSuccess) {
      set_error("device allocation of the ILU selection work space failed");
      return PDES_ERR_NOMEM;
    }
    p->select_tmp_bytes = bytes;
  }
  if (p->sel_ninst < ninst) {
    if (p->d_inst_sel) hipFree(p->d_inst_sel);
    p->d_inst_sel = nullptr;
    if (hipMalloc((void**)&p->d_inst_sel, ninst * sizeof(int32_t)) != hipSuccess) {
      set_error("device allocation of the ILU instance selection failed");
      return PDES_ERR_NOMEM;
    }
    p->sel_ninst = ninst;
  }
  PDES_HIP(hipMemcpyAsync(p->d_inst_sel, inst_sel, ninst * sizeof(int32_t), hipMemcpyHostToDevice, c->stream));
  size_t bytes = p->select_tmp_bytes;
  PDES_HIP(hipcub::DeviceSelect::If(p->d_select_tmp, bytes, ids, p->d_fsel, p->d_nsel, (int)nf,
                                    SetSelected{p->fset.d_order, p->fset.d_start, c->d_el_inst, p->d_inst_sel}, c->stream));
  bytes = p->select_tmp_bytes;
  PDES_HIP(hipcub::DeviceSelect::If(p->d_select_tmp, bytes, ids, p->d_bsel, p->d_nsel + 1, (int)nb,
                                    SetSelected{p->bset.d_order, p->bset.d_start, c->d_el_inst, p->d_inst_sel}, c->stream));
  int32_t cnt[2] = {0, 0};
  PDES_HIP(hipMemcpyAsync(cnt, p->d_nsel, sizeof(cnt), hipMemcpyDeviceToHost, c->stream));
  PDES_HIP(hipStreamSynchronize(c->stream));
  p->sel_nf = cnt[0];
  p->sel_nb = cnt[1];
  c->ilu_sel = true;
  return PDES_OK;
}

void ilu_hint_clear(pdes_ctx* c) {
  c->ilu_hint_el = -1;
  c->ilu_sel = false;
}

// levels spanned by the elements [el0, el1) (one instance of a packed batch)
int ilu_range_levels(const pdes_ctx* c, int64_t el0, int64_t el1, int* lf, int* lb) {
  const pdes_precond* p = c->pc_obj;
  *lf = *lb = 0;
  if (!p || p->h_fl.empty()) return PDES_ERR_ARG;
  for (int64_t e = el0; e < el1; ++e) {
    *lf = std::max(*lf, p->h_fl[e] + 1);
    *lb = std::max(*lb, p->h_bl[e] + 1);
  }
  return PDES_OK;
}

template <int NP, int ND, int NS, bool DIAGE>
static int ilu_factor(pdes_ctx* c) {
  pdes_jacobian* j = c->jac;
  pdes_precond* p = c->pc_obj;
  const dim3 block(GjShape<NP * ND>::THREADS);
  for (size_t l = 0; l + 1 < p->fptr.size(); ++l) {
    const int64_t cnt = p->fptr[l + 1] - p->fptr[l];
    if (cnt == 0) continue;
    const int32_t* lev = p->d_fel + p->fptr[l];
    if (j->fp64)
      hipLaunchKernelGGL((ilu_factor_level_kernel<NP, ND, NS, DIAGE, double>), dim3((unsigned)cnt), block, 0, c->stream,
                         lev, j->d_rowptr, j->d_colind, p->d_own, (const double*)j->d_vals, c->d_elface,
                         c->d_perm, c->d_nodepos, p->d_inv, j->d_err, c->d_el_inst, c->d_inst_active);
    else
      hipLaunchKernelGGL((ilu_factor_level_kernel<NP, ND, NS, DIAGE, float>), dim3((unsigned)cnt), block, 0, c->stream,
                         lev, j->d_rowptr, j->d_colind, p->d_own, (const float*)j->d_vals, c->d_elface,
                         c->d_perm, c->d_nodepos, p->d_inv, j->d_err, c->d_el_inst, c->d_inst_active);
  }
  PDES_HIP(hipGetLastError());
  return PDES_OK;
}

template <int NP, int ND, int NS, bool DIAGE>
static int ilu_apply(pdes_ctx* c, const double* b, double* x) {
  pdes_jacobian* j = c->jac;
  pdes_precond* p = c->pc_obj;
  constexpr int N = NP * ND;
  constexpr int LPR = ilu_lanes<N, DIAGE>();
  constexpr int EPB = 256 / (N * LPR);
  if (ilu_use_dep(c, p)) {
    const bool sel = c->ilu_sel && c->ilu_hint_el >= 0;
    for (int pass = 0; pass < 2; ++pass) {
      const pdes_precond::Sets& k = pass == 0 ? p->fset : p->bset;
      const int32_t* sets = sel ? (pass == 0 ? p->d_fsel : p->d_bsel) : nullptr;
      const int64_t nsets = sel ? (pass == 0 ? p->sel_nf : p->sel_nb) : k.n;
      if (nsets == 0) continue;
      // forward: b -> y, x set pending; backward: y -> x, y set pending again
      const double* in = pass == 0 ? b : p->d_y;
      double* out = pass == 0 ? p->d_y : x;
      double* reset = pass == 0 ? x : p->d_y;
      if (j->fp64)
        hipLaunchKernelGGL((ilu_sweep_dep_kernel<NP, ND, NS, DIAGE, double>), dim3((unsigned)nsets),
                           dim3(IluSet<NP, ND, NS, DIAGE, double>::THREADS), 0, c->stream, k.d_order, k.d_start,
                           k.d_place, sets, nsets, c->d_elface, j->d_rowptr, j->d_colind, p->d_own,
                           (const double*)j->d_vals, p->d_inv, in, out, reset, pass == 0, c->d_el_inst, c->d_mask,
                           c->d_inst_active, p->d_sync);
      else
        hipLaunchKernelGGL((ilu_sweep_dep_kernel<NP, ND, NS, DIAGE, float>), dim3((unsigned)nsets),
                           dim3(IluSet<NP, ND, NS, DIAGE, float>::THREADS), 0, c->stream, k.d_order, k.d_start,
                           k.d_place, sets, nsets, c->d_elface, j->d_rowptr, j->d_colind, p->d_own,
                           (const float*)j->d_vals, p->d_inv, in, out, reset, pass == 0, c->d_el_inst, c->d_mask,
                           c->d_inst_active, p->d_sync);
    }
    PDES_HIP(hipGetLastError());
    return PDES_OK;
  }
  for (int pass = 0; pass < 2; ++pass) {
    const std::vector<int64_t>& ptr = pass == 0 ? p->fptr : p->bptr;
    const int32_t* els = pass == 0 ? p->d_fel : p->d_bel;
    for (size_t l = 0; l + 1 < ptr.size(); ++l) {
      const int64_t cnt = ptr[l + 1] - ptr[l];
      if (cnt == 0) continue;
      const dim3 grid((unsigned)ceil_div(cnt, EPB));
      if constexpr (LPR > 1) {
        const dim3 block((unsigned)(EPB * N * LPR));
        if (j->fp64)
          hipLaunchKernelGGL((ilu_sweep_level_ml_kernel<NP, ND, double, LPR>), grid, block, 0, c->stream, els + ptr[l],
                             cnt, j->d_rowptr, j->d_colind, p->d_own, (const double*)j->d_vals, p->d_inv, b, x,
                             pass == 0, c->d_el_inst, c->d_mask, c->d_inst_active);
        else
          hipLaunchKernelGGL((ilu_sweep_level_ml_kernel<NP, ND, float, LPR>), grid, block, 0, c->stream, els + ptr[l],
                             cnt, j->d_rowptr, j->d_colind, p->d_own, (const float*)j->d_vals, p->d_inv, b, x,
                             pass == 0, c->d_el_inst, c->d_mask, c->d_inst_active);
        continue;
      }
      if (j->fp64)
        hipLaunchKernelGGL((ilu_sweep_level_kernel<NP, ND, double>), grid, dim3(256), 0, c->stream, els + ptr[l], cnt,
                           j->d_rowptr, j->d_colind, p->d_own, (const double*)j->d_vals, p->d_inv, b, x, pass == 0,
                           c->d_el_inst, c->d_mask, c->d_inst_active);
      else
        hipLaunchKernelGGL((ilu_sweep_level_kernel<NP, ND, float>), grid, dim3(256), 0, c->stream, els + ptr[l], cnt,
                           j->d_rowptr, j->d_colind, p->d_own, (const float*)j->d_vals, p->d_inv, b, x, pass == 0,
                           c->d_el_inst, c->d_mask, c->d_inst_active);
    }
  }
  PDES_HIP(hipGetLastError());
  return PDES_OK;
}

template <int NP, int ND>
static int bj_factor(pdes_ctx* c) {
  pdes_jacobian* j = c->jac;
  pdes_precond* p = c->pc_obj;
  if (c->active_count() == 0) return PDES_OK;
  const dim3 grid((unsigned)c->active_count()), block(GjShape<NP * ND>::THREADS);
  if (j->fp64)
    hipLaunchKernelGGL((bjacobi_factor_kernel<NP, ND, double>), grid, block, 0, c->stream, c->active_list(),
                       j->d_rowptr, j->d_colind, (const double*)j->d_vals, p->d_inv, j->d_err);
  else
    hipLaunchKernelGGL((bjacobi_factor_kernel<NP, ND, float>), grid, block, 0, c->stream, c->active_list(),
                       j->d_rowptr, j->d_colind, (const float*)j->d_vals, p->d_inv, j->d_err);
  PDES_HIP(hipGetLastError());
  return PDES_OK;
}

template <int NP, int ND>
static int bj_apply(pdes_ctx* c, const double* b, double* x) {
  if (c->active_count() == 0) return PDES_OK;
  constexpr int EPB = 256 / (NP * ND);
  const int64_t nel = c->active_count();
  hipLaunchKernelGGL((bjacobi_apply_kernel<NP, ND>), dim3((unsigned)ceil_div(nel, EPB)), dim3(256), 0, c->stream,
                     c->active_list(), nel, c->pc_obj->d_inv, b, x, c->d_el_inst, c->d_mask);
  PDES_HIP(hipGetLastError());
  return PDES_OK;
}

static int pc_factor(pdes_ctx* c) {
  if (c->dim == 2) {
    switch (c->Np) {
      case 3: return bj_factor<3, 4>(c);
      case 6: return bj_factor<6, 4>(c);
      case 10: return bj_factor<10, 4>(c);
      case 15: return bj_factor<15, 4>(c);
      case 7: return bj_factor<7, 4>(c);
      case 12: return bj_factor<12, 4>(c);
      case 18: return bj_factor<18, 4>(c);
      case 27: return bj_factor<27, 4>(c);
    }
  } else {
    switch (c->Np) {
      case 4: return bj_factor<4, 5>(c);
      case 10: return bj_factor<10, 5>(c);
    }
  }
  set_error("no block-Jacobi kernel for this operator");
  return PDES_ERR_UNSUPPORTED;
}

__global__ void copy_kernel(const double* __restrict__ a, double* __restrict__ b, int64_t n) {
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) b[i] = a[i];
}

static int ilu_factor_dispatch(pdes_ctx* c) {
#define PDES_ILU_F(D_, NP_, NF_, NS_, DE_) \
  if (c->dim == D_ && c->Np == NP_ && (c->diag_e != 0) == DE_) return ilu_factor<NP_, D_ + 2, NS_, DE_>(c);
  PDES_FOR_EACH_SHAPE(PDES_ILU_F)
#undef PDES_ILU_F
  set_error("no ILU(0) kernel for this operator");
  return PDES_ERR_UNSUPPORTED;
}

static int ilu_apply_dispatch(pdes_ctx* c, const double* b, double* x) {
#define PDES_ILU_A(D_, NP_, NF_, NS_, DE_) \
  if (c->dim == D_ && c->Np == NP_ && (c->diag_e != 0) == DE_) return ilu_apply<NP_, D_ + 2, NS_, DE_>(c, b, x);
  PDES_FOR_EACH_SHAPE(PDES_ILU_A)
#undef PDES_ILU_A
  set_error("no ILU(0) kernel for this operator");
  return PDES_ERR_UNSUPPORTED;
}

// ILU(0) apply through a captured graph: b is copied into the staging input,
// the graph (all level launches) is replayed, the staging output is copied to
// x.  Falls back to direct launches if the capture is refused.
static int ilu_apply_graphed(pdes_ctx* c, const double* b, double* x) {
  pdes_precond* p = c->pc_obj;
  const size_t bytes = (size_t)c->numDof * sizeof(double);
  if (!p->d_stage_in) {
    if (hipMalloc((void**)&p->d_stage_in, bytes) != hipSuccess ||
        hipMalloc((void**)&p->d_stage_out, bytes) != hipSuccess) {
      set_error("ILU staging allocation failed");
      return PDES_ERR_NOMEM;
    }
  }
  hipGraphExec_t exec = nullptr;
  for (auto& g : p->graphs)
    if (g.mask == c->d_mask && g.vals == c->jac->d_vals && g.fp64 == c->jac->fp64 && g.inv == p->d_inv)
      exec = g.exec;
  if (!exec) {
    hipGraph_t graph = nullptr;
    if (hipStreamBeginCapture(c->stream, hipStreamCaptureModeThreadLocal) != hipSuccess) {
      (void)hipGetLastError();
      return ilu_apply_dispatch(c, b, x);
    }
    const int st = ilu_apply_dispatch(c, p->d_stage_in, p->d_stage_out);
    const hipError_t ec = hipStreamEndCapture(c->stream, &graph);
    if (st) {
      if (graph) hipGraphDestroy(graph);
      return st;
    }
    if (ec != hipSuccess || !graph || hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0) != hipSuccess) {
      if (graph) hipGraphDestroy(graph);
      (void)hipGetLastError();
      return ilu_apply_dispatch(c, b, x);
    }
    hipGraphDestroy(graph);
    p->graphs.push_back({c->d_mask, c->jac->d_vals, c->jac->fp64, p->d_inv, exec});
  }
  PDES_HIP(hipMemcpyAsync(p->d_stage_in, b, bytes, hipMemcpyDeviceToDevice, c->stream));
  PDES_HIP(hipGraphLaunch(exec, c->stream));
  PDES_HIP(hipMemcpyAsync(x, p->d_stage_out, bytes, hipMemcpyDeviceToDevice, c->stream));
  return PDES_OK;
}

int pc_apply(pdes_ctx* c, const double* b, double* x) {
  // the dependency-driven sweeps are two launches, one a triangle; the
  // level-by-level ones are replayed from a captured graph
  if (c->pc_obj && c->pc_obj->kind == PDES_PC_ILU0)
    return c->use_graphs && !c->capturing && !ilu_use_dep(c, c->pc_obj) ? ilu_apply_graphed(c, b, x)
                                                                        : ilu_apply_dispatch(c, b, x);
  if (!c->pc_obj || c->pc_obj->kind == PDES_PC_NONE) {
    const int64_t n = c->numDof;
    hipLaunchKernelGGL(copy_kernel, dim3((unsigned)std::min<int64_t>(8192, ceil_div(n, 256))), dim3(256), 0,
                       c->stream, b, x, n);
    PDES_HIP(hipGetLastError());
    return PDES_OK;
  }
  if (c->dim == 2) {
    switch (c->Np) {
      case 3: return bj_apply<3, 4>(c, b, x);
      case 6: return bj_apply<6, 4>(c, b, x);
      case 10: return bj_apply<10, 4>(c, b, x);
      case 15: return bj_apply<15, 4>(c, b, x);
      case 7: return bj_apply<7, 4>(c, b, x);
      case 12: return bj_apply<12, 4>(c, b, x);
      case 18: return bj_apply<18, 4>(c, b, x);
      case 27: return bj_apply<27, 4>(c, b, x);
    }
  } else {
    switch (c->Np) {
      case 4: return bj_apply<4, 5>(c, b, x);
      case 10: return bj_apply<10, 5>(c, b, x);
    }
  }
  set_error("no block-Jacobi kernel for this operator");
  return PDES_ERR_UNSUPPORTED;
}

// What a captured sequence of preconditioner applications depends on besides
// device data: the kind, the factor and matrix buffers, and for ILU(0) the
// sweep kind and, for the dependency-driven sweeps over compacted lists of
// sets, their lengths (launch sizes).
void pc_graph_key(const pdes_ctx* c, int64_t key[6]) {
  const pdes_precond* p = c->pc_obj;
  for (int i = 0; i < 6; ++i) key[i] = 0;
  if (!p) return;
  key[0] = p->kind;
  key[1] = (int64_t)(intptr_t)p->d_inv;
  key[2] = c->jac ? (int64_t)(intptr_t)c->jac->d_vals : 0;
  key[3] = c->jac ? (int64_t)c->jac->fp64 : 0;
  if (p->kind == PDES_PC_ILU0) {
    const bool dep = ilu_use_dep(c, p);
    const bool sel = dep && c->ilu_sel && c->ilu_hint_el >= 0;
    key[4] = dep ? 1 + (sel ? 1 : 0) : 0;
    key[5] = sel ? p->sel_nf * (int64_t(1) << 32) + p->sel_nb : 0;
  }
}

// the error word of the dependency-driven sweeps (a wait that gave up): the
// preconditioner applications since the last check are not to be trusted
int pc_check(pdes_ctx* c) {
  pdes_precond* p = c->pc_obj;
  if (!p || p->kind != PDES_PC_ILU0 || !p->d_sync) return PDES_OK;
  int32_t err = 0;
  PDES_HIP(hipMemcpyAsync(&err, p->d_sync + ILU_SYNC_ERR, sizeof(int32_t), hipMemcpyDeviceToHost, c->stream));
  PDES_HIP(hipStreamSynchronize(c->stream));
  if (err) {
    PDES_HIP(hipMemsetAsync(p->d_sync + ILU_SYNC_ERR, 0, sizeof(int32_t), c->stream));
    set_error("an ILU(0) sweep gave up waiting for a neighbour element (its result is invalid)");
    return PDES_ERR_HIP;
  }
  return PDES_OK;
}

// floats that the inverse of an element block of n unknowns takes
int64_t pc_block_floats(int n) {
#define PDES_BLOCK_FLOATS(D_, NP_, NF_, NS_, DE_) \
  if (NP_ * (D_ + 2) == n) return InvLayout<NP_ * (D_ + 2)>::SIZE;
  PDES_FOR_EACH_SHAPE(PDES_BLOCK_FLOATS)
#undef PDES_BLOCK_FLOATS
  return (int64_t)n * n;
}

int pc_setup(pdes_ctx* c, int kind) {
  PDES_CHECK(kind == PDES_PC_NONE || kind == PDES_PC_BJACOBI || kind == PDES_PC_ILU0, PDES_ERR_UNSUPPORTED,
             "preconditioner kind %d is not available", kind);
  if (!c->pc_obj) c->pc_obj = new pdes_precond();
  pdes_precond* p = c->pc_obj;
  p->kind = kind;
  if (kind == PDES_PC_NONE) { p->factored = true; return PDES_OK; }
  PDES_CHECK(c->jac && c->jac->assembled, PDES_ERR_ARG, "assemble the Jacobian before the preconditioner");
  const int n = c->Np * c->nd;
  if (!p->d_inv || p->n != n) {
    if (p->d_inv) hipFree(p->d_inv);
    for (auto& g : p->graphs) hipGraphExecDestroy(g.exec);
    p->graphs.clear();
    p->n = n;
    if (hipMalloc((void**)&p->d_inv, (size_t)c->numEl * pc_block_floats(n) * sizeof(float)) != hipSuccess) {
      set_error("device allocation of the block-Jacobi factors failed");
      return PDES_ERR_NOMEM;
    }
  }
  int st;
  if (kind == PDES_PC_ILU0) {
    if (!p->ilu_ready && (st = ilu_structure(c, p)) != 0) return st;
    st = ilu_factor_dispatch(c);
    // the dependency-driven sweeps' vector holds ILU_PENDING between
    // applications; set it again with each factorization, so that an
    // application cut short between its two sweeps cannot leave values
    // behind for the next factorization's sweeps
    if (!st) {
      const int64_t ny = std::max<int64_t>(1, c->numDof);
      hipLaunchKernelGGL(ilu_pending_fill, dim3((unsigned)ceil_div(ny, 256)), dim3(256), 0, c->stream, p->d_y, ny);
      PDES_HIP(hipGetLastError());
    }
  } else {
    st = pc_factor(c);
  }
  if (st) return st;
  p->factored = true;
  return PDES_OK;
}

// ---------------------------------------------------------------------------
// GMRES building blocks
// ---------------------------------------------------------------------------
// CGS2 against the basis V_0 .. V_{m-1} (h = V^T w, w -= V h, twice, then
// w /= ||w||) in four launches, each passing once over the basis:
//   cgs_pass<MG, false>  partial dots of w
//   cgs_pass<MG, true>   sums them to h, w -= V h, and the partial dots of the
//                        new w from the basis values still in registers
//   cgs_norm             sums those, w -= V h, partial sum of w^2
//   cgs_finish           sums that, w /= ||w||, the Hessenberg column to the host
// Small systems are bound by the number of dependent launches and by the
// latency inside each, large ones by the basis traffic; both fall with the
// passes fused.  A workgroup's sums over its slice go to partial[i][block] and
// every workgroup of the next launch adds them up for itself in block order,
// so the bits depend on n only.  Up to n = 524,288 there are at most 256
// workgroups (at n = 131,000 and 30 vectors the second pass takes 11.6 us with
// 256, 15.6 with 128, 24 with 64); beyond, 512 and a launch of multidot_reduce
// before each use (at n = 300,000 a step takes 58 us the first way and 62 the
// second).  Separate kernels for each dot, update and sum (11 launches and a
// wait of the host a step) took 73 us a step at n = 9,600 with the operator
// and the preconditioner, these take 38.
constexpr int CGS_MAX_BLOCKS = 512;
// The coefficients of up to this many basis vectors are summed into LDS by every
// workgroup; those of longer cycles once, by multidot_reduce, and read from
// memory (LONG), so that the length of a cycle has no bound but the basis's
// memory.  Beyond it the pass over the basis takes longer than the extra launch.
constexpr int CGS_LDS_ROWS = 1024;

static int cgs_blocks(int64_t n) {
  const int64_t full = std::max<int64_t>(1, ceil_div(n, CGS_THREADS));
  if (full <= 8 * CGS_SELF_REDUCE) return (int)std::min<int64_t>(CGS_SELF_REDUCE, full);
  return (int)std::min<int64_t>(CGS_MAX_BLOCKS, full);
}

// AXPY: h = sums of pin's rows (nb_in each), w -= sum_i h_i V_i (kept in hsave
// by workgroup 0).  Then pout[i][block] = sum over the block's slice of V_i . w.
// The first 8 MG basis values of an entry stay in registers for both uses; the
// basis vectors beyond (m > 32) are read again, 32 at a time.
template <int MG, bool AXPY, bool LONG>
__global__ void __launch_bounds__(CGS_THREADS)
cgs_pass(const double* __restrict__ V, int m, int64_t ldv, double* __restrict__ w, int64_t n,
         const double* __restrict__ pin, int nb_in, double* __restrict__ hsave, double* __restrict__ pout) {
  constexpr int NV = 8 * MG;
  extern __shared__ double sh_h[];
  __shared__ double sh_w[CGS_THREADS / 64][NV];
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  auto h = [&](int i) { return LONG ? pin[i] : sh_h[i]; };
  if constexpr (AXPY) {
    if constexpr (!LONG) sum_partial_rows(pin, m, nb_in, nb_in, sh_h);
    if (blockIdx.x == 0)
      for (int i = tid; i < m; i += CGS_THREADS) hsave[i] = h(i);
  }
  const int64_t stride = (int64_t)gridDim.x * CGS_THREADS, t0 = (int64_t)blockIdx.x * CGS_THREADS + tid;
  for (int i0 = 0; i0 < m; i0 += NV) {
    double acc[NV];
#pragma unroll
    for (int i = 0; i < NV; ++i) acc[i] = 0.0;
    for (int64_t t = t0; t < n; t += stride) {
      double v[NV];
#pragma unroll
      for (int i = 0; i < NV; ++i) v[i] = i0 + i < m ? V[(int64_t)(i0 + i) * ldv + t] : 0.0;
      double wt = w[t];
      if (AXPY && i0 == 0) {
#pragma unroll
        for (int i = 0; i < NV; ++i)
          if (i < m) wt -= h(i) * v[i];
        for (int i = NV; i < m; ++i) wt -= h(i) * V[(int64_t)i * ldv + t];
        w[t] = wt;
      }
#pragma unroll
      for (int i = 0; i < NV; ++i) acc[i] += v[i] * wt;
    }
    const double x = wave_sums<NV>(acc);
    if (lane % (64 / NV) == 0) sh_w[wave][lane / (64 / NV)] = x;
    __syncthreads();
    if (tid < NV && i0 + tid < m) {
      double y = 0.0;
#pragma unroll
      for (int k = 0; k < CGS_THREADS / 64; ++k) y += sh_w[k][tid];
      pout[(int64_t)(i0 + tid) * gridDim.x + blockIdx.x] = y;
    }
    __syncthreads();
  }
}

// w -= sum_i h_i V_i with h the sums of pin's rows, and the partial sum of w^2
// (m = 0: w = b - w, the residual of a cycle's start)
template <int MG, bool LONG>
__global__ void __launch_bounds__(CGS_THREADS)
cgs_norm(const double* __restrict__ V, int m, int64_t ldv, const double* __restrict__ b, const double* w, double* out,
         int64_t n, const double* __restrict__ pin, int nb_in, double* __restrict__ hsave,
         double* __restrict__ pout) {
  extern __shared__ double sh_h[];
  __shared__ double sh_w[CGS_THREADS / 64];
  const int tid = threadIdx.x;
  auto h = [&](int i) { return LONG ? pin[i] : sh_h[i]; };
  if (m > 0) {
    if constexpr (!LONG) sum_partial_rows(pin, m, nb_in, nb_in, sh_h);
    if (blockIdx.x == 0)
      for (int i = tid; i < m; i += CGS_THREADS) hsave[i] = h(i);
  }
  const int64_t stride = (int64_t)gridDim.x * CGS_THREADS;
  double acc = 0.0;
  for (int64_t t = (int64_t)blockIdx.x * CGS_THREADS + tid; t < n; t += stride) {
    double wt = m > 0 ? w[t] : (w ? b[t] - w[t] : b[t]);
    for (int i0 = 0; i0 < m; i0 += 8 * MG) {
      double v[8 * MG];
#pragma unroll
      for (int i = 0; i < 8 * MG; ++i) v[i] = i0 + i < m ? V[(int64_t)(i0 + i) * ldv + t] : 0.0;
#pragma unroll
      for (int i = 0; i < 8 * MG; ++i)
        if (i0 + i < m) wt -= h(i0 + i) * v[i];
    }
    out[t] = wt;
    acc += wt * wt;
  }
  acc = wave_sum(acc);
  if ((tid & 63) == 0) sh_w[tid >> 6] = acc;
  __syncthreads();
  if (tid == 0) {
    double y = 0.0;
#pragma unroll
    for (int k = 0; k < CGS_THREADS / 64; ++k) y += sh_w[k];
    pout[blockIdx.x] = y;
  }
}

// w /= ||w|| (left alone when the norm is not positive); the column h1 + h2
// and the norm go to host memory that the host reads after the step's event
__global__ void __launch_bounds__(CGS_THREADS)
cgs_finish(double* __restrict__ w, int64_t n, const double* __restrict__ pin, int nb_in, int m,
           const double* __restrict__ h1, const double* __restrict__ h2, double* __restrict__ host) {
  __shared__ double sh_h[8];
  sum_partial_rows(pin, 1, nb_in, nb_in, sh_h);
  const double hn = sqrt(sh_h[0]);
  if (blockIdx.x == 0) {
    for (int i = threadIdx.x; i < m; i += CGS_THREADS) host[i] = h1[i] + h2[i];
    if (threadIdx.x == 0) host[m] = hn;
  }
  const double inv = hn > 0.0 ? 1.0 / hn : 1.0;
  const int64_t stride = (int64_t)gridDim.x * CGS_THREADS;
  for (int64_t t = (int64_t)blockIdx.x * CGS_THREADS + threadIdx.x; t < n; t += stride) w[t] = inv * w[t];
}

// out[i] = sum of partial[i][0 .. nb)
__global__ void __launch_bounds__(CGS_THREADS)
multidot_reduce(const double* __restrict__ partial, int nb, double* __restrict__ out) {
  __shared__ double sh[CGS_THREADS / 64];
  double acc = 0.0;
  for (int b = threadIdx.x; b < nb; b += CGS_THREADS) acc += partial[(int64_t)blockIdx.x * nb + b];
  acc = wave_sum(acc);
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = acc;
  __syncthreads();
  if (threadIdx.x == 0) {
    double y = 0.0;
#pragma unroll
    for (int k = 0; k < CGS_THREADS / 64; ++k) y += sh[k];
    out[blockIdx.x] = y;
  }
}

// y = a*x (+ y if accumulate)
__global__ void scale_kernel(const double* __restrict__ x, double* __restrict__ y, double a, int accumulate, int64_t n) {
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; t < n; t += stride)
    y[t] = accumulate ? y[t] + a * x[t] : a * x[t];
}

// y = sum_i c[i] V_i  (c on the host, passed through a small device buffer)
__global__ void combine_kernel(const double* __restrict__ V, int m, int64_t ldv, const double* __restrict__ cf,
                               double* __restrict__ y, int64_t n) {
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; t < n; t += stride) {
    double acc = 0.0;
    for (int i = 0; i < m; ++i) acc += cf[i] * V[(int64_t)i * ldv + t];
    y[t] = acc;
  }
}

static unsigned grid_for(int64_t n) { return (unsigned)std::max<int64_t>(1, std::min<int64_t>(8192, ceil_div(n, 256))); }

struct GmresWork;
static void gmres_free(GmresWork& W);

struct GmresWork {
  double* V = nullptr;      // (restart+1) x n
  double* w = nullptr;
  double* z = nullptr;
  double* partial = nullptr;    // two sets of block partials, [restart+1][CGS_MAX_BLOCKS] each
  double* coef = nullptr;       // h of the two passes, reduced rows, solution coefficients
  // pinned host buffer, [3][restart+2]: the Hessenberg columns of the step that
  // the host reads and of the one enqueued ahead of it, the solution coefficients
  double* hcol = nullptr;
  hipEvent_t ev[2] = {nullptr, nullptr};
  int restart = 0;
  int64_t n = 0;
};

static int gmres_alloc(pdes_ctx* c, GmresWork& W, int restart) {
  if (c->gmres_ws) {
    GmresWork* cached = (GmresWork*)c->gmres_ws;
    if (cached->restart == restart && cached->n == c->numDof) { W = *cached; return PDES_OK; }
    gmres_free(*cached);
    delete cached;
    c->gmres_ws = nullptr;
  }
  W.restart = restart;
  W.n = c->numDof;
  const size_t n = (size_t)c->numDof;
  if (hipMalloc((void**)&W.V, (size_t)(restart + 1) * n * sizeof(double)) != hipSuccess ||
      hipMalloc((void**)&W.w, n * sizeof(double)) != hipSuccess ||
      hipMalloc((void**)&W.z, n * sizeof(double)) != hipSuccess ||
      hipMalloc((void**)&W.partial, (size_t)2 * (restart + 1) * CGS_MAX_BLOCKS * sizeof(double)) != hipSuccess ||
      hipMalloc((void**)&W.coef, (size_t)4 * (restart + 2) * sizeof(double)) != hipSuccess ||
      hipHostMalloc((void**)&W.hcol, (size_t)3 * (restart + 2) * sizeof(double)) != hipSuccess ||
      hipEventCreateWithFlags(&W.ev[0], hipEventDisableTiming) != hipSuccess ||
      hipEventCreateWithFlags(&W.ev[1], hipEventDisableTiming) != hipSuccess) {
    set_error("GMRES workspace allocation failed");
    gmres_free(W);
    return PDES_ERR_NOMEM;
  }
  return PDES_OK;
}

static void gmres_keep(pdes_ctx* c, GmresWork& W) {
  if (!c->gmres_ws) c->gmres_ws = new GmresWork(W);
}

static void gmres_free(GmresWork& W) {
  if (W.V) hipFree(W.V);
  if (W.w) hipFree(W.w);
  if (W.z) hipFree(W.z);
  if (W.partial) hipFree(W.partial);
  if (W.coef) hipFree(W.coef);
  if (W.hcol) hipHostFree(W.hcol);
  for (hipEvent_t& e : W.ev)
    if (e) hipEventDestroy(e);
  W = GmresWork();
}

void gmres_release(pdes_ctx* c) {
  if (c->gmres_ws) {
    gmres_free(*(GmresWork*)c->gmres_ws);
    delete (GmresWork*)c->gmres_ws;
    c->gmres_ws = nullptr;
  }
}

// rows of block partials as the next launch reads them: as they are, or
// summed once where there are many
static void cgs_rows(pdes_ctx* c, GmresWork& W, int m, double*& rows, int& nb) {
  if (nb <= CGS_SELF_REDUCE && m <= CGS_LDS_ROWS) return;
  double* out = W.coef + 2 * (W.restart + 2);
  hipLaunchKernelGGL(multidot_reduce, dim3(m), dim3(CGS_THREADS), 0, c->stream, rows, nb, out);
  rows = out;
  nb = 1;
}

template <bool AXPY>
static void launch_cgs_pass(pdes_ctx* c, GmresWork& W, int m, double* w, const double* pin, int nb_in, double* pout,
                            int nb) {
  const bool lng = AXPY && m > CGS_LDS_ROWS;
  const size_t lds = AXPY && !lng ? (size_t)m * sizeof(double) : 0;
  auto go = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3(nb), dim3(CGS_THREADS), lds, c->stream, W.V, m, W.n, w, W.n, pin, nb_in, W.coef,
                       pout);
  };
  if (m <= 8) go(cgs_pass<1, AXPY, false>);
  else if (m <= 16) go(cgs_pass<2, AXPY, false>);
  else if (!lng) go(cgs_pass<4, AXPY, false>);
  else go(cgs_pass<4, AXPY, AXPY>);
}

// w is made orthogonal to V_0 .. V_{m-1} and normalised; the column (m
// coefficients and the norm) goes to the host slot of step m - 1, which the next
// step but one writes again
static int cgs2_step(pdes_ctx* c, GmresWork& W, int m, double* w) {
  const int nb0 = cgs_blocks(W.n);
  double* pa = W.partial;
  double* pb = W.partial + (size_t)(W.restart + 1) * CGS_MAX_BLOCKS;
  double* h1 = W.coef;
  double* h2 = W.coef + W.restart + 2;
  launch_cgs_pass<false>(c, W, m, w, nullptr, 0, pa, nb0);
  double* rows = pa;
  int nb = nb0;
  cgs_rows(c, W, m, rows, nb);
  launch_cgs_pass<true>(c, W, m, w, rows, nb, pb, nb0);
  rows = pb;
  nb = nb0;
  cgs_rows(c, W, m, rows, nb);
  auto norm = [&](auto kernel) {
    const size_t lds = m > CGS_LDS_ROWS ? 0 : (size_t)m * sizeof(double);
    hipLaunchKernelGGL(kernel, dim3(nb0), dim3(CGS_THREADS), lds, c->stream, W.V, m, W.n,
                       (const double*)nullptr, w, w, W.n, rows, nb, h2, pa);
  };
  if (m <= 8) norm(cgs_norm<1, false>);
  else if (m <= 16) norm(cgs_norm<2, false>);
  else if (m <= CGS_LDS_ROWS) norm(cgs_norm<4, false>);
  else norm(cgs_norm<4, true>);
  rows = pa;
  nb = nb0;
  cgs_rows(c, W, 1, rows, nb);
  hipLaunchKernelGGL(cgs_finish, dim3(nb0), dim3(CGS_THREADS), 0, c->stream, w, W.n, rows, nb, m, h1, h2,
                     W.hcol + (size_t)((m - 1) & 1) * (W.restart + 2));
  PDES_HIP(hipGetLastError());
  return PDES_OK;
}

// V_0 = (b - w) / ||b - w|| (w null: b / ||b||); the norm goes to the host
static int cgs_start(pdes_ctx* c, GmresWork& W, const double* b, double* w) {
  const int nb0 = cgs_blocks(W.n);
  hipLaunchKernelGGL((cgs_norm<1, false>), dim3(nb0), dim3(CGS_THREADS), 0, c->stream, (const double*)nullptr, 0, W.n, b, w, W.V,
                     W.n, (const double*)nullptr, 0, (double*)nullptr, W.partial);
  double* rows = W.partial;
  int nb = nb0;
  cgs_rows(c, W, 1, rows, nb);
  hipLaunchKernelGGL(cgs_finish, dim3(nb0), dim3(CGS_THREADS), 0, c->stream, W.V, W.n, rows, nb, 0,
                     (const double*)nullptr, (const double*)nullptr, W.hcol);
  PDES_HIP(hipGetLastError());
  return PDES_OK;
}

static int apply_op(pdes_ctx* c, int mode, const double* x, double* y) {
  if (mode == 0) return launch_spmv(c, x, y, 1.0, nullptr, 0.0);
  int st = launch_residual(c, c->d_q, x, nullptr, y, false);
  if (!st && c->hom_lambda >= 0.0)
    st = launch_homotopy(c, c->d_q, x, 1.0 - c->hom_lambda, c->hom_lambda, nullptr, y);
  return st ? st : launch_ptc_shift(c, x, y);
}

// how far above the tolerance the residual estimate has to be for the next
// Arnoldi step to be enqueued ahead of it
constexpr double GMRES_NEAR = 4.0;

// GMRES(restart), right preconditioned, x0 = x on entry (device vectors).
int gmres_device(pdes_ctx* c, const double* b, double* x, double rtol, double atol, int restart, int maxit,
                 int mode, int* iters, double* resnorm, bool x_zero) {
  GmresWork W;
  int st = gmres_alloc(c, W, restart);
  if (st) return st;
  const int64_t n = W.n;
  std::vector<double> H((size_t)(restart + 1) * restart, 0.0), cs(restart), sn(restart), g(restart + 1);
  int total = 0;
  double beta = 0.0, beta0 = -1.0;
  if (x_zero) PDES_HIP(hipMemsetAsync(x, 0, n * sizeof(double), c->stream));
  // one Arnoldi step: launches only; its Hessenberg column is on the host
  // once its event has passed
  auto enqueue = [&](int j) -> int {
    double* Vn = W.V + (int64_t)(j + 1) * n;
    int sst;
    if ((sst = pc_apply(c, W.V + (int64_t)j * n, W.z)) != 0) return sst;
    if ((sst = apply_op(c, mode, W.z, Vn)) != 0) return sst;
    if ((sst = cgs2_step(c, W, j + 1, Vn)) != 0) return sst;
    PDES_HIP(hipEventRecord(W.ev[j & 1], c->stream));
    return PDES_OK;
  };
  while (true) {
    // r = b - A x  -> V_0 = r / ||r||
    if (x_zero && total == 0) {
      if ((st = cgs_start(c, W, b, nullptr)) != 0) goto done;
    } else {
      if ((st = apply_op(c, mode, x, W.w)) != 0) goto done;
      if ((st = cgs_start(c, W, b, W.w)) != 0) goto done;
    }
    PDES_HIP(hipStreamSynchronize(c->stream));
    beta = W.hcol[0];
    if (beta0 < 0) beta0 = beta;
    const double tol = std::max(rtol * beta0, atol);
    if (beta <= tol || total >= maxit) break;
    std::fill(g.begin(), g.end(), 0.0);
    g[0] = beta;
    int jdone = 0, enqueued = 0;
    double res_est = beta;
    for (int j = 0; j < restart && total < maxit; ++j) {
      if (enqueued == j && (st = enqueue(enqueued++)) != 0) goto done;
      // The next step is enqueued before this one's column is read, so the
      // device does not wait for the host in between (about 20 us a step),
      // unless the estimate is within a factor GMRES_NEAR of the tolerance and
      // this step may be the last: a step past the last one only costs time.
      if (enqueued == j + 1 && enqueued < restart && total + 1 < maxit && res_est > GMRES_NEAR * tol &&
          (st = enqueue(enqueued++)) != 0)
        goto done;
      PDES_HIP(hipEventSynchronize(W.ev[j & 1]));
      const double* col = W.hcol + (size_t)(j & 1) * (restart + 2);
      const double hn = col[j + 1];
      for (int i = 0; i <= j; ++i) H[(size_t)i * restart + j] = col[i];
      H[(size_t)(j + 1) * restart + j] = hn;
      // Givens
      for (int i = 0; i < j; ++i) {
        double a = H[(size_t)i * restart + j], bb = H[(size_t)(i + 1) * restart + j];
        H[(size_t)i * restart + j] = cs[i] * a + sn[i] * bb;
        H[(size_t)(i + 1) * restart + j] = -sn[i] * a + cs[i] * bb;
      }
      double a = H[(size_t)j * restart + j], bb = H[(size_t)(j + 1) * restart + j];
      double r = std::hypot(a, bb);
      cs[j] = r > 0 ? a / r : 1.0;
      sn[j] = r > 0 ? bb / r : 0.0;
      H[(size_t)j * restart + j] = r;
      H[(size_t)(j + 1) * restart + j] = 0.0;
      g[j + 1] = -sn[j] * g[j];
      g[j] = cs[j] * g[j];
      res_est = std::fabs(g[j + 1]);
      ++total;
      jdone = j + 1;
      if (res_est <= tol || hn == 0.0) break;
    }
    // y = H^-1 g ; x += M^-1 V y
    {
      // (the stream may still be running a step past the last one, which
      // writes its host slot, V_{jdone+1} and the work vectors only)
      std::vector<double> y(jdone);
      for (int i = jdone - 1; i >= 0; --i) {
        double s = g[i];
        for (int k = i + 1; k < jdone; ++k) s -= H[(size_t)i * restart + k] * y[k];
        y[i] = s / H[(size_t)i * restart + i];
      }
      double* ypin = W.hcol + (size_t)2 * (restart + 2);
      double* yd = W.coef + 3 * (restart + 2);
      for (int i = 0; i < jdone; ++i) ypin[i] = y[i];
      PDES_HIP(hipMemcpyAsync(yd, ypin, jdone * sizeof(double), hipMemcpyHostToDevice, c->stream));
      hipLaunchKernelGGL(combine_kernel, dim3(grid_for(n)), dim3(256), 0, c->stream, W.V, jdone, n, yd, W.w, n);
      if ((st = pc_apply(c, W.w, W.z)) != 0) goto done;
      if (x_zero && total == jdone)
        hipLaunchKernelGGL(scale_kernel, dim3(grid_for(n)), dim3(256), 0, c->stream, W.z, x, 1.0, 0, n);
      else
        hipLaunchKernelGGL(scale_kernel, dim3(grid_for(n)), dim3(256), 0, c->stream, W.z, x, 1.0, 1, n);
    }
    // The Givens estimate res_est is the residual of x + M^-1 V y only when
    // M^-1 is applied exactly; the block preconditioners apply it in FP32, so
    // the loop returns to the top, where the true residual b - A x decides
    // convergence (and, when it is still too large, seeds the next cycle).
    x_zero = false;
  }
done:
  gmres_keep(c, W);
  if (st) return st;
  if ((st = pc_check(c)) != 0) return st;
  if (iters) *iters = total;
  if (resnorm) *resnorm = beta;
  return PDES_OK;
}

}  // namespace pdes

using namespace pdes;

extern "C" {

int pdes_pc_setup(pdes_ctx* c, int kind) {
  PDES_CHECK(c, PDES_ERR_ARG, "null context");
  int st = pc_setup(c, kind);
  if (st) return st;
  if (kind != PDES_PC_NONE) {
    int32_t err = 0;
    PDES_HIP(hipMemcpyAsync(&err, c->jac->d_err, sizeof(int32_t), hipMemcpyDeviceToHost, c->stream));
    PDES_HIP(hipStreamSynchronize(c->stream));
    if (err) {
      PDES_HIP(hipMemsetAsync(c->jac->d_err, 0, sizeof(int32_t), c->stream));
      set_error("singular element block in the preconditioner factorisation");
      return PDES_ERR_PHYS;
    }
  }
  return PDES_OK;
}

int pdes_pc_apply(pdes_ctx* c, const double* b, double* x) {
  PDES_CHECK(c && b && x, PDES_ERR_ARG, "null argument");
  PDES_HIP(hipMemcpyAsync(c->d_work, b, c->numDof * sizeof(double), hipMemcpyHostToDevice, c->stream));
  int st = pc_apply(c, c->d_work, c->d_work2);
  if (st) return st;
  PDES_HIP(hipMemcpyAsync(x, c->d_work2, c->numDof * sizeof(double), hipMemcpyDeviceToHost, c->stream));
  PDES_HIP(hipStreamSynchronize(c->stream));
  return pc_check(c);
}

int pdes_gmres(pdes_ctx* c, const double* b_host, double* x_host, double rtol, double atol, int restart,
               int maxit, int mode, int* iters, double* final_resnorm) {
  PDES_CHECK(c && b_host && x_host && restart > 0 && maxit >= 0, PDES_ERR_ARG, "bad argument");
  PDES_CHECK(mode == 1 || (c->jac && c->jac->assembled), PDES_ERR_ARG, "assemble the Jacobian for mode 0");
  PDES_HIP(hipMemcpyAsync(c->d_work, b_host, c->numDof * sizeof(double), hipMemcpyHostToDevice, c->stream));
  PDES_HIP(hipMemcpyAsync(c->d_work2, x_host, c->numDof * sizeof(double), hipMemcpyHostToDevice, c->stream));
  int st = gmres_device(c, c->d_work, c->d_work2, rtol, atol, restart, maxit, mode, iters, final_resnorm, false);
  if (st) return st;
  PDES_HIP(hipMemcpyAsync(x_host, c->d_work2, c->numDof * sizeof(double), hipMemcpyDeviceToHost, c->stream));
  PDES_HIP(hipStreamSynchronize(c->stream));
  return PDES_OK;
}

// calcAdjoint (src/optimization/steady_adjoint.jl:30-66): J^T psi = -dJ/dq
// at the current state, with J assembled here, its blocks transposed in
// place for the solve (so the chosen preconditioner is built from J^T, as
// linearSolveTranspose applies the transposed preconditioner) and restored
// afterwards, with the preconditioner rebuilt from J.
int pdes_adjoint_solve(pdes_ctx* c, int kind, const int32_t* bcnums, int nbc, int pc_kind, int fp64_blocks,
                       double rtol, double atol, int restart, int maxit, double* psi, int* iters,
                       double* final_resnorm) {
  PDES_CHECK(c && psi && restart > 0 && maxit >= 0, PDES_ERR_ARG, "bad argument");
  const int64_t n = c->numDof;
  int st = jacobian_setup(c, fp64_blocks);
  if (st) return st;
  c->ptc_on = false;
  if ((st = assemble(c))) return st;
  // rhs = -dJ/dq in d_work, psi in d_work2 (x0 = 0)
  if ((st = functional_grad_device(c, kind, bcnums, nbc, c->d_work))) return st;
  hipLaunchKernelGGL(scale_kernel, dim3(grid_for(n)), dim3(256), 0, c->stream, c->d_work, c->d_work, -1.0, 0, n);
  hipLaunchKernelGGL(scale_kernel, dim3(grid_for(n)), dim3(256), 0, c->stream, c->d_work, c->d_work2, 0.0, 0, n);
  PDES_HIP(hipGetLastError());
  if ((st = transpose_jacobian(c))) return st;
  int gst = pc_setup(c, pc_kind);
  if (!gst) gst = gmres_device(c, c->d_work, c->d_work2, rtol, atol, restart, maxit, 0, iters, final_resnorm, true);
  // restore J and its preconditioner whatever the solve returned
  if ((st = transpose_jacobian(c))) return st;
  if ((st = pc_setup(c, pc_kind))) return st;
  if (gst) return gst;
  PDES_HIP(hipMemcpyAsync(psi, c->d_work2, n * sizeof(double), hipMemcpyDeviceToHost, c->stream));
  PDES_HIP(hipStreamSynchronize(c->stream));
  return PDES_OK;
}

int pdes_newton_solve(pdes_ctx* c, const pdes_newton_opts* o, pdes_newton_report* rep) {
  PDES_CHECK(c && o && rep, PDES_ERR_ARG, "null argument");
  PDES_CHECK(!o->globalize_euler || o->euler_tau > 0, PDES_ERR_ARG, "euler_tau must be positive");
  auto t0 = std::chrono::steady_clock::now();
  *rep = pdes_newton_report{};
  const int64_t n = c->numDof;
  int st;
  double* res = c->d_res;
  // every exit, the early returns of the HIP checks included, turns the
  // implicit-Euler term off and frees the workspace
  struct Guard {
    pdes_ctx* c;
    double* dq = nullptr;
    double* rhs = nullptr;
    ~Guard() {
      c->ptc_on = false;
      hipStreamSynchronize(c->stream);
      if (dq) hipFree(dq);
      if (rhs) hipFree(rhs);
    }
  } guard{c};
  PDES_CHECK(hipMalloc((void**)&guard.dq, n * sizeof(double)) == hipSuccess &&
             hipMalloc((void**)&guard.rhs, n * sizeof(double)) == hipSuccess, PDES_ERR_NOMEM, "Newton workspace");
  double* const dq = guard.dq;
  double* const rhs = guard.rhs;
  auto norm_res = [&](double* out) -> int {
    int s2 = launch_residual(c, c->d_q, nullptr, res, nullptr, c->phys.check_positivity != 0);
    if (!s2 && c->hom_lambda >= 0.0)
      s2 = launch_homotopy(c, c->d_q, nullptr, 1.0 - c->hom_lambda, c->hom_lambda, res, nullptr);
    if (s2) return s2;
    s2 = launch_wnorm2(c, res, c->d_Minv, n, 0);
    return s2 ? s2 : wait_norm(c, out);
  };
  double nrm = 0, tau = 0, prev_nrm = 0;
  if ((st = norm_res(&nrm)) != 0) goto fin;
  rep->res_norm0 = nrm;
  rep->res_norm = nrm;
  if (nrm < o->res_abstol) { rep->converged = 1; goto fin; }
  if ((st = jacobian_setup(c, o->fp64_blocks)) != 0) goto fin;
  for (int it = 1; it <= o->itermax; ++it) {
    if (o->globalize_euler) {
      // updateEuler at each Jacobian evaluation (globalization.jl:237-262)
      if (it == 1) {
        tau = o->euler_tau;
        if (o->scale_euler) tau *= 1.0 / nrm;
      } else {
        tau *= prev_nrm / nrm;
      }
      prev_nrm = nrm;
      if ((st = set_ptc_scale(c, &tau, 1)) != 0) goto fin;
    }
    // doRecalculation: Jacobian and preconditioner every iteration (recalc_freq 1)
    if ((st = c->hom_lambda >= 0.0 ? assemble_homotopy(c, c->hom_lambda) : assemble(c)) != 0) goto fin;
    if ((st = pdes_pc_setup(c, o->pc_kind)) != 0) goto fin;
    hipLaunchKernelGGL(scale_kernel, dim3(grid_for(n)), dim3(256), 0, c->stream, res, rhs, -1.0, 0, n);
    int kits = 0;
    double kres = 0;
    if ((st = gmres_device(c, rhs, dq, o->krylov_reltol, o->krylov_abstol, o->gmres_restart, o->krylov_itermax,
                           o->jv_mode, &kits, &kres, true)) != 0)
      goto fin;
    rep->total_krylov_iters += kits;
    hipLaunchKernelGGL(scale_kernel, dim3(grid_for(n)), dim3(256), 0, c->stream, dq, c->d_q, 1.0, 1, n);
    // step norm: norm(delta_q_vec)
    if ((st = launch_wnorm2(c, dq, nullptr, n, 1)) != 0) goto fin;
    if ((st = norm_res(&nrm)) != 0) goto fin;
    rep->step_norm = std::sqrt(c->h_norm->sum[1]);
    rep->res_norm = nrm;
    rep->iterations = it;
    // checkConvergence (newton.jl:402-455)
    if (nrm < o->res_abstol || nrm / rep->res_norm0 < o->res_reltol || rep->step_norm <= o->step_tol) {
      rep->converged = 1;
      break;
    }
  }
fin:
  rep->elapsed_s = std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
  return st;
}

// predictorCorrectorHomotopy (src/NonlinearSolvers/predictor_corrector.jl:
// HomotopyData :63-148, the loop :226-326, updateTolerances :381-440,
// calcTangentVector :454-476, calcdHdLambda :495-530, takePredictorStep
// :535-595).  H(q, lambda) = (1 - lambda) R(q) + lambda D(q), lambda from 1 to
// 0: each predictor iteration runs a Newton corrector on H (tolerance
// homotopy_tol = 1e-2 relative while lambda > 0, res_reltol at lambda = 0,
// at most 30 iterations), then solves dH/dq t = dH/dlambda = D - R with the
// corrector's last Jacobian and preconditioner, normalises t with the SBP
// norm, sets the step h from the angle between successive tangents (limit
// psi_max) and the corrector's step length (limit 1), and takes
// lambda -= h, q += h t.  The loop ends on the physics residual:
// ||R|| <= res_abstol or ||R|| / ||R_0|| <= res_reltol, or itermax
// predictor iterations.
int pdes_homotopy_solve(pdes_ctx* c, const pdes_newton_opts* o, double psi_max, pdes_newton_report* rep) {
  PDES_CHECK(c && o && rep, PDES_ERR_ARG, "null argument");
  PDES_CHECK(psi_max > 0, PDES_ERR_ARG, "psi_max must be positive");
  PDES_CHECK(!o->globalize_euler, PDES_ERR_UNSUPPORTED, "homotopy with implicit-Euler globalization is not available");
  auto t0 = std::chrono::steady_clock::now();
  *rep = pdes_newton_report{};
  const int64_t n = c->numDof;
  const double eps = 2.220446049250313e-16;
  std::vector<double> M(n), t(n), t1(n), q(n), q0(n);
  // every exit, the early returns of the HIP checks included, leaves the
  // context solving the physics again and frees the workspace
  struct Guard {
    pdes_ctx* c;
    double* d_t = nullptr;
    double* d_rhs = nullptr;
    ~Guard() {
      c->hom_lambda = -1.0;
      hipStreamSynchronize(c->stream);
      if (d_t) hipFree(d_t);
      if (d_rhs) hipFree(d_rhs);
    }
  } guard{c};
  int st = PDES_OK;
  PDES_CHECK(hipMalloc((void**)&guard.d_t, n * sizeof(double)) == hipSuccess &&
             hipMalloc((void**)&guard.d_rhs, n * sizeof(double)) == hipSuccess, PDES_ERR_NOMEM, "homotopy workspace");
  double* const d_t = guard.d_t;
  double* const d_rhs = guard.d_rhs;
  auto phys_norm = [&](double* out) -> int {
    c->hom_lambda = -1.0;
    int s2 = launch_residual(c, c->d_q, nullptr, c->d_res, nullptr, c->phys.check_positivity != 0);
    if (!s2) s2 = launch_wnorm2(c, c->d_res, c->d_Minv, n, 0);
    return s2 ? s2 : wait_norm(c, out);
  };
  // calcNorm (Utils.jl:427-449) and calcL2InnerProduct (:476-493): M-weighted
  auto mdot = [&](const std::vector<double>& a, const std::vector<double>& b) {
    double acc = 0.0;
    for (int64_t i = 0; i < n; ++i) acc += a[i] * M[i] * b[i];
    return acc;
  };
  double lambda = 1.0, h = 0.05, h_max = 0.1, delta_max = 1.0, hom_tol = 1e-2, tan_norm_1 = 0.0;
  double res_norm = 0.0;
  int iter = 1;
  lambda -= h;   // the Jacobian at lambda = 1 is ill-conditioned; start one step in
  {
    std::vector<double> minv(n);
    PDES_HIP(hipMemcpyAsync(minv.data(), c->d_Minv, n * sizeof(double), hipMemcpyDeviceToHost, c->stream));
    PDES_HIP(hipStreamSynchronize(c->stream));
    for (int64_t i = 0; i < n; ++i) M[i] = 1.0 / minv[i];
  }
  if ((st = phys_norm(&res_norm)) != 0) goto done;
  rep->res_norm0 = res_norm;
  while (res_norm > rep->res_norm0 * o->res_reltol && res_norm > o->res_abstol && iter < o->itermax) {
    // updateTolerances
    if (std::fabs(lambda) <= eps) hom_tol = o->res_reltol;
    // corrector
    PDES_HIP(hipMemcpyAsync(q0.data(), c->d_q, n * sizeof(double), hipMemcpyDeviceToHost, c->stream));
    c->hom_lambda = lambda;
    pdes_newton_opts no = *o;
    no.res_reltol = hom_tol;
    no.itermax = 30;
    pdes_newton_report nrep{};
    if ((st = pdes_newton_solve(c, &no, &nrep)) != 0) goto done;
    rep->total_krylov_iters += nrep.total_krylov_iters;
    if (std::fabs(lambda) > eps) {
      // tangent: dH/dq t = D(q) - R(q), with the corrector's last operator
      if ((st = launch_residual(c, c->d_q, nullptr, c->d_res, nullptr, false)) != 0) goto done;
      if ((st = launch_homotopy(c, c->d_q, nullptr, 0.0, 1.0, d_rhs, nullptr)) != 0) goto done;
      hipLaunchKernelGGL(scale_kernel, dim3(grid_for(n)), dim3(256), 0, c->stream, c->d_res, d_rhs, -1.0, 1, n);
      if (nrep.iterations == 0) {
        if ((st = jacobian_setup(c, o->fp64_blocks)) != 0) goto done;
        if ((st = assemble_homotopy(c, lambda)) != 0) goto done;
        if ((st = pdes_pc_setup(c, o->pc_kind)) != 0) goto done;
      }
      int kits = 0;
      double kres = 0;
      if ((st = gmres_device(c, d_rhs, d_t, o->krylov_reltol, o->krylov_abstol, o->gmres_restart, o->krylov_itermax,
                             o->jv_mode, &kits, &kres, true)) != 0)
        goto done;
      rep->total_krylov_iters += kits;
      PDES_HIP(hipMemcpyAsync(t.data(), d_t, n * sizeof(double), hipMemcpyDeviceToHost, c->stream));
      PDES_HIP(hipMemcpyAsync(q.data(), c->d_q, n * sizeof(double), hipMemcpyDeviceToHost, c->stream));
      PDES_HIP(hipStreamSynchronize(c->stream));
      // takePredictorStep
      double tan_norm = std::sqrt(mdot(t, t) + 1.0);
      for (int64_t i = 0; i < n; ++i) t[i] /= tan_norm;
      for (int64_t i = 0; i < n; ++i) q0[i] = q[i] - q0[i];
      const double delta = std::sqrt(mdot(q0, q0));
      double psi = psi_max;
      if (iter > 1) {
        const double arg = std::min(1.0, std::max(-1.0, mdot(t1, t) + 1.0 / (tan_norm * tan_norm_1)));
        psi = std::acos(arg);
      }
      const double fac = std::max(psi / psi_max, std::sqrt(delta / delta_max));
      h /= fac;
      h = std::min(h, h_max);
      lambda = std::max(0.0, lambda - h);
      if (lambda < eps) lambda = 0.0;
      for (int64_t i = 0; i < n; ++i) q[i] += h * t[i];
      PDES_HIP(hipMemcpyAsync(c->d_q, q.data(), n * sizeof(double), hipMemcpyHostToDevice, c->stream));
      t1.swap(t);
      tan_norm_1 = tan_norm;
    }
    if ((st = phys_norm(&res_norm)) != 0) goto done;
    rep->iterations = iter;
    ++iter;
  }
  rep->res_norm = res_norm;
  rep->converged = (res_norm <= o->res_abstol || res_norm <= rep->res_norm0 * o->res_reltol) ? 1 : 0;
done:
  rep->elapsed_s = std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
  return st;
}

}  // extern "C"
