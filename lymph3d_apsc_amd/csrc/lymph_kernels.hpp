// lymph_kernels.hpp -- gfx950 kernels of the PolyDG leapfrog path.
//
// Data layout in HBM (one context):
//  * operator K and A_dg: one block row per polyhedron, blocks of 3Np x 3Np
//    FP64 in "column-pair" order: entry (r, c) of block b sits at
//      b*N3*N3C + ((c>>1)*N3 + r)*2 + (c&1),     N3 = 3Np, N3C = N3 rounded up
//    to even (padding column zero).  A 64-lane wave with lane = row r reads one
//    column pair of a block as a single 16-byte load per lane: N3*16 contiguous
//    bytes per wave instruction, every byte of the block read exactly once.
//  * mass factors R (upper, M = R^T R): packed row-major upper triangle,
//    Np(Np+1)/2 doubles per polyhedron (the bytes the step must read).
//  * vectors: 3Np doubles per polyhedron, component-major inside.
#pragma once
#include "lymph_math.hpp"

namespace lymph {

template <int P>
struct Dims {
  static constexpr int NP = np_of(P);
  static constexpr int N3 = 3 * NP;
  static constexpr int N3C = (N3 + 1) & ~1;
  static constexpr int NPAIR = N3C / 2;
  static constexpr int NQ1 = P + 1;
  static constexpr int NQ3 = NQ1 * NQ1 * NQ1;
  static constexpr int NQ2 = NQ1 * NQ1;
  static constexpr int NPK = NP * (NP + 1) / 2;
  static constexpr size_t BS = (size_t)N3 * N3C;
};

// Operator blocks are read exactly once per step.  Where the operator does not
// stay in the caches until the next step, non-temporal loads (NT) keep them
// from displacing the coefficient vectors (which neighbours re-read).
typedef double lymph_dv2 __attribute__((ext_vector_type(2)));
typedef float lymph_fv4 __attribute__((ext_vector_type(4)));
typedef float lymph_fv2 __attribute__((ext_vector_type(2)));
template <bool NT = true>
__device__ inline double2 load_stream(const double* p) {
  const auto* q = reinterpret_cast<const lymph_dv2*>(p);
  const lymph_dv2 t = NT ? __builtin_nontemporal_load(q) : *q;
  return make_double2(t.x, t.y);
}
template <bool NT = true>
__device__ inline float4 load_stream(const float* p) {
  const auto* q = reinterpret_cast<const lymph_fv4*>(p);
  const lymph_fv4 t = NT ? __builtin_nontemporal_load(q) : *q;
  return make_float4(t.x, t.y, t.z, t.w);
}
// the tail columns of a 32-bit block row (N3 % 4 of them; 1 or 2 for p <= 4)
template <bool NT, int T>
__device__ inline void load_tail(const float* p, float (&v)[T]) {
  static_assert(T == 1 || T == 2, "tail of 1 or 2 columns");
  if constexpr (T == 2) {
    const auto* q = reinterpret_cast<const lymph_fv2*>(p);
    const lymph_fv2 t = NT ? __builtin_nontemporal_load(q) : *q;
    v[0] = t.x;
    v[1] = t.y;
  } else {
    v[0] = NT ? __builtin_nontemporal_load(p) : *p;
  }
}

LYMPH_HD size_t kpos(int N3, int r, int c) {
  return ((size_t)(c >> 1) * N3 + r) * 2 + (c & 1);
}

// Layout of a 32-bit block: the first 4*NQ columns as column quads (entry
// (r, c) at ((c>>2)*N3 + r)*4 + (c&3)), then the T = N3 % 4 tail columns
// row by row (at 4*NQ*N3 + r*T + c - 4*NQ); no padding columns, so the block
// stream is exactly N3^2 floats (the block stride is rounded up to 4 floats
// to keep every block 16-byte aligned).
template <int P>
struct Dims32 {
  static constexpr int N3 = 3 * np_of(P);
  static constexpr int NQ = N3 / 4, T = N3 % 4;
  static constexpr size_t BS = ((size_t)N3 * N3 + 3) / 4 * 4;
};
// The 48-bit apply's 16-bit corrections: column quads taken in pairs, a
// row's 8 values of quads 2k, 2k+1 contiguous (one 16-byte load); the last
// quad of an odd count row by row at 4 values per row (one 8-byte load, no
// half-empty slots to come in with the lines); then the N3 % 4 tail columns
// row by row; blocks padded to 8 values (none at p = 1, 3).
template <int P>
struct Dims16 {
  static constexpr int N3 = 3 * np_of(P);
  static constexpr int NQ = N3 / 4, T = N3 % 4, NPF = NQ / 2, NPR = (NQ + 1) / 2;
  static constexpr size_t HALF0 = (size_t)NPF * N3 * 8;
  static constexpr size_t TAIL0 = HALF0 + (size_t)(NQ % 2) * N3 * 4;
  static constexpr size_t BS = (TAIL0 + (size_t)N3 * T + 7) / 8 * 8;
};
LYMPH_HD size_t kpos16(int N3, int r, int c) {
  const int c0 = N3 / 4 * 4, nq = N3 / 4, npf = nq / 2;
  const size_t half0 = (size_t)npf * N3 * 8;
  if (c < c0) {
    const int q = c >> 2;
    if (q < 2 * npf) return ((size_t)(q >> 1) * N3 + r) * 8 + (q & 1) * 4 + (c & 3);
    return half0 + (size_t)r * 4 + (c & 3);
  }
  return half0 + (size_t)(nq % 2) * N3 * 4 + (size_t)r * (N3 % 4) + (c - c0);
}
// The corrections' loads: 8 (a quad pair's row) or 4 (the last quad's row)
// halves, non-temporal like the operator's own.
typedef _Float16 lymph_hv4 __attribute__((ext_vector_type(4)));
typedef _Float16 lymph_hv8 __attribute__((ext_vector_type(8)));
template <bool NT = true>
__device__ inline lymph_hv8 load_stream_h8(const _Float16* p) {
  const auto* q = reinterpret_cast<const lymph_hv8*>(p);
  return NT ? __builtin_nontemporal_load(q) : *q;
}
template <bool NT = true>
__device__ inline lymph_hv4 load_stream_h4(const _Float16* p) {
  const auto* q = reinterpret_cast<const lymph_hv4*>(p);
  return NT ? __builtin_nontemporal_load(q) : *q;
}
LYMPH_HD size_t kpos32(int N3, int r, int c) {
  const int c0 = N3 / 4 * 4;
  if (c < c0) return ((size_t)(c >> 2) * N3 + r) * 4 + (c & 3);
  return (size_t)c0 * N3 + (size_t)r * (N3 % 4) + (c - c0);
}
LYMPH_HD int pk_off(int NP, int i) { return i * NP - i * (i - 1) / 2; }
// Doubles per block product of the pairs-once steps: whole 128-byte lines, so
// that each product's store covers its lines entirely (the padding lanes
// write zeros) instead of leaving partial lines that other waves complete.
LYMPH_HD constexpr int prod_stride(int n3) { return (n3 + 15) & ~15; }

struct MeshDev {
  const double* tet_xyz;  // n_tet*12
  const int* tet_poly;
  const int* neigh;       // n_tet*4
  const int* bc_space;    // n_tet*4
  const double* normal;   // n_tet*12
  const double* area;     // n_tet*4
  const double* rho;
  const double* lam;
  const double* mu;
  const double* bbox;     // n_poly*6
  const double* hk;       // n_poly
  const int* ptet_ptr;    // n_poly+1
  const int* ptet;        // n_tet
  const int* row_ptr;     // n_poly+1
  const int* col;         // n_blk
  const int* face_blk;    // n_tet*4 block index of the neighbour block, -1 if none
  const double* qtet;     // NQ3*4
  const double* wtet;     // NQ3
  const double* qtri;     // NQ2*4
  const double* wtri;     // NQ2
  const int* blist;       // NP*3
};

// ---------------------------------------------------------------------------
// Basis tables.  At a point the basis functions are products of 1-D values
// v_d[k] = L_k(x_d) / sqrt(h_d) and their derivatives; each 1-D value costs a
// square root and a division, so a workgroup forms them once per point,
// dimension and degree (tab1d) and the products from LDS (basis_row), in
// basis_at's operand order.  Tables run over the functions first ([q][f]):
// lanes hold neighbouring functions, and their reads fall in distinct banks
// ([f][q] put all of them in one).
// ---------------------------------------------------------------------------
// Row d of affine_map's matrix from the tet's vertices (same expressions).
__device__ __forceinline__ void affine_row(const double* __restrict__ v, int d, double (&r)[4]) {
  const double x1 = v[d], x2 = v[3 + d], x3 = v[6 + d], x4 = v[9 + d];
  r[0] = ((0.0 + -1 * x1) + 1 * x2) + 0 * x3 + 0 * x4;
  r[1] = ((0.0 + -1 * x1) + 0 * x2) + 1 * x3 + 0 * x4;
  r[2] = ((0.0 + -1 * x1) + 0 * x2) + 0 * x3 + 1 * x4;
  r[3] = ((0.0 + 1 * x1) + 0 * x2) + 0 * x3 + 0 * x4;
}
// Coordinate d of map_point / face_point from row d.
__device__ __forceinline__ double map_coord(const double (&r)[4], const double* __restrict__ nod4) {
  double s = 0.0;
#pragma unroll
  for (int l = 0; l < 4; ++l) s = s + r[l] * nod4[l];
  return s;
}
__device__ __forceinline__ double face_coord(const double (&r)[4], int face, const double* __restrict__ tri4) {
  double s = 0.0;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    double t = 0.0;
#pragma unroll
    for (int l = 0; l < 4; ++l) t = t + r[l] * node_map(face, l, q);
    s = s + t * tri4[q];
  }
  return s;
}

// 1-D values of one bounding box at NQ points: v[d][k][q], dv[d][k][q]
template <int P, int NQ>
struct Tab1 {
  double v[3][P + 1][NQ], dv[3][P + 1][NQ];
};
template <int P, int NQ>
__device__ __forceinline__ void tab1d(Tab1<P, NQ>& t, int d, int q, double x, double lo, double hi) {
  const double hb = (hi - lo) / 2.0;
  const double mb = (hi + lo) / 2.0;
  const double sq = sqrt(hb);
  const double xp = (x - mb) / hb;
#pragma unroll
  for (int k = 0; k <= P; ++k) {
    t.v[d][k][q] = leg(k, xp) / sq;
    t.dv[d][k][q] = dleg(k, xp) / (hb * sq);
  }
}
// phi and gradient of the function with degrees (a, b, c) at point q
template <int P, int NQ>
__device__ __forceinline__ void basis_row(const Tab1<P, NQ>& t, int a, int b, int c, int q, double& phi, double& d0,
                                          double& d1, double& d2) {
  const double v0 = t.v[0][a][q], v1 = t.v[1][b][q], v2 = t.v[2][c][q];
  phi = v0 * v1 * v2;
  d0 = t.dv[0][a][q] * v1 * v2;
  d1 = v0 * t.dv[1][b][q] * v2;
  d2 = v0 * v1 * t.dv[2][c][q];
}

// ---------------------------------------------------------------------------
// Operator build: MAKE_MATRICES_FREE (src/matrix_free.f90:27-464).  A group of
// TG threads per polyhedron, a basis pair (m, n) with its nine component
// entries per thread; the tets are
// processed in order (volume term, then faces 1..4), and the self block's
// entries stay in registers to the end, so every entry accumulates in the
// reference's order and is written once; a neighbour's block is stored at its
// first face and added to at the others.
//
// REF evaluates the reference's terms in its operand order.  !REF uses that
// the face and volume terms of MAKE_STIFFNESS_VOLUME / MAKE_STIFFNESS_FACE are
// bilinear in the basis values, so each is a combination of a few quadrature
// sums per basis pair (m, n):
//   volume:  D_ab = sum_q w|J| d_a phi_m d_b phi_n  (a, b = x, y, z)
//     V_ii = (l+2m) D_ii + m sum_{a != i} D_aa,  V_ij = l D_ij + m D_ji;
//   face:    PP = sum w phiP_m phiP_n,  PQ = sum w phiP_m phiQ_n,
//            BP_a = sum w d_a phiP_m phiP_n,  BPt_a = sum w d_a phiP_n phiP_m,
//            CP_a = sum w d_a phiP_m phiQ_n,  DQ_a = sum w d_a phiQ_n phiP_m,
//     with T(i,j;X) = i==j ? (l+2m) n_i X_i + m sum_{a != i} n_a X_a
//                          : l n_j X_i + m n_i X_j,
//     S+ = s ar PP c_ij, I+ = k ar T(i,j;BP), I+^T = k ar T(j,i;BPt),
//     I- = -ar/2 T(i,j;CP), I-^T = ar/2 T(i,j;DQ), S- = -s ar PQ c_ij,
//     c_ii = dd_i, c_ij = n_i n_j / 2, k = 1 (Dirichlet) or 1/2 (interior);
// sums are regrouped relative to the reference, so entries agree with it to
// rounding (1e-15 relative), not bit for bit.  The mass blocks are summed the
// same way in both.
//
// Bound by FP64 instructions (no contraction: the reference's roundings).  A
// face's transposed consistency term of entry (i, j; m, n) is its plain one of
// (j, i; n, m), so REF exchanges it through LDS instead of summing it again.
// What it replaced read its tables with every lane in one bank, evaluated each
// function's 1-D values (three square roots, six divisions) per point anew and
// added every tet and face into the blocks in memory.  Milliseconds, then ->
// now, reference / factored order, both operators, agglomerated cubes: p = 1
// (64,000 polyhedra) 17.6 -> 1.3 / 7.1 -> 1.1; p = 2 (32,768) 35.9 -> 6.5 / 11.7
// -> 4.0; p = 3 (13,824) 123 -> 20 / 29.6 -> 10.5; p = 4 (4,096) 233 -> 32 / 31
// -> 11.  At p = 3 the reference order keeps the vector units 62% busy, 58% of
// the time with FP64; the factored one 40%, with as many LDS instructions for a
// quarter of the FP64 ones.
// ---------------------------------------------------------------------------
template <int P, bool ONE = false>
struct Build {
  static constexpr int PAIRS = np_of(P) * np_of(P);
  // p = 1: 16 pairs, four polyhedra a wave (ONE: one); p = 2: 100 pairs in two
  // waves; p = 3: 400 in seven; p = 4: 1225 in two workgroups of ten (two pairs
  // a thread in one spilled 210 registers)
  static constexpr int GP = P == 1 && !ONE ? 4 : 1;
  static constexpr int TG = P == 1 ? (ONE ? 64 : 16) : (P == 2 ? 128 : (P == 3 ? 448 : 640));
  static constexpr int SPLIT = (PAIRS + TG - 1) / TG;
  static constexpr int SHARE = (PAIRS + SPLIT - 1) / SPLIT;  // pairs per workgroup
  static constexpr int TPB = GP * TG;
  static constexpr int NQ2 = (P + 1) * (P + 1), NQ3 = NQ2 * (P + 1);
  static constexpr int NB = GP > 1 ? 2 : 8;  // tets fetched at a time
  static constexpr int QC = P <= 2 ? NQ3 : 2 * NQ2 <= 32 ? 32 : NQ2;  // volume points per table
  static_assert(NQ3 % QC == 0, "whole chunks of the volume rule");
};

// acc[3 i + j] += c I(i, j), the consistency term sigma(grad) : (phi (x) n) of
// :504-515 with the component pattern: gradient (G0, G1, G2) on one side,
// value ph on the other.
__device__ __forceinline__ void face_terms(double (&acc)[9], double c, double G0, double G1, double G2, double ph,
                                           double lam, double mu, double l2m, double n1, double n2, double n3) {
  const double a0 = l2m * G0 * ph, a1 = l2m * G1 * ph, a2 = l2m * G2 * ph;
  const double u0 = mu * G0 * ph, u1 = mu * G1 * ph, u2 = mu * G2 * ph;
  const double l0 = lam * G0 * ph, l1 = lam * G1 * ph, l2 = lam * G2 * ph;
  const double w0 = u0 * n1, w1 = u1 * n2, w2 = u2 * n3;
  acc[0] = acc[0] + c * (a0 * n1 + w1 + w2);
  acc[4] = acc[4] + c * (a1 * n2 + w0 + w2);
  acc[8] = acc[8] + c * (a2 * n3 + w1 + w0);
  acc[1] = acc[1] + c * (l0 * n2 + u1 * n1);
  acc[2] = acc[2] + c * (l0 * n3 + u2 * n1);
  acc[3] = acc[3] + c * (l1 * n1 + u0 * n2);
  acc[5] = acc[5] + c * (l1 * n3 + u2 * n2);
  acc[6] = acc[6] + c * (l2 * n1 + u0 * n3);
  acc[7] = acc[7] + c * (l2 * n2 + u1 * n3);
}

// What a workgroup needs of a few tets ahead, fetched for all of them at once
// (one walk tet -> neighbour -> polyhedron -> its box per polyhedron instead
// of one per face).
struct BuildFace {
  double n[3], ar, sigma, bb[6];  // normal, area, penalty, the neighbour's box
  int Q, blk;                     // neighbour polyhedron (-1: Dirichlet), its block; Q = -2: no term
};
struct BuildTet {
  double v[12], aJ, rho, lam, mu;
  BuildFace f[4];
};

template <int P, bool REF, bool ADG, bool ONE = false>
__global__ __launch_bounds__((Build<P, ONE>::TPB), !REF && (P == 2 || P == 3) ? 4 : 2) void k_build(
    MeshDev m, double alpha, double theta, double* __restrict__ K, double* __restrict__ A, double* __restrict__ M,
    double* __restrict__ Mm, int n_poly) {
  using D = Dims<P>;
  using B = Build<P, ONE>;
  constexpr int NP = D::NP, N3 = D::N3, NQ3 = D::NQ3, NQ2 = D::NQ2, QC = B::QC, GP = B::GP, TG = B::TG,
                PAIRS = B::PAIRS;
  constexpr bool XCHG = REF && B::SPLIT == 1;  // the transposed pair's term is in this workgroup
  constexpr int VOLSZ = 4 * NP * QC, FACESZ = 8 * NP * NQ2, NB = B::NB;
  union Tabs {
    Tab1<P, QC> vol;
    Tab1<P, NQ2> face[2];
  };
  __shared__ double shT[GP][VOLSZ > FACESZ ? VOLSZ : FACESZ];
  __shared__ Tabs sh1[GP];
  __shared__ double shw[GP][QC > NQ2 ? QC : NQ2][2];
  __shared__ double shX[GP][XCHG ? 9 : 1][XCHG ? PAIRS : 1];
  __shared__ BuildTet shS[GP][NB];
  __shared__ double sq3[NQ3 * 4], sw3[NQ3], sq2[NQ2 * 4], sw2[NQ2], sbb[GP][6];
  __shared__ int sbl[NP * 3];
  const int tid = threadIdx.x, grp = GP == 1 ? 0 : tid / TG, lt = GP == 1 ? tid : tid % TG;
  const int Pr = (int)(blockIdx.x / B::SPLIT) * GP + grp, half = blockIdx.x % B::SPLIT;
  const bool poly = GP == 1 || Pr < n_poly;
  const int Pp = poly ? Pr : n_poly - 1;  // a group past the end computes along and stores nothing
  double* const T = shT[grp];
  Tabs& t1 = sh1[grp];
  double(*const sw)[2] = shw[grp];
  for (int i = tid; i < NP * 3; i += B::TPB) sbl[i] = m.blist[i];
  for (int i = tid; i < NQ3 * 4; i += B::TPB) sq3[i] = m.qtet[i];
  for (int i = tid; i < NQ2 * 4; i += B::TPB) sq2[i] = m.qtri[i];
  for (int i = tid; i < NQ3; i += B::TPB) sw3[i] = m.wtet[i];
  for (int i = tid; i < NQ2; i += B::TPB) sw2[i] = m.wtri[i];
  double* const bbP = sbb[grp];
  if (lt < 6) bbP[lt] = m.bbox[(size_t)Pp * 6 + lt];
  const double hkP = m.hk[Pp];
  const int r0 = m.row_ptr[Pp], r1 = m.row_ptr[Pp + 1];
  const int pr = half * B::SHARE + lt;
  const bool on = lt < B::SHARE && pr < PAIRS;
  // lanes along the rows: their stores cover whole lines of the column-pair layout
  const int mm = on ? pr % NP : 0, nn = on ? pr / NP : 0;
  double sK[9], sA[9], sM = 0.0, sMr = 0.0;
#pragma unroll
  for (int e = 0; e < 9; ++e) sK[e] = sA[e] = 0.0;
  // entry (i, j) of this thread's pair in a block
  auto at = [&](int i, int j) { return (uint32_t)kpos(N3, i * NP + mm, j * NP + nn); };
  // blocks of this row stored already (bit = block - r0; longer rows: cleared here)
  unsigned long long seen = 0ull;
  if (poly && on)
    for (int b = r0 + 64; b < r1; ++b)
      for (int e = 0; e < 9; ++e) {
        K[(size_t)b * D::BS + at(e / 3, e % 3)] = 0.0;
        if (ADG) A[(size_t)b * D::BS + at(e / 3, e % 3)] = 0.0;
      }
  const int a0 = m.ptet_ptr[Pp], cnt = m.ptet_ptr[Pp + 1] - a0;
  int steps = cnt;  // the workgroup's polyhedra walk their tets together
  if constexpr (GP > 1) {
#pragma unroll
    for (int o = TG; o < 64; o <<= 1) steps = max(steps, __shfl_xor(steps, o, 64));
  }
  for (int a = 0; a < steps; ++a) {
    if (a % NB == 0) {
      __syncthreads();
      for (int i = lt; i < 4 * NB; i += TG) {
        const int c = a + i / 4, f = i % 4;
        if (c >= cnt) continue;
        BuildTet& ts = shS[grp][i / 4];
        const int t = m.ptet[a0 + c], e2 = m.neigh[t * 4 + f];
        const double lam = m.lam[t], mu = m.mu[t];
        double v[12];
        for (int e = 0; e < 12; ++e) v[e] = m.tet_xyz[(size_t)t * 12 + e];
        const int Q = e2 >= 0 ? m.tet_poly[e2] : -1;
        BuildFace& fs = ts.f[f];
        // neither a face inside the polyhedron nor a Neumann face has a term
        fs.Q = (e2 >= 0 ? Q != Pp : e2 != -2) ? Q : -2;
        fs.blk = m.face_blk[t * 4 + f];
        for (int d = 0; d < 3; ++d) fs.n[d] = m.normal[(t * 4 + f) * 3 + d];
        fs.ar = m.area[t * 4 + f];
        const double hkQ = Q >= 0 ? m.hk[Q] : hkP;
        const double Dbar = lam + 2 * mu;
        const double hmin = hkP < hkQ ? hkP : hkQ;
        fs.sigma = alpha * (P * P) / hmin * Dbar;
        if (Q >= 0)
          for (int e = 0; e < 6; ++e) fs.bb[e] = m.bbox[(size_t)Q * 6 + e];
        if (f == 0) {
          double Fk[12], Jdet;
          affine_map(v, Fk, Jdet);
          for (int e = 0; e < 12; ++e) ts.v[e] = v[e];
          ts.aJ = fabs(Jdet);
          ts.rho = m.rho[t];
          ts.lam = lam;
          ts.mu = mu;
        }
      }
      __syncthreads();
    }
    const bool tet = a < cnt;
    const BuildTet& ts = shS[grp][tet ? a % NB : 0];
    const double lam = ts.lam, mu = ts.mu;
    const double l2m = lam + 2 * mu;
    // mass (MAKE_MATRICES_FREE :224-233 with MAKE_MASS_VOLUME) and volume
    // stiffness (MAKE_STIFFNESS_VOLUME, assemble_element :24-77)
    double s[9], ms = 0.0;
#pragma unroll
    for (int e = 0; e < 9; ++e) s[e] = 0.0;
#pragma unroll 1
    for (int q0 = 0; q0 < NQ3; q0 += QC) {
      for (int i = lt; i < 3 * QC; i += TG) {
        const int d = i / QC, q = i % QC;
        double r[4];
        affine_row(ts.v, d, r);
        tab1d<P, QC>(t1.vol, d, q, map_coord(r, &sq3[(q0 + q) * 4]), bbP[2 * d], bbP[2 * d + 1]);
        if (d == 0) sw[q][0] = sw3[q0 + q] * ts.aJ;
      }
      __syncthreads();
      double *phi = T, *dphi = T + NP * QC;  // [q][f], [d][q][f]
      for (int e = lt; e < NP * QC; e += TG) {
        const int q = e / NP, f = e % NP;
        basis_row<P, QC>(t1.vol, sbl[f * 3], sbl[f * 3 + 1], sbl[f * 3 + 2], q, phi[e], dphi[e],
                         dphi[NP * QC + e], dphi[2 * NP * QC + e]);
      }
      __syncthreads();
#pragma unroll 2
      for (int q = 0; q < QC; ++q) {
        const double wj = sw[q][0];
        ms = ms + wj * phi[q * NP + mm] * phi[q * NP + nn];
        const double x0 = dphi[q * NP + mm], x1 = dphi[(QC + q) * NP + mm], x2 = dphi[(2 * QC + q) * NP + mm];
        const double y0 = dphi[q * NP + nn], y1 = dphi[(QC + q) * NP + nn], y2 = dphi[(2 * QC + q) * NP + nn];
        if constexpr (REF) {
          const double u0 = mu * x0, u1 = mu * x1, u2 = mu * x2;
          const double b0 = u0 * y0, b1 = u1 * y1, b2 = u2 * y2;
          const double l0 = lam * x0, l1 = lam * x1, l2 = lam * x2;
          s[0] = s[0] + wj * (l2m * x0 * y0 + b1 + b2);
          s[4] = s[4] + wj * (l2m * x1 * y1 + b0 + b2);
          s[8] = s[8] + wj * (l2m * x2 * y2 + b0 + b1);
          s[1] = s[1] + wj * (l0 * y1 + u1 * y0);
          s[2] = s[2] + wj * (l0 * y2 + u2 * y0);
          s[3] = s[3] + wj * (l1 * y0 + u0 * y1);
          s[5] = s[5] + wj * (l1 * y2 + u2 * y1);
          s[6] = s[6] + wj * (l2 * y0 + u0 * y2);
          s[7] = s[7] + wj * (l2 * y1 + u1 * y2);
        } else {
          const double z0 = wj * y0, z1 = wj * y1, z2 = wj * y2;
          s[0] += x0 * z0; s[1] += x0 * z1; s[2] += x0 * z2;
          s[3] += x1 * z0; s[4] += x1 * z1; s[5] += x1 * z2;
          s[6] += x2 * z0; s[7] += x2 * z1; s[8] += x2 * z2;
        }
      }
      __syncthreads();  // the tables' reads are done before they are filled again
    }
    if (tet) {
      sM = sM + ms;
      sMr = sMr + ms * ts.rho;
#pragma unroll
      for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int j = 0; j < 3; ++j) {
          const int e = 3 * i + j;
          double val = s[e];
          if constexpr (!REF) {
            if (i == j)
              val = l2m * s[e] + mu * s[4 * ((i + 1) % 3)] + mu * s[4 * ((i + 2) % 3)];
            else
              val = lam * s[e] + mu * s[3 * j + i];
          }
          sK[e] = sK[e] + val;
          if (ADG) sA[e] = sA[e] + val;
        }
    }
    // faces (MAKE_STIFFNESS_FACE, assemble_element :404-661; insertion
    // src/matrix_free.f90:371-441)
#pragma unroll 1
    for (int f = 0; f < 4; ++f) {
      const BuildFace& fs = ts.f[f];
      const int Q = tet ? fs.Q : -2;
      const bool act = Q != -2, interior = Q >= 0;
      if (GP == 1 ? !act : !__any(act)) continue;
      const double n1 = fs.n[0], n2 = fs.n[1], n3 = fs.n[2];
      const double ar = fs.ar;
      const double d11 = fabs(n1) * fabs(n1) + 0.5 * (fabs(n2) * fabs(n2)) + 0.5 * (fabs(n3) * fabs(n3));
      const double d22 = fabs(n2) * fabs(n2) + 0.5 * (fabs(n1) * fabs(n1)) + 0.5 * (fabs(n3) * fabs(n3));
      const double d33 = fabs(n3) * fabs(n3) + 0.5 * (fabs(n1) * fabs(n1)) + 0.5 * (fabs(n2) * fabs(n2));
      for (int i = lt; i < 3 * NQ2 * (interior ? 2 : 1); i += TG) {
        const int side = i / (3 * NQ2), d = i / NQ2 % 3, q = i % NQ2;
        double r[4];
        affine_row(ts.v, d, r);
        const double x = face_coord(r, f, &sq2[q * 4]);
        const double* bb = side ? fs.bb : bbP;
        tab1d<P, NQ2>(t1.face[side], d, q, x, bb[2 * d], bb[2 * d + 1]);
        if (side == 0 && d == 0) {
          const double w = sw2[q];
          sw[q][0] = REF ? (interior ? 0.5 * w * ar : w * ar) : w;
          sw[q][1] = fs.sigma * w;
        }
      }
      __syncthreads();
      double *p1 = T, *p2 = T + NP * NQ2, *g1 = T + 2 * NP * NQ2, *g2 = T + 5 * NP * NQ2;  // [q][f], [d][q][f]
      constexpr int SG = NP * NQ2;
      for (int e = lt; e < SG * (interior ? 2 : 1); e += TG) {
        const int side = e / SG, o = e % SG, q = o / NP, fb = o % NP;
        double* g = side ? g2 : g1;
        basis_row<P, NQ2>(t1.face[side], sbl[fb * 3], sbl[fb * 3 + 1], sbl[fb * 3 + 2], q,
                          (side ? p2 : p1)[o], g[o], g[SG + o], g[2 * SG + o]);
      }
      __syncthreads();
      // the neighbour's block: first face to touch it stores, the others add
      const int blk = interior ? fs.blk : r0;
      const int bit = blk - r0;
      const bool fresh = bit < 64 && !(seen >> (bit & 63) & 1ull);
      if (interior && bit < 64) seen |= 1ull << bit;
      double* Kb = K + (size_t)blk * D::BS;
      double* Ab = ADG ? A + (size_t)blk * D::BS : nullptr;
      if constexpr (REF) {
        double i1[9], i1t[9];  // the term and its transpose: entry (j, i) of the pair (n, m)
        // S_E1 (:476-490): the same for (i, j) and (j, i); entries 00 11 22 01 02 12
        double s1[6] = {0, 0, 0, 0, 0, 0};
#pragma unroll
        for (int e = 0; e < 9; ++e) i1[e] = i1t[e] = 0.0;
#pragma unroll 1
        for (int q = 0; q < NQ2; ++q) {
          const double c = sw[q][0], swq = sw[q][1];
          const double am = p1[q * NP + mm], an = p1[q * NP + nn];
          const double pp = am * an, hp = 0.5 * am * an;
          s1[0] = s1[0] + swq * (pp * d11) * ar;
          s1[1] = s1[1] + swq * (pp * d22) * ar;
          s1[2] = s1[2] + swq * (pp * d33) * ar;
          s1[3] = s1[3] + swq * (hp * n1 * n2) * ar;
          s1[4] = s1[4] + swq * (hp * n1 * n3) * ar;
          s1[5] = s1[5] + swq * (hp * n2 * n3) * ar;
          face_terms(i1, c, g1[q * NP + mm], g1[SG + q * NP + mm], g1[2 * SG + q * NP + mm], an, lam, mu, l2m, n1,
                     n2, n3);
          if constexpr (!XCHG)
            face_terms(i1t, c, g1[q * NP + nn], g1[SG + q * NP + nn], g1[2 * SG + q * NP + nn], am, lam, mu, l2m, n1,
                       n2, n3);
        }
        if constexpr (XCHG) {
          if (on)
#pragma unroll
            for (int e = 0; e < 9; ++e) shX[grp][e][nn * NP + mm] = i1[e];
          __syncthreads();
#pragma unroll
          for (int e = 0; e < 9; ++e) i1t[e] = shX[grp][e][mm * NP + nn];
        }
        if (act) {
#pragma unroll
          for (int i = 0; i < 3; ++i)
#pragma unroll
            for (int j = 0; j < 3; ++j) {
              const int e = 3 * i + j;
              const double v1 = s1[i == j ? i : i + j + 2];
              sK[e] = sK[e] + v1;
              if (ADG) sA[e] = sA[e] + v1;
              sK[e] = sK[e] + theta * i1[e] - i1t[3 * j + i];
            }
        }
        if (interior && on) {
          double s2[6] = {0, 0, 0, 0, 0, 0}, i2[9], it2[9];
#pragma unroll
          for (int e = 0; e < 9; ++e) i2[e] = it2[e] = 0.0;
#pragma unroll 1
          for (int q = 0; q < NQ2; ++q) {
            const double c = sw[q][0], swq = sw[q][1];
            const double am = p1[q * NP + mm], an = p2[q * NP + nn];
            const double pp = am * an, hp = 0.5 * am * an;
            s2[0] = s2[0] - swq * (pp * d11) * ar;
            s2[1] = s2[1] - swq * (pp * d22) * ar;
            s2[2] = s2[2] - swq * (pp * d33) * ar;
            s2[3] = s2[3] - swq * (hp * n1 * n2) * ar;
            s2[4] = s2[4] - swq * (hp * n1 * n3) * ar;
            s2[5] = s2[5] - swq * (hp * n2 * n3) * ar;
            face_terms(i2, -c, g1[q * NP + mm], g1[SG + q * NP + mm], g1[2 * SG + q * NP + mm], an, lam, mu, l2m,
                       n1, n2, n3);
            face_terms(it2, c, g2[q * NP + nn], g2[SG + q * NP + nn], g2[2 * SG + q * NP + nn], am, lam, mu, l2m,
                       n1, n2, n3);
          }
          if (poly) {
#pragma unroll
            for (int i = 0; i < 3; ++i)
#pragma unroll
              for (int j = 0; j < 3; ++j) {
                const uint32_t o = at(i, j);
                const double v2 = s2[i == j ? i : i + j + 2];
                const double kb = fresh ? 0.0 : Kb[o];
                Kb[o] = kb + theta * i2[3 * i + j] + v2 - it2[3 * i + j];
                if (ADG) Ab[o] = (fresh ? 0.0 : Ab[o]) + v2;
              }
          }
        }
      } else {
        const double kk = interior ? 0.5 : 1.0, sigma = fs.sigma;
        const double nv[3] = {n1, n2, n3};
        const double dd[3] = {d11, d22, d33};
        // T(i,j;X): the traction pattern
        auto Tij = [&](int i, int j, const double* X) -> double {
          if (i == j) return l2m * nv[i] * X[i] + mu * nv[(i + 1) % 3] * X[(i + 1) % 3] +
                             mu * nv[(i + 2) % 3] * X[(i + 2) % 3];
          return lam * nv[j] * X[i] + mu * nv[i] * X[j];
        };
        if (act && on) {
          double PPs = 0.0, BP[3] = {0, 0, 0}, BPt[3] = {0, 0, 0};
#pragma unroll 2
          for (int q = 0; q < NQ2; ++q) {
            const double w = sw[q][0];
            const double am = p1[q * NP + mm], an = p1[q * NP + nn];
            const double wpm = w * am, wpn = w * an;
            PPs += wpm * an;
#pragma unroll
            for (int d = 0; d < 3; ++d) {
              BP[d] += g1[d * SG + q * NP + mm] * wpn;
              BPt[d] += g1[d * SG + q * NP + nn] * wpm;
            }
          }
#pragma unroll
          for (int i = 0; i < 3; ++i)
#pragma unroll
            for (int j = 0; j < 3; ++j) {
              const double cij = (i == j) ? dd[i] : 0.5 * nv[i] * nv[j];
              const double s1 = sigma * ar * PPs * cij;
              const double i1 = kk * ar * Tij(i, j, BP);
              const double i1t = kk * ar * Tij(j, i, BPt);
              sK[3 * i + j] = sK[3 * i + j] + s1;
              if (ADG) sA[3 * i + j] = sA[3 * i + j] + s1;
              sK[3 * i + j] = sK[3 * i + j] + theta * i1 - i1t;
            }
        }
        if (interior && on) {
          double PQs = 0.0, CP[3] = {0, 0, 0}, DQ[3] = {0, 0, 0};
#pragma unroll 2
          for (int q = 0; q < NQ2; ++q) {
            const double w = sw[q][0];
            const double wpm = w * p1[q * NP + mm], qn = p2[q * NP + nn];
            const double wqn = w * qn;
            PQs += wpm * qn;
#pragma unroll
            for (int d = 0; d < 3; ++d) {
              CP[d] += g1[d * SG + q * NP + mm] * wqn;
              DQ[d] += g2[d * SG + q * NP + nn] * wpm;
            }
          }
          if (poly)
#pragma unroll
            for (int i = 0; i < 3; ++i)
#pragma unroll
              for (int j = 0; j < 3; ++j) {
                const double cij = (i == j) ? dd[i] : 0.5 * nv[i] * nv[j];
                const double i2 = -0.5 * ar * Tij(i, j, CP);
                const double it2 = 0.5 * ar * Tij(i, j, DQ);
                const double s2 = -(sigma * ar * PQs * cij);
                const uint32_t o = at(i, j);
                const double kb = fresh ? 0.0 : Kb[o];
                Kb[o] = kb + theta * i2 + s2 - it2;
                if (ADG) Ab[o] = (fresh ? 0.0 : Ab[o]) + s2;
              }
        }
      }
      __syncthreads();  // as after a volume chunk
    }
  }
  if (!poly) return;
  double* Ks = K + (size_t)r0 * D::BS;
  double* As = ADG ? A + (size_t)r0 * D::BS : nullptr;
  if (on) {
    M[(size_t)Pp * NP * NP + mm * NP + nn] = sMr;
    Mm[(size_t)Pp * NP * NP + mm * NP + nn] = sM;
#pragma unroll
    for (int e = 0; e < 9; ++e) {
      Ks[at(e / 3, e % 3)] = sK[e];
      if (ADG) As[at(e / 3, e % 3)] = sA[e];
    }
  }
  if constexpr (N3 % 2 == 1) {  // the padding column
    for (int i = lt; i < (r1 - r0) * N3; i += TG) {
      const size_t o = (size_t)(r0 + i / N3) * D::BS + kpos(N3, i % N3, N3);
      K[o] = 0.0;
      if (ADG) A[o] = 0.0;
    }
  }
}

// Cholesky of both mass blocks of a polyhedron (cholesky,
// src/vet_mat_operations.f90:84-120), one wave per polyhedron: the block is
// staged in LDS by coalesced loads, each row j of the packed upper factor is
// computed across the wave (every lane forms the pivot, lane i > j the entry
// (j, i)) with each entry's sum over k in the serial order, and the factor
// leaves as one coalesced store.  status[0] set to 1 if a block is not SPD.
template <int P>
__global__ __launch_bounds__(64) void k_cholesky(const double* __restrict__ M,
                                                 const double* __restrict__ Mm,
                                                 double* __restrict__ RM, double* __restrict__ RMm,
                                                 int n_poly, int* __restrict__ status) {
  using D = Dims<P>;
  constexpr int NP = D::NP, NPK = D::NPK;
  static_assert(NP <= 64, "one lane per row of the factor");
  __shared__ double sA[NP * NP];
  __shared__ double sR[NPK];
  const int lane = threadIdx.x;
  const int Pp = blockIdx.x;
  if (Pp >= n_poly) return;
  for (int which = 0; which < 2; ++which) {
    const double* A = (which ? Mm : M) + (size_t)Pp * NP * NP;
    double* R = (which ? RMm : RM) + (size_t)Pp * NPK;
    __syncthreads();  // the previous block's LDS reads are done
    for (int e = lane; e < NP * NP; e += 64) sA[e] = A[e];
    __syncthreads();
    for (int j = 0; j < NP; ++j) {
      double s = sA[j * NP + j];
      for (int k = 0; k < j; ++k) {
        const double rkj = sR[pk_off(NP, k) + (j - k)];
        s = s - rkj * rkj;
      }
      if (!(s > 0.0)) {  // the same value on every lane: the wave leaves together
        if (lane == 0) atomicOr(status, 1);
        return;
      }
      const double rjj = sqrt(s);
      double rji = 0.0;
      if (lane > j && lane < NP) {
        double s2 = sA[j * NP + lane];
        for (int k = 0; k < j; ++k)
          s2 = s2 - sR[pk_off(NP, k) + (j - k)] * sR[pk_off(NP, k) + (lane - k)];
        rji = s2 / rjj;
      }
      // row j is read from the next step on (this step reads rows k < j only)
      if (lane == j) sR[pk_off(NP, j)] = rjj;
      if (lane > j && lane < NP) sR[pk_off(NP, j) + (lane - j)] = rji;
      __syncthreads();
    }
    for (int e = lane; e < NPK; e += 64) R[e] = sR[e];
  }
}

// ---------------------------------------------------------------------------
// RHS (MAKE_RHS_FREE, src/matrix_free.f90:467-843) and L2 projection
// (COMPUTE_MODAL_COEFFICIENTS_FREE, :847-997).  One workgroup per polyhedron,
// entry (i, m) owned by one thread; bound by the data's sines and the basis
// values, both formed once per point (tab1d): p = 3, 13,824 polyhedra, RHS 2.07
// -> 0.88 ms, projection 0.98 -> 0.56 ms.
// ---------------------------------------------------------------------------
template <int P>
constexpr int rhs_threads() { return P <= 2 ? 128 : 256; }
// p = 1: from so many polyhedra on the chip is full and one wave a polyhedron
// does; below, a second one shortens the walk over a polyhedron's tets.  us of a
// right-hand side with 64 / 128 threads: 22 polyhedra of 300 to 600 tets 3019 /
// 2641, 2,338 of 4 to 40 341 / 303, 1,728 of 6 80 / 77; 3,524 of 50 to 100 1015 /
// 1182, 4,096 of 6 128 / 149.
constexpr int kRhsWave = 2560;
// NQ points' data(q) and 3 NQ one-dimensional values tab(i) over a workgroup: the
// data on the first wave, the values on the others where there are (one wave
// would run the two one after the other) and the data fit one, or else all in a
// row
template <int NQ, int TPB, class Data, class Tab>
__device__ __forceinline__ void data_and_tabs(int tid, Data&& data, Tab&& tab) {
  if constexpr (NQ < 64 && TPB > 64) {
    if (tid < 64) {
      if (tid < NQ) data(tid);
    } else {
      for (int i = tid - 64; i < 3 * NQ; i += TPB - 64) tab(i);
    }
  } else {
    for (int i = tid; i < 4 * NQ; i += TPB) {
      if (i < NQ) data(i);
      else tab(i - NQ);
    }
  }
}

template <int P, int TPB = rhs_threads<P>()>
__global__ __launch_bounds__(TPB, 4) void k_rhs(MeshDev m, int prob, double alpha, double theta,
                                             double* __restrict__ rhs,
                                             const double* __restrict__ tabv = nullptr,
                                             const double* __restrict__ tabf = nullptr) {
  using D = Dims<P>;
  constexpr int NP = D::NP, N3 = D::N3, NQ3 = D::NQ3, NQ2 = D::NQ2;
  constexpr int VOLSZ = NP * NQ3, FACESZ = 4 * NP * NQ2;
  union Tabs {
    Tab1<P, NQ3> vol;
    Tab1<P, NQ2> face;
  };
  __shared__ double T[VOLSZ > FACESZ ? VOLSZ : FACESZ];
  __shared__ Tabs t1;
  __shared__ double sval[NQ3 * 3];
  __shared__ int sbl[NP * 3];
  const int tid = threadIdx.x;
  const int Pp = blockIdx.x;
  for (int i = tid; i < NP * 3; i += TPB) sbl[i] = m.blist[i];
  const double* bbP = m.bbox + (size_t)Pp * 6;
  double* r = rhs + (size_t)Pp * N3;
  const int ci = tid / NP, mm = tid % NP;  // this thread's entry
  double racc = 0.0;  // running rhs entry of this thread
  for (int a = m.ptet_ptr[Pp]; a < m.ptet_ptr[Pp + 1]; ++a) {
    const int t = m.ptet[a];
    const double* vt = m.tet_xyz + (size_t)t * 12;
    double v[12], Fk[12], Jdet;
    for (int i = 0; i < 12; ++i) v[i] = vt[i];
    affine_map(v, Fk, Jdet);
    const double aJ = fabs(Jdet);
    const double rho = m.rho[t], lam = m.lam[t], mu = m.mu[t];
    __syncthreads();
    data_and_tabs<NQ3, TPB>(
        tid,
        [&](int i) {  // the data, times the weight
          double val[3];
          if (tabv) {  // values of the caller's forcing at k_rhs_points' volume points
            for (int c = 0; c < 3; ++c) val[c] = tabv[((size_t)t * NQ3 + i) * 3 + c];
          } else {
            double x[3];
            map_point(Fk, &m.qtet[i * 4], x);
            forcing(prob, lam, mu, x, rho, val);
          }
          const double aw = aJ * m.wtet[i];
          for (int c = 0; c < 3; ++c) sval[i * 3 + c] = aw * val[c];
        },
        [&](int i) {
          const int d = i / NQ3, q = i % NQ3;
          double rw[4];
          affine_row(vt, d, rw);
          tab1d<P, NQ3>(t1.vol, d, q, map_coord(rw, &m.qtet[q * 4]), bbP[2 * d], bbP[2 * d + 1]);
        });
    __syncthreads();
    for (int e = tid; e < NP * NQ3; e += TPB) {
      const int q = e / NP, f = e % NP;
      T[e] = t1.vol.v[0][sbl[f * 3]][q] * t1.vol.v[1][sbl[f * 3 + 1]][q] * t1.vol.v[2][sbl[f * 3 + 2]][q];
    }
    __syncthreads();
    if (tid < N3) {
      double s = 0.0;
#pragma unroll 4
      for (int q = 0; q < NQ3; ++q) s = s + sval[q * 3 + ci] * T[q * NP + mm];
      racc = racc + s;
    }
    for (int f = 0; f < 4; ++f) {
      const int e2 = m.neigh[t * 4 + f];
      if (e2 >= 0) continue;  // only boundary faces carry data
      __syncthreads();
      const double* nrm = &m.normal[(t * 4 + f) * 3];
      const int tag = m.bc_space[t * 4 + f];
      data_and_tabs<NQ2, TPB>(
          tid,
          [&](int i) {
            if (tabf) {  // the caller's Dirichlet / Neumann data at k_rhs_points' face points
              for (int c = 0; c < 3; ++c) sval[i * 3 + c] = tabf[(((size_t)t * 4 + f) * NQ2 + i) * 3 + c];
            } else {
              double xr[3];
              face_point_rhs(Fk, f, &m.qtri[i * 4], xr);
              if (e2 == -1) dirichlet(prob, xr, tag, &sval[i * 3]);
              else neumann(prob, lam, mu, nrm, xr, tag, &sval[i * 3]);
            }
          },
          [&](int i) {
            const int d = i / NQ2, q = i % NQ2;
            double rw[4];
            affine_row(vt, d, rw);
            tab1d<P, NQ2>(t1.face, d, q, face_coord(rw, f, &m.qtri[q * 4]), bbP[2 * d], bbP[2 * d + 1]);
          });
      __syncthreads();
      constexpr int SG = NP * NQ2;
      for (int e = tid; e < SG; e += TPB) {
        const int q = e / NP, fb = e % NP;
        basis_row<P, NQ2>(t1.face, sbl[fb * 3], sbl[fb * 3 + 1], sbl[fb * 3 + 2], q, T[e], T[SG + e], T[2 * SG + e],
                          T[3 * SG + e]);
      }
      __syncthreads();
      if (tid < N3) {
        const int i = ci;
        const double n1 = nrm[0], n2 = nrm[1], n3 = nrm[2];
        const double ar = m.area[t * 4 + f];
        const double l2m = lam + 2 * mu;
        const double sigma = alpha * (P * P) / m.hk[Pp] * (lam + 2 * mu);
        double s = 0.0;
        for (int q = 0; q < NQ2; ++q) {
          const double w = m.wtri[q];
          const double* dd = &sval[q * 3];
          const double ph = T[q * NP + mm];
          if (e2 == -1) {
            const double gg1 = T[SG + q * NP + mm], gg2 = T[2 * SG + q * NP + mm], gg3 = T[3 * SG + q * NP + mm];
            double tm, t2;
            if (i == 0) {
              tm = l2m * gg1 * dd[0] * n1 + mu * gg2 * dd[0] * n2 + mu * gg3 * dd[0] * n3 +
                   lam * gg1 * dd[1] * n2 + mu * gg2 * dd[1] * n1 + lam * gg1 * dd[2] * n3 +
                   mu * gg3 * dd[2] * n1;
              t2 = ph * dd[0] * (fabs(n1) * fabs(n1) + 0.5 * (fabs(n2) * fabs(n2)) + 0.5 * (fabs(n3) * fabs(n3))) +
                   0.5 * ph * dd[1] * n1 * n2 + 0.5 * ph * dd[2] * n1 * n3;
            } else if (i == 1) {
              tm = l2m * gg2 * dd[1] * n2 + mu * gg1 * dd[1] * n1 + mu * gg3 * dd[1] * n3 +
                   lam * gg2 * dd[0] * n1 + mu * gg1 * dd[0] * n2 + lam * gg2 * dd[2] * n3 +
                   mu * gg3 * dd[2] * n2;
              t2 = ph * dd[1] * (fabs(n2) * fabs(n2) + 0.5 * (fabs(n1) * fabs(n1)) + 0.5 * (fabs(n3) * fabs(n3))) +
                   0.5 * ph * dd[0] * n1 * n2 + 0.5 * ph * dd[2] * n2 * n3;
            } else {
              tm = l2m * gg3 * dd[2] * n3 + mu * gg1 * dd[2] * n1 + mu * gg2 * dd[2] * n2 +
                   lam * gg3 * dd[0] * n1 + mu * gg1 * dd[0] * n3 + lam * gg3 * dd[1] * n2 +
                   mu * gg2 * dd[1] * n3;
              t2 = ph * dd[2] * (fabs(n3) * fabs(n3) + 0.5 * (fabs(n1) * fabs(n1)) + 0.5 * (fabs(n2) * fabs(n2))) +
                   0.5 * ph * dd[0] * n1 * n3 + 0.5 * ph * dd[1] * n2 * n3;
            }
            s = s + theta * w * tm * ar + sigma * w * t2 * ar;
          } else {
            s = s + w * ph * dd[i] * ar;
          }
        }
        if (s != 0.0) racc = racc + s;
      }
    }
  }
  if (tid < N3) r[tid] = racc;
}

// Physical points where MAKE_RHS_FREE evaluates its data (as k_rhs computes
// them): volume quadrature points vpts[(t*NQ3 + q)*3 + d] (forcing) and the
// data points of every tet face fpts[((t*4 + f)*NQ2 + q)*3 + d] (Dirichlet /
// Neumann data; src/matrix_free.f90:711, :781-801).  One thread per point.
template <int P>
__global__ void k_rhs_points(MeshDev m, int n_tet, double* __restrict__ vpts,
                             double* __restrict__ fpts) {
  using D = Dims<P>;
  constexpr int NQ3 = D::NQ3, NQ2 = D::NQ2, PER = NQ3 + 4 * NQ2;
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= (size_t)n_tet * PER) return;
  const int t = (int)(i / PER), k = (int)(i % PER);
  double v[12], Fk[12], Jdet;
  for (int j = 0; j < 12; ++j) v[j] = m.tet_xyz[(size_t)t * 12 + j];
  affine_map(v, Fk, Jdet);
  if (k < NQ3) {
    map_point(Fk, &m.qtet[k * 4], vpts + ((size_t)t * NQ3 + k) * 3);
  } else {
    const int f = (k - NQ3) / NQ2, q = (k - NQ3) % NQ2;
    face_point_rhs(Fk, f, &m.qtri[q * 4], fpts + (((size_t)t * 4 + f) * NQ2 + q) * 3);
  }
}

// LDS ordering within one wave (the rocPRIM wave barrier: fences at
// wavefront scope around a code-motion barrier); enough for a workgroup of
// one wave, and it does not wait on the wave's global loads and stores.
__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Broadcast lane `l`'s double to the whole wave (v_readlane on both halves).
__device__ __forceinline__ double lane_bcast(double v, int l) {
  const int lo = __builtin_amdgcn_readlane(__double2loint(v), l);
  const int hi = __builtin_amdgcn_readlane(__double2hiint(v), l);
  return __hiloint2double(hi, lo);
}

// A divisor b of many quotients: y = 1 / b rounded, then quot() gives a / b to
// the bits of the division in five dependent operations instead of a dozen
// (Markstein, IBM J. Res. Dev. 34, 1990: the remainder a - b q is exact in one
// fused multiply-add, the first correction makes q faithful, the second rounds
// it correctly), for divisors that are plain() and numerators that are
// quotable().  Quotients that are zero, infinite or NaN are q = a y, which has
// the division's sign.
struct Divisor {
  double b, y;
  __device__ __forceinline__ explicit Divisor(double v) : b(v), y(1.0 / v) {}
  __device__ __forceinline__ bool plain() const { return fabs(b) > 0x1p-100 && fabs(b) < 0x1p100; }
};
__device__ __forceinline__ double quot(double a, const Divisor& d) {
  const double q0 = a * d.y;
  const double q1 = fma(fma(-d.b, q0, a), d.y, q0);
  const double q2 = fma(fma(-d.b, q1, a), d.y, q1);
  constexpr int kNonzeroFinite = 0x008 | 0x010 | 0x080 | 0x100;  // -normal, -subnormal, +subnormal, +normal
  return __builtin_amdgcn_class(q0, kNonzeroFinite) ? q2 : q0;
}
// Numerators whose quotients by a plain divisor are exact above: the quotient
// stays within 2^-960 and 2^1000, the last bit of the remainder (2^-106 of the
// numerator) above the smallest subnormal.  The solves test the numerators that
// they used once at their end and divide if one fails: in a wave front's first
// trace, next to overflow, or with infinities and NaN.
__device__ __forceinline__ bool quotable(double a) {
  const double m = fabs(a);
  return (m >= 0x1p-860 && m <= 0x1p900) || m == 0.0;
}

// M^-1 w = R^-1 R^-T w (solve_LU with L = R^T, src/vet_mat_operations.f90:
// 123-153) across a group of 3Np lanes from lane `base`, one entry of the
// vector per lane: r = component x Np + row (other lanes' results are not
// used).  The forward sweep broadcasts y_j = s_j / R_jj and the rows below
// subtract R_ji y_j, in ascending j as the reference does; the backward sweep
// runs the columns from the last, the rows above subtracting R_ij x_j.  NP
// dependent steps per sweep instead of Np(Np+1)/2 on one lane.  A lane past its
// own step goes on, subtracting zeros (R[NPK] is one), so that it keeps its
// numerator and the selects stay off the chain.  The solves are the tail of a step on few polyhedra: with divisions
// and selects on the chain 162 single-tet polyhedra took 6.2, 10.4 and 30.9 us
// a step at p = 2, 3, 4, now 5.2, 7.3 and 23.5.
template <int NP, bool PLAIN>
__device__ __forceinline__ double solve_group_as(const double* __restrict__ R, const Divisor& d, double w, int ii,
                                                 int from, bool& ok) {
  constexpr int ZERO = NP * (NP + 1) / 2;
  double y = 0.0;
#pragma unroll
  for (int j = 0; j < NP; ++j) {
    const double t = PLAIN ? quot(w, d) : w / d.b;
    if (ii == j) y = t;
    w = w - R[ii > j ? pk_off(NP, j) + ii - j : ZERO] * __shfl(t, from + j, 64);
  }
  ok = !PLAIN || quotable(w);
  const int ri = pk_off(NP, ii);
  w = y;
#pragma unroll
  for (int j = NP - 1; j >= 0; --j) {
    const double t = PLAIN ? quot(w, d) : w / d.b;
    if (ii == j) y = t;
    w = w - R[ii < j ? ri + j - ii : ZERO] * __shfl(t, from + j, 64);
  }
  ok = ok && (!PLAIN || quotable(w));
  return y;
}
template <int NP>
__device__ __forceinline__ double solve_group(const double* __restrict__ R, const Divisor& d, double w, int base,
                                              int r, bool on) {
  const int cc = on ? r / NP : 0, ii = on ? r % NP : 0, from = on ? base + cc * NP : 0;
  bool ok;
  if (__all(!on || d.plain())) {
    const double y = solve_group_as<NP, true>(R, d, w, ii, from, ok);
    if (__all(!on || ok)) return y;
  }
  return solve_group_as<NP, false>(R, d, w, ii, from, ok);
}

// R^-T of three right-hand sides across one wave, lane i on row i of all three
// (NP <= 64): broadcasts y_j = s_j / R_jj from lane j, the rows below subtract
// R_ji y_j (ascending j, as the reference).
template <int NP>
__device__ __forceinline__ void forward_rows(const double* __restrict__ R, double& x0, double& x1, double& x2, int i) {
  static_assert(NP <= 64, "one lane per row");
#pragma unroll 5
  for (int j = 0; j < NP; ++j) {
    const int rj = pk_off(NP, j);
    const double rjj = R[rj];
    const double y0 = __shfl(x0, j, 64) / rjj, y1 = __shfl(x1, j, 64) / rjj, y2 = __shfl(x2, j, 64) / rjj;
    if (i == j) {
      x0 = y0;
      x1 = y1;
      x2 = y2;
    } else if (i > j && i < NP) {
      const double r = R[rj + (i - j)];
      x0 = x0 - r * y0;
      x1 = x1 - r * y1;
      x2 = x2 - r * y2;
    }
  }
}

// R^-1 of three right-hand sides across one wave, lane i on row i of all three
// (NP <= 64), the columns from the last; d: the divisor R_ii of lane i.
// Broadcasts by v_readlane (24.2 us above with __shfl).
template <int NP, bool PLAIN>
__device__ __forceinline__ bool back_rows_as(const double* __restrict__ R, const Divisor& d, double (&x)[3], int i) {
  constexpr int ZERO = NP * (NP + 1) / 2;
  double y[3] = {0.0, 0.0, 0.0};
  const int ri = pk_off(NP, i < NP ? i : 0);
#pragma unroll 5
  for (int j = NP - 1; j >= 0; --j) {
    const double r = R[i < j ? ri + j - i : ZERO];
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      const double t = PLAIN ? quot(x[c], d) : x[c] / d.b;
      if (i == j) y[c] = t;
      x[c] = x[c] - r * lane_bcast(t, j);
    }
  }
  const bool ok = !PLAIN || i >= NP || (quotable(x[0]) && quotable(x[1]) && quotable(x[2]));
#pragma unroll
  for (int c = 0; c < 3; ++c) x[c] = y[c];
  return ok;
}
template <int NP>
__device__ __forceinline__ void back_rows(const double* __restrict__ R, const Divisor& d, double (&x)[3], int i) {
  if (__all(i >= NP || d.plain())) {
    double y[3] = {x[0], x[1], x[2]};
    const bool ok = back_rows_as<NP, true>(R, d, y, i);
    if (__all(ok)) {
#pragma unroll
      for (int c = 0; c < 3; ++c) x[c] = y[c];
      return;
    }
  }
  back_rows_as<NP, false>(R, d, x, i);
}

// M^-1: both sweeps
template <int NP, bool PLAIN>
__device__ __forceinline__ bool solve_rows_as(const double* __restrict__ R, const Divisor& d, double (&x)[3], int i) {
  constexpr int ZERO = NP * (NP + 1) / 2;
  double y[3] = {0.0, 0.0, 0.0};
#pragma unroll 5
  for (int j = 0; j < NP; ++j) {
    const double r = R[i < NP && i > j ? pk_off(NP, j) + i - j : ZERO];
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      const double t = PLAIN ? quot(x[c], d) : x[c] / d.b;
      if (i == j) y[c] = t;
      x[c] = x[c] - r * lane_bcast(t, j);
    }
  }
  const bool ok = !PLAIN || i >= NP || (quotable(x[0]) && quotable(x[1]) && quotable(x[2]));
#pragma unroll
  for (int c = 0; c < 3; ++c) x[c] = y[c];
  return back_rows_as<NP, PLAIN>(R, d, x, i) && ok;
}
template <int NP>
__device__ __forceinline__ void solve_rows(const double* __restrict__ R, const Divisor& d, double (&x)[3], int i) {
  if (__all(i >= NP || d.plain())) {
    double y[3] = {x[0], x[1], x[2]};
    const bool ok = solve_rows_as<NP, true>(R, d, y, i);
    if (__all(ok)) {
#pragma unroll
      for (int c = 0; c < 3; ++c) x[c] = y[c];
      return;
    }
  }
  solve_rows_as<NP, false>(R, d, x, i);
}

// R^-1 y in place on one lane, every row's terms in ascending columns as the
// reference adds them.  The projections keep this order: the 32-bit apply
// turns a last-bit change of the initial data into 1e-6 of the state within
// 100 steps.  The products of four columns are formed ahead of the chain.
template <int NP>
__device__ __forceinline__ void back_ascending(const double* __restrict__ R, double* __restrict__ x) {
#pragma unroll 1
  for (int i = NP - 1; i >= 0; --i) {
    const double* __restrict__ Ri = R + pk_off(NP, i) - i;
    double s = x[i];
#pragma unroll 4
    for (int j = i + 1; j < NP; ++j) s = s - Ri[j] * x[j];
    x[i] = s / Ri[i];
  }
}

template <int P, int TPB = rhs_threads<P>()>
__global__ __launch_bounds__(TPB, 4) void k_project(MeshDev m, int fn, const double* __restrict__ RMm,
                                                 double* __restrict__ out,
                                                 const double* __restrict__ tabv) {
  using D = Dims<P>;
  constexpr int NP = D::NP, N3 = D::N3, NQ3 = D::NQ3;
  __shared__ double phi[NP * NQ3];
  __shared__ Tab1<P, NQ3> t1;
  __shared__ double sval[NQ3 * 3];
  __shared__ double sb[N3];
  __shared__ double sR[D::NPK];
  __shared__ int sbl[NP * 3];
  const int tid = threadIdx.x;
  const int Pp = blockIdx.x;
  for (int i = tid; i < NP * 3; i += TPB) sbl[i] = m.blist[i];
  for (int i = tid; i < D::NPK; i += TPB) sR[i] = RMm[(size_t)Pp * D::NPK + i];
  const double* bbP = m.bbox + (size_t)Pp * 6;
  const int ci = tid / NP, mm = tid % NP;
  double acc = 0.0;
  for (int a = m.ptet_ptr[Pp]; a < m.ptet_ptr[Pp + 1]; ++a) {
    const int t = m.ptet[a];
    const double* vt = m.tet_xyz + (size_t)t * 12;
    double v[12], Fk[12], Jdet;
    for (int i = 0; i < 12; ++i) v[i] = vt[i];
    affine_map(v, Fk, Jdet);
    const double aJ = fabs(Jdet);
    __syncthreads();
    data_and_tabs<NQ3, TPB>(
        tid,
        [&](int i) {  // the field, times the weight
          double val[3];
          if (tabv) {  // the caller's field at k_rhs_points' volume points
            for (int c = 0; c < 3; ++c) val[c] = tabv[((size_t)t * NQ3 + i) * 3 + c];
          } else {
            double x[3];
            map_point(Fk, &m.qtet[i * 4], x);
            field(fn, x, val);
          }
          const double aw = aJ * m.wtet[i];
          for (int c = 0; c < 3; ++c) sval[i * 3 + c] = aw * val[c];
        },
        [&](int i) {
          const int d = i / NQ3, q = i % NQ3;
          double rw[4];
          affine_row(vt, d, rw);
          tab1d<P, NQ3>(t1, d, q, map_coord(rw, &m.qtet[q * 4]), bbP[2 * d], bbP[2 * d + 1]);
        });
    __syncthreads();
    for (int e = tid; e < NP * NQ3; e += TPB) {
      const int q = e / NP, f = e % NP;
      phi[e] = t1.v[0][sbl[f * 3]][q] * t1.v[1][sbl[f * 3 + 1]][q] * t1.v[2][sbl[f * 3 + 2]][q];
    }
    __syncthreads();
    if (tid < N3)
#pragma unroll 4
      for (int q = 0; q < NQ3; ++q) acc = acc + sval[q * 3 + ci] * phi[q * NP + mm];
  }
  if (tid < N3) sb[tid] = acc;
  __syncthreads();
  if (tid < 64) {  // one wave sweeps forward, a lane per component back
    const bool row = tid < NP;
    double x0 = row ? sb[tid] : 0.0, x1 = row ? sb[NP + tid] : 0.0, x2 = row ? sb[2 * NP + tid] : 0.0;
    forward_rows<NP>(sR, x0, x1, x2, tid);
    if (row) {
      sb[tid] = x0;
      sb[NP + tid] = x1;
      sb[2 * NP + tid] = x2;
    }
    wave_lds_sync();
    if (tid < 3) back_ascending<NP>(sR, sb + tid * NP);
  }
  __syncthreads();
  if (tid < N3) out[(size_t)Pp * N3 + tid] = sb[tid];
}

__global__ void k_fill(double* __restrict__ a, double v, size_t n) {
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) a[i] = v;
}

// ---------------------------------------------------------------------------
// The leapfrog step (TIME_STEP_MATRIX_FREE, src/matrix_free.f90:1230-1385;
// FIRST_TIME_STEP_MATRIX_FREE :1100-1227) fused in one kernel: one wave per
// polyhedron, lane r = row r of the block row.  Per block the wave streams
// the block's column pairs (16 B per lane per load), with the neighbour's
// coefficients as wave-uniform (scalar) loads: the halo exchange of
// src/exchange_data.f90 becomes the on-device gather col[b].  Then
// w = -Ku + F_s + F_d g, three triangular-solve pairs with the packed mass
// factor, and the update.
//   MODE 0: out = (c1*x + 2*u) - wa            (c1 = dt^2, u = x_apply, wa = u^{n-1})
//   MODE 1: out = (c1*x + u) + c2*wa           (c1 = dt^2/2, u = u^0, wa = v^0, c2 = dt)
//   MODE 2: part[P] = sum_r u_r (K u)_r        (DG error: K = A_dg, u = uh - uex)
// ---------------------------------------------------------------------------
// Polyhedron of this workgroup.  Workgroups are dealt to the 8 XCDs round
// robin (workgroup b runs on XCD b % 8), each XCD with its own L2; the grid is
// padded to a multiple of 8 and XCD x is given the x-th eighth of the
// polyhedra, so neighbours -- whose coefficient blocks a row re-reads -- mostly
// share an L2.  A bijection of [0, grid); ids >= n_poly are padding.
__device__ inline int step_poly() {
  const int per = (int)(gridDim.x >> 3);
  return (int)(blockIdx.x & 7) * per + (int)(blockIdx.x >> 3);
}
inline unsigned step_grid(int n_poly) { return 8u * (unsigned)((n_poly + 7) / 8); }

// With a dispatch order (order[i] = polyhedron of slot i, step_grid entries,
// padding slots holding n_poly): each XCD's share of the polyhedra is walked
// longest block row first, so on meshes of uneven polyhedra the long rows
// start early instead of forming the tail of the launch.  Every polyhedron is
// still computed by one workgroup exactly as without it.
__device__ inline int step_poly(const int* __restrict__ order) {
  const int i = step_poly();
  return order ? order[i] : i;
}

// The vectors a row's update reads besides the block products.  With several
// waves per polyhedron (few polyhedra: latency counts) they are fetched before
// the blocks, otherwise after them, where other waves cover the wait and the
// registers are free.
template <int N3, int RPL>
struct StepEnds {
  double s[RPL], d[RPL], u[RPL], a[RPL];
  __device__ __forceinline__ void load(const double* __restrict__ rs, const double* __restrict__ rd,
                                       const double* __restrict__ uu, const double* __restrict__ wa, size_t o,
                                       int lane) {
#pragma unroll
    for (int k = 0; k < RPL; ++k) {
      const int r = lane + 64 * k;
      const bool row = r < N3;
      s[k] = row ? rs[o + r] : 0.0;
      d[k] = row ? rd[o + r] : 0.0;
      u[k] = row ? uu[o + r] : 0.0;
      a[k] = row ? wa[o + r] : 0.0;
    }
  }
};

// UNR = column pairs whose loads are issued together (register footprint vs
// loads in flight).  XS = how the neighbour's coefficients reach the lanes:
// 0 = wave-uniform scalar loads per pair, 1 = one coalesced vector load per
// block (lane c holds x[c]) broadcast with v_readlane, so the inner loop waits
// only on the block's own HBM loads.  Chosen per degree by lymph_autotune.
template <int P, int MODE, int UNR, int XS, int WPP, bool NT>
__global__ __launch_bounds__(64 * WPP) void k_leapfrog(const double* __restrict__ K,
                                                 const int* __restrict__ row_ptr,
                                                 const int* __restrict__ col,
                                                 const double* __restrict__ Rp,
                                                 const double* __restrict__ rs,
                                                 const double* __restrict__ rd,
                                                 const double* __restrict__ u,
                                                 const double* __restrict__ wa,
                                                 double* __restrict__ out, double g, double c1,
                                                 double c2, const int* __restrict__ gsel,
                                                 const double* __restrict__ gtab, int n_poly,
                                                 const int* __restrict__ order) {
  using D = Dims<P>;
  constexpr int NP = D::NP, N3 = D::N3, NPAIR = D::NPAIR;
  constexpr int RPL = (N3 + 63) / 64;
  __shared__ double sw[N3];
  __shared__ double sR[D::NPK + 1];  // the factor and a zero
  extern __shared__ double sblk[];  // WPP > 1: per-block products [block][row]
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int Pp = step_poly(order);
  if (Pp >= n_poly) return;  // padding workgroups of the last XCD share
  if (MODE != 2)
    for (int k = threadIdx.x; k <= D::NPK; k += 64 * WPP) sR[k] = k < D::NPK ? Rp[(size_t)Pp * D::NPK + k] : 0.0;
  StepEnds<N3, RPL> ends;
  const int drow = RPL == 1 ? (lane < N3 ? lane % NP : 0) : (lane < NP ? lane : 0);  // the lane's row in the solve
  Divisor diag(1.0);
  if constexpr (WPP > 1 && MODE != 2)
    if (wv == 0) {
      ends.load(rs, rd, u, wa, (size_t)Pp * N3, lane);
      diag = Divisor(Rp[(size_t)Pp * D::NPK + pk_off(NP, drow)]);
    }
  double acc[RPL];
#pragma unroll
  for (int k = 0; k < RPL; ++k) acc[k] = 0.0;
  const int b0 = row_ptr[Pp], b1 = row_ptr[Pp + 1];
  // WPP waves share a polyhedron's blocks round robin; each block's product
  // goes to LDS and wave 0 adds them in block order, the reference's order
  for (int b = b0 + wv; b < b1; b += WPP) {
    const int cb = __builtin_amdgcn_readfirstlane(col[b]);
    const double* __restrict__ xv = u + (size_t)cb * N3;
    const double* __restrict__ Kb = K + (size_t)b * D::BS;
    double xl[RPL];
    if (XS == 1) {
#pragma unroll
      for (int k = 0; k < RPL; ++k) {
        const int r = lane + 64 * k;
        xl[k] = r < N3 ? xv[r] : 0.0;
      }
    }
    double s[RPL];
#pragma unroll
    for (int k = 0; k < RPL; ++k) s[k] = 0.0;
#pragma unroll 1
    for (int c0 = 0; c0 < NPAIR; c0 += UNR) {
      double2 kv[UNR][RPL];
#pragma unroll
      for (int uu = 0; uu < UNR; ++uu) {
        const int c2i = c0 + uu;
#pragma unroll
        for (int k = 0; k < RPL; ++k) {
          const int r = lane + 64 * k;
          if ((NPAIR % UNR == 0 || c2i < NPAIR) && r < N3)
            kv[uu][k] = load_stream<NT>(Kb + ((size_t)c2i * N3 + r) * 2);
        }
      }
#pragma unroll
      for (int uu = 0; uu < UNR; ++uu) {
        const int c2i = c0 + uu;
        if (NPAIR % UNR == 0 || c2i < NPAIR) {
          const bool odd_tail = (N3 % 2 == 1) && (c2i == NPAIR - 1);
          double x0, x1;
          if (XS == 1) {
            const int ca = 2 * c2i, cbb = 2 * c2i + 1;
            const double xa = (RPL > 1 && (ca >> 6)) ? xl[RPL - 1] : xl[0];
            const double xb = (RPL > 1 && (cbb >> 6)) ? xl[RPL - 1] : xl[0];
            x0 = lane_bcast(xa, ca & 63);
            x1 = odd_tail ? 0.0 : lane_bcast(xb, cbb & 63);
          } else {
            x0 = xv[2 * c2i];
            x1 = odd_tail ? 0.0 : xv[2 * c2i + 1];
          }
#pragma unroll
          for (int k = 0; k < RPL; ++k) {
            const int r = lane + 64 * k;
            if (r < N3) {
              s[k] = s[k] + kv[uu][k].x * x0;
              if (!odd_tail) s[k] = s[k] + kv[uu][k].y * x1;
            }
          }
        }
      }
    }
    if constexpr (WPP == 1) {
#pragma unroll
      for (int k = 0; k < RPL; ++k) acc[k] = (b == b0) ? s[k] : acc[k] + s[k];
    } else {
#pragma unroll
      for (int k = 0; k < RPL; ++k) {
        const int r = lane + 64 * k;
        if (r < N3) sblk[(size_t)(b - b0) * N3 + r] = s[k];
      }
    }
  }
  if constexpr (WPP > 1) {
    __syncthreads();
#pragma unroll
    for (int k = 0; k < RPL; ++k) {
      const int r = lane + 64 * k;
      if (r < N3 && wv == 0) {
        double a = sblk[r];
#pragma unroll 4
        for (int j = 1; j < b1 - b0; ++j) a = a + sblk[(size_t)j * N3 + r];
        acc[k] = a;
      }
    }
  }
  const size_t o = (size_t)Pp * N3;
  if (MODE == 2) {
#pragma unroll
    for (int k = 0; k < RPL; ++k) {
      const int r = lane + 64 * k;
      if (r < N3 && wv == 0) sw[r] = acc[k];
    }
    __syncthreads();
    if (threadIdx.x == 0) {
      double el = 0.0;
      for (int r = 0; r < N3; ++r) el = el + u[o + r] * sw[r];
      out[Pp] = el;
    }
    return;
  }
  if constexpr (WPP == 1) __syncthreads();  // sR
  if (wv != 0) return;  // no barrier of the workgroup follows
  if constexpr (WPP == 1) ends.load(rs, rd, u, wa, o, lane);
  // time factor: one scalar, or per source group (ensembles whose instances
  // carry their own wavelet; the table is filled for this step)
  const double gp = gsel ? gtab[gsel[Pp]] : g;
  double w[RPL];
#pragma unroll
  for (int k = 0; k < RPL; ++k) w[k] = -acc[k] + ends.s[k] + ends.d[k] * gp;
  if constexpr (WPP == 1) diag = Divisor(sR[pk_off(NP, drow)]);
  if constexpr (RPL == 1) {  // one row per lane: the wave solves across its lanes
    w[0] = solve_group<NP>(sR, diag, w[0], 0, lane, lane < N3);
  } else {  // lane i takes row i of the three components
#pragma unroll
    for (int k = 0; k < RPL; ++k)
      if (lane + 64 * k < N3) sw[lane + 64 * k] = w[k];
    wave_lds_sync();
    const bool row = lane < NP;
    double x[3];
#pragma unroll
    for (int c = 0; c < 3; ++c) x[c] = row ? sw[c * NP + lane] : 0.0;
    solve_rows<NP>(sR, diag, x, lane);
    if (row)
#pragma unroll
      for (int c = 0; c < 3; ++c) sw[c * NP + lane] = x[c];
    wave_lds_sync();
#pragma unroll
    for (int k = 0; k < RPL; ++k) w[k] = lane + 64 * k < N3 ? sw[lane + 64 * k] : 0.0;
  }
#pragma unroll
  for (int k = 0; k < RPL; ++k) {
    const int r = lane + 64 * k;
    if (r < N3) {
      if (MODE == 0)
        out[o + r] = c1 * w[k] + 2.0 * ends.u[k] - ends.a[k];
      else
        out[o + r] = c1 * w[k] + ends.u[k] + c2 * ends.a[k];
    }
  }
}

// Step with every face pair's block stored once, in two launches.  With SIPG
// and one material on both traces of each face, K_QP = K_PQ^T to rounding, so
// only the self blocks and K_PQ for Q > P are kept (Ks; sidx[b] >= 0 the
// stored block of full-row block b, < 0 a block of the neighbour's row), and
// of each self block (K_PP = K_PP^T to rounding) only its upper triangle:
// column pair c2i's rows 0..2c2i+1 packed from entry 2 c2i (c2i + 1)
// (self_upper_off), half the bytes of the full block.
// k_sym_products: one wave per stored block K_PQ, the self blocks first
// (stored index = polyhedron, ssrc[P] its full-row slot) and then the pair
// blocks (pinfo: full-row slot b in P's row, P, Q, slot of (Q, P)), each
// XCD taking a contiguous share of both, so that the block's loads depend on
// nothing loaded: P's product K_PQ u_Q (FMA-free chain over ascending columns,
// as k_leapfrog) into prod[b], and for a pair block the neighbour's product
// K_QP u_P = K_PQ^T u_P into prod[tdst[b]], the slot of block (Q, P) of Q's
// row.  Lane i holds row i of K_PQ and u_P[i]; the products K_PQ[i][c] u_P[i]
// go to LDS in three chunks of CW columns and lane c adds column c's
// products over ascending rows: the same chain Q's own row would run over
// K_QP's columns, so with K_QP = K_PQ^T exactly (the 32-bit copies) the
// transposed product is the full-row product bit for bit.  A self block's
// product is its upper triangle's row product plus the transposed product
// of its strict upper triangle, both with u_P.  Each wave's stores come after
// all of its loads.  k_sym_update: per polyhedron, the row's products summed
// in block order, then M^-1 = S S^T with S = R^-1 (packed like R) as two
// triangular products through LDS, and the update of k_leapfrog.  p <= 3
// (3Np <= 64 rows, whole column pairs).
__host__ __device__ constexpr int self_upper_off(int c2i) { return 2 * c2i * (c2i + 1); }

// One stored block of k_sym_products (self: a self block's packed upper
// triangle; otherwise a pair block K_PQ with its transposed product).  Kb is
// the block's base plus the lane's offset.  A wave holds its registers until
// its stores are acknowledged, so a pair block's row product is stored before
// the LDS transpose (u_P is loaded with the block: no load follows a store).
template <int P>
__device__ __forceinline__ void sym_block(bool self, const double* __restrict__ Kb, int b, int Pp, int Qq,
                                          int td, const double* __restrict__ u,
                                          double* __restrict__ prod, double* __restrict__ sT,
                                          int lane) {
  using D = Dims<P>;
  constexpr int N3 = D::N3, NPAIR = D::NPAIR, PS = prod_stride(N3);
  constexpr int CW = N3 / 3, CP = CW / 2, LDT = N3 + 1;
  const bool row = lane < N3;
  double2 kv[NPAIR];
#pragma unroll
  for (int c2i = 0; c2i < NPAIR; ++c2i) {
    const bool ld = row && (!self || lane <= 2 * c2i + 1);
    kv[c2i] = ld ? load_stream(Kb + (self ? self_upper_off(c2i) : c2i * N3 * 2))
                 : make_double2(0.0, 0.0);
    if (self && lane == 2 * c2i + 1) kv[c2i].x = 0.0;  // K_PP[lane][lane - 1]: below the diagonal
  }
  const double xl = row ? u[(size_t)Qq * N3 + lane] : 0.0;
  const double up = self ? xl : (row ? u[(size_t)Pp * N3 + lane] : 0.0);  // P's own coefficients
  double s = 0.0;
#pragma unroll
  for (int c2i = 0; c2i < NPAIR; ++c2i) {
    const double x0 = lane_bcast(xl, 2 * c2i), x1 = lane_bcast(xl, 2 * c2i + 1);
    s = s + kv[c2i].x * x0;
    s = s + kv[c2i].y * x1;
  }
  if (!self && lane < PS) prod[(size_t)b * PS + lane] = s;  // lanes past the rows hold zeros
  double st = 0.0;
#pragma unroll
  for (int h = 0; h < 3; ++h) {
    wave_lds_sync();  // the previous chunk's reads are done
    if (row) {
#pragma unroll
      for (int k = 0; k < CP; ++k) {
        sT[(2 * k) * LDT + lane] = kv[h * CP + k].x * up;
        sT[(2 * k + 1) * LDT + lane] = kv[h * CP + k].y * up;
      }
      // the self block's diagonal is in its row product only (a wave's LDS
      // writes land in program order)
      if (self && lane >= h * CW && lane < (h + 1) * CW) sT[(lane - h * CW) * LDT + lane] = 0.0;
    }
    wave_lds_sync();
    if (lane >= h * CW && lane < (h + 1) * CW) {
      const double* __restrict__ colp = sT + (lane - h * CW) * LDT;
      double v = 0.0;
#pragma unroll
      for (int r = 0; r < N3; ++r) v = v + colp[r];
      st = v;
    }
  }
  if (lane < PS) {
    if (self)
      prod[(size_t)b * PS + lane] = s + st;
    else
      prod[(size_t)td * PS + lane] = st;
  }
}

template <int P>
__global__ __launch_bounds__(64) void k_sym_products(const double* __restrict__ Ks,
                                                     const int* __restrict__ ssrc,
                                                     const int4* __restrict__ pinfo,
                                                     const double* __restrict__ u,
                                                     double* __restrict__ prod, int n_poly,
                                                     int n_pair, int self_per, int pair_per) {
  using D = Dims<P>;
  constexpr int N3 = D::N3, NPAIR = D::NPAIR;
  static_assert(N3 <= 64 && N3 % 2 == 0, "one lane per row, whole column pairs");
  static_assert((N3 / 3) % 2 == 0, "whole column pairs per chunk");
  static_assert(self_upper_off(NPAIR) <= D::BS, "packed self block fits its slot");
  __shared__ double sT[(N3 / 3) * (N3 + 1)];  // odd stride: a column read spreads over the banks
  const int lane = threadIdx.x;
  // XCD-aware: workgroup i of XCD x takes self block x self_per + i, or pair
  // x pair_per + (i - self_per); padding workgroups of the last shares leave
  const int xcd = (int)(blockIdx.x & 7), i = (int)(blockIdx.x >> 3);
  const bool self = i < self_per;
  int sb;
  if (self) {
    sb = xcd * self_per + i;
    if (sb >= n_poly) return;
  } else {
    const int j = xcd * pair_per + (i - self_per);
    if (j >= n_pair) return;
    sb = n_poly + j;
  }
  int4 q;
  if (self)
    q = make_int4(ssrc[sb], sb, sb, -1);
  else
    q = pinfo[sb - n_poly];
  sym_block<P>(self, Ks + (size_t)sb * D::BS + 2 * lane, q.x, q.y, q.z, q.w, u, prod, sT, lane);
}

// k_sym_products at small degree (3Np <= 32: p = 1, 2): one wave carries
// G = 64 / 3Np stored blocks, lane = (block, row), so short rows do not leave
// lanes idle.  Per block the sums of sym_block in its order: the row product
// K_PQ u_Q (FMA-free chain over ascending columns, u_Q broadcast from LDS),
// then the block's products K_PQ[i][c] u_P[i] in LDS at once (a self block's
// diagonal zeroed) and lane (block, c) adding column c over ascending rows;
// so the two kernels agree bit for bit.  Stores cover the rows only (the
// update reads no padding).
template <int P>
__global__ __launch_bounds__(64) void k_sym_products_packed(const double* __restrict__ Ks,
                                                            const int* __restrict__ ssrc,
                                                            const int4* __restrict__ pinfo,
                                                            const double* __restrict__ u,
                                                            double* __restrict__ prod, int n_poly,
                                                            int n_stored) {
  using D = Dims<P>;
  constexpr int N3 = D::N3, NPAIR = D::NPAIR, PS = prod_stride(N3);
  static_assert(N3 <= 32 && N3 % 2 == 0, "packed stored blocks need 3Np <= 32, whole column pairs");
  static_assert(self_upper_off(NPAIR) <= D::BS, "packed self block fits its slot");
  constexpr int G = 64 / N3;
  __shared__ double sX[G][N3];          // u_Q of each block
  __shared__ double sT[G][N3][N3 + 1];  // K_PQ[i][c] u_P[i]; odd row stride
  const int lane = threadIdx.x, sub = lane / N3, r = lane % N3;
  // XCD-aware: workgroups are dealt to the XCDs round robin; XCD x takes a
  // contiguous eighth of the waves, hence of the stored blocks
  const int per = (int)(gridDim.x >> 3);
  const int w = (int)(blockIdx.x & 7) * per + (int)(blockIdx.x >> 3);
  const int sb = w * G + sub;
  const bool on = sub < G && sb < n_stored;
  const bool self = sb < n_poly;
  int b = 0, Pp = 0, Qq = 0, td = 0;
  if (on) {
    if (self) {
      b = ssrc[sb];
      Pp = Qq = sb;
    } else {
      const int4 q = pinfo[sb - n_poly];
      b = q.x;
      Pp = q.y;
      Qq = q.z;
      td = q.w;
    }
  }
  const double* __restrict__ Kb = Ks + (size_t)(on ? sb : 0) * D::BS;
  double2 kv[NPAIR];
#pragma unroll
  for (int c2i = 0; c2i < NPAIR; ++c2i) {
    const bool ld = on && (!self || r <= 2 * c2i + 1);
    kv[c2i] = ld ? load_stream(Kb + (self ? self_upper_off(c2i) + 2 * r : ((size_t)c2i * N3 + r) * 2))
                 : make_double2(0.0, 0.0);
    if (self && r == 2 * c2i + 1) kv[c2i].x = 0.0;  // K_PP[r][r - 1]: below the diagonal
  }
  const double xl = on ? u[(size_t)Qq * N3 + r] : 0.0;
  const double up = on ? u[(size_t)Pp * N3 + r] : 0.0;
  if (on) sX[sub][r] = xl;
  __syncthreads();
  double s = 0.0;
  if (on) {
#pragma unroll
    for (int c2i = 0; c2i < NPAIR; ++c2i) {
      s = s + kv[c2i].x * sX[sub][2 * c2i];
      s = s + kv[c2i].y * sX[sub][2 * c2i + 1];
    }
  }
  if (on) {
#pragma unroll
    for (int c2i = 0; c2i < NPAIR; ++c2i) {
      sT[sub][r][2 * c2i] = kv[c2i].x * up;
      sT[sub][r][2 * c2i + 1] = kv[c2i].y * up;
    }
    if (self) sT[sub][r][r] = 0.0;  // the diagonal is in the row product only
  }
  __syncthreads();
  double st = 0.0;
  if (on) {
    double v = 0.0;  // column r of this block over ascending rows
#pragma unroll
    for (int i = 0; i < N3; ++i) v = v + sT[sub][i][r];
    st = v;
  }
  if (on) {
    if (self) {
      prod[(size_t)b * PS + r] = s + st;
    } else {
      prod[(size_t)b * PS + r] = s;
      prod[(size_t)td * PS + r] = st;
    }
  }
}

// K_PP's upper triangle in the packed layout of k_sym_products, one thread
// per stored entry: the self blocks listed in self_s (stored index s, taken
// from full-row slot src[s]).
template <int P>
__global__ void k_pack_self_upper(const double* __restrict__ K, double* __restrict__ Ks,
                                  const int* __restrict__ src, const int* __restrict__ self_s,
                                  int n_self) {
  using D = Dims<P>;
  constexpr int N3 = D::N3, NPAIR = D::NPAIR, NE = self_upper_off(NPAIR);
  const size_t id = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (id >= (size_t)n_self * NE) return;
  const int k = (int)(id / NE), e = (int)(id % NE);
  int c2i = 0;  // column pair of packed entry e: self_upper_off(c2i) <= e < self_upper_off(c2i + 1)
  while (self_upper_off(c2i + 1) <= e) ++c2i;
  const int r = (e - self_upper_off(c2i)) >> 1, h = e & 1;
  const int s = self_s[k];
  Ks[(size_t)s * D::BS + e] = K[(size_t)src[s] * D::BS + ((size_t)c2i * N3 + r) * 2 + h];
}

template <int P, int MODE>
__global__ __launch_bounds__(64) void k_sym_update(const double* __restrict__ prod,
                                                   const int* __restrict__ row_ptr,
                                                   const double* __restrict__ Sp,
                                                   const double* __restrict__ rs,
                                                   const double* __restrict__ rd,
                                                   const double* __restrict__ u,
                                                   const double* __restrict__ wa,
                                                   double* __restrict__ out, double g, double c1,
                                                   double c2, const int* __restrict__ gsel,
                                                   const double* __restrict__ gtab, int n_poly,
                                                   const int* __restrict__ order) {
  using D = Dims<P>;
  constexpr int NP = D::NP, N3 = D::N3;
  static_assert(N3 <= 64, "one lane per row");
  static_assert(MODE == 0 || MODE == 1, "leapfrog and first step");
  __shared__ double sS[D::NPK];
  __shared__ double sv[N3];
  const int lane = threadIdx.x;
  const bool row = lane < N3;
  const int Pp = step_poly(order);
  if (Pp >= n_poly) return;
  for (int k = lane; k < D::NPK; k += 64) sS[k] = Sp[(size_t)Pp * D::NPK + k];
  const int b0 = row_ptr[Pp], b1 = row_ptr[Pp + 1];
  const size_t o = (size_t)Pp * N3;
  double vs = 0.0, vd = 0.0, vu = 0.0, va = 0.0;
  if (row) {
    vs = rs[o + lane];
    vd = rd[o + lane];
    vu = u[o + lane];
    va = wa[o + lane];
  }
  // the row's products, eight loads in flight at a time, added in block order
  double acc = 0.0;
  if (row) {
    for (int b = b0; b < b1; b += 8) {
      double v[8];
#pragma unroll
      for (int k = 0; k < 8; ++k)
        v[k] = b + k < b1 ? prod[(size_t)(b + k) * prod_stride(N3) + lane] : 0.0;
#pragma unroll
      for (int k = 0; k < 8; ++k)
        if (b + k < b1) acc = (b + k == b0) ? v[k] : acc + v[k];
    }
  }
  const double gp = gsel ? gtab[gsel[Pp]] : g;
  const int cc = row ? lane / NP : 0, ii = lane % NP;
  const double* __restrict__ vc = sv + cc * NP;  // this lane's component
  if (row) sv[lane] = -acc + vs + vd * gp;
  __syncthreads();  // sS, sv
  // z = S^T w: z_i = sum_{j <= i} S_ji w_j
  double z = 0.0;
  if (row) {
#pragma unroll
    for (int j = 0; j < NP; ++j)
      if (j <= ii) z = z + sS[pk_off(NP, j) + (ii - j)] * vc[j];
  }
  __syncthreads();
  if (row) sv[lane] = z;
  __syncthreads();
  // M^-1 w = S z: x_i = sum_{j >= i} S_ij z_j
  double w = 0.0;
  if (row) {
#pragma unroll
    for (int j = 0; j < NP; ++j)
      if (j >= ii) w = w + sS[pk_off(NP, ii) + (j - ii)] * vc[j];
    if (MODE == 0)
      out[o + lane] = c1 * w + 2.0 * vu - va;
    else
      out[o + lane] = c1 * w + vu + c2 * va;
  }
}

// k_sym_update at small degree (3Np <= 32: p = 1, 2): G = 64 / 3Np
// polyhedra per wave, lane = (polyhedron, row), each with its own S and
// vector in LDS; the sums of k_sym_update in its order, so the two agree bit
// for bit.
template <int P, int MODE>
__global__ __launch_bounds__(64) void k_sym_update_packed(const double* __restrict__ prod,
                                                          const int* __restrict__ row_ptr,
                                                          const double* __restrict__ Sp,
                                                          const double* __restrict__ rs,
                                                          const double* __restrict__ rd,
                                                          const double* __restrict__ u,
                                                          const double* __restrict__ wa,
                                                          double* __restrict__ out, double g,
                                                          double c1, double c2,
                                                          const int* __restrict__ gsel,
                                                          const double* __restrict__ gtab, int n_poly) {
  using D = Dims<P>;
  constexpr int NP = D::NP, N3 = D::N3;
  static_assert(N3 <= 32, "packed update needs 3Np <= 32");
  static_assert(MODE == 0 || MODE == 1, "leapfrog and first step");
  constexpr int G = 64 / N3;
  __shared__ double sS[G][D::NPK];
  __shared__ double sv[G][N3];
  const int lane = threadIdx.x, sub = lane / N3, r = lane % N3;
  const int P0 = step_poly() * G;
  const int Pp = P0 + sub;
  const bool act = sub < G && Pp < n_poly;
  for (int k = lane; k < G * D::NPK; k += 64) {
    const int sp = k / D::NPK, e = k % D::NPK;
    if (P0 + sp < n_poly) sS[sp][e] = Sp[(size_t)(P0 + sp) * D::NPK + e];
  }
  const size_t o = (size_t)Pp * N3 + r;
  double vs = 0.0, vd = 0.0, vu = 0.0, va = 0.0, acc = 0.0;
  if (act) {
    vs = rs[o];
    vd = rd[o];
    vu = u[o];
    va = wa[o];
    const int b0 = row_ptr[Pp], b1 = row_ptr[Pp + 1];
    for (int b = b0; b < b1; b += 8) {  // the row's products, added in block order
      double v[8];
#pragma unroll
      for (int k = 0; k < 8; ++k) v[k] = b + k < b1 ? prod[(size_t)(b + k) * prod_stride(N3) + r] : 0.0;
#pragma unroll
      for (int k = 0; k < 8; ++k)
        if (b + k < b1) acc = (b + k == b0) ? v[k] : acc + v[k];
    }
  }
  const int cc = r / NP, ii = r % NP;
  const double* __restrict__ vc = &sv[act ? sub : 0][cc * NP];  // this lane's component
  if (act) {
    const double gp = gsel ? gtab[gsel[Pp]] : g;
    sv[sub][r] = -acc + vs + vd * gp;
  }
  __syncthreads();  // sS, sv
  double z = 0.0;  // z = S^T w: z_i = sum_{j <= i} S_ji w_j
  if (act) {
#pragma unroll
    for (int j = 0; j < NP; ++j)
      if (j <= ii) z = z + sS[sub][pk_off(NP, j) + (ii - j)] * vc[j];
  }
  __syncthreads();
  if (act) sv[sub][r] = z;
  __syncthreads();
  if (act) {  // M^-1 w = S z: x_i = sum_{j >= i} S_ij z_j
    double w = 0.0;
#pragma unroll
    for (int j = 0; j < NP; ++j)
      if (j >= ii) w = w + sS[sub][pk_off(NP, ii) + (j - ii)] * vc[j];
    if (MODE == 0)
      out[o] = c1 * w + 2.0 * vu - va;
    else
      out[o] = c1 * w + vu + c2 * va;
  }
}

// The pairs-once steps of the 32- and 48-bit applies (mass-orthonormal
// basis, no solves): ~K_QP = R_Q^-T K_PQ^T R_P^-1 = ~K_PQ^T, so the stored
// list of the FP64 step applies to the FP32 blocks (column quads, 3Np a
// multiple of 12 so that each of three chunks is whole quads: p = 3).  A
// self block keeps its upper triangle by column quads: quad q's rows
// 0..4q+3 from float self32_off(q), row r at self32_off(q) + 4r (and the
// 48-bit corrections by quad pairs: pair k's rows 0..min(8k+7, 3Np-1) from
// half self16_off(k), row r at self16_off(k) + self16_w(k) r, 8 halves per
// row, 4 for the last quad of an odd count); entries below the diagonal that
// a quad's rows carry are zeroed on load.
//
// One wave per polyhedron walks its row's stored blocks.  Lane i holds row i
// of the block; the block's entries go to LDS in three chunks of CW columns,
// and lane c runs column c's chain over ascending rows r with u_P[r] -- the
// chain Q's own full row runs over block (Q, P), so where the two rounded
// blocks are exact transposes the transposed product equals the full rows'
// bit for bit.  Then each lane's row chain over ascending columns: from zero
// for a pair block, and for a self block continuing its own column chain
// (the strict upper triangle's column r holds row r's entries left of the
// diagonal, in the full row's order), so a self block's product is also the
// full rows' product bit for bit.  (Summing the transposed products in three
// row groups instead made the 32-bit state drift from FP64 faster over long
// runs, increasingly with the mesh size: 7x the full rows' drift after 1000
// steps at 40^3.)
//
// A wave adds the row products of its stored blocks in FP64 (block order)
// and stores that sum once, rowp[P]; only a pair block's transposed product
// is stored per block, in the slot of block (Q, P) of Q's row.
// k_sym_update32 adds to rowp[P] the transposed products of the blocks kept
// in the neighbours' rows (sidx < 0), in block order, in FP64, and applies
// k_leapfrog32's update.
//
// 32-bit: products and per-block sums in FP32 as k_leapfrog32, transposed
// products stored as floats (prod_stride(3Np) per block, half the bytes of a
// 64-bit product; PT = double: the 48-bit apply's, k_sym_products48).
LYMPH_HD constexpr int self32_off(int q) { return 8 * q * (q + 1); }
LYMPH_HD constexpr int self16_rows(int n3, int k) { return 8 * k + 8 < n3 ? 8 * k + 8 : n3; }
LYMPH_HD constexpr int self16_w(int n3, int k) { return 2 * k + 1 < n3 / 4 ? 8 : 4; }
LYMPH_HD constexpr int self16_off(int n3, int k) {
  int o = 0;
  for (int i = 0; i < k; ++i) o += self16_w(n3, i) * self16_rows(n3, i);
  return o;
}

// A self block's upper triangle in the packed layouts above, from the
// full-row block of slot src[s] (s < n_self): one thread per packed entry.
template <int P>
__global__ void k_pack_self32(const float* __restrict__ K, float* __restrict__ Ks,
                              const int* __restrict__ src, int n_self) {
  constexpr int N3 = Dims32<P>::N3, NE = self32_off(Dims32<P>::NQ);
  const size_t id = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (id >= (size_t)n_self * NE) return;
  const int s = (int)(id / NE), e = (int)(id % NE);
  int q = 0;
  while (self32_off(q + 1) <= e) ++q;
  const int r = (e - self32_off(q)) >> 2, c = 4 * q + (e & 3);
  Ks[(size_t)s * Dims32<P>::BS + e] = K[(size_t)src[s] * Dims32<P>::BS + kpos32(N3, r, c)];
}
template <int P>
__global__ void k_pack_self16(const _Float16* __restrict__ K, _Float16* __restrict__ Ks,
                              const int* __restrict__ src, int n_self) {
  constexpr int N3 = Dims32<P>::N3, NE = self16_off(N3, Dims16<P>::NPR);
  const size_t id = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (id >= (size_t)n_self * NE) return;
  const int s = (int)(id / NE), e = (int)(id % NE);
  int k = 0;
  while (self16_off(N3, k + 1) <= e) ++k;
  const int w = self16_w(N3, k), r = (e - self16_off(N3, k)) / w, h = (e - self16_off(N3, k)) % w;
  const int c = 8 * k + h;  // quad 2k + h / 4, column h % 4 of it
  Ks[(size_t)s * Dims16<P>::BS + e] = K[(size_t)src[s] * Dims16<P>::BS + kpos16(N3, r, c)];
}

template <int P>
__global__ __launch_bounds__(64) void k_sym_products32(const float* __restrict__ Ks,
                                                       const int* __restrict__ row_ptr,
                                                       const int* __restrict__ col,
                                                       const int* __restrict__ sidx,
                                                       const int* __restrict__ tdst,
                                                       const double* __restrict__ u,
                                                       float* __restrict__ prod,
                                                       double* __restrict__ rowp, int n_poly,
                                                       const int* __restrict__ order) {
  constexpr int N3 = Dims32<P>::N3, NQ = Dims32<P>::NQ;
  static_assert(N3 <= 64 && N3 % 12 == 0, "one lane per row, whole quads per chunk");
  static_assert(self32_off(NQ) <= (int)Dims32<P>::BS, "packed self block fits its slot");
  constexpr int CW = N3 / 3, CQ = CW / 4;
  // one chunk row by row (lanes past the rows write padding rows): a lane
  // stores its quads with 16-byte writes, and a column read over 20 lanes
  // touches 20 distinct banks
  __shared__ __align__(16) float sT[64 * CW];
  __shared__ __align__(16) float sX[64];  // u_Q of the current block, read by the row chains
  const int lane = threadIdx.x;
  const bool row = lane < N3;
  const int rl = row ? lane : N3 - 1;  // lanes past the rows load the last row's (cached) lines
  const int Pp = step_poly(order);
  if (Pp >= n_poly) return;  // padding workgroups of the last XCD share
  const int b0 = row_ptr[Pp], b1 = row_ptr[Pp + 1];
  const int lcb = lane < b1 - b0 ? col[b0 + lane] : 0;
  const int lsi = lane < b1 - b0 ? sidx[b0 + lane] : 0;
  const int ltd = lane < b1 - b0 ? tdst[b0 + lane] : 0;
  const float up = (float)u[(size_t)Pp * N3 + rl];
  double racc = 0.0;  // the row products of this wave's stored blocks, in block order
  for (int b = b0; b < b1; ++b) {
    const int j = b - b0;
    const int si = j < 64 ? __builtin_amdgcn_readlane(lsi, j) : __builtin_amdgcn_readfirstlane(sidx[b]);
    if (si < 0) continue;  // written by the neighbour's wave
    const int cb = j < 64 ? __builtin_amdgcn_readlane(lcb, j) : __builtin_amdgcn_readfirstlane(col[b]);
    const int td = j < 64 ? __builtin_amdgcn_readlane(ltd, j) : __builtin_amdgcn_readfirstlane(tdst[b]);
    const bool pair = cb != Pp;
    const float* __restrict__ Kb = Ks + (size_t)si * Dims32<P>::BS;
    const float xl = (float)u[(size_t)cb * N3 + rl];
    // the self blocks' row clamps and masks are formed per block: hoisted
    // out of the loop they would hold 60 masks in scalar registers
    int rb = rl;
    asm volatile("" : "+v"(rb));
    // one load path for both kinds (an address select per quad), so that the
    // chunks wait on their own quads only
    float4 kq[NQ];
#pragma unroll
    for (int q = 0; q < NQ; ++q)
      kq[q] = load_stream(Kb + (pair ? (q * N3 + rb) * 4 : self32_off(q) + 4 * (rb < 4 * q + 3 ? rb : 4 * q + 3)));
    if (!pair) {  // the upper triangle's rows only
#pragma unroll
      for (int q = 0; q < NQ; ++q) {
        if (4 * q + 0 < rb) kq[q].x = 0.0f;
        if (4 * q + 1 < rb) kq[q].y = 0.0f;
        if (4 * q + 2 < rb) kq[q].z = 0.0f;
        if (4 * q + 3 < rb) kq[q].w = 0.0f;
      }
    }
    float st = 0.0f;
#pragma unroll
    for (int h = 0; h < 3; ++h) {
      wave_lds_sync();  // the previous chunk's (and block's) reads are done
      if (h == 0) sX[lane] = xl;  // lanes past the rows write padding
#pragma unroll
      for (int k = 0; k < CQ; ++k) {
        const float4 v = kq[h * CQ + k];
        *reinterpret_cast<float4*>(sT + lane * CW + 4 * k) =
            make_float4(v.x * up, v.y * up, v.z * up, v.w * up);
      }
      // a self block's diagonal belongs to its rows only (a wave's LDS
      // writes land in program order)
      if (!pair && lane >= h * CW && lane < (h + 1) * CW) sT[lane * CW + (lane - h * CW)] = 0.0f;
      wave_lds_sync();
      if (lane >= h * CW && lane < (h + 1) * CW) {  // column's chain over ascending rows
        const float* __restrict__ colp = sT + (lane - h * CW);
        float v = 0.0f;
#pragma unroll
        for (int r = 0; r < N3; ++r) v = v + colp[r * CW];
        st = v;
      }
    }
    float s = pair ? 0.0f : st;
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
      const float4 xq = *reinterpret_cast<const float4*>(sX + 4 * q);  // a broadcast
      s = s + kq[q].x * xq.x;
      s = s + kq[q].y * xq.y;
      s = s + kq[q].z * xq.z;
      s = s + kq[q].w * xq.w;
    }
    // the block's row chain ends here: left free, the compiler interleaves it
    // with the next block's loads and holds both in registers
    asm volatile("" : "+v"(s));
    racc = racc + (double)s;
    if (pair && lane < prod_stride(N3)) prod[(size_t)td * prod_stride(N3) + lane] = row ? st : 0.0f;
  }
  if (lane < prod_stride(N3)) rowp[(size_t)Pp * prod_stride(N3) + lane] = row ? racc : 0.0;
}

template <int P, int MODE, typename PT = float>
__global__ __launch_bounds__(64) void k_sym_update32(const PT* __restrict__ prod,
                                                     const double* __restrict__ rowp,
                                                     const int* __restrict__ sidx,
                                                     const int* __restrict__ row_ptr,
                                                     const double* __restrict__ rs,
                                                     const double* __restrict__ rd,
                                                     const double* __restrict__ u,
                                                     const double* __restrict__ wa,
                                                     double* __restrict__ out, double g, double c1,
                                                     double c2, const int* __restrict__ gsel,
                                                     const double* __restrict__ gtab, int n_poly,
                                                     const int* __restrict__ order) {
  constexpr int N3 = Dims32<P>::N3;
  static_assert(N3 <= 64, "one lane per row");
  static_assert(MODE == 0 || MODE == 1, "leapfrog and first step");
  const int lane = threadIdx.x;
  if (lane >= N3) return;  // no barrier in this kernel
  const int Pp = step_poly(order);
  if (Pp >= n_poly) return;
  const int b0 = row_ptr[Pp], b1 = row_ptr[Pp + 1];
  const size_t o = (size_t)Pp * N3;
  const double vs = rs[o + lane], vd = rd[o + lane], vu = u[o + lane], va = wa[o + lane];
  // the wave's own row products (summed by the products pass), then the
  // neighbours' transposed products in block order
  double acc = rowp[(size_t)Pp * prod_stride(N3) + lane];
  for (int b = b0; b < b1; b += 8) {
    double v[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const bool theirs = b + k < b1 && sidx[b + k] < 0;
      v[k] = theirs ? (double)prod[(size_t)(b + k) * prod_stride(N3) + lane] : 0.0;
    }
#pragma unroll
    for (int k = 0; k < 8; ++k)
      if (b + k < b1 && sidx[b + k] < 0) acc = acc + v[k];
  }
  const double gp = gsel ? gtab[gsel[Pp]] : g;
  const double w = -acc + vs + vd * gp;
  if (MODE == 0)
    out[o + lane] = c1 * w + 2.0 * vu - va;
  else
    out[o + lane] = c1 * w + vu + c2 * va;
}

// Symmetry of the operator, pair by pair: ratio[w] = max |K_PQ - K_QP^T| /
// max |K_PQ| for the blocks pb[w] = K_PQ and pt[w] = K_QP (column-pair
// layout, whole pairs: 3Np even).
template <int P>
__global__ __launch_bounds__(64) void k_pair_asym(const double* __restrict__ K,
                                                  const int* __restrict__ pb,
                                                  const int* __restrict__ pt, int n_pairs,
                                                  double* __restrict__ ratio) {
  using D = Dims<P>;
  constexpr int N3 = D::N3;
  static_assert(N3 % 2 == 0, "whole column pairs");
  const int w = blockIdx.x;
  if (w >= n_pairs) return;
  const double* A = K + (size_t)pb[w] * D::BS;
  const double* B = K + (size_t)pt[w] * D::BS;
  double dmax = 0.0, amax = 0.0;
  for (int e = threadIdx.x; e < N3 * N3; e += 64) {
    const int r = e % N3, c = e / N3;
    const double a = A[((size_t)(c >> 1) * N3 + r) * 2 + (c & 1)];   // K_PQ[r][c]
    const double bt = B[((size_t)(r >> 1) * N3 + c) * 2 + (r & 1)];  // K_QP[c][r]
    const double d = fabs(a - bt);
    dmax = (d > dmax || d != d) ? d : dmax;  // a NaN makes the pair fail
    amax = fabs(a) > amax ? fabs(a) : amax;
  }
  for (int off = 32; off > 0; off >>= 1) {
    const double od = __shfl_xor(dmax, off, 64), oa = __shfl_xor(amax, off, 64);
    dmax = (od > dmax || od != od) ? od : dmax;
    amax = oa > amax ? oa : amax;
  }
  if (threadIdx.x == 0) ratio[w] = dmax == 0.0 ? 0.0 : dmax / amax;
}

// Ks[s] = K[src[s]], whole blocks of bs entries.
template <class T>
__global__ void k_gather_blocks(const T* __restrict__ K, T* __restrict__ Ks,
                                const int* __restrict__ src, int n, size_t bs) {
  const size_t total = (size_t)n * bs;
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < total;
       i += (size_t)gridDim.x * blockDim.x) {
    const size_t s = i / bs, k = i - s * bs;
    Ks[i] = K[(size_t)src[s] * bs + k];
  }
}

// Barrier of the packed kernels: a whole workgroup for one-wave workgroups;
// with several waves per workgroup each wave owns its own LDS region and
// polyhedra (and its own loop trip count), so only the wave's own LDS
// traffic is ordered (the rocPRIM wave barrier: fences at wavefront scope
// around a code-motion barrier; a wave's LDS operations complete in order).
template <int WPW>
__device__ inline void lsync() {
  if constexpr (WPW == 1) {
    __syncthreads();
  } else {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  }
}

// Packed variant of the step for small blocks (3Np <= 32: p = 1, 2): one
// wave carries G = 64 / 3Np polyhedra, lane = (polyhedron, row), so lanes are
// not left idle by short rows.  Each polyhedron walks its own block row; the
// neighbour's coefficients go through LDS (one segment per polyhedron); the
// block products are added in block order and the solves and update are the
// ones of k_leapfrog, so results are bit-identical to it.  TB = 64 (FP64
// operator in column pairs), 32 (mass-orthonormal FP32 operator in column
// quads, no solves) or 48 (the FP32 operator plus its 16-bit corrections Kr,
// with k_leapfrog48's arithmetic in its order: bit-identical to it).
template <int P, int MODE, int TB, int WPW, bool NT>
__global__ __launch_bounds__(64 * WPW) void k_leapfrog_packed(const void* __restrict__ Kv,
                                                        const _Float16* __restrict__ Kr,
                                                        const int* __restrict__ row_ptr,
                                                        const int* __restrict__ col,
                                                        const double* __restrict__ Rp,
                                                        const double* __restrict__ rs,
                                                        const double* __restrict__ rd,
                                                        const double* __restrict__ u,
                                                        const double* __restrict__ wa,
                                                        double* __restrict__ out, double g,
                                                        double c1, double c2,
                                                        const int* __restrict__ gsel,
                                                        const double* __restrict__ gtab,
                                                        int n_poly) {
  using D = Dims<P>;
  constexpr int NP = D::NP, N3 = D::N3, NPAIR = D::NPAIR;
  static_assert(N3 <= 32, "packed step needs 3Np <= 32");
  constexpr int G = 64 / N3;
  constexpr int NQUAD = Dims32<P>::NQ, TAIL = Dims32<P>::T;
  // neighbour coefficients, double-buffered by block parity: one barrier per block
  __shared__ double sxa[WPW][2][G][N3 + 1];
  __shared__ double swa[WPW][G][N3];
  __shared__ double sRa[WPW][G][D::NPK + 1];  // the factors, each and a zero
  const int wv = threadIdx.x >> 6;
  double(&sx)[2][G][N3 + 1] = sxa[wv];
  double(&sw)[G][N3] = swa[wv];
  double(&sR)[G][D::NPK + 1] = sRa[wv];
  const int lane = threadIdx.x & 63;
  const int sub = lane / N3, r = lane % N3;
  const int P0 = (step_poly() * WPW + wv) * G;
  const int Pp = P0 + sub;
  const bool act = sub < G && Pp < n_poly;
  if (MODE != 2 && TB == 64)
    for (int k = lane; k < G * (D::NPK + 1); k += 64) {
      const int sp = k / (D::NPK + 1), e = k % (D::NPK + 1), Q = P0 + sp;
      if (Q < n_poly) sR[sp][e] = e < D::NPK ? Rp[(size_t)Q * D::NPK + e] : 0.0;
    }
  const int b0 = act ? row_ptr[Pp] : 0, cnt = act ? row_ptr[Pp + 1] - b0 : 0;
  double xn = cnt > 0 ? u[(size_t)col[b0] * N3 + r] : 0.0;  // neighbour value of the next block
  double acc = 0.0;
  for (int j = 0; __any(j < cnt); ++j) {
    const bool on = j < cnt;
    const int b = b0 + j;
    const int buf = j & 1;
    // the block's loads and the next neighbour value are issued before the
    // barrier, so they overlap the exchange of this block's coefficients
    double2 kd[TB == 64 ? NPAIR : 1];
    float4 kf[TB != 64 ? NQUAD : 1];
    float kt[TB != 64 && TAIL > 0 ? TAIL : 1];
    lymph_hv8 kr[TB == 48 ? (NQUAD + 1) / 2 : 1];
    float krt[TB == 48 && TAIL > 0 ? TAIL : 1];
    if (on) {
      if constexpr (TB == 64) {
        const double* Kb = static_cast<const double*>(Kv) + (size_t)b * D::BS;
#pragma unroll
        for (int c2i = 0; c2i < NPAIR; ++c2i) kd[c2i] = load_stream<NT>(Kb + ((size_t)c2i * N3 + r) * 2);
      } else {
        const float* Kb = static_cast<const float*>(Kv) + (size_t)b * Dims32<P>::BS;
#pragma unroll
        for (int q = 0; q < NQUAD; ++q) kf[q] = load_stream<NT>(Kb + ((size_t)q * N3 + r) * 4);
        if constexpr (TAIL > 0) load_tail<NT>(Kb + (size_t)4 * NQUAD * N3 + (size_t)r * TAIL, kt);
        if constexpr (TB == 48) {
          const _Float16* Rb = Kr + (size_t)b * Dims16<P>::BS;
#pragma unroll
          for (int k = 0; k < (NQUAD + 1) / 2; ++k) {
            if (2 * k + 1 < NQUAD) {
              kr[k] = load_stream_h8<NT>(Rb + ((size_t)k * N3 + r) * 8);
            } else {  // the last quad of an odd count: 4 values per row
              const lymph_hv4 h = load_stream_h4<NT>(Rb + Dims16<P>::HALF0 + (size_t)r * 4);
              kr[k] = lymph_hv8{h.x, h.y, h.z, h.w, 0, 0, 0, 0};
            }
          }
          if constexpr (TAIL > 0) {
#pragma unroll
            for (int j = 0; j < TAIL; ++j) krt[j] = (float)Rb[Dims16<P>::TAIL0 + (size_t)r * TAIL + j];
          }
        }
      }
      sx[buf][sub][r] = xn;
      if (j + 1 < cnt) xn = u[(size_t)col[b + 1] * N3 + r];
    }
    lsync<WPW>();
    if (on) {
      double s = 0.0;
      if constexpr (TB == 64) {
#pragma unroll
        for (int c2i = 0; c2i < NPAIR; ++c2i) {
          const bool odd_tail = (N3 % 2 == 1) && (c2i == NPAIR - 1);
          s = s + kd[c2i].x * sx[buf][sub][2 * c2i];
          if (!odd_tail) s = s + kd[c2i].y * sx[buf][sub][2 * c2i + 1];
        }
      } else if constexpr (TB == 48) {  // k_leapfrog48's chains
        double sd = 0.0;
        float sc = 0.0f;
#pragma unroll
        for (int q = 0; q < NQUAD; ++q) {
          double xq[4];
#pragma unroll
          for (int jj = 0; jj < 4; ++jj) xq[jj] = (4 * q + jj < N3) ? sx[buf][sub][4 * q + jj] : 0.0;
          const lymph_hv8 t8 = kr[q >> 1];
          const int o4 = (q & 1) * 4;
          sd = fma((double)kf[q].x, xq[0], sd);
          sd = fma((double)kf[q].y, xq[1], sd);
          sd = fma((double)kf[q].z, xq[2], sd);
          sd = fma((double)kf[q].w, xq[3], sd);
          sc = fmaf(kf[q].x * (float)t8[o4 + 0], (float)xq[0], sc);
          sc = fmaf(kf[q].y * (float)t8[o4 + 1], (float)xq[1], sc);
          sc = fmaf(kf[q].z * (float)t8[o4 + 2], (float)xq[2], sc);
          sc = fmaf(kf[q].w * (float)t8[o4 + 3], (float)xq[3], sc);
        }
        if constexpr (TAIL > 0) {
#pragma unroll
          for (int j = 0; j < TAIL; ++j) {
            const double xt = sx[buf][sub][4 * NQUAD + j];
            sd = fma((double)kt[j], xt, sd);
            sc = fmaf(kt[j] * krt[j], (float)xt, sc);
          }
        }
        s = sd + (double)sc * 0x1p-24;
      } else {
        float sf = 0.0f;
#pragma unroll
        for (int q = 0; q < NQUAD; ++q) {
          float xq[4];
#pragma unroll
          for (int jj = 0; jj < 4; ++jj)
            xq[jj] = (4 * q + jj < N3) ? (float)sx[buf][sub][4 * q + jj] : 0.0f;
          sf = sf + kf[q].x * xq[0];
          sf = sf + kf[q].y * xq[1];
          sf = sf + kf[q].z * xq[2];
          sf = sf + kf[q].w * xq[3];
        }
        if constexpr (TAIL > 0) {
#pragma unroll
          for (int j = 0; j < TAIL; ++j) sf = sf + kt[j] * (float)sx[buf][sub][4 * NQUAD + j];
        }
        s = (double)sf;
      }
      acc = (j == 0) ? s : acc + s;
    }
  }
  const size_t o = (size_t)Pp * N3 + r;
  if (MODE == 2) {
    if (act) sw[sub][r] = acc;
    lsync<WPW>();
    if (act && r == 0) {
      double el = 0.0;
      for (int k = 0; k < N3; ++k) el = el + u[(size_t)Pp * N3 + k] * sw[sub][k];
      out[Pp] = el;
    }
    return;
  }
  double w = 0.0;
  if (act) {
    const double gp = gsel ? gtab[gsel[Pp]] : g;
    w = -acc + rs[o] + rd[o] * gp;
  }
  if constexpr (TB == 64) {
    lsync<WPW>();  // sR
    const double* R = sR[act ? sub : 0];
    w = solve_group<NP>(R, Divisor(act ? R[pk_off(NP, r % NP)] : 1.0), w, sub * N3, r, act);
  }
  if (act) {
    if (MODE == 0)
      out[o] = c1 * w + 2.0 * u[o] - wa[o];
    else
      out[o] = c1 * w + u[o] + c2 * wa[o];
  }
}

// Packed step with a joint block walk (3Np <= 32): the G polyhedra of a wave
// own the contiguous block range row_ptr[P0] .. row_ptr[P0 + G]; at loop
// iteration j lane group s takes block B0 + j G + s, so each iteration
// streams G consecutive blocks and no cache line is left half read for a
// later iteration (32-bit blocks of 576 B at p = 1 end mid-line).  Each
// block's product goes to LDS; each row then adds its own blocks in block
// order, so results are bit-identical to k_leapfrog (TB = 48: to
// k_leapfrog48, with Kr its 16-bit corrections).  Dynamic LDS: the products
// of the wave's longest block range (G x longest row x 3Np doubles).
template <int P, int MODE, int TB, int WPW, bool NT>
__global__ __launch_bounds__(64 * WPW) void k_leapfrog_joint(const void* __restrict__ Kv,
                                                       const _Float16* __restrict__ Kr,
                                                       const int* __restrict__ row_ptr,
                                                       const int* __restrict__ col,
                                                       const double* __restrict__ Rp,
                                                       const double* __restrict__ rs,
                                                       const double* __restrict__ rd,
                                                       const double* __restrict__ u,
                                                       const double* __restrict__ wa,
                                                       double* __restrict__ out, double g,
                                                       double c1, double c2,
                                                       const int* __restrict__ gsel,
                                                       const double* __restrict__ gtab,
                                                       int n_poly, int prod_stride) {
  using D = Dims<P>;
  constexpr int NP = D::NP, N3 = D::N3, NPAIR = D::NPAIR;
  static_assert(N3 <= 32, "joint packed step needs 3Np <= 32");
  constexpr int G = 64 / N3;
  constexpr int NQUAD = Dims32<P>::NQ, TAIL = Dims32<P>::T;
  __shared__ double sxa[WPW][2][G][N3 + 1];
  __shared__ double swa[WPW][G][N3];
  __shared__ double sRa[WPW][G][D::NPK + 1];  // the factors, each and a zero
  const int wv = threadIdx.x >> 6;
  double(&sx)[2][G][N3 + 1] = sxa[wv];
  double(&sw)[G][N3] = swa[wv];
  double(&sR)[G][D::NPK + 1] = sRa[wv];
  extern __shared__ double prod_all[];  // per wave: [block - B0][row]
  const int lane = threadIdx.x & 63;
  const int sub = lane / N3, r = lane % N3;
  const int P0 = (step_poly() * WPW + wv) * G;
  const int Pp = P0 + sub;
  const bool act = sub < G && Pp < n_poly;
  if (MODE != 2 && TB == 64)
    for (int k = lane; k < G * (D::NPK + 1); k += 64) {
      const int sp = k / (D::NPK + 1), e = k % (D::NPK + 1), Q = P0 + sp;
      if (Q < n_poly) sR[sp][e] = e < D::NPK ? Rp[(size_t)Q * D::NPK + e] : 0.0;
    }
  if (P0 >= n_poly) return;  // padding group: the wave exits before any barrier
  double* prod = prod_all + (size_t)wv * prod_stride;
  const int B0 = row_ptr[P0], B1 = row_ptr[min(P0 + G, n_poly)];
  const int nblk = B1 - B0;
  int bj = B0 + sub;  // this lane group's block at iteration 0
  double xn = (sub < G && bj < B1) ? u[(size_t)col[bj] * N3 + r] : 0.0;
  for (int j = 0; j * G < nblk; ++j, bj += G) {
    const bool on = sub < G && bj < B1;
    const int buf = j & 1;
    double2 kd[TB == 64 ? NPAIR : 1];
    float4 kf[TB != 64 ? NQUAD : 1];
    float kt[TB != 64 && TAIL > 0 ? TAIL : 1];
    lymph_hv8 kr[TB == 48 ? (NQUAD + 1) / 2 : 1];
    float krt[TB == 48 && TAIL > 0 ? TAIL : 1];
    if (on) {
      if constexpr (TB == 64) {
        const double* Kb = static_cast<const double*>(Kv) + (size_t)bj * D::BS;
#pragma unroll
        for (int c2i = 0; c2i < NPAIR; ++c2i) kd[c2i] = load_stream<NT>(Kb + ((size_t)c2i * N3 + r) * 2);
      } else {
        const float* Kb = static_cast<const float*>(Kv) + (size_t)bj * Dims32<P>::BS;
#pragma unroll
        for (int q = 0; q < NQUAD; ++q) kf[q] = load_stream<NT>(Kb + ((size_t)q * N3 + r) * 4);
        if constexpr (TAIL > 0) load_tail<NT>(Kb + (size_t)4 * NQUAD * N3 + (size_t)r * TAIL, kt);
        if constexpr (TB == 48) {
          const _Float16* Rb = Kr + (size_t)bj * Dims16<P>::BS;
#pragma unroll
          for (int kk = 0; kk < (NQUAD + 1) / 2; ++kk) {
            if (2 * kk + 1 < NQUAD) {
              kr[kk] = load_stream_h8<NT>(Rb + ((size_t)kk * N3 + r) * 8);
            } else {  // the last quad of an odd count: 4 values per row
              const lymph_hv4 h = load_stream_h4<NT>(Rb + Dims16<P>::HALF0 + (size_t)r * 4);
              kr[kk] = lymph_hv8{h.x, h.y, h.z, h.w, 0, 0, 0, 0};
            }
          }
          if constexpr (TAIL > 0) {
#pragma unroll
            for (int jj = 0; jj < TAIL; ++jj) krt[jj] = (float)Rb[Dims16<P>::TAIL0 + (size_t)r * TAIL + jj];
          }
        }
      }
      sx[buf][sub][r] = xn;
      if (bj + G < B1) xn = u[(size_t)col[bj + G] * N3 + r];
    }
    lsync<WPW>();
    if (on) {
      double s = 0.0;
      if constexpr (TB == 64) {
#pragma unroll
        for (int c2i = 0; c2i < NPAIR; ++c2i) {
          const bool odd_tail = (N3 % 2 == 1) && (c2i == NPAIR - 1);
          s = s + kd[c2i].x * sx[buf][sub][2 * c2i];
          if (!odd_tail) s = s + kd[c2i].y * sx[buf][sub][2 * c2i + 1];
        }
      } else if constexpr (TB == 48) {  // k_leapfrog48's chains
        double sd = 0.0;
        float sc = 0.0f;
#pragma unroll
        for (int q = 0; q < NQUAD; ++q) {
          double xq[4];
#pragma unroll
          for (int jj = 0; jj < 4; ++jj) xq[jj] = sx[buf][sub][4 * q + jj];
          const lymph_hv8 t8 = kr[q >> 1];
          const int o4 = (q & 1) * 4;
          sd = fma((double)kf[q].x, xq[0], sd);
          sd = fma((double)kf[q].y, xq[1], sd);
          sd = fma((double)kf[q].z, xq[2], sd);
          sd = fma((double)kf[q].w, xq[3], sd);
          sc = fmaf(kf[q].x * (float)t8[o4 + 0], (float)xq[0], sc);
          sc = fmaf(kf[q].y * (float)t8[o4 + 1], (float)xq[1], sc);
          sc = fmaf(kf[q].z * (float)t8[o4 + 2], (float)xq[2], sc);
          sc = fmaf(kf[q].w * (float)t8[o4 + 3], (float)xq[3], sc);
        }
        if constexpr (TAIL > 0) {
#pragma unroll
          for (int jj = 0; jj < TAIL; ++jj) {
            const double xt = sx[buf][sub][4 * NQUAD + jj];
            sd = fma((double)kt[jj], xt, sd);
            sc = fmaf(kt[jj] * krt[jj], (float)xt, sc);
          }
        }
        s = sd + (double)sc * 0x1p-24;
      } else {
        float sf = 0.0f;
#pragma unroll
        for (int q = 0; q < NQUAD; ++q) {
          float xq[4];
#pragma unroll
          for (int jj = 0; jj < 4; ++jj) xq[jj] = (float)sx[buf][sub][4 * q + jj];
          sf = sf + kf[q].x * xq[0];
          sf = sf + kf[q].y * xq[1];
          sf = sf + kf[q].z * xq[2];
          sf = sf + kf[q].w * xq[3];
        }
        if constexpr (TAIL > 0) {
#pragma unroll
          for (int jj = 0; jj < TAIL; ++jj) sf = sf + kt[jj] * (float)sx[buf][sub][4 * NQUAD + jj];
        }
        s = (double)sf;
      }
      prod[(size_t)(bj - B0) * N3 + r] = s;
    }
  }
  lsync<WPW>();
  double acc = 0.0;
  if (act) {  // this row's blocks, in block order
    const int a0 = row_ptr[Pp] - B0, a1 = row_ptr[Pp + 1] - B0;
    acc = prod[(size_t)a0 * N3 + r];
    for (int k = a0 + 1; k < a1; ++k) acc = acc + prod[(size_t)k * N3 + r];
  }
  const size_t o = (size_t)Pp * N3 + r;
  if (MODE == 2) {
    if (act) sw[sub][r] = acc;
    lsync<WPW>();
    if (act && r == 0) {
      double el = 0.0;
      for (int k = 0; k < N3; ++k) el = el + u[(size_t)Pp * N3 + k] * sw[sub][k];
      out[Pp] = el;
    }
    return;
  }
  double w = 0.0;
  if (act) {
    const double gp = gsel ? gtab[gsel[Pp]] : g;
    w = -acc + rs[o] + rd[o] * gp;
  }
  if constexpr (TB == 64) {
    lsync<WPW>();  // sR
    const double* R = sR[act ? sub : 0];
    w = solve_group<NP>(R, Divisor(act ? R[pk_off(NP, r % NP)] : 1.0), w, sub * N3, r, act);
  }
  if (act) {
    if (MODE == 0)
      out[o] = c1 * w + 2.0 * u[o] - wa[o];
    else
      out[o] = c1 * w + u[o] + c2 * wa[o];
  }
}

// ---------------------------------------------------------------------------
// FP32-apply variant of the step: the operator blocks, taken to the
// mass-orthonormal basis in FP64 (k_ortho_operator below), are held in FP32 in
// "column-quad" order (entry (r, c) at ((c>>2)*N3 + r)*4 + (c&3); a lane
// reads four columns of its row as one 16-byte load, half the bytes of the
// FP64 stream); products and the per-block sum are FP32; the sum over blocks,
// the RHS, the basis transforms and the update stay FP64.
// ---------------------------------------------------------------------------

// ---------------------------------------------------------------------------
// 32-bit apply in the mass-orthonormal basis.  With M_P = R_P^T R_P per
// polyhedron, the variables ~u = R u turn the leapfrog step into
//   ~u^{n+1} = 2 ~u^n - ~u^{n-1} + dt^2 (~F - ~K ~u^n),
//   ~K_PQ = R_P^-T K_PQ R_Q^-1,   ~F = R^-T F,
// the same iteration with M^-1 turned into the identity.  ~K is scaled like
// M^-1 K whatever the conditioning of the bounding-box Legendre basis on the
// polyhedron, so rounding it to FP32 perturbs the iteration by FP32 rounding
// relative to itself.  Rounding K in the original basis perturbs M^-1 K by
// that rounding times cond(M_P) -- up to 2e8 at p = 4 on agglomerates of
// 4-40 tets, enough to make the iteration diverge.  The 32-bit step also
// needs no triangular solves.
// ---------------------------------------------------------------------------

// S = R^-1 (upper triangular, packed like R), one thread per (polyhedron, column)
template <int P>
__global__ void k_inv_upper(const double* __restrict__ RM, double* __restrict__ S, int n_poly) {
  using D = Dims<P>;
  constexpr int NP = D::NP;
  const int id = blockIdx.x * blockDim.x + threadIdx.x;
  if (id >= n_poly * NP) return;
  const int Pp = id / NP, j = id % NP;
  const double* R = RM + (size_t)Pp * D::NPK;
  double* Sp = S + (size_t)Pp * D::NPK;
  double x[NP];  // column j of R^-1: R x = e_j, x[i] = 0 for i > j
#pragma unroll
  for (int i = 0; i < NP; ++i) x[i] = 0.0;
  for (int i = j; i >= 0; --i) {
    double s = (i == j) ? 1.0 : 0.0;
    for (int k = i + 1; k <= j; ++k) s = s - R[pk_off(NP, i) + (k - i)] * x[k];
    x[i] = s / R[pk_off(NP, i)];
  }
  for (int i = 0; i <= j; ++i) Sp[pk_off(NP, i) + (j - i)] = x[i];
}

// The 48-bit apply keeps an operator entry k as its FP32 rounding hi and a
// 16-bit correction t = (k - hi) / hi * 2^24 (|t| <= 1 since hi is k
// rounded to nearest; FP16 keeps 11 significant bits of it), so that
// hi (1 + t 2^-24) carries about 35 bits: a relative error of 2^-36 where
// the FP32 rounding leaves 2^-25.
__device__ __forceinline__ _Float16 split_residual(double k, float hi) {
  if (hi == 0.0f) return (_Float16)0.0f;
  return (_Float16)(float)((k - (double)hi) / (double)hi * 0x1p24);
}

// ~K_PQ = S_P^T K_PQ S_Q rounded to FP32 in the column-quad layout; one
// workgroup per block, one component strip (Np rows) at a time:
// T = X S_Q (per column component), Z = S_P^T T.
template <int P>
__global__ __launch_bounds__(256) void k_ortho_operator(const double* __restrict__ K,
                                                        const double* __restrict__ S,
                                                        const int* __restrict__ blk_row,
                                                        const int* __restrict__ col,
                                                        float* __restrict__ K32,
                                                        _Float16* __restrict__ K16, size_t b0) {
  using D = Dims<P>;
  constexpr int NP = D::NP, N3 = D::N3, NPK = D::NPK;
  __shared__ double SP[NPK], SQ[NPK];
  __shared__ double X[NP * N3], T[NP * N3];
  const int tid = threadIdx.x;
  const size_t b = b0 + blockIdx.x;
  const int Pp = blk_row[b], Q = col[b];
  for (int k = tid; k < NPK; k += blockDim.x) {
    SP[k] = S[(size_t)Pp * NPK + k];
    SQ[k] = S[(size_t)Q * NPK + k];
  }
  const double* Kb = K + b * D::BS;
  float* Ob = K32 + b * Dims32<P>::BS;
  _Float16* Rb = K16 ? K16 + b * Dims16<P>::BS : nullptr;  // unused slots zeroed by the host
  for (int i = 0; i < 3; ++i) {
    __syncthreads();
    for (int e = tid; e < NP * N3; e += blockDim.x) {
      const int r = e / N3, c = e % N3;
      X[e] = Kb[kpos(N3, i * NP + r, c)];
    }
    __syncthreads();
    for (int e = tid; e < NP * N3; e += blockDim.x) {  // T = X S_Q, S_Q upper
      const int r = e / N3, c = e % N3, j = c / NP, cc = c % NP;
      double s = 0.0;
      for (int k = 0; k <= cc; ++k) s = s + X[r * N3 + j * NP + k] * SQ[pk_off(NP, k) + (cc - k)];
      T[e] = s;
    }
    __syncthreads();
    for (int e = tid; e < NP * N3; e += blockDim.x) {  // Z = S_P^T T
      const int r = e / N3, c = e % N3;
      double s = 0.0;
      for (int k = 0; k <= r; ++k) s = s + SP[pk_off(NP, k) + (r - k)] * T[k * N3 + c];
      const float hi = (float)s;
      const size_t o = kpos32(N3, i * NP + r, c);
      Ob[o] = hi;
      if (Rb) Rb[kpos16(N3, i * NP + r, c)] = split_residual(s, hi);
    }
  }
  // the floats that round the block stride up to a multiple of 4
  constexpr int PAD = (int)(Dims32<P>::BS - (size_t)N3 * N3);
  if constexpr (PAD > 0)
    if (tid < PAD) Ob[(size_t)N3 * N3 + tid] = 0.0f;
}

// Mass-orthonormal transforms with one wave per polyhedron, lane i on row i
// of all three components: MODE 0 ~u = R u (row i sums R_ik x_k over k >= i
// in ascending k, x_k broadcast from lane k); MODE 2 ~F = R^-T F (forward
// substitution swept by columns: y_j = s_j / R_jj from lane j, then every row
// below subtracts R_ji y_j, so row i subtracts in ascending k as a serial
// loop would).  `list` (n entries) restricts the transform to the listed
// polyhedra; null = the first n.
template <int P, int MODE>
__global__ __launch_bounds__(64) void k_tilde(const double* __restrict__ RM,
                                              const double* __restrict__ in,
                                              double* __restrict__ out,
                                              const int* __restrict__ list, int n) {
  using D = Dims<P>;
  constexpr int NP = D::NP;
  static_assert(NP <= 64, "one lane per row");
  static_assert(MODE == 0 || MODE == 2, "mode 1 is k_tilde_back");
  const int w = blockIdx.x;
  if (w >= n) return;
  const int Pp = list ? list[w] : w;
  const int i = threadIdx.x;
  const bool row = i < NP;
  const double* R = RM + (size_t)Pp * D::NPK;
  const double* x = in + (size_t)Pp * D::N3;
  double* y = out + (size_t)Pp * D::N3;
  double x0 = 0.0, x1 = 0.0, x2 = 0.0;
  if (row) {
    x0 = x[i];
    x1 = x[NP + i];
    x2 = x[2 * NP + i];
  }
  if constexpr (MODE == 0) {
    const int ri = row ? pk_off(NP, i) : 0;
    double s0 = 0.0, s1 = 0.0, s2 = 0.0;
#pragma unroll
    for (int k = 0; k < NP; ++k) {
      const double a0 = __shfl(x0, k, 64), a1 = __shfl(x1, k, 64), a2 = __shfl(x2, k, 64);
      if (row && i <= k) {
        const double r = R[ri + (k - i)];
        s0 = s0 + r * a0;
        s1 = s1 + r * a1;
        s2 = s2 + r * a2;
      }
    }
    if (row) {
      y[i] = s0;
      y[NP + i] = s1;
      y[2 * NP + i] = s2;
    }
  } else {
#pragma unroll
    for (int j = 0; j < NP; ++j) {
      const int rj = pk_off(NP, j);
      const double rjj = R[rj];
      const double y0 = __shfl(x0, j, 64) / rjj;
      const double y1 = __shfl(x1, j, 64) / rjj;
      const double y2 = __shfl(x2, j, 64) / rjj;
      if (i == j) {
        y[i] = y0;
        y[NP + i] = y1;
        y[2 * NP + i] = y2;
      } else if (row && i > j) {
        const double r = R[rj + (i - j)];
        x0 = x0 - r * y0;
        x1 = x1 - r * y1;
        x2 = x2 - r * y2;
      }
    }
  }
}

// u = R^-1 ~u (mode 1 of the transforms above) with one wave per polyhedron:
// back_rows, the factor staged in LDS in one trip (read from memory column by
// column, with divisions on the chain, 64 polyhedra took 16 us at p = 4, now 8).
template <int P>
__global__ __launch_bounds__(64) void k_tilde_back(const double* __restrict__ RM,
                                                   const double* __restrict__ in,
                                                   double* __restrict__ out,
                                                   const int* __restrict__ list, int n) {
  using D = Dims<P>;
  constexpr int NP = D::NP;
  __shared__ double sR[D::NPK + 1];  // the factor and a zero
  const int w = blockIdx.x;
  if (w >= n) return;
  const int Pp = list ? list[w] : w;
  const int i = threadIdx.x;
  const bool row = i < NP;
  const double* R = RM + (size_t)Pp * D::NPK;
  const Divisor d(R[pk_off(NP, row ? i : 0)]);
  for (int k = i; k <= D::NPK; k += 64) sR[k] = k < D::NPK ? R[k] : 0.0;
  double x[3];
#pragma unroll
  for (int c = 0; c < 3; ++c) x[c] = row ? in[(size_t)Pp * D::N3 + c * NP + i] : 0.0;
  wave_lds_sync();
  back_rows<NP>(sR, d, x, i);
  if (row)
#pragma unroll
    for (int c = 0; c < 3; ++c) out[(size_t)Pp * D::N3 + c * NP + i] = x[c];
}

template <int P, int MODE, int UNR, int WPP, bool NT>
__global__ __launch_bounds__(64 * WPP) void k_leapfrog32(const float* __restrict__ K,
                                                   const int* __restrict__ row_ptr,
                                                   const int* __restrict__ col,
                                                   const double* __restrict__ Rp,
                                                   const double* __restrict__ rs,
                                                   const double* __restrict__ rd,
                                                   const double* __restrict__ u,
                                                   const double* __restrict__ wa,
                                                   double* __restrict__ out, double g, double c1,
                                                   double c2, const int* __restrict__ gsel,
                                                   const double* __restrict__ gtab, int n_poly,
    const int* __restrict__ order) {
  // all vectors in the mass-orthonormal basis (K is ~K); Rp is unused
  using D = Dims<P>;
  constexpr int N3 = D::N3, NQUAD = Dims32<P>::NQ, TAIL = Dims32<P>::T;
  constexpr int RPL = (N3 + 63) / 64;
  extern __shared__ double sblk[];  // WPP > 1: per-block products [block][row]
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int Pp = step_poly(order);
  if (Pp >= n_poly) return;  // padding workgroups of the last XCD share
  double acc[RPL];
#pragma unroll
  for (int k = 0; k < RPL; ++k) acc[k] = 0.0;
  StepEnds<N3, RPL> ends;
  if constexpr (WPP > 1)
    if (wv == 0) ends.load(rs, rd, u, wa, (size_t)Pp * N3, lane);
  const int b0 = row_ptr[Pp], b1 = row_ptr[Pp + 1];
  for (int b = b0 + wv; b < b1; b += WPP) {
    const int cb = __builtin_amdgcn_readfirstlane(col[b]);
    const double* __restrict__ xv = u + (size_t)cb * N3;
    const float* __restrict__ Kb = K + (size_t)b * Dims32<P>::BS;
    float xl[RPL];
#pragma unroll
    for (int k = 0; k < RPL; ++k) {
      const int r = lane + 64 * k;
      xl[k] = r < N3 ? (float)xv[r] : 0.0f;
    }
    float s[RPL];
#pragma unroll
    for (int k = 0; k < RPL; ++k) s[k] = 0.0f;
#pragma unroll 1
    for (int q0 = 0; q0 < NQUAD; q0 += UNR) {
      float4 kv[UNR][RPL];
#pragma unroll
      for (int uu = 0; uu < UNR; ++uu) {
        const int q = q0 + uu;
#pragma unroll
        for (int k = 0; k < RPL; ++k) {
          const int r = lane + 64 * k;
          if ((NQUAD % UNR == 0 || q < NQUAD) && r < N3)
            kv[uu][k] = load_stream<NT>(Kb + ((size_t)q * N3 + r) * 4);
        }
      }
#pragma unroll
      for (int uu = 0; uu < UNR; ++uu) {
        const int q = q0 + uu;
        if (NQUAD % UNR == 0 || q < NQUAD) {
          float xq[4];
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const int c = 4 * q + j;
            const float src = (RPL > 1 && (c >> 6)) ? xl[RPL - 1] : xl[0];
            xq[j] = (c < N3) ? __int_as_float(__builtin_amdgcn_readlane(__float_as_int(src), c & 63))
                             : 0.0f;
          }
#pragma unroll
          for (int k = 0; k < RPL; ++k) {
            const int r = lane + 64 * k;
            if (r < N3) {
              s[k] = s[k] + kv[uu][k].x * xq[0];
              s[k] = s[k] + kv[uu][k].y * xq[1];
              s[k] = s[k] + kv[uu][k].z * xq[2];
              s[k] = s[k] + kv[uu][k].w * xq[3];
            }
          }
        }
      }
    }
    if constexpr (TAIL > 0) {  // last N3 % 4 columns, stored row by row
      constexpr int C0 = 4 * NQUAD;
      float xt[TAIL];
#pragma unroll
      for (int j = 0; j < TAIL; ++j) {
        const int c = C0 + j;
        const float src = (RPL > 1 && (c >> 6)) ? xl[RPL - 1] : xl[0];
        xt[j] = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(src), c & 63));
      }
#pragma unroll
      for (int k = 0; k < RPL; ++k) {
        const int r = lane + 64 * k;
        if (r < N3) {
          float kt[TAIL];
          load_tail<NT>(Kb + (size_t)C0 * N3 + (size_t)r * TAIL, kt);
#pragma unroll
          for (int j = 0; j < TAIL; ++j) s[k] = s[k] + kt[j] * xt[j];
        }
      }
    }
    if constexpr (WPP == 1) {
#pragma unroll
      for (int k = 0; k < RPL; ++k) acc[k] = (b == b0) ? (double)s[k] : acc[k] + (double)s[k];
    } else {
#pragma unroll
      for (int k = 0; k < RPL; ++k) {
        const int r = lane + 64 * k;
        if (r < N3) sblk[(size_t)(b - b0) * N3 + r] = (double)s[k];
      }
    }
  }
  if constexpr (WPP > 1) {
    __syncthreads();
    if (wv != 0) return;  // no barrier follows in this kernel
#pragma unroll
    for (int k = 0; k < RPL; ++k) {
      const int r = lane + 64 * k;
      if (r < N3) {
        double a = sblk[r];
#pragma unroll 4
        for (int j = 1; j < b1 - b0; ++j) a = a + sblk[(size_t)j * N3 + r];
        acc[k] = a;
      }
    }
  }
  const size_t o = (size_t)Pp * N3;
  if constexpr (WPP == 1) ends.load(rs, rd, u, wa, o, lane);
  // time factor: one scalar, or per source group (ensembles whose instances
  // carry their own wavelet; the table is filled for this step)
  const double gp = gsel ? gtab[gsel[Pp]] : g;
#pragma unroll
  for (int k = 0; k < RPL; ++k) {
    const int r = lane + 64 * k;
    if (r < N3) {
      const double w = -acc[k] + ends.s[k] + ends.d[k] * gp;
      if (MODE == 0)
        out[o + r] = c1 * w + 2.0 * ends.u[k] - ends.a[k];
      else
        out[o + r] = c1 * w + ends.u[k] + c2 * ends.a[k];
    }
  }
}

// The 48-bit apply: k_leapfrog32's walk over ~K (mass-orthonormal basis, no
// solves) with each entry hi (1 + t 2^-24) (split_residual): hi x summed in
// FP64 fused multiply-adds from the FP64 coefficients, the correction
// (hi t) x in FP32 and scaled by 2^-24 once per block, then the block
// products added in block order in FP64 and k_leapfrog32's update.  6 bytes
// per operator entry; the state stays within about 1e-9 of the FP64 step's
// over 1000 steps where the 32-bit apply drifts to 1e-5.

template <int P, int MODE, int UNR, int WPP, bool NT>
__global__ __launch_bounds__(64 * WPP) void k_leapfrog48(const float* __restrict__ K,
                                                   const _Float16* __restrict__ Kr,
                                                   const int* __restrict__ row_ptr,
                                                   const int* __restrict__ col,
                                                   const double* __restrict__ rs,
                                                   const double* __restrict__ rd,
                                                   const double* __restrict__ u,
                                                   const double* __restrict__ wa,
                                                   double* __restrict__ out, double g, double c1,
                                                   double c2, const int* __restrict__ gsel,
                                                   const double* __restrict__ gtab, int n_poly,
                                                   const int* __restrict__ order) {
  using D = Dims<P>;
  constexpr int N3 = D::N3, NQUAD = Dims32<P>::NQ, TAIL = Dims32<P>::T;
  constexpr int RPL = (N3 + 63) / 64;
  static_assert(UNR % 2 == 0, "whole quad pairs per load group");
  extern __shared__ double sblk[];  // WPP > 1: per-block products [block][row]
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int Pp = step_poly(order);
  if (Pp >= n_poly) return;  // padding workgroups of the last XCD share
  double acc[RPL];
#pragma unroll
  for (int k = 0; k < RPL; ++k) acc[k] = 0.0;
  StepEnds<N3, RPL> ends;
  if constexpr (WPP > 1)
    if (wv == 0) ends.load(rs, rd, u, wa, (size_t)Pp * N3, lane);
  const int b0 = row_ptr[Pp], b1 = row_ptr[Pp + 1];
  for (int b = b0 + wv; b < b1; b += WPP) {
    const int cb = __builtin_amdgcn_readfirstlane(col[b]);
    const double* __restrict__ xv = u + (size_t)cb * N3;
    const float* __restrict__ Kb = K + (size_t)b * Dims32<P>::BS;
    const _Float16* __restrict__ Rb = Kr + (size_t)b * Dims16<P>::BS;
    double xl[RPL];
#pragma unroll
    for (int k = 0; k < RPL; ++k) {
      const int r = lane + 64 * k;
      xl[k] = r < N3 ? xv[r] : 0.0;
    }
    double s[RPL];
    float sc[RPL];
#pragma unroll
    for (int k = 0; k < RPL; ++k) {
      s[k] = 0.0;
      sc[k] = 0.0f;
    }
#pragma unroll 1
    for (int q0 = 0; q0 < NQUAD; q0 += UNR) {  // UNR even: whole quad pairs
      float4 kv[UNR][RPL];
      lymph_hv8 tv[UNR / 2][RPL];
#pragma unroll
      for (int uu = 0; uu < UNR; ++uu) {
        const int q = q0 + uu;
#pragma unroll
        for (int k = 0; k < RPL; ++k) {
          const int r = lane + 64 * k;
          if (q < NQUAD && r < N3) {
            kv[uu][k] = load_stream<NT>(Kb + ((size_t)q * N3 + r) * 4);
            if ((uu & 1) == 0) {
              if (q + 1 < NQUAD) {
                tv[uu / 2][k] = load_stream_h8<NT>(Rb + ((size_t)(q >> 1) * N3 + r) * 8);
              } else {  // the last quad of an odd count: 4 values per row
                const lymph_hv4 h = load_stream_h4<NT>(Rb + Dims16<P>::HALF0 + (size_t)r * 4);
                tv[uu / 2][k] = lymph_hv8{h.x, h.y, h.z, h.w, 0, 0, 0, 0};
              }
            }
          }
        }
      }
#pragma unroll
      for (int uu = 0; uu < UNR; ++uu) {
        const int q = q0 + uu;
        if (q < NQUAD) {
          double xq[4];
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const int c = 4 * q + j;
            const double src = (RPL > 1 && (c >> 6)) ? xl[RPL - 1] : xl[0];
            xq[j] = (c < N3) ? lane_bcast(src, c & 63) : 0.0;
          }
#pragma unroll
          for (int k = 0; k < RPL; ++k) {
            const int r = lane + 64 * k;
            if (r < N3) {
              const float4 h = kv[uu][k];
              const lymph_hv8 t8 = tv[uu / 2][k];
              const int o4 = (uu & 1) * 4;
              s[k] = fma((double)h.x, xq[0], s[k]);
              s[k] = fma((double)h.y, xq[1], s[k]);
              s[k] = fma((double)h.z, xq[2], s[k]);
              s[k] = fma((double)h.w, xq[3], s[k]);
              sc[k] = fmaf(h.x * (float)t8[o4 + 0], (float)xq[0], sc[k]);
              sc[k] = fmaf(h.y * (float)t8[o4 + 1], (float)xq[1], sc[k]);
              sc[k] = fmaf(h.z * (float)t8[o4 + 2], (float)xq[2], sc[k]);
              sc[k] = fmaf(h.w * (float)t8[o4 + 3], (float)xq[3], sc[k]);
            }
          }
        }
      }
    }
    if constexpr (TAIL > 0) {  // last N3 % 4 columns, stored row by row
      constexpr int C0 = 4 * NQUAD;
#pragma unroll
      for (int k = 0; k < RPL; ++k) {
        const int r = lane + 64 * k;
#pragma unroll
        for (int j = 0; j < TAIL; ++j) {
          const int c = C0 + j;
          const double src = (RPL > 1 && (c >> 6)) ? xl[RPL - 1] : xl[0];
          const double xt = lane_bcast(src, c & 63);
          if (r < N3) {
            const float h = Kb[(size_t)C0 * N3 + (size_t)r * TAIL + j];
            const float t = (float)Rb[Dims16<P>::TAIL0 + (size_t)r * TAIL + j];
            s[k] = fma((double)h, xt, s[k]);
            sc[k] = fmaf(h * t, (float)xt, sc[k]);
          }
        }
      }
    }
#pragma unroll
    for (int k = 0; k < RPL; ++k) s[k] = s[k] + (double)sc[k] * 0x1p-24;
    if constexpr (WPP == 1) {
#pragma unroll
      for (int k = 0; k < RPL; ++k) acc[k] = (b == b0) ? s[k] : acc[k] + s[k];
    } else {
#pragma unroll
      for (int k = 0; k < RPL; ++k) {
        const int r = lane + 64 * k;
        if (r < N3) sblk[(size_t)(b - b0) * N3 + r] = s[k];
      }
    }
  }
  if constexpr (WPP > 1) {
    __syncthreads();
    if (wv != 0) return;  // no barrier follows in this kernel
#pragma unroll
    for (int k = 0; k < RPL; ++k) {
      const int r = lane + 64 * k;
      if (r < N3) {
        double a = sblk[r];
#pragma unroll 4
        for (int j = 1; j < b1 - b0; ++j) a = a + sblk[(size_t)j * N3 + r];
        acc[k] = a;
      }
    }
  }
  const size_t o = (size_t)Pp * N3;
  if constexpr (WPP == 1) ends.load(rs, rd, u, wa, o, lane);
  const double gp = gsel ? gtab[gsel[Pp]] : g;
#pragma unroll
  for (int k = 0; k < RPL; ++k) {
    const int r = lane + 64 * k;
    if (r < N3) {
      const double w = -acc[k] + ends.s[k] + ends.d[k] * gp;
      if (MODE == 0)
        out[o + r] = c1 * w + 2.0 * ends.u[k] - ends.a[k];
      else
        out[o + r] = c1 * w + ends.u[k] + c2 * ends.a[k];
    }
  }
}

// The pairs-once step of the 48-bit apply: k_sym_products32's walk over the
// stored list and its packed self blocks, with k_leapfrog48's arithmetic
// (hi x in FP64 fused multiply-adds, (hi t) x in FP32, joined with the 2^-24
// scale per block), products stored as doubles (prod_stride(3Np) per block)
// and summed by k_sym_update32<P, MODE, double>.  Here the row chain of each
// chunk runs first and writes the chunk's hi and hi t to LDS as it forms
// them; the chunk's columns then run their chains over ascending rows with
// u_P[r], the chain Q's own row runs over block (Q, P), so a pair block's
// products are the full rows' bit for bit where the two stored blocks round
// alike.  A self block's product is its upper triangle's row chain (diagonal
// included) plus its strict upper triangle's column chain: the full row's
// terms in another order, which moves its FP64 sum by rounding only.  p = 3
// (3Np = 60: whole quads per chunk, no tail columns).
template <int P>
__global__ __launch_bounds__(64) void k_sym_products48(const float* __restrict__ Ks,
                                                       const _Float16* __restrict__ Kr,
                                                       const int* __restrict__ row_ptr,
                                                       const int* __restrict__ col,
                                                       const int* __restrict__ sidx,
                                                       const int* __restrict__ tdst,
                                                       const double* __restrict__ u,
                                                       double* __restrict__ prod,
                                                       double* __restrict__ rowp, int n_poly,
                                                       const int* __restrict__ order) {
  constexpr int N3 = Dims32<P>::N3, NQ = Dims32<P>::NQ, NPR = Dims16<P>::NPR;
  constexpr int PS = prod_stride(N3);
  static_assert(N3 <= 64 && N3 % 12 == 0 && Dims32<P>::T == 0, "one lane per row, whole quads per chunk");
  static_assert(self32_off(NQ) <= (int)Dims32<P>::BS, "packed self block fits its slot");
  static_assert(self16_off(N3, NPR) <= (int)Dims16<P>::BS, "packed self corrections fit their slot");
  constexpr int CW = N3 / 3, CQ = CW / 4;
  // one chunk's hi and hi t row by row (lanes past the rows write padding
  // rows): 16-byte writes, and a column read over 20 lanes hits 20 banks
  __shared__ __align__(16) float sH[64 * CW], sC[64 * CW];
  __shared__ __align__(16) double sU[N3];  // u_P, read by the column chains
  __shared__ __align__(16) double sX[64];  // u_Q of the current block, read by the row chains
  const int lane = threadIdx.x;
  const bool row = lane < N3;
  const int rl = row ? lane : N3 - 1;  // lanes past the rows load the last row's (cached) lines
  const int Pp = step_poly(order);
  if (Pp >= n_poly) return;  // padding workgroups of the last XCD share
  const int b0 = row_ptr[Pp], b1 = row_ptr[Pp + 1];
  const int lcb = lane < b1 - b0 ? col[b0 + lane] : 0;
  const int lsi = lane < b1 - b0 ? sidx[b0 + lane] : 0;
  const int ltd = lane < b1 - b0 ? tdst[b0 + lane] : 0;
  if (row) sU[lane] = u[(size_t)Pp * N3 + lane];  // ordered before its reads by the chunks' syncs
  double racc = 0.0;  // the row products of this wave's stored blocks, in block order
  for (int b = b0; b < b1; ++b) {
    const int j = b - b0;
    const int si = j < 64 ? __builtin_amdgcn_readlane(lsi, j) : __builtin_amdgcn_readfirstlane(sidx[b]);
    if (si < 0) continue;  // written by the neighbour's wave
    const int cb = j < 64 ? __builtin_amdgcn_readlane(lcb, j) : __builtin_amdgcn_readfirstlane(col[b]);
    const int td = j < 64 ? __builtin_amdgcn_readlane(ltd, j) : __builtin_amdgcn_readfirstlane(tdst[b]);
    const float* __restrict__ Kb = Ks + (size_t)si * Dims32<P>::BS;
    const _Float16* __restrict__ Rb = Kr + (size_t)si * Dims16<P>::BS;
    const double xl = u[(size_t)cb * N3 + rl];
    const bool pair = cb != Pp;
    // the self blocks' row clamps and masks are formed per block: hoisted
    // out of the loop they would hold 60 masks in scalar registers
    int rb = rl;
    asm volatile("" : "+v"(rb));
    // one load path for both kinds (an address select per load), so that the
    // chunks wait on their own loads only
    float4 kq[NQ];
    lymph_hv8 tq[NPR];
#pragma unroll
    for (int q = 0; q < NQ; ++q)
      kq[q] = load_stream(Kb + (pair ? (q * N3 + rb) * 4 : self32_off(q) + 4 * (rb < 4 * q + 3 ? rb : 4 * q + 3)));
#pragma unroll
    for (int k = 0; k < NPR; ++k) {
      const int last = self16_rows(N3, k) - 1;
      const int self_at = self16_off(N3, k) + self16_w(N3, k) * (rb < last ? rb : last);
      if (2 * k + 1 < NQ) {
        tq[k] = load_stream_h8(Rb + (pair ? (k * N3 + rb) * 8 : self_at));
      } else {  // the last quad of an odd count: 4 values per row
        const lymph_hv4 h = load_stream_h4(Rb + (pair ? (int)Dims16<P>::HALF0 + rb * 4 : self_at));
        tq[k] = lymph_hv8{h.x, h.y, h.z, h.w, 0, 0, 0, 0};
      }
    }
    if (!pair) {  // the upper triangle's rows only
#pragma unroll
      for (int q = 0; q < NQ; ++q) {
        if (4 * q + 0 < rb) kq[q].x = 0.0f;
        if (4 * q + 1 < rb) kq[q].y = 0.0f;
        if (4 * q + 2 < rb) kq[q].z = 0.0f;
        if (4 * q + 3 < rb) kq[q].w = 0.0f;
      }
    }
    // three chunks of CW columns: the row chain continues over the chunk's
    // quads, each entry's hi and hi t going to LDS as they are formed, then
    // the chunk's columns run their chains
    wave_lds_sync();  // the previous block's reads of sX are done
    sX[lane] = xl;  // lanes past the rows write padding
    wave_lds_sync();
    double s = 0.0, st = 0.0;
    float sc = 0.0f;
#pragma unroll
    for (int h = 0; h < 3; ++h) {
      wave_lds_sync();  // the previous chunk's reads are done
#pragma unroll
      for (int k = 0; k < CQ; ++k) {
        const int q = h * CQ + k;
        const double2 xa = *reinterpret_cast<const double2*>(sX + 4 * q);  // broadcasts
        const double2 xb = *reinterpret_cast<const double2*>(sX + 4 * q + 2);
        const double xq[4] = {xa.x, xa.y, xb.x, xb.y};
        const float hv[4] = {kq[q].x, kq[q].y, kq[q].z, kq[q].w};
        const lymph_hv8 t8 = tq[q >> 1];
        const int o4 = (q & 1) * 4;
        float hc[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          hc[j] = hv[j] * (float)t8[o4 + j];
          s = fma((double)hv[j], xq[j], s);
          sc = fmaf(hc[j], (float)xq[j], sc);
        }
        *reinterpret_cast<float4*>(sH + lane * CW + 4 * k) = kq[q];
        *reinterpret_cast<float4*>(sC + lane * CW + 4 * k) = make_float4(hc[0], hc[1], hc[2], hc[3]);
      }
      // the chunk's row chain is complete here: otherwise the compiler defers
      // it past the column chains and keeps every broadcast u_Q live
      asm volatile("" : "+v"(s), "+v"(sc));
      // a self block's diagonal belongs to its rows only (a wave's LDS
      // writes land in program order)
      if (!pair && lane >= h * CW && lane < (h + 1) * CW) {
        sH[lane * CW + (lane - h * CW)] = 0.0f;
        sC[lane * CW + (lane - h * CW)] = 0.0f;
      }
      wave_lds_sync();
      if (lane >= h * CW && lane < (h + 1) * CW) {  // column's chain over ascending rows
        const float* __restrict__ hp = sH + (lane - h * CW);
        const float* __restrict__ cp = sC + (lane - h * CW);
        double v = 0.0;
        float vc = 0.0f;
#pragma unroll
        for (int r = 0; r < N3; ++r) {
          const double ur = sU[r];  // the same address in every lane: a broadcast
          v = fma((double)hp[r * CW], ur, v);
          vc = fmaf(cp[r * CW], (float)ur, vc);
        }
        st = v + (double)vc * 0x1p-24;
      }
    }
    s = s + (double)sc * 0x1p-24;
    if (!pair) s = s + st;  // the strict upper triangle's transposed product
    asm volatile("" : "+v"(s));  // as in k_sym_products32
    racc = racc + s;
    if (pair && lane < PS) prod[(size_t)td * PS + lane] = row ? st : 0.0;
  }
  if (lane < PS) rowp[(size_t)Pp * PS + lane] = row ? racc : 0.0;  // zeros past the rows
}

// L2 error terms du_i^T M_modal du_i per (polyhedron, component)
// (COMPUTE_ERROR_L2_MATRIX_FREE, src/matrix_free.f90:1406-1416).
template <int P>
__global__ void k_l2_terms(const double* __restrict__ Mm, const double* __restrict__ uh,
                           const double* __restrict__ ue, double* __restrict__ part, int n_poly) {
  using D = Dims<P>;
  constexpr int NP = D::NP;
  const int id = blockIdx.x * blockDim.x + threadIdx.x;
  if (id >= 3 * n_poly) return;
  const int Pp = id / 3, i = id % 3;
  const size_t o = (size_t)Pp * D::N3 + i * NP;
  double du[NP];
  for (int mm = 0; mm < NP; ++mm) du[mm] = uh[o + mm] - ue[o + mm];
  const double* A = Mm + (size_t)Pp * NP * NP;
  double el = 0.0;
  for (int mm = 0; mm < NP; ++mm) {
    double s = 0.0;
    for (int nn = 0; nn < NP; ++nn) s = s + A[mm * NP + nn] * du[nn];
    el = el + du[mm] * s;
  }
  part[id] = el;
}

// Sum of n error terms by one workgroup in a fixed order: thread t adds terms
// t, t + 1024, ... eight at a time, then a tree over the threads.  (One thread
// adding them one after the other, as the reference's element loop does, took
// 3.3 ms on average for 28,606 and 85,818 terms; this 9.4 us.)
__global__ __launch_bounds__(1024) void k_sum_terms(const double* __restrict__ part, int n, double* __restrict__ out) {
  __shared__ double red[1024];
  double s = 0.0;
#pragma unroll 8
  for (int i = threadIdx.x; i < n; i += 1024) s = s + part[i];
  red[threadIdx.x] = s;
  __syncthreads();
  for (int w = 512; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) red[threadIdx.x] = red[threadIdx.x] + red[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) out[0] = red[0];
}

__global__ void k_sub(const double* __restrict__ a, const double* __restrict__ b,
                      double* __restrict__ c, size_t n) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) c[i] = a[i] - b[i];
}

// flag[0] = 1 if some a[i] is NaN or infinite (flag cleared by k_set_int
// first; every writer stores the same value, so no atomics are needed)
__global__ void k_set_int(int* __restrict__ flag, int v) { flag[0] = v; }
__global__ void k_nonfinite(const double* __restrict__ a, size_t n, int* __restrict__ flag) {
  bool bad = false;
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (size_t)gridDim.x * blockDim.x)
    bad |= !isfinite(a[i]);
  if (__any(bad) && bad) flag[0] = 1;
}

__global__ void k_scale(double* __restrict__ a, double g, size_t n) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) a[i] = 0.0 * 0.0 + a[i] * g;
}

// poly-major u[P*N3 + d]  <->  reference column-major u(npoly, N3): u[d*npoly + P]
__global__ void k_to_poly(const double* __restrict__ f, double* __restrict__ p, int n_poly, int n3) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < (size_t)n_poly * n3) {
    const int P = (int)(i / n3), d = (int)(i % n3);
    p[i] = f[(size_t)d * n_poly + P];
  }
}
__global__ void k_to_fortran(const double* __restrict__ p, double* __restrict__ f, int n_poly, int n3) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < (size_t)n_poly * n3) {
    const int d = (int)(i / n_poly), P = (int)(i % n_poly);
    f[i] = p[(size_t)P * n3 + d];
  }
}

// Receivers: value of the modal field at a point, sum_i u_i Lx Ly Lz on the
// polyhedron's bounding box, as EXPORT_SOLUTION evaluates it
// (src/solution_processing.f90:150-170); out[r*3 + comp] of record row `row`.
// One wave per receiver, a basis function per lane, the terms added in the
// functions' order: 64 receivers at p = 4 take 5 us, with a thread per
// component 14.  Beyond kSampleWaves receivers the threads fill the chip
// (k_sample_many, the same bits): wave / thread us, p = 1 and 4, 2,000 receivers
// 5.3 / 5.6 and 8.6 / 16.8, 8,000 10.1 / 7.1 and 17.1 / 17.2, 100,000 52 / 10 and
// 141 / 54.
constexpr int kSampleWaves = 4096;
template <int P>
__global__ __launch_bounds__(64) void k_sample(const double* __restrict__ u, const int* __restrict__ rpoly,
                         const double* __restrict__ rxyz, const double* __restrict__ bbox,
                         const int* __restrict__ blist, int n, double* __restrict__ out) {
  using D = Dims<P>;
  constexpr int NP = D::NP;
  const int r = blockIdx.x, i = threadIdx.x;
  if (r >= n) return;
  const int Pp = rpoly[r];
  const double* bb = bbox + (size_t)Pp * 6;
  const int f = i < NP ? i : 0;
  double v[3];
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    const double hb = (bb[2 * d + 1] - bb[2 * d]) / 2.0, mb = (bb[2 * d + 1] + bb[2 * d]) / 2.0;
    v[d] = leg(blist[f * 3 + d], (rxyz[r * 3 + d] - mb) / hb) / sqrt(hb);
  }
  double t[3], s[3] = {0.0, 0.0, 0.0};
#pragma unroll
  for (int c = 0; c < 3; ++c) t[c] = u[(size_t)Pp * D::N3 + c * NP + f] * v[0] * v[1] * v[2];
#pragma unroll
  for (int j = 0; j < NP; ++j)
#pragma unroll
    for (int c = 0; c < 3; ++c) s[c] = s[c] + lane_bcast(t[c], j);
  if (i < 3) out[r * 3 + i] = i == 0 ? s[0] : (i == 1 ? s[1] : s[2]);
}

template <int P>
__global__ void k_sample_many(const double* __restrict__ u, const int* __restrict__ rpoly,
                              const double* __restrict__ rxyz, const double* __restrict__ bbox,
                              const int* __restrict__ blist, int n, double* __restrict__ out) {
  using D = Dims<P>;
  constexpr int NP = D::NP;
  const int id = blockIdx.x * blockDim.x + threadIdx.x;
  if (id >= 3 * n) return;
  const int r = id / 3, comp = id % 3;
  const int Pp = rpoly[r];
  const double* bb = bbox + (size_t)Pp * 6;
  double xp[3], sq[3];
  for (int d = 0; d < 3; ++d) {
    const double hb = (bb[2 * d + 1] - bb[2 * d]) / 2.0, mb = (bb[2 * d + 1] + bb[2 * d]) / 2.0;
    xp[d] = (rxyz[(size_t)r * 3 + d] - mb) / hb;
    sq[d] = sqrt(hb);
  }
  const double* uu = u + (size_t)Pp * D::N3 + comp * NP;
  double s = 0.0;
  for (int i = 0; i < NP; ++i) {
    const double vx = leg(blist[i * 3 + 0], xp[0]) / sq[0];
    const double vy = leg(blist[i * 3 + 1], xp[1]) / sq[1];
    const double vz = leg(blist[i * 3 + 2], xp[2]) / sq[2];
    s = s + uu[i] * vx * vy * vz;
  }
  out[id] = s;
}

// Point forces: rhs[P_k][i*Np+m] += f_k,i phi_m(x_k), sources applied in order
// (one workgroup, a barrier between sources so two sources in one
// polyhedron accumulate in order).
template <int P>
__global__ __launch_bounds__(128) void k_point_sources(const double* __restrict__ sxyz,
                                                       const int* __restrict__ spoly,
                                                       const double* __restrict__ sf, int n,
                                                       const double* __restrict__ bbox,
                                                       const int* __restrict__ blist,
                                                       double* __restrict__ rhs,
                                                       const int* __restrict__ tet_poly) {
  using D = Dims<P>;
  constexpr int NP = D::NP, N3 = D::N3;
  for (int k = 0; k < n; ++k) {
    // spoly holds polyhedra, or tets when their polyhedron map is given
    const int Pp = tet_poly ? tet_poly[spoly[k]] : spoly[k];
    const double* bb = bbox + (size_t)Pp * 6;
    for (int e = threadIdx.x; e < N3; e += blockDim.x) {
      const int i = e / NP, m = e % NP;
      double v[3];
      for (int d = 0; d < 3; ++d) {
        const double hb = (bb[2 * d + 1] - bb[2 * d]) / 2.0, mb = (bb[2 * d + 1] + bb[2 * d]) / 2.0;
        v[d] = leg(blist[m * 3 + d], (sxyz[k * 3 + d] - mb) / hb) / sqrt(hb);
      }
      const size_t o = (size_t)Pp * N3 + e;
      rhs[o] = rhs[o] + sf[k * 3 + i] * v[0] * v[1] * v[2];
    }
    __syncthreads();
  }
}


// Double-couple sources, the SISM branch of MAKE_RHS_FREE
// (src/matrix_free.f90:600-664): for source k in order, in tet stet[k] of
// polyhedron P, the moment density M = ((s n^T + n s^T) M0) / V with V =
// |det4| / 6 of the tet (moment_density, src/problem_data_and_properties.f90:
// 317-335; volume, src/find_tet.f90:184-210), and MAKE_DOUBLE_COUPLE
// (src/assemble_element.f90:116-167): couple[i*Np+m] = sum_q (w_q |J|)
// sum_j M_ij d_j phi_m(x_q) over the tet's quadrature points with P's basis,
// then rhs[P] += couple.  One workgroup, thread = entry (i, m), sources in
// order so that sources sharing a polyhedron add as the reference adds them.
__device__ inline double det4_rows(const double* v) {  // rows (x_r, y_r, z_r, 1)
#define A_(i, j) ((j) == 4 ? 1.0 : v[((i) - 1) * 3 + ((j) - 1)])
  return A_(1, 1) * (A_(2, 2) * (A_(3, 3) * A_(4, 4) - A_(3, 4) * A_(4, 3)) -
                     A_(2, 3) * (A_(3, 2) * A_(4, 4) - A_(3, 4) * A_(4, 2)) +
                     A_(2, 4) * (A_(3, 2) * A_(4, 3) - A_(3, 3) * A_(4, 2))) -
         A_(1, 2) * (A_(2, 1) * (A_(3, 3) * A_(4, 4) - A_(3, 4) * A_(4, 3)) -
                     A_(2, 3) * (A_(3, 1) * A_(4, 4) - A_(3, 4) * A_(4, 1)) +
                     A_(2, 4) * (A_(3, 1) * A_(4, 3) - A_(3, 3) * A_(4, 1))) +
         A_(1, 3) * (A_(2, 1) * (A_(3, 2) * A_(4, 4) - A_(3, 4) * A_(4, 2)) -
                     A_(2, 2) * (A_(3, 1) * A_(4, 4) - A_(3, 4) * A_(4, 1)) +
                     A_(2, 4) * (A_(3, 1) * A_(4, 2) - A_(3, 2) * A_(4, 1))) -
         A_(1, 4) * (A_(2, 1) * (A_(3, 2) * A_(4, 3) - A_(3, 3) * A_(4, 2)) -
                     A_(2, 2) * (A_(3, 1) * A_(4, 3) - A_(3, 3) * A_(4, 1)) +
                     A_(2, 3) * (A_(3, 1) * A_(4, 2) - A_(3, 2) * A_(4, 1)));
#undef A_
}

template <int P>
__global__ __launch_bounds__(128) void k_double_couples(MeshDev m, const int* __restrict__ stet,
                                                        const double* __restrict__ strike,
                                                        const double* __restrict__ normal,
                                                        const double* __restrict__ m0, int n,
                                                        double* __restrict__ rhs) {
  using D = Dims<P>;
  constexpr int NP = D::NP, N3 = D::N3, NQ3 = D::NQ3;
  __shared__ double spt[NQ3 * 3];
  __shared__ int sbl[NP * 3];
  const int tid = threadIdx.x;
  for (int i = tid; i < NP * 3; i += blockDim.x) sbl[i] = m.blist[i];
  for (int k = 0; k < n; ++k) {
    const int t = stet[k];
    const int Pp = m.tet_poly[t];
    double v[12], Fk[12], Jdet;
    for (int i = 0; i < 12; ++i) v[i] = m.tet_xyz[(size_t)t * 12 + i];
    affine_map(v, Fk, Jdet);
    const double vol = fabs(det4_rows(v)) / 6.0;
    double mom[9];
    for (int i = 0; i < 3; ++i)
      for (int j = 0; j < 3; ++j)
        mom[i * 3 + j] = ((strike[3 * k + i] * normal[3 * k + j] + strike[3 * k + j] * normal[3 * k + i]) *
                          m0[k]) / vol;
    __syncthreads();  // the previous source's points are no longer read
    for (int q = tid; q < NQ3; q += blockDim.x) map_point(Fk, &m.qtet[q * 4], &spt[q * 3]);
    __syncthreads();
    double bb[6];
    for (int d = 0; d < 6; ++d) bb[d] = m.bbox[(size_t)Pp * 6 + d];
    for (int e = tid; e < N3; e += blockDim.x) {
      const int i = e / NP, mm = e % NP;
      double acc = 0.0;
      for (int q = 0; q < NQ3; ++q) {
        double ph, g[3];
        basis_at(&sbl[mm * 3], bb, &spt[q * 3], ph, g[0], g[1], g[2]);
        double reduct = 0.0;
        for (int j = 0; j < 3; ++j) reduct = reduct + mom[i * 3 + j] * g[j];
        acc = acc + m.wtet[q] * fabs(Jdet) * reduct;
      }
      const size_t o = (size_t)Pp * N3 + e;
      rhs[o] = rhs[o] + acc;
    }
  }
}

// Per-group Ricker time factors of one step: gtab[i] = ricker(f0[i], t0[i], t).
__global__ void k_ricker_table(const double* __restrict__ f0, const double* __restrict__ t0,
                               int n, double t, double* __restrict__ gtab) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) gtab[i] = ricker(f0[i], t0[i], t);
}

}  // namespace lymph
