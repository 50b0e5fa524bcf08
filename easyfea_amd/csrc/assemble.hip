// Elastic stiffness assembled row by row: the CSR values straight from the
// mesh, without the element matrices in between.
//
// Writing every element matrix and gathering its entries into their slots
// moves the matrix several times (64^3 HEXA8: 1.2 GB of element entries
// written, then read back one 8-byte gather at a time through 0.6 GB of
// indices, for 0.52 GB of values; 422 + 661 us, and 1.2 GB of memory).  Here a
// group of lanes owns a node and walks its elements in increasing order; lane j
// of the group adds the element's DIM x DIM block of (the node, the element's
// node j) to the row's slots in LDS, where a wave's nodes are laid out as in the
// CSR array, so that the end is one contiguous store.  The element's geometry is
// computed once per node of it (8 times for HEXA8): lane p of the group forms
// sqrt(w |det|) J^-1 of point p and the gradient of the node's own function, and
//   S = sum_p (sqrt(w |det|) grad N_a) (sqrt(w |det|) grad N_b)^T
// gives the block of any law constant in the element:
//   isotropic   K_ij = lam S_ij + mu S_ji + mu d_ij tr S
//   general     K_ij = sum_kl C_ikjl S_kl
// One wave per block (nothing to synchronise), entries summed in increasing
// element order (deterministic).  Bound: latency.  The rows (15.5 KB for 8
// HEXA8 nodes) and the registers (reference gradients held, 250) leave 7 waves
// on a CU, 1.75 per SIMD, for steps that pass through LDS twice, a division
// and a root; FP64 issue is 180 us of the 64^3 HEXA8 mesh's 490 (1083 with
// element matrices), its 0.52 GB store 60 us at the chip's copy rate.  Reference
// gradients in LDS were 10 us slower, recomputing the node's own gradient in
// every lane 55 us, the Lame constants' divisions in the steps 5 us.
//
// Replaces Operators.Bilinear.LinearizedElasticity (FEM/Operators/
// Bilinear.py:62-79) followed by _Simu.__Assemble_csr (Simulations/
// _simu.py:1051-1055).
#include "efea_common.h"

namespace efea {

// The plan of the assembly by rows, from the scatter map: the entries that a
// node's own (diagonal) slot sums are its incidences, elements increasing.
__device__ inline int place(const int* __restrict__ cols, int p0, int p1, int j) {
  int lo = p0, hi = p1 - 1;  // j is in the row
  while (lo < hi) {
    const int mid = (lo + hi) / 2;
    if (cols[mid] < j) lo = mid + 1; else hi = mid;
  }
  return lo - p0;
}
__device__ inline int64_t own_slot(const int* __restrict__ node_ptr, const int* __restrict__ node_cols, int dn, int n) {
  const int p0 = node_ptr[n], p1 = node_ptr[n + 1];
  return (int64_t)dn * dn * p0 + (p1 > p0 ? dn * place(node_cols, p0, p1, n) : 0);
}

// counts[n + 1]: the node's incidences (counts[0] = 0).
__global__ void __launch_bounds__(256) k_row_counts(int Nn, int dn, const int* __restrict__ node_ptr,
                                                    const int* __restrict__ node_cols, const int* __restrict__ seg,
                                                    int* __restrict__ counts) {
  const int n = blockIdx.x * 256 + threadIdx.x;
  if (n == 0) counts[0] = 0;
  if (n >= Nn) return;
  const int64_t s = own_slot(node_ptr, node_cols, dn, n);
  counts[n + 1] = node_ptr[n + 1] > node_ptr[n] ? seg[s + 1] - seg[s] : 0;
}

// A wave per node, a lane per (incidence, element node).  repeated (may be null):
// set where an element names a node twice.
__global__ void __launch_bounds__(64) k_row_plan(int dn, int nPe, const int* __restrict__ node_ptr,
                                                 const int* __restrict__ node_cols, const int* __restrict__ seg,
                                                 const int* __restrict__ perm, const int* __restrict__ connect,
                                                 const int* __restrict__ inc_ptr, int* __restrict__ inc,
                                                 unsigned short* __restrict__ pos, int* __restrict__ repeated) {
  const int n = blockIdx.x, nd = nPe * dn;
  const int p0 = node_ptr[n], p1 = node_ptr[n + 1], i0 = inc_ptr[n], num = inc_ptr[n + 1] - i0;
  if (num <= 0) return;
  const int first = seg[own_slot(node_ptr, node_cols, dn, n)];
  for (int q = threadIdx.x; q < num * nPe; q += 64) {
    const int k = q / nPe, lj = q % nPe, entry = perm[first + k];
    const int e = entry / (nd * nd), li = entry % (nd * nd) / nd / dn;
    if (lj == 0) {
      inc[i0 + k] = e * 16 + li;
      if (repeated && entry % nd / dn != li) *repeated = 1;
    }
    pos[(int64_t)(i0 + k) * nPe + lj] = (unsigned short)place(node_cols, p0, p1, connect[(int64_t)e * nPe + lj]);
  }
}

int row_counts(int Nn, int dof_n, const int* node_ptr, const int* node_cols, const int* seg, int* counts,
               hipStream_t s) {
  hipLaunchKernelGGL(k_row_counts, dim3((unsigned)((Nn + 255) / 256)), dim3(256), 0, s, Nn, dof_n, node_ptr, node_cols,
                     seg, counts);
  return check_launch("row_counts");
}

int row_plan(int Nn, int dof_n, int nPe, const int* node_ptr, const int* node_cols, const int* seg, const int* perm,
             const int* connect, const int* inc_ptr, int* inc, unsigned short* pos, int* repeated, hipStream_t s) {
  hipLaunchKernelGGL(k_row_plan, dim3((unsigned)Nn), dim3(64), 0, s, dof_n, nPe, node_ptr, node_cols, seg, perm,
                     connect, inc_ptr, inc, pos, repeated);
  return check_launch("row_plan");
}

// LDS a block may use for its rows (the groups' arrays, 0.9 to 6.2 KB, come on
// top): three blocks on a CU, two of HEXA8.  Longer rows than this allows (HEXA8:
// 85 nodes, TETRA10: 170) go through element matrices.
constexpr size_t ASM_ROWS_MAX = 48 * 1024;

struct AsmMesh {
  int Nn;
  const int* node_ptr;
  const int* inc_ptr;            // elements of each node ...
  const int* inc;                // ... element * 16 + the node's number in it, elements increasing
  const unsigned short* pos;     // (incidence, element node): place in the node's row
  const int* connect;
  const double* coord;
  const double* tab;
};

struct AsmLaw {
  const double* E;
  int E_stride;
  double lam1, mu1;  // Lame constants of E = 1
  double thickness;
  const double* D;  // Kelvin-Mandel 6 x 6 (general law)
  int D_stride;
};

// The LDS operations of a wave complete in order; this keeps the compiler from
// moving them past each other.
__device__ inline void wave_order() { asm volatile("" ::: "memory"); }

template <int ET, int NPG, bool GENERAL>
__global__ void __launch_bounds__(64) k_assemble(AsmMesh M, AsmLaw L, double* __restrict__ values) {
  constexpr int NPE = Elem<ET>::NPE, DIM = Elem<ET>::DIM, DD = DIM * DIM;
  constexpr int GL = NPE <= 4 ? 4 : (NPE <= 8 ? 8 : 16), NG = 64 / GL;
  using TB = Tab<NPG, NPE, DIM>;
  // per group the coordinates, then (once they are read) the points' Jacobians
  // and gradients; an odd stride keeps the groups off each other's banks
  constexpr int PG = DD + DIM, GS = (NPG > 1 && NPG * PG > NPE * DIM ? NPG * PG : NPE * DIM) | 1;
  __shared__ double sX[NG][GS];
  extern __shared__ double rows[];
  const int lane = threadIdx.x, grp = lane / GL, j = lane % GL, jn = j < NPE ? j : 0;
  const int n0 = blockIdx.x * NG, n = n0 + grp;
  const bool have = n < M.Nn;
  const int nn = have ? n : M.Nn - 1;
  const int r0 = M.node_ptr[n0], r1 = M.node_ptr[n0 + NG < M.Nn ? n0 + NG : M.Nn];
  const int p0 = M.node_ptr[nn], cnt = M.node_ptr[nn + 1] - p0;
  const int k0 = M.inc_ptr[nn], num = have ? M.inc_ptr[nn + 1] - k0 : 0;
  const int total = DD * (r1 - r0);
  for (int i = lane; i < total; i += 64) rows[i] = 0.0;
  double* mine = rows + DD * (p0 - r0);
  wave_order();
  // reference gradients: of node j at every point, of every node at point j
  const int jp = j < NPG ? j : 0;
  auto ref = [&](int p, int a, int d) { return M.tab[TB::DN + (p * DIM + d) * NPE + a]; };
  double dNb[NPG][DIM], dNp[NPE][DIM];
#pragma unroll
  for (int d = 0; d < DIM; ++d) {
#pragma unroll
    for (int p = 0; p < NPG; ++p) dNb[p][d] = ref(p, jn, d);
#pragma unroll
    for (int a = 0; a < NPE; ++a) dNp[a][d] = ref(jp, a, d);
  }
  const double wp = M.tab[TB::W + jp];
  // the element of step k, the coordinates of its node j: loaded ahead, index
  // by index, so that a step's three dependent loads are behind it
  auto code = [&](int k) { return num > 0 ? M.inc[k0 + (k < num ? k : num - 1)] : 0; };
  auto node = [&](int c) { return num > 0 ? M.connect[(int64_t)(c >> 4) * NPE + jn] : nn; };
  int c0 = code(0), c1 = code(1), c2 = code(2);
  int m1 = node(c1);
  double X[DIM], X1[DIM];
  {
    const int m0 = node(c0);
#pragma unroll
    for (int d = 0; d < DIM; ++d) X[d] = M.coord[(int64_t)m0 * 3 + d];
  }
  for (int k = 0; __any(k < num); ++k) {
#pragma unroll
    for (int d = 0; d < DIM; ++d) X1[d] = M.coord[(int64_t)m1 * 3 + d];
    const int m2 = node(c2), c3 = code(k + 3);
    const int64_t e = c0 >> 4;
    double dNa[DIM];
#pragma unroll
    for (int d = 0; d < DIM; ++d) dNa[d] = ref(jp, c0 & 15, d);
    const int kk = k < num ? k : 0;
    const int at = num > 0 ? M.pos[(int64_t)(k0 + kk) * NPE + jn] : 0;
    double E = 0;
    if constexpr (!GENERAL) E = L.E[L.E_stride ? e : 0];
    if (j < NPE) {
#pragma unroll
      for (int d = 0; d < DIM; ++d) sX[grp][j * DIM + d] = X[d];
    }
    wave_order();
    // sqrt(w |det|) J^-1 at point j (one point: J^-1 in every lane, w |det| apart)
    // and the scaled gradient of this node's function there
    double inv[DD], ga[DIM], w = 0;
    if (NPG == 1 || j < NPG) {
      double F[DIM][DIM];
#pragma unroll
      for (int i = 0; i < DD; ++i) F[i / DIM][i % DIM] = 0;
#pragma unroll
      for (int a = 0; a < NPE; ++a)
#pragma unroll
        for (int d = 0; d < DIM; ++d)
#pragma unroll
          for (int c = 0; c < DIM; ++c) F[d][c] += dNp[a][d] * sX[grp][a * DIM + c];
      double det;
      if constexpr (DIM == 2) {
        det = F[0][0] * F[1][1] - F[1][0] * F[0][1];
        inv[0] = F[1][1];
        inv[1] = -F[0][1];
        inv[2] = -F[1][0];
        inv[3] = F[0][0];
      } else {
        inv[0] = F[1][1] * F[2][2] - F[1][2] * F[2][1];
        inv[1] = F[0][2] * F[2][1] - F[0][1] * F[2][2];
        inv[2] = F[0][1] * F[1][2] - F[0][2] * F[1][1];
        inv[3] = F[1][2] * F[2][0] - F[1][0] * F[2][2];
        inv[4] = F[0][0] * F[2][2] - F[0][2] * F[2][0];
        inv[5] = F[0][2] * F[1][0] - F[0][0] * F[1][2];
        inv[6] = F[1][0] * F[2][1] - F[1][1] * F[2][0];
        inv[7] = F[0][1] * F[2][0] - F[0][0] * F[2][1];
        inv[8] = F[0][0] * F[1][1] - F[0][1] * F[1][0];
        det = F[0][0] * inv[0] + F[0][1] * inv[3] + F[0][2] * inv[6];
      }
      w = fabs(det) * wp;
      const double s = (NPG == 1 ? 1.0 : sqrt(w)) / det;
#pragma unroll
      for (int i = 0; i < DD; ++i) inv[i] *= s;
#pragma unroll
      for (int i = 0; i < DIM; ++i) {
        ga[i] = 0;
#pragma unroll
        for (int d = 0; d < DIM; ++d) ga[i] += inv[i * DIM + d] * dNa[d];
      }
      wave_order();
      if constexpr (NPG > 1) {
#pragma unroll
        for (int i = 0; i < DD; ++i) sX[grp][j * PG + i] = inv[i];
#pragma unroll
        for (int i = 0; i < DIM; ++i) sX[grp][j * PG + DD + i] = ga[i];
      }
    }
    wave_order();
    double S[DIM][DIM];
#pragma unroll
    for (int i = 0; i < DD; ++i) S[i / DIM][i % DIM] = 0;
#pragma unroll
    for (int p = 0; p < NPG; ++p) {
      double J[DD], gb[DIM];
#pragma unroll
      for (int i = 0; i < DD; ++i) J[i] = NPG == 1 ? inv[i] : sX[grp][p * PG + i];
      if constexpr (NPG > 1) {
#pragma unroll
        for (int i = 0; i < DIM; ++i) ga[i] = sX[grp][p * PG + DD + i];
      }
#pragma unroll
      for (int i = 0; i < DIM; ++i) {
        gb[i] = 0;
#pragma unroll
        for (int d = 0; d < DIM; ++d) gb[i] += J[i * DIM + d] * dNb[p][d];
      }
#pragma unroll
      for (int i = 0; i < DIM; ++i)
#pragma unroll
        for (int c = 0; c < DIM; ++c) S[i][c] += ga[i] * gb[c];
    }
    const double scale = (NPG == 1 ? w : 1.0) * (DIM == 2 ? L.thickness : 1.0);
    double K[DIM][DIM];
    if constexpr (GENERAL) {
      // rows and columns of D: xx yy zz yz xz xy; the shear rows of B carry 1/sqrt(2)
      const double* __restrict__ D = L.D + (L.D_stride ? e * 36 : 0);
      constexpr int V[3][3] = {{0, 5, 4}, {5, 1, 3}, {4, 3, 2}};
#pragma unroll
      for (int i = 0; i < DIM; ++i)
#pragma unroll
        for (int c = 0; c < DIM; ++c) {
          double s = 0;
#pragma unroll
          for (int a = 0; a < DIM; ++a)
#pragma unroll
            for (int b = 0; b < DIM; ++b) {
              const int I = V[i][a], J = V[c][b];
              const double f = (I > 2 ? 0.70710678118654752440 : 1.0) * (J > 2 ? 0.70710678118654752440 : 1.0);
              s += (f * D[I * 6 + J]) * S[a][b];
            }
          K[i][c] = s * scale;
        }
    } else {
      const double lam = E * L.lam1, mu = E * L.mu1;
      double tr = 0;
#pragma unroll
      for (int i = 0; i < DIM; ++i) tr += S[i][i];
#pragma unroll
      for (int i = 0; i < DIM; ++i)
#pragma unroll
        for (int c = 0; c < DIM; ++c)
          K[i][c] = scale * (lam * S[i][c] + mu * S[c][i] + (i == c ? mu * tr : 0.0));
    }
    if (k < num && j < NPE) {
#pragma unroll
      for (int i = 0; i < DIM; ++i)
#pragma unroll
        for (int c = 0; c < DIM; ++c) mine[(i * cnt + at) * DIM + c] += K[i][c];
    }
    wave_order();
    c0 = c1;
    c1 = c2;
    c2 = c3;
    m1 = m2;
#pragma unroll
    for (int d = 0; d < DIM; ++d) X[d] = X1[d];
  }
  wave_order();
  double* out = values + (int64_t)DD * r0;
  for (int i = lane; i < total; i += 64) out[i] = rows[i];
}

template <int ET, int NPG, bool GENERAL>
static int assemble_launch(const AsmMesh& M, const AsmLaw& L, int max_neighbours, double* values, hipStream_t s) {
  constexpr int NPE = Elem<ET>::NPE, DIM = Elem<ET>::DIM;
  constexpr int NG = 64 / (NPE <= 4 ? 4 : (NPE <= 8 ? 8 : 16));
  const size_t lds = 8 * (size_t)NG * max_neighbours * DIM * DIM;
  if (lds > ASM_ROWS_MAX) {
    set_error("elastic_assemble: rows of %d neighbours need %zu bytes of LDS, at most %zu", max_neighbours, lds,
              ASM_ROWS_MAX);
    return EFEA_ERR_SIZE;
  }
  hipLaunchKernelGGL((k_assemble<ET, NPG, GENERAL>), dim3((unsigned)((M.Nn + NG - 1) / NG)), dim3(64), lds, s, M, L,
                     values);
  return check_launch("elastic_assemble");
}

int assemble_max_neighbours(int elem_type) {
#define MAXN(ETV)                                                                                        \
  if (elem_type == ETV)                                                                                  \
    return (int)(ASM_ROWS_MAX / (8 * (64 / (Elem<ETV>::NPE <= 4 ? 4 : (Elem<ETV>::NPE <= 8 ? 8 : 16))) * \
                                 Elem<ETV>::DIM * Elem<ETV>::DIM));
  MAXN(ET_TRI3) MAXN(ET_QUAD4) MAXN(ET_HEXA8) MAXN(ET_TETRA4) MAXN(ET_TETRA10)
#undef MAXN
  return 0;
}

int elastic_assemble(int elem_type, int Nn, const int* node_ptr, int max_neighbours, const int* inc_ptr,
                     const int* inc, const unsigned short* pos, const int* connect, const double* coord,
                     const double* tab, int nPg, const double* E, int E_stride, double nu, int plane_stress,
                     double thickness, const double* D, int D_stride, double* values, hipStream_t s) {
  const AsmMesh M{Nn, node_ptr, inc_ptr, inc, pos, connect, coord, tab};
  const bool plane = plane_stress && (elem_type == ET_TRI3 || elem_type == ET_QUAD4);
  const double lam1 = plane ? nu / (1 - nu * nu) : nu / ((1 + nu) * (1 - 2 * nu));
  const AsmLaw L{E, E_stride, lam1, 1 / (2 * (1 + nu)), thickness, D, D_stride};
#define RUN(ETV, NPGV)                                                                               \
  if (elem_type == ETV && nPg == NPGV) {                                                             \
    if constexpr (ETV == ET_HEXA8 || ETV == ET_TETRA10) {                                            \
      if (D) return assemble_launch<ETV, NPGV, true>(M, L, max_neighbours, values, s);               \
    }                                                                                                \
    if (!D) return assemble_launch<ETV, NPGV, false>(M, L, max_neighbours, values, s);               \
  }
  RUN(ET_TRI3, 1)
  RUN(ET_QUAD4, 4)
  RUN(ET_HEXA8, 8)
  RUN(ET_TETRA4, 1)
  RUN(ET_TETRA10, 4)
#undef RUN
  set_error("elastic_assemble: unsupported element %d with %d points%s", elem_type, nPg, D ? " and a general law" : "");
  return EFEA_ERR_ARG;
}

}  // namespace efea
