// Resident PCG: a whole solve in one launch, for systems whose matrix fits the
// chip's registers (256 CUs x 512 KiB).
//
// The launch-per-step solvers pay two launch boundaries (2 to 4 us each) and
// two or three dependent memory round trips per iteration: on the systems
// here (1,000 to 260,000 nodes in 2D, 33,000 in 3D, a million scalar nodes)
// that is most of an iteration.  Here one block per CU keeps its nodes' matrix
// values, mask, block-Jacobi inverse and the vectors x, r, p, s in registers
// and the preconditioned residual u (with the neighbours' values, the halo) in
// LDS for the whole solve.  Per iteration the blocks exchange only u at
// the nodes other blocks read, and one set of partial sums:
//   u = M r                         (own nodes; published where others need it)
//   w = A u                         after the halo has arrived
//   gamma = (r, u), delta = (w, u), (r, r) and, two-level, P^T w
//                                   block sums published, every block adds all
//   beta = gamma / gamma_old, alpha = gamma / (delta - beta gamma / alpha_old)
//   p = u + beta p, s = w + beta s, x += alpha p, r -= alpha s
//   zs = Ac^-1 P^T w + beta zs, z -= alpha zs
//                                   the block's rows of Ac^-1 P^T r, kept as r is
//   u = B^-1 r + P z
// This is Chronopoulos and Gear's form of the preconditioned CG (one reduction
// per iteration): the iterates and the stopping test (Strakos-Tichy delayed
// A-norm estimate, residual test) are the classic solve's.  Unlike the
// pipelined recurrences (pcg2p.hip, pcgp.hip) only s = A p is kept by
// recurrence, and u and w are formed anew, so no residual replacement is
// needed.
//
// Exchange.  CDNA4's XCDs have separate L2 caches, and a device-scope fence
// writes a whole L2 back; so data goes through relaxed agent-scope atomic
// stores and loads (write-through and L2-bypassing), and a value is its own
// flag: the buffers hold the bit pattern EMPTY (a NaN no arithmetic produces)
// until the value arrives, and a reader polls the values themselves.
// Buffers rotate (halo: 2, sums: 3); an owner sets its slots of the next
// buffer back to EMPTY while it publishes the current one, which is safe
// because
//   - everybody has read halo k - 1 when the sums of k - 1 are complete, and
//     an owner's reset of that buffer is waited for before its sums of k go
//     out, without which nobody starts to read halo k + 1;
//   - everybody has read the sums of k - 2 when those of k - 1 are complete,
//     and the reset is waited for before the owner's sums of k go out.
// Every wait is bounded by `wait_ticks` of the 100 MHz clock: a block that
// gives up leaves the kernel (so every other block's waits end too) and marks
// the result failed; the caller redoes the solve with the launch-per-step
// iteration.  The waits need all blocks on the chip at once: a plan has at
// most one block per CU, kernels of other streams only delay the blocks they
// keep out, and the resident solves of a process are queued one after the
// other (each waits for the event of the last one), so that two of them never
// hold half of the chip each.
// (hipLaunchCooperativeKernel gives the same by sending the launch through
// the runtime's transfer queue: 110 to 140 us more per solve in a program that
// had used several streams.)
//
// What bounds it: the two exchanges (a store to memory and a load from it past
// the L2s, about 1 us each way; 2,500 to 3,500 cycles for the halo, 3,000 for
// the sums of 6 blocks, 5,800 of 256), then the block's own chain of LDS reads
// and barriers.  Measured per iteration, the launch-per-step solve before and
// this one: QUAD4 32^2 (6 blocks) 15.9 -> 5.1 us, 360 x 39 (64) 16.5 -> 5.3,
// TRI3 251 x 249 (256) 22 -> 6.6, notched TRI3 200^2 (161) 20 -> 8.0 and its
// scalar system (80) 10.9 -> 4.2, HEXA8 30^3 (236) 42.6 -> 11.7, 31^3 (256)
// 40 -> 12.0, scalar QUAD4 700^2 (240) 28 -> 6.0, 1024^2 (229) 50 -> 12.5;
// block Jacobi on 360 x 39 10.2 -> 4.0.
//
// It replaces the same call as efea_solve_pcg: __Solver_1
// (Simulations/Solvers.py:502-553) with _Solve_Axb's backends
// (Solvers.py:225-394).
#include <mutex>
#include <vector>

#include "coarse_device.h"
#include "resident.h"

namespace efea {

typedef unsigned long long u64;
constexpr u64 EMPTY = ~0ull;
constexpr int RT = 512;           // threads per block: 2 waves per SIMD, 256 registers each
constexpr int RNW = RT / 64;
constexpr int RES_LDS = 160 * 1024 - 512;  // dynamic LDS a block may ask for

__device__ inline u64 ld_agent(const u64* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ inline void st_agent(u64* p, u64 v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ inline void publish(u64* p, double v) {
  u64 b = (u64)__double_as_longlong(v);
  if (b == EMPTY) b = 0x7ff8000000000000ull;  // some other NaN
  st_agent(p, b);
}

// Waits until U published values are there, all loads in flight together.
template <int U>
__device__ inline bool poll(const u64* const (&src)[U], double (&out)[U], u64 wait_ticks) {
  u64 t0 = 0;
  for (int spin = 0;; ++spin) {
    u64 v[U];
#pragma unroll
    for (int i = 0; i < U; ++i) v[i] = ld_agent(src[i]);
    bool miss = false;
#pragma unroll
    for (int i = 0; i < U; ++i) miss |= v[i] == EMPTY;
    if (!miss) {
#pragma unroll
      for (int i = 0; i < U; ++i) out[i] = __longlong_as_double((long long)v[i]);
      return true;
    }
    if ((spin & 15) == 15 || wait_ticks == 0) {
      const u64 now = wall_clock64();
      if (t0 == 0) t0 = now;
      if (now - t0 >= wait_ticks) return false;
    }
  }
}

// Half of a block's waves collect the scalars, the others the restriction:
// thread 256 + c reads entries of source offset | destination <<
// 16 | last << 31 (-1 for none), kept in LDS.  Entries up to a last one belong
// together (the pieces of one component) and are added before they are stored,
// so that a component takes one LDS word however many blocks hold its aggregate.
constexpr int CT = RT / 2;  // threads that collect the restriction
constexpr int RU = 5;         // entries in flight per thread (more would spill)
template <int U>
__device__ inline bool collect(const u64* __restrict__ cur, const int* items, int n, double* __restrict__ to,
                               u64 wait_ticks) {
  double sum = 0;
  for (int i0 = 0; i0 < n; i0 += U) {
    int item[U];
#pragma unroll
    for (int i = 0; i < U; ++i) item[i] = i0 + i < n ? items[(i0 + i) * CT] : -1;
    if (item[0] == -1) break;
    const u64* src[U];
#pragma unroll
    for (int i = 0; i < U; ++i) src[i] = cur + ((item[i] == -1 ? item[0] : item[i]) & 0xffff);
    double o[U];
    if (!poll(src, o, wait_ticks)) return false;
#pragma unroll
    for (int i = 0; i < U; ++i) {
      if (item[i] != -1) sum += o[i];
      if (item[i] < -1) {
        to[(item[i] >> 16) & 0x7fff] = sum;
        sum = 0;
      }
    }
  }
  return true;
}

// This wave's share of the three scalars' sums over the blocks: four lanes per
// block (the fourth reads along), so that a wave's load takes 16 whole lines.
template <int U>
__device__ inline bool collect_scalars(const u64* __restrict__ cur, int line, int nblk, double* __restrict__ to,
                                       u64 wait_ticks) {
  const int lane = threadIdx.x & 63, b0 = (threadIdx.x >> 6) * 16 + (lane >> 2), j = lane & 3;
  const u64* src[U];
#pragma unroll
  for (int i = 0; i < U; ++i) {
    const int b = b0 + 64 * i;
    src[i] = cur + (b < nblk ? b : (b0 < nblk ? b0 : 0)) * line + (j < 3 ? j : 0);
  }
  double o[U], s = 0;
  if (!poll(src, o, wait_ticks)) return false;
#pragma unroll
  for (int i = 0; i < U; ++i) s += b0 + 64 * i < nblk ? o[i] : 0.0;
  s = ror_add<4>(s);
  s = ror_add<8>(s);
  s = swap_add<true>(s, s);
  s = swap_add<false>(s, s);
  if (lane < 3) to[lane] = s;
  return true;
}

template <int DN> struct ResLanes { static constexpr int G = DN == 1 ? 1 : (DN == 2 ? 2 : 4); };
// Neighbour positions kept per lane: a scalar row's first slot is its own
// node, whose position needs no table.
template <int DN, int S> struct ResSlots { static constexpr int N = DN == 1 ? S - 1 : S; };

// A block's published sums: its three scalars and its pieces' restrictions, on
// 64-byte lines of their own (blocks that share a line slow every poll of it:
// 256 blocks' all-to-all took 8,700 cycles with the scalars of all blocks side
// by side, 5,800 with a line per block).
template <int NM, typename Plan>
__host__ __device__ inline int res_line(const Plan& P) {
  return (3 + (P.nagg > 0 ? P.max_pieces * NM : 0) + 7) / 8 * 8;
}

// Columns of the restriction in LDS: whole waves of two per lane, zero-padded.
__host__ __device__ inline int res_columns(int nc) { return (nc + 127) / 128 * 128; }
// Offsets (in doubles) of a block's LDS arrays.
struct ResLds {
  int u, pay, rel, ch, z, zs, rows, item, idx, p, total;
};

template <int DN, bool TWO, typename Plan>
__host__ __device__ inline ResLds res_lds(const Plan& P, int S, int NP, bool BIG, bool cache_rows) {
  constexpr int NM = Modes<DN>::NM, G = ResLanes<DN>::G;
  const int nloc = RT / G * NP, nc = TWO ? res_columns(P.nagg * NM) : 0;
  ResLds L;
  int o = 0;
  L.u = o; o += (nloc + P.max_halo) * DN;
  o += o & 1;
  L.pay = o; o += nc;
  L.rel = o; o += TWO ? nloc * 3 : 0;
  o += o & 1;
  L.ch = o; o += (3 + (TWO ? P.max_pieces * NM : 0)) * RNW * NP;
  L.z = o; o += TWO ? P.max_pieces * NM : 0;
  L.zs = o; o += TWO ? P.max_pieces * NM : 0;
  o += o & 1;
  L.rows = o; o += (TWO && cache_rows) ? P.max_pieces * NM * nc : 0;
  L.item = o; o += TWO ? P.ncollect * CT / 2 : 0;
  L.idx = o; o += BIG ? NP * ((S + 2) / 4) * RT : 0;
  L.p = o; o += BIG ? nloc : 0;
  L.total = o;
  return L;
}

// The plan as a kernel argument.  `gap` decides which arguments share a scalar
// load and so what the compiler keeps in scalar registers.  An iteration of the
// two-level variants with and without it: QUAD4 32^2 5.24 and 5.40 us, 360 x 39
// 5.38 and 5.55, TRI3 251 x 249 6.68 and 6.75, HEXA8 31^3 11.86 and 11.91 (30^3
// 11.73 and 11.52); 8 bytes behind the plan instead: 31^3 12.97.
struct KernelPlan {
  int dof_n, slots, passes, nblk, max_halo, nex, nagg, npiece, max_pieces, ncollect;
  const int* rows;
  const unsigned short* lidx;
  const int *halo_ptr, *halo_ex, *pub, *pub_ptr, *pub_pos, *self, *piece_ptr, *piece_agg;
  const void* gap;
  const int *chunk_piece, *collect;

  explicit KernelPlan(const ResidentPlan& P)
      : dof_n(P.dof_n), slots(P.slots), passes(P.passes), nblk(P.nblk), max_halo(P.max_halo), nex(P.nex),
        nagg(P.nagg), npiece(P.npiece), max_pieces(P.max_pieces), ncollect(P.ncollect), rows(P.rows), lidx(P.lidx),
        halo_ptr(P.halo_ptr), halo_ex(P.halo_ex), pub(P.pub), pub_ptr(P.pub_ptr), pub_pos(P.pub_pos), self(P.self),
        piece_ptr(P.piece_ptr), piece_agg(P.piece_agg), gap(nullptr), chunk_piece(P.chunk_piece),
        collect(P.collect) {}
};

struct ResWork {
  double *r, *u, *p, *s;   // a paused solve's vectors
  double *z, *zs;          // its rows of Ac^-1 P^T r and of the same for s
  double* xp;              // BIG: x in position order
  double* vs;              // BIG: the values of the streamed passes, per block, pass and slot
  u64 *hx, *pay;
  PcgState* st;
};

struct ResArgs {
  const int* node_ptr;
  const double* vals;
  const unsigned char* known;
  const double* Minv;
  const double* b;
  double* x;
  const double* rel;
  const double* Ainv;
  int ld;
  double tolr2, tolA2;
  int limit;       // iterations this launch may add
  int resume;      // continue a paused solve
  int cache_rows;  // the block's rows of Ac^-1 are kept in LDS
  u64 wait_ticks;
  PollBuf* out;    // host-visible result
};

__global__ void __launch_bounds__(256) k_res_empty(int64_t n, u64* __restrict__ a, PollBuf* out) {
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) a[i] = EMPTY;
  if (blockIdx.x == 0 && threadIdx.x == 0) out->failed = 0;
}

// BIG (scalar, most passes): the block's neighbour positions and p live in
// LDS, x in L2 (updated while the halo is on its way), u only in LDS, and B^-1
// is the division by the diagonal.  Of the values at most 72 registers' worth
// stay (9 slots: 4 passes of 9), the other passes are read from the cache in
// every product, laid out for it at the start: with more kept the compiler
// spilled, and a spilled word waits behind the streamed ones.  QUAD4 1024^2
// scalar, 164 iterations: 4 passes kept 10.9 ms for three solves, 6 kept 11.2,
// 7 kept 12.6, all 9 kept (180 words per thread spilled) 25.4; launch-per-step
// 27.7.  It is bound by the product: 13,000 of 33,000 cycles per iteration,
// LDS reads and the latency of the streamed passes.
template <int S, int NP, bool BIG>
struct ResPasses {
  static constexpr int KEPT = !BIG || 2 * S * NP <= 72 ? NP : 72 / (2 * S);
};
template <int DN, int S, int NP, bool TWO, bool BIG>
__global__ void __launch_bounds__(RT, 2)
k_resident(KernelPlan P, ResArgs A, ResWork W) {
  constexpr int NM = Modes<DN>::NM, G = ResLanes<DN>::G, NPC = 64 / G, NLOC = RT / G * NP;
  constexpr int SN = ResSlots<DN, S>::N, S2 = (SN + 1) / 2, NR = BIG ? 1 : NP;
  constexpr int NV = ResPasses<S, NP, BIG>::KEPT;  // passes whose values stay in registers
  static_assert(!BIG || (DN == 1 && !TWO), "BIG is scalar block Jacobi");
  extern __shared__ double lds[];
  __shared__ double ring[RING], lsc[16];  // lsc: sums of the scalars, 4 per collecting wave
  __shared__ int lfail;
  const ResLds L = res_lds<DN, TWO>(P, S, NP, BIG, A.cache_rows != 0);
  double* lu = lds + L.u;
  double* lpay = lds + L.pay;
  double* lrel = lds + L.rel;
  double* lch = lds + L.ch;
  double* lz = lds + L.z;
  double* lzs = lds + L.zs;
  double* lrow = lds + L.rows;
  // BIG: the neighbours' byte offsets in lu, four to a word
  constexpr int SH = (SN + 3) / 4;
  u64* lidx = (u64*)(lds + L.idx);
  double* lp = lds + L.p;

  const int t = threadIdx.x, lane = t & 63, wv = t >> 6, q = lane / G, g = lane % G;
  const int blk = blockIdx.x;
  const int nc = TWO ? P.nagg * NM : 0, nc2 = res_columns(nc), line = res_line<NM>(P);
  const int64_t hstride = (int64_t)P.nex * DN;
  const bool own = g < DN;
  if (t == 0) lfail = 0;
  if (t < RING) ring[t] = 0;
  // the lane's position of pass p
  auto at = [&](int p) { return G == 1 ? p * RT + t : (p * RNW + wv) * NPC + q; };
  // between passes: several passes' loads in flight would spill
  auto fence = [] {
    if constexpr (NP > 1) __builtin_amdgcn_sched_barrier(0);
  };
  // a uniform address, formed anew each time: the loop's own copies of what is
  // added to it would fill the registers
  using Global = __attribute__((address_space(1))) double;
  auto fresh = [](double* a) {
    auto* f = (Global*)a;
    asm volatile("" : "+s"(f));
    return f;
  };

  // ---- the block's nodes, matrix values and neighbour positions
  int node[NR], pubx[NR], piece[NR];
  unsigned li[NR][BIG ? 1 : S2];
  double v[NV][S][DN][DN], Mi[NR][DN], dg[NP - NV + 1];
  double xv[NR], rv[NP], pv[NR], sv[NP], uv[NR];
  unsigned kmask = 0;
#pragma unroll
  for (int p = 0; p < NP; ++p) {
    const int64_t gp = (int64_t)blk * NLOC + at(p);
    const int nd = P.rows[gp];
    const bool have = nd >= 0;
    const int n = have ? nd : 0;
    const int p0 = A.node_ptr[n], cnt = A.node_ptr[n + 1] - p0;
    // a node of no element has an empty row: its loads (dropped) go to the first
    // values, where p0 of a last such node would be past the end
    const int64_t base = (int64_t)DN * DN * (cnt > 0 ? p0 : 0);
    const int self = DN == 1 ? P.self[gp] : 0;
    double* vs = W.vs + ((int64_t)blk * (NP - NV) + (p - NV)) * S * RT + t;  // a streamed pass
    bool diag = false, off = false;  // BIG: not zero
#pragma unroll
    for (int s = 0; s < S; ++s) {
      int j = g + s * G;
      const bool ok = have && j < cnt;
      if constexpr (DN == 1) j = s == 0 ? self : (s - 1 < self ? s - 1 : s);
      const int jj = ok ? j : 0;
#pragma unroll
      for (int a = 0; a < DN; ++a)
#pragma unroll
        for (int b = 0; b < DN; ++b) {
          const double vv = A.vals[base + (int64_t)a * DN * cnt + (int64_t)jj * DN + b];
          if (p < NV) {
            v[p][s][a][b] = ok ? vv : 0.0;
          } else {
            vs[s * RT] = ok ? vv : 0.0;
            if (s == 0) dg[p - NV] = ok ? vv : 0.0;
          }
          if (BIG && ok && vv != 0.0) (s == 0 ? diag : off) = true;
        }
    }
    if constexpr (!BIG) {
#pragma unroll
      for (int s = 0; s < S2; ++s) li[p][s] = 0;
    }
    u64 four = 0;
#pragma unroll
    for (int s = 0; s < SN; ++s) {
      const unsigned i = P.lidx[(((int64_t)blk * NP + p) * SN + s) * RT + t];
      if constexpr (BIG) {
        four |= (u64)(8 * i) << (16 * (s & 3));
        if ((s & 3) == 3 || s == SN - 1) {
          lidx[(p * SH + s / 4) * RT + t] = four;
          four = 0;
        }
      } else {
        li[p][s / 2] |= i << (16 * (s & 1));
      }
    }
    const int64_t i = (int64_t)n * DN + (own ? g : 0);
    const bool act = have && own;
    const bool kn = !act || (A.known && A.known[i]);
    if (kn) kmask |= 1u << p;
    rv[p] = sv[p] = 0.0;
    if constexpr (BIG) {
      // A row of zeros keeps its x, as it does with efea_bj_setup's 1 in place of
      // the zero diagonal.  Where only the diagonal is zero, or b is not, the
      // solve breaks down at once and the classic iteration takes it.
      if (!kn && !diag) {
        kmask |= 1u << p;
        if (off || !(A.b[i] == 0.0)) rv[p] = __longlong_as_double(0x7ff8000000000000ll);
      }
      lp[at(p)] = 0.0;
    } else {
      node[p] = nd;
      pubx[p] = own ? P.pub[gp] : -1;
      piece[p] = TWO ? P.chunk_piece[blk * RNW * NP + p * RNW + wv] : -1;
#pragma unroll
      for (int b = 0; b < DN; ++b) Mi[p][b] = kn ? 0.0 : A.Minv[i * DN + b];  // row g of the node's inverse
      xv[p] = act ? A.x[i] : 0.0;
      pv[p] = uv[p] = 0.0;
    }
    if constexpr (TWO) {
      if (g == 0) {
#pragma unroll
        for (int d = 0; d < 3; ++d) lrel[at(p) * 3 + d] = have ? A.rel[3 * (int64_t)n + d] : 0.0;
      }
    }
    fence();
  }
  const int pc0 = TWO ? P.piece_ptr[blk] : 0, npc = TWO ? P.piece_ptr[blk + 1] - pc0 : 0;
  const int nrow = npc * NM, mine = 3 + nrow;  // rows of Ac^-1, published sums
  for (int i = t; i < (3 + (TWO ? P.max_pieces * NM : 0)) * RNW * NP; i += RT) lch[i] = 0.0;
  if constexpr (TWO) {
    if (A.cache_rows) {
      for (int r = 0; r < nrow; ++r) {
        const double* __restrict__ row = A.Ainv + (int64_t)(P.piece_agg[pc0 + r / NM] * NM + r % NM) * A.ld;
        for (int c = t; c < nc2; c += RT) lrow[r * nc2 + c] = c < nc ? row[c] : 0.0;
      }
    }
    for (int c = nc + t; c < nc2; c += RT) lpay[c] = 0.0;
    for (int r = t; r < nrow; r += RT) {
      lz[r] = A.resume ? W.z[pc0 * NM + r] : 0.0;
      lzs[r] = A.resume ? W.zs[pc0 * NM + r] : 0.0;
    }
  }
  int* litem = (int*)(lds + L.item);
  if constexpr (TWO) {
    for (int i = t; i < P.ncollect * CT; i += RT) litem[i] = P.collect[i];
  }
  const int h0 = P.halo_ptr[blk], nh = (P.halo_ptr[blk + 1] - h0) * DN;
  constexpr int HU = DN == 3 ? 3 : 2;
  int hoff[HU];
#pragma unroll
  for (int i = 0; i < HU; ++i) {
    const int e = t + i * RT;
    hoff[i] = e < nh ? P.halo_ex[h0 + e / DN] * DN + e % DN : 0;
  }
  // BIG: the block's published positions, in exchange order
  const int e0 = BIG ? P.pub_ptr[blk] : 0, ne = BIG ? P.pub_ptr[blk + 1] - e0 : 0;
  int ppos[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) ppos[i] = BIG && t + i * RT < ne ? P.pub_pos[e0 + t + i * RT] : 0;

  // the position in lu of slot s of pass p (after the first, own, slot of a scalar row)
  auto nb = [&](int p, int s) -> int {
    unsigned w = li[p][s / 2];
    asm volatile("" : "+v"(w));  // unpacked here each time: unpacked once, they would fill the registers
    return (int)((w >> (16 * (s & 1))) & 0xffffu);
  };
  // the own values of lu to the other blocks (halo buffer k & 1; the other one
  // and the sums after next are emptied)
  auto put = [&](const double (&val)[NR], int k) {
    u64* cur = W.hx + (k & 1) * hstride;
    u64* nxt = W.hx + ((k + 1) & 1) * hstride;
    if constexpr (BIG) {
      __syncthreads();
      for (int i = t; i < ne; i += RT) {
        const int pp = i == t ? ppos[0] : (i == t + RT ? ppos[1] : P.pub_pos[e0 + i]);
        publish(cur + e0 + i, lu[pp]);
        st_agent(nxt + e0 + i, EMPTY);
      }
    } else {
#pragma unroll
      for (int p = 0; p < NP; ++p) {
        if (own) lu[at(p) * DN + g] = val[p];
        if (pubx[p] >= 0) {
          const int64_t e = (int64_t)pubx[p] * DN + g;
          publish(cur + e, val[p]);
          st_agent(nxt + e, EMPTY);
        }
      }
    }
    if (t < mine) st_agent(W.pay + ((int64_t)((k + 1) % 3) * P.nblk + blk) * line + t, EMPTY);
  };
  auto halo = [&](int k) -> bool {
    const u64* cur = W.hx + (k & 1) * hstride;
    bool ok = true;
    if (t < nh) {
      const u64* src[HU];
#pragma unroll
      for (int i = 0; i < HU; ++i) src[i] = cur + (t + i * RT < nh ? hoff[i] : hoff[0]);
      double o[HU];
      ok = poll(src, o, A.wait_ticks);
#pragma unroll
      for (int i = 0; i < HU; ++i)
        if (ok && t + i * RT < nh) lu[NLOC * DN + t + i * RT] = o[i];
    }
    for (int e = t + HU * RT; e < nh && ok; e += RT) {
      const u64* src[1] = {cur + (int64_t)P.halo_ex[h0 + e / DN] * DN + e % DN};
      double o[1];
      ok = poll(src, o, A.wait_ticks);
      if (ok) lu[NLOC * DN + e] = o[0];
    }
    if (!ok) lfail = 1;
    __syncthreads();
    return lfail == 0;
  };
  // component g of A lu at the lane's node (owner lanes), 0 at known rows
  auto product = [&](double (&y)[NP]) {
    auto pass = [&](int p, const double (&vp)[S][DN][DN]) {
      double sum[DN];
#pragma unroll
      for (int a = 0; a < DN; ++a) sum[a] = 0;
#pragma unroll
      for (int s = 0; s < S; ++s) {
        const double* uu = lu + (DN == 1 ? (s == 0 ? at(p) : nb(p, s - 1)) : nb(p, s) * DN);
        double ub[DN];
#pragma unroll
        for (int b = 0; b < DN; ++b) ub[b] = uu[b];
#pragma unroll
        for (int a = 0; a < DN; ++a)
#pragma unroll
          for (int b = 0; b < DN; ++b) sum[a] += vp[s][a][b] * ub[b];
      }
      double r;
      if constexpr (DN == 1) {
        r = sum[0];
      } else if constexpr (DN == 2) {
        const double other = __shfl_xor(g == 0 ? sum[1] : sum[0], 1, 64);
        r = (g == 0 ? sum[0] : sum[1]) + other;
      } else {
#pragma unroll
        for (int a = 0; a < DN; ++a) {
          sum[a] += __shfl_xor(sum[a], 1, 64);
          sum[a] += __shfl_xor(sum[a], 2, 64);
        }
        r = g == 0 ? sum[0] : (g == 1 ? sum[1] : sum[2]);
      }
      y[p] = ((kmask >> p) & 1u) ? 0.0 : r;
      // formed here: sunk to its first use, past a branch, it would keep every operand live
      asm volatile("" : "+v"(y[p]));
      fence();
    };
    if constexpr (!BIG) {
#pragma unroll
      for (int p = 0; p < NP; ++p) pass(p, v[p]);
    } else {
      // a streamed pass's values are on their way while the passes before it are
      // formed, a pass's offsets while the one before is
      constexpr int NS = NP - NV, ND = NS > 0 ? NS : 1;
      u64 ix[SH];
      auto split = [](int i) { return (i * NV + ND - 1) / ND; };  // kept passes before streamed pass i
      auto offsets = [&](int p, u64 (&w)[SH]) {
#pragma unroll
        for (int h = 0; h < SH; ++h) w[h] = lidx[(p * SH + h) * RT + t];
      };
      auto big = [&](int p, int next, const double (&vp)[S][DN][DN]) {
        double ub[S];
        ub[0] = lu[at(p)];
#pragma unroll
        for (int s = 1; s < S; ++s)
          ub[s] = *(const double*)((const char*)lu + (unsigned)((ix[(s - 1) / 4] >> (16 * ((s - 1) & 3))) & 0xffffu));
        offsets(next, ix);
        fence();
        double sum = 0;
#pragma unroll
        for (int s = 0; s < S; ++s) sum += vp[s][0][0] * ub[s];
        y[p] = ((kmask >> p) & 1u) ? 0.0 : sum;
        asm volatile("" : "+v"(y[p]));  // as above
        fence();
      };
      offsets(0, ix);
#pragma unroll
      for (int i = 0; i < ND; ++i) {
        double w[S][DN][DN];
        if constexpr (NS > 0) {
          const Global* vs = fresh(W.vs + (int64_t)blk * NS * S * RT);
#pragma unroll
          for (int s = 0; s < S; ++s) w[s][0][0] = vs[(unsigned)((i * S + s) * RT + t)];
          fence();
        }
        const int p0 = split(i), p1 = split(i + 1);
#pragma unroll
        for (int p = p0; p < p1; ++p) big(p, NS > 0 && p + 1 == p1 ? NV + i : (p + 1 < NP ? p + 1 : 0), v[p]);
        if constexpr (NS > 0) big(NV + i, i + 1 < NS ? (p1 < split(i + 2) ? p1 : NV + i + 1) : 0, w);
      }
    }
  };
  // block sums of three scalars and of P^T rest per piece, published as sums k,
  // then every block's read into lpay
  auto sums = [&](double s0, double s1, double s2, const double (&rest)[NP], int k, bool read) -> bool {
    // the values' place in wave_sum4's rows
    const int row = lane >> 4, w4 = row == 1 ? 2 : (row == 2 ? 1 : row);
    constexpr int CS = TWO ? RNW * NP : RNW;  // column of lch: a value of each chunk
    if constexpr (TWO) {
#pragma unroll
      for (int p = 0; p < NP; ++p) {
        const double* rn = lrel + at(p) * 3;
        double rc[6];
#pragma unroll
        for (int m = 0; m < NM; ++m) rc[m] = own ? pmode<DN>(rn, g, m) * rest[p] : 0.0;  // rest = 0 at known DOFs
        const double v1 = wave_sum4(rc[0], rc[1], rc[2], NM == 6 ? rc[3] : (p == 0 ? s0 : 0.0));
        const double v2 = NM == 6 ? wave_sum4(rc[4], rc[5], p == 0 ? s0 : 0.0, p == 0 ? s1 : 0.0) : 0.0;
        if ((lane & 15) == 0) {
          double* to = lch + (3 + piece[p] * NM) * CS + p * RNW + wv;  // the other chunks of this column stay 0
          const bool in = piece[p] >= 0;
          if constexpr (NM == 6) {
            if (in) to[w4 * CS] = v1;
            if (w4 < 2) {
              if (in) to[(4 + w4) * CS] = v2;
            } else if (p == 0) {
              lch[(w4 - 2) * CS + wv] = v2;
            }
          } else {
            if (w4 < 3) {
              if (in) to[w4 * CS] = v1;
            } else if (p == 0) {
              lch[wv] = v1;
            }
          }
        }
      }
      if constexpr (NM == 6) {
        const double v = wave_sum4(s2, 0.0, 0.0, 0.0);
        if (lane == 0) lch[2 * CS + wv] = v;
      } else {
        const double v = wave_sum4(s1, s2, 0.0, 0.0);
        if ((lane & 15) == 0 && w4 < 2) lch[(1 + w4) * CS + wv] = v;
      }
    } else {
      const double v = wave_sum4(s0, s1, s2, 0.0);
      if ((lane & 15) == 0 && w4 < 3) lch[w4 * CS + wv] = v;
    }
    // the slots put() emptied are in place before this block's sums go out
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    u64* cur = W.pay + (int64_t)(k % 3) * P.nblk * line;
    if (t < mine) {
      const double* col = lch + t * CS;
      double val = 0;
#pragma unroll
      for (int cb = 0; cb < CS; cb += RNW) {
        double c8[RNW];
#pragma unroll
        for (int w = 0; w < RNW; ++w) c8[w] = col[cb + w];
        val += ((c8[0] + c8[1]) + (c8[2] + c8[3])) + ((c8[4] + c8[5]) + (c8[6] + c8[7]));
      }
      publish(cur + (int64_t)blk * line + t, val);
    }
    if (!read) return true;
    bool ok = true;
    if (wv < RNW / 2) {
      double* to = lsc + 4 * wv;
      ok = P.nblk <= 64 ? collect_scalars<1>(cur, line, P.nblk, to, A.wait_ticks)
                        : (P.nblk <= 128 ? collect_scalars<2>(cur, line, P.nblk, to, A.wait_ticks)
                                         : collect_scalars<4>(cur, line, P.nblk, to, A.wait_ticks));
    } else if constexpr (TWO) {
      const int* items = litem + t - (RT - CT);
      ok = P.ncollect <= 1 ? collect<1>(cur, items, P.ncollect, lpay, A.wait_ticks)
                           : (P.ncollect <= 3 ? collect<3>(cur, items, P.ncollect, lpay, A.wait_ticks)
                                              : collect<RU>(cur, items, P.ncollect, lpay, A.wait_ticks));
    }
    if (!ok) lfail = 1;
    __syncthreads();
    return lfail == 0;
  };
  auto scalar = [&](int j) { return (lsc[j] + lsc[4 + j]) + (lsc[8 + j] + lsc[12 + j]); };
  // row r of Ac^-1 times the collected restriction (the whole wave); the loads
  // of a pass are issued together (left to itself the compiler waits for each
  // pair before it loads the next)
  auto row_product = [&](int r) -> double {
    constexpr int U = 3;
    const int n = nc2 / 128;  // passes of two columns per lane
    double z = 0, z1 = 0;
    const double2* rc = (const double2*)lpay + lane;
    for (int i = 0; i < n; i += U) {
      double2 a[U], b[U];
#pragma unroll
      for (int u = 0; u < U; ++u) b[u] = rc[64 * (i + u < n ? i + u : n - 1)];
      if (A.cache_rows) {
        const double2* row = (const double2*)(lrow + r * nc2) + lane;
#pragma unroll
        for (int u = 0; u < U; ++u) a[u] = row[64 * (i + u < n ? i + u : n - 1)];
      } else {
        const double* __restrict__ row = A.Ainv + (int64_t)(P.piece_agg[pc0 + r / NM] * NM + r % NM) * A.ld;
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const int c = 128 * (i + u) + 2 * lane;  // past the last column rc is zero
          a[u].x = row[c < nc ? c : 0];
          a[u].y = row[c + 1 < nc ? c + 1 : 0];
        }
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int u = 0; u < U; ++u) {
        if (i + u < n) {
          z += a[u].x * b[u].x;
          z1 += a[u].y * b[u].y;
        }
      }
    }
    return wave_sum1(z + z1);
  };
  // zs = Ac^-1 P^T w + beta zs, z -= alpha zs, a wave per row (first: row wv's
  // product, formed ahead of alpha and beta); set: z = Ac^-1 P^T r instead
  auto coarse_step = [&](double first, double alpha, double beta, bool set) {
    if constexpr (TWO) {
      for (int r = wv; r < nrow; r += RNW) {
        const double zr = r == wv ? first : row_product(r);
        if (lane == 0) {
          const double s = set ? 0.0 : zr + beta * lzs[r];
          lz[r] = set ? zr : lz[r] - alpha * s;
          lzs[r] = s;
        }
      }
    }
  };
  auto first_row = [&]() -> double { return TWO && wv < nrow ? row_product(wv) : 0.0; };
  // u = B^-1 r + P z
  auto precondition = [&]() {
    if constexpr (TWO) __syncthreads();
    if constexpr (BIG) {
#pragma unroll
      for (int p = 0; p < NP; ++p) {
        lu[at(p)] = ((kmask >> p) & 1u) ? 0.0 : rv[p] / (p < NV ? v[p < NV ? p : 0][0][0][0] : dg[p < NV ? 0 : p - NV]);
        fence();
      }
    } else {
#pragma unroll
      for (int p = 0; p < NP; ++p) {
        double z = 0;
#pragma unroll
        for (int b = 0; b < DN; ++b) {
          const double rb = DN == 1 ? rv[p] : __shfl(rv[p], (lane & ~(G - 1)) + b, 64);
          z += Mi[p][b] * rb;
        }
        if constexpr (TWO) {
          const int j = piece[p];
          if (j >= 0 && own) {
            const double* rn = lrel + at(p) * 3;
#pragma unroll
            for (int m = 0; m < NM; ++m) z += pmode<DN>(rn, g, m) * lz[j * NM + m];
          }
        }
        uv[p] = ((kmask >> p) & 1u) ? 0.0 : z;
      }
    }
  };
  // the own u of pass p
  auto uown = [&](int p) -> double {
    if constexpr (BIG)
      return lu[at(p)];
    else
      return uv[p];
  };

  double Sall = 0, Sw = 0, xAx0 = 0, bb = 0, a_prev = 0, g_prev = 0, del = 0, rr = 0, beta = 0;
  int head = 0, iters = 0, done = 0, k = 0, added = 0;
  bool first = true, good = true, xpend = false;
  // BIG: x += a_prev p of the last step
  auto update_x = [&]() {
    if constexpr (BIG) {
      Global* xp = fresh(W.xp + (int64_t)blk * NLOC);
      double xo[NP];
#pragma unroll
      for (int p = 0; p < NP; ++p) xo[p] = xp[(unsigned)at(p)];
#pragma unroll
      for (int p = 0; p < NP; ++p) xp[(unsigned)at(p)] = xo[p] + a_prev * lp[at(p)];
      xpend = false;
    }
  };
  // BIG: x of the nodes into lu
  auto x_to_lu = [&]() {
    if constexpr (BIG) {
      const double* xp = W.xp + (int64_t)blk * NLOC;
#pragma unroll
      for (int p = 0; p < NP; ++p) lu[at(p)] = xp[at(p)];
    }
  };
  if (A.resume) {
    const PcgState* st = W.st;
    Sall = st->Sall;
    xAx0 = st->xAx0;
    bb = st->bb;
    a_prev = st->alpha;
    g_prev = st->rz;
    head = st->head;
    iters = st->iters;
    first = st->fresh != 0;
    Sw = st->Sw;
    rr = st->rr;
    __syncthreads();  // the zeroes above
    if (t < RING) ring[t] = st->ring[t];
#pragma unroll
    for (int p = 0; p < NP; ++p) {
      const int nd = BIG ? P.rows[(int64_t)blk * NLOC + at(p)] : node[BIG ? 0 : p];
      if constexpr (BIG) lu[at(p)] = 0.0;  // a position without a node enters the sums too
      if (nd >= 0 && own) {
        const int64_t i = (int64_t)nd * DN + g;
        rv[p] = W.r[i];
        sv[p] = W.s[i];
        if constexpr (BIG) {
          lu[at(p)] = W.u[i];
          lp[at(p)] = W.p[i];
        } else {
          uv[p] = W.u[i];
          pv[p] = W.p[i];
        }
      }
      fence();
    }
    __syncthreads();
  } else {
    // r = b - A x, x.A x over the unknown rows, rc = P^T r
    if constexpr (BIG) {
      double* xp = W.xp + (int64_t)blk * NLOC;
#pragma unroll
      for (int p = 0; p < NP; ++p) {
        const int nd = P.rows[(int64_t)blk * NLOC + at(p)];
        xp[at(p)] = nd >= 0 ? A.x[nd] : 0.0;
        fence();
      }
      x_to_lu();
    }
    put(xv, k);
    good = halo(k);
    if (good) {
      double y[NP], ax = 0, r2 = 0;
      product(y);
#pragma unroll
      for (int p = 0; p < NP; ++p) {
        const int nd = BIG ? P.rows[(int64_t)blk * NLOC + at(p)] : node[BIG ? 0 : p];
        if (!((kmask >> p) & 1u)) rv[p] = A.b[(int64_t)nd * DN + g] - y[p];
        ax += (BIG ? lu[at(p)] : xv[BIG ? 0 : p]) * y[p];
        r2 += rv[p] * rv[p];
        fence();
      }
      good = sums(ax, r2, 0.0, rv, k, true);
    }
    if (good) {
      xAx0 = scalar(0);
      bb = rr = scalar(1);
      if (rr == 0) done = 1;
      coarse_step(first_row(), 0.0, 0.0, true);
      precondition();
    }
    ++k;
  }
  double inv_g = 1.0 / g_prev, inv_a = 1.0 / a_prev;  // unused on the first iteration
  while (good && !done && added < A.limit) {
    put(uv, k);
    if (xpend) update_x();
    good = halo(k);
    if (!good) break;
    double y[NP], s0 = 0, s1 = 0, s2 = 0;
    product(y);
#pragma unroll
    for (int p = 0; p < NP; ++p) {
      const double u = uown(p);
      s0 += rv[p] * u;
      s1 += y[p] * u;
      s2 += rv[p] * rv[p];
    }
    // what closes the previous iteration is known before the sums arrive
    if (!first) {
      const double term = a_prev * g_prev;
      Sall += term;
      Sw = 0;  // the window summed afresh: the new term replaces the oldest
#pragma unroll
      for (int i = 0; i < RING; ++i) Sw += i == head ? term : ring[i];
      if (t == 0) ring[head] = term;  // the other threads do not use this entry before the next barrier
      head = (head + 1) % RING;
      ++iters;
    }
    good = sums(s0, s1, s2, y, k, true);
    ++k;
    if (!good) break;
    const double gam = scalar(0);
    del = scalar(1);
    rr = scalar(2);
    const double z0 = first_row();
    double alpha;
    if (first) {
      beta = 0;
      alpha = gam / del;
    } else {
      beta = gam * inv_g;
      alpha = gam / (del - beta * gam * inv_a);
    }
    a_prev = alpha;
    g_prev = gam;
    first = false;
    const double scale = Sall > xAx0 ? Sall : xAx0;
    const bool finite = isfinite(rr) && isfinite(gam) && isfinite(del) && isfinite(Sw);
    if (finite && ((iters >= RING && Sw <= A.tolA2 * scale) || rr <= A.tolr2 * bb || gam == 0)) {
      done = 1;  // converged (gam = 0: r = 0 exactly), whatever this step's alpha
      break;
    }
    if (!finite || !(alpha > 0) || !isfinite(alpha)) {
      done = 2;  // breakdown: the caller redoes the solve with the classic iteration
      break;
    }
    coarse_step(z0, alpha, beta, false);
#pragma unroll
    for (int p = 0; p < NP; ++p) {
      sv[p] = y[p] + beta * sv[p];
      rv[p] -= alpha * sv[p];
      if constexpr (BIG) {
        lp[at(p)] = lu[at(p)] + beta * lp[at(p)];
        fence();
      } else {
        pv[p] = uv[p] + beta * pv[p];
        xv[p] += alpha * pv[p];
      }
    }
    xpend = BIG;
    precondition();
    inv_g = 1.0 / g_prev;
    inv_a = 1.0 / a_prev;
    ++added;
  }
  // the solution, and the residual b - A x of it
  if (good) {
    if (xpend) update_x();
#pragma unroll
    for (int p = 0; p < NP; ++p) {
      const int nd = BIG ? P.rows[(int64_t)blk * NLOC + at(p)] : node[BIG ? 0 : p];
      if (nd >= 0 && own) {
        const int64_t i = (int64_t)nd * DN + g;
        A.x[i] = BIG ? W.xp[(int64_t)blk * NLOC + at(p)] : xv[BIG ? 0 : p];
        if (!done) {
          W.r[i] = rv[p];
          W.u[i] = uown(p);
          W.p[i] = BIG ? lp[at(p)] : pv[BIG ? 0 : p];
          W.s[i] = sv[p];
        }
      }
      fence();
    }
    if constexpr (TWO) {
      if (!done) {
        for (int r = t; r < nrow; r += RT) {
          W.z[pc0 * NM + r] = lz[r];
          W.zs[pc0 * NM + r] = lzs[r];
        }
      }
    }
    x_to_lu();
    put(xv, k);
    good = halo(k);
  }
  if (good) {
    double y[NP], r2 = 0;
    product(y);
#pragma unroll
    for (int p = 0; p < NP; ++p) {
      const int nd = BIG ? P.rows[(int64_t)blk * NLOC + at(p)] : node[BIG ? 0 : p];
      const double r = ((kmask >> p) & 1u) ? 0.0 : A.b[(int64_t)nd * DN + g] - y[p];
      r2 += r * r;
      fence();
    }
    good = sums(r2, 0.0, 0.0, y, k, blk == 0);
  }
  if (!good) {
    if (t == 0) A.out->failed = 1;
    return;
  }
  if (blk == 0) {
    const double rt = scalar(0);
    if (t == 0) {
      PcgState st;
      st.rz = st.rz_prev = g_prev;
      st.alpha = a_prev;
      st.beta = beta;
      st.pq = del;
      st.rr = rr;
      st.rrmax = st.rrmax_prev = rr;
      st.bb = bb;
      st.tolr2 = A.tolr2;
      st.tolA2 = A.tolA2;
      st.delta2 = 0;
      st.Sall = Sall;
      st.Sw = Sw;
      st.xAx0 = xAx0;
      for (int i = 0; i < RING; ++i) st.ring[i] = ring[i];
      st.head = head;
      st.done = done;
      st.iters = iters;
      st.nrepl = 0;
      st.fresh = first;
      st.justrep = st.par = st.par_next = st.stop = 0;
      *W.st = st;
      A.out->st = st;
      A.out->rr = rt;
    }
  }
}

// The kernel variants: dof_n, slots per lane, passes, BIG.  A
// block holds RT / lanes * passes nodes, of at most lanes * slots neighbours
// each; the largest pass count of each slot count is what 256 registers hold.
#define EFEA_RESIDENT(X)                                                                    \
  X(1, 7, 1, false) X(1, 7, 2, false) X(1, 7, 4, false) X(1, 7, 9, true)                     \
  X(1, 9, 1, false) X(1, 9, 2, false) X(1, 9, 4, false) X(1, 9, 9, true)                     \
  X(1, 16, 1, false) X(1, 16, 2, false) X(1, 28, 1, false) X(1, 28, 2, false)               \
  X(2, 4, 1, false) X(2, 4, 2, false) X(2, 4, 4, false)                                     \
  X(2, 5, 1, false) X(2, 5, 2, false) X(2, 5, 4, false) X(2, 8, 1, false) X(2, 8, 2, false) \
  X(3, 4, 1, false) X(3, 4, 2, false) X(3, 7, 1, false)

static inline int res_modes(int dof_n) { return dof_n == 1 ? 1 : (dof_n == 2 ? 3 : 6); }

// BIG's x in position order (allotted for every scalar plan).
static inline size_t res_xp_bytes(const ResidentPlan& P) {
  return P.dof_n == 1 ? align256(8 * (size_t)P.nblk * RT * P.passes) : 0;
}

// BIG's streamed passes.
static inline size_t res_vs_bytes(const ResidentPlan& P) {
#define STREAM(D, SV, NPV, BIG)                             \
  if (P.dof_n == D && P.slots == SV && P.passes == NPV)     \
    return align256(8 * (size_t)P.nblk * RT * SV * (NPV - ResPasses<SV, NPV, BIG>::KEPT));
  EFEA_RESIDENT(STREAM)
#undef STREAM
  return 0;
}

static inline size_t res_words(const ResidentPlan& P, size_t* halo) {
  const int line = P.dof_n == 1 ? res_line<1>(P) : (P.dof_n == 2 ? res_line<3>(P) : res_line<6>(P));
  *halo = align256(16 * (size_t)P.nex * P.dof_n) / 8;
  return *halo + 3 * (size_t)P.nblk * line;
}

size_t resident_workspace_bytes(int Nnode, int dof_n, const ResidentPlan& P) {
  const size_t vb = align256(8 * (size_t)Nnode * dof_n), cb = align256(8 * (size_t)P.npiece * res_modes(dof_n));
  size_t halo;
  return 4 * vb + 2 * cb + res_xp_bytes(P) + res_vs_bytes(P) + align256(8 * res_words(P, &halo)) + align256(sizeof(PcgState));
}

static ResWork res_carve(void* ws, int Nnode, int dof_n, const ResidentPlan& P, int64_t* nwords) {
  const size_t vb = align256(8 * (size_t)Nnode * dof_n), cb = align256(8 * (size_t)P.npiece * res_modes(dof_n));
  char* c = (char*)ws;
  ResWork W;
  W.r = (double*)c; c += vb;
  W.u = (double*)c; c += vb;
  W.p = (double*)c; c += vb;
  W.s = (double*)c; c += vb;
  W.z = (double*)c; c += cb;
  W.zs = (double*)c; c += cb;
  W.xp = (double*)c; c += res_xp_bytes(P);
  W.vs = (double*)c; c += res_vs_bytes(P);
  size_t halo;
  *nwords = (int64_t)res_words(P, &halo);
  W.hx = (u64*)c;
  W.pay = W.hx + halo;
  c += align256(8 * (size_t)*nwords);
  W.st = (PcgState*)c;
  return W;
}

int resident_shape(int dof_n, int max_neighbours, int min_passes, int* lanes, int* slots, int* passes) {
  int best = 0;
#define SHAPE(D, SV, NPV, BIG)                                                                      \
  if (!best && D == dof_n && ResLanes<D>::G * SV >= max_neighbours && NPV >= min_passes) {          \
    best = 1;                                                                                       \
    *lanes = ResLanes<D>::G;                                                                        \
    *slots = SV;                                                                                    \
    *passes = NPV;                                                                                  \
  }
  EFEA_RESIDENT(SHAPE)
#undef SHAPE
  return best;
}

// LDS bytes a block of the plan needs without (rows = 0) or with its rows of
// the coarse inverse in LDS; 0 when no kernel variant matches.
static size_t res_lds_bytes(const ResidentPlan& P, int two, int rows) {
#define LDSB(D, SV, NPV, BIG)                                                             \
  if (P.dof_n == D && P.slots == SV && P.passes == NPV)                                   \
    return 8 * (size_t)(two ? res_lds<D, true>(P, SV, NPV, BIG, rows != 0).total          \
                            : res_lds<D, false>(P, SV, NPV, BIG, false).total);
  EFEA_RESIDENT(LDSB)
#undef LDSB
  return 0;
}

int resident_fits(const ResidentPlan& P) {
  const size_t n = res_lds_bytes(P, P.nagg > 0, 0);
  const int nm = res_modes(P.dof_n), mine = 3 + P.max_pieces * nm, line = (mine + 7) / 8 * 8;
  // BIG keeps byte offsets of lu's entries in 16 bits
  if (P.dof_n == 1 && P.passes == 9 && RT * P.passes + P.max_halo > 8191) return 0;
  return n > 0 && n <= (size_t)RES_LDS && P.nblk <= 256 && (P.nagg == 0 || P.ncollect >= 1) && mine <= RT &&
         P.nblk * line <= 65536 && res_columns(P.nagg * nm) <= 32767;
}

template <int DN, int S, int NP, bool TWO, bool BIG>
static int res_launch(const ResidentPlan& P, const ResArgs& A, const ResWork& W, size_t lds, int dev, hipStream_t s) {
  auto* fn = &k_resident<DN, S, NP, TWO, BIG>;
  static thread_local int ready = -1;  // device whose limit was raised by this thread
  if (ready != dev) {
    if (hipFuncSetAttribute((const void*)fn, hipFuncAttributeMaxDynamicSharedMemorySize, RES_LDS) != hipSuccess) {
      (void)hipGetLastError();
      return 1;
    }
    ready = dev;
  }
  hipLaunchKernelGGL(fn, dim3((unsigned)P.nblk), dim3(RT), lds, s, KernelPlan(P), A, W);
  return hipGetLastError() == hipSuccess ? 0 : 1;
}

constexpr int RES_DEVICES = 64;
static std::mutex res_mutex;
// The event recorded behind the last resident solve queued on each device.
static hipEvent_t res_last[RES_DEVICES];
// Events of threads that have ended, for the next ones (never destroyed:
// res_last may still name one; leaked, so that they outlive every thread).
static std::vector<hipEvent_t>* const res_free = new std::vector<hipEvent_t>[RES_DEVICES];

struct ResEvents {
  hipEvent_t ev[RES_DEVICES][2] = {};
  ~ResEvents() {
    std::lock_guard<std::mutex> lock(res_mutex);
    for (int d = 0; d < RES_DEVICES; ++d)
      for (hipEvent_t e : ev[d])
        if (e) res_free[d].push_back(e);
  }
};

// This thread's event of poll slot `slot` on device dev (null: creation failed).
static hipEvent_t res_event(int dev, int slot) {
  static thread_local ResEvents own;
  hipEvent_t& e = own.ev[dev][slot];
  if (e) return e;
  {
    std::lock_guard<std::mutex> lock(res_mutex);
    if (!res_free[dev].empty()) {
      e = res_free[dev].back();
      res_free[dev].pop_back();
      return e;
    }
  }
  if (hipEventCreateWithFlags(&e, hipEventDisableTiming | hipEventReleaseToSystem) != hipSuccess) {
    (void)hipGetLastError();
    e = nullptr;
  }
  return e;
}

// phase PCGP_WHOLE: the solve to its end; PCGP_START queues it with at most
// first_check iterations and returns; PCGP_FINISH waits for that and, if the
// stopping test had not been met, continues the solve (*resumed = 1).
int solve_resident(const ResidentPlan& P, int Nnode, const int* node_ptr, const double* vals,
                   const unsigned char* known, const double* Minv, const double* rel, const double* Ainv, int ld,
                   const double* b, double* x, void* ws, double tol_r, double tol_A, int maxit, int first_check,
                   double wait_ms, hipStream_t s, double* info, int phase, int* resumed) {
  if (resumed) *resumed = 0;
  const int slot = phase == PCGP_WHOLE ? 0 : 1;
  PollBuf* pb = poll_buffer(slot);
  int dev = 0, cus = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev >= RES_DEVICES ||
      hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) {
    set_error("resident: no device");
    return EFEA_ERR_HIP;
  }
  const hipEvent_t done = res_event(dev, slot);
  if (!pb || !done) {
    set_error("resident: pinned host allocation failed");
    return EFEA_ERR_HIP;
  }
  if (P.nblk > cus) {
    set_error("resident: a plan of %d blocks on a device of %d CUs", P.nblk, cus);
    return EFEA_ERR_ARG;
  }
  const int two = P.nagg > 0;
  size_t lds = res_lds_bytes(P, two, 1);
  ResArgs A;
  A.cache_rows = two && lds <= (size_t)RES_LDS;
  if (!A.cache_rows) lds = res_lds_bytes(P, two, 0);
  int64_t nwords = 0;
  const ResWork W = res_carve(ws, Nnode, P.dof_n, P, &nwords);
  A.node_ptr = node_ptr;
  A.vals = vals;
  A.known = known;
  A.Minv = Minv;
  A.b = b;
  A.x = x;
  A.rel = rel;
  A.Ainv = Ainv;
  A.ld = ld;
  A.tolr2 = tol_r * tol_r;
  A.tolA2 = tol_A * tol_A;
  A.wait_ticks = (u64)((wait_ms > 0 ? wait_ms : 250.0) * 1e5);  // 100 MHz; 0: give up at the first miss
  A.out = pb;
  auto launch = [&](int limit, int resume) -> int {
    A.limit = limit;
    A.resume = resume;
    const unsigned nb = (unsigned)((nwords + 1023) / 1024 < 1024 ? (nwords + 1023) / 1024 : 1024);
    std::lock_guard<std::mutex> lock(res_mutex);
    // also on what looks like the last solve's stream: a handle may name another
    // stream by now, or one for each thread (hipStreamPerThread)
    hipEvent_t& last = res_last[dev];
    if (last && hipStreamWaitEvent(s, last, 0) != hipSuccess) {
      set_error("resident: the last solve's event could not be waited for");
      return EFEA_ERR_HIP;
    }
    hipLaunchKernelGGL(k_res_empty, dim3(nb ? nb : 1), dim3(256), 0, s, nwords, W.hx, pb);
    int rc = 1;
#define RUN(D, SV, NPV, BIG)                                                                \
  if (P.dof_n == D && P.slots == SV && P.passes == NPV) {                                   \
    if constexpr (D == 1)                                                                   \
      rc = two ? 1 : res_launch<D, SV, NPV, false, BIG>(P, A, W, lds, dev, s);              \
    else                                                                                    \
      rc = two ? res_launch<D, SV, NPV, true, BIG>(P, A, W, lds, dev, s)                    \
               : res_launch<D, SV, NPV, false, BIG>(P, A, W, lds, dev, s);                  \
  }
    EFEA_RESIDENT(RUN)
#undef RUN
    if (rc) {
      set_error("resident: the launch of %d blocks was refused", P.nblk);
      return EFEA_ERR_NOCONV;
    }
    if (hipEventRecord(done, s) != hipSuccess) {
      set_error("resident: event not recorded");
      return EFEA_ERR_HIP;
    }
    last = done;
    return 0;
  };
  auto refused = [&](int rc) {
    if (rc == EFEA_ERR_NOCONV && info) {
      info[0] = info[2] = 0;
      info[1] = 1;
      info[3] = 2;
    }
    return rc;
  };
  if (phase != PCGP_FINISH) {
    const int e = launch(phase == PCGP_START && first_check < maxit ? first_check : maxit, 0);
    if (phase == PCGP_START) {
      if (e == EFEA_ERR_NOCONV) {  // the finish reports it
        if (hipStreamSynchronize(s) != hipSuccess) return EFEA_ERR_HIP;
        pb->failed = 2;
        return 0;
      }
      return e;
    }
    if (e) return refused(e);
  }
  // (the solve's end, not that of what the caller queued behind it)
  if (hipEventSynchronize(done) != hipSuccess) {
    set_error("resident: state readback failed");
    return EFEA_ERR_HIP;
  }
  if (phase == PCGP_FINISH && !pb->failed && !pb->st.done && first_check < maxit) {
    if (resumed) *resumed = 1;
    if (int e = launch(maxit - first_check, 1)) return refused(e);
    if (hipEventSynchronize(done) != hipSuccess) {
      set_error("resident: state readback failed");
      return EFEA_ERR_HIP;
    }
  }
  if (pb->failed) {
    set_error(pb->failed == 1 ? "resident: a block waited longer than its limit for another"
                              : "resident: the launch of %d blocks was refused", P.nblk);
    refused(EFEA_ERR_NOCONV);
    info[2] = pb->failed == 1;
    return EFEA_ERR_NOCONV;
  }
  const PcgState fin = pb->st;
  return pcg_finish_info(&fin, pb->rr, info);
}

}  // namespace efea
