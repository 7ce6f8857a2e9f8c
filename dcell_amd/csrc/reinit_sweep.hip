// reinit_sweep.hip -- the parallel reinitialisation on gfx950
// (dcl_reinitialize_parallel): LevelSetReinitialize
// (LevelSetMethod/FastMarching.c:10-146) computed by sweeps over the whole
// window instead of one accepted node at a time.
//
// The boundary values are the fast marching's (the distance to the
// orthogonal projection at every projection record) and so is the update:
// AccumulateCoef (FastMarching2D.c:33-94) over the axes, then the larger
// root.  What the fast marching decides by its order -- which neighbours
// are already accepted when a node is pushed, and which push's value the
// node keeps -- a sweep decides from the neighbours' values: each push is
// replayed in the order of the pushing neighbours' values (the boundary
// nodes' pushes first), with the neighbours accepted by then, and the node
// keeps the least value pushed before its own value comes up.  Every sweep
// recomputes every node from the previous sweep's values (two buffers), so
// the result does not depend on scheduling; sweeps end when no node moves by
// more than band_width * 1e-9.  Nodes whose order is decided by their last
// bits can trade values in a cycle: once the count of moving nodes has
// fallen and then stops falling, a node's value may only go down, which ends
// every cycle.
//
// Work skips what cannot change.  A node whose stencil (the node and two
// nodes each way along each axis) held no change in the previous sweep would
// come out as it is, so a change marks the nodes whose stencil holds it, and
// each sweep recomputes only the marked nodes; the output buffer already
// holds the others' values (both buffers start equal, and a node not
// recomputed did not change in the sweep before).  The boundary values are
// the changes before the first sweep.  A sweep is two launches: one lists
// the marked nodes (each chunk of 1024 nodes carries a flag set with its
// marks, so a block reads its chunks' flags at once and scans only the
// marked chunks, one wave each with 16 marks per lane, clearing them) and, in
// blocks of its own, sums the moved nodes of the sweep before and decides;
// the other updates the listed nodes, one thread each, so that whole waves
// run the chain of updates.  Lists are gathered per block in LDS and
// published with one atomic each: an atomic per wave on one counter would
// queue (6 ns each).
//
// A batch of level sets runs in one launch per step, over all nodes (in
// raster order) and all records, each block finding its level set by a
// binary search.
#include <math.h>
#include <string.h>

#include "dcl_host.hpp"
#include "dcl_reinit.hpp"

namespace dcl {

constexpr int RS_B = 256;
constexpr double RS_TOL = 1e-9;  // settled: no node moves by more than band_width * RS_TOL
constexpr int RS_OUT = 3;        // the mask of a stencil node outside the window
constexpr int RS_CH = 1024;      // nodes per chunk of the mark scan (one wave, 16 per lane)
constexpr int RS_STAGE = 3072;   // list entries a block gathers before publishing them
// blocks of the mark scan: each publishes its entries with an atomic on one
// counter, and fewer leave waves idle.  ms with 512, 1024, 2048 and 4096: a
// 256^3 step 1.64, 1.60, 1.78, 2.05; level sets of edges 32 to 48, 4 of them
// 0.81, 0.76, 0.79, 0.79, 64 of them 2.75, 2.73, 3.02, 3.30; 256 of 32 to 64
// 11.8, 10.5, 10.1, 10.4; 1000 of 24 to 32 21.3, 19.9, 19.2, 19.3; 64 of 96
// 10.5, 9.2, 8.5, 8.9.
constexpr int RS_NEED_GRID = 1024;
constexpr int RS_GRID = 4096;       // blocks of the update, each taking listed nodes in turn
constexpr int RS_GROUP = 4;         // sweeps queued between looks at the count of level sets still sweeping

struct RsCell {
  double* buf[2];        // buf[0]: the caller's phi, buf[1]: scratch
  unsigned char* mask;   // 0: a - side node, 1: a + side node, 2: a boundary node
  unsigned char* nd[2];  // marks: sweep k + 1 recomputes the nodes marked in nd[k & 1]
  unsigned char* cd[2];  // per chunk of RS_CH nodes: it holds a mark in nd[k & 1]
  KWin w;
  int d3;
  double bw, inf, tol;
  long long qb0, qb1;  // the level set's raster blocks (RS_B nodes each) in the batch
  long long cb0;       // its first chunk (RS_CH nodes) in the batch
  long long rb0, rb1;  // its record blocks (RS_B records each) in the batch
  const dcl_irregular_node* nodes;
  int64_t count;
  dcl_icoor* band;
  int64_t band_cap;
};

struct RsState {
  int k;        // sweeps done
  int settle;   // values may only go down
  int falling;  // the count of moving nodes has fallen
  int done;     // 1 settled, 2 NaN update, 3 out of sweeps
  long long last;  // the previous sweep's count, -1 before the first
  int nan;
  int pad;
};

enum { RS_ACTIVE = 0, RS_SETTLED = 1, RS_NAN = 2, RS_SWEEPS = 3 };
enum { RS_KEY_RASTER = 0, RS_KEY_RECORD = 1, RS_KEY_CHUNK = 2 };

// the level set of batch block g: the last one whose first block is <= g
template <int KEY>
__device__ __forceinline__ int rs_find(const RsCell* __restrict__ cells, int ncells, long long g) {
  int lo = 0, hi = ncells - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    const long long f = KEY == RS_KEY_RASTER ? cells[mid].qb0 : KEY == RS_KEY_RECORD ? cells[mid].rb0 : cells[mid].cb0;
    if (f <= g) lo = mid;
    else hi = mid - 1;
  }
  return lo;
}

__device__ __forceinline__ int64_t rs_nodes(const RsCell& c) { return (int64_t)c.w.nx * c.w.ny * c.w.nz; }

// A level set's arrays are named by a table in memory, so their pointers are
// cast to the global address space (the compiler would take them for flat).
template <typename T>
using rs_gptr = __attribute__((address_space(1))) T*;
typedef unsigned rs_u32x4 __attribute__((ext_vector_type(4)));

// a node changed: the nodes whose stencil holds it (itself and two nodes
// each way along each axis) are recomputed in the next sweep
template <int DIM>
__device__ __forceinline__ void rs_mark(const RsCell& c, unsigned char* nd_, unsigned char* cd_, int64_t i, int lx,
                                        int ly, int lz) {
  const rs_gptr<unsigned char> nd = (rs_gptr<unsigned char>)nd_, cd = (rs_gptr<unsigned char>)cd_;
  const int64_t sy = c.w.nx, sz = (int64_t)c.w.nx * c.w.ny;
  nd[i] = 1;
  cd[i / RS_CH] = 1;
#pragma unroll
  for (int o = -2; o <= 2; ++o) {
    if (o == 0) continue;
    if (lx + o >= 0 && lx + o < c.w.nx) {
      nd[i + o] = 1;
      cd[(i + o) / RS_CH] = 1;
    }
    if (ly + o >= 0 && ly + o < c.w.ny) {
      nd[i + o * sy] = 1;
      cd[(i + o * sy) / RS_CH] = 1;
    }
    if (DIM == 3 && lz + o >= 0 && lz + o < c.w.nz) {
      nd[i + o * sz] = 1;
      cd[(i + o * sz) / RS_CH] = 1;
    }
  }
}

// what the first sweep finds: per level set its state, per sweep the counts
// of active level sets and listed nodes, and the partial counts of a sweep
struct RsStart {
  RsState* state;
  int *active, *ncount;
  unsigned long long* parts;
  int ncells, sweeps, nparts;
};

// FMM_InitializeEikonal (FastMarching.c:46-58): phi to +-PHI_INF in both
// buffers; the mask keeps each node's side.  The grid sets z up too: three
// fills and an upload before it took 20 us of a call.
__global__ __launch_bounds__(RS_B) void rs_reset_k(const RsCell* __restrict__ cells, int ncells, long long nq,
                                                   RsStart z) {
  const long long g = blockIdx.x, all = (long long)gridDim.x * RS_B;
  for (long long e = g * RS_B + threadIdx.x; e < z.ncells; e += all) z.state[e] = {0, 0, 0, 0, -1, 0, 0};
  for (long long e = g * RS_B + threadIdx.x; e < z.sweeps; e += all) z.active[e] = z.ncount[e] = 0;
  for (long long e = g * RS_B + threadIdx.x; e < z.nparts; e += all) z.parts[e] = 0;
  if (g >= nq) return;
  const RsCell& c = cells[rs_find<RS_KEY_RASTER>(cells, ncells, g)];
  const int64_t i = (g - c.qb0) * RS_B + threadIdx.x;
  if (i >= rs_nodes(c)) return;
  const bool pos = c.buf[0][i] > 0;
  const double v = pos ? c.inf : -c.inf;
  c.mask[i] = pos ? 1 : 0;
  c.buf[0][i] = v;
  c.buf[1][i] = v;
  c.nd[0][i] = 0;
  c.nd[1][i] = 0;
  if (i % RS_CH == 0) {
    c.cd[0][i / RS_CH] = 0;
    c.cd[1][i / RS_CH] = 0;
  }
}

// FMM_InitializeEikonal (FastMarching.c:60-74): the boundary values, which
// mark the first sweep's nodes
template <int DIM>
__global__ __launch_bounds__(RS_B) void rs_bc_k(const RsCell* __restrict__ cells, int ncells, long long nr) {
#pragma clang fp contract(off)
  const long long g = blockIdx.x;
  if (g >= nr) return;
  const RsCell& c = cells[rs_find<RS_KEY_RECORD>(cells, ncells, g)];
  const int64_t i = (g - c.rb0) * RS_B + threadIdx.x;
  if (i >= c.count) return;
  const dcl_irregular_node n = c.nodes[i];
  if (n.axis != -1 || !ri_inside(c.w, c.d3, n.pos.x, n.pos.y, n.pos.z)) return;
  const double r = c.d3 ? sqrt(n.op.x * n.op.x + n.op.y * n.op.y + n.op.z * n.op.z)
                         : sqrt(n.op.x * n.op.x + n.op.y * n.op.y);
  const int64_t j = ri_index(c.w, c.d3, n.pos.x, n.pos.y, n.pos.z);
  const double v = n.sign_center * r;
  c.buf[0][j] = v;
  c.buf[1][j] = v;
  c.mask[j] = 2;
  rs_mark<DIM>(c, c.nd[0], c.cd[0], j, n.pos.x - c.w.px, n.pos.y - c.w.py, c.d3 ? n.pos.z - c.w.pz : 0);
}

// The acceptance-time code of a neighbour of value v and mask m as the side
// `sign` sees it, q = sign * v: its value for an accepted node of this side,
// which pushes its neighbours at that time; -1 for a boundary node with q >= 0,
// which pushes before the side's pops; RS_T_STATIC for a - side node that the
// + side finds final, which does not push; INFINITY for a node never accepted.
constexpr double RS_T_STATIC = -2.0;

__device__ __forceinline__ double rs_tcode(double inf, int sign, double v, int m) {
  const double q = sign * v;
  const bool own = m == (sign > 0 ? 1 : 0), bc = m == 2, other = (sign > 0) & (m == 0);
  const bool known = (q < inf) & (own | ((0 <= q) & (bc | other)));
  const double t = own ? q : bc ? -1.0 : RS_T_STATIC;
  return known ? t : INFINITY;
}

// One direction of an axis as a node's pushes see it: AccumulateCoef's
// (FastMarching2D.c:33-94) differences from the node, which is not accepted
// and counts as inf, to its neighbour (value p) and the node beyond it.  The
// terms depend on the acceptances only through which of the two hold, so
// they are formed once; a push at time T takes the second-order ones from e2
// on, the first-order ones from e1 on.
struct RsSide {
  double p, q;    // the neighbour's value; (4 p - beyond) / 3
  double D2;      // the second-order difference
  double e1, e2;  // the times from which each order holds (INFINITY: never)
};

// t1, t2: the acceptance-time codes of the neighbour and the node beyond
__device__ __forceinline__ RsSide rs_side(double inf, double p, double t1, double beyond, double t2) {
#pragma clang fp contract(off)
  RsSide s;
  s.p = p;
  s.q = (4 * p - beyond) / 3;
  s.D2 = (3 * inf - 4 * p + beyond) / 2.;
  const bool first = (0 <= p) & (p < inf);  // inf - p > 0
  const bool second = first & (0 <= beyond) & (beyond < inf) & (s.D2 > 0);
  s.e1 = first ? t1 : INFINITY;
  s.e2 = second ? fmax(t1, t2) : INFINITY;
  return s;
}

// the node's value from its stencil: nv the values and nt the
// acceptance-time codes (for the node's side) of the nodes two each way
// along each axis (-2, -1, +1, +2); NaN for a NaN update.  Each push takes
// the larger difference of each axis's two directions (the + one when
// equal), sums the terms in axis order and solves the quadratic; the larger
// root's numerator falls back to -B where the discriminant is negative.
template <int DIM>
__device__ __forceinline__ double rs_node(double inf, double bw, int sign, const double (&nv)[DIM][4],
                                          const double (&nt)[DIM][4]) {
#pragma clang fp contract(off)
  double cand = INFINITY;
  RsSide sd[DIM][2];       // [axis][0: +, 1: -]
  double push[DIM][2];     // push times not yet replayed
#pragma unroll
  for (int a = 0; a < DIM; ++a) {
    sd[a][0] = rs_side(inf, sign * nv[a][2], nt[a][2], sign * nv[a][3], nt[a][3]);
    sd[a][1] = rs_side(inf, sign * nv[a][1], nt[a][1], sign * nv[a][0], nt[a][0]);
    push[a][0] = nt[a][2] == RS_T_STATIC ? INFINITY : nt[a][2];
    push[a][1] = nt[a][1] == RS_T_STATIC ? INFINITY : nt[a][1];
  }
  // at most 2 * DIM distinct push times, then one pass that finds none
#pragma unroll 1
  for (int guard = 0; guard <= 2 * DIM; ++guard) {
    double T = INFINITY;
#pragma unroll
    for (int a = 0; a < DIM; ++a) T = fmin(T, fmin(push[a][0], push[a][1]));
    if (T == INFINITY || !(T < cand)) break;
    double A = 0, B = 0, C = -1;
#pragma unroll
    for (int a = 0; a < DIM; ++a) {
      const RsSide &sp = sd[a][0], &sm = sd[a][1];
      const bool p1 = sp.e1 <= T, p2 = sp.e2 <= T, m1 = sm.e1 <= T, m2 = sm.e2 <= T;
      const double Dp = p2 ? sp.D2 : p1 ? inf - sp.p : 0.0;
      const double Dm = m2 ? sm.D2 : m1 ? inf - sm.p : 0.0;
      const bool minus = Dm > Dp;
      const bool second = minus ? m2 : p2, first = minus ? m1 : p1;
      const double x = minus ? (m2 ? sm.q : sm.p) : (p2 ? sp.q : sp.p);
      // 9/4, -9/2 x, 9/4 x x; or 1, -2 x, x x; or nothing
      const double ka = second ? 9. / 4. : 1., kb = second ? -9. / 2. : -2.;
      const bool some = first | second;
      A += some ? ka : 0.;
      B += some ? kb * x : 0.;
      C += some ? ka * x * x : 0.;
#pragma unroll
      for (int d = 0; d < 2; ++d) push[a][d] = push[a][d] <= T ? INFINITY : push[a][d];
    }
    const double disc = sqrt(B * B - 4 * A * C);
    const double d1 = (disc != disc ? -B : -B + disc) / (2 * A);
    if (d1 != d1) return NAN;
    if (d1 < cand) cand = d1;
  }
  return cand <= bw ? sign * cand : sign * inf;
}

// the block-wide exclusive prefix of v (RS_B threads) and the total
__device__ __forceinline__ int rs_scan(int v, unsigned* wsum, int* total) {
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  int x = v;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int t = __shfl_up(x, o, 64);
    if (lane >= o) x += t;
  }
  if (lane == 63) wsum[wv] = (unsigned)x;
  __syncthreads();
  int pre = 0;
  for (int w = 0; w < wv; ++w) pre += (int)wsum[w];
  *total = (int)(wsum[0] + wsum[1] + wsum[2] + wsum[3]);
  __syncthreads();
  return pre + x - v;
}

// after a sweep, one wave per level set: the count of moving nodes decides
// whether it has settled and whether its values may only go down from the
// next sweep on.  active: the level sets still sweeping.
__device__ __forceinline__ void rs_state_of(RsState* __restrict__ st, int i, int max_sweeps, int* __restrict__ active,
                                            unsigned long long* __restrict__ parts, int nparts, int pstride) {
  const int lane = threadIdx.x & 63;
  if (st[i].done) return;
  unsigned long long c = 0;
  if (lane < nparts) {
    c = parts[(long long)lane * pstride + i];
    parts[(long long)lane * pstride + i] = 0;
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) c += __shfl_xor(c, o, 64);
  if (lane != 0) return;
  RsState s = st[i];
  s.k++;
  if (s.nan) {
    s.done = RS_NAN;
  } else if (c == 0) {
    s.done = RS_SETTLED;
  } else {
    if (s.last >= 0 && (long long)c < s.last) s.falling = 1;
    else if (s.last >= 0 && s.falling) s.settle = 1;
    s.last = (long long)c;
    if (s.k >= max_sweeps) s.done = RS_SWEEPS;
  }
  st[i] = s;
  if (!s.done) atomicAdd(active, 1);
}

// The nodes sweep `sweep` recomputes: the marked ones, read and cleared 16 at
// a time (the marks of the sweep after next are written into these bytes).
// One wave per marked chunk; a block's entries are gathered in LDS and
// published with one atomic, entries past the LDS space with one per chunk.
// The last nstate blocks step the level sets' states after the sweep before
// (sweep > 0), which the next update needs and the mark scan does not: which
// marks a sweep reads depends on its number alone, and a level set settled
// just now only lists nodes that the update then leaves out.
__global__ __launch_bounds__(RS_B) void rs_need_k(const RsCell* __restrict__ cells, int ncells,
                                                  RsState* __restrict__ st, long long nch, int sweep, int scan_blocks,
                                                  int2* __restrict__ nlist, int* __restrict__ ncount, int max_sweeps,
                                                  int* __restrict__ active, unsigned long long* __restrict__ parts,
                                                  int nparts, int pstride) {
  __shared__ int2 stage[RS_STAGE];
  __shared__ unsigned wsum[RS_B / 64];
  __shared__ int at, held, cut;  // entries reserved; the first reservation past the LDS space
  __shared__ int live[RS_B];  // this round's chunks holding marks, as batch chunk indices
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  if ((int)blockIdx.x >= scan_blocks) {
    const int i = ((int)blockIdx.x - scan_blocks) * (RS_B / 64) + wv;
    if (i < ncells) rs_state_of(st, i, max_sweeps, active, parts, nparts, pstride);
    return;
  }
  if (tid == 0) {
    held = 0;
    cut = RS_STAGE;
  }
  // the block's chunks are blockIdx.x + q * scan_blocks; their flags are read
  // RS_B at a time, one per thread, and the marked ones taken by the waves in
  // turn
  const long long per = (nch - blockIdx.x + scan_blocks - 1) / scan_blocks;
  for (long long q0 = 0; q0 < per; q0 += RS_B) {
    const long long g = blockIdx.x + (q0 + tid) * scan_blocks;
    bool has = false;
    if (q0 + tid < per) {
      const int ci = rs_find<RS_KEY_CHUNK>(cells, ncells, g);
      const RsCell& c = cells[ci];
      const rs_gptr<unsigned char> cdk = (rs_gptr<unsigned char>)c.cd[sweep & 1];
      has = cdk[g - c.cb0] != 0;
      if (has) cdk[g - c.cb0] = 0;
    }
    int nlive;
    const int slot = rs_scan(has ? 1 : 0, wsum, &nlive);
    if (has) live[slot] = (int)g;
    __syncthreads();
    for (int e = wv; e < nlive; e += RS_B / 64) {
      const long long gc = live[e];
      const int ci = __builtin_amdgcn_readfirstlane(rs_find<RS_KEY_CHUNK>(cells, ncells, gc));
      const RsCell& c = cells[ci];
      const int64_t n = rs_nodes(c);
      const int64_t i0 = (gc - c.cb0) * RS_CH + 16 * lane;
      // the mark arrays are padded to 256 bytes
      const rs_gptr<rs_u32x4> nd = (rs_gptr<rs_u32x4>)(c.nd[sweep & 1] + i0);
      rs_u32x4 w = {0u, 0u, 0u, 0u};
      if (i0 < n) w = *nd;
      // marks are 0 or 1 per byte: bit j of m = byte j
      unsigned m = 0;
#pragma unroll
      for (int j = 0; j < 4; ++j) m |= ((((w[j] & 0x01010101u) * 0x01020408u) >> 24) & 0xfu) << (4 * j);
      if (i0 + 16 > n && i0 < n) m &= (1u << (int)(n - i0)) - 1u;
      if (m) *nd = rs_u32x4{0u, 0u, 0u, 0u};
      const int cnt = __popc(m);
      int pre = cnt;
#pragma unroll
      for (int o = 1; o < 64; o <<= 1) {
        const int t = __shfl_up(pre, o, 64);
        if (lane >= o) pre += t;
      }
      const int tot = __shfl(pre, 63);
      if (tot == 0) continue;
      int base = 0;
      if (lane == 63) base = atomicAdd(&held, tot);
      base = __shfl(base, 63);
      const bool fits = base + tot <= RS_STAGE;
      if (!fits) {
        if (lane == 63) {
          atomicMin(&cut, base);
          base = atomicAdd(ncount, tot);
        }
        base = __shfl(base, 63);
      }
      int pos = base + pre - cnt;
      for (; m; m &= m - 1) {
        const int2 ent = make_int2(ci, (int)(i0 + __ffs((int)m) - 1));
        if (fits) stage[pos++] = ent;
        else nlist[pos++] = ent;
      }
    }
    __syncthreads();
  }
  const int n = min(held, cut);  // uniform: every reservation is made
  if (n > 0) {
    if (tid == 0) at = atomicAdd(ncount, n);
    __syncthreads();
    for (int q = tid; q < n; q += RS_B) nlist[at + q] = stage[q];
  }
}

__global__ __launch_bounds__(RS_B) void rs_state_k(RsState* __restrict__ st, int ncells, int max_sweeps,
                                                   int* __restrict__ active, unsigned long long* __restrict__ parts,
                                                   int nparts, int pstride) {
  const int i = blockIdx.x * (RS_B / 64) + (threadIdx.x >> 6);
  if (i < ncells) rs_state_of(st, i, max_sweeps, active, parts, nparts, pstride);
}

// the listed nodes' new values, one thread each.  A wave works its nodes of
// one level set at a time (nearly always all of them), so that the level
// set's arrays are the same for the lanes at work, and every load of a node's
// stencil is issued before the first is waited for: nodes outside the window
// load the node itself instead.  At 256^3 with 600 000 listed nodes 71 -> 37 us
// against a level set per lane (a loop over its values around every load) and
// the terms of each axis formed anew at every push.  Three waves per SIMD: at
// 168 registers nothing spills; two (173) took 6% more per reinitialisation,
// four spilled and took 18% more.  The per-sweep counts of moving nodes are
// added into nparts partial sums per level set, each on its own 128-byte
// line (part p of level set i at p * pstride + i).
template <int DIM>
__device__ __forceinline__ bool rs_update_node(const RsCell& c, RsState* __restrict__ st, int64_t i) {
#pragma clang fp contract(off)
  if (st->done) return false;
  const int k = st->k, settle = st->settle;
  const rs_gptr<const double> in = (rs_gptr<const double>)((k & 1) ? c.buf[1] : c.buf[0]);
  const rs_gptr<double> out = (rs_gptr<double>)((k & 1) ? c.buf[0] : c.buf[1]);
  const rs_gptr<const unsigned char> mask = (rs_gptr<const unsigned char>)c.mask;
  const int64_t sy = c.w.nx, sz = (int64_t)c.w.nx * c.w.ny;
  const int lz = DIM == 3 ? (int)((unsigned)i / (unsigned)sz) : 0;
  const int r2 = (int)(i - lz * sz);
  const int ly = (int)((unsigned)r2 / (unsigned)c.w.nx), lx = r2 - ly * c.w.nx;
  double nv[DIM][4], nt[DIM][4];
  int mm[DIM][4];
  const int m = mask[i];
  const double old = in[i];
#pragma unroll
  for (int a = 0; a < DIM; ++a) {
    const int p = a == 0 ? lx : a == 1 ? ly : lz;
    const int lim = a == 0 ? c.w.nx : a == 1 ? c.w.ny : c.w.nz;
    const int64_t st_ = a == 0 ? 1 : a == 1 ? sy : sz;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int o = q < 2 ? q - 2 : q - 1;
      const bool inside = (unsigned)(p + o) < (unsigned)lim;
      const int64_t at = inside ? i + o * st_ : i;
      nv[a][q] = in[at];
      const int b = mask[at];
      mm[a][q] = inside ? b : RS_OUT;
    }
  }
  if (m == 2) return false;
  const int sg = m ? 1 : -1;
#pragma unroll
  for (int a = 0; a < DIM; ++a)
#pragma unroll
    for (int q = 0; q < 4; ++q) nt[a][q] = rs_tcode(c.inf, sg, nv[a][q], mm[a][q]);
  const double u = rs_node<DIM>(c.inf, c.bw, sg, nv, nt);
  if (u != u) atomicOr(&st->nan, 1);
  double v = old;
  if (!settle || sg * u < sg * v) v = u;
  out[i] = v;
  if (__double_as_longlong(v) != __double_as_longlong(old))
    rs_mark<DIM>(c, (k & 1) ? c.nd[0] : c.nd[1], (k & 1) ? c.cd[0] : c.cd[1], i, lx, ly, lz);
  return fabs(v - old) > c.tol;
}

template <int DIM>
__global__ __launch_bounds__(RS_B) __attribute__((amdgpu_waves_per_eu(3, 8))) void rs_update_k(
    const RsCell* __restrict__ cells, RsState* __restrict__ st, const int2* __restrict__ nlist,
    const int* __restrict__ ncount, unsigned long long* __restrict__ parts, int nparts, int pstride) {
  const int n = *ncount;
  for (int e0 = blockIdx.x * RS_B; e0 < n; e0 += gridDim.x * RS_B) {
    const int e = e0 + threadIdx.x;
    bool moved = false;
    int ci = -1;
    int64_t i = 0;
    if (e < n) {
      const int2 w = nlist[e];
      ci = w.x;
      i = w.y;
    }
    for (unsigned long long todo = __ballot(ci >= 0); todo;) {
      const int cu = __builtin_amdgcn_readlane(ci, __builtin_ctzll(todo));
      if (ci == cu) moved = rs_update_node<DIM>(cells[cu], st + cu, i);
      todo &= ~__ballot(ci == cu);
    }
    // one atomic per wave where the wave's nodes are of one level set
    const int c0 = __builtin_amdgcn_readfirstlane(ci);
    const bool uni = __ballot(ci != c0 && ci >= 0) == 0ull;
    const unsigned long long mb = __ballot(moved);
    if (uni) {
      if (mb && (threadIdx.x & 63) == 0)
        atomicAdd(&parts[(long long)((e0 / RS_B + (threadIdx.x >> 6)) % nparts) * pstride + c0],
                  (unsigned long long)__popcll(mb));
    } else if (moved) {
      atomicAdd(&parts[(long long)((e0 / RS_B) % nparts) * pstride + ci], 1ull);
    }
  }
}

// the exclusive rank of a true predicate within the block (RS_B threads)
__device__ __forceinline__ unsigned rs_rank(bool p, unsigned* sh) {
  const unsigned long long bal = __ballot(p);
  const unsigned lane_pre =
      __builtin_amdgcn_mbcnt_hi((unsigned)(bal >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)bal, 0u));
  const int wv = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0) sh[wv] = (unsigned)__popcll(bal);
  __syncthreads();
  unsigned pre = 0;
  for (int k = 0; k < wv; ++k) pre += sh[k];
  __syncthreads();
  return pre + lane_pre;
}

__device__ __forceinline__ long long rs_prefix(const unsigned* counts, const unsigned long long* sums, long long b) {
  return (long long)counts[b] + (long long)sums[b / SCAN_TILE];
}

// rs_final_k and rs_side_write_k run one raster block (RS_B nodes) per wave,
// nodes e * 64 + lane for e = 0 .. RS_B / 64 - 1 (raster order: e, then
// lane); rs_final_k issues its loads before its stores and keeps each row's
// ballot of each side, from which rs_side_write_k ranks the band nodes.
constexpr int RS_WPB = RS_B / 64;  // raster blocks per workgroup
constexpr int RS_ROWS = RS_B / 64; // 64-node rows per raster block

// the result into the caller's buffer where the last sweep wrote the other
// one, then the band counts: each side per raster block (the block past the
// last level set counts nothing, so the scans' last entry is the total), and
// each row's ballot of each side for rs_side_write_k
__global__ __launch_bounds__(RS_B) void rs_final_k(const RsCell* __restrict__ cells, int ncells, long long nq,
                                                   long long nq1, const RsState* __restrict__ st,
                                                   unsigned* __restrict__ c0, unsigned* __restrict__ c1,
                                                   unsigned long long* __restrict__ sides) {
  const long long g = (long long)blockIdx.x * RS_WPB + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  unsigned n0 = 0, n1 = 0;
  if (g < nq) {  // uniform over the wave
    const int ci = rs_find<RS_KEY_RASTER>(cells, ncells, g);
    const RsCell& c = cells[ci];
    const int64_t n = rs_nodes(c);
    const bool odd = st[ci].k & 1;
    const int64_t i0 = (g - c.qb0) * RS_B + lane;
    const double* src = c.buf[odd ? 1 : 0];
    // every row's loads first: the copy's stores could alias later rows'
    // loads and would otherwise serialise them
    double v[RS_ROWS];
    int m[RS_ROWS];
#pragma unroll
    for (int e = 0; e < RS_ROWS; ++e) {
      const int64_t i = i0 + e * 64;
      v[e] = i < n ? src[i] : 0.0;
      m[e] = i < n ? (int)c.mask[i] : 2;
    }
    unsigned long long mine = 0;  // lane 2e / 2e + 1: row e's - / + side ballot
#pragma unroll
    for (int e = 0; e < RS_ROWS; ++e) {
      const int64_t i = i0 + e * 64;
      if (odd && i < n) c.buf[0][i] = v[e];
      const bool fin = fabs(v[e]) < c.inf;
      const unsigned long long b0 = __ballot(m[e] == 0 && fin), b1 = __ballot(m[e] == 1 && fin);
      n0 += (unsigned)__popcll(b0);
      n1 += (unsigned)__popcll(b1);
      if (lane == 2 * e) mine = b0;
      if (lane == 2 * e + 1) mine = b1;
    }
    if (lane < 2 * RS_ROWS) sides[g * (2 * RS_ROWS) + lane] = mine;
  }
  if (lane == 0 && g < nq1) {
    c0[g] = n0;
    c1[g] = n1;
  }
}

__device__ __forceinline__ bool rs_is_bc(const RsCell& c, int64_t i, dcl_icoor* pos) {
  if (i >= c.count) return false;
  const dcl_irregular_node& n = c.nodes[i];
  *pos = n.pos;
  return n.axis == -1 && ri_inside(c.w, c.d3, n.pos.x, n.pos.y, n.pos.z);
}

// boundary records per record block
__global__ __launch_bounds__(RS_B) void rs_bc_count_k(const RsCell* __restrict__ cells, int ncells, long long nr,
                                                      unsigned* __restrict__ counts) {
  const long long g = blockIdx.x;
  bool p = false;
  if (g < nr) {
    const RsCell& c = cells[rs_find<RS_KEY_RECORD>(cells, ncells, g)];
    dcl_icoor q;
    p = rs_is_bc(c, (g - c.rb0) * RS_B + threadIdx.x, &q);
  }
  const int cnt = __syncthreads_count(p);
  if (threadIdx.x == 0) counts[g] = (unsigned)cnt;
}

// the band of each level set: [boundary nodes in record order | - side |
// + side], each side in raster order
__global__ __launch_bounds__(RS_B) void rs_bc_write_k(const RsCell* __restrict__ cells, int ncells, long long nr,
                                                      const unsigned* __restrict__ rc,
                                                      const unsigned long long* __restrict__ rs) {
  __shared__ unsigned sh[RS_B / 64];
  const long long g = blockIdx.x;
  if (g >= nr) return;
  const RsCell& c = cells[rs_find<RS_KEY_RECORD>(cells, ncells, g)];
  dcl_icoor q = {0, 0, 0};
  const bool p = rs_is_bc(c, (g - c.rb0) * RS_B + threadIdx.x, &q);
  const unsigned r = rs_rank(p, sh);
  if (!p) return;
  const int64_t pos = rs_prefix(rc, rs, g) - rs_prefix(rc, rs, c.rb0) + r;
  if (pos < c.band_cap) c.band[pos] = q;
}

// the band nodes of raster block g, ranked by rs_final_k's ballots
__device__ __forceinline__ void rs_side_block(const RsCell* __restrict__ cells, int ncells, long long g, int lane,
                                              const unsigned* __restrict__ rc,
                                              const unsigned long long* __restrict__ rs,
                                              const unsigned* __restrict__ c0,
                                              const unsigned long long* __restrict__ s0,
                                              const unsigned* __restrict__ c1,
                                              const unsigned long long* __restrict__ s1,
                                              const unsigned long long* __restrict__ sides) {
  const RsCell& c = cells[rs_find<RS_KEY_RASTER>(cells, ncells, g)];
  const long long p0 = rs_prefix(c0, s0, g), p1 = rs_prefix(c1, s1, g);
  const long long nbc = rs_prefix(rc, rs, c.rb1) - rs_prefix(rc, rs, c.rb0);
  const long long n0 = rs_prefix(c0, s0, c.qb1) - rs_prefix(c0, s0, c.qb0);
  const long long base0 = nbc + p0 - rs_prefix(c0, s0, c.qb0);
  const long long base1 = nbc + n0 + p1 - rs_prefix(c1, s1, c.qb0);
  const int64_t plane = (int64_t)c.w.nx * c.w.ny;
  const int64_t i0 = (g - c.qb0) * RS_B + lane;
  const unsigned long long lt = (1ull << lane) - 1ull;  // the lanes below this one
  const unsigned long long* sb = sides + g * (2 * RS_ROWS);
  long long r0 = 0, r1 = 0;  // band nodes of each side in the rows before
#pragma unroll
  for (int e = 0; e < RS_ROWS; ++e) {
    const unsigned long long b0 = sb[2 * e], b1 = sb[2 * e + 1];
    const bool k0 = (b0 >> lane) & 1ull, k1 = (b1 >> lane) & 1ull;
    if (k0 || k1) {
      const int64_t pos = k0 ? base0 + r0 + __popcll(b0 & lt) : base1 + r1 + __popcll(b1 & lt);
      if (pos < c.band_cap) {
        const int64_t i = i0 + e * 64;
        const int z = c.d3 ? (int)(i / plane) : 0, rr = (int)(i - (int64_t)z * plane);
        const int y = rr / c.w.nx, x = rr - y * c.w.nx;
        dcl_icoor q;
        q.x = c.w.px + x;
        q.y = c.w.py + y;
        q.z = c.w.pz + z;
        c.band[pos] = q;
      }
    }
    r0 += __popcll(b0);
    r1 += __popcll(b1);
  }
}

// the two sides of the band, from the counts' scans and rs_final_k's
// ballots: one raster block per wave; a block without band nodes reads its
// two counts and stops
__global__ __launch_bounds__(RS_B) void rs_side_write_k(const RsCell* __restrict__ cells, int ncells, long long nq,
                                                        const unsigned* __restrict__ rc,
                                                        const unsigned long long* __restrict__ rs,
                                                        const unsigned* __restrict__ c0,
                                                        const unsigned long long* __restrict__ s0,
                                                        const unsigned* __restrict__ c1,
                                                        const unsigned long long* __restrict__ s1,
                                                        const unsigned long long* __restrict__ sides) {
  const long long g = (long long)blockIdx.x * RS_WPB + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (g >= nq) return;  // uniform over the wave; no block barrier below
  if (rs_prefix(c0, s0, g + 1) == rs_prefix(c0, s0, g) && rs_prefix(c1, s1, g + 1) == rs_prefix(c1, s1, g)) return;
  rs_side_block(cells, ncells, g, lane, rc, rs, c0, s0, c1, s1, sides);
}

// per level set: boundary nodes, - side, + side
__global__ __launch_bounds__(RS_B) void rs_totals_k(const RsCell* __restrict__ cells, int ncells,
                                                    const unsigned* __restrict__ rc,
                                                    const unsigned long long* __restrict__ rs,
                                                    const unsigned* __restrict__ c0,
                                                    const unsigned long long* __restrict__ s0,
                                                    const unsigned* __restrict__ c1,
                                                    const unsigned long long* __restrict__ s1,
                                                    unsigned long long* __restrict__ totals) {
  const int i = blockIdx.x * RS_B + threadIdx.x;
  if (i >= ncells) return;
  const RsCell& c = cells[i];
  totals[3 * i] = (unsigned long long)(rs_prefix(rc, rs, c.rb1) - rs_prefix(rc, rs, c.rb0));
  totals[3 * i + 1] = (unsigned long long)(rs_prefix(c0, s0, c.qb1) - rs_prefix(c0, s0, c.qb0));
  totals[3 * i + 2] = (unsigned long long)(rs_prefix(c1, s1, c.qb1) - rs_prefix(c1, s1, c.qb0));
}

static size_t rs_al(size_t b) { return (b + 255) / 256 * 256; }

}  // namespace dcl

using namespace dcl;

extern "C" int dcl_reinitialize_parallel(dcl_reinit_cell* cells, int ncells, int max_sweeps, int* sweeps,
                                         void* stream) {
  if (ncells < 0) return set_error(DCL_ERR_ARG_SIZ, "ncells < 0");
  if (ncells > 0 && !cells) return set_error(DCL_ERR_ARG_NULL, "cells is NULL");
  if (max_sweeps < 0) return set_error(DCL_ERR_ARG_SIZ, "max_sweeps < 0");
  if (ncells == 0) return 0;
  if (ncells > (1 << 20)) return set_error(DCL_ERR_ARG_SIZ, "at most 2^20 level sets per call");
  if (max_sweeps == 0) max_sweeps = 256;
  hipStream_t s = as_stream(stream);
  int d3 = -1;
  long long nodes = 0, nq = 0, nr = 0, nch = 0;
  size_t cell_bytes = 0;
  for (int i = 0; i < ncells; ++i) {
    const dcl_reinit_cell& u = cells[i];
    if (!u.phi) return set_error(DCL_ERR_ARG_NULL, "level set %d: phi is NULL", i);
    DCL_TRY(check_window(&u.win, "phi", 1));
    if (u.count < 0 || (u.count > 0 && !u.nodes))
      return set_error(DCL_ERR_ARG_NULL, "level set %d: bad irregular-node list", i);
    if (u.count > INT32_MAX) return set_error(DCL_ERR_ARG_SIZ, "level set %d: more than 2^31 - 1 records", i);
    if (u.band_capacity < 0 || (u.band_capacity > 0 && !u.band))
      return set_error(DCL_ERR_ARG_NULL, "level set %d: bad band output", i);
    if (!(u.band_width > 0) || !(u.phi_inf > u.band_width))
      return set_error(DCL_ERR_ARG_WRONG, "level set %d: need 0 < band_width < phi_inf", i);
    const int c3 = u.win.n.z >= 2;
    if (d3 >= 0 && c3 != d3) return set_error(DCL_ERR_ARG_WRONG, "a batch mixes 2D and 3D level sets");
    d3 = c3;
    const int64_t n = win_nodes(u.win);
    nodes += n;
    nq += (n + RS_B - 1) / RS_B;
    nch += (n + RS_CH - 1) / RS_CH;
    nr += (u.count + RS_B - 1) / RS_B;
    cell_bytes += rs_al(sizeof(double) * (size_t)n) + 3 * rs_al((size_t)n) +
                  2 * rs_al((size_t)((n + RS_CH - 1) / RS_CH));
  }
  if (nodes >= INT32_MAX || nr >= INT32_MAX)
    return set_error(DCL_ERR_ARG_SIZ, "a batch of more than 2^31 - 1 nodes or record blocks");
  // one more raster and record block, counting nothing: the scans' totals
  const long long nq1 = nq + 1, nr1 = nr + 1;
  const int nparts = ncells >= 4096 ? 1 : (4096 / ncells < 64 ? 4096 / ncells : 64);
  const int pstride = ncells < 16 ? 16 : ncells;
  const size_t bytes = rs_al(sizeof(RsCell) * ncells) + rs_al(sizeof(RsState) * ncells) +
                       rs_al(sizeof(unsigned long long) * (size_t)nparts * pstride) +
                       2 * rs_al(sizeof(int) * (size_t)(max_sweeps + 1)) + rs_al(sizeof(int2) * (size_t)nodes) +
                       rs_al(sizeof(unsigned long long) * 3 * (size_t)ncells) +
                       2 * rs_al(sizeof(unsigned) * (size_t)nq1) +
                       2 * rs_al(sizeof(unsigned long long) * (size_t)scan_tiles(nq1)) +
                       rs_al(sizeof(unsigned) * (size_t)nr1) +
                       rs_al(sizeof(unsigned long long) * (size_t)scan_tiles(nr1)) +
                       rs_al(sizeof(unsigned long long) * 3) +
                       rs_al(sizeof(unsigned long long) * 2 * RS_ROWS * (size_t)nq) + cell_bytes;
  void* sc = nullptr;
  DCL_TRY(scratch(bytes, &sc));
  char* base = static_cast<char*>(sc);
  auto take = [&](size_t b) {
    char* p = base;
    base += rs_al(b);
    return p;
  };
  RsCell* dcells = reinterpret_cast<RsCell*>(take(sizeof(RsCell) * ncells));
  RsState* dstate = reinterpret_cast<RsState*>(take(sizeof(RsState) * ncells));
  unsigned long long* parts =
      reinterpret_cast<unsigned long long*>(take(sizeof(unsigned long long) * (size_t)nparts * pstride));
  int* active = reinterpret_cast<int*>(take(sizeof(int) * (size_t)(max_sweeps + 1)));
  int* ncount = reinterpret_cast<int*>(take(sizeof(int) * (size_t)(max_sweeps + 1)));
  int2* nlist = reinterpret_cast<int2*>(take(sizeof(int2) * (size_t)nodes));
  unsigned long long* totals = reinterpret_cast<unsigned long long*>(take(sizeof(unsigned long long) * 3 * ncells));
  unsigned* c0 = reinterpret_cast<unsigned*>(take(sizeof(unsigned) * (size_t)nq1));
  unsigned* c1 = reinterpret_cast<unsigned*>(take(sizeof(unsigned) * (size_t)nq1));
  unsigned long long* s0 = reinterpret_cast<unsigned long long*>(take(sizeof(unsigned long long) * scan_tiles(nq1)));
  unsigned long long* s1 = reinterpret_cast<unsigned long long*>(take(sizeof(unsigned long long) * scan_tiles(nq1)));
  unsigned* rc = reinterpret_cast<unsigned*>(take(sizeof(unsigned) * (size_t)nr1));
  unsigned long long* rsum = reinterpret_cast<unsigned long long*>(take(sizeof(unsigned long long) * scan_tiles(nr1)));
  unsigned long long* grand = reinterpret_cast<unsigned long long*>(take(sizeof(unsigned long long) * 3));
  unsigned long long* sides =
      reinterpret_cast<unsigned long long*>(take(sizeof(unsigned long long) * 2 * RS_ROWS * (size_t)nq));

  RsCell* host = static_cast<RsCell*>(malloc(sizeof(RsCell) * ncells));
  RsState* hstate = static_cast<RsState*>(malloc(sizeof(RsState) * ncells));
  unsigned long long* htot = static_cast<unsigned long long*>(malloc(sizeof(unsigned long long) * 3 * ncells));
  if (!host || !hstate || !htot) {
    free(host);
    free(hstate);
    free(htot);
    return set_error(DCL_ERR_MEM, "host memory");
  }
  long long q0 = 0, r0 = 0, h0 = 0;
  for (int i = 0; i < ncells; ++i) {
    const dcl_reinit_cell& u = cells[i];
    RsCell& c = host[i];
    const int64_t n = win_nodes(u.win);
    c.buf[0] = static_cast<double*>(u.phi);
    c.buf[1] = reinterpret_cast<double*>(take(sizeof(double) * (size_t)n));
    c.mask = reinterpret_cast<unsigned char*>(take((size_t)n));
    c.nd[0] = reinterpret_cast<unsigned char*>(take((size_t)n));
    c.nd[1] = reinterpret_cast<unsigned char*>(take((size_t)n));
    c.cd[0] = reinterpret_cast<unsigned char*>(take((size_t)((n + RS_CH - 1) / RS_CH)));
    c.cd[1] = reinterpret_cast<unsigned char*>(take((size_t)((n + RS_CH - 1) / RS_CH)));
    c.w = kwin(u.win);
    c.d3 = d3;
    c.bw = u.band_width;
    c.inf = u.phi_inf;
    c.tol = u.band_width * RS_TOL;
    c.qb0 = q0;
    q0 += (n + RS_B - 1) / RS_B;
    c.qb1 = q0;
    c.cb0 = h0;
    h0 += (n + RS_CH - 1) / RS_CH;
    c.rb0 = r0;
    r0 += (u.count + RS_B - 1) / RS_B;
    c.rb1 = r0;
    c.nodes = u.nodes;
    c.count = u.count;
    c.band = u.band;
    c.band_cap = u.band_capacity;
  }
  int rc_ = 0;
  {
    hipError_t e = hipMemcpyAsync(dcells, host, sizeof(RsCell) * ncells, hipMemcpyHostToDevice, s);
    if (e != hipSuccess) rc_ = hip_fail(e, "reinit upload", __FILE__, __LINE__);
  }
  if (!rc_) {
    hipLaunchKernelGGL(rs_reset_k, dim3((unsigned)nq), dim3(RS_B), 0, s, dcells, ncells, nq,
                       RsStart{dstate, active, ncount, parts, ncells, max_sweeps + 1, nparts * pstride});
    if (nr > 0) {
      if (d3) hipLaunchKernelGGL(rs_bc_k<3>, dim3((unsigned)nr), dim3(RS_B), 0, s, dcells, ncells, nr);
      else hipLaunchKernelGGL(rs_bc_k<2>, dim3((unsigned)nr), dim3(RS_B), 0, s, dcells, ncells, nr);
    }
    if (hipGetLastError() != hipSuccess) rc_ = set_error(DCL_ERR_LIB, "reinit reset / boundary launch failed");
  }
  // the sweeps, in groups of RS_GROUP: once a group is queued, the count of
  // level sets still sweeping late in the group before it is awaited (through
  // pinned memory), so the GPU always holds the next group; a level set
  // that has settled skips the sweeps queued after it
  static thread_local int* pin = nullptr;
  if (!pin && !rc_) {
    hipError_t e = hipHostMalloc(reinterpret_cast<void**>(&pin), 2 * sizeof(int), hipHostMallocDefault);
    if (e != hipSuccess) {
      pin = nullptr;
      rc_ = hip_fail(e, "reinit pinned count", __FILE__, __LINE__);
    }
  }
  hipEvent_t ev[2] = {nullptr, nullptr};
  for (int q = 0; q < 2 && !rc_; ++q) {
    hipError_t e = hipEventCreateWithFlags(&ev[q], hipEventDisableTiming);
    if (e != hipSuccess) rc_ = hip_fail(e, "reinit events", __FILE__, __LINE__);
  }
  const unsigned ng = (unsigned)(nch < RS_NEED_GRID ? nch : RS_NEED_GRID), nst = grid1d(ncells, RS_B / 64);
  bool settled = false;
  for (int j0 = 0, grp = 0; j0 < max_sweeps && !rc_ && !settled; j0 += RS_GROUP, ++grp) {
    const int j1 = j0 + RS_GROUP < max_sweeps ? j0 + RS_GROUP : max_sweeps;
    for (int j = j0; j < j1; ++j) {
      // with the state after sweep j - 1, into active[j - 1]
      hipLaunchKernelGGL(rs_need_k, dim3(ng + (j > 0 ? nst : 0u)), dim3(RS_B), 0, s, dcells, ncells, dstate, nch, j,
                         (int)ng, nlist, ncount + j, max_sweeps, active + (j > 0 ? j - 1 : 0), parts, nparts, pstride);
      if (d3)
        hipLaunchKernelGGL(rs_update_k<3>, dim3(RS_GRID), dim3(RS_B), 0, s, dcells, dstate, nlist, ncount + j, parts,
                           nparts, pstride);
      else
        hipLaunchKernelGGL(rs_update_k<2>, dim3(RS_GRID), dim3(RS_B), 0, s, dcells, dstate, nlist, ncount + j, parts,
                           nparts, pstride);
    }
    if (hipGetLastError() != hipSuccess) {
      rc_ = set_error(DCL_ERR_LIB, "reinit sweep launch failed");
      break;
    }
    if (j1 < 2) continue;
    hipError_t e = hipMemcpyAsync(pin + (grp & 1), active + (j1 - 2), sizeof(int), hipMemcpyDeviceToHost, s);
    if (e == hipSuccess) e = hipEventRecord(ev[grp & 1], s);
    if (e == hipSuccess && grp > 0) {
      e = hipEventSynchronize(ev[(grp - 1) & 1]);
      if (e == hipSuccess && pin[(grp - 1) & 1] == 0) settled = true;
    }
    if (e != hipSuccess) rc_ = hip_fail(e, "reinit sweeps", __FILE__, __LINE__);
  }
  if (!rc_ && !settled) {  // the last sweep's state
    hipLaunchKernelGGL(rs_state_k, dim3(nst), dim3(RS_B), 0, s, dstate, ncells, max_sweeps, active + (max_sweeps - 1),
                       parts, nparts, pstride);
    if (hipGetLastError() != hipSuccess) rc_ = set_error(DCL_ERR_LIB, "reinit state launch failed");
  }
  for (int q = 0; q < 2; ++q)
    if (ev[q]) (void)hipEventDestroy(ev[q]);
  if (!rc_) {
    hipError_t e = hipMemcpyAsync(hstate, dstate, sizeof(RsState) * ncells, hipMemcpyDeviceToHost, s);
    if (e == hipSuccess) e = hipStreamSynchronize(s);
    if (e != hipSuccess) rc_ = hip_fail(e, "reinit sweeps", __FILE__, __LINE__);
  }
  for (int i = 0; i < ncells && !rc_; ++i) {
    const RsState& q = hstate[i];
    if (sweeps) sweeps[i] = q.k;
    if (q.done == RS_NAN) rc_ = set_error(DCL_ERR_LIB, "level set %d: NaN in a reinitialisation update", i);
    else if (q.done != RS_SETTLED)
      rc_ = set_error(DCL_ERR_LIB, "level set %d: reinitialisation did not settle in %d sweeps", i, max_sweeps);
  }
  // the result, then the band
  if (!rc_) {
    hipLaunchKernelGGL(rs_final_k, dim3((unsigned)((nq1 + RS_WPB - 1) / RS_WPB)), dim3(RS_B), 0, s, dcells,
                       ncells, nq, nq1, dstate, c0, c1, sides);
    hipLaunchKernelGGL(rs_bc_count_k, dim3((unsigned)nr1), dim3(RS_B), 0, s, dcells, ncells, nr, rc);
    if (hipGetLastError() != hipSuccess) rc_ = set_error(DCL_ERR_LIB, "reinit band launch failed");
  }
  if (!rc_) {
    const ScanArrays sn = {{c0, c1}, {s0, s1}, {grand, grand + 1}};
    rc_ = scan_counts(sn, 2, nq1, s);
  }
  if (!rc_) {
    const ScanArrays sr = {{rc, nullptr}, {rsum, nullptr}, {grand + 2, nullptr}};
    rc_ = scan_counts(sr, 1, nr1, s);
  }
  if (!rc_) {
    if (nr > 0) hipLaunchKernelGGL(rs_bc_write_k, dim3((unsigned)nr), dim3(RS_B), 0, s, dcells, ncells, nr, rc, rsum);
    hipLaunchKernelGGL(rs_side_write_k, dim3((unsigned)((nq + RS_WPB - 1) / RS_WPB)), dim3(RS_B), 0, s, dcells,
                       ncells, nq, rc, rsum, c0, s0, c1, s1, sides);
    hipLaunchKernelGGL(rs_totals_k, dim3(grid1d(ncells, RS_B)), dim3(RS_B), 0, s, dcells, ncells, rc, rsum, c0, s0,
                       c1, s1, totals);
    if (hipGetLastError() != hipSuccess) rc_ = set_error(DCL_ERR_LIB, "reinit band launch failed");
  }
  if (!rc_) {
    hipError_t e = hipMemcpyAsync(htot, totals, sizeof(unsigned long long) * 3 * ncells, hipMemcpyDeviceToHost, s);
    if (e == hipSuccess) e = hipStreamSynchronize(s);
    if (e != hipSuccess) rc_ = hip_fail(e, "reinit band", __FILE__, __LINE__);
  }
  for (int i = 0; i < ncells && !rc_; ++i)
    cells[i].band_count = (int64_t)(htot[3 * i] + htot[3 * i + 1] + htot[3 * i + 2]);
  if (rc_) (void)hipStreamSynchronize(s);
  free(host);
  free(hstate);
  free(htot);
  return rc_;
}
