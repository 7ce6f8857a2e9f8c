// reinit.hip -- reinitialisation on gfx950: LevelSetReinitialize
// (LevelSetMethod/FastMarching.c:10-146) with the second-order neighbour
// updates of FastMarching3D.c:14-101 / FastMarching2D.c:33-185 and the
// binary min-heap of Common/Heap.c:59-139.
//
// The fast marching method accepts nodes one at a time in heap order, and
// which neighbours count as known when a node is updated (first or second
// order, which side) depends on that order, equal keys included.  The GPU
// keeps that order exactly: one wave runs one sign pass of one level set
// with the reference's heap (the same comparisons, so equal keys pop in the
// same order), and the lanes compute the updates of the accepted node's
// neighbours side by side.  The parallelism is across passes and level sets:
// the - pass writes only nodes whose phi is -PHI_INF and reads only
// non-negative values of -phi (the + pass the mirror image), so the two
// passes of a level set run as two concurrent waves with the same result as
// the reference's sequential order, and a batch of level sets (DCell's
// cells) runs as 2 x ncells waves.
//
// Steps: reset phi to +-PHI_INF (reinit_reset_k), write the boundary values
// at the projection records (reinit_bc_k), then the passes (reinit_fmm_k);
// the - pass also lists the boundary nodes in record order.  The band is
// assembled as [boundary nodes | - pass | + pass] by copies.
//
// Departures from the reference, where it reads out of bounds or leaves a
// value unset: a neighbour outside the window is not pushed and a record
// outside it is skipped (the reference reads them unchecked; LevelSetResize
// keeps the band away from the edge), a pushed 2D node's z is the window's
// (the reference leaves it unset), and a NaN update or a full heap stops the
// pass with an error instead of exiting.
//
// One accepted node is a chain of dependent steps, so the wave shortens the
// chain: the heap's sifts are done by all lanes at once (a pop compares six
// levels of siblings per LDS round trip and follows the ballot; an insert
// reads all ancestors of the new slot together), with the same comparisons
// and the same final heap as the reference's one-level-at-a-time loops, and
// the popped node's value and its neighbours' stencils are loaded before the
// sift, one lane per neighbour and axis.  Measured on 24 level sets of edges
// 32 to 64 (FP64): 345 ms with lane 0 sifting, 67 ms; what is left is the
// latency of one wave's instructions (about 1000 cycles per pop, 465 per
// insert, 880 per accepted node's updates).  One wave fills a CU's LDS, so
// more than 128 level sets run in rounds: 256 of edges 32 to 64 462 -> 146 ms,
// 300 of 32 to 40 325 -> 92 ms.
//
// The heap's first 13311 slots sit in LDS, where nearly every pop and push
// spends most of its steps; deeper ones are in memory.
#include <math.h>

#include "dcl_host.hpp"
#include "dcl_reinit.hpp"

namespace dcl {

// a heap entry: the tentative value and the node: its offset in the window
// (below 2^31), and RI_INNER where it is 3 or more nodes from every face of
// the window, so that every value its push reads is there
constexpr unsigned RI_INNER = 0x80000000u;
struct RiEntry {
  double v;
  unsigned key;
};

// The heap: slots 1 .. RI_LDS - 1 in LDS (values and keys apart, 156 KB: one
// wave per CU), the deeper ones in memory.  IN_LDS: the caller knows that
// every slot it uses is in LDS.
constexpr unsigned RI_LDS = 13312;
struct __align__(16) RiLds {  // the keys first: both arrays within reach of a 16-bit offset
  unsigned k[RI_LDS];
  double v[RI_LDS];
};
static_assert(sizeof(RiLds::k) < 65536 && sizeof(RiLds::k) % 16 == 0, "the values' offset in LDS");
struct RiSlot {  // an entry in memory
  double v;
  unsigned long long key;
};
struct RiHeap {
  double* lv;
  unsigned* lk;
  __attribute__((address_space(1))) RiSlot* mem;
  template <bool IN_LDS>
  __device__ __forceinline__ RiEntry get(unsigned i) const {
    RiEntry e;
    if (IN_LDS || i < RI_LDS) {
      e.v = lv[i];
      e.key = lk[i];
    } else {
      e.v = mem[i].v;
      e.key = (unsigned)mem[i].key;
    }
    return e;
  }
  // slots i (even) and i + 1, both in LDS
  __device__ __forceinline__ void pair(unsigned i, RiEntry& a, RiEntry& b) const {
    typedef double f64x2 __attribute__((ext_vector_type(2)));
    typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
    const f64x2 v = *reinterpret_cast<const f64x2*>(lv + i);
    const u32x2 k = *reinterpret_cast<const u32x2*>(lk + i);
    a.v = v.x, a.key = k.x;
    b.v = v.y, b.key = k.y;
  }
  template <bool IN_LDS>
  __device__ __forceinline__ void set(unsigned i, const RiEntry& e) const {
    if (IN_LDS || i < RI_LDS) {
      lv[i] = e.v;
      lk[i] = e.key;
    } else {
      mem[i].v = e.v;
      mem[i].key = e.key;
    }
  }
};

// unsigned division by a constant of the launch, exact for numerators below
// 2^31 (round-up multiplier: 2^(l-1) < d <= 2^l, mul = ceil(2^(31+l) / d))
struct RiDiv {
  unsigned mul, shift;
  __device__ __forceinline__ unsigned operator()(unsigned n) const {
    return (unsigned)(((unsigned long long)n * mul) >> shift);
  }
};
__device__ __forceinline__ RiDiv ri_div(unsigned d) {
  RiDiv r;
  int l = 0;
  while ((1u << l) < d) ++l;
  r.mul = (unsigned)(((1ull << (31 + l)) + d - 1) / d);
  r.shift = 31 + l;
  return r;
}

struct RiCell {
  double* phi;
  KWin w;
  int d3;
  const dcl_irregular_node* nodes;
  int64_t count;
  double bw, inf;
  RiSlot* heap[2];
  int64_t heap_cap;
  dcl_icoor* list[3];  // boundary nodes, - pass, + pass
  int64_t list_cap;
  long long* stat;  // boundary count, - pass count, + pass count, error
};

enum { RI_OK = 0, RI_NAN = 1, RI_HEAP = 2, RI_STEPS = 3 };

__global__ __launch_bounds__(256) void reinit_reset_k(double* __restrict__ phi, int64_t n, double inf) {
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) {
    const double v = phi[i];
    phi[i] = v > 0 ? inf : -inf;
  }
}

// FMM_InitializeEikonal (FastMarching.c:60-74): phi at each projection record
// is the signed distance to its orthogonal projection
__global__ __launch_bounds__(256) void reinit_bc_k(RiCell c) {
#pragma clang fp contract(off)
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= c.count) return;
  const dcl_irregular_node n = c.nodes[i];
  if (n.axis != -1) return;
  if (!ri_inside(c.w, c.d3, n.pos.x, n.pos.y, n.pos.z)) return;
  const double r = c.d3 ? sqrt(n.op.x * n.op.x + n.op.y * n.op.y + n.op.z * n.op.z)
                         : sqrt(n.op.x * n.op.x + n.op.y * n.op.y);
  c.phi[ri_index(c.w, c.d3, n.pos.x, n.pos.y, n.pos.z)] = n.sign_center * r;
}

// phi as this pass sees it.  Lane 0 of the wave writes the accepted nodes
// and other lanes read them back: accesses of one wave reach its CU's L1 in
// order, so a wavefront-scope fence (ri_wave_sync) is all that needs.  The
// other pass may write nodes of the opposite sign at any time; whether a
// read sees the old -+PHI_INF or the new value, it is of the opposite sign,
// which this pass treats the same either way, so no wider coherence is
// needed.
//
// The pointers come from a table in memory, so the compiler takes them for
// flat ones, and a flat load is also waited for by every wait for LDS: the
// accesses name the global address space.
#define RI_GLOBAL __attribute__((address_space(1)))
__device__ __forceinline__ double ri_load(const double* p) {
  return __hip_atomic_load((const RI_GLOBAL double*)p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
__device__ __forceinline__ void ri_store(double* p, double v) {
  __hip_atomic_store((RI_GLOBAL double*)p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// writes of one lane (LDS, memory) visible to the other lanes of its wave
__device__ __forceinline__ void ri_wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

__device__ __forceinline__ double ri_lane_f64(double v, int lane) {
  const unsigned long long b = (unsigned long long)__double_as_longlong(v);
  const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)b, lane);
  const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)(b >> 32), lane);
  return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

// The end of a path that read heap slots in memory: its loads are done, so
// that the code after it, which the LDS-only path also runs, has no reason to
// wait for the loads and stores of phi that are in flight.
__device__ __forceinline__ void ri_mem_done() { __builtin_amdgcn_s_waitcnt(0x0f70); }  // vmcnt(0)

// HeapInsert (Common/Heap.c:59-91), all lanes of the wave: lane t compares
// the item with the t-th ancestor of the new slot c.  The item rises to the
// first ancestor below it; the ancestors it passes each move down one slot.
template <bool IN_LDS>
__device__ __forceinline__ void ri_heap_insert_at(const RiHeap& H, unsigned c, const RiEntry& item) {
  const int lane = threadIdx.x;
  const int depth = 31 - __builtin_clz(c);  // ancestors of slot c
  const unsigned slot = c >> (lane & 31);   // lanes past the root: slot 0, read and not used
  const RiEntry parent = H.get<IN_LDS>(slot >> 1);
  // the root stops the item at the latest
  const uint64_t stops = __builtin_amdgcn_ballot_w64(parent.v - item.v < 0) | (~0ull << depth);
  const int stop = __builtin_ctzll(stops);
  ri_wave_sync();  // every lane has read its parent before any slot changes
  RiEntry e;
  e.v = lane == stop ? item.v : parent.v;
  e.key = lane == stop ? item.key : parent.key;
  if (lane <= stop) H.set<IN_LDS>(slot, e);
  if (!IN_LDS) ri_mem_done();
  ri_wave_sync();
}
__device__ __forceinline__ void ri_heap_insert(const RiHeap& H, unsigned& len, const RiEntry& item) {
  const unsigned c = len++;
  if (c < RI_LDS) ri_heap_insert_at<true>(H, c, item);
  else ri_heap_insert_at<false>(H, c, item);
}

// What a lane holds through the whole pass.  Lane j (1 .. 63) stands for the
// j-th node, in breadth-first order, of a subtree of six levels that a pop
// works at a time; lane 8 n + 2 a + d, a below the dimension, works neighbour
// n (STAR order) of an accepted node along axis a, towards + (d = 0) or -.
struct RiLane {
  int depth1;      // depth of node j's children below the subtree's root
  unsigned pos2;   // the left child's place among the nodes of that depth
  int parent;      // j / 2
  uint64_t line;   // bits of j and its ancestors but the root
  uint64_t above;  // bits of its ancestors, the root among them
  bool on;         // the lane has a neighbour and an axis
  bool back;       // its first value is the accepted node itself
  int axis, dir;
  int dx, dy, dz;  // the neighbour's offset
  int delta, st;   // the same as an offset in the window, and the step along the axis
};

// HeapPop (Common/Heap.c:94-139) of a heap of at least one entry, all lanes
// of the wave; the top itself is read by the caller.  The reference moves the
// last entry (bubble) down from the root along the smaller child (the left
// one where the right is not below it) while it is above that child.  Here a
// round takes six levels: every lane compares its node's children and the
// smaller one with bubble, two ballots carry the outcomes to all lanes, and
// a lane whose ancestors all lead to it without stopping bubble knows that
// its node is on the path: it takes up its smaller child, or bubble where
// that stops it.  A heap of 8192 entries is two rounds, each one LDS round
// trip.
//
// One round from the subtree's root; true when bubble has found its slot,
// else root is the next one's.  A missing child counts as above everything.
template <bool IN_LDS>
__device__ __forceinline__ bool ri_pop_round(const RiHeap& H, const RiLane& t, const RiEntry& bubble, unsigned len,
                                             unsigned& root) {
  // the left child's slot (past LDS and the heap's end it may pass 32 bits)
  const uint64_t at = IN_LDS ? (uint64_t)((root << t.depth1) + t.pos2) : ((uint64_t)root << t.depth1) + t.pos2;
  const bool has = at < len, both = at + 1 < len;
  const unsigned left = (unsigned)at, node = left >> 1;
  RiEntry l, r;
  if (IN_LDS) {
    H.pair(left < RI_LDS - 2 ? left : RI_LDS - 2, l, r);
  } else {
    l = H.get<false>(has ? left : 0u);
    r = H.get<false>(both ? left + 1 : 1u);
  }
  l.v = has ? l.v : INFINITY;
  r.v = both ? r.v : INFINITY;
  const bool right = r.v - l.v < 0;
  const uint64_t rm = __builtin_amdgcn_ballot_w64(right);
  RiEntry e;
  e.v = right ? r.v : l.v;
  e.key = right ? r.key : l.key;
  // An infinite bubble (a tentative value that overflowed) stops above an
  // infinite or a missing child, where the difference is NaN; the reference
  // goes on past an infinite one, which moves infinite entries only, and these
  // are never accepted.
  const bool stop = !(bubble.v - e.v > 0);
  const uint64_t sm = __builtin_amdgcn_ballot_w64(stop);
  // the node is its parent's smaller child
  const uint64_t cm =
      __builtin_amdgcn_ballot_w64(((unsigned)(rm >> t.parent) & 1u) == (unsigned)(threadIdx.x & 1));
  const bool led = (cm & t.line) == t.line, free = (sm & t.above) == 0;
  const uint64_t path = __builtin_amdgcn_ballot_w64(led) & __builtin_amdgcn_ballot_w64(free);
  const int last = 63 - __builtin_clzll(path);
  root = 2 * (unsigned)__builtin_amdgcn_readlane((int)node, last) + ((unsigned)(rm >> last) & 1u);
  ri_wave_sync();  // every lane has read its children before any slot changes
  e.v = stop ? bubble.v : e.v;
  e.key = stop ? bubble.key : e.key;
  if (led & free) H.set<IN_LDS>(node, e);
  return (sm >> last) & 1ull;
}
template <bool IN_LDS>
__device__ __forceinline__ void ri_heap_pop_of(const RiHeap& H, const RiLane& t, unsigned len) {
  const RiEntry bubble = H.get<IN_LDS>(len);
  unsigned root = 1;
  if (IN_LDS) {  // at most 13 levels below the root
    if (!ri_pop_round<true>(H, t, bubble, len, root))
      if (!ri_pop_round<true>(H, t, bubble, len, root)) ri_pop_round<true>(H, t, bubble, len, root);
  } else {
    while (!ri_pop_round<false>(H, t, bubble, len, root)) {
    }
    ri_mem_done();
  }
  ri_wave_sync();
}
static_assert(RI_LDS <= 1u << 14, "a pop in LDS takes three rounds at most");
__device__ __forceinline__ void ri_heap_pop(const RiHeap& H, const RiLane& t, unsigned& hlen) {
  const unsigned len = --hlen;
  if (len == 1) return;
  if (len < RI_LDS) ri_heap_pop_of<true>(H, t, len);
  else ri_heap_pop_of<false>(H, t, len);
}

// STAR (Common/Common.h:49-51)
__device__ __forceinline__ int ri_star(int n, int a) { return (n >> 1) == a ? ((n & 1) ? -1 : 1) : 0; }

template <int NN>
__device__ __forceinline__ RiLane ri_lane(const KWin& w, int lane) {
  constexpr int DIM = NN == 6 ? 3 : 2;
  RiLane t;
  // lane 0 stands for no node: its children lie past any heap, and it is on
  // no path (two siblings are never both the smaller one)
  const int depth = 31 - __builtin_clz((unsigned)(lane | 1));
  t.depth1 = depth + 1;
  t.pos2 = lane ? 2 * ((unsigned)lane - (1u << depth)) : 0x80000000u;
  t.parent = lane >> 1;
  t.line = lane ? 0 : ~0ull;
  t.above = 0;
  for (int j = lane; j > 1; j >>= 1) {
    t.line |= 1ull << j;
    t.above |= 1ull << (j >> 1);
  }
  const int n = lane >> 3, a = (lane >> 1) & 3, d = lane & 1;
  t.on = n < NN && a < DIM;
  t.back = t.on && a == n >> 1 && d != (n & 1);
  t.axis = a;
  t.dir = d ? -1 : 1;
  t.dx = t.on ? ri_star(n, 0) : 0;
  t.dy = t.on ? ri_star(n, 1) : 0;
  t.dz = t.on && DIM == 3 ? ri_star(n, 2) : 0;
  t.delta = (t.dz * w.ny + t.dy) * w.nx + t.dx;
  t.st = !t.on ? 0 : t.dir * (a == 0 ? 1 : a == 1 ? w.nx : w.nx * w.ny);
  return t;
}

// What a lane holds of a push (FMM_PushNeighbors3D / 2D) of the node at
// offset id, (lx, ly, lz) in the window: the values of its neighbour and of
// the two nodes beyond it along its axis and direction (phi itself; the pass
// sees sign * phi, and PHI_INF outside the window).
struct RiSten {
  double raw[3];
  bool has[3];  // the node lies in the window
  bool in;      // the neighbour does
};

// inner: every value is there, the coordinates are not used.  Every lane
// loads (the node itself where it has nothing to load), so that nothing
// waits between the loads.
template <int NN>
__device__ __forceinline__ RiSten ri_sten(const RiCell& c, const RiLane& t, int id, int lx, int ly, int lz,
                                          bool inner) {
  constexpr int DIM = NN == 6 ? 3 : 2;
  RiSten s;
  int at[3];
  if (inner) {
    s.in = t.on;
#pragma unroll
    for (int m = 0; m < 3; ++m) {
      s.has[m] = true;
      at[m] = id + t.delta + m * t.st;
    }
  } else {
    const int x = lx + t.dx, y = ly + t.dy, z = lz + t.dz;
    s.in = t.on && (unsigned)x < (unsigned)c.w.nx && (unsigned)y < (unsigned)c.w.ny &&
           (DIM == 2 || (unsigned)z < (unsigned)c.w.nz);
    const int p = t.axis == 0 ? x : t.axis == 1 ? y : z;
    const int ext = !s.in ? 0 : t.axis == 0 ? c.w.nx : t.axis == 1 ? c.w.ny : c.w.nz;
#pragma unroll
    for (int m = 0; m < 3; ++m) {
      s.has[m] = (unsigned)(p + m * t.dir) < (unsigned)ext;
      at[m] = s.has[m] ? id + t.delta + m * t.st : id;
    }
  }
#pragma unroll
  for (int m = 0; m < 3; ++m) s.raw[m] = ri_load(c.phi + at[m]);
  return s;
}

// v of the lane that CTRL names for this one (DPP: quad_perm 0x00 .. 0xff,
// row_shl:k 0x100 + k)
template <int CTRL>
__device__ __forceinline__ double ri_dpp(double v) {
  const unsigned long long b = (unsigned long long)__double_as_longlong(v);
  const int lo = __builtin_amdgcn_mov_dpp((int)(unsigned)b, CTRL, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_mov_dpp((int)(unsigned)(b >> 32), CTRL, 0xf, 0xf, true);
  return __longlong_as_double((long long)(((unsigned long long)(unsigned)hi << 32) | (unsigned)lo));
}

// the value pushed to neighbour n, in lane 8 n; valid and nan there as the
// reference decides them.  back: the accepted node got the value v after the
// loads.  One direction of AccumulateCoef (FastMarching2D.c:33-94) per lane,
// the larger of the two taken by the even lanes, then the sums over the axes
// in axis order.
template <int NN>
__device__ __forceinline__ double ri_update(const RiCell& c, int sign, const RiLane& t, const RiSten& s, bool back,
                                            double v, bool& valid, bool& nan) {
#pragma clang fp contract(off)
  const double inf = c.inf;
  const double p0 = s.has[0] ? sign * s.raw[0] : inf;
  double p1 = s.has[1] ? sign * s.raw[1] : inf;
  const double p2 = s.has[2] ? sign * s.raw[2] : inf;
  if (back) p1 = v;
  valid = s.in && !(p0 < c.bw);
  const double D2 = (3 * p0 - 4 * p1 + p2) / 2.;
  const double D1 = p0 - p1;
  const bool known = (0 <= p1) & (p1 < inf);
  const bool second = known & (0 <= p2) & (p2 < inf) & (D2 > 0), first = known & (D1 > 0);
  const double q = (4 * p1 - p2) / 3;
  double a = second ? 9. / 4. : first ? 1. : 0.;
  double b = second ? -9. / 2. * q : first ? -2. * p1 : 0.;
  double cc = second ? 9. / 4. * q * q : first ? p1 * p1 : 0.;
  const double D = second ? D2 : first ? D1 : 0.;
  // quad_perm [1,0,3,2]: the other direction's
  const double ao = ri_dpp<0xb1>(a), bo = ri_dpp<0xb1>(b), co = ri_dpp<0xb1>(cc), Do = ri_dpp<0xb1>(D);
  const bool minus = Do > D;  // in the even lanes
  a = minus ? ao : a;
  b = minus ? bo : b;
  cc = minus ? co : cc;
  // axis 0, 1, 2 of neighbour n: lanes 8 n, 8 n + 2 and 8 n + 4
  double A = 0, B = 0, C = -1;
  A += a;
  B += b;
  C += cc;
  A += ri_dpp<0xaa>(a);
  B += ri_dpp<0xaa>(b);
  C += ri_dpp<0xaa>(cc);
  if (NN == 6) {
    A += ri_dpp<0x104>(a);
    B += ri_dpp<0x104>(b);
    C += ri_dpp<0x104>(cc);
  }
  const double disc = sqrt(B * B - 4 * A * C);
  double d1 = (-B + disc) / (2 * A);
  if (valid && d1 != d1) d1 = -B / (2 * A);
  nan = valid && d1 != d1;
  return d1;
}

// the lanes 8 n, where ri_update leaves neighbour n's results
constexpr uint64_t RI_LEAD = 0x0101010101010101ull;

// the heap key of the lane's neighbour of the node at (lx, ly, lz), offset id
template <int NN>
__device__ __forceinline__ unsigned ri_key(const KWin& w, const RiLane& t, int id, int lx, int ly, int lz) {
  const int x = lx + t.dx, y = ly + t.dy, z = lz + t.dz;
  const bool inner = x >= 3 && x <= w.nx - 4 && y >= 3 && y <= w.ny - 4 && (NN == 4 || (z >= 3 && z <= w.nz - 4));
  return (unsigned)(id + t.delta) | (inner ? RI_INNER : 0u);
}

// the inserts of one push in STAR order: d1 and key of neighbour n in lane
// 8 n, valid their mask
__device__ __forceinline__ int ri_insert_all(unsigned cap, unsigned key, double d1, uint64_t valid, const RiHeap& H,
                                             unsigned& hlen) {
#pragma unroll 1
  for (uint64_t m = valid; m; m &= m - 1) {
    const int q = __builtin_ctzll(m);
    RiEntry e;
    e.v = ri_lane_f64(d1, q);
    e.key = (unsigned)__builtin_amdgcn_readlane((int)key, q);
    if (hlen >= cap) return RI_HEAP;
    ri_heap_insert(H, hlen, e);
  }
  return RI_OK;
}

// one wave per (level set, sign): FMM_InitializeEikonal's pushes
// (FastMarching.c:76-93) and FMM_SolveEikonal (:97-146)
template <int NN>
__global__ __launch_bounds__(64) void reinit_fmm_k(const RiCell* __restrict__ cells) {
#pragma clang fp contract(off)
  const RiCell c = cells[blockIdx.x >> 1];
  const int pass = blockIdx.x & 1;
  const int sign = pass ? 1 : -1;
  const int lane = threadIdx.x;
  __shared__ RiLds lds;
  double* lds_v = lds.v;
  unsigned* lds_k = lds.k;
  const RiHeap H = {lds_v, lds_k, (RI_GLOBAL RiSlot*)(pass ? c.heap[1] : c.heap[0])};
  dcl_icoor* accepted = pass ? c.list[2] : c.list[1];
  // heap slots are 32-bit (a heap of 2^31 entries is 32 GB, hours of pushes)
  const unsigned cap = (unsigned)(c.heap_cap < 0x7fffffff ? c.heap_cap : 0x7fffffff);
  const RiLane tl = ri_lane<NN>(c.w, lane);
  const RiDiv by_row = ri_div((unsigned)c.w.nx), by_plane = ri_div((unsigned)(c.w.nx * c.w.ny));
  unsigned hlen = 1;
  int64_t nbc = 0, nacc = 0;
  int err = RI_OK;
  // the boundary nodes, in record order
  for (int64_t base = 0; base < c.count && err == RI_OK; base += 64) {
    const int64_t r = base + lane;
    bool bc = false;
    int x = 0, y = 0, z = 0;
    double v = -1.0;
    if (r < c.count) {
      const dcl_irregular_node n = c.nodes[r];
      bc = n.axis == -1 && ri_inside(c.w, c.d3, n.pos.x, n.pos.y, n.pos.z);
      x = n.pos.x, y = n.pos.y, z = n.pos.z;
      if (bc) v = sign * ri_load(c.phi + ri_index(c.w, c.d3, x, y, z));
    }
    const uint64_t bm = __ballot(bc);
    if (pass == 0 && bc) {
      const int64_t at = nbc + __popcll(bm & ((1ull << lane) - 1ull));
      if (at < c.list_cap) {
        dcl_icoor q;
        q.x = x, q.y = y, q.z = z;
        c.list[0][at] = q;
      }
    }
    nbc += __popcll(bm);
    x -= c.w.px;
    y -= c.w.py;
    z = c.d3 ? z - c.w.pz : 0;
    uint64_t pm = __ballot(bc && v >= 0.);
    while (pm && err == RI_OK) {
      const int l = __builtin_ctzll(pm);
      pm &= pm - 1;
      const int bx = __builtin_amdgcn_readlane(x, l), by = __builtin_amdgcn_readlane(y, l),
                bz = __builtin_amdgcn_readlane(z, l);
      const int id = (bz * c.w.ny + by) * c.w.nx + bx;
      const RiSten s = ri_sten<NN>(c, tl, id, bx, by, bz, false);
      bool valid, nan;
      const double d1 = ri_update<NN>(c, sign, tl, s, false, 0.0, valid, nan);
      if (__builtin_amdgcn_ballot_w64(nan) & RI_LEAD)
        err = RI_NAN;
      else
        err = ri_insert_all(cap, ri_key<NN>(c.w, tl, id, bx, by, bz), d1, __builtin_amdgcn_ballot_w64(valid) & RI_LEAD,
                            H, hlen);
    }
  }
  // FMM_SolveEikonal; every pop either ends the pass or is followed by at
  // most NN pushes, and a node is accepted again only at a value below its
  // last, so a bounded number of pops always suffices: the cap only keeps a
  // corrupted input from running without end
  const int64_t max_pops = 64 * ((int64_t)c.w.nx * c.w.ny * (c.d3 ? c.w.nz : 1) + c.count) + (1 << 20);
  int64_t pops = 0;
  while (hlen > 1 && err == RI_OK) {
    if (++pops > max_pops) {
      err = RI_STEPS;
      break;
    }
    const unsigned top = (unsigned)__builtin_amdgcn_readfirstlane((int)lds_k[1]);
    const double v = ri_lane_f64(lds_v[1], 0);
    if (v > c.bw) break;
    const int id = (int)(top & ~RI_INNER);
    const bool inner = (top & RI_INNER) != 0;
    const int lz = NN == 6 ? (int)by_plane((unsigned)id) : 0;
    const int row = id - lz * (c.w.nx * c.w.ny);
    const int ly = (int)by_row((unsigned)row), lx = row - ly * c.w.nx;
    double* q = c.phi + id;
    // the node's value and its neighbours' stencils are on their way while
    // the heap closes up (a node accepted before at a value as low is
    // dropped, and its loads with it)
    const double cur = ri_load(q);
    const RiSten s = ri_sten<NN>(c, tl, id, lx, ly, lz, inner);
    ri_heap_pop(H, tl, hlen);
    if (v >= sign * cur) continue;
    if (lane == 0) {
      if (nacc < c.list_cap) {
        dcl_icoor p;
        p.x = c.w.px + lx, p.y = c.w.py + ly;
        p.z = c.w.pz + lz;  // 2D: the window's z (see orc_reinitialize)
        RI_GLOBAL int* to = (RI_GLOBAL int*)(accepted + nacc);
        to[0] = p.x, to[1] = p.y, to[2] = p.z;
      }
      ri_store(q, sign * v);
    }
    ++nacc;
    // the stencils were loaded before the node got its value
    bool valid, nan;
    const double d1 = ri_update<NN>(c, sign, tl, s, tl.back, v, valid, nan);
    if (__builtin_amdgcn_ballot_w64(nan) & RI_LEAD) {
      err = RI_NAN;
      break;
    }
    err = ri_insert_all(cap, ri_key<NN>(c.w, tl, id, lx, ly, lz), d1, __builtin_amdgcn_ballot_w64(valid) & RI_LEAD, H,
                        hlen);
  }
  if (lane == 0) {
    if (pass == 0) c.stat[0] = nbc;
    c.stat[1 + pass] = nacc;
    if (err != RI_OK) c.stat[3] = err;
  }
}

}  // namespace dcl

using namespace dcl;

extern "C" int dcl_reinitialize(dcl_reinit_cell* cells, int ncells, int64_t heap_capacity, void* stream) {
  if (ncells < 0) return set_error(DCL_ERR_ARG_SIZ, "ncells < 0");
  if (ncells > 0 && !cells) return set_error(DCL_ERR_ARG_NULL, "cells is NULL");
  if (heap_capacity < 0) return set_error(DCL_ERR_ARG_SIZ, "heap_capacity < 0");
  if (ncells == 0) return 0;
  if (ncells > (1 << 20)) return set_error(DCL_ERR_ARG_SIZ, "at most 2^20 level sets per call");
  hipStream_t s = as_stream(stream);
  // scratch: cell descriptors | stats | per cell: 2 heaps, 3 lists
  size_t bytes = ((sizeof(RiCell) * ncells + 255) / 256) * 256 + ((sizeof(long long) * 4 * ncells + 255) / 256) * 256;
  for (int i = 0; i < ncells; ++i) {
    dcl_reinit_cell& u = cells[i];
    if (!u.phi) return set_error(DCL_ERR_ARG_NULL, "level set %d: phi is NULL", i);
    DCL_TRY(check_window(&u.win, "phi", 1));
    if (u.count < 0 || (u.count > 0 && !u.nodes))
      return set_error(DCL_ERR_ARG_NULL, "level set %d: bad irregular-node list", i);
    if (u.count > INT32_MAX) return set_error(DCL_ERR_ARG_SIZ, "level set %d: more than 2^31 - 1 records", i);
    if (u.band_capacity < 0 || (u.band_capacity > 0 && !u.band))
      return set_error(DCL_ERR_ARG_NULL, "level set %d: bad band output", i);
    if (!(u.band_width > 0) || !(u.phi_inf > u.band_width))
      return set_error(DCL_ERR_ARG_WRONG, "level set %d: need 0 < band_width < phi_inf", i);
    const int64_t hc = heap_capacity ? heap_capacity : 2 * u.count + 4096;
    bytes += 2 * (((sizeof(RiSlot) * (size_t)(hc + 1)) + 255) / 256) * 256;
    bytes += 3 * (((sizeof(dcl_icoor) * (size_t)(u.band_capacity > 0 ? u.band_capacity : 1)) + 255) / 256) * 256;
  }
  void* sc = nullptr;
  DCL_TRY(scratch(bytes, &sc));
  char* base = static_cast<char*>(sc);
  RiCell* dcells = reinterpret_cast<RiCell*>(base);
  base += ((sizeof(RiCell) * ncells + 255) / 256) * 256;
  long long* stats = reinterpret_cast<long long*>(base);
  base += ((sizeof(long long) * 4 * ncells + 255) / 256) * 256;
  RiCell* host = static_cast<RiCell*>(malloc(sizeof(RiCell) * ncells));
  long long* hstat = static_cast<long long*>(malloc(sizeof(long long) * 4 * ncells));
  if (!host || !hstat) {
    free(host);
    free(hstat);
    return set_error(DCL_ERR_MEM, "host memory");
  }
  int d3 = -1, mixed = 0;
  for (int i = 0; i < ncells; ++i) {
    const dcl_reinit_cell& u = cells[i];
    RiCell& c = host[i];
    c.phi = static_cast<double*>(u.phi);
    c.w = kwin(u.win);
    c.d3 = u.win.n.z >= 2;
    if (d3 >= 0 && d3 != c.d3) mixed = 1;
    d3 = c.d3;
    c.nodes = u.nodes;
    c.count = u.count;
    c.bw = u.band_width;
    c.inf = u.phi_inf;
    c.heap_cap = heap_capacity ? heap_capacity : 2 * u.count + 4096;
    for (int p = 0; p < 2; ++p) {
      c.heap[p] = reinterpret_cast<RiSlot*>(base);
      base += ((sizeof(RiSlot) * (size_t)(c.heap_cap + 1) + 255) / 256) * 256;
    }
    c.list_cap = u.band_capacity;
    for (int p = 0; p < 3; ++p) {
      c.list[p] = reinterpret_cast<dcl_icoor*>(base);
      base += ((sizeof(dcl_icoor) * (size_t)(u.band_capacity > 0 ? u.band_capacity : 1) + 255) / 256) * 256;
    }
    c.stat = stats + 4 * i;
  }
  int rc = 0;
  if (mixed) rc = set_error(DCL_ERR_ARG_WRONG, "a batch mixes 2D and 3D level sets");
  if (!rc) {
    hipError_t e = hipMemcpyAsync(dcells, host, sizeof(RiCell) * ncells, hipMemcpyHostToDevice, s);
    if (e == hipSuccess) e = hipMemsetAsync(stats, 0, sizeof(long long) * 4 * ncells, s);
    if (e != hipSuccess) rc = hip_fail(e, "reinit upload", __FILE__, __LINE__);
  }
  for (int i = 0; i < ncells && !rc; ++i) {
    const RiCell& c = host[i];
    const int64_t n = win_nodes(cells[i].win);
    const unsigned rb = grid1d(n, 256) < 4096u ? grid1d(n, 256) : 4096u;
    hipLaunchKernelGGL(reinit_reset_k, dim3(rb), dim3(256), 0, s, c.phi, n, c.inf);
    if (c.count > 0) hipLaunchKernelGGL(reinit_bc_k, dim3(grid1d(c.count, 256)), dim3(256), 0, s, c);
    if (hipGetLastError() != hipSuccess) rc = set_error(DCL_ERR_LIB, "reinit reset / boundary launch failed");
  }
  if (!rc) {
    if (d3)
      hipLaunchKernelGGL(reinit_fmm_k<6>, dim3(2 * ncells), dim3(64), 0, s, dcells);
    else
      hipLaunchKernelGGL(reinit_fmm_k<4>, dim3(2 * ncells), dim3(64), 0, s, dcells);
    if (hipGetLastError() != hipSuccess) rc = set_error(DCL_ERR_LIB, "reinit fast marching launch failed");
  }
  if (!rc) {
    hipError_t e = hipMemcpyAsync(hstat, stats, sizeof(long long) * 4 * ncells, hipMemcpyDeviceToHost, s);
    if (e == hipSuccess) e = hipStreamSynchronize(s);
    if (e != hipSuccess) rc = hip_fail(e, "reinit", __FILE__, __LINE__);
  }
  // the band: [boundary nodes | - pass | + pass], clipped to the capacity
  for (int i = 0; i < ncells && !rc; ++i) {
    const long long* st = hstat + 4 * i;
    if (st[3] == RI_NAN) {
      rc = set_error(DCL_ERR_LIB, "level set %d: NaN in a fast marching update", i);
      break;
    }
    if (st[3] == RI_STEPS) {
      rc = set_error(DCL_ERR_LIB, "level set %d: fast marching did not finish", i);
      break;
    }
    if (st[3] == RI_HEAP) {
      rc = set_error(DCL_ERR_ARG_SIZ, "level set %d: fast marching heap full (capacity %lld)", i,
                     (long long)host[i].heap_cap);
      break;
    }
    dcl_reinit_cell& u = cells[i];
    int64_t at = 0;
    for (int p = 0; p < 3 && !rc; ++p) {
      const int64_t len = st[p];
      const int64_t take = at >= u.band_capacity ? 0 : (len < u.band_capacity - at ? len : u.band_capacity - at);
      if (take > 0) {
        hipError_t e = hipMemcpyAsync(u.band + at, host[i].list[p], sizeof(dcl_icoor) * (size_t)take,
                                      hipMemcpyDeviceToDevice, s);
        if (e != hipSuccess) rc = hip_fail(e, "reinit band copy", __FILE__, __LINE__);
      }
      at += len;
    }
    u.band_count = at;
  }
  if (!rc) {
    hipError_t e = hipStreamSynchronize(s);
    if (e != hipSuccess) rc = hip_fail(e, "reinit", __FILE__, __LINE__);
  }
  free(host);
  free(hstat);
  return rc;
}
