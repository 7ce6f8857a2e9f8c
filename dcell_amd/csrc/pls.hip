// pls.hip -- particle level set on gfx950.
//
//   dcl_pls_advect       ParticleLS_AdvectParticles3D / 2D (ParticleLS3D.c:6-36,
//                        ParticleLS2D.c:6-36): RK2 midpoint, one thread per particle
//   dcl_pls_correct      ParticleLS_ErrorCorrection3D / 2D (ParticleLS3D.c:40-116,
//                        ParticleLS2D.c:40-115)
//   dcl_pls_adjust_radii ParticleLS_AdjustRadii (ParticleLS.c:158-185)
//
// The correction keeps phi+ and phi- as ordered-integer keys of the particle
// extrema only (the reference copies phi into two whole grids first,
// ParticleLS3D.c:60-61); max(phi, P+) is the reference's phi+ because max is
// order-free.  Escaped particles scatter with integer atomic max/min and
// list the touched nodes; the merge then visits only touched nodes (dense) or
// the band, and puts the keys back to their neutral values, so no full-grid
// pass is needed per call.  Each block of particles lists its nodes in a
// region of its own with its own count (a block's particles touch at most
// 2^dim nodes each, so the regions fit the workspace by the check on the
// call): one list with one counter queued every touched corner's atomic on
// one address, 1.62 ms for the escape pass of 8.8M FP32 particles at 256^3
// (moved by a tenth of a cell since their radii were set) against 0.060 ms
// with the regions, where reading the particles (140 MB, 26 us) and 8 phi
// values each is what is left; the merge 0.062 against 0.014 ms.
#include <new>

#include "dcl_buf.hpp"
#include "dcl_host.hpp"

namespace dcl {

template <typename T>
__device__ __forceinline__ T psign(T a) { return a >= T(0) ? (a == T(0) ? T(0) : T(1)) : T(-1); }

// |X - a|^2 summed left to right without FMA contraction, so the FP64 corner
// values round exactly as the reference's expression (ParticleLS3D.c:85-87)
__device__ __forceinline__ double dist2(double dx, double dy, double dz, bool three) {
#pragma clang fp contract(off)
  double r = dx * dx + dy * dy;
  if (three) r = r + dz * dz;
  return r;
}

// --------------------------------------------------------------- advect
// How the velocity is read: with pointers; with buffer loads (3D, velocity
// window below 2 GiB: 32-bit offsets, and with 3 FP32 components an x pair of
// faces is one 16-byte load); or, on top of these, from LDS boxes (exactly 3
// components a node, a window no smaller than a box)
enum { ADV_PTR, ADV_BUF, ADV_BOX };

// The box of velocity nodes that a wave stages.  Particles lie in memory as
// they were seeded, node by node along x, so the 64 of a wave sit around a few
// neighbouring nodes of one row, and the 24 corner pairs that each interpolates
// are nearly the same: gathered, they were 24 loads of 64 lanes per particle
// against the 3 (FP64: 5) that bring the box.  8 nodes along x hold 4 cells
// of particles, and 5 along y and z one cell, with the RK2 midpoint half a
// cell away to either side; where a row of particles ends within a wave, the
// rest of it has a second box, and lanes that neither box holds gather.
// 8.8M FP32 particles in a band of the 256^3 window 227 -> 122 us: the texture
// path was 94% busy, now the vector units are (82%; 420 instructions per
// particle of which 84 are the six divisions by the spacing, against 52 us
// for reading and writing the particles).
constexpr int BOX_X = 8, BOX_Y = 5, BOX_Z = 5;
constexpr int BOX_NODES = BOX_X * BOX_Y * BOX_Z;
// Fewest particles that a wave stages a box for: a box costs the loads of a
// quarter of one gathered interpolation.  Particles in no order would stage
// boxes for a few lanes each and gather the others all the same.
constexpr int BOX_MIN = 8;

template <typename T>
struct VelBox {
  int o[3];  // the box's lowest node

  __device__ __forceinline__ void place(const KVel& v, int x, int y, int z) {
    o[0] = clampi(x - 1, 0, v.w.nx - BOX_X);
    o[1] = clampi(y - 1, 0, v.w.ny - BOX_Y);
    o[2] = clampi(z - 1, 0, v.w.nz - BOX_Z);
  }
  // whether all corners of the split (b0, b1) lie in the box (b0 <= b1 <= b0 + 1)
  __device__ __forceinline__ bool holds(const int b0[3], const int b1[3]) const {
    return (b0[0] >= o[0]) & (b1[0] <= o[0] + BOX_X - 2) & (b0[1] >= o[1]) & (b1[1] <= o[1] + BOX_Y - 2) &
           (b0[2] >= o[2]) & (b1[2] <= o[2] + BOX_Z - 2);
  }
  // one 16-byte load per chunk of a row; rows lie in LDS as they do in memory
  __device__ __forceinline__ void stage(rsrc_t rv, const KVel& v, T* lds, int lane) const {
    constexpr int CH = 16 / (int)sizeof(T), RC = BOX_X * 3 / CH;  // elements of a chunk, chunks of a row
    constexpr int NC = 3 * BOX_NODES / CH, PER = (NC + 63) / 64;
    const int sy = v.w.nx * 3, sz = v.w.ny * sy, base = o[2] * sz + o[1] * sy + o[0] * 3;
    T q[PER][CH];
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int c = min(lane + 64 * i, NC - 1), row = c / RC;
      const int e = base + (row / BOX_Y) * sz + (row % BOX_Y) * sy + (c % RC) * CH;
      if constexpr (CH == 4)
        BL<T>::four(rv, e * (int)sizeof(T), 0, q[i]);
      else
        BL<T>::two(rv, e * (int)sizeof(T), 0, q[i]);
    }
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int c = lane + 64 * i;
      if (c >= NC) break;
#pragma unroll
      for (int k = 0; k < CH; ++k) lds[c * CH + k] = q[i][k];
    }
  }
  // mac_vel_buf_split from the box at lds
  __device__ __forceinline__ void vel(const T* lds, const int b0[3], const int b1[3], const T f0[3], const T f1[3],
                                      T V[3]) const {
    constexpr int sx = 3, sy = BOX_X * sx, sz = BOX_Y * sy;
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      const int ix = c == 0 ? b1[0] : b0[0], iy = c == 1 ? b1[1] : b0[1], iz = c == 2 ? b1[2] : b0[2];
      const T* b = lds + (iz - o[2]) * sz + (iy - o[1]) * sy + (ix - o[0]) * sx + c;
      const T x1 = c == 0 ? f1[0] : f0[0], y1 = c == 1 ? f1[1] : f0[1], z1 = c == 2 ? f1[2] : f0[2];
      V[c] = vtri(b[0], b[sx], b[sy], b[sy + sx], b[sz], b[sz + sx], b[sz + sy], b[sz + sy + sx], x1, y1, z1);
    }
  }
};

// both velocities of a particle's step (at X and at the midpoint) from the
// boxes of its wave
template <typename T>
__device__ __forceinline__ void box_vels(rsrc_t rv, KVel v, const double X[3], double dt, const double dh[3],
                                         T* lds, T V2[3]) {
  v.dof = 3, v.udof = 0, v.cs = 1;
  const int lane = threadIdx.x & 63;
  int b0[3], b1[3];
  T f0[3], f1[3], V1[3];
  mac_split<T, 3>(v, X, b0, b1, f0, f1);
  VelBox<T> A, B;
  A.place(v, __builtin_amdgcn_readfirstlane(b0[0]), __builtin_amdgcn_readfirstlane(b0[1]),
          __builtin_amdgcn_readfirstlane(b0[2]));
  const bool inA = A.holds(b0, b1);
  const unsigned long long ma = __builtin_amdgcn_ballot_w64(inA);
  const bool useA = __popcll(ma) >= BOX_MIN;
  bool inB = false;
  if (~ma) {
    const int l = __ffsll(~ma) - 1;
    B.place(v, __builtin_amdgcn_readlane(b0[0], l), __builtin_amdgcn_readlane(b0[1], l),
            __builtin_amdgcn_readlane(b0[2], l));
    inB = B.holds(b0, b1) && !inA;
  } else {
    B = A;
  }
  const bool useB = __popcll(__builtin_amdgcn_ballot_w64(inB)) >= BOX_MIN;
  if (useA) A.stage(rv, v, lds, lane);
  if (useB) B.stage(rv, v, lds + 3 * BOX_NODES, lane);
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  const bool second = inB && useB, boxed = second || (inA && useA);
  const T* box = second ? lds + 3 * BOX_NODES : lds;
  VelBox<T> own;
#pragma unroll
  for (int a = 0; a < 3; ++a) own.o[a] = second ? B.o[a] : A.o[a];
  if (boxed)
    own.vel(box, b0, b1, f0, f1, V1);
  else
    mac_vel_buf_split<T>(rv, v, b0, b1, f0, f1, V1);
  double Xm[3];
#pragma unroll
  for (int a = 0; a < 3; ++a) Xm[a] = X[a] + dt / 2 * (double)V1[a] / dh[a];
  mac_split<T, 3>(v, Xm, b0, b1, f0, f1);
  if (boxed && own.holds(b0, b1))
    own.vel(box, b0, b1, f0, f1, V2);
  else
    mac_vel_buf_split<T>(rv, v, b0, b1, f0, f1, V2);
}

template <typename T, int DIM, int MODE>
__global__ __launch_bounds__(256) void pls_advect_k(T* __restrict__ P, int64_t n,
                                                    const T* __restrict__ vel, KVel v,
                                                    double dhx, double dhy, double dhz, double dt,
                                                    unsigned vbytes) {
  const int64_t m = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const double dh[3] = {dhx, dhy, dhz};
  if constexpr (MODE == ADV_BOX) {
    __shared__ __attribute__((aligned(16))) T boxes[256 / 64][2][3 * BOX_NODES];
    // the wave's lanes past the end go along with its last particle
    if (m - (threadIdx.x & 63) >= n) return;
    T* p = P + 4 * (m < n ? m : n - 1);
    const double X[3] = {(double)p[0], (double)p[1], (double)p[2]};
    T V2[3];
    box_vels<T>(make_rsrc(vel, vbytes), v, X, dt, dh, boxes[threadIdx.x / 64][0], V2);
    if (m >= n) return;
#pragma unroll
    for (int a = 0; a < 3; ++a) p[a] = (T)(X[a] + dt * (double)V2[a] / dh[a]);
    return;
  }
  if (m >= n) return;
  T* p = P + 4 * m;
  double X[3] = {(double)p[0], (double)p[1], (double)p[2]};
  T V1[3], V2[3];
  const rsrc_t rv = make_rsrc(vel, vbytes);
  if (MODE == ADV_BUF)
    mac_vel_buf<T>(rv, v, X, V1);
  else
    mac_vel<T, DIM>(vel, v, X, V1);
  double Xm[3] = {X[0], X[1], X[2]};
#pragma unroll
  for (int a = 0; a < DIM; ++a) Xm[a] = X[a] + dt / 2 * (double)V1[a] / dh[a];
  if (MODE == ADV_BUF)
    mac_vel_buf<T>(rv, v, Xm, V2);
  else
    mac_vel<T, DIM>(vel, v, Xm, V2);
#pragma unroll
  for (int a = 0; a < DIM; ++a) p[a] = (T)(X[a] + dt * (double)V2[a] / dh[a]);
}

// ------------------------------------------------------------- correct
struct PlsK {
  KWin w;
  int flags;
  unsigned epoch;
};

// one particle: where it has escaped, its 2^dim corner values into the keys
// and the corners inside the window into the block's region
template <typename T, int DIM>
__device__ __forceinline__ void pls_escape_one(const T* __restrict__ p, const T* __restrict__ phi,
                                               typename KeyOf<T>::type* __restrict__ kpos,
                                               typename KeyOf<T>::type* __restrict__ kneg,
                                               int* __restrict__ region, unsigned* listed, const PlsK& K) {
  const double X[3] = {(double)p[0], (double)p[1], (double)p[2]};
  const T r = p[3];
  const T dist = grid_interp<T, DIM>(phi, K.w, X);
  const T sign = psign(r);
  if (!(sign * dist < T(0) && fabs(dist) > fabs(r))) return;
  const int Ax = (int)floor(X[0]);
  const int Ay = (int)floor(X[1]);
  const int Az = DIM == 3 ? (int)floor((K.flags & DCL_PLS_REF_AZ) ? X[1] : X[2]) : K.w.pz;
#pragma unroll
  for (int k = 0; k < (DIM == 3 ? 2 : 1); ++k)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int ax = Ax + i, ay = Ay + j, az = Az + k;
        const int lx = ax - K.w.px, ly = ay - K.w.py, lz = DIM == 3 ? az - K.w.pz : 0;
        if (lx < 0 || lx >= K.w.nx || ly < 0 || ly >= K.w.ny || lz < 0 || lz >= K.w.nz) continue;
        const double r2 = dist2(X[0] - ax, X[1] - ay, X[2] - az, DIM == 3);
        const T phi_p = sign * (sign * r - (T)sqrt(r2));
        const int id = (lz * K.w.ny + ly) * K.w.nx + lx;
        if (sign > T(0)) atomicMax(&kpos[id], okey(phi_p));
        else atomicMin(&kneg[id], okey(phi_p));
        region[atomicAdd(listed, 1u)] = id;
      }
}

constexpr int PLS_B = 256;  // particles per block of the escape pass
// node slots of one block's event region
template <int DIM>
constexpr int pls_region() {
  return PLS_B * (DIM == 3 ? 8 : 4);
}

// escape test + corner scatter, one thread per particle.  The block's
// touched nodes go to its region of events, their number to counts.
template <typename T, int DIM>
__global__ __launch_bounds__(PLS_B) void pls_escape_k(const T* __restrict__ P, int64_t n,
                                                      const T* __restrict__ phi,
                                                      typename KeyOf<T>::type* __restrict__ kpos,
                                                      typename KeyOf<T>::type* __restrict__ kneg,
                                                      int* __restrict__ events, unsigned* __restrict__ counts,
                                                      PlsK K) {
  __shared__ unsigned listed;
  if (threadIdx.x == 0) listed = 0;
  __syncthreads();
  const int64_t m = (int64_t)blockIdx.x * PLS_B + threadIdx.x;
  int* region = events + (int64_t)blockIdx.x * pls_region<DIM>();
  if (m < n) pls_escape_one<T, DIM>(P + 4 * m, phi, kpos, kneg, region, &listed, K);
  __syncthreads();
  if (threadIdx.x == 0) counts[blockIdx.x] = listed;
}
template <typename T>
__device__ __forceinline__ T merged(T ph, typename KeyOf<T>::type kp, typename KeyOf<T>::type kn) {
  const T pp = okey_val(kp), pn = okey_val(kn);
  const T phi_pos = pp < ph ? ph : pp;   // PetscMax(phi_p, phi_pos)
  const T phi_neg = pn < ph ? pn : ph;   // PetscMin(phi_p, phi_neg)
  return fabs(phi_pos) <= fabs(phi_neg) ? phi_pos : phi_neg;
}

// The listed nodes of every region, one wave per region (nearly all are
// empty: a wave reads its region's count and ends).
template <typename F>
__device__ __forceinline__ void pls_each_event(const int* __restrict__ events, const unsigned* __restrict__ counts,
                                               unsigned regions, int region_size, F body) {
  const unsigned b = blockIdx.x * (256 / 64) + threadIdx.x / 64;
  if (b >= regions) return;
  const unsigned ne = counts[b];
  for (unsigned e = threadIdx.x & 63; e < ne; e += 64) body(events[(int64_t)b * region_size + e]);
}

// dense merge: the first event of a node (per call epoch) owns it
template <typename T>
__global__ __launch_bounds__(256) void pls_merge_events_k(T* __restrict__ phi,
                                                          typename KeyOf<T>::type* __restrict__ kpos,
                                                          typename KeyOf<T>::type* __restrict__ kneg,
                                                          unsigned* __restrict__ claim,
                                                          const int* __restrict__ events,
                                                          const unsigned* __restrict__ counts, unsigned regions,
                                                          int region_size, PlsK K) {
  pls_each_event(events, counts, regions, region_size, [&](int id) {
    if (atomicExch(&claim[id], K.epoch) == K.epoch) return;
    typedef typename KeyOf<T>::type Key;
    const Key kp = kpos[id], kn = kneg[id];
    phi[id] = merged<T>(phi[id], kp, kn);
    kpos[id] = okey(-(T)INFINITY);
    kneg[id] = okey((T)INFINITY);
  });
}

// band merge (the reference's loop over ls->band, ParticleLS3D.c:104-113)
template <typename T, bool COMPACT>
__global__ __launch_bounds__(256) void pls_merge_band_k(T* phi, T* out,
                                                        const typename KeyOf<T>::type* __restrict__ kpos,
                                                        const typename KeyOf<T>::type* __restrict__ kneg,
                                                        const dcl_icoor* __restrict__ band, int64_t n,
                                                        PlsK K, int dim) {
  const int64_t b = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (b >= n) return;
  const dcl_icoor q = band[b];
  const int lx = q.x - K.w.px, ly = q.y - K.w.py, lz = dim == 3 ? q.z - K.w.pz : 0;
  const bool inside = lx >= 0 && lx < K.w.nx && ly >= 0 && ly < K.w.ny && lz >= 0 && lz < K.w.nz;
  if (!inside) {
    if (COMPACT) out[b] = T(0);
    return;
  }
  const int id = (lz * K.w.ny + ly) * K.w.nx + lx;
  const T v = merged<T>(phi[id], kpos[id], kneg[id]);
  if (COMPACT) out[b] = v;
  else phi[id] = v;
}

// put the keys of touched nodes back to neutral (band mode); idempotent writes
template <typename T>
__global__ __launch_bounds__(256) void pls_reset_events_k(typename KeyOf<T>::type* __restrict__ kpos,
                                                          typename KeyOf<T>::type* __restrict__ kneg,
                                                          const int* __restrict__ events,
                                                          const unsigned* __restrict__ counts, unsigned regions,
                                                          int region_size) {
  pls_each_event(events, counts, regions, region_size, [&](int id) {
    kpos[id] = okey(-(T)INFINITY);
    kneg[id] = okey((T)INFINITY);
  });
}

template <typename T>
__global__ __launch_bounds__(256) void pls_fill_keys_k(typename KeyOf<T>::type* kpos,
                                                       typename KeyOf<T>::type* kneg,
                                                       unsigned* claim, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  kpos[i] = okey(-(T)INFINITY);
  kneg[i] = okey((T)INFINITY);
  claim[i] = 0u;
}

// --------------------------------------------------------------- radii
template <typename T, int DIM>
__global__ __launch_bounds__(256) void pls_radii_k(T* __restrict__ P, int64_t n,
                                                   const T* __restrict__ phi, KWin w, T rmin, T rmax) {
  const int64_t m = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (m >= n) return;
  T* p = P + 4 * m;
  const double X[3] = {(double)p[0], (double)p[1], (double)p[2]};
  const T dist = grid_interp<T, DIM>(phi, w, X);
  const T sign = psign(p[3]);
  const T sphi = sign * dist;
  if (rmin < sphi && sphi < rmax) p[3] = sign * sphi;
  else if (sphi > rmax) p[3] = sign * rmax;
  else if (sphi < rmin) p[3] = sign * rmin;
}

}  // namespace dcl

using namespace dcl;

struct dcl_pls_ws_s {
  int precision;
  int64_t max_nodes, max_events;
  void* kpos;
  void* kneg;
  unsigned* claim;
  int* events;       // max_events node slots, cut into one region per block of particles
  unsigned* counts;  // nodes listed in each region
  unsigned epoch;
};

static int check_particles(const void* particles, int64_t count, int dim, int precision) {
  DCL_TRY(check_precision(precision));
  if (count < 0) return set_error(DCL_ERR_ARG_SIZ, "particle count %lld < 0", (long long)count);
  if (count > 0 && !particles) return set_error(DCL_ERR_ARG_NULL, "particles is NULL");
  if (dim != 2 && dim != 3) return set_error(DCL_ERR_ARG_WRONG, "dim %d is neither 2 nor 3", dim);
  return 0;
}

extern "C" int dcl_pls_advect(void* particles, int64_t count, const dcl_velocity* vel, dcl_coor dh,
                              double dt, int dim, int precision, void* stream) {
  DCL_TRY(check_particles(particles, count, dim, precision));
  DCL_TRY(check_velocity(vel, dim));
  if (!(dh.x > 0 && dh.y > 0 && (dim == 2 || dh.z > 0)))
    return set_error(DCL_ERR_ARG_WRONG, "dh must be positive");
  if (count == 0) return 0;
  const KVel v = kvel(*vel);
  hipStream_t s = as_stream(stream);
  const unsigned g = grid1d(count, 256);
  const long long vb = win_nodes(vel->win) * vel->dof * (long long)(precision == DCL_F64 ? 8 : 4);
  int mode = dim == 3 && buf_ok(0, vb) ? ADV_BUF : ADV_PTR;
  if (mode == ADV_BUF && v.dof == 3 && v.w.nx >= BOX_X && v.w.ny >= BOX_Y && v.w.nz >= BOX_Z) mode = ADV_BOX;
#define DCL_ADV(T, D, M)                                                                             \
  hipLaunchKernelGGL((pls_advect_k<T, D, M>), dim3(g), dim3(256), 0, s, static_cast<T*>(particles),  \
                     count, static_cast<const T*>(vel->data), v, dh.x, dh.y, dh.z, dt, (unsigned)vb)
#define DCL_ADV_T(T)                             \
  if (dim == 2) DCL_ADV(T, 2, ADV_PTR);          \
  else if (mode == ADV_PTR) DCL_ADV(T, 3, ADV_PTR);   \
  else if (mode == ADV_BUF) DCL_ADV(T, 3, ADV_BUF);   \
  else DCL_ADV(T, 3, ADV_BOX)
  if (precision == DCL_F64) {
    DCL_ADV_T(double);
  } else {
    DCL_ADV_T(float);
  }
#undef DCL_ADV_T
#undef DCL_ADV
  DCL_LAUNCHED("pls_advect");
  return 0;
}

extern "C" int dcl_pls_ws_create(int64_t max_nodes, int64_t max_events, int precision, void* stream,
                                 dcl_pls_ws* out) {
  DCL_TRY(check_precision(precision));
  if (!out) return set_error(DCL_ERR_ARG_NULL, "ws is NULL");
  *out = nullptr;
  if (max_nodes <= 0 || max_nodes >= ((int64_t)1 << 31))
    return set_error(DCL_ERR_ARG_SIZ, "max_nodes %lld out of range", (long long)max_nodes);
  if (max_events <= 0 || max_events >= ((int64_t)1 << 40))
    return set_error(DCL_ERR_ARG_SIZ, "max_events %lld out of range", (long long)max_events);
  dcl_pls_ws ws = new (std::nothrow) dcl_pls_ws_s();
  if (!ws) return set_error(DCL_ERR_MEM, "host allocation failed");
  ws->precision = precision;
  ws->max_nodes = max_nodes;
  ws->max_events = max_events;
  ws->epoch = 0;
  const size_t kb = precision == DCL_F64 ? 8 : 4;
  int rc = 0;
  void* p[5] = {nullptr, nullptr, nullptr, nullptr, nullptr};
  // as many regions as the smaller (2D) ones that max_events holds
  const size_t regions = (size_t)((max_events + pls_region<2>() - 1) / pls_region<2>());
  const size_t bytes[5] = {kb * max_nodes, kb * max_nodes, 4 * (size_t)max_nodes, 4 * (size_t)max_events,
                           sizeof(unsigned) * regions};
  for (int i = 0; i < 5 && !rc; ++i) rc = dcl_malloc(&p[i], bytes[i]);
  if (rc) {
    for (int i = 0; i < 5; ++i) dcl_free(p[i]);
    delete ws;
    return rc;
  }
  ws->kpos = p[0];
  ws->kneg = p[1];
  ws->claim = static_cast<unsigned*>(p[2]);
  ws->events = static_cast<int*>(p[3]);
  ws->counts = static_cast<unsigned*>(p[4]);
  hipStream_t s = as_stream(stream);
  const unsigned g = grid1d(max_nodes, 256);
  if (precision == DCL_F64)
    hipLaunchKernelGGL((pls_fill_keys_k<double>), dim3(g), dim3(256), 0, s,
                       static_cast<unsigned long long*>(ws->kpos),
                       static_cast<unsigned long long*>(ws->kneg), ws->claim, max_nodes);
  else
    hipLaunchKernelGGL((pls_fill_keys_k<float>), dim3(g), dim3(256), 0, s,
                       static_cast<unsigned*>(ws->kpos), static_cast<unsigned*>(ws->kneg), ws->claim,
                       max_nodes);
  hipError_t e = hipGetLastError();
  if (e == hipSuccess) e = hipStreamSynchronize(s);
  if (e != hipSuccess) {
    for (int i = 0; i < 5; ++i) dcl_free(p[i]);
    delete ws;
    return hip_fail(e, "pls workspace init", __FILE__, __LINE__);
  }
  *out = ws;
  return 0;
}

extern "C" int dcl_pls_ws_destroy(dcl_pls_ws ws) {
  if (!ws) return 0;
  DCL_HIP(hipDeviceSynchronize());
  dcl_free(ws->kpos);
  dcl_free(ws->kneg);
  dcl_free(ws->claim);
  dcl_free(ws->events);
  dcl_free(ws->counts);
  delete ws;
  return 0;
}

template <typename T>
static int pls_correct_t(const void* particles, int64_t count, void* phi, const dcl_window* win,
                         const dcl_icoor* band, int64_t band_len, void* band_values, int flags,
                         int dim, dcl_pls_ws ws, hipStream_t s) {
  typedef typename KeyOf<T>::type Key;
  PlsK K;
  K.w = kwin(*win);
  K.flags = flags;
  K.epoch = ++ws->epoch == 0 ? ++ws->epoch : ws->epoch;
  Key* kp = static_cast<Key*>(ws->kpos);
  Key* kn = static_cast<Key*>(ws->kneg);
  T* ph = static_cast<T*>(phi);
  const unsigned regions = grid1d(count, PLS_B);
  const int rsize = dim == 3 ? pls_region<3>() : pls_region<2>();
  if (count > 0) {
    if (dim == 3)
      hipLaunchKernelGGL((pls_escape_k<T, 3>), dim3(regions), dim3(PLS_B), 0, s, static_cast<const T*>(particles),
                         count, ph, kp, kn, ws->events, ws->counts, K);
    else
      hipLaunchKernelGGL((pls_escape_k<T, 2>), dim3(regions), dim3(PLS_B), 0, s, static_cast<const T*>(particles),
                         count, ph, kp, kn, ws->events, ws->counts, K);
    DCL_LAUNCHED("pls_escape");
  }
  const unsigned ge = (regions + 3) / 4;
  if (!band) {
    if (regions == 0) return 0;
    hipLaunchKernelGGL((pls_merge_events_k<T>), dim3(ge), dim3(256), 0, s, ph, kp, kn, ws->claim, ws->events,
                       ws->counts, regions, rsize, K);
    DCL_LAUNCHED("pls_merge_events");
    return 0;
  }
  if (band_len > 0) {
    const unsigned gb = grid1d(band_len, 256);
    if (band_values)
      hipLaunchKernelGGL((pls_merge_band_k<T, true>), dim3(gb), dim3(256), 0, s, ph,
                         static_cast<T*>(band_values), kp, kn, band, band_len, K, dim);
    else
      hipLaunchKernelGGL((pls_merge_band_k<T, false>), dim3(gb), dim3(256), 0, s, ph, ph, kp, kn, band,
                         band_len, K, dim);
    DCL_LAUNCHED("pls_merge_band");
  }
  if (regions > 0) {
    hipLaunchKernelGGL((pls_reset_events_k<T>), dim3(ge), dim3(256), 0, s, kp, kn, ws->events, ws->counts, regions,
                       rsize);
    DCL_LAUNCHED("pls_reset_events");
  }
  return 0;
}

extern "C" int dcl_pls_correct(const void* particles, int64_t count, void* phi, const dcl_window* win,
                               const dcl_icoor* band, int64_t band_len, void* band_values, int flags,
                               int dim, int precision, dcl_pls_ws ws, void* stream) {
  DCL_TRY(check_particles(particles, count, dim, precision));
  if (!phi) return set_error(DCL_ERR_ARG_NULL, "phi is NULL");
  if (!ws) return set_error(DCL_ERR_ARG_NULL, "workspace is NULL");
  DCL_TRY(check_window(win, "phi", 2));
  if ((win->n.z < 2 ? 2 : 3) != dim) return set_error(DCL_ERR_ARG_WRONG, "window is not %dD", dim);
  if (ws->precision != precision)
    return set_error(DCL_ERR_ARG_WRONG, "workspace precision differs from the call's");
  if (win_nodes(*win) > ws->max_nodes)
    return set_error(DCL_ERR_ARG_SIZ, "window has %lld nodes, workspace holds %lld",
                     (long long)win_nodes(*win), (long long)ws->max_nodes);
  const int64_t corners = dim == 3 ? 8 : 4;
  if (count > ws->max_events / corners)
    return set_error(DCL_ERR_ARG_SIZ, "%lld particles may touch %lld corners; workspace holds %lld events",
                     (long long)count, (long long)(count * corners), (long long)ws->max_events);
  if (band && band_len < 0) return set_error(DCL_ERR_ARG_SIZ, "band_len < 0");
  hipStream_t s = as_stream(stream);
  if (precision == DCL_F64)
    return pls_correct_t<double>(particles, count, phi, win, band, band_len, band_values, flags, dim, ws, s);
  return pls_correct_t<float>(particles, count, phi, win, band, band_len, band_values, flags, dim, ws, s);
}

extern "C" int dcl_pls_adjust_radii(void* particles, int64_t count, const void* phi,
                                    const dcl_window* win, double rmin, double rmax, int dim,
                                    int precision, void* stream) {
  DCL_TRY(check_particles(particles, count, dim, precision));
  if (!phi) return set_error(DCL_ERR_ARG_NULL, "phi is NULL");
  DCL_TRY(check_window(win, "phi", 2));
  if ((win->n.z < 2 ? 2 : 3) != dim) return set_error(DCL_ERR_ARG_WRONG, "window is not %dD", dim);
  if (count == 0) return 0;
  const KWin w = kwin(*win);
  hipStream_t s = as_stream(stream);
  const unsigned g = grid1d(count, 256);
#define DCL_RAD(T, D)                                                                           \
  hipLaunchKernelGGL((pls_radii_k<T, D>), dim3(g), dim3(256), 0, s, static_cast<T*>(particles), \
                     count, static_cast<const T*>(phi), w, (T)rmin, (T)rmax)
  if (precision == DCL_F64) {
    if (dim == 3) DCL_RAD(double, 3); else DCL_RAD(double, 2);
  } else {
    if (dim == 3) DCL_RAD(float, 3); else DCL_RAD(float, 2);
  }
#undef DCL_RAD
  DCL_LAUNCHED("pls_adjust_radii");
  return 0;
}
