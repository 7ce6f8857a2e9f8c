// dcl_host.hpp -- host-side helpers shared by the C-ABI translation units:
// the per-thread error message, HIP error mapping and argument checks.
#pragma once

#include <hip/hip_runtime.h>
#include <stdarg.h>
#include <stdint.h>
#include <stdio.h>

#include "dcell_lsm.h"
#include "dcl_common.hpp"

namespace dcl {

int set_error(int code, const char* fmt, ...);
int hip_fail(hipError_t e, const char* what, const char* file, int line);

inline hipStream_t as_stream(void* s) { return reinterpret_cast<hipStream_t>(s); }

// window element count (times dof) must fit the kernels' 32-bit offsets
inline int64_t win_nodes(const dcl_window& w) {
  const int64_t nz = w.n.z < 2 ? 1 : w.n.z;
  return (int64_t)w.n.x * w.n.y * nz;
}

int check_window(const dcl_window* w, const char* name, int min_n, int dof = 1);
// planes: the entry point also takes component planes (dof 1)
int check_velocity(const dcl_velocity* v, int dim, bool planes = false);
int check_precision(int precision);

// whether two buffers have memory in common
inline bool overlap(const void* a, int64_t abytes, const void* b, int64_t bbytes) {
  const char *p = static_cast<const char*>(a), *q = static_cast<const char*>(b);
  return p < q + bbytes && q < p + abytes;
}

inline unsigned grid1d(int64_t n, int block) { return (unsigned)((n + block - 1) / block); }

// compute units of the current device (queried once per device; 256 if the
// query fails)
int device_cus();

// Device scratch owned by the calling host thread on the current device
// (grown on demand, kept until the process ends).  Only the synchronous
// entry points (reductions with host results) use it, and they synchronize
// their stream before returning, so the buffer is free again on return.
int scratch(size_t bytes, void** ptr);

// A few words of pinned host memory for the result of a synchronous entry
// point: its last kernel writes them there and wait() synchronises the
// stream.  A kernel and its result come back in 13.9 us that way, against
// 22.6 us with a copy to the caller's pageable word, which is staged and
// awaited by itself.  The words are one of HR_SLOTS of the process, allocated
// together by the first call that needs one (all in use: an allocation of the
// call's own).  A call gives them back when it returns, also with an error
// between take() and wait(): the destructor then waits for the stream.  They
// stay taken only where the stream cannot be waited for, since a kernel may
// still write them.
class HostResult {
 public:
  static constexpr int HR_SLOTS = 64, HR_BYTES = 64;
  HostResult() = default;
  ~HostResult();
  HostResult(const HostResult&) = delete;
  HostResult& operator=(const HostResult&) = delete;
  int take(hipStream_t s);
  int wait();
  template <typename V>
  V* as() const { return static_cast<V*>(p_); }

 private:
  void* p_ = nullptr;
  int slot_ = -1;
  hipStream_t s_ = nullptr;
  bool waited_ = false;
};

// Exclusive scan of per-block counts (scan.hip), in two levels over tiles of
// SCAN_TILE counts: afterwards the exclusive prefix of count i is
// counts[i] + sums[i / SCAN_TILE] and *total is the sum.  A tile's prefix must
// stay below 2^32 (counts below 2^22).  Asynchronous on stream s; scans
// narrays (1 or 2) arrays of the same length n at once.
constexpr int SCAN_TILE = 1024;
struct ScanArrays {
  unsigned* counts[2];
  unsigned long long* sums[2];   // scan_tiles(n) entries each
  unsigned long long* total[2];  // one entry each
};
inline int64_t scan_tiles(int64_t n) { return (n + SCAN_TILE - 1) / SCAN_TILE; }
int scan_counts(const ScanArrays& a, int narrays, int64_t n, hipStream_t s);

}  // namespace dcl

#define DCL_HIP(call)                                                          \
  do {                                                                         \
    hipError_t e__ = (call);                                                   \
    if (e__ != hipSuccess) return dcl::hip_fail(e__, #call, __FILE__, __LINE__); \
  } while (0)

#define DCL_LAUNCHED(name)                                                     \
  do {                                                                         \
    hipError_t e__ = hipGetLastError();                                        \
    if (e__ != hipSuccess) return dcl::hip_fail(e__, name, __FILE__, __LINE__); \
  } while (0)

#define DCL_TRY(call)          \
  do {                         \
    int rc__ = (call);         \
    if (rc__) return rc__;     \
  } while (0)
