// step.hip -- one dense level-set update: SL step phi0 -> phi followed by
// the 19-point (3D) / 9-point (2D) curvature of the new phi.  3D: the SL and
// the curvature kernel one after the other.  2D with the velocity on phi's
// window: one fused launch (dcl_step2d.hpp), unless kappa takes memory of phi0
// or the velocity, which the fused launch still reads when it writes kappa.
#include "dcl_host.hpp"
#include "dcl_step2d.hpp"

namespace dcl {
int sl_launch(const void* phi0, void* phi, const dcl_window* win, const dcl_velocity* vel,
              const dcl_icoor* band, int64_t band_len, void* band_values, double dt,
              int precision, int interp, int backtrace, hipStream_t s);
int check_sl_args(const void* phi0, void* phi, const dcl_window* win, const dcl_velocity* vel,
                  const dcl_icoor* band, int64_t band_len, void* band_values, int precision,
                  int interp, int backtrace);
int curv_launch(const void* phi, void* kappa, const dcl_window* win, const dcl_icoor* band,
                int64_t n, void* bv, int precision, int stencil, hipStream_t s);
int sl_params(const dcl_window* win, const dcl_velocity* vel, double dt, SLP& P);

template <typename T, int INTERP, int BT, int R>
__global__ __launch_bounds__(Step2<R>::NT) void step2d_k(const T* __restrict__ phi0, T* __restrict__ phi,
                                                         T* __restrict__ kappa, const T* __restrict__ vel, SLP P,
                                                         T dx, T dy, Curv2R<T> cr) {
  __shared__ Step2Lds<T, R> S;
  const int cols = step2d_cols(P.w.nx, R);
  step2d_tile<T, INTERP, BT, R>(phi0, phi, kappa, vel, P, dx, dy, cr, (int)blockIdx.x * cols,
                                (int)blockIdx.y * Step2<R>::OY, cols, S);
}

template <typename T, int INTERP, int BT>
static int step2d_launch(const T* phi0, T* phi, T* kappa, const T* vel, const SLP& P, T dx, T dy, hipStream_t s) {
  const Curv2R<T> cr = curv2d_recips<T>(dx, dy);
  const int nx = P.w.nx, ny = P.w.ny;
  const int rows = step2d_rows(step2d_tiles(nx, ny, 4), step2d_tiles(nx, ny, 2), device_cus());
  const int cols = step2d_cols(nx, rows), oy = S2_TY * rows - 2;
  const dim3 grid((nx + cols - 1) / cols, (ny + oy - 1) / oy), block(S2_TX, S2_TY);
  if (rows == 4)
    hipLaunchKernelGGL((step2d_k<T, INTERP, BT, 4>), grid, block, 0, s, phi0, phi, kappa, vel, P, dx, dy, cr);
  else if (rows == 2)
    hipLaunchKernelGGL((step2d_k<T, INTERP, BT, 2>), grid, block, 0, s, phi0, phi, kappa, vel, P, dx, dy, cr);
  else
    hipLaunchKernelGGL((step2d_k<T, INTERP, BT, 1>), grid, block, 0, s, phi0, phi, kappa, vel, P, dx, dy, cr);
  DCL_LAUNCHED("step2d");
  return 0;
}

template <typename T>
static int step2d(const void* phi0, void* phi, void* kappa, const dcl_window* win, const dcl_velocity* vel, double dt,
                  int interp, int backtrace, hipStream_t s) {
  SLP P;
  sl_params(win, vel, dt, P);
  const T dx = (T)win->d.x, dy = (T)win->d.y;
  const T* p0 = static_cast<const T*>(phi0);
  const T* v = static_cast<const T*>(vel->data);
  T* p = static_cast<T*>(phi);
  T* k = static_cast<T*>(kappa);
  if (interp == DCL_CUBIC && backtrace == DCL_RK2) return step2d_launch<T, DCL_CUBIC, DCL_RK2>(p0, p, k, v, P, dx, dy, s);
  if (interp == DCL_CUBIC) return step2d_launch<T, DCL_CUBIC, DCL_EULER>(p0, p, k, v, P, dx, dy, s);
  if (backtrace == DCL_RK2) return step2d_launch<T, DCL_LINEAR, DCL_RK2>(p0, p, k, v, P, dx, dy, s);
  return step2d_launch<T, DCL_LINEAR, DCL_EULER>(p0, p, k, v, P, dx, dy, s);
}

// the fused 2D step stages the velocity at phi's nodes; its grid's second
// dimension holds at most 65535 tiles (two rows each where they are smallest)
static bool step2d_takes(const void* phi0, const void* kappa, const dcl_window& w, const dcl_velocity& vel,
                         int precision) {
  const dcl_window& v = vel.win;
  if (w.n.z >= 2 || v.p.x != w.p.x || v.p.y != w.p.y || v.n.x != w.n.x || v.n.y != w.n.y || w.n.y > 100000)
    return false;
  const int64_t bytes = win_nodes(w) * (precision == DCL_F64 ? 8 : 4);
  return !overlap(kappa, bytes, phi0, bytes) && !overlap(kappa, bytes, vel.data, bytes * (vel.dof == 1 ? 2 : vel.dof));
}
}  // namespace dcl

using namespace dcl;

extern "C" int dcl_levelset_step(const void* phi0, void* phi, void* kappa, const dcl_window* win,
                                 const dcl_velocity* vel, double dt, int precision, int interp,
                                 int backtrace, void* stream) {
  DCL_TRY(check_sl_args(phi0, phi, win, vel, nullptr, 0, nullptr, precision, interp, backtrace));
  if (!kappa) return set_error(DCL_ERR_ARG_NULL, "kappa is NULL");
  if (kappa == phi || kappa == phi0)
    return set_error(DCL_ERR_ARG_WRONG, "kappa must not alias phi or phi0");
  hipStream_t s = as_stream(stream);
  if (step2d_takes(phi0, kappa, *win, *vel, precision))
    return precision == DCL_F64 ? step2d<double>(phi0, phi, kappa, win, vel, dt, interp, backtrace, s)
                                : step2d<float>(phi0, phi, kappa, win, vel, dt, interp, backtrace, s);
  DCL_TRY(sl_launch(phi0, phi, win, vel, nullptr, 0, nullptr, dt, precision, interp, backtrace, s));
  return curv_launch(phi, kappa, win, nullptr, 0, nullptr, precision, DCL_CURV_STD, s);
}
