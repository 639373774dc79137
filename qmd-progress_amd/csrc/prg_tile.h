// Device helpers shared by the GEMM kernels: XCD-aware tile scheduling and
// deterministic workgroup reductions.
#pragma once

#include <hip/hip_runtime.h>

namespace prg {
namespace tile {

constexpr int kThreads = 256;

// Workgroups are dispatched round-robin over the 8 XCDs; give XCD x the
// contiguous logical range [x*nb/8, (x+1)*nb/8).
__device__ __forceinline__ int xcd_remap(int b, int nb) {
  const int per = nb / 8, rem = nb % 8;
  const int xcd = b % 8, idx = b / 8;
  return (xcd < rem) ? xcd * (per + 1) + idx : rem * (per + 1) + (xcd - rem) * per + idx;
}

// Upper-triangle tile t -> (I, J), I <= J, column-by-column, from an estimate
// of J.
__device__ __forceinline__ void sym_tile_from(int j, int t, int& I, int& J) {
  while ((j + 1) * (j + 2) / 2 <= t) ++j;
  while (j * (j + 1) / 2 > t) --j;
  J = j;
  I = t - j * (j + 1) / 2;
}
__device__ __forceinline__ void sym_tile(int t, int& I, int& J) {
  sym_tile_from((int)((sqrt(8.0 * (double)t + 1.0) - 1.0) * 0.5), t, I, J);
}

// Upper-triangle tile t -> (I, J) of nt tile rows in bands of w columns, row by
// row inside a band (its last w x w triangle column by column): consecutive
// tiles form blocks of about w columns, so the workgroups of an XCD that run
// together read few panels each, and each panel is read by few of them.  (In
// column order, 32 of them read the same panel at the same time, and with a
// leading dimension of many powers of two that panel sits in one or two of
// the L2's 16 channels.)
template <int w>
__device__ __forceinline__ void sym_tile_banded(int t, int nt, int& I, int& J) {
  int i, j;
  // single precision is enough for the estimate
  auto at = [&](int u) {
    sym_tile_from((int)((sqrtf(8.0f * (float)u + 1.0f) - 1.0f) * 0.5f), u, i, j);
  };
  at(t);
  const int first = j / w * w, wb = min(w, nt - first);  // band of column j
  const int u = t - first * (first + 1) / 2;
  if (u < first * wb) {
    I = (wb == w) ? u / w : u / wb;
    J = first + u - I * wb;
  } else {
    at(u - first * wb);
    I = first + i;
    J = first + j;
  }
}

// Full tile t -> (I, J) with groups of 8 tile-rows sharing B panels.
__device__ __forceinline__ void full_tile(int t, int nt, int& I, int& J) {
  const int G = 8;
  const int group = t / (G * nt);
  const int first = group * G;
  const int gsize = min(nt - first, G);
  const int in = t % (G * nt);
  I = first + in % gsize;
  J = in / gsize;
}

// Deterministic workgroup sum of NQ per-thread values (BT threads); threads
// 0 .. NQ - 1 store them.
template <int NQ, int BT = kThreads>
__device__ __forceinline__ void block_store_partials(double (&v)[NQ], double* dst) {
  __shared__ double red[BT / 64][NQ];
#pragma unroll
  for (int q = 0; q < NQ; ++q) {
    double x = v[q];
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) x += __shfl_xor(x, off);
    v[q] = x;
  }
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  if (lane == 0) {
#pragma unroll
    for (int q = 0; q < NQ; ++q) red[w][q] = v[q];
  }
  __syncthreads();
  if (threadIdx.x < NQ) {
    double s = 0.0;
#pragma unroll
    for (int ww = 0; ww < BT / 64; ++ww) s += red[ww][threadIdx.x];
    dst[threadIdx.x] = s;
  }
}


// Lane-crossing move inside rows of 16 lanes (DPP control CTRL).
template <int CTRL>
__device__ __forceinline__ double dpp_move(double x) {
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(x), CTRL, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(x), CTRL, 0xf, 0xf, true);
  return __hiloint2double(hi, lo);
}
__device__ __forceinline__ double read_lane(double x, int lane) {
  return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(x), lane),
                          __builtin_amdgcn_readlane(__double2loint(x), lane));
}

// Sums of four values over a wave, the same in every lane, in a fixed order:
// the first two exchanges also split the values over the 16-lane rows (two,
// then one per lane), the other four are moves inside a row, which cost a
// vector instruction instead of an LDS round trip.
__device__ __forceinline__ void wave_sum4(double (&v)[4]) {
  const int lane = threadIdx.x & 63;
  const bool h = lane & 32, q = lane & 16;
  const double s0 = h ? v[0] : v[2], s1 = h ? v[1] : v[3];
  double k0 = (h ? v[2] : v[0]) + __shfl_xor(s0, 32);
  double k1 = (h ? v[3] : v[1]) + __shfl_xor(s1, 32);
  double x = (q ? k1 : k0) + __shfl_xor(q ? k0 : k1, 16);
  x += dpp_move<0xB1>(x);   // quad_perm(1, 0, 3, 2)
  x += dpp_move<0x4E>(x);   // quad_perm(2, 3, 0, 1)
  x += dpp_move<0x141>(x);  // row_half_mirror
  x += dpp_move<0x140>(x);  // row_mirror
#pragma unroll
  for (int i = 0; i < 4; ++i) v[i] = read_lane(x, 16 * i);
}

// Workgroup sums of four per-thread values (BT threads), stored as one record.
template <int BT>
__device__ __forceinline__ void block_store4(double (&v)[4], double* dst) {
  __shared__ double red[BT / 64][4];
  wave_sum4(v);
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  if (lane == 0) {
#pragma unroll
    for (int q = 0; q < 4; ++q) red[w][q] = v[q];
  }
  __syncthreads();
  if (threadIdx.x < 4) {
    double s = 0.0;
#pragma unroll
    for (int ww = 0; ww < BT / 64; ++ww) s += red[ww][threadIdx.x];
    dst[threadIdx.x] = s;
  }
}

// One entry of the SP2 update z from x (the current X) and y (X^2) as the
// sparse BML formats compute it, each product and sum thresholded (|a| <=
// thr dropped): alg1 forms d = thr(X - X^2) then thr(X -+ d)
// (src/prg_sp2_mod.F90:783-784, :811-823), the other variants thr(X^2) then
// thr(X^2) or thr(2X - thr(X^2)) (:450-453, :328-337).  y is replaced by the
// thresholded X^2 (X - d for alg1) that the idempotency sums read.  apply =
// 0 leaves X unchanged.
__device__ __forceinline__ double thr_drop(double v, double thr) {
  return fabs(v) > thr ? v : 0.0;
}
struct SparseUpdate {
  double z, y;
};
__device__ __forceinline__ SparseUpdate sp2_sparse_update(double x, double y, int apply,
                                                          int sigma, bool alg1, double thr) {
  // alg1: d = thr(X - X^2); X^2 seen by the sums as X - d
  const double d = thr_drop(x - y, thr);
  const double yt = alg1 ? x - d : thr_drop(y, thr);
  const double up = alg1 ? (sigma ? x - d : x + d) : (sigma ? yt : 2.0 * x - yt);
  return SparseUpdate{apply ? thr_drop(up, thr) : x, yt};
}

}  // namespace tile
}  // namespace prg
