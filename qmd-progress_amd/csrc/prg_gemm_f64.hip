// FP64 MFMA GEMM family for gfx950 (v_mfma_f64_16x16x4_f64) on the tiles of
// prg_f64_tile.h: operands straight to registers, the tile edge chosen by how
// its tiles fill the CUs, or staged 128-wide tiles where those fill them better.  For symmetric products (X*X, X*D + D*X, products
// of commuting symmetric matrices) only the upper-triangle tiles are computed;
// the epilogue writes each tile and its transpose, so the result is exactly
// symmetric and the executed flops are half of the algorithmic 2 N^3.
// Workgroup ids are remapped so that each of the 8 XCDs walks a contiguous
// range of output tiles (its own L2 keeps the shared panels).
//
// Epilogues are fused: the SP2 branch update (X <- X^2 or 2X - X^2, decided on
// the device before the product from ||X||_F^2 = Tr X^2), the trace and
// Frobenius partial sums for the next branch decision, and the idempotency
// sums ||X - X^2||_F^2 (genseq) or its core-row restriction (submatrix).
#include "prg_internal.h"

#include "prg_f64_tile.h"
#include "prg_plan.h"
#include "prg_tile.h"

namespace prg {
namespace {

using tile::xcd_remap;
using tile::sym_tile_banded;
using tile::full_tile;
using tile::block_store4;
using f64tile::d4;

// Tile columns of a band: the workgroups an XCD runs at a time cover a block
// of about 6 x 5 to 6 x 10 tiles.
constexpr int kBand = 6;

template <typename S>
__device__ __forceinline__ void zero(d4 (&acc)[S::MB][S::NB]) {
#pragma unroll
  for (int m = 0; m < S::MB; ++m)
#pragma unroll
    for (int n = 0; n < S::NB; ++n) acc[m][n] = d4{0.0, 0.0, 0.0, 0.0};
}

// ------------------------------------------------------------- general GEMM
struct GemmArgs {
  const double* A[2];
  const double* B[2];
  int npair, ld, kdim, nt, n, sym;
  double alpha, beta, gamma;
  const double* Cin;
  double* C;
  const double* dotE;  // optional: partial <C, E> (elementwise product sum)
  double* part;        // per tile [Tr C, ||C||^2, <C, E>, 0] or null
};

// The epilogue of a gemm tile: v = alpha y + beta Cin + gamma I, stored (FUSE
// bit 0: with Cin, bit 1: with <C, E>; in the type, because a branch in each
// group of entries costs the registers of the whole tile).  Symmetric
// products (PLACE = 1, 2): off-diagonal tiles (1) are mirrored; inside a
// diagonal tile (2) the upper half is mirrored onto the lower one, so that the output is exactly symmetric also for two-product
// sums (A0 B0 + A1 B1 accumulates its (r, c) and (c, r) entries in different
// orders).  sums: the lane's part of [Tr C, ||C||^2, <C, E>].
template <typename S, int FUSE, int PLACE>
__device__ __forceinline__ void gemm_finish(const GemmArgs& g, d4 (&acc)[S::MB][S::NB],
                                            int ks, int r0, int c0, double* lds,
                                            const f64tile::Entries<S>& cin, double (&sums)[4]) {
  const int ld = g.ld;
  f64tile::finish_tile<S>(acc, ks, lds, [&](auto grp, auto& y) {
    const int r = ks;
    constexpr int G = decltype(grp)::value, W = f64tile::kWidth<S, G>;
    const int col0 = f64tile::entry_col<S, G>(c0, r);
    double e[S::MB][W];
    if (FUSE & 2) f64tile::load_entries<S, G, W>(g.dotE, ld, r0, c0, r, e);
#pragma unroll
    for (int w = 0; w < W; ++w) {
      const int col = col0 + w;
#pragma unroll
      for (int m = 0; m < S::MB; ++m) {
        const int row = f64tile::entry_row<S>(r0, m);
        double v = y[m][w] * g.alpha;
        if (FUSE & 1) v += g.beta * cin.v[G][m][w];
        const bool diag = PLACE != 1 && (row == col);
        if (PLACE != 1) v += (diag && row < g.n) ? g.gamma : 0.0;
        y[m][w] = v;
        const bool in = !S::kRagged || (row < ld && col < ld);
        if (PLACE != 1) sums[0] += (diag && in) ? v : 0.0;
        // a diagonal tile's upper entries stand for the lower ones too
        const bool counted = in && (PLACE != 2 || row <= col);
        const double vw = !counted ? 0.0 : (PLACE == 2 && !diag) ? 2.0 * v : v;
        sums[1] += counted ? vw * v : 0.0;
        if (FUSE & 2) sums[2] += counted ? vw * e[m][w] : 0.0;
      }
    }
    if (PLACE == 2) {
      f64tile::store_upper<S, W>(g.C, ld, r0, col0, y);
    } else {
      f64tile::store_entries<S, G, W>(g.C, ld, r0, c0, r, y);
      if (PLACE == 1) f64tile::store_mirrored<S, G, W>(g.C, ld, r0, c0, r, y);
    }
  });
  if (PLACE == 1) {
    sums[1] *= 2.0;
    sums[2] *= 2.0;
  }
}

// BT: B is read as stored (not symmetric).
template <typename S, bool BT, int FUSE>
__global__ __launch_bounds__(S::NT, 2) void gemm_kernel(GemmArgs g) {
  __shared__ double lds[S::kLdsDoubles];
  const int t = xcd_remap(blockIdx.x, gridDim.x);
  int I, J;
  if (g.sym) sym_tile_banded<kBand>(t, g.nt, I, J); else full_tile(t, g.nt, I, J);
  const int ks = f64tile::k_wave(), r0 = I * S::TM, c0 = J * S::TM, ld = g.ld;
  int first, count;
  f64tile::k_share<S>(g.kdim / S::CK, ks, first, count);
  d4 acc[S::MB][S::NB];
  zero<S>(acc);
  f64tile::WaveProduct<S, BT> product;
  product.start(g.A[0], g.B[0], g.A[1], g.B[1], g.npair, g.ld, r0, c0, first * S::CK, count);
  f64tile::Entries<S> cin;
  product.run(acc, [&] {
    if (FUSE & 1) cin.load(g.Cin, ld, r0, c0, ks);
  });
  double sums[4] = {0.0, 0.0, 0.0, 0.0};
  if (!g.sym)
    gemm_finish<S, FUSE, 0>(g, acc, ks, r0, c0, lds, cin, sums);
  else if (I != J)
    gemm_finish<S, FUSE, 1>(g, acc, ks, r0, c0, lds, cin, sums);
  else
    gemm_finish<S, FUSE, 2>(g, acc, ks, r0, c0, lds, cin, sums);
  if (g.part) block_store4<S::NT>(sums, g.part + 4 * (size_t)t);
}

// --------------------------------------------------------- staged tiles
// The same products on 128 x 128 tiles, one per workgroup: 16-deep slabs of
// both panels go through LDS with the next slab in registers, four waves in a
// 2 x 2 grid of 4 x 4 MFMA blocks.  B is read along its columns, 64 bytes per
// thread, where a 48-wide tile's fragments of an operand that is not symmetric
// take 64 bytes of each of 16 columns; with two workgroups per CU 67 to 69
// TFLOP/s, whatever the leading dimension.  What it costs is the tiles' size
// (see staged_is_faster).
namespace staged {
constexpr int BM = 128, BK = 16, NT = 256;
struct Slabs {
  double A[BK][BM + 4], B[BK][BM + 4];  // rows padded
};

// acc = the tile (I, J) of A[0] B[0] (+ A[1] B[1]).
__device__ __forceinline__ void product(const double* const (&A)[2], const double* const (&B)[2],
                                        int npair, int ld, int kdim, int I, int J, Slabs& lds,
                                        d4 (&acc)[4][4]) {
  typedef f64tile::d2 d2;
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, wm = w & 1, wn = w >> 1;
  const int ar = (tid & 63) * 2, ak = tid >> 6;  // A: rows ar, ar + 1; k = ak + 4 q
  const int bj = tid >> 1, bk = (tid & 1) * 8;   // B: column bj; k = bk .. bk + 7
  const int slabs = kdim / BK, total = slabs * npair;
  d2 ra[4], rb[4];
  auto load = [&](int s) {
    const int p = s >= slabs, k0 = (s - p * slabs) * BK;
    const double* Ap = (p ? A[1] : A[0]) + (size_t)I * BM + ar;
    const double* Bp = (p ? B[1] : B[0]) + (size_t)(J * BM + bj) * ld + k0 + bk;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      ra[q] = *(const d2*)(Ap + (size_t)(k0 + ak + 4 * q) * ld);
      rb[q] = *(const d2*)(Bp + 2 * q);
    }
  };
#pragma unroll
  for (int m = 0; m < 4; ++m)
#pragma unroll
    for (int n = 0; n < 4; ++n) acc[m][n] = d4{0.0, 0.0, 0.0, 0.0};
  load(0);
  for (int s = 0; s < total; ++s) {
    __syncthreads();
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      lds.A[ak + 4 * q][ar] = ra[q].x;
      lds.A[ak + 4 * q][ar + 1] = ra[q].y;
      lds.B[bk + 2 * q][bj] = rb[q].x;
      lds.B[bk + 2 * q + 1][bj] = rb[q].y;
    }
    __syncthreads();
    if (s + 1 < total) load(s + 1);
#pragma unroll
    for (int kk = 0; kk < BK / 4; ++kk) {
      const int kr = kk * 4 + (lane >> 4);
      double a[4], b[4];
#pragma unroll
      for (int m = 0; m < 4; ++m) a[m] = lds.A[kr][wm * 64 + m * 16 + (lane & 15)];
#pragma unroll
      for (int n = 0; n < 4; ++n) b[n] = lds.B[kr][wn * 64 + n * 16 + (lane & 15)];
#pragma unroll
      for (int m = 0; m < 4; ++m)
#pragma unroll
        for (int n = 0; n < 4; ++n)
          acc[m][n] = __builtin_amdgcn_mfma_f64_16x16x4f64(b[n], a[m], acc[m][n], 0, 0, 0);
    }
  }
}

// f(row, column, entry) for the lane's entries, one MFMA block at a time (the
// loads of a block's entries are not hoisted over another's: registers).
template <typename F>
__device__ __forceinline__ void for_entries(const d4 (&acc)[4][4], int I, int J, F&& f) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int row0 = I * BM + (w & 1) * 64 + (lane & 15), col0 = J * BM + (w >> 1) * 64 + (lane >> 4);
#pragma unroll
  for (int m = 0; m < 4; ++m)
#pragma unroll
    for (int n = 0; n < 4; ++n) {
#pragma unroll
      for (int r = 0; r < 4; ++r) f(row0 + 16 * m, col0 + 16 * n + 4 * r, acc[m][n][r]);
      __builtin_amdgcn_sched_barrier(0);
    }
}
}  // namespace staged

template <bool SYM>
__global__ __launch_bounds__(staged::NT, 2) void gemm_staged_kernel(GemmArgs g) {
  __shared__ staged::Slabs lds;
  const int t = xcd_remap(blockIdx.x, gridDim.x), ld = g.ld;
  int I, J;
  if (SYM) tile::sym_tile(t, I, J); else full_tile(t, g.nt, I, J);
  d4 acc[4][4];
  staged::product(g.A, g.B, g.npair, ld, g.kdim, I, J, lds, acc);
  double sums[4] = {0.0, 0.0, 0.0, 0.0};
  staged::for_entries(acc, I, J, [&](int row, int col, double y) {
    if (SYM && row > col) return;  // the lower half of a diagonal tile
    const bool diag = (row == col);
    const double wgt = SYM && !diag ? 2.0 : 1.0;
    const size_t idx = row + (size_t)col * ld;
    double v = y * g.alpha;
    if (g.beta != 0.0) v += g.beta * g.Cin[idx];
    v += (diag && row < g.n) ? g.gamma : 0.0;
    sums[0] += diag ? v : 0.0;
    sums[1] += wgt * v * v;
    if (g.dotE) sums[2] += wgt * v * g.dotE[idx];
    g.C[idx] = v;
    if (SYM && !diag) g.C[col + (size_t)row * ld] = v;
  });
  if (g.part) block_store4<staged::NT>(sums, g.part + 4 * (size_t)t);
}

// ------------------------------------------------------------- SP2 step
struct Sp2Args {
  const double* buf[2];  // ping-pong X buffers
  const double* dbuf[2]; // ping-pong D buffers (response step)
  int ld, kdim, nt, ntiles;
  int cur;               // which buffer holds X
  int lazy;              // multiply before the step is planned
  Sp2Link link;
  double* part;  // per tile [||Xn||^2, Tr Xn, idem, Tr Y]
};

// The SP2 update of a finished product tile: z = cb x + ca y with (ca, cb) =
// (1, 0) for X^2, (-1, 2) for 2X - X^2, (0, 1) when the product is only
// measured (X unchanged); sums: the lane's part of [||Xn||^2, Tr Xn,
// ||X - X^2||^2 (core rows for submatrix), Tr Y].  MIRROR: the tile stands
// for its transposed place too.  Diagonal tiles are symmetric by themselves:
// entries (r, c) and (c, r) add the same products in the same order.  THR:
// with the sparse formats' thresholding.
template <typename S, bool THR, bool MIRROR>
__device__ __forceinline__ void sp2_finish(const Sp2Args& g, const Sp2State* st,
                                           d4 (&acc)[S::MB][S::NB], int ks,
                                           int r0, int c0, double* lds,
                                           const f64tile::Entries<S>& xs, double (&sums)[4]) {
  const int ld = g.ld, cur = g.cur, apply = st->apply, sigma = st->sigma;
  const int variant = st->variant;
  double* Xn = const_cast<double*>(g.buf[cur ^ 1]);
  const double ca = apply ? (sigma ? 1.0 : -1.0) : 0.0;
  const double cb = apply ? (sigma ? 0.0 : 2.0) : 1.0;
  const bool core_only = (variant == V_SUBMATRIX);
  const int core = st->core;
  const double thr = st->threshold;
  const bool alg1 = (variant == V_ALG1 || variant == V_ALG1_GENSEQ || variant == V_SEQ_ALG1);
  f64tile::finish_tile<S>(acc, ks, lds, [&](auto grp, auto& y) {
    const int r = ks;
    constexpr int G = decltype(grp)::value, W = f64tile::kWidth<S, G>;
    const int col0 = f64tile::entry_col<S, G>(c0, r);
#pragma unroll
    for (int w = 0; w < W; ++w) {
      const int col = col0 + w;
#pragma unroll
      for (int m = 0; m < S::MB; ++m) {
        const int row = f64tile::entry_row<S>(r0, m);
        const double xv = xs.v[G][m][w];
        // rows and columns past the buffer repeat its last ones
        double yv = (!S::kRagged || (row < ld && col < ld)) ? y[m][w] : 0.0, z;
        if (THR) {
          const tile::SparseUpdate u = tile::sp2_sparse_update(xv, yv, apply, sigma, alg1, thr);
          z = u.z;
          yv = u.y;
        } else {
          z = fma(cb, xv, ca * yv);
        }
        const double dxy = xv - yv;
        sums[0] = fma(z, z, sums[0]);
        if (core_only) {
          sums[2] += ((row < core ? 1.0 : 0.0) + (MIRROR && col < core ? 1.0 : 0.0)) * dxy * dxy;
        } else {
          sums[2] = fma(dxy, dxy, sums[2]);
        }
        if (!MIRROR) {
          sums[1] += (row == col) ? z : 0.0;
          sums[3] += (row == col) ? yv : 0.0;
        }
        y[m][w] = z;
      }
    }
    f64tile::store_entries<S, G, W>(Xn, ld, r0, c0, r, y);
    if (MIRROR) f64tile::store_mirrored<S, G, W>(Xn, ld, r0, c0, r, y);
  });
  if (MIRROR) {
    sums[0] *= 2.0;
    if (!core_only) sums[2] *= 2.0;
  }
}

// The response's update of a finished Y = X D + D X: Dn = Y (sigma = 1) or
// 2 D - Y.
template <typename S>
__device__ __forceinline__ void response_finish(const Sp2Args& g, const Sp2State* st,
                                                d4 (&acc)[S::MB][S::NB],
                                                int ks, bool mirror, int r0, int c0,
                                                double* lds, const f64tile::Entries<S>& ds) {
  const int cur = g.cur, sigma = st->sigma, ld = g.ld;
  const double ca = sigma ? 1.0 : -1.0, cb = sigma ? 0.0 : 2.0;
  double* Dn = const_cast<double*>(g.dbuf[cur ^ 1]);
  f64tile::finish_tile<S>(acc, ks, lds, [&](auto grp, auto& y) {
    const int r = ks;
    constexpr int G = decltype(grp)::value, W = f64tile::kWidth<S, G>;
    const int col0 = f64tile::entry_col<S, G>(c0, r);
#pragma unroll
    for (int w = 0; w < W; ++w)
#pragma unroll
      for (int m = 0; m < S::MB; ++m)
        y[m][w] = fma(cb, ds.v[G][m][w], ca * y[m][w]);
    if (mirror) {
      f64tile::store_entries<S, G, W>(Dn, ld, r0, c0, r, y);
      f64tile::store_mirrored<S, G, W>(Dn, ld, r0, c0, r, y);
    } else {
      // X D + D X accumulates its (r, c) and (c, r) entries in different
      // orders: inside a diagonal tile the upper half is mirrored
      f64tile::store_upper<S, W>(Dn, ld, r0, col0, y);
    }
  });
}

// One SP2 step: absorb the previous step's sums and plan (sp2_link, wave 0; a
// launch of its own does both above 1280 tiles), product, update.  The current X is known before the
// plan: every step before the last toggles the buffers (g.cur), and the last
// plans nothing after it.  So the product's first operands are on their way
// while wave 0 plans, and (g.lazy) the other waves multiply meanwhile: the
// plan is needed by the update only.  The launch that finds the loop ended
// computes a product that is thrown away.  (N = 1300: 53.1 us per step with
// every workgroup waiting for its plan, 49.4 so.  A test in the main loop
// whether to go on cost the 48-wide tile a fifth.)
// RESP: the response step Y = X D + D X (both products in the same
// accumulators), Dn = Y or 2 D - Y, in the same launch, its workgroups (twice
// the work) first.  Partial sums of the X tile t go to part[4 t].
// FULL: all tiles, B as stored: X need not be symmetric (the response's is; of
// its tiles the upper triangle's are mirrored as in the other form).
template <typename S, bool THR, bool RESP, bool FULL>
__global__ __launch_bounds__(S::NT, 2) void sp2_step_kernel(Sp2Args g) {
  __shared__ double lds[S::kLdsDoubles];
  __shared__ __attribute__((aligned(16))) char head[kSp2HeadBytes];
  Sp2LinkReads reads;
  sp2_link_read(g.link, reads);
  const bool resp = RESP && (int)blockIdx.x < g.ntiles;
  const int t = xcd_remap(blockIdx.x - (RESP && !resp ? g.ntiles : 0), g.ntiles);
  int I, J, first, count;
  if (FULL) full_tile(t, g.nt, I, J); else sym_tile_banded<kBand>(t, g.nt, I, J);
  const int ks = f64tile::k_wave(), r0 = I * S::TM, c0 = J * S::TM, ld = g.ld;
  f64tile::k_share<S>(g.kdim / S::CK, ks, first, count);
  const double* X = g.buf[g.cur];
  const double* D = g.dbuf[g.cur];
  f64tile::WaveProduct<S, FULL> product;
  product.start(X, resp ? D : X, D, X, resp ? 2 : 1, ld, r0, c0, first * S::CK, count);
  sp2_link(g.link, reads, head);
  if (!reads.planned) return;
  const volatile Sp2State* hv = (const volatile Sp2State*)head;
  if (!g.lazy) {
    __syncthreads();
    if (!hv->planned) return;
  }
  d4 acc[S::MB][S::NB];
  zero<S>(acc);
  f64tile::Entries<S> xs;
  product.run(acc, [&] { xs.load(resp ? D : X, ld, r0, c0, ks); });
  if (g.lazy) {
    __syncthreads();
    if (!hv->planned) return;
  }
  const Sp2State* st = (const Sp2State*)head;
  if (resp) {
    if (!st->apply || I > J) return;
    response_finish<S>(g, st, acc, ks, I != J, r0, c0, lds, xs);
    return;
  }
  double sums[4] = {0.0, 0.0, 0.0, 0.0};
  if (!FULL && I != J)
    sp2_finish<S, THR, true>(g, st, acc, ks, r0, c0, lds, xs, sums);
  else
    sp2_finish<S, THR, false>(g, st, acc, ks, r0, c0, lds, xs, sums);
  block_store4<S::NT>(sums, g.part + 4 * (size_t)t);
}

// The step on staged tiles, planned by a launch of its own: the X update, or
// (RESP) the response's.
template <bool RESP>
__global__ __launch_bounds__(staged::NT, 2) void sp2_staged_kernel(Sp2Args g) {
  __shared__ staged::Slabs lds;
  const Sp2State* st = g.link.in;
  if (!st->planned || (RESP && !st->apply)) return;
  const int ld = g.ld, apply = st->apply, sigma = st->sigma;
  const double ca = apply ? (sigma ? 1.0 : -1.0) : 0.0, cb = apply ? (sigma ? 0.0 : 2.0) : 1.0;
  const double* X = g.buf[g.cur];
  const double* D = g.dbuf[g.cur];
  const int t = xcd_remap(blockIdx.x, gridDim.x);
  int I, J;
  tile::sym_tile(t, I, J);
  d4 acc[4][4];
  if (RESP) {
    double* Dn = const_cast<double*>(g.dbuf[g.cur ^ 1]);
    staged::product({X, D}, {D, X}, 2, ld, g.kdim, I, J, lds, acc);
    staged::for_entries(acc, I, J, [&](int row, int col, double y) {
      if (row > col) return;  // X D + D X adds (r, c) and (c, r) in different orders
      const double z = fma(cb, D[row + (size_t)col * ld], ca * y);
      Dn[row + (size_t)col * ld] = z;
      Dn[col + (size_t)row * ld] = z;
    });
    return;
  }
  double* Xn = const_cast<double*>(g.buf[g.cur ^ 1]);
  const int core = st->variant == V_SUBMATRIX ? st->core : 0x7fffffff;
  const bool mirror = (I != J);
  const double wz = mirror ? 2.0 : 1.0;
  double sums[4] = {0.0, 0.0, 0.0, 0.0};
  staged::product({X, X}, {X, X}, 1, ld, g.kdim, I, J, lds, acc);
  staged::for_entries(acc, I, J, [&](int row, int col, double y) {
    const size_t idx = row + (size_t)col * ld;
    const double x = X[idx], z = fma(cb, x, ca * y), d = x - y;
    const bool diag = (row == col);
    sums[0] += wz * z * z;
    sums[1] += diag ? z : 0.0;
    sums[2] += ((row < core ? 1.0 : 0.0) + (mirror && col < core ? 1.0 : 0.0)) * d * d;
    sums[3] += diag ? y : 0.0;
    Xn[idx] = z;
    // on a diagonal tile the lane rewrites its own entry
    Xn[mirror ? col + (size_t)row * ld : idx] = z;
  });
  block_store4<staged::NT>(sums, g.part + 4 * (size_t)t);
}

template <typename S, bool BT>
void launch_gemm_fused(const GemmArgs& g, int nb, int fuse) {
  void (*k)(GemmArgs) = fuse == 0   ? gemm_kernel<S, BT, 0>
                        : fuse == 1 ? gemm_kernel<S, BT, 1>
                        : fuse == 2 ? gemm_kernel<S, BT, 2>
                                    : gemm_kernel<S, BT, 3>;
  hipLaunchKernelGGL(k, dim3(nb), dim3(S::NT), 0, stream(), g);
}

template <typename S>
void launch_gemm(const GemmArgs& g, int nb, bool b_as_stored, int fuse) {
  if (b_as_stored)
    launch_gemm_fused<S, true>(g, nb, fuse);
  else
    launch_gemm_fused<S, false>(g, nb, fuse);
}

// The tiles of a product.
struct GemmShape {
  int edge, tiles, kdim;
  double flops() const { return (double)tiles * 2.0 * edge * edge * kdim; }
};
GemmShape gemm_shape(int n, int ld, bool sym, bool b_symmetric) {
  const int edge = f64tile::staged_is_faster(ld, sym, b_symmetric) ? staged::BM
                                                                   : f64tile::tile_edge(ld, sym);
  // the padding of the operands is zero, so K ends at n's chunk
  return GemmShape{edge, f64tile::tile_count(ld, edge, sym), (n + 31) / 32 * 32};
}

// The tiles of an SP2 step.  Up to 128 rows all of them, so that a matrix which
// is not symmetric is squared as the reference squares it; larger ones are
// taken as symmetric.  (N = 100: 6.8 us per step on 64 workgroups, 7.0 on the
// 36 of one triangle.)
bool step_is_full(int ld) { return ld == kTile; }
GemmShape step_shape(int n, int ld, bool thresholded = false) {
  GemmShape s = gemm_shape(n, ld, true, true);
  if (s.edge == staged::BM && thresholded) {
    s.edge = f64tile::tile_edge(ld, true);
    s.tiles = f64tile::tile_count(ld, s.edge, true);
  }
  if (step_is_full(ld)) {
    s.edge = 16;
    s.tiles = f64tile::tile_count(ld, s.edge, false);
  }
  return s;
}

}  // namespace

int gemm(int npair, const DMat* A, const DMat* B, double alpha, double beta, const DMat* Cin,
         double gamma, DMat C, int sym, double* d_part, int* ntiles, const DMat* dotE,
         bool b_symmetric) {
  if (npair < 1 || npair > 2) {
    set_error(ERR_ARG, "gemm: npair must be 1 or 2");
    return ERR_ARG;
  }
  const int ld = C.ld;
  for (int p = 0; p < npair; ++p) {
    if (A[p].ld != ld || B[p].ld != ld || !A[p].p || !B[p].p) {
      set_error(ERR_ARG, "gemm: operand layout mismatch");
      return ERR_ARG;
    }
  }
  if (beta != 0.0 && (!Cin || Cin->ld != ld || !Cin->p)) {
    set_error(ERR_ARG, "gemm: beta != 0 needs an input C of the same layout");
    return ERR_ARG;
  }
  if (ld % kTile != 0 || ld <= 0) {
    set_error(ERR_ARG, "gemm: leading dimension must be a positive multiple of 128");
    return ERR_ARG;
  }
  GemmArgs g;
  for (int p = 0; p < 2; ++p) {
    g.A[p] = A[p < npair ? p : 0].p;
    g.B[p] = B[p < npair ? p : 0].p;
  }
  const GemmShape shape = gemm_shape(C.n, ld, sym != 0, b_symmetric);
  g.npair = npair;
  g.ld = ld;
  g.kdim = shape.kdim;
  g.nt = (ld + shape.edge - 1) / shape.edge;
  g.n = C.n;
  g.sym = sym;
  g.alpha = alpha;
  g.beta = beta;
  g.gamma = gamma;
  g.Cin = Cin ? Cin->p : nullptr;
  g.C = C.p;
  g.dotE = dotE ? dotE->p : nullptr;
  g.part = d_part;
  const int nb = shape.tiles;
  if (ntiles) *ntiles = nb;
  if (shape.edge == staged::BM) {
    hipLaunchKernelGGL(sym ? gemm_staged_kernel<true> : gemm_staged_kernel<false>, dim3(nb),
                       dim3(staged::NT), 0, stream(), g);
    PRG_HIP_CHECK(hipGetLastError());
    return OK;
  }
  const int fuse = (beta != 0.0 ? 1 : 0) | (dotE ? 2 : 0);
#define PRG_CALL(S) launch_gemm<S>(g, nb, !b_symmetric, fuse)
  PRG_F64_SHAPE_DISPATCH(shape.edge, PRG_CALL)
#undef PRG_CALL
  PRG_HIP_CHECK(hipGetLastError());
  return OK;
}

double gemm_flops(int n, int ld, bool sym, bool b_symmetric) {
  return gemm_shape(n, ld, sym, b_symmetric).flops();
}

double sp2_step_flops(int n, int ld) { return step_shape(n, ld).flops(); }

int gemm_tiles(int ld, int sym) {
  return f64tile::tile_count(ld, f64tile::tile_edge(ld, sym != 0), sym != 0);
}

// (of the 48-wide tiles where the staged ones are fewer)
int sp2_step_tiles(int ld) { return step_shape(ld, ld, true).tiles; }

int sp2_step(const DMat& x0, const DMat& x1, const DMat* d0, const DMat* d1, const Sp2Link& link,
             double* d_part, int* ntiles, bool thresholded, int cur) {
  Sp2Args g;
  g.cur = cur;
  g.buf[0] = x0.p;
  g.buf[1] = x1.p;
  g.dbuf[0] = d0 ? d0->p : nullptr;
  g.dbuf[1] = d1 ? d1->p : nullptr;
  g.ld = x0.ld;
  const GemmShape shape = step_shape(x0.n, x0.ld, thresholded);
  const int edge = shape.edge;
  g.kdim = shape.kdim;
  g.nt = (x0.ld + edge - 1) / edge;
  g.ntiles = shape.tiles;
  g.lazy = link.part != nullptr;
  g.link = link;
  g.part = d_part;
  if (ntiles) *ntiles = g.ntiles;
  auto launch = [&](auto shape_type, auto full) {
    typedef decltype(shape_type) S;
    constexpr bool F = decltype(full)::value;
    void (*k)(Sp2Args) = d0            ? sp2_step_kernel<S, false, true, F>
                         : thresholded ? sp2_step_kernel<S, true, false, F>
                                       : sp2_step_kernel<S, false, false, F>;
    hipLaunchKernelGGL(k, dim3(d0 ? 2 * g.ntiles : g.ntiles), dim3(S::NT), 0, stream(), g);
  };
  if (edge == staged::BM) {
    if (d0)
      hipLaunchKernelGGL(sp2_staged_kernel<true>, dim3(g.ntiles), dim3(staged::NT), 0, stream(), g);
    hipLaunchKernelGGL(sp2_staged_kernel<false>, dim3(g.ntiles), dim3(staged::NT), 0, stream(), g);
  } else if (step_is_full(x0.ld)) {
    launch(f64tile::S16{}, std::true_type{});
  } else {
#define PRG_CALL(S) launch(S{}, std::false_type{})
    PRG_F64_SHAPE_DISPATCH(edge, PRG_CALL)
#undef PRG_CALL
  }
  PRG_HIP_CHECK(hipGetLastError());
  return OK;
}

}  // namespace prg
