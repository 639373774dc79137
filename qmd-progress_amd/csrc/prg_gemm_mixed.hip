// Mixed-precision SP2 products for gfx950.
//
// PRG_PREC_F16SPLIT: X (symmetric, |x| <= 1) is carried as an FP64 master and
// two FP16 planes, hi = fp16(x) and lo = fp16((x - hi) * 2^11), so that
// x ~= hi + 2^-11 lo (about 22 significant bits).  One fused kernel computes
//   X^2 ~= hi*hi + 2^-11 (hi*lo + lo*hi)
// with v_mfma_f32_16x16x32_f16 (FP32 accumulation, two accumulator sets),
// applies the SP2 branch update in FP64 against the master copy, writes the
// next master and its hi/lo planes, and emits the same trace / Frobenius
// partial sums as the FP64 kernel, so the FP64 bookkeeping and stopping rules
// are shared.  The dropped lo*lo term is 2^-22 relative.
//
// PRG_PREC_BF16SPLIT is the same kernel on BF16 planes, hi = bf16(x) and
// lo = bf16((x - hi) * 2^8) (about 16 significant bits), with
// v_mfma_f32_16x16x32_bf16.
//
// Because the planes are symmetric, the A operand (rows of the I panel) and
// the B operand (columns of the J panel) are both read as contiguous slabs of
// a plane.
#include "prg_sp2.h"
#include "prg_lds_dma.h"
#include "prg_tile.h"

namespace prg {
namespace {

using tile::block_store4;
using tile::sym_tile;
using tile::sym_tile_banded;
using tile::xcd_remap;

typedef float f4 __attribute__((ext_vector_type(4)));

// The two 16-bit split formats: element type, lo scale (2^(mantissa bits)),
// and the 16x16x32 MFMA with FP32 accumulation.
template <typename T>
struct Split;
template <>
struct Split<_Float16> {
  typedef _Float16 v8 __attribute__((ext_vector_type(8)));
  static constexpr double kScale = 2048.0;
  static __device__ __forceinline__ f4 mfma(v8 a, v8 b, f4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
  }
};
template <>
struct Split<__bf16> {
  typedef __bf16 v8 __attribute__((ext_vector_type(8)));
  static constexpr double kScale = 256.0;
  static __device__ __forceinline__ f4 mfma(v8 a, v8 b, f4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
  }
};

constexpr int BM = 128, NT = 256;
constexpr int KB = 32;                 // halves of K per slab and per plane block
constexpr int kRing = 64 * 1024;       // the slabs in LDS: two workgroups per CU

// Planes are stored in blocks of 32 columns, element (r, k) at
// (k / 32) 32 ld + 32 r + k % 32: the 128 rows of a slab are 8 KB in one piece.
__device__ __forceinline__ size_t plane_at(int r, int k, int ld) {
  return (size_t)(k >> 5) * KB * ld + (size_t)r * KB + (k & 31);
}

// One tile of A B (both symmetric, by their planes) over the whole K, 128 x 128
// (H = 4) or 64 x 64 (H = 2): four waves in a 2 x 2 grid, each H x H blocks of
// 16 x 16.  The slabs are copied global -> LDS directly (dma16), the ring's
// other slabs (1 or 3) while this one is multiplied; a panel of a slab is 2 H
// chunks of 16 rows x 64 bytes, wave w copies chunks w + 4 q.  Within a
// row the 16-byte chunk g sits in slot g ^ ((row >> 1) & 3), which keeps the
// fragment reads of 8 consecutive rows on distinct banks.  Two workgroups
// share a CU: one multiplies while the other waits for its slab and reads its
// fragments.
//
// Bound: the operand stream from L2, 32 KB per slab of 3 x 128 x 128 x 32
// products (42 B/clk per CU at the 16-bit peak).  Registers: 128 for the two
// accumulator sets, 64 for a slab's fragments.
template <typename T, int H>
__device__ __forceinline__ void split_tile(const T* ahi, const T* alo, const T* bhi, const T* blo,
                                           int ld, int I, int J, int8_t* ring, f4 (&hh)[H][H],
                                           f4 (&xx)[H][H]) {
  constexpr int E = 32 * H;            // tile edge
  constexpr int kPanel = E * KB * 2;   // bytes of one operand plane's slab
  constexpr int kSlab = 4 * kPanel;    // A hi, A lo, B hi, B lo
  constexpr int D = kRing / kSlab;     // slabs in the ring
  constexpr int CPP = H / 2;           // chunks of a panel per wave
  typedef typename Split<T>::v8 h8;
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6), wm = w & 1, wn = w >> 1;
  const int lrow = lane >> 2;
  const uint32_t voff = (uint32_t)(lrow * 64 + 16 * ((lane & 3) ^ ((lrow >> 1) & 3)));
  const uint32_t ring0 = __builtin_amdgcn_readfirstlane(lds_dma::lds_addr(ring));
  const size_t kblock = (size_t)KB * ld * sizeof(T);
  const uint64_t panel[4] = {
      lds_dma::uniform64((uint64_t)(uintptr_t)(ahi + (size_t)I * E * KB)),
      lds_dma::uniform64((uint64_t)(uintptr_t)(alo + (size_t)I * E * KB)),
      lds_dma::uniform64((uint64_t)(uintptr_t)(bhi + (size_t)J * E * KB)),
      lds_dma::uniform64((uint64_t)(uintptr_t)(blo + (size_t)J * E * KB))};
  auto issue = [&](int s) {
    const size_t off = (size_t)s * kblock;
    const uint32_t slot = ring0 + kSlab * (s % D);
#pragma unroll
    for (int q = 0; q < 4 * CPP; ++q) {
      const int c = w + 4 * (q % CPP);  // chunk of its panel
      lds_dma::dma16(panel[q / CPP] + off + 1024 * c, voff,
                     __builtin_amdgcn_readfirstlane(slot + kPanel * (q / CPP) + 1024 * c));
    }
  };
  const int fo = (lane & 15) * 64 + 16 * ((lane >> 4) ^ (((lane & 15) >> 1) & 3));
  const int8_t* fa = ring + wm * (E / 2) * 64 + fo;
  const int8_t* fb = ring + 2 * kPanel + wn * (E / 2) * 64 + fo;
#pragma unroll
  for (int m = 0; m < H; ++m)
#pragma unroll
    for (int n = 0; n < H; ++n) {
      hh[m][n] = f4{0.f, 0.f, 0.f, 0.f};
      xx[m][n] = f4{0.f, 0.f, 0.f, 0.f};
    }
  const int slabs = ld / KB;
#pragma unroll
  for (int s = 0; s < D - 1; ++s)
    if (s < slabs) issue(s);
  for (int s = 0; s < slabs; ++s) {
    // slab s has landed in every wave (the D - 2 after it may be in flight),
    // and every wave has read slab s - 1
    if (s + D - 2 < slabs)
      lds_dma::wait_vm_barrier<(D - 2) * 4 * CPP>();
    else
      lds_dma::wait_vm_barrier<0>();
    if (s + D - 1 < slabs) issue(s + D - 1);
    const int o = kSlab * (s % D);
    h8 ah[H], al[H], bh[H], bl[H];
#pragma unroll
    for (int m = 0; m < H; ++m) ah[m] = *(const h8*)(fa + o + 1024 * m);
#pragma unroll
    for (int n = 0; n < H; ++n) bh[n] = *(const h8*)(fb + o + 1024 * n);
#pragma unroll
    for (int n = 0; n < H; ++n) bl[n] = *(const h8*)(fb + o + kPanel + 1024 * n);
#pragma unroll
    for (int m = 0; m < H; ++m) al[m] = *(const h8*)(fa + o + kPanel + 1024 * m);
#pragma unroll
    for (int m = 0; m < H; ++m)
#pragma unroll
      for (int n = 0; n < H; ++n) hh[m][n] = Split<T>::mfma(bh[n], ah[m], hh[m][n]);
#pragma unroll
    for (int m = 0; m < H; ++m)
#pragma unroll
      for (int n = 0; n < H; ++n) xx[m][n] = Split<T>::mfma(bl[n], ah[m], xx[m][n]);
#pragma unroll
    for (int m = 0; m < H; ++m)
#pragma unroll
      for (int n = 0; n < H; ++n) xx[m][n] = Split<T>::mfma(bh[n], al[m], xx[m][n]);
  }
}

// Operands were swapped, so a lane holds (A B)[row][col] with
// row = lane % 16 and col = 4 (lane / 16) + r inside each 16 x 16 block.
template <int H>
struct SplitAt {
  int lane, row0, col0;  // the lane's first row and column
  int w;
  __device__ SplitAt(int I, int J) {
    lane = threadIdx.x & 63;
    w = threadIdx.x >> 6;
    row0 = 32 * H * I + (w & 1) * 16 * H + (lane & 15);
    col0 = 32 * H * J + (w >> 1) * 16 * H + 4 * (lane >> 4);
  }
};

constexpr int kBand = 8;  // tile columns of a band: an XCD's 64 workgroups cover 8 x 8 tiles

// The tiles of a launch: the first `full` upper-triangle 128 x 128 ones (in
// banded order), and the rest as four 64 x 64 ones each.
struct SplitTile {
  int I, J;
  bool quarter;
  // false: a quarter below the diagonal, left to its mirror
  __device__ bool find(int nt, int full) {
    quarter = (int)blockIdx.x >= full;
    const int q = (int)blockIdx.x - full;
    sym_tile_banded<kBand>(quarter ? full + q / 4 : xcd_remap(blockIdx.x, full), nt, I, J);
    if (quarter) {
      I = 2 * I + (q & 1);
      J = 2 * J + ((q >> 1) & 1);
    }
    return I <= J;
  }
};

struct F16Args {
  const double* buf[2];         // FP64 master ping-pong (lower triangle)
  const void* hi[2];            // hi planes ping-pong (T)
  const void* lo[2];            // lo planes ping-pong (T)
  int ld, nt, full;
  Sp2State* st;
  double* part;
};


// The upper-triangle tile (I, J) of X^2 and the SP2 update.  The FP64 master
// lives in the lower triangle (and the whole of each diagonal tile), where a
// lane's four columns are 32 contiguous bytes; the loop's end restores the
// upper one.  Both positions of the planes are written: (row,
// col) by the lane's four columns at a time, (col, row) after a transposition
// of each wave's block through LDS, 8 bytes per lane each.
template <typename T, int H>
__device__ __forceinline__ void sp2_split_tile(const F16Args& g, const volatile Sp2State* stv,
                                               int I, int J, int8_t* ring, double (&sums)[4]) {
  constexpr double kScale = Split<T>::kScale;
  constexpr int kPitch = 16 * H + 4;  // halves per row of a wave's block in LDS
  const int apply = stv->apply, sigma = stv->sigma, cur = stv->cur;
  // prg_sp2_submatrix: the idempotency sum runs over the first `core` rows
  // (and, by symmetry, the mirrored columns) only
  const int core_lim = (stv->variant == V_SUBMATRIX) ? stv->core : 0x7fffffff;
  const int ld = g.ld;
  f4 hh[H][H], xx[H][H];
  split_tile<T, H>((const T*)g.hi[cur], (const T*)g.lo[cur], (const T*)g.hi[cur], (const T*)g.lo[cur],
                   ld, I, J, ring, hh, xx);
  const double* X = g.buf[cur];
  double* Xn = const_cast<double*>(g.buf[cur ^ 1]);
  T* hin = (T*)const_cast<void*>(g.hi[cur ^ 1]);
  T* lon = (T*)const_cast<void*>(g.lo[cur ^ 1]);
  const double ca = apply ? (sigma ? 1.0 : -1.0) : 0.0;
  const double cb = apply ? (sigma ? 0.0 : 2.0) : 1.0;
  const SplitAt<H> at(I, J);
  typedef T t4 __attribute__((ext_vector_type(4)));
  // every wave is done with the ring: its LDS takes the waves' blocks
  lds_dma::wait_vm_barrier<0>();
  T* block = (T*)ring + (size_t)at.w * 16 * H * kPitch;
  if (I != J) {
#pragma unroll
    for (int m = 0; m < H; ++m) {
      const int row = at.row0 + 16 * m;
      const double wrow = row < core_lim ? 1.0 : 0.0;
      t4 lov[H];
#pragma unroll
      for (int n = 0; n < H; ++n) {
        const int col = at.col0 + 16 * n;
        const double2* xp = (const double2*)(X + col + (size_t)row * ld);
        const double2 u = xp[0], v = xp[1];
        const double xs[4] = {u.x, u.y, v.x, v.y};
        double z[4];
        t4 h, l;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const double y = (double)hh[m][n][r] + (1.0 / kScale) * (double)xx[m][n][r];
          z[r] = fma(cb, xs[r], ca * y);
          const double d = xs[r] - y;
          sums[0] += 2.0 * z[r] * z[r];
          sums[2] += (wrow + (col + r < core_lim ? 1.0 : 0.0)) * d * d;
          h[r] = (T)z[r];
          l[r] = (T)((z[r] - (double)h[r]) * kScale);
        }
        double2* zp = (double2*)(Xn + col + (size_t)row * ld);
        zp[0] = double2{z[0], z[1]};
        zp[1] = double2{z[2], z[3]};
        const size_t pi = plane_at(row, col, ld);
        *(t4*)(hin + pi) = h;
        *(t4*)(lon + pi) = l;
        *(t4*)(block + (16 * m + (at.lane & 15)) * kPitch + 16 * n + 4 * (at.lane >> 4)) = h;
        lov[n] = l;
        __builtin_amdgcn_sched_barrier(0);
      }
      // the lo halves wait in the accumulators' place for the second pass
#pragma unroll
      for (int n = 0; n < H; ++n) {
        const uint2 b = __builtin_bit_cast(uint2, lov[n]);
        hh[m][n][0] = __uint_as_float(b.x);
        hh[m][n][1] = __uint_as_float(b.y);
      }
    }
    // Transposed store of the wave's block: lane b handles the 4 x 4 blocks
    // (row block b % RB, column blocks b / RB + CB q), RB lanes covering the
    // 4 RB rows, i.e. runs of 64 bytes per column.
    auto mirror = [&](T* plane) {
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
      constexpr int RB = 4 * H, CB = 64 / RB;
      const int rb = 4 * (at.lane % RB), cb0 = 4 * (at.lane / RB);
      const int rowb = 32 * H * I + (at.w & 1) * 16 * H + rb;
      const int colb = 32 * H * J + (at.w >> 1) * 16 * H + cb0;
#pragma unroll
      for (int q = 0; q < RB / CB; ++q) {
        t4 e[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) e[i] = *(const t4*)(block + (rb + i) * kPitch + cb0 + 4 * CB * q);
#pragma unroll
        for (int j = 0; j < 4; ++j)
          *(t4*)(plane + plane_at(colb + 4 * CB * q + j, rowb, ld)) =
              t4{e[0][j], e[1][j], e[2][j], e[3][j]};
      }
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
    };
    mirror(hin);
#pragma unroll
    for (int m = 0; m < H; ++m)
#pragma unroll
      for (int n = 0; n < H; ++n)
        *(uint2*)(block + (16 * m + (at.lane & 15)) * kPitch + 16 * n + 4 * (at.lane >> 4)) =
            uint2{__float_as_uint(hh[m][n][0]), __float_as_uint(hh[m][n][1])};
    mirror(lon);
  } else {
    // inside a diagonal tile the upper half is written to both places (the
    // hi.lo and lo.hi terms of (r, c) and (c, r) accumulate in different
    // orders), so X_next is exactly symmetric
#pragma unroll
    for (int m = 0; m < H; ++m) {
      const int row = at.row0 + 16 * m;
#pragma unroll
      for (int n = 0; n < H; ++n) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int col = at.col0 + 16 * n + r;
          if (row > col) continue;
          const bool diag = (row == col);
          const double y = (double)hh[m][n][r] + (1.0 / kScale) * (double)xx[m][n][r];
          const size_t idx = row + (size_t)col * ld, tdx = col + (size_t)row * ld;
          const double x = X[tdx];
          const double z = fma(cb, x, ca * y);
          const double d = x - y;
          const double wc =
              (row < core_lim ? 1.0 : 0.0) + ((!diag && col < core_lim) ? 1.0 : 0.0);
          sums[0] += (diag ? 1.0 : 2.0) * z * z;
          sums[2] += wc * d * d;
          sums[1] += diag ? z : 0.0;
          sums[3] += diag ? y : 0.0;
          const T h = (T)z;
          const T l = (T)((z - (double)h) * kScale);
          Xn[idx] = z;
          Xn[tdx] = z;
          hin[plane_at(row, col, ld)] = h;
          hin[plane_at(col, row, ld)] = h;
          lon[plane_at(row, col, ld)] = l;
          lon[plane_at(col, row, ld)] = l;
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  }
}

template <typename T>
__global__ __launch_bounds__(NT, 2) void sp2_f16split_kernel(F16Args g) {
  __shared__ __attribute__((aligned(1024))) int8_t ring[kRing];
  const volatile Sp2State* stv = g.st;
  if (!stv->planned) return;
  double sums[4] = {0.0, 0.0, 0.0, 0.0};
  SplitTile tl;
  if (tl.find(g.nt, g.full)) {
    if (tl.quarter)
      sp2_split_tile<T, 2>(g, stv, tl.I, tl.J, ring, sums);
    else
      sp2_split_tile<T, 4>(g, stv, tl.I, tl.J, ring, sums);
  }
  block_store4<NT>(sums, g.part + 4 * (size_t)blockIdx.x);
}

// X (current buffer) from its lower triangle: the upper 64 x 64 blocks are
// the transposes of their mirror blocks, through LDS.
__global__ void sp2_mirror_kernel(double* x0, double* x1, const Sp2State* __restrict__ s, int ld) {
  __shared__ double t[64][65];
  double* x = s->cur ? x1 : x0;
  const int br = blockIdx.x * 64, bc = blockIdx.y * 64;
  if (br <= bc) return;  // blocks below the diagonal, whose transposes are written
  const int tx = threadIdx.x & 63, ty = threadIdx.x >> 6;
  for (int j = ty; j < 64; j += 4) t[j][tx] = x[(br + tx) + (size_t)(bc + j) * ld];
  __syncthreads();
  for (int j = ty; j < 64; j += 4) x[(bc + tx) + (size_t)(br + j) * ld] = t[tx][j];
}

struct SplitGemmArgs {
  const void* ahi;
  const void* alo;
  const void* bhi;
  const void* blo;
  const double* Cin;  // beta term, or null
  const double* E;    // <C, E> partial, or null
  double* C;
  double* part;       // per tile [Tr C, ||C||_F^2, <C, E>, 0], or null
  double alpha, beta, gamma;
  int ld, n, nt, full;
};

// C = alpha A B + beta Cin + gamma I (gamma on the n x n diagonal) for
// symmetric, commuting A and B from their hi/lo planes: one workgroup per
// upper-triangle tile, the tile mirrored; inside a diagonal tile
// the upper half is mirrored onto the lower one, so C is exactly symmetric.
// FUSE bit 0: with Cin, bit 1: with <C, E>.
template <typename T, int FUSE, int H>
__device__ __forceinline__ void split_gemm_tile(const SplitGemmArgs& g, int I, int J, int8_t* ring,
                                                double (&sums)[4]) {
  constexpr double kScale = Split<T>::kScale;
  const int ld = g.ld;
  f4 hh[H][H], xx[H][H];
  split_tile<T, H>((const T*)g.ahi, (const T*)g.alo, (const T*)g.bhi, (const T*)g.blo, ld, I, J,
                   ring, hh, xx);
  const SplitAt<H> at(I, J);
  if (I != J) {
    // the (col, row) position is 32 contiguous bytes per lane
#pragma unroll
    for (int m = 0; m < H; ++m) {
      const int row = at.row0 + 16 * m;
#pragma unroll
      for (int n = 0; n < H; ++n) {
        const int col = at.col0 + 16 * n;
        const size_t tdx = col + (size_t)row * ld;
        double v[4];
#pragma unroll
        for (int r = 0; r < 4; ++r)
          v[r] = g.alpha * ((double)hh[m][n][r] + (1.0 / kScale) * (double)xx[m][n][r]);
        if (FUSE & 1) {
          const double2* cp = (const double2*)(g.Cin + tdx);
          const double2 a = cp[0], b = cp[1];
          v[0] += g.beta * a.x;
          v[1] += g.beta * a.y;
          v[2] += g.beta * b.x;
          v[3] += g.beta * b.y;
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) sums[1] += 2.0 * v[r] * v[r];
        if (FUSE & 2) {
          const double2* ep = (const double2*)(g.E + tdx);
          const double2 a = ep[0], b = ep[1];
          sums[2] += 2.0 * (v[0] * a.x + v[1] * a.y + v[2] * b.x + v[3] * b.y);
        }
        double2* tp = (double2*)(g.C + tdx);
        tp[0] = double2{v[0], v[1]};
        tp[1] = double2{v[2], v[3]};
#pragma unroll
        for (int r = 0; r < 4; ++r) g.C[row + (size_t)(col + r) * ld] = v[r];
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  } else {
#pragma unroll
    for (int m = 0; m < H; ++m) {
      const int row = at.row0 + 16 * m;
#pragma unroll
      for (int n = 0; n < H; ++n) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int col = at.col0 + 16 * n + r;
          if (row > col) continue;  // lower half of a diagonal tile
          const bool diag = (row == col);
          const size_t idx = row + (size_t)col * ld;
          double v = g.alpha * ((double)hh[m][n][r] + (1.0 / kScale) * (double)xx[m][n][r]);
          if (FUSE & 1) v += g.beta * g.Cin[idx];
          v += (diag && row < g.n) ? g.gamma : 0.0;
          const double we = diag ? 1.0 : 2.0;
          sums[0] += diag ? v : 0.0;
          sums[1] += we * v * v;
          if (FUSE & 2) sums[2] += we * v * g.E[idx];
          g.C[idx] = v;
          g.C[col + (size_t)row * ld] = v;
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  }
}

template <typename T, int FUSE>
__global__ __launch_bounds__(NT, 2) void split_gemm_kernel(SplitGemmArgs g) {
  __shared__ __attribute__((aligned(1024))) int8_t ring[kRing];
  double sums[4] = {0.0, 0.0, 0.0, 0.0};
  SplitTile tl;
  if (tl.find(g.nt, g.full)) {
    if (tl.quarter)
      split_gemm_tile<T, FUSE, 2>(g, tl.I, tl.J, ring, sums);
    else
      split_gemm_tile<T, FUSE, 4>(g, tl.I, tl.J, ring, sums);
  }
  if (g.part) block_store4<NT>(sums, g.part + 4 * (size_t)blockIdx.x);
}

// hi/lo planes of a symmetric FP64 matrix (whole ld x ld buffer, padding stays
// zero) in the blocked layout.  One workgroup per 64 x 64 block (I, J) of the
// upper triangle: its entries are read once, as (k, r) with a thread's four
// k's in 32 contiguous bytes, and both planes get the block and, through LDS,
// its transpose.  Bound: HBM, 4 bytes read and 4 written per entry; N = 4096:
// 27.2 us (134 MB, 4.9 TB/s; 40.1 us when the whole matrix was read).
template <typename T>
__global__ __launch_bounds__(NT) void split_f16_kernel(const double* __restrict__ x,
                                                       T* __restrict__ hi, T* __restrict__ lo,
                                                       int ld) {
  typedef T t4 __attribute__((ext_vector_type(4)));
  constexpr int B = 64, kPitch = B + 4;
  __shared__ __attribute__((aligned(16))) T th[B * kPitch], tl[B * kPitch];
  int I, J;
  sym_tile(blockIdx.x, I, J);
  const int g = threadIdx.x & 15, y = threadIdx.x >> 4;
  const bool mirror = I != J;
#pragma unroll
  for (int p = 0; p < 4; ++p) {
    const int rl = 16 * p + y, r = B * I + rl, k = B * J + 4 * g;
    const double2* xp = (const double2*)(x + k + (size_t)r * ld);
    const double2 a = xp[0], b = xp[1];
    const double z[4] = {a.x, a.y, b.x, b.y};
    t4 h, l;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      h[j] = (T)z[j];
      l[j] = (T)((z[j] - (double)h[j]) * Split<T>::kScale);
    }
    const size_t at = plane_at(r, k, ld);
    *(t4*)(hi + at) = h;
    *(t4*)(lo + at) = l;
    if (mirror) {
      *(t4*)(th + rl * kPitch + 4 * g) = h;
      *(t4*)(tl + rl * kPitch + 4 * g) = l;
    }
  }
  if (!mirror) return;
  __syncthreads();
  // the 4 x 4 block of rows 4 g .. and k's 4 y .., transposed
  auto transposed = [&](const T* t, T* plane) {
    t4 e[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) e[i] = *(const t4*)(t + (4 * g + i) * kPitch + 4 * y);
#pragma unroll
    for (int j = 0; j < 4; ++j)
      *(t4*)(plane + plane_at(B * J + 4 * y + j, B * I + 4 * g, ld)) =
          t4{e[0][j], e[1][j], e[2][j], e[3][j]};
  };
  transposed(th, hi);
  transposed(tl, lo);
}

// How many of the upper triangle's 128 x 128 tiles a launch keeps whole: all
// but those of the last round over the chip's two workgroups per CU, if that
// round holds few.  Whole, a lone tile takes as long as a round (its operand
// stream has the CU to itself but nothing to hide behind); its quarters, with
// three slabs in flight, about half of that.  BF16 products with their split
// pass, last rounds whole / quartered: 1024 (36 tiles) 52 / 36 us, 1920 (120)
// 75 / 55, 2176 (153) 83 / 78, 2432 (190) 90 / 86, 2560 (210) 95 / 98; behind
// full rounds 4096 (16) 301 / 253, 4352 (83) 322 / 307, 4608 (154) 344 / 343,
// 4736 (191) 362 / 362, 5888 (57) 665 / 606.  Quarters gain up to about 200
// tiles of an only round and 160 behind full ones; the smaller number serves
// both, which leaves 4 % at 171 and 190 tiles of an only round.
constexpr int kSlots = 2 * 256, kQuarterMax = 160;
int split_full_tiles(int nt) {
  const int tiles = nt * (nt + 1) / 2, rest = tiles % kSlots;
  return rest <= kQuarterMax ? tiles - rest : tiles;
}

}  // namespace

int split_step_tiles(int ld) {
  const int nt = ld / BM, full = split_full_tiles(nt);
  return full + 4 * (nt * (nt + 1) / 2 - full);
}

int split_f16(const DMat& x, void* hi, void* lo, bool bf16) {
  const int nb = x.ld / 64;
  const dim3 grid(nb * (nb + 1) / 2);
  if (bf16)
    hipLaunchKernelGGL(split_f16_kernel<__bf16>, grid, dim3(NT), 0, stream(), x.p, (__bf16*)hi,
                       (__bf16*)lo, x.ld);
  else
    hipLaunchKernelGGL(split_f16_kernel<_Float16>, grid, dim3(NT), 0, stream(), x.p,
                       (_Float16*)hi, (_Float16*)lo, x.ld);
  PRG_HIP_CHECK(hipGetLastError());
  return OK;
}

int sp2_step_mixed(const DMat& x0, const DMat& x1, Sp2State* d_state, double* d_part,
                   int* ntiles, int prec) {
  if (prec == PRG_PREC_INT8CRT) return crt_step(x0, x1, d_state, d_part, ntiles, crt_moduli());
  if (prec != PRG_PREC_F16SPLIT && prec != PRG_PREC_BF16SPLIT) {
    set_error(ERR_ARG, "unknown precision mode");
    return ERR_ARG;
  }
  const bool bf16 = (prec == PRG_PREC_BF16SPLIT);
  const int ld = x0.ld;
  const size_t plane = 2 * (size_t)ld * ld;  // bytes of one 16-bit plane
  int st = OK;
  char* planes = (char*)workspace(bf16 ? "bf16_planes" : "f16_planes", 4 * plane, &st);
  if (st) return st;
  F16Args g;
  g.buf[0] = x0.p;
  g.buf[1] = x1.p;
  g.hi[0] = planes;
  g.lo[0] = planes + plane;
  g.hi[1] = planes + 2 * plane;
  g.lo[1] = planes + 3 * plane;
  g.ld = ld;
  g.nt = ld / BM;
  g.st = d_state;
  g.part = d_part;
  g.full = split_full_tiles(g.nt);
  const int nb = split_step_tiles(ld);
  if (ntiles) *ntiles = nb;
  if (bf16)
    hipLaunchKernelGGL(sp2_f16split_kernel<__bf16>, dim3(nb), dim3(NT), 0, stream(), g);
  else
    hipLaunchKernelGGL(sp2_f16split_kernel<_Float16>, dim3(nb), dim3(NT), 0, stream(), g);
  PRG_HIP_CHECK(hipGetLastError());
  return OK;
}

int sp2_mirror(const DMat& x0, const DMat& x1, const Sp2State* d_state) {
  const int nb = x0.ld / 64;
  hipLaunchKernelGGL(sp2_mirror_kernel, dim3(nb, nb), dim3(NT), 0, stream(), x0.p, x1.p, d_state,
                     x0.ld);
  PRG_HIP_CHECK(hipGetLastError());
  return OK;
}

int sp2_mixed_prepare(const DMat& x0, int prec) {
  if (prec == PRG_PREC_INT8CRT) return crt_prepare(x0, crt_moduli());
  if (prec != PRG_PREC_F16SPLIT && prec != PRG_PREC_BF16SPLIT) return OK;
  const bool bf16 = (prec == PRG_PREC_BF16SPLIT);
  const int ld = x0.ld;
  const size_t plane = 2 * (size_t)ld * ld;
  int st = OK;
  char* planes = (char*)workspace(bf16 ? "bf16_planes" : "f16_planes", 4 * plane, &st);
  if (st) return st;
  return split_f16(x0, planes, planes + plane, bf16);
}

// Operands that a caller promises not to change while held (the matrix and the
// current iterate of a Newton-Schulz or CG solve): their planes are formed
// once and reused by every split product that names them until the hold ends.
namespace {
struct SplitHeld {
  const double* key = nullptr;
  int depth = 0;
  bool valid = false;
  int ld = 0;
};
SplitHeld g_split_held[2];
// (the second one's planes: as in the int8 products)
const char* const kSplitHeldPlanes[2] = {"splitg_planes_held", "splitg_planes_a"};

int split_held_slot(const double* p) {
  for (int i = 0; i < 2; ++i)
    if (g_split_held[i].depth > 0 && g_split_held[i].key == p) return i;
  return -1;
}
}  // namespace

void split_hold_operand(const double* p) {
  int i = split_held_slot(p);
  for (int j = 0; i < 0 && j < 2; ++j)
    if (g_split_held[j].depth == 0) {
      g_split_held[j].key = p;
      g_split_held[j].valid = false;
      i = j;
    }
  if (i >= 0) ++g_split_held[i].depth;
}

void split_release_operand(const double* p) {
  const int i = split_held_slot(p);
  if (i >= 0 && --g_split_held[i].depth == 0) {
    g_split_held[i].key = nullptr;
    g_split_held[i].valid = false;
  }
}

int split_gemm(const DMat& A, const DMat& B, DMat C, double alpha, double beta, const DMat* Cin,
               double gamma, double* part, int* nparts, const DMat* dotE) {
  const int ld = C.ld;
  if (A.ld != ld || B.ld != ld || (Cin && Cin->ld != ld) || (dotE && dotE->ld != ld) ||
      ld % BM != 0) {
    set_error(ERR_ARG,
              "BF16 split products: operand leading dimensions differ or are not multiples of 128");
    return ERR_ARG;
  }
  const size_t plane = 2 * (size_t)ld * ld;  // bytes of one BF16 plane
  const bool same = (A.p == B.p);
  const int ha = split_held_slot(A.p), hb = same ? -1 : split_held_slot(B.p);
  int st = OK;
  const bool both = ha < 0 && hb < 0 && !same;
  if (both) g_split_held[1].valid = false;
  const char* scratch_a = both ? "splitg_planes_a" : "splitg_planes_b";
  char* pa = (char*)workspace(ha >= 0 ? kSplitHeldPlanes[ha] : scratch_a, 2 * plane, &st);
  char* pb = same ? pa
                  : (char*)workspace(hb >= 0 ? kSplitHeldPlanes[hb] : "splitg_planes_b", 2 * plane,
                                     &st);
  if (st) return st;
  auto form = [&](const DMat& X, char* planes, int h) -> int {
    if (h >= 0 && g_split_held[h].valid && g_split_held[h].ld == ld) return OK;
    const int e = split_f16(X, planes, planes + plane, true);
    if (!e && h >= 0) {
      g_split_held[h].valid = true;
      g_split_held[h].ld = ld;
    }
    return e;
  };
  if ((st = form(A, pa, ha))) return st;
  if (!same && (st = form(B, pb, hb))) return st;
  SplitGemmArgs g;
  g.ahi = pa;
  g.alo = pa + plane;
  g.bhi = pb;
  g.blo = pb + plane;
  g.Cin = (Cin && beta != 0.0) ? Cin->p : nullptr;
  g.E = dotE ? dotE->p : nullptr;
  g.C = C.p;
  g.part = part;
  g.alpha = alpha;
  g.beta = beta;
  g.gamma = gamma;
  g.ld = ld;
  g.n = C.n;
  g.nt = ld / BM;
  g.full = split_full_tiles(g.nt);
  const int nb = split_step_tiles(ld);
  if (nparts) *nparts = nb;
  const int fuse = (g.Cin ? 1 : 0) | (g.E ? 2 : 0);
  void (*k)(SplitGemmArgs) = fuse == 0   ? split_gemm_kernel<__bf16, 0>
                             : fuse == 1 ? split_gemm_kernel<__bf16, 1>
                             : fuse == 2 ? split_gemm_kernel<__bf16, 2>
                                         : split_gemm_kernel<__bf16, 3>;
  hipLaunchKernelGGL(k, dim3(nb), dim3(NT), 0, stream(), g);
  PRG_HIP_CHECK(hipGetLastError());
  return OK;
}

}  // namespace prg
