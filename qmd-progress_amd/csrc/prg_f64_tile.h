// FP64 MFMA tiles whose operands go straight from memory to registers.
//
// v_mfma_f64_16x16x4_f64 occupies its SIMD for 64 cycles and takes 512 bytes
// of each operand, so a CU whose four SIMDs each work on blocks of B x B such
// products of their own K range draws 64 / B bytes per cycle (21 for B = 3),
// within what a CU gets from L2.  So nothing is staged in LDS and the main
// loop has no barrier: the four waves of a workgroup share one 16 B x 16 B
// tile and split K; each lane loads its fragments as 16-byte row pairs (rows
// 2i and 2i + 1 of a 32-row group go to two MFMA blocks), a chunk of CK k's
// ahead of their use, and the four sums meet in LDS once, in a fixed order.
//
// Small tiles of independent workgroups balance over the 256 CUs where 128 x
// 128 tiles with operands in LDS left them idle (36 tiles at N = 1024, 2080
// for 256 CUs at 8192), and two or three workgroups per CU cover each other's
// first loads and epilogues.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>
#include <type_traits>

namespace prg {
namespace f64tile {

typedef double d4 __attribute__((ext_vector_type(4)));
typedef double d2 __attribute__((ext_vector_type(2)));

// A tile of B x B MFMA blocks, K split over KS = 4 waves.
template <int B>
struct Shape {
  static constexpr int MB = B, NB = B, KS = 4;
  static constexpr int TM = 16 * B, NT = 64 * KS;
  // k's per chunk: the fragments of one chunk are in flight while the previous
  // one is multiplied
  static constexpr int CK = (B >= 3) ? 16 : 32;
  static constexpr int kLdsDoubles = KS * MB * NB * 256;
  // the padded size is a multiple of 128: only the other edges overhang it
  static constexpr bool kRagged = 128 % TM != 0;
};

// Rows (columns) of a wave's group of NBK 16-wide blocks that lane index i
// (0..15) holds: blocks come in pairs of interleaved rows (2i, 2i + 1 of 32
// consecutive rows); an odd last block holds row i of its 16.
template <int NBK>
__device__ __forceinline__ int block_row(int b, int i) {
  return (b < (NBK & ~1)) ? 32 * (b >> 1) + 2 * i + (b & 1) : 16 * b + i;
}

// One wave's product: acc += sum_p A_p[r0.., k] B_p[k, c0..] over `count`
// chunks of CK k's from kbeg, for the npair (1 or 2) operand pairs in turn.
// A is column major, A[i + k ld].  BT = false: B is symmetric and read as
// B[j + k ld]; BT = true: B is read as stored, B[k + j ld] (two consecutive
// k's per lane; the lanes' k order inside 8 is then 2 kq + s for both
// operands).  Rows and columns from ld on are clamped into the matrix; their
// results are not stored.  acc[m][n][r] is (A B)[row][col] with
// row = block_row(m, lane % 16), col = block_row(n, lane / 16 + 4 r).
//
// What the loop may hold follows from how FP64 MFMAs issue (measured, cycles
// per MFMA of 64): back to back 72.8 from one wave of a SIMD, 68.3 with two;
// one vector ALU instruction after each: 84.8; a load after every second one:
// 81.5; the same loads in one burst per 9: 75.9.  So the loop is MFMAs, then
// the substep's loads together, each with a scalar base that steps through K
// and a fixed 32-bit lane offset (64-bit lane addresses are vector adds).
template <typename S, bool BT>
struct WaveProduct {
  static constexpr int MB = S::MB, NB = S::NB, D = S::CK / 4;
  static constexpr int MP = MB / 2, MS = MB & 1, NP = NB / 2, NS = NB & 1;
  uint32_t ao[MP + MS], bo[BT ? NB : NP + NS];  // lane offsets in bytes
  d2 ra[D][MP + 1], rb[D][NP + 1];              // row pairs; [..][MP].x: the odd block
  d2 rt[BT ? D / 2 : 1][BT ? NB : 1];
  const char *pa, *pb, *pa2, *pb2;  // next substep's operands; the second pair's first
  size_t step;                      // bytes from one substep's column to the next
  int count, total;

  __device__ __forceinline__ void load_a(int t, int i) {
    if (i < MP)
      ra[t][i] = *(const d2*)(pa + ao[i]);
    else
      ra[t][MP].x = *(const double*)(pa + ao[i]);
  }
  __device__ __forceinline__ void load_b(int t, int i) {
    if constexpr (BT)
      rt[t >> 1][i] = *(const d2*)(pb + bo[i]);
    else if (i < NP)
      rb[t][i] = *(const d2*)(pb + bo[i]);
    else
      rb[t][NP].x = *(const double*)(pb + bo[i]);
  }
  // Loads substep t of the next chunk (BT: the B fragments of substeps t - 1
  // and t, with the odd one) and steps on.
  __device__ __forceinline__ void load(int t) {
#pragma unroll
    for (int i = 0; i < MP + MS; ++i) load_a(t, i);
    if constexpr (BT) {
      if (t & 1) {
#pragma unroll
        for (int i = 0; i < NB; ++i) load_b(t, i);
      }
      // columns k and k + 1 of a lane's pair, then 8 on
      pa += (t & 1) ? 7 * step : step;
      if (t & 1) pb += 8 * sizeof(double);
    } else {
#pragma unroll
      for (int i = 0; i < NP + NS; ++i) load_b(t, i);
      pa += step;
      pb += step;
    }
  }

  // Loads the first chunk.
  __device__ __forceinline__ void start(const double* A, const double* B, const double* A2,
                                        const double* B2, int npair, int ld, int r0, int c0,
                                        int kbeg, int nchunk) {
    const int lane = threadIdx.x & 63, l15 = lane & 15, kq = lane >> 4;
    count = nchunk;
    total = npair * nchunk;
    if (total <= 0) return;
    const uint32_t ko = (uint32_t)((BT ? 2 * kq : kq) * ld);
#pragma unroll
    for (int p = 0; p < MP; ++p) ao[p] = 8 * (ko + min(r0 + 32 * p + 2 * l15, ld - 2));
    if (MS) ao[MP] = 8 * (ko + min(r0 + 32 * MP + l15, ld - 1));
    const size_t k0 = (size_t)kbeg * ld * sizeof(double);
    pa = (const char*)A + k0;
    pa2 = (const char*)A2 + k0;
    if constexpr (BT) {
      const int cb = min(c0, ld - 1);  // the panel's first column
      const size_t b0 = ((size_t)cb * ld + kbeg) * sizeof(double);
#pragma unroll
      for (int n = 0; n < NB; ++n)
        bo[n] = 8 * ((uint32_t)(min(c0 + block_row<NB>(n, l15), ld - 1) - cb) * ld + 2 * kq);
      pb = (const char*)B + b0;
      pb2 = (const char*)B2 + b0;
      step = (size_t)ld * sizeof(double);
    } else {
#pragma unroll
      for (int p = 0; p < NP; ++p) bo[p] = 8 * (ko + min(c0 + 32 * p + 2 * l15, ld - 2));
      if (NS) bo[NP] = 8 * (ko + min(c0 + 32 * NP + l15, ld - 1));
      pb = (const char*)B + k0;
      pb2 = (const char*)B2 + k0;
      step = (size_t)4 * ld * sizeof(double);
    }
#pragma unroll
    for (int t = 0; t < D; ++t) load(t);
  }

  __device__ __forceinline__ void compute(int t, d4 (&acc)[MB][NB]) {
#pragma unroll
    for (int m = 0; m < MB; ++m) {
      const double a = (m < 2 * MP) ? ra[t][m >> 1][m & 1] : ra[t][MP].x;
#pragma unroll
      for (int n = 0; n < NB; ++n) {
        double b;
        if constexpr (BT)
          b = rt[t >> 1][n][t & 1];
        else
          b = (n < 2 * NP) ? rb[t][n >> 1][n & 1] : rb[t][NP].x;
        acc[m][n] = __builtin_amdgcn_mfma_f64_16x16x4f64(b, a, acc[m][n], 0, 0, 0);
      }
    }
  }

  // The loop; `last` runs before the last chunk's MFMAs (what it loads is
  // there when they are done).
  template <typename F>
  __device__ __forceinline__ void run(d4 (&acc)[MB][NB], F&& last) {
    if (total <= 0) {
      last();
      return;
    }
    for (int c = 1; c < total; ++c) {
      if (c == count) {
        pa = pa2;
        pb = pb2;
      }
#pragma unroll
      for (int t = 0; t < D; ++t) {
        compute(t, acc);
        load(t);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    last();
#pragma unroll
    for (int t = 0; t < D; ++t) compute(t, acc);
  }
};

// This wave along K.
__device__ __forceinline__ int k_wave() {
  return __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
}

// Its share [first, first + count) of the nchunk chunks of K.
template <typename S>
__device__ __forceinline__ void k_share(int nchunk, int ks, int& first, int& count) {
  first = nchunk * ks / S::KS;
  count = nchunk * (ks + 1) / S::KS - first;
}

// Columns of a wave's block come in groups: group g holds blocks 2 g and
// 2 g + 1 (their columns interleave: two consecutive ones per lane), an odd
// last block is a group of one.
template <typename S>
constexpr int kGroups = (S::NB + 1) / 2;
template <typename S, int G>
constexpr int kWidth = (2 * G + 1 < S::NB) ? 2 : 1;

// Row of block m, first column of group G, of the lane's entries of
// accumulator register r, from the wave's first row r0 and column c0.
template <typename S>
__device__ __forceinline__ int entry_row(int r0, int m) {
  return r0 + block_row<S::MB>(m, threadIdx.x & 15);
}
template <typename S, int G>
__device__ __forceinline__ int entry_col(int c0, int r) {
  return c0 + block_row<S::NB>(2 * G, ((threadIdx.x & 63) >> 4) + 4 * r);
}

// Sums the tile over its KS waves (in wave order) and calls
// f(integral_constant<G>, y) for every column group G of accumulator register
// r = ks, the register wave ks finishes: y[m][w] is the entry at row
// entry_row(m), column entry_col<G>(r) + w.
template <typename S, int G, typename F>
__device__ __forceinline__ void finish_groups(const double* src, F&& f) {
  constexpr int MB = S::MB, NB = S::NB, W = kWidth<S, G>;
  double y[MB][W];
#pragma unroll
  for (int m = 0; m < MB; ++m)
#pragma unroll
    for (int w = 0; w < W; ++w) {
      const int b = m * NB + 2 * G + w;
      double s = src[b * 256];
#pragma unroll
      for (int k = 1; k < S::KS; ++k) s += src[(k * MB * NB + b) * 256];
      y[m][w] = s;
    }
  f(std::integral_constant<int, G>{}, y);
  if constexpr (G + 1 < kGroups<S>) finish_groups<S, G + 1>(src, f);
}

template <typename S, typename F>
__device__ __forceinline__ void finish_tile(const d4 (&acc)[S::MB][S::NB], int ks, double* lds,
                                            F&& f) {
  constexpr int MB = S::MB, NB = S::NB;
  const int lane = threadIdx.x & 63;
  double* slot = lds + ks * MB * NB * 256 + lane;
#pragma unroll
  for (int m = 0; m < MB; ++m)
#pragma unroll
    for (int n = 0; n < NB; ++n)
#pragma unroll
      for (int r = 0; r < 4; ++r) slot[(m * NB + n) * 256 + r * 64] = acc[m][n][r];
  __syncthreads();
  finish_groups<S, 0>(lds + ks * 64 + lane, f);
}

// Element offset of this lane inside a group, apart from what is the same for
// the whole wave: rows of a pair (ROW2) or of an odd block, columns of a
// group of two (COL2) or of one, in a column-major matrix of leading
// dimension ld, or (MIRROR) in its transposed place.
template <bool ROW2, bool COL2, bool MIRROR>
__device__ __forceinline__ uint32_t lane_offset(int ld) {
  const uint32_t i = (ROW2 ? 2 : 1) * (threadIdx.x & 15);
  const uint32_t j = (COL2 ? 2 : 1) * ((threadIdx.x & 63) >> 4);
  return MIRROR ? j + i * (uint32_t)ld : i + j * (uint32_t)ld;
}
// First column of group G, register r, past c0 + the lane's part.
template <typename S, int G>
__device__ __forceinline__ int group_col(int r) {
  return kWidth<S, G> == 2 ? 32 * G + 8 * r : 16 * (S::NB - 1) + 4 * r;
}

// Reads (writes) the entries of group G of register r from (to) a
// column-major matrix, rows in pairs, 16 bytes per lane.  Entries of an
// overhanging tile outside the ld x ld buffer read as 0 and are not written.
template <typename S, int G, int W>
__device__ __forceinline__ void load_entries(const double* __restrict__ X, int ld, int r0, int c0,
                                             int r, double (&x)[S::MB][W]) {
  constexpr int MB = S::MB;
  const int cg = c0 + group_col<S, G>(r);
  const double* U = X + (size_t)cg * ld + r0;
  const uint32_t l2 = lane_offset<true, W == 2, false>(ld);
  const uint32_t l1 = lane_offset<false, W == 2, false>(ld);
#pragma unroll
  for (int w = 0; w < W; ++w) {
    const bool cin = !S::kRagged || entry_col<S, G>(c0, r) + w < ld;
#pragma unroll
    for (int p = 0; p < MB / 2; ++p) {
      d2 v = d2{0.0, 0.0};
      if (cin && (!S::kRagged || entry_row<S>(r0, 2 * p) < ld))
        v = *(const d2*)(U + ((size_t)w * ld + 32 * p) + l2);
      x[2 * p][w] = v.x;
      x[2 * p + 1][w] = v.y;
    }
    if (MB & 1)
      x[MB - 1][w] = (cin && (!S::kRagged || entry_row<S>(r0, MB - 1) < ld))
                         ? U[(size_t)w * ld + 16 * (MB - 1) + l1]
                         : 0.0;
  }
}

template <typename S, int G, int W>
__device__ __forceinline__ void store_entries(double* __restrict__ X, int ld, int r0, int c0,
                                              int r, const double (&z)[S::MB][W]) {
  constexpr int MB = S::MB;
  const int cg = c0 + group_col<S, G>(r);
  double* U = X + (size_t)cg * ld + r0;
  const uint32_t l2 = lane_offset<true, W == 2, false>(ld);
  const uint32_t l1 = lane_offset<false, W == 2, false>(ld);
#pragma unroll
  for (int w = 0; w < W; ++w) {
    const bool cin = !S::kRagged || entry_col<S, G>(c0, r) + w < ld;
#pragma unroll
    for (int p = 0; p < MB / 2; ++p)
      if (cin && (!S::kRagged || entry_row<S>(r0, 2 * p) < ld))
        *(d2*)(U + ((size_t)w * ld + 32 * p) + l2) = d2{z[2 * p][w], z[2 * p + 1][w]};
    if (MB & 1)
      if (cin && (!S::kRagged || entry_row<S>(r0, MB - 1) < ld))
        U[(size_t)w * ld + 16 * (MB - 1) + l1] = z[MB - 1][w];
  }
}

// The transposed copy: entry (row, col) at (col, row); the two columns of a
// group are consecutive there.
template <typename S, int G, int W>
__device__ __forceinline__ void store_mirrored(double* __restrict__ X, int ld, int r0, int c0,
                                               int r, const double (&z)[S::MB][W]) {
  constexpr int MB = S::MB;
  const bool cin = !S::kRagged || entry_col<S, G>(c0, r) < ld;
  double* U = X + (size_t)r0 * ld + (c0 + group_col<S, G>(r));
  const uint32_t l2 = lane_offset<true, W == 2, true>(ld);
  const uint32_t l1 = lane_offset<false, W == 2, true>(ld);
#pragma unroll
  for (int m = 0; m < MB; ++m) {
    if (cin && (!S::kRagged || entry_row<S>(r0, m) < ld)) {
      double* p = (m < (MB & ~1)) ? U + (size_t)(32 * (m >> 1) + (m & 1)) * ld + l2
                                  : U + (size_t)(16 * (MB - 1)) * ld + l1;
      if constexpr (W == 2)
        *(d2*)p = d2{z[m][0], z[m][1]};
      else
        *p = z[m][0];
    }
  }
}

// The entries of X that this wave's register of the tile needs, fetched ahead.
template <typename S>
struct Entries {
  double v[kGroups<S>][S::MB][2];
  template <int G = 0>
  __device__ __forceinline__ void load(const double* __restrict__ X, int ld, int r0, int c0,
                                       int r) {
    constexpr int W = kWidth<S, G>;
    double t[S::MB][W];
    load_entries<S, G, W>(X, ld, r0, c0, r, t);
#pragma unroll
    for (int m = 0; m < S::MB; ++m)
#pragma unroll
      for (int w = 0; w < W; ++w) v[G][m][w] = t[m][w];
    if constexpr (G + 1 < kGroups<S>) load<G + 1>(X, ld, r0, c0, r);
  }
};

// A diagonal tile of a sum whose (r, c) and (c, r) entries may differ in the
// last bit: the upper half, written to both places.
template <typename S, int W>
__device__ __forceinline__ void store_upper(double* __restrict__ X, int ld, int r0, int col0,
                                            const double (&z)[S::MB][W]) {
#pragma unroll
  for (int w = 0; w < W; ++w)
#pragma unroll
    for (int m = 0; m < S::MB; ++m) {
      const int row = entry_row<S>(r0, m), col = col0 + w;
      if (row <= col && (!S::kRagged || col < ld)) {
        X[row + (size_t)col * ld] = z[m][w];
        X[col + (size_t)row * ld] = z[m][w];
      }
    }
}

typedef Shape<1> S16;
typedef Shape<2> S32;
typedef Shape<3> S48;

// Tile edge for `tiles(edge)` tiles: the least of (rounds of 256 tiles) x
// edge^2 x w, w the time per MFMA relative to the 48-wide tile's: 1.1 at 32
// (32 instead of 21 operand bytes per cycle and CU), 2 at 16 (which also pays
// each workgroup's fixed cost most often).  Measured, us per SP2 step at
// edges 16 / 32 / 48: N = 300 9.1 / 10.0 / 15.8; 512 14.2 / 12.1 / 19.1;
// 700 23.6 / 19.1 / 21.3; 1024 - / 31.2 / 25.8; 1300 - / 49.4 / 51.2; 1500 - /
// 67.5 / 84.5; 2048 - / 158 / 148; 2600 - / 313 / 321; 4096 - / 1148 / 1067.
// (64-, 96- and 128-wide tiles of 2 x 2 waves: 187, 152 and 262 us at 2048,
// 1309, 1101 and 1443 us at 4096.)  The response's step launches twice the
// tiles, half of them over two products, at the edge chosen for the plain one:
// N = 700 2 x 300 tiles of 32, 32.5 us.
inline double edge_cost(int tiles, int e) {
  const double rounds = (tiles + 255) / 256;
  return rounds * e * e * (e == 48 ? 1.0 : e == 32 ? 1.1 : 2.0);
}
template <typename F>
inline int best_edge(F&& tiles) {
  int best = 48;
  for (int e : {32, 16})
    if (edge_cost(tiles(e), e) < edge_cost(tiles(best), best)) best = e;
  return best;
}

// Tiles of that edge of an ld x ld result (upper-triangle tiles of a
// symmetric one).
inline int tile_count(int ld, int edge, bool sym) {
  const int nb = (ld + edge - 1) / edge;
  return sym ? nb * (nb + 1) / 2 : nb * nb;
}
inline int tile_edge(int ld, bool sym) {
  return best_edge([&](int e) { return tile_count(ld, e, sym); });
}

// Whether a product takes less time on the staged 128-wide tiles
// (gemm_staged_kernel), two workgroups per CU: a round of 512 of them takes as
// long as 12.95 rounds of 48-wide ones (243 us against 18.7 us at K = 1000) if
// the operands are not symmetric, as 13.8 (17.6 us) if they are; a single
// round of at most 256, one per CU, 0.58 of that.
// Z^T A Z and Z A Z^T (two products each), ms, 48-wide / staged:
// ld 1920 0.58, 0.54 / 0.65, 0.61; 2048 0.73, 0.65 / 0.69, 0.65; 2560 1.35,
// 1.23 / 1.41, 1.34; 2816 1.77, 1.54 / 1.60, 1.53; 3072 2.16, 1.90 / 3.17,
// 3.02; 4096 4.62, 4.34 / 4.45, 4.05; 5632 11.5, 11.4 / 11.0, 11.1; 6144 13.7,
// 13.5 / 15.0, 15.0; 6400 16.5, 16.7 / 15.7, 15.7; 8192 34.2, 34.2 / 32.0, 32.0.
// Symmetric products: 6912 4.92 / 5.07; 7936 7.6 / 7.7; 8064 8.09 / 7.85; 8192
// 8.3 / 9.2; 9088 11.6 / 11.0; 10112 16.0 / 17.2; 11520 23.5 / 22.3; 12288 28.7
// / 29.4.  Below 2048 staged tiles (1 to 3 rounds) the two are within 1 %.
inline bool staged_is_faster(int ld, bool sym, bool b_symmetric) {
  const int tiles = tile_count(ld, 128, sym), edge = tile_edge(ld, sym);
  if (sym && (!b_symmetric || tiles < 2016)) return false;
  const double rounds = tiles <= 256 ? 0.58 : (tiles + 511) / 512;
  return (sym ? 13.8 : 12.95) * rounds * 48 * 48 < edge_cost(tile_count(ld, edge, sym), edge);
}

#define PRG_F64_SHAPE_DISPATCH(EDGE, CALL) \
  switch (EDGE) {                          \
    case 16: CALL(f64tile::S16); break;    \
    case 32: CALL(f64tile::S32); break;    \
    default: CALL(f64tile::S48); break;    \
  }

}  // namespace f64tile
}  // namespace prg
