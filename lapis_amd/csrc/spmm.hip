// CSR x dense SpMM for gfx950:  C[i,:] = C[i,:] + sum_kk val[kk] * B[crd[kk],:]
// (row-major B and C).  Replaces the i -> kk -> j nest the sparsifier emits for
// CSR x dense linalg.matmul (examples/spmm_dcsr_opdsl.py:73-110).
#include <algorithm>
#include <cstdlib>
#include <cstring>
#include <mutex>
#include <type_traits>

#include "common.hpp"
#include "plan.hpp"

namespace lapis {

// 16 bytes of a row of B or C.  Global memory takes 128-bit accesses at any address that is a multiple of
// four, so the vectors only promise the alignment of their elements: any leading dimension, any base.
template <typename T>
struct RowVec;
template <>
struct RowVec<float> {
  typedef v4f type;
  typedef float loose __attribute__((ext_vector_type(4), aligned(4)));
  static constexpr int width = 4;
};
template <>
struct RowVec<double> {
  typedef v2d type;
  typedef double loose __attribute__((ext_vector_type(2), aligned(8)));
  static constexpr int width = 2;
};

// How a launch deals B's columns and A's rows to lanes.
//   Columns: chunk c holds the columns [chunk_first(c), chunk_first(c + 1)), a multiple of the vector width
//   wide except the last, which takes what is left and is at least one vector wide.
//   Rows: a group of lpr * par lanes takes one row of A; 64 / (lpr * par) groups to a wavefront.  In a group
//   `lpr` lanes cover the chunk of a row of B, so the group takes `par` non-zeros of its row per step.
struct SpmmShape {
  int chunks;      // column chunks
  int k;
  int chunk_width, wider;  // vectors of a chunk, and how many of the first chunks have one more
  int lpr, par;
  unsigned lpr_inv, group_inv;  // 65536 / lpr + 1, 65536 / (lpr * par) + 1: a lane's number divided without a division
  int groups;      // 64 / (lpr * par)
  int row_blocks;  // workgroups per chunk
  template <int VW>
  __device__ __forceinline__ int chunk_first(int c) const {
    return c >= chunks ? k : VW * (c * chunk_width + min(c, wider));
  }
};

__device__ __forceinline__ int lane_get(int byte_of_lane, int v) { return __builtin_amdgcn_ds_bpermute(byte_of_lane, v); }
__device__ __forceinline__ float lane_get(int byte_of_lane, float v) {
  return __builtin_bit_cast(float, lane_get(byte_of_lane, __builtin_bit_cast(int, v)));
}
__device__ __forceinline__ double lane_get(int byte_of_lane, double v) {
  v2i w = __builtin_bit_cast(v2i, v);
  w.x = lane_get(byte_of_lane, w.x);
  w.y = lane_get(byte_of_lane, w.y);
  return __builtin_bit_cast(double, w);
}

// A wavefront owns `groups` consecutive rows; their entries are one contiguous stretch of crd/val, which it
// stages in its own part of LDS with coalesced loads, all in flight together (window by window when the rows
// hold more than kStaged entries), the column already turned into the byte offset of its row of B.  A lane of a
// group holds one 128-bit vector (VW elements; VW = 1 for k smaller than a vector) of its group's row of
// C and reads every par-th entry of the row from LDS.  A batch of up to DEPTH steps loads its rows of B first,
// without any condition (past the row end a lane repeats the last non-zero's row), then adds them in order:
// DEPTH gathered rows in flight per lane.  The `par` partial rows of a group are added with shuffles at the end.
// A lane whose vector would pass the end of its chunk takes the chunk's last VW columns instead: it
// computes (and stores) the same numbers as its neighbour, so no access needs a guard for a ragged k.
//
// What bounds short rows is the chain of dependent loads of a wavefront (positions, entries, rows of B, row of
// C), not bandwidth: staging makes it one trip per wavefront instead of one per LPR entries, and the row of C
// is asked for first.  Measured (us; entries handed round by bpermute, LPR or 64 per trip -> staged):
//   7-point 97^3, fp64   k = 3: 342 -> 34   k = 10: 393 -> 66   k = 64: 387 -> 355
//   27-point x 3, 30^3   k = 3 fp64: 47 -> 26   k = 10 fp32: 83 -> 30   k = 64 fp32: 77 -> 66
//   random, 32 per row, 15 000 rows, k = 10 fp32: 9.9 -> 7.7; 1 M rows, k = 64 fp32 (rows of B from HBM): 1216 -> 1207
// Each XCD takes a contiguous part of the rows, so that neighbouring rows find each other's rows of B in its L2.  Dealt
// round-robin instead, us, 7-point grids in fp64, k = 64: 70^3 130 -> 153, 95^3 334 -> 325, 97^3 358 -> 352, 100^3
// 393 -> 501, 115^3 595 -> 763; fp32, k = 64, 100^3: 181 -> 225; 27-point x 3, 45^3, fp64, k = 64: 423 -> 403, k = 100:
// 764 -> 807.  (A rule that dealt round-robin where 1024 non-zeros span more than 8 MB of B rested on 97^3 alone.)
// WIDE: B is 4 GB or more and the offsets take 64 bits.
// Entries per wavefront and window: 384, 18 KB per workgroup in fp64, and registers for seven wavefronts per SIMD
// (against 512 entries and 76 registers, six wavefronts: 7-point 97^3 fp64, k = 10: 75 us -> 68, k = 33: 228 -> 207;
// 27-point x 3, 30^3, k = 10: 45 -> 38; scattered columns in an L2-sized B, 100 000 rows of 60, k = 33 fp64, pay 2 %:
// 226 -> 232; registers for eight spill: 88 at the first).
constexpr int kStaged = 384;
template <typename T, int VW, int DEPTH, bool WIDE>
__device__ __forceinline__ void spmm_rows_body(int nrows, const SpmmShape &sh, const int *__restrict__ pos,
                                               const int *__restrict__ crd, const T *__restrict__ val,
                                               const T *__restrict__ B, long long ldb, T *__restrict__ C,
                                               long long ldc) {
  typedef typename std::conditional<VW == 1, T, typename RowVec<T>::loose>::type V;
  __shared__ T s_val[4][kStaged];
  __shared__ unsigned s_off[4][kStaged];
  const unsigned nblocks = (unsigned)sh.row_blocks * (unsigned)sh.chunks, id = linear_block();
  if (id >= nblocks) return;
  unsigned block = xcd_contiguous_block(id, nblocks);
  int cfirst = 0, cend = sh.k;
  if (sh.chunks > 1) {
    const int chunk = (int)(block / (unsigned)sh.row_blocks);
    block = block % (unsigned)sh.row_blocks;
    cfirst = sh.chunk_first<VW>(chunk);
    cend = sh.chunk_first<VW>(chunk + 1);
  }
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  T *wval = s_val[wave];
  unsigned *woff = s_off[wave];
  const int gs = sh.lpr * sh.par;
  const int group = (lane * sh.group_inv) >> 16, sub = lane - group * gs;
  const int e = (sub * sh.lpr_inv) >> 16, l = sub - e * sh.lpr;
  const long long row0 = ((long long)block * 4 + wave) * sh.groups;
  if (row0 >= nrows) return;
  const int rows_here = (int)min((long long)sh.groups, nrows - row0);
  const bool mine = group < rows_here;  // lanes past the last group of a wavefront have no row
  const int ps = pos[row0 + min(group, rows_here)], pe = pos[row0 + min(group + 1, rows_here)];
  // the row of C is asked for before anything that depends on the positions
  const int col = min(cfirst + l * VW, cend - VW);
  const bool writes = mine && e == 0 && cfirst + l * VW < cend;
  T *cp = C + (row0 + group) * ldc + col;
  V cin = {};
  if (writes) cin = load_stream(reinterpret_cast<const V *>(cp));
  const int first = __shfl(ps, 0, 64), end = __shfl(pe, 63, 64);
  const unsigned col_bytes = (unsigned)(col * (int)sizeof(T));
  T acc[VW];
#pragma unroll
  for (int i = 0; i < VW; ++i) acc[i] = T(0);
  for (int w0 = first; w0 < end;) {
    const int count = min(kStaged, end - w0);
#pragma unroll
    for (int i = 0; i < kStaged / 64; ++i) {
      const int j = i * 64 + lane;
      if (j < count) {
        const unsigned c = (unsigned)load_stream(crd + w0 + j);
        woff[j] = WIDE ? c : c * (unsigned)(ldb * sizeof(T));
        wval[j] = load_stream(val + w0 + j);
      }
    }
    wave_lds_sync();
    int t = max(ps, w0) - w0;
    const int hi = min(pe - w0, kStaged);
    auto batch = [&](auto unr) {
      constexpr int UNR = decltype(unr)::value;
      T a[UNR];
      V b[UNR];
#pragma unroll
      for (int u = 0; u < UNR; ++u) {
        const int at = min(t + u * sh.par + e, hi - 1);
        const unsigned o = woff[at];
        a[u] = wval[at];
        const char *bp = reinterpret_cast<const char *>(B);
        if (WIDE)
          b[u] = *reinterpret_cast<const V *>(bp + ((unsigned long long)o * (unsigned long long)ldb * sizeof(T) + col_bytes));
        else
          b[u] = *reinterpret_cast<const V *>(bp + (o + col_bytes));
      }
#pragma unroll
      for (int u = 0; u < UNR; ++u) {
        if (t + u * sh.par + e < hi) {
          if constexpr (VW == 1) {
            acc[0] = acc[0] + a[u] * b[u];
          } else {
#pragma unroll
            for (int i = 0; i < VW; ++i) acc[i] = acc[i] + a[u] * b[u][i];
          }
        }
      }
      t += UNR * sh.par;
    };
    if (DEPTH >= 4)
      for (; hi - t > 2 * sh.par;) batch(std::integral_constant<int, 4>());
    if (DEPTH >= 2)
      for (; hi - t > sh.par;) batch(std::integral_constant<int, 2>());
    for (; hi - t > 0;) batch(std::integral_constant<int, 1>());
    if (end - w0 <= kStaged) break;
    w0 += kStaged;
    wave_lds_sync();  // the next window goes into the same LDS
  }
  for (int o = sh.par >> 1; o > 0; o >>= 1) {  // lane e of the group adds lane e + o; the total ends in e = 0
    const int src = min(lane + o * sh.lpr, 63) * 4;
#pragma unroll
    for (int i = 0; i < VW; ++i) acc[i] = acc[i] + lane_get(src, acc[i]);
  }
  if (writes) {
    if constexpr (VW == 1) {
      cin = acc[0] + cin;
    } else {
#pragma unroll
      for (int i = 0; i < VW; ++i) cin[i] = acc[i] + cin[i];
    }
    store_stream(reinterpret_cast<V *>(cp), cin);
  }
}

// Two names for the one body: profiles and lapis_hip_spmm_last_kernel tell the two regimes apart.
template <typename T, int VW, int DEPTH, bool WIDE>
__global__ __launch_bounds__(256) void spmm_wave_row_kernel(int nrows, SpmmShape shape, const int *__restrict__ pos,
                                                            const int *__restrict__ crd, const T *__restrict__ val,
                                                            const T *__restrict__ B, long long ldb, T *__restrict__ C,
                                                            long long ldc) {
  spmm_rows_body<T, VW, DEPTH, WIDE>(nrows, shape, pos, crd, val, B, ldb, C, ldc);
}
template <typename T, int VW, int DEPTH, bool WIDE>
__global__ __launch_bounds__(256, 7) void spmm_group_row_kernel(int nrows, SpmmShape shape, const int *__restrict__ pos,
                                                             const int *__restrict__ crd, const T *__restrict__ val,
                                                             const T *__restrict__ B, long long ldb, T *__restrict__ C,
                                                             long long ldc) {
  spmm_rows_body<T, VW, DEPTH, WIDE>(nrows, shape, pos, crd, val, B, ldb, C, ldc);
}

// LDS-staged row blocks, for matrices with a band around the diagonal.  A workgroup of
// 16 wavefronts owns `rb` consecutive rows of A.  It first copies the rows
// [row0 - halo, row0 + rb + halo) of B into LDS, LPR 128-bit vectors per row, fully
// coalesced; then every wavefront walks its rows as the kernel above does, and a
// non-zero whose column lies in the staged window reads its B row from LDS, any other
// from global memory.  A B row that several rows of the block use crosses the L2 -> CU
// path once instead of once per use; on this chip that path, not HBM, is what bounds a
// stencil SpMM (about 260 G lines per second for the whole chip).  k = LPR * VW exactly.
template <typename T, int LPR>
__global__ __launch_bounds__(1024) void spmm_rowblock_lds_kernel(int nrows, int ncols, int rb, int halo,
                                                                 const int *__restrict__ pos,
                                                                 const int *__restrict__ crd,
                                                                 const T *__restrict__ val, const T *__restrict__ B,
                                                                 long long ldb, T *__restrict__ C, long long ldc) {
  typedef typename RowVec<T>::type V;
  constexpr int VW = RowVec<T>::width;
  constexpr int G = 64 / LPR;
  extern __shared__ __align__(16) unsigned char spmm_lds[];
  V *tile = reinterpret_cast<V *>(spmm_lds);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const long long row0 = (long long)blockIdx.x * rb;
  const int wlo = (int)std::max<long long>(0, row0 - halo);
  const int whi = (int)std::min<long long>(ncols, row0 + rb + halo);
  const int nvec = (whi - wlo) * LPR;
  for (int v = tid; v < nvec; v += 1024) {
    const int r = v / LPR, c = v % LPR;
    tile[v] = *reinterpret_cast<const V *>(B + (long long)(wlo + r) * ldb + c * VW);
  }
  __syncthreads();
  const int g = lane / LPR;
  const int l = lane % LPR;
  const long long row_end = std::min<long long>(nrows, row0 + rb);
  for (long long row = row0 + wave; row < row_end; row += 16) {
    const int start = pos[row];
    const int end = pos[row + 1];
    V acc = {};
    for (int base = start; base < end; base += 64) {
      const int cnt = min(64, end - base);
      int c_l = 0;
      T a_l = T(0);
      if (lane < cnt) {
        c_l = load_stream(crd + base + lane);
        a_l = load_stream(val + base + lane);
      }
      for (int t0 = 0; t0 < cnt; t0 += G) {
        const int t = t0 + g;
        const int cj = __shfl(c_l, t & 63, 64);
        const T aj = __shfl(a_l, t & 63, 64);
        if (t < cnt) {
          V b;
          if (cj >= wlo && cj < whi)
            b = tile[(cj - wlo) * LPR + l];
          else
            b = *reinterpret_cast<const V *>(B + (long long)cj * ldb + l * VW);
#pragma unroll
          for (int e = 0; e < VW; ++e) acc[e] = acc[e] + aj * b[e];
        }
      }
    }
#pragma unroll
    for (int o = LPR; o < 64; o <<= 1) {
#pragma unroll
      for (int e = 0; e < VW; ++e) acc[e] = acc[e] + __shfl_xor(acc[e], o, 64);
    }
    if (g == 0) {
      V *cp = reinterpret_cast<V *>(C + row * ldc + l * VW);
      V cin = *cp;
#pragma unroll
      for (int e = 0; e < VW; ++e) cin[e] = acc[e] + cin[e];
      *cp = cin;
    }
  }
}

// Batched CSRV product of examples/bspmm.py:22-50: A is CSR over (n1, n2) and every
// non-zero carries nh values (a trailing dense batch); out(i, d, h) += A(i, c, h) * V(c, d, h).
// A row of V is K = dh*nh consecutive floats, and column j of it is multiplied by value j % nh of the
// non-zero.  A group of lpr lanes takes one row of A and one chunk of its columns, four per lane; the
// chunk's sums start from `out` and take the non-zeros in order, one rounding per product and per sum,
// as the reference's nest does.  A wavefront stages the coordinates and the values of its rows in LDS, `window`
// entries of every row at a time; up to 4 rows of V are asked for before the first is added.
// HV: nh is a multiple of 4, so a lane's four values are neighbours, one 128-bit LDS read.
// All coordinates and values of a window are asked for at once, values four at a time; the stretches of two rows lie
// kRowPad floats apart, since the lanes of all groups read the same entry of their row together, which without the
// padding is the same bank; and seven wavefronts per SIMD (six where nh is no multiple of 4) keep enough rows of V in
// flight (eight rows per lane instead of four: no faster, and twice as slow where they cost the wavefronts).
// Measured at 16384 rows of 32, dh = 32, nh = 8: 195 us with a wavefront per row that read each value and coordinate
// from global memory for every 64 columns, 45.3 us now: 537 MB of rows of V at 11.8 TB/s, of which some 190 MB come from
// beyond L2 (246 MB fetched in all, the entries of A read once per part of V among them; 58 % of L2's requests hit).
constexpr int kStagedBatched = 1024;        // values per wavefront and window
constexpr int kStagedBatchedEntries = 256;  // non-zeros per wavefront and window at most
constexpr int kRowPad = 8;  // floats between the stretches of two rows
constexpr int kCoords = kStagedBatchedEntries / 64, kVectors = kStagedBatched / 256;  // of a lane per window
constexpr int kBatchedGroups = 8;           // rows per wavefront at most: rows are long against narrow chunks
template <bool HV, bool WIDE>
__global__ __launch_bounds__(256, HV ? 7 : 6) void bspmm_csrv_kernel(int n1, SpmmShape sh, int nh, int window_log2,
                                                         const int *__restrict__ pos, const int *__restrict__ crd,
                                                         const float *__restrict__ val, const float *__restrict__ V,
                                                         float *__restrict__ out) {
  typedef RowVec<float>::loose W;
  __shared__ __align__(16) float s_val[4][kStagedBatched + kBatchedGroups * kRowPad];
  __shared__ unsigned s_off[4][kStagedBatchedEntries + kBatchedGroups];
  const unsigned nblocks = (unsigned)sh.row_blocks * (unsigned)sh.chunks, id = linear_block();
  if (id >= nblocks) return;
  unsigned block = xcd_contiguous_block(id, nblocks);
  const int chunk = (int)(block / (unsigned)sh.row_blocks);
  block = block % (unsigned)sh.row_blocks;
  const int cfirst = sh.chunk_first<4>(chunk), cend = sh.chunk_first<4>(chunk + 1);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  unsigned *woff = s_off[wave];
  float *wval = s_val[wave];
  const int group = (lane * sh.lpr_inv) >> 16, l = lane - group * sh.lpr;
  const long long row0 = ((long long)block * 4 + wave) * sh.groups;
  if (row0 >= n1) return;
  const int rows_here = (int)min((long long)sh.groups, n1 - row0);
  const int ps = pos[row0 + min(group, rows_here)], pe = pos[row0 + min(group + 1, rows_here)];
  const long long K = sh.k;
  const int col = min(cfirst + l * 4, cend - 4);
  const bool writes = group < rows_here && cfirst + l * 4 < cend;
  const int window = 1 << window_log2;
  int h[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) h[i] = (col + i) % nh;
  float *op = out + (row0 + group) * K + col;
  W acc = {};
  if (writes) acc = *reinterpret_cast<const W *>(op);
  int done = 0;                                      // entries of each row already taken
  const int mine = group < rows_here ? pe - ps : 0;  // entries of this lane's row
  // What a lane stages of every window (all lanes run every trip: the shuffles need their source lanes active):
  // coordinate slot j = entry done + j % window of row j / window, and four values at a time, vector q = floats 4 rest..
  // of the stretch of row q / per_row.
  const int slots = sh.groups << window_log2, per_row = ((nh << window_log2) + 3) >> 2;
  const unsigned per_row_inv = (1u << 22) / (unsigned)per_row + 1;  // q * inv >> 22 == q / per_row for q, per_row <= 1024
  while (__ballot(done < mine)) {
    // (every lane runs every step: the shuffles need their source lanes active)
    unsigned c[kCoords];
    W v[kVectors] = {};
    int ln = lane;
    asm volatile("" : "+v"(ln));  // the slots' numbers are worked out again in every window: kept, they cost 30 registers
#pragma unroll
    for (int i = 0; i < kCoords; ++i) {
      const int j = i * 64 + ln, from = min((j >> window_log2) * sh.lpr, 63), at = done + (j & (window - 1));
      const int first = __shfl(ps, from, 64), count = __shfl(mine, from, 64);
      c[i] = 0;
      if (j < slots && at < count) c[i] = (unsigned)load_stream(crd + first + at);
    }
#pragma unroll
    for (int i = 0; i < kVectors; ++i) {
      const unsigned q = i * 64 + ln, row = (q * per_row_inv) >> 22;
      const int rest = 4 * (int)(q - row * per_row), from = min((int)row * sh.lpr, 63);
      const int first = __shfl(ps, from, 64), count = __shfl(mine, from, 64);
      const int floats = min(count - done, window) * nh - rest;  // of the row's stretch from here on
      const float *vp = val + ((long long)first + done) * nh + rest;
      if ((int)row < sh.groups) {
        if (HV || floats >= 4) {
          if (floats > 0) v[i] = *reinterpret_cast<const W *>(vp);
        } else {
#pragma unroll
          for (int e = 0; e < 3; ++e) v[i][e] = e < floats ? vp[e] : 0.0f;
        }
      }
    }
#pragma unroll
    for (int i = 0; i < kCoords; ++i) {
      const int j = i * 64 + ln;
      if (j < slots) woff[j + (j >> window_log2)] = WIDE ? c[i] : c[i] * (unsigned)(K * 4);
    }
#pragma unroll
    for (int i = 0; i < kVectors; ++i) {
      const unsigned q = i * 64 + ln, row = (q * per_row_inv) >> 22;
      if ((int)row < sh.groups) *reinterpret_cast<v4f *>(wval + q * 4 + row * kRowPad) = v[i];
    }
    wave_lds_sync();
    const int hi = min(mine - done, window);
    const unsigned *goff = woff + (group << window_log2) + group;
    const float *gval = wval + (group << window_log2) * nh + group * kRowPad;
    int t = 0;
    auto batch = [&](auto unr) {
      constexpr int UNR = decltype(unr)::value;
      W b[UNR];
#pragma unroll
      for (int u = 0; u < UNR; ++u) {
        const unsigned o = goff[min(t + u, hi - 1)];
        if (WIDE)
          b[u] = *reinterpret_cast<const W *>(V + (long long)o * K + col);
        else
          b[u] = *reinterpret_cast<const W *>(reinterpret_cast<const char *>(V) + (o + (unsigned)(col * 4)));
      }
#pragma unroll
      for (int u = 0; u < UNR; ++u) {
        if (t + u < hi) {
          const float *au = gval + (t + u) * nh;
          v4f a;
          if (HV) {
            a = *reinterpret_cast<const v4f *>(au + h[0]);
          } else {
#pragma unroll
            for (int i = 0; i < 4; ++i) a[i] = au[h[i]];
          }
#pragma unroll
          for (int i = 0; i < 4; ++i) acc[i] = a[i] * b[u][i] + acc[i];
        }
      }
      t += UNR;
    };
    for (; hi - t > 2;) batch(std::integral_constant<int, 4>());
    for (; hi - t > 0;) batch(std::integral_constant<int, 2>());
    done += window;
    wave_lds_sync();  // the next window goes into the same LDS
  }
  if (writes) *reinterpret_cast<W *>(op) = acc;
}

// K smaller than a vector (or past int32): a lane per element of `out`.
__global__ __launch_bounds__(256) void bspmm_csrv_scalar_kernel(long long n1, long long K, int nh,
                                                                const int *__restrict__ pos,
                                                                const int *__restrict__ crd,
                                                                const float *__restrict__ val,
                                                                const float *__restrict__ V, float *__restrict__ out) {
  for (long long t = (long long)blockIdx.x * 256 + threadIdx.x; t < n1 * K; t += (long long)gridDim.x * 256) {
    const long long row = t / K, j = t % K;
    float acc = out[t];
    for (int e = pos[row]; e < pos[row + 1]; ++e) {
      const float prod = val[(long long)e * nh + j % nh] * V[(long long)crd[e] * K + j];
      acc = prod + acc;
    }
    out[t] = acc;
  }
}

template <typename T>
struct SpmmArgs {
  int64_t nrows, k;
  const int *pos, *crd;
  const T *val, *B;
  int64_t ldb;
  T *C;
  int64_t ldc;
  hipStream_t st;
};

// Cuts k columns into chunks of at most `vectors_max` vectors of VW elements (a ragged rest counts as one
// more) and deals `nrows` rows to groups of lanes per chunk, `par` non-zeros of a row at a time.
inline SpmmShape make_shape(int64_t nrows, int64_t k, int vw, int vectors_max, int par) {
  SpmmShape s;
  s.k = (int)k;
  const int vectors = (int)(k / vw);
  const int rest = k % vw != 0;
  s.chunks = (int)ceil_div(vectors + rest, vectors_max);
  while (ceil_div(vectors, s.chunks) + rest > vectors_max) ++s.chunks;
  s.lpr = (int)ceil_div(vectors, s.chunks) + rest;
  s.chunk_width = vectors / s.chunks;
  s.wider = vectors % s.chunks;
  s.par = par;
  while (s.par > 1 && s.lpr * s.par > 64) s.par /= 2;
  s.groups = 64 / (s.lpr * s.par);
  s.lpr_inv = 65536 / s.lpr + 1;
  s.group_inv = 65536 / (s.lpr * s.par) + 1;
  s.row_blocks = (int)ceil_div(nrows, 4 * s.groups);
  return s;
}

// smallest power of two >= n, at most 64
inline int pow2_up(int64_t n) {
  int p = 1;
  while (p < 64 && p < n) p *= 2;
  return p;
}

template <typename T, int VW, int DEPTH, bool WIDE>
int launch_spmm_rows(const SpmmArgs<T> &a, const SpmmShape &shape) {
  const int64_t blocks = (int64_t)shape.row_blocks * shape.chunks;
  if (blocks > 0x7fffffffLL)
    return set_error(LAPIS_HIP_ERR_INVALID_ARGUMENT, "spmm: %lld rows times %d column chunks exceed the grid limit",
                     (long long)a.nrows, shape.chunks);
  if (shape.groups == 1)
    launch_timed(spmm_wave_row_kernel<T, VW, DEPTH, WIDE>, grid_of(blocks), dim3(256), a.st, (int)a.nrows, shape, a.pos,
                 a.crd, a.val, a.B, (long long)a.ldb, a.C, (long long)a.ldc);
  else
    launch_timed(spmm_group_row_kernel<T, VW, DEPTH, WIDE>, grid_of(blocks), dim3(256), a.st, (int)a.nrows, shape, a.pos,
                 a.crd, a.val, a.B, (long long)a.ldb, a.C, (long long)a.ldc);
  LAPIS_LAUNCH_CHECK();
  return LAPIS_HIP_OK;
}

constexpr int kSpmmLdsBytes = 128 * 1024;  // staged rows of B per workgroup of the LDS kernel

// Row block and halo of the LDS kernel for rows of `row_bytes` bytes: a quarter of the
// staged rows on either side of the block, from the halo widths the plan has statistics for.
void lds_block_shape(int64_t row_bytes, int *rb, int *halo, int *halo_index) {
  const int64_t rows = kSpmmLdsBytes / row_bytes;
  const int widths[4] = {32, 64, 128, 256};
  int i = 0;
  while (i + 1 < 4 && widths[i + 1] * 4 <= rows) ++i;
  *halo = widths[i];
  *halo_index = i;
  *rb = (int)std::max<int64_t>(16, rows - 2 * widths[i]);
}

template <typename T, int LPR>
int launch_rowblock_lds(int64_t nrows, int64_t ncols, int rb, int halo, const int *pos, const int *crd, const T *val,
                        const T *B, int64_t ldb, T *C, int64_t ldc, hipStream_t st) {
  auto kernel = spmm_rowblock_lds_kernel<T, LPR>;
  static std::once_flag attribute_once;
  static hipError_t attribute_status = hipSuccess;
  std::call_once(attribute_once, [&] {
    attribute_status = hipFuncSetAttribute(reinterpret_cast<const void *>(kernel),
                                           hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
  });
  LAPIS_HIP_TRY(attribute_status);
  const size_t lds = (size_t)(rb + 2 * halo) * LPR * 16;
  const dim3 grid((unsigned)ceil_div(nrows, rb)), block(1024);
  hipEvent_t e0, e1;
  if (timing_next_events(&e0, &e1))
    hipExtLaunchKernelGGL(kernel, grid, block, lds, st, e0, e1, 0, (int)nrows, (int)ncols, rb, halo, pos, crd, val, B,
                          (long long)ldb, C, (long long)ldc);
  else
    hipLaunchKernelGGL(kernel, grid, block, lds, st, (int)nrows, (int)ncols, rb, halo, pos, crd, val, B, (long long)ldb, C,
                       (long long)ldc);
  LAPIS_LAUNCH_CHECK();
  return LAPIS_HIP_OK;
}

// name of the kernel the calling thread's last SpMM ran (lapis_hip_spmm_last_kernel)
static thread_local const char *g_last_spmm_kernel = "";

template <typename T>
int spmm_impl(const char *what, const lapis_hip_csr_plan *plan, int64_t nrows, int64_t ncols, int64_t k,
              const int32_t *pos, const int32_t *crd, const T *val, const T *B, int64_t ldb, T *C, int64_t ldc,
              lapis_hip_stream_t stream) {
  LAPIS_CHECK_INIT();
  LAPIS_REQUIRE(nrows >= 0 && ncols >= 0 && k >= 0, "%s: negative dimension", what);
  LAPIS_REQUIRE(nrows <= INT32_MAX - 64 && ncols <= INT32_MAX && k <= INT32_MAX, "%s: dimension exceeds int32", what);
  LAPIS_REQUIRE(ldb >= k && ldc >= k, "%s: leading dimension smaller than k=%lld", what, (long long)k);
  if (plan && (plan->stats.nrows != nrows || plan->stats.ncols != ncols || plan->pos != pos))
    return set_error(LAPIS_HIP_ERR_PLAN_MISMATCH, "%s: plan was built for a %lld x %lld matrix at positions %p", what,
                     (long long)plan->stats.nrows, (long long)plan->stats.ncols, (const void *)plan->pos);
  if (nrows == 0 || k == 0) return LAPIS_HIP_OK;
  LAPIS_REQUIRE(pos && C, "%s: null positions or C", what);
  LAPIS_REQUIRE(ncols == 0 || (crd && val && B), "%s: null coordinates, values or B", what);
  if (ncols == 0) return LAPIS_HIP_OK;  // a matrix without columns has no non-zeros
  hipStream_t st = as_stream(stream);
  constexpr int VW = RowVec<T>::width;
  const char *force = getenv("LAPIS_HIP_SPMM_KERNEL");  // "lds" / "wave" / "group": tuning and tests
  if (force && !strcmp(force, "lds")) {
    // Never chosen automatically: measured on MI355X it loses to the kernels below wherever it applies
    // (7-point stencil 100^3, k = 64 fp32: 0.625 ms against 0.195 ms; 27-point x 3 unknowns 60^3: 1.55 against
    // 0.60 ms).  The window a block stages is read from L2 once per block, halo included (twice B in
    // all), the block cannot start on its rows before the window is in, and the reuse it serves -- a
    // B row used by neighbouring rows -- is reuse the 32 KB vector cache of the CU already catches.
    const bool vec = aligned16(B) && aligned16(C) && (ldb % VW == 0) && (ldc % VW == 0) && (k % VW == 0);
    const int64_t lpr = vec ? k / VW : 0;
    if (lpr >= 4 && lpr <= 64 && (lpr & (lpr - 1)) == 0) {
      int rb = 0, halo = 0, hi = 0;
      lds_block_shape(k * (int64_t)sizeof(T), &rb, &halo, &hi);
      g_last_spmm_kernel = "spmm_rowblock_lds_kernel";
      switch (lpr) {
        case 4: return launch_rowblock_lds<T, 4>(nrows, ncols, rb, halo, pos, crd, val, B, ldb, C, ldc, st);
        case 8: return launch_rowblock_lds<T, 8>(nrows, ncols, rb, halo, pos, crd, val, B, ldb, C, ldc, st);
        case 16: return launch_rowblock_lds<T, 16>(nrows, ncols, rb, halo, pos, crd, val, B, ldb, C, ldc, st);
        case 32: return launch_rowblock_lds<T, 32>(nrows, ncols, rb, halo, pos, crd, val, B, ldb, C, ldc, st);
        default: return launch_rowblock_lds<T, 64>(nrows, ncols, rb, halo, pos, crd, val, B, ldb, C, ldc, st);
      }
    }
  }

  const int vw = k >= VW ? VW : 1;
  const int vectors = (int)std::min<int64_t>(64, ceil_div(k, vw));  // lanes per row of B
  const int wave_row = 64 / pow2_up(vectors);                       // par that gives a wavefront one row
  int par = wave_row;
  int depth = 4;
  if (plan && plan->stats.mean_row_len > 0.0) {
    const lapis_hip_csr_stats &ps = plan->stats;
    const double mean = ps.mean_row_len;
    const double span_bytes = ps.mean_chunk_col_span * (double)(k * sizeof(T));
    const bool local = ps.mean_chunk_col_span >= 0.0 && span_bytes <= 32.0 * 1024 * 1024;
    const bool even = mean <= 256.0 && (double)ps.max_row_len <= 4.0 * std::max(mean, 8.0);
    if (even) {
      // Several rows per wavefront, as many as leave their entries room in the staged window and a group at
      // least 8 steps; where the rows of B come from HBM (columns of 1024 non-zeros spread over more than
      // 32 MB of B) as few as the 8 steps allow (1 M rows of 32, k = 64 fp32: 1203 us against 1290 with 4 rows
      // per wavefront); and in a matrix of few rows more lanes per row until there are wavefronts for the
      // chip (15 000 rows of 32, k = 3 fp64: 7.0 us against 12.0).
      auto groups = [&](int q) { return 64 / (vectors * q); };
      par = 1;
      while (par < wave_row && 2 * par * 8.0 <= mean && (!local || groups(par) * mean > kStaged)) par *= 2;
      while (par < wave_row && 2 * par * 3.0 <= mean && ceil_div(nrows, groups(par)) < 2500) par *= 2;
    }
    // Rows of B in flight per lane: 4, but where the columns are all over a B that L2 does not hold more requests
    // only lengthen each other's way, and the registers they take are wavefronts lost: 2 (50 000 rows of 60,
    // k = 64 fp32: 55 us against 70), and 1 for rows of B of up to 16 vectors from HBM (1 M rows of 32, k = 64 fp32:
    // 1209 us against 1242; k = 64 fp64, 32 vectors, would lose 10 %).
    const bool scattered = ps.mean_chunk_col_span > 0.25 * (double)ncols;
    if (scattered && span_bytes > 8.0 * 1024 * 1024) depth = !local && vectors <= 16 && mean >= 16.0 ? 1 : 2;
  }
  if (force) par = !strcmp(force, "group") && vectors <= 32 ? 1 : wave_row;
  const SpmmShape shape = make_shape(nrows, k, vw, vectors, par);
  g_last_spmm_kernel = shape.groups == 1 ? "spmm_wave_row_kernel" : "spmm_group_row_kernel";
  const SpmmArgs<T> args{nrows, k, pos, crd, val, B, ldb, C, ldc, st};
  const bool wide = (double)ncols * (double)ldb * sizeof(T) >= 4294967296.0;
  if (vw == 1)
    return wide ? launch_spmm_rows<T, 1, 4, true>(args, shape) : launch_spmm_rows<T, 1, 4, false>(args, shape);
  if (wide) return launch_spmm_rows<T, VW, 2, true>(args, shape);
  switch (depth) {
    case 1: return launch_spmm_rows<T, VW, 1, false>(args, shape);
    case 2: return launch_spmm_rows<T, VW, 2, false>(args, shape);
    default: return launch_spmm_rows<T, VW, 4, false>(args, shape);
  }
}

}  // namespace lapis

using namespace lapis;

extern "C" const char *lapis_hip_spmm_last_kernel(void) { return g_last_spmm_kernel; }

extern "C" int lapis_hip_spmm_csr_f32_i32(int64_t nrows, int64_t ncols, int64_t k, const int32_t *pos,
                                          const int32_t *crd, const float *val, const float *B, int64_t ldb,
                                          float *C, int64_t ldc, lapis_hip_stream_t stream) {
  return spmm_impl<float>("spmm_csr_f32", nullptr, nrows, ncols, k, pos, crd, val, B, ldb, C, ldc, stream);
}
extern "C" int lapis_hip_spmm_csr_f32_i32_plan(const lapis_hip_csr_plan *plan, int64_t nrows, int64_t ncols, int64_t k,
                                               const int32_t *pos, const int32_t *crd, const float *val, const float *B,
                                               int64_t ldb, float *C, int64_t ldc, lapis_hip_stream_t stream) {
  return spmm_impl<float>("spmm_csr_f32_plan", plan, nrows, ncols, k, pos, crd, val, B, ldb, C, ldc, stream);
}
extern "C" int lapis_hip_spmm_csr_f64_i32(int64_t nrows, int64_t ncols, int64_t k, const int32_t *pos,
                                          const int32_t *crd, const double *val, const double *B, int64_t ldb,
                                          double *C, int64_t ldc, lapis_hip_stream_t stream) {
  return spmm_impl<double>("spmm_csr_f64", nullptr, nrows, ncols, k, pos, crd, val, B, ldb, C, ldc, stream);
}
extern "C" int lapis_hip_spmm_csr_f64_i32_plan(const lapis_hip_csr_plan *plan, int64_t nrows, int64_t ncols, int64_t k,
                                               const int32_t *pos, const int32_t *crd, const double *val,
                                               const double *B, int64_t ldb, double *C, int64_t ldc,
                                               lapis_hip_stream_t stream) {
  return spmm_impl<double>("spmm_csr_f64_plan", plan, nrows, ncols, k, pos, crd, val, B, ldb, C, ldc, stream);
}

extern "C" int lapis_hip_bspmm_csrv_f32_i32(int64_t n1, int64_t n2, int64_t dh, int64_t nh, const int32_t *pos,
                                            const int32_t *crd, const float *val, const float *V, float *out,
                                            lapis_hip_stream_t stream) {
  LAPIS_CHECK_INIT();
  LAPIS_REQUIRE(n1 >= 0 && n2 >= 0 && dh >= 0 && nh >= 0, "bspmm_csrv: negative dimension");
  LAPIS_REQUIRE(n1 <= INT32_MAX - 64 && n2 <= INT32_MAX && dh <= INT32_MAX && nh <= INT32_MAX,
                "bspmm_csrv: dimension exceeds int32");
  if (n1 == 0 || dh == 0 || nh == 0) return LAPIS_HIP_OK;
  LAPIS_REQUIRE(pos && out, "bspmm_csrv: null positions or output");
  LAPIS_REQUIRE(n2 == 0 || (crd && val && V), "bspmm_csrv: null coordinates, values or V");
  if (n2 == 0) return LAPIS_HIP_OK;
  hipStream_t st = as_stream(stream);
  const int64_t K = dh * nh;
  if (K < 4 || K > INT32_MAX || nh > kStagedBatched) {
    const int64_t want = ceil_div(n1 * K, 256);
    hipLaunchKernelGGL(bspmm_csrv_scalar_kernel, dim3((unsigned)std::min<int64_t>(want, 1 << 20)), dim3(256), 0, st,
                       (long long)n1, (long long)K, (int)nh, pos, crd, val, V, out);
    LAPIS_LAUNCH_CHECK();
    return LAPIS_HIP_OK;
  }
  // As many columns of a row per group as there are, 256 at most, except where an XCD's 4 MB of L2 hold more of a part
  // of V than of the whole: 512 bytes per part, 256 where the row is no multiple of 1024, so that the parts of the XCDs'
  // rows still lie on every channel of L2.  us, 16 384 rows of 32, in 64 / 32 / 16 vectors per part:
  //   K = 192, nh = 3: 45 / 42 / 33    K = 256, nh = 8: 56 / 47 / 53    K = 320, nh = 8: 69 / 65 / 59
  //   K = 384, nh = 4: 82 / 65 / 60    K = 512, nh = 8: 110 / 83 / 92   K = 1024, nh = 8: 227 / 171 / 180
  // Not for rows that are no multiple of 256 bytes (parts begin inside a line, which is fetched twice: K = 200: 58.0, in
  // two 56.7), nor where a part is beyond 16 MB (60 000 rows of 6, K = 256: 67, in two 70) or the whole within 8 MB
  // (6000 rows of 32, K = 320: 24, in five 29), nor where a window would hold fewer than 32 entries of a row.
  int vectors = (int)std::min<int64_t>(64, ceil_div(K, 4));
  const double v_bytes = (double)n2 * (double)K * sizeof(float);
  if (K % 64 == 0 && K >= 192) {
    const int part = K % 256 ? 16 : 32;
    if (v_bytes > 8388608.0 && v_bytes * part <= 16777216.0 * (double)(K / 4) && nh * (64 / part) * 32 <= kStagedBatched)
      vectors = part;
  }
  SpmmShape shape = make_shape(n1, K, 4, vectors, 1);
  // at least 4 entries of every row per window
  const int slots = (int)std::min<int64_t>(kStagedBatchedEntries, kStagedBatched / nh);
  shape.groups = std::max(1, std::min({shape.groups, kBatchedGroups, slots / 4}));
  // Two wavefronts per SIMD before a wavefront takes several rows: a few rows are bound by the trips of each wavefront
  // (514 rows of 52, K = 56: 15.0 us -> 12.8; 4587 of 62, K = 36: 18.5 -> 14.7; 9811 of 31, K = 16: 11.1 -> 10.2, and
  // 12.3 with four per SIMD).
  while (shape.groups > 1 && ceil_div(n1, shape.groups) * shape.chunks < 2048) shape.groups = (shape.groups + 1) / 2;
  shape.row_blocks = (int)ceil_div(n1, 4 * shape.groups);
  int window_log2 = 0;
  while ((2 << window_log2) * shape.groups <= slots) ++window_log2;
  const int64_t blocks = (int64_t)shape.row_blocks * shape.chunks;
  if (blocks > 0x7fffffffLL)
    return set_error(LAPIS_HIP_ERR_INVALID_ARGUMENT, "bspmm_csrv: %lld rows of %lld elements exceed the grid limit",
                     (long long)n1, (long long)K);
  const bool wide = v_bytes >= 4294967296.0;
#define LAPIS_BSPMM_LAUNCH(HV, WIDE)                                                                                  \
  hipLaunchKernelGGL((bspmm_csrv_kernel<HV, WIDE>), grid_of(blocks), dim3(256), 0, st, (int)n1, shape, (int)nh,             \
                     window_log2, pos, crd, val, V, out)
  if (nh % 4 == 0) {
    if (wide) LAPIS_BSPMM_LAUNCH(true, true); else LAPIS_BSPMM_LAUNCH(true, false);
  } else {
    if (wide) LAPIS_BSPMM_LAUNCH(false, true); else LAPIS_BSPMM_LAUNCH(false, false);
  }
#undef LAPIS_BSPMM_LAUNCH
  LAPIS_LAUNCH_CHECK();
  return LAPIS_HIP_OK;
}
