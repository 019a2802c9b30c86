// CSR SpMV over chunks of whole rows, for matrices without very long rows.
//
// The row-split kernel (spmv.hip) cuts the non-zeros into equal chunks wherever the cuts fall and completes the
// rows they hit in a second launch.  Where no row is long the cuts can be moved to row boundaries: every row
// lies in one chunk, there is one launch, and in CG the p.Ap of a chunk is complete when its wavefront is.
//
// Chunk c holds the rows r with floor((pos[r] + r) / weight) == c, so it is bounded in rows as well as in
// entries; `weight` is chosen from the longest row so that no chunk has more than CAP entries.  desc[c] =
// (first row, first entry) of chunk c: with it a wavefront asks for its positions, values, coordinates and
// its part of y at once, then gathers x, then adds up -- three dependent latencies.
//
// Bound by memory: the matrix is streamed once.  Measured on MI355X, us a product among others of the same matrix and
// vectors, on one box: the row-block and row-split kernels it replaces, this one, and the time of the bare bytes at the rate
// of a large copy (6.1 TB/s):
//   5-point grid 1000^2    fp64  21.7  14.1 (14.4)
//   7-point grid 100^3     fp64  25.7  17.3 (18.2)    fp32  21.8  13.8 (11.7)
//   7-point grid 180^3     fp64   126   117 (107)     fp32    92    77 ( 68)
//   27-node mesh of 35^3   fp64  32.1  19.7 (20.3)    fp32  27.9  14.8 (13.6)
//   27-node mesh of 60^3   fp64   130   107 (103)     fp32    99    76 ( 68)
// (below the bare bytes where the last-level cache holds the matrix from one product to the next; with another matrix every
// time 100^3 takes 20.8 in fp64, and the mesh of 60^3, which no cache holds, 106.9).  With four neighbouring entries in a
// lane instead of one, and guarded loads, the lanes of a gather are four entries apart and touch that many more lines:
// 18.6 at 100^3 and 23.7 on the mesh of 35^3 in fp64.
// Tried and not kept: staging columns and values in LDS and gathering x in the row phase (40 to 50 % slower: the
// gathers have to be issued right behind the loads), and 16-bit coordinates per chunk (fp64 slower, fp32 a few
// percent faster: not worth a second copy of the coordinates).
#include <algorithm>

#include "blas1.hpp"
#include "common.hpp"
#include "plan.hpp"

namespace lapis {

// buf[lo..hi) with stride `step`, in ascending order, four reads in flight
template <typename T>
__device__ __forceinline__ T sum_strided(const T *buf, int lo, int hi, int step) {
  T acc = T(0);
  for (int j = lo; j < hi; j += 4 * step) {
    T v[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) v[u] = buf[min(j + u * step, hi - 1)];
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (j + u * step < hi) acc = acc + v[u];
  }
  return acc;
}

constexpr int kLongPart = 32;  // entries per lane from which the whole wavefront takes a row

template <typename T, int CAP, int WAVES, bool NT>
__global__ __launch_bounds__(64 * WAVES) void spmv_rowchunk_kernel(
    int nchunks, const v2i *__restrict__ desc, const int *__restrict__ pos, const int *__restrict__ crd,
    const T *__restrict__ val, const T *__restrict__ x, T *__restrict__ y, int accumulate, int contiguous,
    double *__restrict__ xy_partials, int to_host, const unsigned long long *__restrict__ skip) {
  constexpr int STEPS = CAP / 64;
  __shared__ __align__(16) T lds[WAVES * CAP];
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  T *buf = lds + wave * CAP;
  double xy = 0.0;
  if (skip && *skip != 0) return;  // nobody reads this product any more
  // groups of WAVES chunks: of the whole matrix in turn, or the XCD's own contiguous part of them in turn
  const int groups = (nchunks + WAVES - 1) / WAVES;
  int g0 = blockIdx.x, gend = groups, gstep = gridDim.x;
  if (contiguous) {
    const int xcd = blockIdx.x % kXcds, q = groups / kXcds, rest = groups % kXcds;
    g0 = xcd * q + min(xcd, rest) + (int)(blockIdx.x / kXcds);
    gend = (xcd + 1) * q + min(xcd + 1, rest);
    gstep = ((int)gridDim.x - xcd + kXcds - 1) / kXcds;
  }
  for (int grp = g0; grp < gend; grp += gstep) {
    const int c = __builtin_amdgcn_readfirstlane(grp * WAVES + wave);
    if (c >= nchunks) break;
    const v2i d0 = desc[c], d1 = desc[c + 1];
    const int r0 = d0.x, r1 = d1.x, e0 = d0.y, count = d1.y - d0.y;
    if (r0 >= r1) continue;
    const int nr = r1 - r0;
    // lanes per row: few rows per chunk are long ones, and several lanes add up each of them
    int shift = 0;
    while ((nr << (shift + 1)) <= 64) ++shift;
    const int sub = lane & ((1 << shift) - 1);
    int r = r0 + (lane >> shift);
    int ps = 0, pe = 0;
    T yr = T(0), xr = T(0);
    if (r < r1) {
      ps = ldv<NT>(pos + r);
      pe = ldv<NT>(pos + r + 1);
      if (accumulate) yr = y[r];
      if (xy_partials) xr = x[r];
    }
    // Values and columns of the chunk, entry by entry: neighbouring lanes take neighbouring entries, whose x mostly share
    // lines, and slots past the end repeat the last entry, so that no load waits behind a condition.  (A chunk of empty
    // rows reads an entry of its neighbour's.)
    const int eb = count > 0 ? e0 : max(e0 - 1, 0), kmax = max(count - 1, 0);
    T v[STEPS];
    int col[STEPS];
#pragma unroll
    for (int s = 0; s < STEPS; ++s) {
      const int k = min(s * 64 + lane, kmax);
      v[s] = ldv<NT>(val + eb + k);
      col[s] = ldv<NT>(crd + eb + k);
    }
#pragma unroll
    for (int s = 0; s < STEPS; ++s) buf[s * 64 + lane] = v[s] * x[col[s]];
    wave_lds_sync();
    for (int g = r0;;) {
      const int lo = ps - e0, hi = pe - e0;
      unsigned long long longs = __ballot((hi - lo) >> shift > kLongPart);
      T acc = sum_strided(buf, lo + sub, (hi - lo) >> shift > kLongPart ? lo : hi, 1 << shift);
      for (int o = 1; o < (1 << shift); o <<= 1) acc = acc + __shfl_xor(acc, o, 64);
      while (longs) {  // rows much longer than their lanes' share of the wavefront: all of it adds them up, row by row
        const int src = __builtin_ctzll(longs);
        longs &= ~(((1ull << (1 << shift)) - 1) << src);
        const int lhi = __shfl(hi, src, 64);
        T part = T(0);
        for (int j = __shfl(lo, src, 64) + lane; j < lhi; j += 64) part = part + buf[j];
        part = group_sum<64>(part);
        if (lane >> shift == src >> shift) acc = part;
      }
      if (r < r1 && sub == 0) {
        y[r] = accumulate ? acc + yr : acc;
        xy = xy + (double)xr * (double)acc;
      }
      g += 64 >> shift;
      if (g >= r1) break;
      r = g + (lane >> shift);
      ps = pe = e0;
      if (r < r1) {
        ps = ldv<NT>(pos + r);
        pe = ldv<NT>(pos + r + 1);
        if (accumulate) yr = y[r];
        if (xy_partials) xr = x[r];
      }
    }
    wave_lds_sync();  // the next chunk goes into the same LDS
  }
  if (xy_partials) {
    __shared__ double wave_xy[WAVES];
    xy = group_sum<64>(xy);
    if (lane == 0) wave_xy[wave] = xy;
    __syncthreads();
    if (threadIdx.x == 0) {
      double s = wave_xy[0];
      for (int w = 1; w < WAVES; ++w) s = s + wave_xy[w];
      if (to_host)
        tell_host(xy_partials + blockIdx.x, s);
      else
        xy_partials[blockIdx.x] = s;
    }
  }
}

// ---- plan-time kernels ---------------------------------------------------------------------------

// desc[c] = (first row with floor((pos[r] + r) / weight) >= c, its position), rows past the end counted as empty
__global__ __launch_bounds__(256) void rowchunk_desc_kernel(int nrows, int weight, int nchunks, const int *__restrict__ pos,
                                                            v2i *__restrict__ desc) {
  const long long r = (long long)blockIdx.x * 256 + threadIdx.x;
  if (r > nrows) return;
  const long long at = pos[r];
  const long long here = r == nrows ? nchunks : (at + r) / weight;
  const long long before = r == 0 ? -1 : ((long long)pos[r - 1] + r - 1) / weight;
  const v2i d = {(int)r, (int)at};
  for (long long c = before + 1; c <= here; ++c) desc[c] = d;
}

// ---- host ----------------------------------------------------------------------------------------

void free_rowchunk(lapis_hip_csr_plan *p) {
  if (p->rowchunk_desc) (void)hipFree(p->rowchunk_desc);
  p->rowchunk_desc = nullptr;
  p->rowchunk_cap = 0;
  p->rowchunk_use = false;
}

int build_rowchunk(lapis_hip_csr_plan *p, int value_bytes, hipStream_t st) {
  const lapis_hip_csr_stats &s = p->stats;
  if (s.nnz == 0 || s.max_row_len > kRowchunkLongestRow) return LAPIS_HIP_OK;
  // Short rows with a few long ones among them are left to the row-block kernel: the chunk has to hold four of the
  // longest and is mostly rows (100 000 rows of 5, every 50th 250: 9.5 us here, 8.1 there; 500 000 of 3 and 100: 25.8 and
  // 25.0).  From a mean of 16 the chunks win (2013 power-law rows of 31 on average, up to 201: 6.4 us against 11.5, the
  // whole wavefront adding up a long row; 100 000 rows of 20, every tenth 100: 17.3 against 19.8).
  if (s.max_row_len > 64 && s.max_row_len > 3.0 * s.mean_row_len && s.mean_row_len < 16.0) return LAPIS_HIP_OK;
  // Entries per wavefront, 4 wavefronts per workgroup.  A matrix the 256 MB last-level cache holds: 256 in fp64 (512:
  // +3 % in CG on 1024^2), 512 in fp32 (7-point 152^3: 39.1 us against 41.6).  From HBM more of it is asked for at once:
  // 512 (7-point 180^3: 116.9 us against 118.4 in fp64, 76.5 against 79.2 in fp32), 1024 where rows are long (27-node
  // mesh 60^3: 114 us against 125 in fp64, 77 against 80 in fp32; in cache, at 35^3, it loses: 21.2 against 19.3).
  // A chunk's rows fill it less well the longer they are, so the longest stays within a quarter of it.
  const bool cached = s.nnz * (value_bytes + 4) <= (256ll << 20);
  int cap = !cached && s.mean_row_len >= 32.0 ? 1024 : cached && value_bytes == 8 ? 256 : 512;
  while (cap < 4 * s.max_row_len) cap *= 2;
  p->rowchunk_weight = (int)((int64_t)cap * (s.max_row_len + 1) / s.max_row_len - s.max_row_len);
  p->rowchunk_n = (int)((s.nnz + s.nrows) / p->rowchunk_weight + 1);
  LAPIS_HIP_TRY(hipMalloc(&p->rowchunk_desc, sizeof(v2i) * ((size_t)p->rowchunk_n + 1)));
  p->rowchunk_cap = cap;
  // Every XCD a contiguous run of chunks while the last-level cache holds the matrix: the parts of x that neighbours share
  // are read into one L2 instead of eight (7-point 130^3 fp64, 184 MB: 33.7 us against 44.7; grid 1500^2 27.5 against
  // 32.1).  A larger matrix comes from HBM, which eight distant streams suit less than one moving window (mesh 50^3
  // fp64, 350 MB: 74.5 us against 72.8): round-robin there.
  p->rowchunk_contiguous = cached;
  hipLaunchKernelGGL(rowchunk_desc_kernel, dim3((unsigned)ceil_div(s.nrows + 1, 256)), dim3(256), 0, st, (int)s.nrows,
                     p->rowchunk_weight, p->rowchunk_n, p->pos, static_cast<v2i *>(p->rowchunk_desc));
  LAPIS_LAUNCH_CHECK();
  return LAPIS_HIP_OK;
}

// Workgroups of a product that also sums x . y.  In cache, up to 16 384 groups of chunks, 2048 workgroups take several in
// turn; beyond, and from HBM, workgroups that stay drift apart and the front that moves through memory frays (CG, 100
// iterations: 140^3 8.87 ms against 8.37 with a workgroup per group, 164^3 14.6 against 13.6), and the caller adds up
// more partial sums instead.
int rowchunk_xy_blocks(const lapis_hip_csr_plan *p) {
  const int64_t groups = ceil_div(p->rowchunk_n, 4);
  return (int)(p->rowchunk_contiguous && groups <= 16384 ? std::min<int64_t>(groups, 2048) : groups);
}

template <typename T, int CAP>
int launch_rowchunk_cap(const lapis_hip_csr_plan *p, const int *crd, const T *val, const T *x, T *y, hipStream_t st,
                        int accumulate, double *xy_partials, bool to_host, int *count,
                        const unsigned long long *skip) {
  constexpr int kWaves = 4;
  int64_t blocks = ceil_div(p->rowchunk_n, kWaves);
  if (count) *count = (int)(blocks = rowchunk_xy_blocks(p));
  auto kernel = p->nontemporal ? spmv_rowchunk_kernel<T, CAP, kWaves, true> : spmv_rowchunk_kernel<T, CAP, kWaves, false>;
  launch_timed(kernel, dim3((unsigned)blocks), dim3(64 * kWaves), st, p->rowchunk_n,
               (const v2i *)p->rowchunk_desc, p->pos, crd, val, x, y, accumulate, (int)p->rowchunk_contiguous,
               xy_partials, (int)to_host, skip);
  LAPIS_LAUNCH_CHECK();
  return LAPIS_HIP_OK;
}

template <typename T>
int launch_rowchunk_any(const lapis_hip_csr_plan *p, const int *crd, const T *val, const T *x, T *y, hipStream_t st,
                        int accumulate, double *xy_partials, bool to_host, int *count,
                        const unsigned long long *skip) {
  switch (p->rowchunk_cap) {
    case 256: return launch_rowchunk_cap<T, 256>(p, crd, val, x, y, st, accumulate, xy_partials, to_host, count, skip);
    case 512: return launch_rowchunk_cap<T, 512>(p, crd, val, x, y, st, accumulate, xy_partials, to_host, count, skip);
    default: return launch_rowchunk_cap<T, 1024>(p, crd, val, x, y, st, accumulate, xy_partials, to_host, count, skip);
  }
}

template <typename T>
int launch_rowchunk(const lapis_hip_csr_plan *p, const int *crd, const T *val, const T *x, T *y, hipStream_t st,
                    int accumulate) {
  return launch_rowchunk_any<T>(p, crd, val, x, y, st, accumulate, nullptr, false, nullptr, nullptr);
}
template int launch_rowchunk<double>(const lapis_hip_csr_plan *, const int *, const double *, const double *, double *,
                                     hipStream_t, int);
template int launch_rowchunk<float>(const lapis_hip_csr_plan *, const int *, const float *, const float *, float *,
                                    hipStream_t, int);

template <typename T>
int launch_rowchunk_xy(const lapis_hip_csr_plan *p, const int *crd, const T *val, const T *x, T *y, hipStream_t st,
                       double *xy_partials, bool to_host, int *count, const unsigned long long *skip) {
  return launch_rowchunk_any<T>(p, crd, val, x, y, st, 0, xy_partials, to_host, count, skip);
}
template int launch_rowchunk_xy<double>(const lapis_hip_csr_plan *, const int *, const double *, const double *, double *,
                                        hipStream_t, double *, bool, int *, const unsigned long long *);
template int launch_rowchunk_xy<float>(const lapis_hip_csr_plan *, const int *, const float *, const float *, float *,
                                       hipStream_t, double *, bool, int *, const unsigned long long *);

}  // namespace lapis
