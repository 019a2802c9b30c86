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
// Bound by memory: the matrix is streamed once.  Measured on MI355X, kernel time against the row-block and
// row-split kernels it replaces, and the time of the bare bytes at the rate of a large copy (6.1 TB/s):
//   5-point grid 1000^2    fp64  19.1 ->  14.9 us (14.4)    fp32  15.4 -> 10.4 us ( 9.2)
//   7-point grid 100^3     fp64  24.1 ->  21.0 us (18.2)    fp32  19.3 -> 13.0 us (11.7)
//   7-point grid 192^3     fp64   148 ->   142 us (130)     fp32   107 ->   97 us ( 83)
//   27-node mesh of 20^3   fp64  27.9 ->   6.9 us ( 3.6)    fp32  26.1 ->  6.3 us ( 2.4)
//   27-node mesh of 60^3   fp64   131 ->   120 us (103)     fp32   100 ->   88 us ( 68)
// Tried and not kept: staging columns and values in LDS and gathering x in the row phase (40 to 50 % slower: the
// gathers have to be issued right behind the loads), and 16-bit coordinates per chunk (fp64 slower, fp32 a few
// percent faster: not worth a second copy of the coordinates).
#include <algorithm>

#include "blas1.hpp"
#include "common.hpp"
#include "plan.hpp"

namespace lapis {

template <typename T>
struct Lanes;  // entries a lane takes per step: 16 bytes of values
template <>
struct Lanes<double> {
  static constexpr int per = 2;
  typedef double vals __attribute__((ext_vector_type(2), aligned(8)));
  typedef int cols __attribute__((ext_vector_type(2), aligned(4)));
  typedef v2d lds;
};
template <>
struct Lanes<float> {
  static constexpr int per = 4;
  typedef float vals __attribute__((ext_vector_type(4), aligned(4)));
  typedef int cols __attribute__((ext_vector_type(4), aligned(4)));
  typedef v4f lds;
};

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

template <typename T, int CAP, int WAVES, bool NT>
__global__ __launch_bounds__(64 * WAVES) void spmv_rowchunk_kernel(
    int nnz, int nchunks, const v2i *__restrict__ desc, const int *__restrict__ pos, const int *__restrict__ crd,
    const T *__restrict__ val, const T *__restrict__ x, T *__restrict__ y, int accumulate, int contiguous,
    double *__restrict__ xy_partials, int to_host, const unsigned long long *__restrict__ skip) {
  typedef Lanes<T> L;
  constexpr int PER = L::per;
  constexpr int STEPS = CAP / (64 * PER);
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
    // values and columns of the chunk
    typename L::vals v[STEPS];
    int col[STEPS][PER];
    if ((long long)e0 + CAP <= nnz) {
#pragma unroll
      for (int s = 0; s < STEPS; ++s) {
        const int k = (s * 64 + lane) * PER;
        if (k < count) {
          v[s] = ldv<NT>(reinterpret_cast<const typename L::vals *>(val + e0 + k));
          const typename L::cols w = ldv<NT>(reinterpret_cast<const typename L::cols *>(crd + e0 + k));
#pragma unroll
          for (int i = 0; i < PER; ++i) col[s][i] = w[i];
        }
      }
    } else {  // the arrays may end inside the last chunks
#pragma unroll
      for (int s = 0; s < STEPS; ++s) {
#pragma unroll
        for (int i = 0; i < PER; ++i) {
          const int k = (s * 64 + lane) * PER + i;
          v[s][i] = k < count ? val[e0 + k] : T(0);
          col[s][i] = k < count ? crd[e0 + k] : 0;
        }
      }
    }
#pragma unroll
    for (int s = 0; s < STEPS; ++s) {
      const int k = (s * 64 + lane) * PER;
      if (k < count) {
        typename L::lds pr;
#pragma unroll
        for (int i = 0; i < PER; ++i) pr[i] = v[s][i] * x[col[s][i]];
        *reinterpret_cast<typename L::lds *>(buf + k) = pr;
      }
    }
    wave_lds_sync();
    for (int g = r0;;) {
      T acc = sum_strided(buf, ps - e0 + sub, pe - e0, 1 << shift);
      for (int o = 1; o < (1 << shift); o <<= 1) acc = acc + __shfl_xor(acc, o, 64);
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
  // One lane adds up a row where a chunk has 64 or more, so a chunk takes as long as its longest row: uneven rows
  // are left to the row-split kernel unless none is long (2425 power-law rows of up to 256: 16 us here, 5 there).
  if (s.nnz == 0 || s.max_row_len > kRowchunkLongestRow) return LAPIS_HIP_OK;
  if (s.max_row_len > 64 && s.max_row_len > 3.0 * s.mean_row_len) return LAPIS_HIP_OK;
  // 256 entries per wavefront, 4 wavefronts per workgroup: the most loads in flight for the LDS they take (512:
  // +2 to +7 %, 1024: +20 to +35 % in fp64).  Long rows in fp32 have half the bytes per entry and fewer rows per
  // byte: 1024 gains 3 % on the large meshes and costs nothing on the small ones.  A chunk's rows fill it less
  // well the longer they are, so the longest stays within a quarter of it.
  int cap = value_bytes == 4 && s.mean_row_len >= 32.0 ? 1024 : 256;
  while (cap < 4 * s.max_row_len) cap *= 2;
  p->rowchunk_weight = (int)((int64_t)cap * (s.max_row_len + 1) / s.max_row_len - s.max_row_len);
  p->rowchunk_n = (int)((s.nnz + s.nrows) / p->rowchunk_weight + 1);
  LAPIS_HIP_TRY(hipMalloc(&p->rowchunk_desc, sizeof(v2i) * ((size_t)p->rowchunk_n + 1)));
  p->rowchunk_cap = cap;
  // Every XCD a contiguous run of chunks while the matrix stays within half of the 256 MB last-level cache: the
  // parts of x that neighbours share are read into one L2 instead of eight (-4 to -12 %).  A larger matrix comes
  // from HBM, which eight distant streams suit less than one moving window (+6 to +10 %): round-robin there.
  p->rowchunk_contiguous = s.nnz * (value_bytes + 4) <= (128ll << 20);
  hipLaunchKernelGGL(rowchunk_desc_kernel, dim3((unsigned)ceil_div(s.nrows + 1, 256)), dim3(256), 0, st, (int)s.nrows,
                     p->rowchunk_weight, p->rowchunk_n, p->pos, static_cast<v2i *>(p->rowchunk_desc));
  LAPIS_LAUNCH_CHECK();
  return LAPIS_HIP_OK;
}

// Workgroups of a product that also sums x . y.  Up to 16 384 groups of chunks, 2048 workgroups take several in turn
// (32 to 36 us at 120^3 either way); beyond, workgroups that stay drift apart and the front that moves through memory
// frays (192^3: 161 us against 138 with a workgroup per group), and the caller adds up more partial sums instead.
int rowchunk_xy_blocks(const lapis_hip_csr_plan *p) {
  const int64_t groups = ceil_div(p->rowchunk_n, 4);
  return (int)(groups <= 16384 ? std::min<int64_t>(groups, 2048) : groups);
}

template <typename T, int CAP>
int launch_rowchunk_cap(const lapis_hip_csr_plan *p, const int *crd, const T *val, const T *x, T *y, hipStream_t st,
                        int accumulate, double *xy_partials, bool to_host, int *count,
                        const unsigned long long *skip) {
  constexpr int kWaves = 4;
  int64_t blocks = ceil_div(p->rowchunk_n, kWaves);
  if (count) *count = (int)(blocks = rowchunk_xy_blocks(p));
  auto kernel = p->nontemporal ? spmv_rowchunk_kernel<T, CAP, kWaves, true> : spmv_rowchunk_kernel<T, CAP, kWaves, false>;
  launch_timed(kernel, dim3((unsigned)blocks), dim3(64 * kWaves), st, (int)p->stats.nnz, p->rowchunk_n,
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
