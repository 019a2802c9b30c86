// The CSR plan object behind lapis_hip_csr_plan (opaque in the C ABI).
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

#include "lapis_hip.h"

struct lapis_hip_csr_plan {
  lapis_hip_csr_stats stats;
  const int32_t *pos;
  const int32_t *crd;  // the coordinates the statistics were read from (null when the plan was made without them)
  int nchunks;
  int chunk;            // non-zeros per wavefront of the row-split kernel (512, 1024 or 2048)
  int waves_per_block;  // wavefronts per workgroup of the row-split kernel
  bool nontemporal;
  int xcd_map;          // 1: contiguous ranges of blocks per XCD (see xcd_contiguous_block)
  // row-split (NNZSPLIT) metadata
  int *chunk_row;    // device, int[nchunks+1]
  void *part_first;  // device, 8 bytes * nchunks
  void *part_last;   // device, 8 bytes * nchunks
  // chunks of whole rows (rowchunk.hip); rowchunk_cap = 0: not for this matrix
  int rowchunk_cap;          // entries per chunk at most
  int rowchunk_weight;       // rows + entries per chunk
  int rowchunk_n;            // chunks
  void *rowchunk_desc;       // device, int2[n + 1]: first row and first entry of a chunk
  bool rowchunk_contiguous;  // neighbouring chunks on one XCD
  bool rowchunk_use;         // the choice of kernel is the plan's own: ROWBLOCK and NNZSPLIT run as row chunks
  // column-blocked (COLBLOCK) copy of the matrix, built on request
  bool colblock_built;
  int colblock_value_bytes;
  int colblock_col_bits;     // low bits of an entry hold the column, the bits above the row inside its row block
  int colblock_slice_log2;   // columns per x slice = 1 << this
  unsigned *colblock_idx;    // device, uint32[nnz]
  void *colblock_val;        // device, T[nnz]
  unsigned *colblock_perm;   // device, uint32[nnz]: CSR position of the entry stored at each position of the copy
  const void *colblock_src_crd;  // the caller's buffers the copy was made from; SpMV calls must pass the same ones
  const void *colblock_src_val;
  int colblock_steps;        // steps per wavefront trip
  int colblock_epl;          // entries per lane per step (1, 2 or 4)
  int colblock_pad;          // 1: workgroups of 8 wavefronts instead of 4
  int colblock_rows;         // rows per wavefront (512 or 1024), or per workgroup in the workgroup-blocked layout
  int colblock_threads;      // threads per workgroup of the workgroup-blocked kernel (256, 512 or 1024)
  int colblock_group;        // 1: workgroup-blocked layout (tiles in column order, row sums shared by a workgroup)
  int colblock_pc_prod;      // > 0: the workgroup kernel with this many producer wavefronts (they only stream)
  int colblock_pc_threads;   // threads per workgroup of that kernel
  int *colblock_fault;       // device int: set by a wavefront of that kernel whose bounded wait ran out
  int colblock_nblocks;      // row blocks of the workgroup-blocked layout
  int colblock_nslices;      // slices of x
  int *colblock_tile_ptr;    // device, int[nblocks * (nslices + 1)]
  // workgroup-blocked layout: work units and the rows kept apart as long rows
  int colblock_nblocks_nat;  // blocks of consecutive rows; blocks from here on hold the long rows
  int colblock_nunits;       // workgroups per launch
  int *colblock_units;       // device, int[4 * nunits]: block, first entry, one past the last, 1 if the block's only unit
  int colblock_nlong;        // rows of colblock_long_threshold entries or more
  int *colblock_long_rows;   // device, int[nlong]: their row numbers, ascending
  int colblock_long_threshold;
  unsigned colblock_pace_fp; // clock ticks per entry (16.16 fixed point) of the time-triggered pacing, 0 = off
  double colblock_free_ms;   // calibration: kernel time without pacing
  double colblock_paced_ms;  // calibration: kernel time at the chosen pace

  // Chunks of whole rows replace the row-block and the row-split kernel wherever the plan itself chose one of these.
  bool runs_rowchunk() const {
    return rowchunk_use && (stats.kernel == LAPIS_HIP_SPMV_ROWBLOCK || stats.kernel == LAPIS_HIP_SPMV_NNZSPLIT);
  }
};

namespace lapis {
// What a pass over the structure finds; made by the kernels of spmv.hip, or by the host where the structure comes from
// host memory (staging.hip).
struct CsrCounts {
  int min_len;
  int max_len;
  int bad;  // bit 0: positions decrease; bit 1: coordinate out of range
  int pad;
  unsigned long long empty_rows;
  double sum_sq;
  unsigned long long span_sum;  // sum over 1024-non-zero chunks of (max column - min column)
  unsigned long long near[4];   // non-zeros with |column - row| <= 32, 64, 128, 256 (device counts only)
};
// A plan from counts made by the host, `first` and `last` being the first and the last position.  Nothing of the
// device is waited for: the plan serves calls on `stream`.
int create_counted_plan(lapis_hip_csr_plan **out, int64_t nrows, int64_t ncols, int64_t nnz, const int32_t *pos,
                        const int32_t *crd, int value_bytes, const CsrCounts &counts, int32_t first, int32_t last,
                        hipStream_t stream);

constexpr int kColblockRowBits = 10;  // the per-wavefront layout keeps up to 1024 rows per wavefront

// bits needed for values 0..n-1
inline int bits_for(int64_t n) {
  int b = 0;
  while (b < 62 && (1LL << b) < n) ++b;
  return b;
}

// Chunks of whole rows; defined in rowchunk.hip.
constexpr int kRowchunkLongestRow = 256;  // a quarter of the largest chunk
int build_rowchunk(lapis_hip_csr_plan *plan, int value_bytes, hipStream_t st);
void free_rowchunk(lapis_hip_csr_plan *plan);
// y += A x, or y = A x with accumulate = 0
template <typename T>
int launch_rowchunk(const lapis_hip_csr_plan *plan, const int *crd, const T *val, const T *x, T *y, hipStream_t st,
                    int accumulate);
// y = A x for a square A, and x . y in rowchunk_xy_blocks(plan) partial sums, one per workgroup; *count becomes their
// number.  The sums may go to pinned host memory.  The whole launch returns at once when *skip (device memory) is not 0.
int rowchunk_xy_blocks(const lapis_hip_csr_plan *plan);
template <typename T>
int launch_rowchunk_xy(const lapis_hip_csr_plan *plan, const int *crd, const T *val, const T *x, T *y, hipStream_t st,
                       double *xy_partials, bool to_host, int *count, const unsigned long long *skip);

// May `plan` serve a product of this matrix?  The error the entry point `what` returns if not: a plan of other sizes or
// positions, null entries, or a column-blocked copy (where the plan runs one) of other buffers.
int check_planned(const char *what, const lapis_hip_csr_plan *plan, int64_t nrows, int64_t ncols, const int32_t *pos,
                  const int32_t *crd, const void *val, int value_bytes);

// y = A x with the checks of the SpMV entry points, and the same with the start of init + x . y (blas1.hpp).
struct HostSum;
template <typename T>
int spmv_overwrite(lapis_hip_csr_plan *plan, int64_t nrows, int64_t ncols, const int32_t *pos, const int32_t *crd,
                   const T *val, const T *x, T *y, lapis_hip_stream_t stream);
template <typename T>
int spmv_dot_start(lapis_hip_csr_plan *plan, int64_t nrows, int64_t ncols, const int32_t *pos, const int32_t *crd,
                   const T *val, const T *x, T *y, double init, lapis_hip_stream_t stream, HostSum **out);

// Workgroup-blocked layout; defined in colgroup.hip.
template <typename T>
int build_colgroup(lapis_hip_csr_plan *plan, const int32_t *crd, const T *val, int slice_log2, hipStream_t st);
template <typename T>
int launch_colgroup(const lapis_hip_csr_plan *plan, const T *x, T *y, hipStream_t st);

// Launches the column-blocked kernel; defined in colblock.hip.
template <typename T>
int launch_colblock(const lapis_hip_csr_plan *plan, const int *pos, const int *crd, const T *val, const T *x, T *y,
                    hipStream_t st);
void free_colblock(lapis_hip_csr_plan *plan);

// Sorts `nnz` 64-bit keys (bits [0, end_bit)).  On success *keys_out holds the sorted keys and
// *perm the position each sorted key had before (both device buffers, the caller frees them).
int sort_keys_with_perm(const unsigned long long *keys_in, int64_t nnz, int begin_bit, int end_bit, unsigned long long **keys_out,
                        unsigned **perm, hipStream_t st);
// out[i] = val[perm[i]]
template <typename T>
int gather_values(const unsigned *perm, const T *val, T *out, int64_t nnz, hipStream_t st);

// y = A x without reading y; defined in spmv.hip.  A caller that passes `deferred_chunk` and gets a
// non-zero chunk length back completes the rows cut at chunk boundaries itself (rowsplit_fix.hpp);
// for a square matrix `xy_chunk` (plan->nchunks doubles) then holds, per chunk, the sum of
// x[r]*y[r] over the rows that lie wholly inside the chunk.
int spmv_overwrite_f64(lapis_hip_csr_plan *plan, int64_t nrows, int64_t ncols, const int32_t *pos,
                       const int32_t *crd, const double *val, const double *x, double *y,
                       lapis_hip_stream_t stream, int *deferred_chunk = nullptr, double *xy_chunk = nullptr);
}  // namespace lapis
