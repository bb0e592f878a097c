// kernels.hpp -- internal interfaces between the .hip translation units.
#pragma once

#include "common.hpp"

namespace tbsla_hip {

// scan.hip: prefix sum of n values (in may equal out); *d_total (device,
// nullable) receives the sum.  workspace: scan_workspace_bytes(n) bytes.
template <typename T>
int scan(const T *in, T *out, long long n, bool inclusive, long long *d_total, void *workspace,
         hipStream_t s);
size_t scan_workspace_bytes(long long n);

// spmv.hip
// d_done (device, nullable): CSR and ELL launches return at once when it
// holds a nonzero value (converged solver iterations queued in a batch).
int spmv_launch(tbsla_hip_matrix_s *m, double *d_r, const double *d_v, int vect_incr,
                bool zero_first, hipStream_t s, const int *d_done = nullptr,
                const int *seg_offs = nullptr, int nseg = 0, const int *seg_done = nullptr);
// the CSR row kernel (csr_rows.hpp) of a block: what was set on the handle,
// else csr_default of its mean row length
struct CsrKernel {
  int V, L, R, NT;
};
CsrKernel csr_default(double mean, double entries);
CsrKernel pick_csr(const tbsla_hip_matrix_s *m);

// vec.hip
int launch_fill(double *d, long long n, double v, hipStream_t s);
int launch_axpy_inplace(double *y, const double *x, long long n, hipStream_t s);  // y += x

// sort.hip: stable LSD radix sort of 32- or 64-bit keys (key_bits significant
// bits, the lowest `low` of which are left unsorted), *payload receiving each key's
// original position.  Buffers of n
// elements from device_alloc; the sort works between them and two of its own
// and leaves in *keys / *payload the pair that holds the result (it frees the
// other).  Synchronises the stream.
template <typename K>
int radix_sort_pairs(K **keys, int **payload, long long n, int key_bits, hipStream_t s,
                     int low = 0);
// Keys taken from column indices: the local column, or `none` outside the block.
struct ColumnKeys {
  const int *cols;
  int f_col;
  unsigned ln_col, none;
  __device__ inline unsigned operator[](long long i) const {
    const unsigned c = (unsigned)(cols[i] - f_col);
    return c < ln_col ? c : none;
  }
};
// radix_sort_pairs<unsigned> of src's n keys, read by the first pass in place of
// *keys (whose contents are ignored)
int radix_sort_columns(const ColumnKeys &src, unsigned **keys, int **payload, long long n,
                       int key_bits, hipStream_t s, int low = 0);
// ptr[b] = the first k with (keys[k] >> shift) >= b, b in [0, nb], of n sorted keys
template <typename K>
int bucket_starts(const K *keys, long long n, int shift, long long nb, int *ptr, hipStream_t s);

// problems.hip: row pointers from per-row counts (exclusive scan; *total,
// host, receives the sum; synchronises the stream)
int counts_to_rowptr(const int *cnt, int *rowptr, long long n, long long *total, hipStream_t s);

// problems.hip: CSR transpose into new arrays (rows = src's local columns)
int csr_transpose_arrays(const tbsla_hip_matrix_s *src, int **rowptr_t, int **colidx_t,
                         double **values_t, hipStream_t s);

// split.hip: the split CSR layout (near-diagonal + column-sliced remote)
int split_launch(tbsla_hip_matrix_s *m, double *y, const double *x, const int *done,
                 hipStream_t s);
int split_build(tbsla_hip_matrix_s *m, int window, int slices, hipStream_t s,
                int layout = TBSLA_HIP_CSR_SPLIT);
int split_params(const tbsla_hip_matrix_s *m, int *window, int *slices, int *layout);
// rows per block of the diagonal layout's LDS-slice remote form, or 0 (no
// layout, no remote entries, or the L2-slice form, whose slice count matters)
int split_lds_block_rows(const tbsla_hip_matrix_s *m);
// PageRank's SpMV and update in one pass of the diagonal layout's LDS-slice
// form (CSR / ELL blocks with that form only; split_pr_blocks gives its
// workgroup count, the number of partials, or 0): b = (beta A b_t + S (1 -
// beta) / n_col) / S over the block's rows with b_t = x, as k_pr_update.
struct PrFuse {
  double *b;
  const double *S;
  double beta, n_col;
  double *p_err, *p_sum;
};
int split_pr_blocks(const tbsla_hip_matrix_s *m);
// A PageRank solve's state
struct PrState {
  double S;      // sum of the current iterate
  double err;    // last L1 change
  int iters;     // iterations done (reference counting)
  int done;      // set when the solve has finished
};
constexpr int kPrBlocks = 1024;  // most workgroups (partials) of an update
// The same on the CSR row kernel (spmv.hip): for a square block on the diagonal
// whose row kernel has a fused form; nb workgroups and partials, those of
// k_pr_update on its grid of nb.  q_err, q_sum: the step before's partials, whose
// finalisation (k_pr_finalize's) this step makes, or null when it has been made.
struct PrPrev {
  const double *q_err, *q_sum;
  int NC;
  double epsilon;
};
bool csr_pr_fits(const tbsla_hip_matrix_s *m);
int csr_pr_launch(const tbsla_hip_matrix_s *m, const double *bt, const PrFuse &pf,
                  const PrPrev &prev, PrState *st, unsigned nb, hipStream_t s);
int split_launch_pr(tbsla_hip_matrix_s *m, const double *bt, const PrFuse &pf, const int *done,
                    hipStream_t s);
// The row pointer of a COO / SCOO block's n row-sorted triplets over their
// row range (built once and kept with the block); *ok false when the
// triplets are not sorted by row
int coo_rowptr(tbsla_hip_matrix_s *m, long long n, bool *ok, hipStream_t s);
// The diagonal layout's arrays when it holds every entry (no remote part):
// offsets (device and host), tiled values (dia_at), count, values' length, the
// build's id (unique in the process: a copy made from one build is stale for any
// other, even one whose arrays reuse the same addresses), and whether the values
// are symmetric bit for bit; else 0.
int split_diag_only(const tbsla_hip_matrix_s *m, const int **doff, const int **hoff,
                    const double **dv, int *ndiag, long long *dv_len, unsigned long long *build_id,
                    int *symmetric);

// solvers.hip: after the values of m changed in place: rebuild the split
// layout (it holds a copy of the values), mark copies of the old values
// stale (values_version), synchronise
int values_changed(tbsla_hip_matrix_s *m, hipStream_t s);

}  // namespace tbsla_hip
