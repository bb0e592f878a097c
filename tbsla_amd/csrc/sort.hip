// sort.hip -- stable LSD radix sort and the COO conversion constructors.
//
// Radix sort of 32- or 64-bit keys carrying each key's original position, and of
// matrix entries by an index of theirs, in digits of at most 8 bits.  Per pass: a
// per-tile digit histogram, one exclusive scan over the digit-major histogram,
// and a stable scatter.  Stability inside a tile comes from processing elements in
// index order: each wavefront owns a contiguous sub-tile, walks it in 64-element
// rounds, finds the lanes that share its digit with one ballot per digit bit and
// ranks itself among them; per-wave counts live in LDS.  The tile's elements are
// then put into LDS in digit order and written from there, so that an output run
// of one digit is written by consecutive lanes.  Integer work only: the
// permutation is unique.
#include <algorithm>
#include <vector>

#include "common.hpp"
#include "kernels.hpp"
#include "radix_tile.hpp"

namespace tbsla_hip {

namespace {

constexpr int kItems = 16;  // keys per thread of a tile

// Tiles: 512 threads for 32-bit keys, 256 for 64-bit ones; both put 32 KB of
// keys through LDS.  With the counts a workgroup takes 42,016 bytes of a CU's
// 163,840 for 32-bit keys and for entries, 37,904 for 64-bit keys: three and four
// fit.
template <typename K>
struct SortTile {
  typedef K key;
  static constexpr int items = kItems;
  static constexpr int threads = sizeof(K) == 4 ? 512 : 256;
  static constexpr int elems = threads * kItems;
  static constexpr int waves = threads / kWave;
};
// of matrix entries (k_entry_scatter)
struct EntryTile {
  typedef unsigned key;
  static constexpr int items = 8;
  static constexpr int threads = 512;
  static constexpr int elems = threads * items;
  static constexpr int waves = threads / kWave;
};

// Digit counts of each tile.  Per-wave counters in LDS; the lanes of a round that
// hold its first lane's digit (most of them in the high digits of a banded or
// sorted input) are counted by that lane instead of added one by one to one
// address.  keys: an array, or a source with its operator[] (ColumnKeys).
template <typename T, typename Src>
__global__ __launch_bounds__(T::threads) void k_digit_hist(
    const Src keys, long long n, int shift, int mask, long long ntiles, int *__restrict__ hist) {
  typedef typename T::key K;
  constexpr int kItems = T::items;
  __shared__ int h[T::waves][kRadix];
  for (int i = threadIdx.x; i < T::waves * kRadix; i += T::threads) (&h[0][0])[i] = 0;
  __syncthreads();
  const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
  const long long base = (long long)blockIdx.x * T::elems + threadIdx.x;
  K key[kItems];
#pragma unroll
  for (int i = 0; i < kItems; i++) {
    const long long e = base + i * T::threads;
    key[i] = e < n ? keys[e] : (K)0;
  }
#pragma unroll
  for (int i = 0; i < kItems; i++) {
    const bool valid = base + i * T::threads < n;
    const int d = (int)(key[i] >> shift) & mask;
    const int first = __builtin_amdgcn_readfirstlane(d);
    const unsigned long long same = __ballot(valid && d == first);
    if (lane == 0 && same) atomicAdd(&h[wave][first], __popcll(same));
    if (valid && d != first) atomicAdd(&h[wave][d], 1);
  }
  __syncthreads();
  for (int d = threadIdx.x; d <= mask; d += T::threads) {
    int c = 0;
    for (int w = 0; w < T::waves; w++) c += h[w][d];
    hist[(long long)d * ntiles + blockIdx.x] = c;
  }
}

// The stable scatter of one pass; pay_in null: the payload of element e is e
// (the first pass).  Bound by its bytes once the output runs are whole: 24 M
// 32-bit keys take 101 us a pass (16 bytes an element, 3.8 TB/s) where
// the scatter from registers, with 64-bit keys read twice, took 290 (2.0 TB/s).
template <typename K, typename Src>
__global__ __launch_bounds__(SortTile<K>::threads) void k_digit_scatter(
    const Src keys_in, const int *__restrict__ pay_in, K *__restrict__ keys_out,
    int *__restrict__ pay_out, long long n, int shift, int bits, long long ntiles,
    const int *__restrict__ offsets) {
  typedef SortTile<K> T;
  __shared__ TileRank<T::threads> sh;
  __shared__ K stage[T::elems];
  const int mask = (1 << bits) - 1;
  const long long tile0 = (long long)blockIdx.x * T::elems;
  const int count = (int)min((long long)T::elems, n - tile0);
  const int sub = tile_sub<kItems>();
  K key[kItems];
  int pay[kItems], pos[kItems];
#pragma unroll
  for (int i = 0; i < kItems; i++) {
    const int e = sub + i * kWave;
    key[i] = e < count ? keys_in[tile0 + e] : (K)0;
  }
#pragma unroll
  for (int i = 0; i < kItems; i++) {
    const int e = sub + i * kWave;
    pay[i] = pay_in ? (e < count ? pay_in[tile0 + e] : 0) : (int)(tile0 + e);
  }
  int start, total;
  rank_tile<T::threads, kItems, K>(sh, key, pos, count, shift, bits, start, total);
  if ((int)threadIdx.x <= mask)
    sh.gofs[threadIdx.x] = offsets[(long long)threadIdx.x * ntiles + blockIdx.x] - start;
#pragma unroll
  for (int i = 0; i < kItems; i++)
    if (sub + i * kWave < count) stage[pos[i]] = key[i];
  __syncthreads();
  int dst[kItems];
#pragma unroll
  for (int i = 0; i < kItems; i++) {
    const int t = threadIdx.x + i * T::threads;
    if (t < count) {
      const K k = stage[t];
      dst[i] = sh.gofs[(int)(k >> shift) & mask] + t;
      keys_out[dst[i]] = k;
    }
  }
  __syncthreads();
  int *pstage = reinterpret_cast<int *>(stage);
#pragma unroll
  for (int i = 0; i < kItems; i++)
    if (sub + i * kWave < count) pstage[pos[i]] = pay[i];
  __syncthreads();
#pragma unroll
  for (int i = 0; i < kItems; i++) {
    const int t = threadIdx.x + i * T::threads;
    if (t < count) pay_out[dst[i]] = pstage[t];
  }
}

// A pass over matrix entries: key (the index sorted by), other (the other index)
// and value move together, so no gather by sorted position follows (4.8 M
// entries: 171 us, a cache line for each value and column).  Tiles of 4096, a
// value of each through LDS at a time: 32 KB.  4.8 M entries take 32 us a pass (32
// bytes an entry, 4.8 TB/s).
constexpr int kEntThreads = EntryTile::threads, kEntItems = EntryTile::items;
constexpr int kEntTile = EntryTile::elems;

__global__ __launch_bounds__(kEntThreads) void k_entry_scatter(
    const int *__restrict__ key_in, const int *__restrict__ other_in,
    const double *__restrict__ val_in, int *__restrict__ key_out, int *__restrict__ other_out,
    double *__restrict__ val_out, long long n, int shift, int bits, long long ntiles,
    const int *__restrict__ offsets) {
  __shared__ TileRank<kEntThreads> sh;
  __shared__ double stage[kEntTile];
  const int mask = (1 << bits) - 1;
  const long long tile0 = (long long)blockIdx.x * kEntTile;
  const int count = (int)min((long long)kEntTile, n - tile0);
  const int sub = tile_sub<kEntItems>();
  unsigned key[kEntItems];
  int other[kEntItems], pos[kEntItems], dst[kEntItems];
  double val[kEntItems];
#pragma unroll
  for (int i = 0; i < kEntItems; i++) {
    const int e = min(sub + i * kWave, count - 1);
    key[i] = key_in[tile0 + e];
    other[i] = other_in[tile0 + e];
    val[i] = val_in[tile0 + e];
  }
  int start, total;
  rank_tile<kEntThreads, kEntItems, unsigned>(sh, key, pos, count, shift, bits, start, total);
  if ((int)threadIdx.x <= mask)
    sh.gofs[threadIdx.x] = offsets[(long long)threadIdx.x * ntiles + blockIdx.x] - start;
  int *istage = reinterpret_cast<int *>(stage);
#pragma unroll
  for (int i = 0; i < kEntItems; i++)
    if (sub + i * kWave < count) istage[pos[i]] = (int)key[i];
  __syncthreads();
#pragma unroll
  for (int i = 0; i < kEntItems; i++) {
    const int t = threadIdx.x + i * kEntThreads;
    if (t < count) {
      const unsigned k = istage[t];
      dst[i] = sh.gofs[(int)(k >> shift) & mask] + t;
      key_out[dst[i]] = (int)k;
    }
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < kEntItems; i++)
    if (sub + i * kWave < count) istage[pos[i]] = other[i];
  __syncthreads();
#pragma unroll
  for (int i = 0; i < kEntItems; i++) {
    const int t = threadIdx.x + i * kEntThreads;
    if (t < count) other_out[dst[i]] = istage[t];
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < kEntItems; i++)
    if (sub + i * kWave < count) stage[pos[i]] = val[i];
  __syncthreads();
#pragma unroll
  for (int i = 0; i < kEntItems; i++) {
    const int t = threadIdx.x + i * kEntThreads;
    if (t < count) val_out[dst[i]] = stage[t];
  }
}

// ptr[b] = the first k with (keys[k] >> shift) >= b, for b in [0, nb]: the
// bucket starts of sorted keys, by binary search (no atomics: counting 24 M
// banded keys by atomic additions took 1053 us, and 4.8 M with hub rows 317).
// Two waves find the ends of their workgroup's 256 buckets among all keys, 64
// probes at a time; the threads then search between them.
template <typename K>
__device__ inline long long first_at_least(const K *__restrict__ keys, int shift, long long lo,
                                           long long hi, long long b) {
  while (lo < hi) {
    const long long mid = (lo + hi) >> 1;
    if ((long long)(keys[mid] >> shift) < b) lo = mid + 1;
    else hi = mid;
  }
  return lo;
}

template <typename K>
__global__ __launch_bounds__(kBlock) void k_bucket_starts(const K *__restrict__ keys, long long n,
                                                          int shift, long long nb,
                                                          int *__restrict__ ptr) {
  __shared__ long long ends[2];
  const long long b0 = (long long)blockIdx.x * kBlock, b = b0 + threadIdx.x;
  const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
  if (wave < 2) {
    const long long want = b0 + wave * kBlock;
    long long lo = 0, hi = n;  // the answer lies in [lo, hi]
    while (hi - lo > kWave) {
      const long long step = (hi - lo) / kWave, at = lo + lane * step;
      const unsigned long long less = __ballot((long long)(keys[at] >> shift) < want);
      const int m = __popcll(less);  // probes below `want`: lanes 0 .. m - 1
      if (m < kWave) hi = lo + m * step;
      lo = m ? lo + (m - 1) * step + 1 : lo;
    }
    const unsigned long long less =
        __ballot(lo + lane < hi && (long long)(keys[min(lo + lane, n - 1)] >> shift) < want);
    if (lane == 0) ends[wave] = lo + __popcll(less);
  }
  __syncthreads();
  if (b <= nb) ptr[b] = (int)first_at_least(keys, shift, ends[0], ends[1], b);
}

// the longest row
__global__ __launch_bounds__(kBlock) void k_max_row(const int *__restrict__ rowptr, long long n,
                                                    int *__restrict__ out) {
  int m = 0;
  for (long long i = (long long)blockIdx.x * kBlock + threadIdx.x; i < n;
       i += (long long)gridDim.x * kBlock)
    m = max(m, rowptr[i + 1] - rowptr[i]);
  if (m > 0) atomicMax(out, m);
}

// ELL slots from row-sorted (col, val) with rowptr: column-major, padded.
__global__ __launch_bounds__(kBlock) void k_rows_to_ell(long long n_rows, int max_col,
                                                        const int *__restrict__ rowptr,
                                                        const int *__restrict__ cols,
                                                        const double *__restrict__ vals,
                                                        int *__restrict__ ecols,
                                                        double *__restrict__ evals) {
  long long r = (long long)blockIdx.x * kBlock + threadIdx.x;
  if (r >= n_rows) return;
  int b = rowptr[r], e = rowptr[r + 1];
  for (int j = 0; j < max_col; j++) {
    size_t s = (size_t)j * n_rows + r;
    bool in = b + j < e;
    ecols[s] = in ? cols[b + j] : 0;
    evals[s] = in ? vals[b + j] : 0.0;
  }
}

// DENSE(COO) (MatrixDENSE.cpp:34-36): per row, the row's triplets in COO
// order (stable row sort), so repeated cells add in the reference's order.
__global__ __launch_bounds__(kBlock) void k_rows_to_dense(long long n_rows, long long ln_col,
                                                          const int *__restrict__ rowptr,
                                                          const int *__restrict__ perm,
                                                          const int *__restrict__ cols,
                                                          const double *__restrict__ vals,
                                                          double *__restrict__ dense) {
  long long r = (long long)blockIdx.x * kBlock + threadIdx.x;
  if (r >= n_rows) return;
  double *row = dense + (size_t)r * ln_col;
  for (int j = rowptr[r]; j < rowptr[r + 1]; j++) {
    int p = perm[j];
    row[cols[p]] += vals[p];
  }
}

__global__ __launch_bounds__(kBlock) void k_zero_d(double *__restrict__ d, long long n) {
  for (long long i = (long long)blockIdx.x * kBlock + threadIdx.x; i < n;
       i += (long long)gridDim.x * kBlock)
    d[i] = 0.0;
}

unsigned stride_grid(long long n) {
  long long g = (n + kBlock - 1) / kBlock;
  if (g > 65536) g = 65536;
  if (g < 1) g = 1;
  return (unsigned)g;
}

int bits_for(long long v) {
  int b = 0;
  while (b < 62 && (1LL << b) <= v) b++;
  return std::max(b, 1);
}

}  // namespace

template <typename K, typename Src>
static int radix_sort_from(const Src *first, K **keys, int **payload, long long n, int key_bits,
                           hipStream_t s, int low = 0) {
  typedef SortTile<K> T;
  if (n <= 0) return TBSLA_HIP_SUCCESS;
  const long long ntiles = (n + T::elems - 1) / T::elems;
  const int passes = std::max(1, (key_bits - low + 7) / 8);
  const int bits = std::max(1, (key_bits - low + passes - 1) / passes);
  const long long hist_n = (1LL << bits) * ntiles;
  K *keys_alt = nullptr;
  int *pay_alt = nullptr, *hist = nullptr;
  void *ws = nullptr;
  auto cleanup = [&]() {
    (void)hipStreamSynchronize(s);
    device_free(keys_alt);
    device_free(pay_alt);
    device_free(hist);
    device_free(ws);
  };
  int st = TBSLA_HIP_SUCCESS;
  if ((st = device_alloc((void **)&keys_alt, (size_t)n * sizeof(K))) ||
      (st = device_alloc((void **)&pay_alt, (size_t)n * 4)) ||
      (st = device_alloc((void **)&hist, (size_t)hist_n * 4)) ||
      (st = device_alloc(&ws, scan_workspace_bytes(hist_n)))) {
    cleanup();
    return st;
  }
  for (int p = 0; p < passes; p++) {
    const int shift = low + bits * p, b = std::min(bits, std::max(1, key_bits - shift));
    const K *kin = *keys;
    if (p == 0 && first)
      k_digit_hist<T><<<(unsigned)ntiles, T::threads, 0, s>>>(*first, n, shift, (1 << b) - 1,
                                                              ntiles, hist);
    else
      k_digit_hist<T><<<(unsigned)ntiles, T::threads, 0, s>>>(kin, n, shift, (1 << b) - 1, ntiles,
                                                              hist);
    st = scan<int>(hist, hist, (1LL << b) * ntiles, false, nullptr, ws, s);
    if (st) break;
    if (p == 0 && first)
      k_digit_scatter<K><<<(unsigned)ntiles, T::threads, 0, s>>>(*first, nullptr, keys_alt, pay_alt,
                                                                 n, shift, b, ntiles, hist);
    else
      k_digit_scatter<K><<<(unsigned)ntiles, T::threads, 0, s>>>(
          kin, p > 0 ? *payload : nullptr, keys_alt, pay_alt, n, shift, b, ntiles, hist);
    std::swap(*keys, keys_alt);
    std::swap(*payload, pay_alt);
  }
  hipError_t e = hipGetLastError();
  cleanup();
  if (st) return st;
  if (e != hipSuccess) return fail(TBSLA_HIP_ERR_HIP, std::string("radix sort: ") + hipGetErrorString(e));
  return TBSLA_HIP_SUCCESS;
}

template <typename K>
int radix_sort_pairs(K **keys, int **payload, long long n, int key_bits, hipStream_t s, int low) {
  return radix_sort_from<K, const K *>(nullptr, keys, payload, n, key_bits, s, low);
}

int radix_sort_columns(const ColumnKeys &src, unsigned **keys, int **payload, long long n,
                       int key_bits, hipStream_t s, int low) {
  return radix_sort_from<unsigned, ColumnKeys>(&src, keys, payload, n, key_bits, s, low);
}

template int radix_sort_pairs<unsigned>(unsigned **, int **, long long, int, hipStream_t, int);
template int radix_sort_pairs<unsigned long long>(unsigned long long **, int **, long long, int,
                                                  hipStream_t, int);

template <typename K>
int bucket_starts(const K *keys, long long n, int shift, long long nb, int *ptr, hipStream_t s) {
  k_bucket_starts<K><<<grid_for(nb + 1), kBlock, 0, s>>>(keys, n, shift, nb, ptr);
  TBSLA_HIP_LAUNCH_CHECK();
  return TBSLA_HIP_SUCCESS;
}

template int bucket_starts<unsigned>(const unsigned *, long long, int, long long, int *,
                                     hipStream_t);
template int bucket_starts<unsigned long long>(const unsigned long long *, long long, int,
                                               long long, int *, hipStream_t);

// The CSR arrays of n COO triplets: stable order by (row, col)
// (csr::compare_row, src/cpp/utils/csr.cpp:3-8): passes over the columns' digits,
// then over the rows'; those over the columns are left out where the triplets are
// in column order already (known from the import, as a column-ordered file gives
// them).  300,007 rows, 4.8 M triplets in column order: 368 -> 189 us (three passes
// and a gather before).
static int coo_rows(const tbsla_hip_matrix_s *coo, long long n, int *rowptr, int *cols,
                    double *vals, hipStream_t s) {
  const int row_bits = bits_for(std::max(coo->n_row, 1));
  const int col_bits = coo->col_sorted ? 0 : bits_for(std::max(coo->n_col, 1));
  const int row_passes = (row_bits + 7) / 8, col_passes = (col_bits + 7) / 8;
  const int passes = row_passes + col_passes;
  const int rb = (row_bits + row_passes - 1) / row_passes;
  const int cb = col_passes ? (col_bits + col_passes - 1) / col_passes : 0;
  const long long ntiles = (n + kEntTile - 1) / kEntTile;
  const long long hist_n = (1LL << std::max(rb, cb)) * std::max(ntiles, 1LL);
  const size_t len = (size_t)std::max(n, 1LL);
  // where a pass's entries go: the result's arrays and others in turn, the last
  // pass's to the result's (its rows, in order, to rows[0])
  int *rows[2] = {nullptr, nullptr}, *oc[2] = {cols, nullptr}, *hist = nullptr;
  double *ov[2] = {vals, nullptr};
  void *ws = nullptr;
  int st;
  if (!(st = device_alloc((void **)&rows[0], len * 4)) &&
      !(st = device_alloc((void **)&rows[1], passes > 1 ? len * 4 : 4)) &&
      !(st = device_alloc((void **)&oc[1], passes > 1 ? len * 4 : 4)) &&
      !(st = device_alloc((void **)&ov[1], passes > 1 ? len * 8 : 8)) &&
      !(st = device_alloc((void **)&hist, (size_t)hist_n * 4)) &&
      !(st = device_alloc(&ws, scan_workspace_bytes(hist_n)))) {
    const int *r_in = coo->rowidx, *c_in = coo->colidx;
    const double *v_in = coo->values;
    for (int p = 0; n > 0 && !st && p < passes; p++) {
      const bool by_row = p >= col_passes;
      const int shift = by_row ? rb * (p - col_passes) : cb * p;
      const int bits = by_row ? std::min(rb, row_bits - shift) : std::min(cb, col_bits - shift);
      const int *key = by_row ? r_in : c_in, *other = by_row ? c_in : r_in;
      const int to = (passes - 1 - p) % 2;
      k_digit_hist<EntryTile><<<(unsigned)ntiles, kEntThreads, 0, s>>>(
          key, n, shift, (1 << bits) - 1, ntiles, hist);
      st = scan<int>(hist, hist, (1LL << bits) * ntiles, false, nullptr, ws, s);
      if (st) break;
      k_entry_scatter<<<(unsigned)ntiles, kEntThreads, 0, s>>>(
          key, other, v_in, by_row ? rows[to] : oc[to], by_row ? oc[to] : rows[to], ov[to], n,
          shift, bits, ntiles, hist);
      r_in = rows[to];
      c_in = oc[to];
      v_in = ov[to];
    }
    if (!st)
      st = bucket_starts<unsigned>(reinterpret_cast<unsigned *>(rows[0]), n, 0, coo->n_row, rowptr,
                                   s);
    const hipError_t e = hipGetLastError();
    if (!st && e != hipSuccess) st = fail(TBSLA_HIP_ERR_HIP, hipGetErrorString(e));
  }
  (void)hipStreamSynchronize(s);
  device_free(rows[0]);
  device_free(rows[1]);
  device_free(oc[1]);
  device_free(ov[1]);
  device_free(hist);
  device_free(ws);
  return st;
}

}  // namespace tbsla_hip

using namespace tbsla_hip;

// <FMT>(const MatrixCOO&): MatrixCSR.cpp:49-96, MatrixELL.cpp:25-79,
// MatrixSCOO.cpp:75-101, MatrixDENSE.cpp:15-37.  The geometry is the COO's,
// with ln_row = n_row and ln_col = n_col.
extern "C" int tbsla_hip_convert(tbsla_hip_matrix_t dst, int format, tbsla_hip_matrix_t coo,
                                 void *stream) {
  if (!dst || !coo || dst == coo) return fail(TBSLA_HIP_ERR_INVALID, "bad handles");
  if (coo->format != TBSLA_HIP_COO) return fail(TBSLA_HIP_ERR_INVALID, "source must be COO");
  if (format < TBSLA_HIP_SCOO || format > TBSLA_HIP_DENSE)
    return fail(TBSLA_HIP_ERR_INVALID, "target must be SCOO, CSR, ELL or DENSE");
  hipStream_t s = static_cast<hipStream_t>(stream);
  release_arrays(dst);
  dst->format = format;
  dst->n_row = coo->n_row;
  dst->n_col = coo->n_col;
  dst->ln_row = coo->n_row;
  dst->ln_col = coo->n_col;
  dst->f_row = coo->f_row;
  dst->f_col = coo->f_col;
  dst->pr = coo->pr;
  dst->pc = coo->pc;
  dst->NR = coo->NR;
  dst->NC = coo->NC;
  dst->nnz = coo->nnz;
  dst->max_col = 0;
  dst->row_sorted = coo->row_sorted;
  // the reference converts nnz triplets; never more than are held
  const long long n = coo->has_arrays ? std::min(coo->nnz, coo->stored) : 0;
  const long long rows = dst->n_row;

  if (format == TBSLA_HIP_SCOO) {
    dst->stored = n;
    dst->has_arrays = n > 0;
    TBSLA_TRY(device_alloc((void **)&dst->rowidx, (size_t)std::max(n, 1LL) * 4));
    TBSLA_TRY(device_alloc((void **)&dst->colidx, (size_t)std::max(n, 1LL) * 4));
    TBSLA_TRY(device_alloc((void **)&dst->values, (size_t)std::max(n, 1LL) * 8));
    if (n > 0) {
      TBSLA_HIP_CHECK(hipMemcpyAsync(dst->rowidx, coo->rowidx, n * 4, hipMemcpyDeviceToDevice, s));
      TBSLA_HIP_CHECK(hipMemcpyAsync(dst->colidx, coo->colidx, n * 4, hipMemcpyDeviceToDevice, s));
      TBSLA_HIP_CHECK(hipMemcpyAsync(dst->values, coo->values, n * 8, hipMemcpyDeviceToDevice, s));
    }
    TBSLA_HIP_CHECK(hipStreamSynchronize(s));
    return TBSLA_HIP_SUCCESS;
  }
  if (format == TBSLA_HIP_ELL && n == 0) {
    dst->nnz = 0;  // MatrixELL.cpp:39-41
    TBSLA_HIP_CHECK(hipStreamSynchronize(s));
    return TBSLA_HIP_SUCCESS;
  }

  int *rowptr = nullptr;
  TBSLA_TRY(device_alloc((void **)&rowptr, (size_t)(rows + 1) * 4));
  if (format == TBSLA_HIP_DENSE) {
    // DENSE needs only a stable row order (cells add in COO order)
    unsigned *keys = nullptr;
    int *perm = nullptr;
    auto drop = [&]() {
      (void)hipStreamSynchronize(s);
      device_free(keys);
      device_free(perm);
      device_free(rowptr);
    };
    const size_t cells = (size_t)rows * (size_t)dst->ln_col;
    int st;
    if ((st = device_alloc((void **)&keys, (size_t)std::max(n, 1LL) * 4)) ||
        (st = device_alloc((void **)&perm, (size_t)std::max(n, 1LL) * 4)) ||
        (st = device_alloc((void **)&dst->values, std::max<size_t>(cells, 1) * 8))) {
      drop();
      return st;
    }
    const unsigned *rows_in = reinterpret_cast<const unsigned *>(coo->rowidx);
    if ((st = radix_sort_from<unsigned, const unsigned *>(&rows_in, &keys, &perm, n,
                                                          bits_for(std::max(coo->n_row, 1)), s)) ||
        (st = bucket_starts<unsigned>(keys, n, 0, rows, rowptr, s))) {
      drop();
      return st;
    }
    k_zero_d<<<stride_grid((long long)cells), kBlock, 0, s>>>(dst->values, (long long)cells);
    if (rows > 0)
      k_rows_to_dense<<<grid_for(rows), kBlock, 0, s>>>(rows, dst->ln_col, rowptr, perm,
                                                        coo->colidx, coo->values, dst->values);
    const hipError_t e = hipGetLastError();
    drop();
    if (e != hipSuccess) return fail(TBSLA_HIP_ERR_HIP, hipGetErrorString(e));
    dst->stored = (long long)cells;
    dst->has_arrays = 1;
    return TBSLA_HIP_SUCCESS;
  }

  int *scol = nullptr;
  double *sval = nullptr;
  TBSLA_TRY(device_alloc((void **)&scol, (size_t)std::max(n, 1LL) * 4));
  TBSLA_TRY(device_alloc((void **)&sval, (size_t)std::max(n, 1LL) * 8));
  {
    const int st = coo_rows(coo, n, rowptr, scol, sval, s);
    if (st) {
      device_free(rowptr);
      device_free(scol);
      device_free(sval);
      return st;
    }
  }
  if (format == TBSLA_HIP_CSR) {
    dst->rowptr = rowptr;
    dst->colidx = scol;
    dst->values = sval;
    dst->stored = n;
    dst->has_arrays = 1;
    return TBSLA_HIP_SUCCESS;
  }
  // ELL: width = longest row
  TBSLA_TRY(ensure_scratch(dst, 256));
  int *d_w = reinterpret_cast<int *>(dst->scratch);
  TBSLA_HIP_CHECK(hipMemsetAsync(d_w, 0, 4, s));
  k_max_row<<<stride_grid(rows), kBlock, 0, s>>>(rowptr, rows, d_w);
  int width = 0;
  TBSLA_HIP_CHECK(hipMemcpyAsync(&width, d_w, 4, hipMemcpyDeviceToHost, s));
  TBSLA_HIP_CHECK(hipStreamSynchronize(s));
  dst->max_col = width;
  const size_t slots = (size_t)rows * (size_t)width;
  TBSLA_TRY(device_alloc((void **)&dst->colidx, std::max<size_t>(slots, 1) * 4));
  TBSLA_TRY(device_alloc((void **)&dst->values, std::max<size_t>(slots, 1) * 8));
  if (rows > 0 && width > 0)
    k_rows_to_ell<<<grid_for(rows), kBlock, 0, s>>>(rows, width, rowptr, scol, sval, dst->colidx,
                                                    dst->values);
  TBSLA_HIP_LAUNCH_CHECK();
  dst->stored = (long long)slots;
  dst->has_arrays = 1;
  TBSLA_HIP_CHECK(hipStreamSynchronize(s));
  device_free(rowptr);
  device_free(scol);
  device_free(sval);
  return TBSLA_HIP_SUCCESS;
}
