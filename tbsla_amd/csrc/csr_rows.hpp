// csr_rows.hpp -- the CSR row kernel (MatrixCSR::Ax, MatrixCSR.cpp:209-224)
// shared by the plain row layout and by the near-diagonal part of the split
// layout.
//
// A wave holds kWave / L lane groups; group g takes R rows (base + r G + g).
// Each lane reads V consecutive entries per trip (one 4 V-byte load of
// column indices and one 8 V-byte load of values), starting from the row's
// first entry rounded down to a multiple of V, so the vector loads stay
// aligned; they may reach V - 1 entries past the row, and past the arrays
// (device_alloc's blocks have room for them).  In a batch of instances (SEG) the
// multiple is counted from the instance's first entry, so that a row is summed
// as in a block of the instance alone; the loads then lie on any entry.  The
// entries are turned in groups of V lanes (lane_transpose), so that x is gathered
// by neighbouring columns; what lies outside the row is not summed (17 entries a
// row, a load per entry at the row's end before: n = 2.5 M 176 -> 143 us, n = 10^6
// 71 -> 57).  Lanes add their entries in trip order and the group adds its lanes
// by a fixed xor tree, so results are deterministic and within rounding of the
// sequential row sum.
//
// NT selects the nontemporal load (the line is not kept in L2 for later
// use): it pays when every line is read whole by one instruction, and
// costs a second fetch when a row's lines are split over trips.  The
// autotuner picks V, L, R and NT per matrix.
#pragma once

#include "common.hpp"

namespace tbsla_hip {

struct CsrRowsArgs {
  long long n_rows;
  const int *rowptr;
  const int *colidx;
  const double *vals;
  const double *x;
  int f_col;
  double *y;
  const int *done;
  // split layout: y[row] = the row's sum + add[row] (its remote products)
  const double *add;
  // optional row segments (instances of a batch): rows [seg_offs[k],
  // seg_offs[k+1]); a wavefront whose rows all lie in one segment with
  // seg_done[k] != 0 returns at once (its rows of y are left as they are)
  const int *seg_offs = nullptr;
  int nseg = 0;
  const int *seg_done = nullptr;
};

// the segment holding row: the largest k with seg_offs[k] <= row
__device__ inline int seg_of_row(const int *offs, int nseg, long long row) {
  int lo = 0, hi = nseg - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (offs[mid] <= row) lo = mid;
    else hi = mid - 1;
  }
  return lo;
}

// ANY: j need not be a multiple of V
template <int V, int NT, bool ANY>
__device__ inline void csr_load(const int *ci, const double *va, int j, int (&c)[V],
                                double (&v)[V]) {
  typedef int vi __attribute__((ext_vector_type(V), aligned((ANY ? 1 : V) * sizeof(int))));
  typedef double vd __attribute__((ext_vector_type(V), aligned((ANY ? 1 : V) * sizeof(double))));
  if (V == 1) {
    c[0] = NT ? __builtin_nontemporal_load(ci + j) : ci[j];
    v[0] = NT ? __builtin_nontemporal_load(va + j) : va[j];
  } else {
    const vi cc = NT ? __builtin_nontemporal_load(reinterpret_cast<const vi *>(ci + j))
                     : *reinterpret_cast<const vi *>(ci + j);
    const vd vv = NT ? __builtin_nontemporal_load(reinterpret_cast<const vd *>(va + j))
                     : *reinterpret_cast<const vd *>(va + j);
#pragma unroll
    for (int k = 0; k < V; k++) {
      c[k] = cc[k];
      v[k] = vv[k];
    }
  }
}

// The sums of the R rows [beg[r], end[r]) of this lane's group, in every lane of
// the group; ent0[r] (SEG): the entry that row r's loads are counted from
template <int V, int L, int R, int NT, bool SEG = false>
__device__ inline void csr_row_sums(const CsrRowsArgs &a, const int (&beg)[R], const int (&end)[R],
                                    int lane, double (&sum)[R], const int (&ent0)[R]) {
  auto down = [&](int e, int r) {  // e rounded down to a load's first entry
    if constexpr (SEG) return e - ((e - ent0[r]) & (V - 1));
    else return e & ~(V - 1);
  };
  int len = 0;
#pragma unroll
  for (int r = 0; r < R; r++) len = max(len, end[r] - down(beg[r], r));
#pragma unroll
  for (int off = kWave / 2; off > 0; off >>= 1) len = max(len, __shfl_xor(len, off, kWave));
  const int trips = (len + V * L - 1) / (V * L);
#pragma unroll
  for (int r = 0; r < R; r++) sum[r] = 0.0;
  // the lane's entries after the turn: slot k is entry V k' + l' of its V lanes' V V
  // entries, l' = lane % V
  const int turned = lane - lane % V;
  for (int t = 0; t < trips; t++) {
    int c[R][V];
    double v[R][V], xv[R][V];
    bool in[R][V];
#pragma unroll
    for (int r = 0; r < R; r++) {
      const int first = down(beg[r], r) + V * t * L;
      // lanes past the row read its last entries again
      const int j = max(min(first + V * lane, down(end[r] - 1, r)), 0);
      csr_load<V, NT, SEG>(a.colidx, a.vals, j, c[r], v[r]);
    }
#pragma unroll
    for (int r = 0; r < R; r++) {
      const int first = down(beg[r], r) + V * t * L;
      if constexpr (V > 1) {
        lane_transpose<V>(c[r]);
        lane_transpose<V>(v[r]);
      }
#pragma unroll
      for (int k = 0; k < V; k++) {
        const int e = first + V * (turned + k) + lane % V;
        in[r][k] = e >= beg[r] && e < end[r];
        xv[r][k] = a.x[in[r][k] ? c[r][k] - a.f_col : 0];
      }
    }
#pragma unroll
    for (int r = 0; r < R; r++)
#pragma unroll
      for (int k = 0; k < V; k++) sum[r] = in[r][k] ? fma(v[r][k], xv[r][k], sum[r]) : sum[r];
  }
#pragma unroll
  for (int r = 0; r < R; r++) sum[r] = group_sum<L>(sum[r]);
}

template <int V, int L, int R, int NT, bool SPLIT, bool SEG>
__global__ __launch_bounds__(kBlock) void k_csr_rows(CsrRowsArgs a) {
  if (a.done && *a.done) return;
  constexpr int G = kWave / L;
  const int lane = threadIdx.x & (L - 1);
  const int g = (threadIdx.x & (kWave - 1)) / L;
  const long long wave = ((long long)blockIdx.x * kBlock + threadIdx.x) / kWave;
  const long long base = wave * (G * R);
  if (base >= a.n_rows) return;
  int seg = 0, seg_end = 0, seg_ent0 = 0;
  if (a.seg_offs) {  // wave-uniform
    const long long last = min(base + G * R, a.n_rows) - 1;
    seg = seg_of_row(a.seg_offs, a.nseg, __builtin_amdgcn_readfirstlane((int)base));
    seg_end = a.seg_offs[seg + 1];
    if constexpr (SEG) seg_ent0 = a.rowptr[a.seg_offs[seg]];
    if (a.seg_done[seg] && last < seg_end) return;
  }
  int beg[R], end[R], ent0[R];
#pragma unroll
  for (int r = 0; r < R; r++) {
    const long long row = base + r * G + g;
    ent0[r] = 0;
    if (row < a.n_rows) {
      beg[r] = a.rowptr[row];
      end[r] = a.rowptr[row + 1];
      if constexpr (SEG) {
        if (row >= seg_end) {  // a later segment: from the row before's on
          do seg_end = a.seg_offs[++seg + 1];
          while (row >= seg_end);
          seg_ent0 = a.rowptr[a.seg_offs[seg]];
        }
        ent0[r] = seg_ent0;
      }
    } else {
      beg[r] = end[r] = 0;
    }
  }
  double sum[R];
  csr_row_sums<V, L, R, NT, SEG>(a, beg, end, lane, sum, ent0);
#pragma unroll
  for (int r = 0; r < R; r++) {
    const long long row = base + r * G + g;
    if (lane == 0 && row < a.n_rows) a.y[row] = SPLIT ? sum[r] + a.add[row] : sum[r];
  }
}

// Schedules with a compiled kernel: V = 1 with L = 1..64 and R = 1, 2, 4;
// V = 2 with L = 4..32 and V = 4 with L = 4..16, both with R = 1, 2.
inline bool csr_rows_valid(int V, int L, int R, int NT) {
  if (NT != 0 && NT != 1) return false;
  if (L < 1 || L > 64 || (L & (L - 1))) return false;
  if (V == 1) return R == 1 || R == 2 || R == 4;
  if (R != 1 && R != 2) return false;
  if (V == 2) return L >= 4 && L <= 32;
  if (V == 4) return L >= 4 && L <= 16;
  return false;
}

template <bool SPLIT, int V, int L, int R, int NT>
void csr_rows_go(const CsrRowsArgs &a, hipStream_t s) {
  const long long rows_per_wave = (long long)(kWave / L) * R;
  const long long waves = (a.n_rows + rows_per_wave - 1) / rows_per_wave;
  const unsigned grid = grid_for(waves * kWave);
  if constexpr (V > 1 && !SPLIT)  // one entry a load: no multiple to count
    if (a.seg_offs) {
      k_csr_rows<V, L, R, NT, false, true><<<grid, kBlock, 0, s>>>(a);
      return;
    }
  k_csr_rows<V, L, R, NT, SPLIT, false><<<grid, kBlock, 0, s>>>(a);
}

template <bool SPLIT, int V, int L, int R>
void csr_rows_nt(const CsrRowsArgs &a, int NT, hipStream_t s) {
  if (NT) csr_rows_go<SPLIT, V, L, R, 1>(a, s);
  else csr_rows_go<SPLIT, V, L, R, 0>(a, s);
}

template <bool SPLIT, int V, int L>
void csr_rows_r(const CsrRowsArgs &a, int R, int NT, hipStream_t s) {
  if (R == 1) csr_rows_nt<SPLIT, V, L, 1>(a, NT, s);
  else if (V > 1 || R == 2) csr_rows_nt<SPLIT, V, L, 2>(a, NT, s);
  else csr_rows_nt<SPLIT, V, L, (V == 1 ? 4 : 2)>(a, NT, s);
}

// Launches the kernel for a schedule that csr_rows_valid accepts.
template <bool SPLIT>
void csr_rows_launch(const CsrRowsArgs &a, int V, int L, int R, int NT, hipStream_t s) {
  if (V == 1) {
    switch (L) {
      case 1: csr_rows_r<SPLIT, 1, 1>(a, R, NT, s); break;
      case 2: csr_rows_r<SPLIT, 1, 2>(a, R, NT, s); break;
      case 4: csr_rows_r<SPLIT, 1, 4>(a, R, NT, s); break;
      case 8: csr_rows_r<SPLIT, 1, 8>(a, R, NT, s); break;
      case 16: csr_rows_r<SPLIT, 1, 16>(a, R, NT, s); break;
      case 32: csr_rows_r<SPLIT, 1, 32>(a, R, NT, s); break;
      default: csr_rows_r<SPLIT, 1, 64>(a, R, NT, s); break;
    }
  } else if (V == 2) {
    switch (L) {
      case 4: csr_rows_r<SPLIT, 2, 4>(a, R, NT, s); break;
      case 8: csr_rows_r<SPLIT, 2, 8>(a, R, NT, s); break;
      case 16: csr_rows_r<SPLIT, 2, 16>(a, R, NT, s); break;
      default: csr_rows_r<SPLIT, 2, 32>(a, R, NT, s); break;
    }
  } else {
    switch (L) {
      case 4: csr_rows_r<SPLIT, 4, 4>(a, R, NT, s); break;
      case 8: csr_rows_r<SPLIT, 4, 8>(a, R, NT, s); break;
      default: csr_rows_r<SPLIT, 4, 16>(a, R, NT, s); break;
    }
  }
}

}  // namespace tbsla_hip
