// cg.hip -- the CG driver (src/mpi/matrix/CG.cpp:32-73, with the swapped
// Ax arguments of :61 corrected) for one system or for a batch of independent
// systems stored block-diagonally in one CSR block.
//
// Iteration i of the reference loop is two kernels (three with M = G G^T):
//
//   K1  beta = rz_new / max(rz_old, nz); p' = z + beta p (own rows);
//       Ap = A (z + beta p) by gathering z and p at the columns; pAp partials.
//       For i > 0 it first applies the reference's test on |r| and counts
//       the iteration (it++ only when not converged, CG.cpp:66-72).
//   K2  alpha = rz / max(pAp, nz); x += alpha p'; r' = r - alpha Ap;
//       z' = D^-1 r' (Jacobi) or t = G^T r' (computed from r and Ap at the
//       columns); r.r and r.z partials.
//   K3  (M = G G^T) z' = G t; r.z partials.
//
// r and p are double-buffered by iteration parity, so no kernel reads what
// another block of the same kernel writes.  Every reduction is one partial
// per workgroup; each consumer workgroup re-sums its system's partials in the
// same fixed order, so all workgroups see bitwise-equal scalars and repeated
// runs give identical bits.  Systems keep their own state (threshold,
// iteration count, convergence, wall-clock time of convergence); a converged
// system's workgroups return at once.  Iterations run in hipGraph-captured
// batches; the host polls a small status copy with one batch in flight.
//
// Precision forms: FP64 (the reference's), or FP32 matrix values, FP32
// accumulation in the SpMV and in the preconditioner, with FP64 vectors and
// dot products and the true FP64 residual r = b - A x every replace_every
// iterations and before convergence is accepted.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <mutex>
#include <tuple>
#include <type_traits>
#include <vector>

#include "common.hpp"
#include "kernels.hpp"

namespace tbsla_hip {

namespace {

constexpr double kNearZero = 1.0e-10;  // CG.cpp:35
constexpr int kMaxBlocksPerSystem = 1024;
constexpr int kBatchBlocksPerSystem = 256;  // default for a batch of systems
constexpr long long kRowsPerBlockLone = 512;  // default rows per workgroup of a lone system
constexpr long long kTwoPassEntries = 1LL << 24;  // K1 in two passes from this many entries

enum SegDone { kRunning = 0, kConverged = 1, kPending = 2, kBreakdown = 3, kInactive = 5 };

struct CgSeg {
  double stop;       // threshold on |r|
  double near_zero;  // clamp of alpha's and beta's divisors
  double rnorm;      // |r| at the last test
  double rnorm0;     // |r0|
  long long t_done;  // wall clock when the system finished
  int iters;         // reference counting
  int done;          // SegDone
  int shift;         // buffer parity of this system relative to the global iteration
  int true_res;      // the current r.r partials belong to a true residual b - A x
  int stop_par;      // buffer parity at the test that ended the recurrence
  int row0, row1;    // rows of the system
  int blk0, blk1;    // workgroups of the system (same in every kernel)
  int rpb;           // rows per workgroup
  int ent0;          // the first entry of row0
  // K2 found the system not running: K1 may leave at once (last here: among the
  // fields that a lone system loads together it cost its solve 0.4 %)
  int left;
};

struct CgCom {
  int ndone;     // systems finished for good
  int npending;  // systems waiting for the true-residual test
  long long t0;  // wall clock at the start of the iteration
  double ratio;  // the first system's |r| over its threshold at its last test
};

struct CgArgs {
  const int *rowptr;
  const int *colidx;
  const double *val64;
  const float *val32;
  int f_col;
  // M = G G^T: rows of G (lower) and of G^T
  const int *g_rp;
  const int *g_ci;
  const double *g_v64;
  const float *g_v32;
  const int *t_rp;
  const int *t_ci;
  const double *t_v64;
  const float *t_v32;
  const double *dinv;
  // M = G G^T with G held on A's stored diagonals of offset <= 0 (a stencil
  // factor): offsets (ascending), tiled values (dia_at) and their FP32 copy;
  // G^T is read from the same slots (G^T_{i,i-o} = G_{i-o,i})
  const int *gdoff;
  const double *gd64;
  const float *gd32;
  int gndiag;
  const double *b;
  double *x;
  double *r[2];
  double *p[2];
  double *z;
  double *ap;
  double *ax;  // A x in FP64 (true residuals)
  double *t64;
  float *t32;
  double *ppap;
  double *prr[2];
  double *prz[2];
  CgSeg *seg;
  CgCom *com;
  const int *block_seg;
  int verify;        // recurrence convergence waits for the true residual
  int stall_window;  // > 0: breakdown when |r| has not dropped below |r0| by then
  int a_nnz;         // stored entries of A
  int g_nnz;         // stored entries of G (and of G^T)
  // A in the diagonal layout (every entry on a stored diagonal): offsets,
  // tiled values (dia_at), their FP32 copy, count, A's columns
  const int *doff;
  const double *dv64;
  const float *dv32;
  int ndiag;
  int ncol;
  // the first 8 offsets of each again, at hand with the arguments (G's last one
  // repeated)
  int doff8[8];
  int gdoff8[8];
};

// What the kernels find at one known address: the arguments, the status counts
// and the state of a lone system (a batch's systems lie at args.seg).  A lone
// system's kernels then load arguments and state in one trip to memory, before
// the rows' data, where arguments, the workgroup's system, that system's state
// and the diagonals' offsets took one each (10^6 rows, mixed: K1 17.1 -> 16.2 us,
// K3 7.9 -> 7.4).
struct CgBlock {
  CgArgs args;
  CgSeg seg;
  CgCom com;
};

// Every kernel reads its arguments from one CgBlock in device memory
// that the solve's cache owns for its whole lifetime: a captured graph then
// names only that block (and its launch shape), never a matrix or work
// buffer, so one instantiated graph serves every later solve of the same
// shape and no graph can refer to memory that has been freed since.
// multi_: a batch of systems, whose workgroups look theirs up in block_seg.
#define CG_ARGS const CgBlock *__restrict__ pa_, int multi_
#define CG_BIND const CgArgs a = cg_bind(&pa_->args)

// The argument block read as constant memory, by scalar loads, and its pointers
// as pointers to global memory.  A pointer that is itself loaded would otherwise
// be a generic one, and what is read through it would go by flat instructions,
// which count as LDS accesses too, take no uniform base and hold a 64-bit
// address each.
#define TBSLA_CONST __attribute__((address_space(4))) const
template <typename T>
__device__ inline T *arg(T *TBSLA_CONST *slot) {
  typedef __attribute__((address_space(1))) T G;
  return (T *)*(G *TBSLA_CONST *)slot;
}

// The workgroup's place in the layout.  A lone system's: the 8 XCDs, which take
// workgroups in turn, each get a contiguous eighth of them, so that rows share an
// L2 with most of the rows that their columns name (64^3, FP64: K1 8.3 -> 7.8 us,
// K2 6.7 -> 5.6; 10^6 rows, mixed, factored: K1 16.2 -> 15.0, K2 15.2 -> 14.3, K3
// 7.4 -> 6.5).  A batch's in turn: its systems differ in rows and iterations, and
// eighths of it in work (96 systems, K1b: 115 us as it is, 135 in eighths; runs
// of 16 or 64 workgroups an XCD, 115 and 119).
__device__ inline int cg_block(int multi) {
  const int i = blockIdx.x / 8, x = blockIdx.x % 8, n = gridDim.x;
  return multi ? blockIdx.x : x * (n / 8) + min(x, n % 8) + i;
}
// pointer i (0 or 1) of a pair
#define CG_AT(field, i) ((i) ? a.field[1] : a.field[0])
// offset i < 8 of A's or of G's diagonals
#define CG_OFF(field, i) ((TBSLA_CONST CgBlock *)pa_)->args.field[i]
// The system of workgroup b: S, and in sg what a kernel of the iteration reads
// of it and none of that launch writes: every wavefront reads it for itself.  K1's
// test writes `done`, and `iters` where it does not read it, so the kernels that
// make the test take `done` from seg_finish alone, one answer for the workgroup;
// sg.done is for those that do not, and `left`, which K2 writes, for K1's first pass
// (96 systems: 9.00 ms by the shared flag alone, 8.80 with it).  A lone system's is
// read at once, with the arguments: CG_HAND names those a kernel needs first, so
// that the compiler asks for all of them before it waits.
#define CG_SYSTEM(b, ...)                                                              \
  CgPart sg = cg_part(&((TBSLA_CONST CgBlock *)pa_)->seg);                             \
  CG_HAND("s"(sg.shift), "s"(sg.row0), "s"(sg.row1), "s"(sg.blk0), "s"(sg.blk1),       \
          "s"(sg.rpb), "s"(sg.near_zero), ##__VA_ARGS__);                              \
  CgSeg *S = a.seg;                                                                    \
  if (multi_) {                                                                        \
    S += ((TBSLA_CONST int *)a.block_seg)[b];                                          \
    sg = cg_part((TBSLA_CONST CgSeg *)S);                                              \
  }
#define CG_HAND(...) asm volatile("" : : __VA_ARGS__)

struct CgPart {
  double stop, near_zero, rnorm0;
  int iters, shift, true_res, stop_par, done;
  int row0, row1, blk0, blk1, rpb, ent0, left;
};

__device__ inline CgPart cg_part(TBSLA_CONST CgSeg *c) {
  return CgPart{c->stop, c->near_zero, c->rnorm0, c->iters, c->shift, c->true_res, c->stop_par, c->done,
                c->row0, c->row1, c->blk0, c->blk1, c->rpb, c->ent0, c->left};
}

// the block's other fields
__device__ inline CgArgs cg_bind(const CgArgs *pa) {
  TBSLA_CONST CgArgs *c = (TBSLA_CONST CgArgs *)pa;
  CgArgs a;
  a.rowptr = arg(&c->rowptr);
  a.colidx = arg(&c->colidx);
  a.val64 = arg(&c->val64);
  a.val32 = arg(&c->val32);
  a.f_col = c->f_col;
  a.g_rp = arg(&c->g_rp);
  a.g_ci = arg(&c->g_ci);
  a.g_v64 = arg(&c->g_v64);
  a.g_v32 = arg(&c->g_v32);
  a.t_rp = arg(&c->t_rp);
  a.t_ci = arg(&c->t_ci);
  a.t_v64 = arg(&c->t_v64);
  a.t_v32 = arg(&c->t_v32);
  a.dinv = arg(&c->dinv);
  a.gdoff = arg(&c->gdoff);
  a.gd64 = arg(&c->gd64);
  a.gd32 = arg(&c->gd32);
  a.gndiag = c->gndiag;
  a.b = arg(&c->b);
  a.x = arg(&c->x);
  for (int i = 0; i < 2; i++) {
    a.r[i] = arg(&c->r[i]);
    a.p[i] = arg(&c->p[i]);
    a.prr[i] = arg(&c->prr[i]);
    a.prz[i] = arg(&c->prz[i]);
  }
  a.z = arg(&c->z);
  a.ap = arg(&c->ap);
  a.ax = arg(&c->ax);
  a.t64 = arg(&c->t64);
  a.t32 = arg(&c->t32);
  a.ppap = arg(&c->ppap);
  a.seg = arg(&c->seg);
  a.com = arg(&c->com);
  a.block_seg = arg(&c->block_seg);
  a.verify = c->verify;
  a.stall_window = c->stall_window;
  a.a_nnz = c->a_nnz;
  a.g_nnz = c->g_nnz;
  a.doff = arg(&c->doff);
  a.dv64 = arg(&c->dv64);
  a.dv32 = arg(&c->dv32);
  a.ndiag = c->ndiag;
  a.ncol = c->ncol;
  return a;
}

// Sums of a system's workgroup partials are taken in one fixed order:
// thread k adds partials k, k+256, ... in order; waves reduce by xor
// butterflies (every lane gets the same bits); wave totals are added in wave
// order.
// Up to three such sums in one pass (one chain of loads); results in every
// thread.  Every workgroup of a system takes them from the same partials in
// the same order, so all hold bitwise-equal totals.
__device__ void seg_sums(const double *__restrict__ p0, const double *__restrict__ p1,
                         const double *__restrict__ p2, int np, int b0, int b1, double *out) {
  __shared__ double lds[3][kBlock / kWave];
  double v[3] = {0.0, 0.0, 0.0};
  for (int i = b0 + (int)threadIdx.x; i < b1; i += kBlock) {
    v[0] += p0[i];
    if (np > 1) v[1] += p1[i];
    if (np > 2) v[2] += p2[i];
  }
#pragma unroll
  for (int k = 0; k < 3; k++) v[k] = group_sum<kWave>(v[k]);
  __syncthreads();
  if ((threadIdx.x & (kWave - 1)) == 0)
#pragma unroll
    for (int k = 0; k < 3; k++) lds[k][threadIdx.x / kWave] = v[k];
  __syncthreads();
#pragma unroll
  for (int k = 0; k < 3; k++) {
    double t = lds[k][0];
#pragma unroll
    for (int w = 1; w < kBlock / kWave; w++) t += lds[k][w];
    out[k] = t;
  }
}

// workgroup sum, result valid in thread 0
__device__ double wg_sum(double v, double *lds) {
  v = group_sum<kWave>(v);
  __syncthreads();
  if ((threadIdx.x & (kWave - 1)) == 0) lds[threadIdx.x / kWave] = v;
  __syncthreads();
  double t = lds[0];
#pragma unroll
  for (int w = 1; w < kBlock / kWave; w++) t += lds[w];
  return t;
}

// The system's done flag as one value for the whole workgroup (another
// workgroup of the same kernel may be writing it).
__device__ int seg_flag(const CgSeg *S, int *s_flag) {
  if (threadIdx.x == 0) *s_flag = __atomic_load_n(&S->done, __ATOMIC_RELAXED);
  __syncthreads();
  return *s_flag;
}

template <int L>
__device__ inline float lane_sum(float v) {
#pragma unroll
  for (int off = L / 2; off > 0; off >>= 1) v += __shfl_xor(v, off, L);
  return v;
}
template <int L>
__device__ inline double lane_sum(double v) {
#pragma unroll
  for (int off = L / 2; off > 0; off >>= 1) v += __shfl_xor(v, off, L);
  return v;
}

// Operands of the first row a thread handles, loaded before the reductions
// they do not depend on.  Entries j = beg + lane + k L (k < P) of the row, in
// the order the row loop visits them; the arithmetic on them is the loop's,
// so results are bitwise those of the plain loop.
template <int P, typename V>
struct RowPrefetch {
  int beg, end;
  int col[P];
  V v[P];
  double s[P], t[P];
};

// One row of A as a group of L lanes reads it in K1: 8 entries per lane.  L = 1:
// the row's first 8, one by one (short rows).  L >= 2: two 16-byte loads of
// column indices (and 16 or 32 bytes of values), 4 entries each, from the row's
// first entry rounded down to a multiple of 4 of its system's entries (so that a
// system is summed alike alone and in a batch, where its quads may lie on any
// 4-byte boundary); lane l's quads are l and l + L, so a row's lines are read
// whole by one instruction instead of 4 L bytes at a time (but for the lines that
// two rows share: no nontemporal hint, which had them fetched twice; 96 systems
// of 85 M entries, mixed, K1b: 252 -> 230 us).  Slots outside the row
// have column 0 of the block and are not summed.  Longer rows continue with the
// entries from `rest` on.  Entry positions are unsigned: slots reach some hundred
// past the row, and a block may end at entry 2^31 - 2.
template <int L, typename V>
struct CgRow {
  static constexpr int P = 8;
  int beg, end, first;
  int col[P];
  V v[P];

  __device__ inline void extent(const int *__restrict__ rowptr, int row, int ent0) {
    beg = rowptr[row];
    end = rowptr[row + 1];
    first = L == 1 ? beg : beg - ((beg - ent0) & 3);
  }
  __device__ inline unsigned at(int lane, int k) const {
    return L == 1 ? (unsigned)beg + k : (unsigned)first + (4 * (lane + (k >> 2) * L) + (k & 3));
  }
  __device__ inline bool in(int lane, int k) const {
    const unsigned e = at(lane, k);
    return e >= (unsigned)beg && e < (unsigned)end;
  }
  __device__ inline unsigned rest(int lane) const {
    return L == 1 ? (unsigned)beg + P : (unsigned)first + 4 * (lane + 2 * L);
  }
  // the entries, clamped into the arrays (the last quad may end up to three
  // entries after the last one: device_alloc's blocks have room for them)
  __device__ inline void load(const int *__restrict__ ci, const V *__restrict__ va, int nnz,
                              int f_col, int lane) {
    if constexpr (L == 1) {
#pragma unroll
      for (int k = 0; k < P; k++) {
        const int j = (int)min(at(lane, k), (unsigned)nnz - 1);
        col[k] = ci[j];
        v[k] = va[j];
      }
    } else {
#pragma unroll
      for (int h = 0; h < 2; h++) quad(ci, va, (int)min(at(lane, 4 * h), (unsigned)nnz - 1), 4 * h);
    }
#pragma unroll
    for (int k = 0; k < P; k++) col[k] = in(lane, k) ? col[k] - f_col : 0;
  }
  __device__ inline void quad(const int *__restrict__ ci, const V *__restrict__ va, int j, int k) {
    typedef int vi __attribute__((ext_vector_type(4), aligned(4)));
    constexpr int W = 16 / sizeof(V);  // values per 16 bytes
    typedef V vv __attribute__((ext_vector_type(W), aligned(sizeof(V))));
    const vi *pc = reinterpret_cast<const vi *>(ci + j);
    const vi c = *pc;
#pragma unroll
    for (int q = 0; q < 4; q++) col[k + q] = c[q];
#pragma unroll
    for (int q = 0; q < 4; q += W) {
      const vv *pv = reinterpret_cast<const vv *>(va + j + q);
      const vv x = *pv;
#pragma unroll
      for (int w = 0; w < W; w++) v[k + q + w] = x[w];
    }
  }
};

// A system's workgroup partials as loaded by seg_issue (raw, unmasked) and
// summed by seg_finish in seg_sums' order.  Loads complete in issue order, so
// K1 and K2 issue them between their row loads and the dependent gathers:
// the reductions then wait for the partials only, and the gathers stay in
// flight through the cross-lane and LDS work.
constexpr int kPartLoads = kMaxBlocksPerSystem / kBlock;
static_assert(kMaxBlocksPerSystem % kBlock == 0, "partials per thread");

struct SegLoad {
  double v[3][kPartLoads];
};

struct SegShared {
  double part[3][kBlock / kWave];
  int flag;
};

__device__ inline void seg_issue(const double *__restrict__ p0, const double *__restrict__ p1,
                                 const double *__restrict__ p2, int np, int b0, int b1,
                                 SegLoad &l) {
#pragma unroll
  for (int k = 0; k < kPartLoads; k++) {
    const int i = min(b0 + (int)threadIdx.x + k * kBlock, b1 - 1);
    l.v[0][k] = p0[i];
    if (np > 1) l.v[1][k] = p1[i];
    if (np > 2) l.v[2][k] = p2[i];
  }
}

// The sums (results in every thread) and the system's done flag as one value
// for the workgroup; the sums are valid only when the flag is kRunning.
__device__ inline int seg_finish(int flag, const SegLoad &l, int np, int b0, int b1,
                                 SegShared &sh, double *out) {
  double v[3] = {0.0, 0.0, 0.0};
#pragma unroll
  for (int k = 0; k < kPartLoads; k++) {
    if (b0 + (int)threadIdx.x + k * kBlock < b1) {
      v[0] += l.v[0][k];
      if (np > 1) v[1] += l.v[1][k];
      if (np > 2) v[2] += l.v[2][k];
    }
  }
#pragma unroll
  for (int k = 0; k < 3; k++)
    if (k < np) v[k] = group_sum<kWave>(v[k]);
  if ((threadIdx.x & (kWave - 1)) == 0)
#pragma unroll
    for (int k = 0; k < 3; k++)
      if (k < np) sh.part[k][threadIdx.x / kWave] = v[k];
  if (threadIdx.x == 0) sh.flag = flag;
  __syncthreads();
  const int f = sh.flag;
  if (f != kRunning) return f;
#pragma unroll
  for (int k = 0; k < 3; k++) {
    if (k < np) {
      double t = sh.part[k][0];
#pragma unroll
      for (int w = 1; w < kBlock / kWave; w++) t += sh.part[k][w];
      out[k] = t;
    }
  }
  return f;
}

// The convergence test of the previous iteration (CG.cpp:66-72) on
// |r| = sqrt(rr), made alike by every workgroup of the system from the same
// sums; the system's first workgroup records the outcome.  Returns it.
__device__ inline int k1_test(const CgArgs &a, CgSeg *S, const CgPart &sg, int b, int par,
                              double rz_new, double rr, int check_only) {
  const double rn = sqrt(rr);
  int fin = kRunning;
  if (rn < sg.stop || rn == 0.0)
    fin = (a.verify && !sg.true_res) ? kPending : kConverged;
  else if (!(rz_new > 0.0) || !isfinite(rz_new) || !isfinite(rr))
    fin = kBreakdown;
  else if (!check_only && a.stall_window > 0 && sg.iters >= a.stall_window && rn >= sg.rnorm0)
    fin = kBreakdown;
  if (b == sg.blk0 && threadIdx.x == 0) {
    S->rnorm = rn;
    if (S == a.seg) a.com->ratio = rn / sg.stop;
    if (fin != kRunning) {
      S->stop_par = par;
      S->t_done = wall_clock64();
      __atomic_store_n(&S->done, fin, __ATOMIC_RELAXED);
      atomicAdd(fin == kPending ? &a.com->npending : &a.com->ndone, 1);
    } else if (check_only) {
      S->iters += 1;  // the count K2 would have made
    }
  }
  return fin;
}

// K1.  check: apply the convergence test of the previous iteration first
// (the count it++ of a passed test is made by K2, which no K1 workgroup
// races with).  check_only: the final test after the last iteration.
template <int L, bool MIX, bool ZBUF>
__global__ __launch_bounds__(kBlock) void k_cg_spmv_p(CG_ARGS, int par_g, int check,
                                                      int check_only) {
  TBSLA_NO_FMA
  CG_BIND;
  typedef typename std::conditional<MIX, float, double>::type V;
  typedef CgRow<L, V> Row;
  constexpr int P = Row::P;
  constexpr int NP = ZBUF ? 3 : 2;
  __shared__ double lds[kBlock / kWave];
  __shared__ SegShared sh;
  const int b = cg_block(multi_);
  CG_SYSTEM(b, "s"(a.p[0]), "s"(a.p[1]), "s"(a.prz[0]), "s"(a.prz[1]), "s"(ZBUF ? a.prr[0] : a.r[0]),
            "s"(ZBUF ? a.prr[1] : a.r[1]), "s"(a.z), "s"(a.ap), "s"(a.ppap),
            "s"(a.rowptr), "s"(a.colidx),
            "s"(MIX ? (const void *)a.val32 : (const void *)a.val64), "s"(a.a_nnz), "s"(a.f_col),
            "s"(sg.stop), "s"(sg.iters), "s"(sg.true_res), "s"(sg.rnorm0), "s"(sg.ent0));
  const int par = (par_g ^ sg.shift) & 1;
  const int b0 = sg.blk0, b1 = sg.blk1;
  const int r0 = sg.row0 + (b - b0) * sg.rpb;
  const int r1 = min(sg.row1, r0 + sg.rpb);
  const int lane = threadIdx.x & (L - 1);
  const double *zv = ZBUF ? a.z : CG_AT(r, par);
  const double *po = CG_AT(p, par);
  const V *val = MIX ? (const V *)a.val32 : (const V *)a.val64;
  const int row_first = r0 + (int)threadIdx.x / L;
  const int rowc = min(row_first, r1 - 1);
  // row extent and own entries, then the row's first entries, then the
  // partials, then the gathers.  No branches between them: a join would make
  // the partials' wait cover the gathers.
  Row f;
  double fs[P], ft[P];
  f.extent(a.rowptr, rowc, sg.ent0);
  const double own_z = zv[rowc], own_p = po[rowc];
  f.load(a.colidx, val, a.a_nnz, a.f_col, lane);
  const int flag = __atomic_load_n(&S->done, __ATOMIC_RELAXED);
  SegLoad sl;
  seg_issue(CG_AT(prz, par ^ 1), CG_AT(prz, par), CG_AT(prr, par ^ 1), NP, b0, b1, sl);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int k = 0; k < P; k++) {
    fs[k] = zv[f.col[k]];
    ft[k] = po[f.col[k]];
  }
  __builtin_amdgcn_sched_barrier(0);  // keep the loads above issued in this order
  double t[3];
  if (seg_finish(flag, sl, NP, b0, b1, sh, t) != kRunning) return;
  const double rz_new = t[0], rz_old = t[1];
  const double rr = ZBUF ? t[2] : rz_new;
  if (check) {
    const int fin = k1_test(a, S, sg, b, par, rz_new, rr, check_only);
    if (fin != kRunning || check_only) return;
  }
  const double beta = rz_new / fmax(rz_old, sg.near_zero);
  double *pn = CG_AT(p, par ^ 1);
  double pap = 0.0;
  constexpr int PASS = kBlock / L;
  // the sum of a loaded row, the entries past its 8 per lane from memory
  auto finish = [&](const Row &w, const double (&sv)[P], const double (&tv)[P], int row, double oz,
                    double op) {
    V acc = 0;
    auto term = [&](V av, double s, double t) {
      const double v = s + beta * t;
      if (MIX) acc = fmaf((float)av, (float)v, (float)acc);
      else acc = fma((double)av, v, (double)acc);
    };
#pragma unroll
    for (int k = 0; k < P; k++)
      if (w.in(lane, k)) term(w.v[k], sv[k], tv[k]);
    constexpr int Q = L == 1 ? 1 : 4;  // consecutive entries of a lane
    for (unsigned j = w.rest(lane); j < (unsigned)w.end; j += Q * L)
#pragma unroll
      for (int q = 0; q < Q; q++)
        if (j + q < (unsigned)w.end) {
          const int c = a.colidx[j + q] - a.f_col;
          term(val[j + q], zv[c], po[c]);
        }
    acc = lane_sum<L>(acc);
    const double own = oz + beta * op;
    if (lane == 0) {
      pn[row] = own;
      a.ap[row] = (double)acc;
      pap += own * (double)acc;
    }
  };
  if (row_first < r1) finish(f, fs, ft, row_first, own_z, own_p);
  // the later rows two at a time: both rows' extents, then entries, then
  // gathers are issued before either is summed
  constexpr int R2 = 2;
  for (int row = row_first + PASS; row < r1; row += R2 * PASS) {
    Row g[R2];
    double gs[R2][P], gt[R2][P], oz[R2], op[R2];
    int rw[R2];
#pragma unroll
    for (int r = 0; r < R2; r++) {
      rw[r] = min(row + r * PASS, r1 - 1);
      g[r].extent(a.rowptr, rw[r], sg.ent0);
      oz[r] = zv[rw[r]];
      op[r] = po[rw[r]];
    }
#pragma unroll
    for (int r = 0; r < R2; r++) g[r].load(a.colidx, val, a.a_nnz, a.f_col, lane);
#pragma unroll
    for (int r = 0; r < R2; r++)
#pragma unroll
      for (int k = 0; k < P; k++) {
        gs[r][k] = zv[g[r].col[k]];
        gt[r][k] = po[g[r].col[k]];
      }
#pragma unroll
    for (int r = 0; r < R2; r++)
      if (row + r * PASS < r1) finish(g[r], gs[r], gt[r], rw[r], oz[r], op[r]);
  }
  pap = wg_sum(pap, lds);
  if (threadIdx.x == 0) a.ppap[b] = pap;
}

// K1 in two passes (for matrices whose gathers miss the caches: each
// gathered entry then pulls one line of p' instead of one of z and one of
// p).  First pass: the partials, the convergence test and beta exactly as
// k_cg_spmv_p, then p' = z + beta p for the workgroup's rows.
template <bool ZBUF>
__global__ __launch_bounds__(kBlock) void k_cg_pnew(CG_ARGS, int par_g, int check,
                                                    int check_only) {
  TBSLA_NO_FMA
  CG_BIND;
  constexpr int NP = ZBUF ? 3 : 2;
  __shared__ SegShared sh;
  const int b = cg_block(multi_);
  CG_SYSTEM(b);
  if (multi_ && sg.left) return;  // finished before the last K2
  const int par = (par_g ^ sg.shift) & 1;
  const int b0 = sg.blk0, b1 = sg.blk1;
  const int r0 = sg.row0 + (b - b0) * sg.rpb;
  const int r1 = min(sg.row1, r0 + sg.rpb);
  const double *zv = ZBUF ? a.z : CG_AT(r, par);
  const double *po = CG_AT(p, par);
  const int flag = __atomic_load_n(&S->done, __ATOMIC_RELAXED);
  SegLoad sl;
  seg_issue(CG_AT(prz, par ^ 1), CG_AT(prz, par), CG_AT(prr, par ^ 1), NP, b0, b1, sl);
  double t[3];
  if (seg_finish(flag, sl, NP, b0, b1, sh, t) != kRunning) return;
  const double rz_new = t[0], rz_old = t[1];
  const double rr = ZBUF ? t[2] : rz_new;
  if (check) {
    const int fin = k1_test(a, S, sg, b, par, rz_new, rr, check_only);
    if (fin != kRunning || check_only) return;
  }
  const double beta = rz_new / fmax(rz_old, sg.near_zero);
  double *pn = CG_AT(p, par ^ 1);
  for (int row = r0 + (int)threadIdx.x; row < r1; row += 2 * kBlock) {
    const int row2 = row + kBlock;
    const double z0 = zv[row], p0 = po[row];
    const double z1 = row2 < r1 ? zv[row2] : 0.0, p1 = row2 < r1 ? po[row2] : 0.0;
    pn[row] = z0 + beta * p0;
    if (row2 < r1) pn[row2] = z1 + beta * p1;
  }
}

// Second pass: Ap' and the partials of p'.Ap' for the rows of systems still
// running (the first pass made this iteration's test), the row schedule of
// k_cg_spmv_p gathering p' alone.  Every value is the one k_cg_spmv_p
// computes: p' is formed by the same expression.
template <int L, bool MIX>
__global__ __launch_bounds__(kBlock) void k_cg_ap(CG_ARGS, int par_g) {
  TBSLA_NO_FMA  // p'.Ap' partials added as k_cg_spmv_p adds them
  CG_BIND;
  typedef typename std::conditional<MIX, float, double>::type V;
  typedef CgRow<L, V> Row;
  constexpr int P = Row::P;
  __shared__ double lds[kBlock / kWave];
  const int b = cg_block(multi_);
  CG_SYSTEM(b);
  if (multi_ && sg.done != kRunning) return;
  if (__atomic_load_n(&S->done, __ATOMIC_RELAXED) != kRunning) return;
  const int par = (par_g ^ sg.shift) & 1;
  const int b0 = sg.blk0;
  const int r0 = sg.row0 + (b - b0) * sg.rpb;
  const int r1 = min(sg.row1, r0 + sg.rpb);
  const int lane = threadIdx.x & (L - 1);
  const double *pn = CG_AT(p, par ^ 1);
  const V *val = MIX ? (const V *)a.val32 : (const V *)a.val64;
  constexpr int PASS = kBlock / L;
  constexpr int R2 = 2;
  double pap = 0.0;
  // rows two at a time: both rows' extents, then entries, then gathers are
  // issued before either is summed
  for (int row = r0 + (int)threadIdx.x / L; row < r1; row += R2 * PASS) {
    Row w[R2];
    int rw[R2];
    double g[R2][P], own[R2];
#pragma unroll
    for (int r = 0; r < R2; r++) {
      rw[r] = min(row + r * PASS, r1 - 1);
      w[r].extent(a.rowptr, rw[r], sg.ent0);
      own[r] = pn[rw[r]];
    }
#pragma unroll
    for (int r = 0; r < R2; r++) w[r].load(a.colidx, val, a.a_nnz, a.f_col, lane);
#pragma unroll
    for (int r = 0; r < R2; r++)
#pragma unroll
      for (int k = 0; k < P; k++) g[r][k] = pn[w[r].col[k]];
#pragma unroll
    for (int r = 0; r < R2; r++) {
      if (row + r * PASS >= r1) break;
      V acc = 0;
      auto term = [&](V av, double x) {
        if (MIX) acc = fmaf((float)av, (float)x, (float)acc);
        else acc = fma((double)av, x, (double)acc);
      };
#pragma unroll
      for (int k = 0; k < P; k++)
        if (w[r].in(lane, k)) term(w[r].v[k], g[r][k]);
      constexpr int Q = L == 1 ? 1 : 4;
      for (unsigned j = w[r].rest(lane); j < (unsigned)w[r].end; j += Q * L)
#pragma unroll
        for (int q = 0; q < Q; q++)
          if (j + q < (unsigned)w[r].end) term(val[j + q], pn[a.colidx[j + q] - a.f_col]);
      acc = lane_sum<L>(acc);
      if (lane == 0) {
        a.ap[rw[r]] = (double)acc;
        pap += own[r] * (double)acc;
      }
    }
  }
  pap = wg_sum(pap, lds);
  if (threadIdx.x == 0) a.ppap[b] = pap;
}

// base[i] by a 32-bit byte offset (one register of address beside the uniform
// base): arrays below 4 GiB
template <typename T>
__device__ inline T ld32(const T *__restrict__ base, unsigned i) {
  return *reinterpret_cast<const T *>(reinterpret_cast<const char *>(base) +
                                      (size_t)(i * (unsigned)sizeof(T)));
}
// the same, or by a 64-bit one where an array may be larger
template <bool WIDE, typename T>
__device__ inline T ldi(const T *__restrict__ base, long long i) {
  if constexpr (WIDE) return base[i];
  else return ld32(base, (unsigned)i);
}

// K1 on A in the diagonal layout: the same steps as k_cg_spmv_p (the
// partials of the previous iteration, the convergence test, beta), then per
// row p' = z + beta p and (A p')_row = sum over the stored diagonals
// (ascending offset, zero slots skipped) of A's slot times p' at the slot's
// column.  KD 3, 5, 7: exactly that many diagonals (the stencils of one to three
// dimensions) in arrays below 4 GiB, a row's loads all in flight; the first row's
// loads (which need no sum) go out before the partials', so the reductions and
// the test run under them.  KD 0: any number of diagonals and any size, eight
// diagonals at a time.  Bound by latency (flag and partials, then a trip per row)
// at 64^3, FP64: 9.7 -> 8.0 us an iteration (KD and the early loads, 0.9; global
// loads for flat ones, 0.8); 10^6 rows, mixed: 19.4 -> 17.1.  Two rows in flight per
// thread were slower (8.3 and 18.6: 204 registers, half the wavefronts).
// SYM: the layout's values are symmetric bit for bit, and a slot below the main
// diagonal is read as its mirror image, from lines that other rows read anyway:
// half the values from memory (64^3, FP64: 7.8 -> 6.9 us; 10^6 rows, mixed: as
// before, 15.1).
template <bool MIX, bool ZBUF, int KD, bool SYM>
__global__ __launch_bounds__(kBlock) void k_cg_spmv_dia(CG_ARGS, int par_g, int check,
                                                        int check_only) {
  TBSLA_NO_FMA
  CG_BIND;
  typedef typename std::conditional<MIX, float, double>::type V;
  constexpr int NP = ZBUF ? 3 : 2;
  constexpr int U = KD > 0 ? KD : 8;
  __shared__ double lds[kBlock / kWave];
  __shared__ SegShared sh;
  const int b = cg_block(multi_);
  CG_SYSTEM(b, "s"(a.p[0]), "s"(a.p[1]), "s"(a.prz[0]), "s"(a.prz[1]), "s"(ZBUF ? a.prr[0] : a.r[0]),
            "s"(ZBUF ? a.prr[1] : a.r[1]), "s"(a.z), "s"(a.ap),
            "s"(MIX ? (const void *)a.dv32 : (const void *)a.dv64), "s"(a.ncol), "s"(a.ppap),
            "s"(sg.stop), "s"(sg.iters), "s"(sg.true_res), "s"(sg.rnorm0), "s"(CG_OFF(doff8, 0)),
            "s"(CG_OFF(doff8, 1)), "s"(CG_OFF(doff8, 2)), "s"(CG_OFF(doff8, 3)),
            "s"(CG_OFF(doff8, 4)), "s"(CG_OFF(doff8, 5)), "s"(CG_OFF(doff8, 6)));
  const int par = (par_g ^ sg.shift) & 1;
  const int b0 = sg.blk0, b1 = sg.blk1;
  const int r0 = sg.row0 + (b - b0) * sg.rpb;
  const int r1 = min(sg.row1, r0 + sg.rpb);
  const double *zv = ZBUF ? a.z : CG_AT(r, par);
  const double *po = CG_AT(p, par);
  const V *dv = MIX ? (const V *)a.dv32 : (const V *)a.dv64;
  const int row_first = r0 + (int)threadIdx.x;
  struct Row {
    V v[U];
    double z[U], p[U], oz, op;
  } f;
  // slots k0 .. k0 + U - 1 of one row (past the last diagonal: the last one
  // again, not used)
  auto load = [&](int row, int k0, Row &w) {
    if constexpr (KD > 0) {
      const unsigned at = (unsigned)dia_at(row, 0, KD);
#pragma unroll
      for (int i = 0; i < U; i++) {
        const unsigned c = (unsigned)min(max(row + CG_OFF(doff8, i), 0), a.ncol - 1);
        if (SYM && i < KD / 2)  // its mirror image's (unused where there is none)
          w.v[i] = ld32(dv, c / kWave * (kWave * KD) + (KD - 1 - i) * kWave + c % kWave);
        else
          w.v[i] = ld32(dv, at + i * kWave);
        w.z[i] = ld32(zv, c);
        w.p[i] = ld32(po, c);
      }
      w.oz = ld32(zv, (unsigned)row);
      w.op = ld32(po, (unsigned)row);
      return;
    }
#pragma unroll
    for (int i = 0; i < U; i++) {
      const int kk = min(k0 + i, a.ndiag - 1);
      const int c = min(max(row + a.doff[kk], 0), a.ncol - 1);
      w.v[i] = dv[dia_at(row, kk, a.ndiag)];
      w.z[i] = zv[c];
      w.p[i] = po[c];
    }
  };
  if (KD > 0) {
    load(min(row_first, r1 - 1), 0, f);
    __builtin_amdgcn_sched_barrier(0);
  }
  const int flag = __atomic_load_n(&S->done, __ATOMIC_RELAXED);
  SegLoad sl;
  seg_issue(CG_AT(prz, par ^ 1), CG_AT(prz, par), CG_AT(prr, par ^ 1), NP, b0, b1, sl);
  __builtin_amdgcn_sched_barrier(0);  // keep the loads above issued in this order
  double t[3];
  if (seg_finish(flag, sl, NP, b0, b1, sh, t) != kRunning) return;
  const double rz_new = t[0], rz_old = t[1];
  const double rr = ZBUF ? t[2] : rz_new;
  if (check) {
    const int fin = k1_test(a, S, sg, b, par, rz_new, rr, check_only);
    if (fin != kRunning || check_only) return;
  }
  const double beta = rz_new / fmax(rz_old, sg.near_zero);
  double *pn = CG_AT(p, par ^ 1);
  double pap = 0.0;
  auto add = [&](const Row &w, int row, int k0, V acc) {
#pragma unroll
    for (int i = 0; i < U; i++) {
      const bool none = SYM && i < KD / 2 && row + CG_OFF(doff8, i) < 0;
      if ((KD > 0 || k0 + i < a.ndiag) && !none && w.v[i] != (V)0) {
        const double pc = w.z[i] + beta * w.p[i];
        if (MIX) acc = fmaf((float)w.v[i], (float)pc, (float)acc);
        else acc = fma((double)w.v[i], pc, (double)acc);
      }
    }
    return acc;
  };
  auto store = [&](int row, double own, V acc) {
    pn[row] = own;
    a.ap[row] = (double)acc;
    pap += own * (double)acc;
  };
  if (KD > 0) {
    for (int row = row_first; row < r1; row += kBlock) {
      if (row != row_first) load(row, 0, f);
      store(row, f.oz + beta * f.op, add(f, row, 0, (V)0));
    }
  } else {
    for (int row = row_first; row < r1; row += kBlock) {
      V acc = 0;
      for (int k = 0; k < a.ndiag; k += U) {
        load(row, k, f);
        acc = add(f, row, k, acc);
      }
      store(row, zv[row] + beta * po[row], acc);
    }
  }
  pap = wg_sum(pap, lds);
  if (threadIdx.x == 0) a.ppap[b] = pap;
}

// K2.  PRE: 0 none, 1 Jacobi, 2 M = G G^T (t = G^T r' here from G^T's CSR
// rows, z = G t in K3).
template <int PRE, bool MIX>
__global__ __launch_bounds__(kBlock) void k_cg_update(CG_ARGS, int par_g, int count) {
  TBSLA_NO_FMA
  CG_BIND;
  typedef typename std::conditional<MIX, float, double>::type V;
  constexpr int P = 4;
  __shared__ double lds[kBlock / kWave];
  __shared__ SegShared sh;
  const int b = cg_block(multi_);
  CG_SYSTEM(b, "s"(a.p[0]), "s"(a.p[1]), "s"(a.prz[0]), "s"(a.prz[1]), "s"(a.prr[0]),
            "s"(a.prr[1]), "s"(a.r[0]), "s"(a.r[1]), "s"(a.x), "s"(a.ap), "s"(a.ppap),
            "s"(a.dinv));
  if (multi_ && sg.done != kRunning) {  // finished before this launch
    if (b == sg.blk0 && threadIdx.x == 0) S->left = 1;
    return;
  }
  const int par = (par_g ^ sg.shift) & 1;
  const int b0 = sg.blk0, b1 = sg.blk1;
  const double *rc = CG_AT(r, par);
  double *rn = CG_AT(r, par ^ 1);
  const double *pn = CG_AT(p, par ^ 1);
  const V *tv = MIX ? (const V *)a.t_v32 : (const V *)a.t_v64;
  const int r0 = sg.row0 + (b - b0) * sg.rpb;
  const int r1 = min(sg.row1, r0 + sg.rpb);
  const int row_first = r0 + (int)threadIdx.x;
  const int rowc = min(row_first, r1 - 1);
  // the first row's operands (see RowPrefetch), then the partials, then the
  // gathers of t = G^T r'
  const double fx = a.x[rowc], fp = pn[rowc], fr = rc[rowc], fap = a.ap[rowc];
  const double fd = PRE == 1 ? a.dinv[rowc] : 0.0;
  // and, without a factor, the second row's
  const int row2 = min(row_first + kBlock, r1 - 1);
  double fx2 = 0.0, fp2 = 0.0, fr2 = 0.0, fap2 = 0.0, fd2 = 0.0;
  if (PRE != 2) {
    fx2 = a.x[row2];
    fp2 = pn[row2];
    fr2 = rc[row2];
    fap2 = a.ap[row2];
    if (PRE == 1) fd2 = a.dinv[row2];
  }
  RowPrefetch<P, V> f;
  f.beg = f.end = 0;
  if (PRE == 2) {
    f.beg = a.t_rp[rowc];
    f.end = a.t_rp[rowc + 1];
#pragma unroll
    for (int k = 0; k < P; k++) {
      const int j = min(f.beg + k, a.g_nnz - 1);
      f.col[k] = a.t_ci[j];
      f.v[k] = tv[j];
    }
  }
  const int flag = __atomic_load_n(&S->done, __ATOMIC_RELAXED);
  SegLoad sl;
  seg_issue(CG_AT(prz, par ^ 1), a.ppap, nullptr, 2, b0, b1, sl);
  __builtin_amdgcn_sched_barrier(0);
  if (PRE == 2) {
#pragma unroll
    for (int k = 0; k < P; k++) {
      f.s[k] = rc[f.col[k] - a.f_col];
      f.t[k] = a.ap[f.col[k] - a.f_col];
    }
  }
  __builtin_amdgcn_sched_barrier(0);  // keep the loads above issued in this order
  double t[3];
  if (seg_finish(flag, sl, 2, b0, b1, sh, t) != kRunning) return;
  const double rz = t[0], pap = t[1];
  const double alpha = rz / fmax(pap, sg.near_zero);
  double rr = 0.0, rzp = 0.0;
  // PRE 2: the first row, then the later rows two at a time (each pair's
  // loads issued before either is updated; sums in row order)
  const int row_end = PRE == 2 ? min(r1, row_first + 1) : r1;
  for (int row = row_first; row < row_end; row += kBlock) {
    const bool first = row == row_first, second = PRE != 2 && row == row_first + kBlock;
    const double xv = first ? fx : second ? fx2 : a.x[row];
    const double pv = first ? fp : second ? fp2 : pn[row];
    const double rv = first ? fr : second ? fr2 : rc[row];
    const double apv = first ? fap : second ? fap2 : a.ap[row];
    a.x[row] = xv + alpha * pv;
    const double ri = rv + (-alpha) * apv;
    rn[row] = ri;
    rr += ri * ri;
    if (PRE == 1) {
      const double zi = ri * (first ? fd : second ? fd2 : a.dinv[row]);
      a.z[row] = zi;
      rzp += ri * zi;
    }
    if (PRE == 2) {
      // t = G^T r' with r'_c = r_c - alpha Ap_c computed as above
      V acc = 0;
#pragma unroll
      for (int k = 0; k < P; k++) {
        if (f.beg + k < f.end) {
          const double rcv = f.s[k] + (-alpha) * f.t[k];
          if (MIX) acc = fmaf((float)f.v[k], (float)rcv, (float)acc);
          else acc = fma((double)f.v[k], rcv, (double)acc);
        }
      }
      for (int j = f.beg + P; j < f.end; j++) {
        const int c = a.t_ci[j] - a.f_col;
        const double rcv = rc[c] + (-alpha) * a.ap[c];
        if (MIX) acc = fmaf((float)tv[j], (float)rcv, (float)acc);
        else acc = fma((double)tv[j], rcv, (double)acc);
      }
      if (MIX) a.t32[row] = (float)acc;
      else a.t64[row] = (double)acc;
    }
  }
  if (PRE == 2) {
    constexpr int R2 = 2;
    for (int row = row_first + kBlock; row < r1; row += R2 * kBlock) {
      RowPrefetch<P, V> g[R2];
      double xv[R2], pv[R2], rv[R2], apv[R2];
      int rw[R2];
#pragma unroll
      for (int r = 0; r < R2; r++) {
        rw[r] = min(row + r * kBlock, r1 - 1);
        xv[r] = a.x[rw[r]];
        pv[r] = pn[rw[r]];
        rv[r] = rc[rw[r]];
        apv[r] = a.ap[rw[r]];
        g[r].beg = a.t_rp[rw[r]];
        g[r].end = a.t_rp[rw[r] + 1];
      }
#pragma unroll
      for (int r = 0; r < R2; r++)
#pragma unroll
        for (int k = 0; k < P; k++) {
          const int j = min(g[r].beg + k, a.g_nnz - 1);
          g[r].col[k] = a.t_ci[j];
          g[r].v[k] = tv[j];
        }
#pragma unroll
      for (int r = 0; r < R2; r++)
#pragma unroll
        for (int k = 0; k < P; k++) {
          g[r].s[k] = rc[g[r].col[k] - a.f_col];
          g[r].t[k] = a.ap[g[r].col[k] - a.f_col];
        }
#pragma unroll
      for (int r = 0; r < R2; r++) {
        if (row + r * kBlock >= r1) break;
        a.x[rw[r]] = xv[r] + alpha * pv[r];
        const double ri = rv[r] + (-alpha) * apv[r];
        rn[rw[r]] = ri;
        rr += ri * ri;
        V acc = 0;
#pragma unroll
        for (int k = 0; k < P; k++) {
          if (g[r].beg + k < g[r].end) {
            const double rcv = g[r].s[k] + (-alpha) * g[r].t[k];
            if (MIX) acc = fmaf((float)g[r].v[k], (float)rcv, (float)acc);
            else acc = fma((double)g[r].v[k], rcv, (double)acc);
          }
        }
        for (int j = g[r].beg + P; j < g[r].end; j++) {
          const int c = a.t_ci[j] - a.f_col;
          const double rcv = rc[c] + (-alpha) * a.ap[c];
          if (MIX) acc = fmaf((float)tv[j], (float)rcv, (float)acc);
          else acc = fma((double)tv[j], rcv, (double)acc);
        }
        if (MIX) a.t32[rw[r]] = (float)acc;
        else a.t64[rw[r]] = (double)acc;
      }
    }
  }
  rr = wg_sum(rr, lds);
  if (PRE == 1) rzp = wg_sum(rzp, lds);
  if (threadIdx.x == 0) {
    CG_AT(prr, par)[b] = rr;
    if (PRE == 0) CG_AT(prz, par)[b] = rr;
    if (PRE == 1) CG_AT(prz, par)[b] = rzp;
    if (b == b0) {
      S->true_res = 0;
      if (count) S->iters += 1;  // the test K1 made on this iteration passed
    }
  }
}

// Slot k of G's diagonal layout for row `src` (0 outside the block): G^T's
// row i holds G_{i-o_k, i} at column i - o_k, i.e. slot (i - o_k, k).
template <typename V>
__device__ inline V gd_slot(const V *__restrict__ gd, long long src, int k, int ndg, long long n) {
  return src < n ? gd[dia_at(src, k, ndg)] : (V)0;
}

// K2 with M = G G^T and G on diagonals: t_i = sum over G^T's row i in
// ascending column (descending offset o_k <= 0) of G_{i-o_k, i} r'_{i-o_k},
// zero slots skipped -- the order and the products of K2's CSR form, so the
// two forms give bitwise the same iterates.  All of a row's loads are issued
// before it is updated, the first row's (which need no sum) before the partials';
// past G's last diagonal that one's again, not used (with a branch around each
// diagonal they took a trip to memory each: 10^6 rows, mixed, 17.3 -> 15.2 us).
template <bool MIX, int KD, bool WIDE>
__global__ __launch_bounds__(kBlock) void k_cg_update_gdia(CG_ARGS, int par_g, int count) {
  TBSLA_NO_FMA
  CG_BIND;
  typedef typename std::conditional<MIX, float, double>::type V;
  // KD: at most that many diagonals of G (4 or 8, chosen on the host)
  __shared__ double lds[kBlock / kWave];
  __shared__ SegShared sh;
  const int b = cg_block(multi_);
  CG_SYSTEM(b, "s"(a.p[0]), "s"(a.p[1]), "s"(a.prz[0]), "s"(a.prz[1]), "s"(a.prr[0]),
            "s"(a.prr[1]), "s"(a.r[0]), "s"(a.r[1]), "s"(a.x), "s"(a.ap), "s"(a.ppap),
            "s"(a.ncol), "s"(a.gndiag), "s"(MIX ? (const void *)a.gd32 : (const void *)a.gd64),
            "s"(CG_OFF(gdoff8, 0)), "s"(CG_OFF(gdoff8, 1)), "s"(CG_OFF(gdoff8, 2)),
            "s"(CG_OFF(gdoff8, 3)));
  if (multi_ && sg.done != kRunning) {  // finished before this launch
    if (b == sg.blk0 && threadIdx.x == 0) S->left = 1;
    return;
  }
  const int par = (par_g ^ sg.shift) & 1;
  const int b0 = sg.blk0, b1 = sg.blk1;
  const double *rc = CG_AT(r, par);
  double *rn = CG_AT(r, par ^ 1);
  const double *pn = CG_AT(p, par ^ 1);
  const V *gd = MIX ? (const V *)a.gd32 : (const V *)a.gd64;
  const int ndg = a.gndiag;
  const long long n = a.ncol;
  const int r0 = sg.row0 + (b - b0) * sg.rpb;
  const int r1 = min(sg.row1, r0 + sg.rpb);
  int off[KD];
#pragma unroll
  for (int k = 0; k < KD; k++) off[k] = CG_OFF(gdoff8, k);
  const int row_first = r0 + (int)threadIdx.x;
  double xv, pv, rv, apv, rs[KD], as[KD];
  V gv[KD];
  auto load = [&](int row) {
    xv = ldi<WIDE>(a.x, row);
    pv = ldi<WIDE>(pn, row);
    rv = ldi<WIDE>(rc, row);
    apv = ldi<WIDE>(a.ap, row);
#pragma unroll
    for (int k = 0; k < KD; k++) {
      const long long src = (long long)row - off[k];
      const long long sc = src < n ? src : row;
      gv[k] = ldi<WIDE>(gd, dia_at(sc, min(k, ndg - 1), ndg));
      rs[k] = ldi<WIDE>(rc, sc);
      as[k] = ldi<WIDE>(a.ap, sc);
    }
  };
  load(min(row_first, r1 - 1));
  __builtin_amdgcn_sched_barrier(0);
  const int flag = __atomic_load_n(&S->done, __ATOMIC_RELAXED);
  SegLoad sl;
  seg_issue(CG_AT(prz, par ^ 1), a.ppap, nullptr, 2, b0, b1, sl);
  __builtin_amdgcn_sched_barrier(0);
  double t[3];
  if (seg_finish(flag, sl, 2, b0, b1, sh, t) != kRunning) return;
  const double rz = t[0], pap = t[1];
  const double alpha = rz / fmax(pap, sg.near_zero);
  double rr = 0.0;
  for (int row = row_first; row < r1; row += kBlock) {
    if (row != row_first) load(row);
    a.x[row] = xv + alpha * pv;
    const double ri = rv + (-alpha) * apv;
    rn[row] = ri;
    rr += ri * ri;
    V acc = 0;
#pragma unroll
    for (int k = KD - 1; k >= 0; k--) {
      if (k < ndg && (long long)row - off[k] < n && gv[k] != (V)0) {
        const double rcv = rs[k] + (-alpha) * as[k];
        if (MIX) acc = fmaf((float)gv[k], (float)rcv, (float)acc);
        else acc = fma((double)gv[k], rcv, (double)acc);
      }
    }
    if (MIX) a.t32[row] = (float)acc;
    else a.t64[row] = (double)acc;
  }
  rr = wg_sum(rr, lds);
  if (threadIdx.x == 0) {
    CG_AT(prr, par)[b] = rr;
    if (b == b0) {
      S->true_res = 0;
      if (count) S->iters += 1;  // the test K1 made on this iteration passed
    }
  }
}

// Which systems a helper kernel serves: the running ones after an iteration
// (buffers of parity par^1 hold the new residual), the ones waiting for the
// true-residual test (their stop_par buffers), or every active one at start.
enum Mode { kAfterIter = 0, kVerify = 1, kStart = 2 };

// __device__ helper: does this workgroup take part, and with which buffers?
// rsel: the r buffer holding the current residual; psel: the r.r / r.z
// partial slot that describes it.
__device__ bool mode_select(const CgSeg *S, int mode, int par_g, int *s_flag, int *rsel) {
  const int f = seg_flag(S, s_flag);
  if (mode == kAfterIter) {
    if (f != kRunning) return false;
    *rsel = ((par_g ^ S->shift) & 1) ^ 1;
  } else if (mode == kVerify) {
    if (f != kPending) return false;
    *rsel = S->stop_par;
  } else {
    if (f == kInactive) return false;
    *rsel = 0;
  }
  return true;
}

// K3: z = G t; r.z partials.  Also the tail of a residual replacement.  The
// first row's entries of G and the values of t they pick are loaded before
// the done flag is shared (as in K1 and K2).
template <bool MIX>
__global__ __launch_bounds__(kBlock) void k_cg_gz(CG_ARGS, int par_g, int mode) {
  TBSLA_NO_FMA
  CG_BIND;
  typedef typename std::conditional<MIX, float, double>::type V;
  constexpr int P = 4;
  __shared__ double lds[kBlock / kWave];
  __shared__ int s_flag;
  const int b = cg_block(multi_);
  CG_SYSTEM(b);
  const int rsel = mode == kAfterIter ? ((par_g ^ sg.shift) & 1) ^ 1
                   : mode == kVerify  ? sg.stop_par
                                      : 0;
  const double *rc = CG_AT(r, rsel);
  const V *gv = MIX ? (const V *)a.g_v32 : (const V *)a.g_v64;
  const V *tv = MIX ? (const V *)a.t32 : (const V *)a.t64;
  const int b0 = sg.blk0;
  const int r0 = sg.row0 + (b - b0) * sg.rpb;
  const int r1 = min(sg.row1, r0 + sg.rpb);
  const int row_first = r0 + (int)threadIdx.x;
  const int rowc = min(row_first, r1 - 1);
  const int flag = __atomic_load_n(&S->done, __ATOMIC_RELAXED);
  RowPrefetch<P, V> f;
  f.beg = a.g_rp[rowc];
  f.end = a.g_rp[rowc + 1];
  const double fr = rc[rowc];
#pragma unroll
  for (int k = 0; k < P; k++) {
    const int j = min(f.beg + k, a.g_nnz - 1);
    f.col[k] = a.g_ci[j];
    f.v[k] = gv[j];
  }
  V tg[P];
#pragma unroll
  for (int k = 0; k < P; k++) tg[k] = tv[f.col[k] - a.f_col];
  __builtin_amdgcn_sched_barrier(0);  // keep the loads above issued in this order
  if (threadIdx.x == 0) s_flag = flag;
  __syncthreads();
  const int fl = s_flag;
  const bool part = mode == kAfterIter ? fl == kRunning
                    : mode == kVerify  ? fl == kPending
                                       : fl != kInactive;
  if (!part) return;
  double rz = 0.0;
  if (row_first < r1) {
    V acc = 0;
#pragma unroll
    for (int k = 0; k < P; k++)
      if (f.beg + k < f.end) {
        if (MIX) acc = fmaf((float)f.v[k], (float)tg[k], (float)acc);
        else acc = fma((double)f.v[k], (double)tg[k], (double)acc);
      }
    for (int j = f.beg + P; j < f.end; j++) {
      if (MIX) acc = fmaf((float)gv[j], (float)tv[a.g_ci[j] - a.f_col], (float)acc);
      else acc = fma((double)gv[j], (double)tv[a.g_ci[j] - a.f_col], (double)acc);
    }
    const double zi = (double)acc;
    a.z[row_first] = zi;
    rz += fr * zi;
  }
  // the later rows two at a time (loads of both issued before either sum)
  constexpr int R2 = 2;
  for (int row = row_first + kBlock; row < r1; row += R2 * kBlock) {
    RowPrefetch<P, V> g[R2];
    double rv[R2];
    V tq[R2][P];
    int rw[R2];
#pragma unroll
    for (int r = 0; r < R2; r++) {
      rw[r] = min(row + r * kBlock, r1 - 1);
      g[r].beg = a.g_rp[rw[r]];
      g[r].end = a.g_rp[rw[r] + 1];
      rv[r] = rc[rw[r]];
    }
#pragma unroll
    for (int r = 0; r < R2; r++)
#pragma unroll
      for (int k = 0; k < P; k++) {
        const int j = min(g[r].beg + k, a.g_nnz - 1);
        g[r].col[k] = a.g_ci[j];
        g[r].v[k] = gv[j];
      }
#pragma unroll
    for (int r = 0; r < R2; r++)
#pragma unroll
      for (int k = 0; k < P; k++) tq[r][k] = tv[g[r].col[k] - a.f_col];
#pragma unroll
    for (int r = 0; r < R2; r++) {
      if (row + r * kBlock >= r1) break;
      V acc = 0;
#pragma unroll
      for (int k = 0; k < P; k++)
        if (g[r].beg + k < g[r].end) {
          if (MIX) acc = fmaf((float)g[r].v[k], (float)tq[r][k], (float)acc);
          else acc = fma((double)g[r].v[k], (double)tq[r][k], (double)acc);
        }
      for (int j = g[r].beg + P; j < g[r].end; j++) {
        if (MIX) acc = fmaf((float)gv[j], (float)tv[a.g_ci[j] - a.f_col], (float)acc);
        else acc = fma((double)gv[j], (double)tv[a.g_ci[j] - a.f_col], (double)acc);
      }
      const double zi = (double)acc;
      a.z[rw[r]] = zi;
      rz += rv[r] * zi;
    }
  }
  rz = wg_sum(rz, lds);
  if (threadIdx.x == 0) CG_AT(prz, rsel ^ 1)[b] = rz;
}

// t = G^T r for the current residual (replacement, verification, start).
template <bool MIX>
__global__ __launch_bounds__(kBlock) void k_cg_gtr(CG_ARGS, int par_g, int mode) {
  TBSLA_NO_FMA
  CG_BIND;
  __shared__ int s_flag;
  const int b = cg_block(multi_);
  CG_SYSTEM(b);
  int rsel;
  if (!mode_select(S, mode, par_g, &s_flag, &rsel)) return;
  const double *rc = CG_AT(r, rsel);
  const int r0 = sg.row0 + (b - sg.blk0) * sg.rpb;
  const int r1 = min(sg.row1, r0 + sg.rpb);
  for (int row = r0 + (int)threadIdx.x; row < r1; row += kBlock) {
    if (MIX) {
      float acc = 0.0f;
      for (int j = a.t_rp[row]; j < a.t_rp[row + 1]; j++)
        acc = fmaf(a.t_v32[j], (float)rc[a.t_ci[j] - a.f_col], acc);
      a.t32[row] = acc;
    } else {
      double acc = 0.0;
      for (int j = a.t_rp[row]; j < a.t_rp[row + 1]; j++)
        acc = fma(a.t_v64[j], rc[a.t_ci[j] - a.f_col], acc);
      a.t64[row] = acc;
    }
  }
}

// k_cg_gtr with G on diagonals (G^T's row in ascending column, zero slots
// skipped, as k_cg_update_gdia).
template <bool MIX>
__global__ __launch_bounds__(kBlock) void k_cg_gtr_gdia(CG_ARGS, int par_g, int mode) {
  TBSLA_NO_FMA
  CG_BIND;
  typedef typename std::conditional<MIX, float, double>::type V;
  __shared__ int s_flag;
  const int b = cg_block(multi_);
  CG_SYSTEM(b);
  int rsel;
  if (!mode_select(S, mode, par_g, &s_flag, &rsel)) return;
  const double *rc = CG_AT(r, rsel);
  const V *gd = MIX ? (const V *)a.gd32 : (const V *)a.gd64;
  const int ndg = a.gndiag;
  const long long n = a.ncol;
  const int r0 = sg.row0 + (b - sg.blk0) * sg.rpb;
  const int r1 = min(sg.row1, r0 + sg.rpb);
  for (int row = r0 + (int)threadIdx.x; row < r1; row += kBlock) {
    V acc = 0;
    for (int k = ndg - 1; k >= 0; k--) {
      const long long src = (long long)row - a.gdoff[k];
      const V g = gd_slot(gd, src, k, ndg, n);
      if (g != (V)0) {
        if (MIX) acc = fmaf((float)g, (float)rc[src], (float)acc);
        else acc = fma((double)g, rc[src], (double)acc);
      }
    }
    if (MIX) a.t32[row] = (float)acc;
    else a.t64[row] = (double)acc;
  }
}

// K3 with G on diagonals: z_i = sum over G's row i in ascending column
// (ascending offset) of G_{i,i+o_k} t_{i+o_k}, zero slots skipped; r.z
// partials.  Rows two per thread and trip, loads of both issued first.
template <bool MIX, int KD, bool WIDE>
__global__ __launch_bounds__(kBlock) void k_cg_gz_gdia(CG_ARGS, int par_g, int mode) {
  TBSLA_NO_FMA
  CG_BIND;
  typedef typename std::conditional<MIX, float, double>::type V;
  constexpr int R2 = 2;
  __shared__ double lds[kBlock / kWave];
  __shared__ int s_flag;
  const int b = cg_block(multi_);
  CG_SYSTEM(b, "s"(a.prz[0]), "s"(a.prz[1]), "s"(a.r[0]), "s"(a.r[1]), "s"(a.z), "s"(a.ncol),
            "s"(a.gndiag), "s"(MIX ? (const void *)a.gd32 : (const void *)a.gd64),
            "s"(MIX ? (const void *)a.t32 : (const void *)a.t64), "s"(CG_OFF(gdoff8, 0)),
            "s"(CG_OFF(gdoff8, 1)), "s"(CG_OFF(gdoff8, 2)), "s"(CG_OFF(gdoff8, 3)));
  const int flag = __atomic_load_n(&S->done, __ATOMIC_RELAXED);
  const int rsel = mode == kAfterIter ? ((par_g ^ sg.shift) & 1) ^ 1
                   : mode == kVerify  ? sg.stop_par
                                      : 0;
  const double *rc = CG_AT(r, rsel);
  const V *gd = MIX ? (const V *)a.gd32 : (const V *)a.gd64;
  const V *tv = MIX ? (const V *)a.t32 : (const V *)a.t64;
  const int ndg = a.gndiag;
  const int r0 = sg.row0 + (b - sg.blk0) * sg.rpb;
  const int r1 = min(sg.row1, r0 + sg.rpb);
  int off[KD];
#pragma unroll
  for (int k = 0; k < KD; k++) off[k] = CG_OFF(gdoff8, k);
  const int row_first = r0 + (int)threadIdx.x;
  V gv[R2][KD], tq[R2][KD];
  double rv[R2];
  int rw[R2];
  auto load = [&](int row) {
#pragma unroll
    for (int r = 0; r < R2; r++) {
      rw[r] = min(row + r * kBlock, r1 - 1);
      rv[r] = ldi<WIDE>(rc, rw[r]);
#pragma unroll
      for (int k = 0; k < KD; k++) {
        const int c = rw[r] + off[k];
        gv[r][k] = ldi<WIDE>(gd, dia_at(rw[r], min(k, ndg - 1), ndg));
        tq[r][k] = ldi<WIDE>(tv, c >= 0 ? c : rw[r]);
      }
    }
  };
  load(row_first);  // before the done flag is shared, as k_cg_gz
  __builtin_amdgcn_sched_barrier(0);
  if (threadIdx.x == 0) s_flag = flag;
  __syncthreads();
  const int fl = s_flag;
  const bool part = mode == kAfterIter ? fl == kRunning
                    : mode == kVerify  ? fl == kPending
                                       : fl != kInactive;
  if (!part) return;
  double rz = 0.0;
  for (int row = row_first; row < r1; row += R2 * kBlock) {
    if (row != row_first) load(row);
#pragma unroll
    for (int r = 0; r < R2; r++) {
      if (row + r * kBlock >= r1) break;
      V acc = 0;
#pragma unroll
      for (int k = 0; k < KD; k++)
        if (k < ndg && gv[r][k] != (V)0) {
          if (MIX) acc = fmaf((float)gv[r][k], (float)tq[r][k], (float)acc);
          else acc = fma((double)gv[r][k], (double)tq[r][k], (double)acc);
        }
      const double zi = (double)acc;
      a.z[rw[r]] = zi;
      rz += rv[r] * zi;
    }
  }
  rz = wg_sum(rz, lds);
  if (threadIdx.x == 0) CG_AT(prz, rsel ^ 1)[b] = rz;
}

// The entries' offsets col - row of kProbeRows rows spread over the block
// (row (k * 2654435761) mod n): out[k * 9] = the row's entry count, then up
// to 8 offsets (a count above 8 rules the diagonal form out).
constexpr int kProbeRows = 64;
__global__ __launch_bounds__(kWave) void k_g_probe(long long n, int f_col,
                                                   const int *__restrict__ rp,
                                                   const int *__restrict__ ci, int *__restrict__ out) {
  const int k = threadIdx.x;
  const long long r = (long long)(((unsigned long long)(k + 1) * 2654435761ULL) % (unsigned long long)n);
  const int beg = rp[r], cnt = rp[r + 1] - beg;
  out[k * 9] = cnt;
  for (int j = 0; j < 8; j++) out[k * 9 + 1 + j] = j < cnt ? (int)((ci[beg + j] - f_col) - r) : 0;
}

// G's entries into its diagonal layout (slots zeroed first): the slot of
// offset col - row among the offsets given; *bad set when an entry lies on
// none of them or two entries of a row share one (G is then applied from its
// CSR rows).
template <typename V>
__global__ __launch_bounds__(kBlock) void k_g_to_dia(long long n, int f_col, int f_row,
                                                     const int *__restrict__ rp,
                                                     const int *__restrict__ ci,
                                                     const double *__restrict__ v,
                                                     const int *__restrict__ off, int ndg,
                                                     V *__restrict__ gd, int *bad) {
  for (long long i = (long long)blockIdx.x * kBlock + threadIdx.x; i < n;
       i += (long long)gridDim.x * kBlock) {
    unsigned used = 0;
    for (int j = rp[i]; j < rp[i + 1]; j++) {
      const long long o = (long long)(ci[j] - f_col) - (i + f_row - f_col);
      int k = -1;
      for (int q = 0; q < ndg; q++)
        if (off[q] == o) k = q;
      if (k < 0 || (used >> k) & 1u) {
        atomicOr(bad, 1);
        continue;
      }
      used |= 1u << k;
      gd[dia_at(i, k, ndg)] = (V)v[j];
    }
  }
}

// r = b - ax (ax = A x in FP64 when use_ax, else 0: a zero start) into the selected
// buffer, z = D^-1 r for Jacobi, and the r.r (r.z) partials.  At the start
// it also zeroes x (unless an initial guess is given) and p, seeds the
// "old r.z" slot with +inf (so the first beta is 0) and leaves b.b partials
// in ppap.
template <int PRE>
__global__ __launch_bounds__(kBlock) void k_cg_residual(CG_ARGS, int use_ax, int par_g, int mode,
                                                        int zero_x) {
  TBSLA_NO_FMA
  CG_BIND;
  const double *ax = use_ax ? a.ax : nullptr;
  __shared__ double lds[kBlock / kWave];
  __shared__ int s_flag;
  const int b = cg_block(multi_);
  CG_SYSTEM(b);
  int rsel;
  if (!mode_select(S, mode, par_g, &s_flag, &rsel)) return;
  double *rc = CG_AT(r, rsel);
  const int b0 = sg.blk0;
  const int r0 = sg.row0 + (b - b0) * sg.rpb;
  const int r1 = min(sg.row1, r0 + sg.rpb);
  double rr = 0.0, rz = 0.0, bb = 0.0;
  for (int row = r0 + (int)threadIdx.x; row < r1; row += kBlock) {
    const double bi = a.b[row];
    const double ri = ax ? bi - ax[row] : bi;
    rc[row] = ri;
    rr += ri * ri;
    if (PRE == 1) {
      const double zi = ri * a.dinv[row];
      a.z[row] = zi;
      rz += ri * zi;
    }
    if (mode == kStart) {
      if (zero_x) a.x[row] = 0.0;
      a.p[0][row] = 0.0;
      bb += bi * bi;
    }
  }
  rr = wg_sum(rr, lds);
  if (PRE == 1) rz = wg_sum(rz, lds);
  if (mode == kStart) bb = wg_sum(bb, lds);
  if (threadIdx.x == 0) {
    CG_AT(prr, rsel ^ 1)[b] = rr;
    if (PRE == 0) CG_AT(prz, rsel ^ 1)[b] = rr;
    if (PRE == 1) CG_AT(prz, rsel ^ 1)[b] = rz;
    if (mode == kStart) {
      CG_AT(prz, 0)[b] = b == b0 ? INFINITY : 0.0;  // the first beta is 0
      a.ppap[b] = bb;
    }
    if (b == b0) S->true_res = 1;
  }
}

// Per-system setup after the start residual: threshold, |r0|, counters.
__global__ __launch_bounds__(kBlock) void k_cg_start(CG_ARGS, double tol, int relative,
                                                     double near_zero) {
  CG_BIND;
  __shared__ double lds[kBlock / kWave];
  __shared__ int s_flag;
  const int b = cg_block(multi_);
  if (b == 0 && threadIdx.x == 0) a.com->t0 = wall_clock64();
  CG_SYSTEM(b);
  if (b != sg.blk0) return;
  if (seg_flag(S, &s_flag) == kInactive) return;
  (void)lds;
  double t[3];
  seg_sums(a.ppap, CG_AT(prr, 1), nullptr, 2, sg.blk0, sg.blk1, t);
  const double bb = t[0], rr = t[1];
  if (threadIdx.x == 0) {
    S->stop = relative ? tol * sqrt(bb) : tol;
    S->near_zero = near_zero;
    S->rnorm0 = sqrt(rr);
    S->rnorm = S->rnorm0;
    S->iters = 0;
    S->ent0 = a.rowptr[sg.row0];
    S->shift = 0;
    S->true_res = 1;
    S->t_done = 0;
  }
}

// After verification: accept (true |r| below the threshold) or resume at
// the next global iteration j from the replaced residual (only j's parity
// matters).
__global__ __launch_bounds__(kBlock) void k_cg_vcheck(CG_ARGS, int j) {
  CG_BIND;
  __shared__ double lds[kBlock / kWave];
  __shared__ int s_flag;
  const int b = cg_block(multi_);
  CG_SYSTEM(b);
  if (b != sg.blk0) return;
  if (seg_flag(S, &s_flag) != kPending) return;
  (void)lds;
  double t[3];
  seg_sums(CG_AT(prr, sg.stop_par ^ 1), nullptr, nullptr, 1, sg.blk0, sg.blk1, t);
  const double rr = t[0];
  if (threadIdx.x == 0) {
    const double rn = sqrt(rr);
    S->rnorm = rn;
    atomicAdd(&a.com->npending, -1);
    if (rn < sg.stop) {
      // t_done keeps the time of the iteration whose test the recurrence
      // passed (k1_test), not the time of this verification
      S->done = kConverged;
      atomicAdd(&a.com->ndone, 1);
    } else {
      // the recurrence had drifted from the true residual: restart from it
      // (beta = 0 at the next iteration: an infinite "old r.z")
      S->shift = (j ^ sg.stop_par) & 1;
      S->done = kRunning;
      S->left = 0;
    }
  }
  __syncthreads();
  if (!(sqrt(rr) < sg.stop)) {
    double *old_rz = CG_AT(prz, sg.stop_par);
    for (int k = sg.blk0 + (int)threadIdx.x; k < sg.blk1; k += kBlock)
      old_rz[k] = k == sg.blk0 ? INFINITY : 0.0;
  }
}

// ax = A x (FP64 matrix) for the rows of the systems the mode selects, in
// the engine's workgroup layout (workgroups of other systems return at
// once); L lanes per row.  kStart: before k_cg_start has stored ent0.
template <int L>
__global__ __launch_bounds__(kBlock) void k_cg_ax(CG_ARGS, int par_g, int mode) {
  CG_BIND;
  double *ax = a.ax;
  __shared__ int s_flag;
  const int b = cg_block(multi_);
  CG_SYSTEM(b);
  int rsel;
  if (!mode_select(S, mode, par_g, &s_flag, &rsel)) return;
  const int r0 = sg.row0 + (b - sg.blk0) * sg.rpb;
  const int r1 = min(sg.row1, r0 + sg.rpb);
  const int lane = threadIdx.x & (L - 1);
  const int ent0 = mode == kStart ? a.rowptr[sg.row0] : sg.ent0;
  typedef CgRow<L, double> Row;
  constexpr int PASS = kBlock / L;
  for (int row = r0 + (int)threadIdx.x / L; row < r1; row += PASS) {
    Row w;
    w.extent(a.rowptr, row, ent0);
    w.load(a.colidx, a.val64, a.a_nnz, a.f_col, lane);
    double g[Row::P];
#pragma unroll
    for (int k = 0; k < Row::P; k++) g[k] = a.x[w.col[k]];
    double acc = 0.0;
#pragma unroll
    for (int k = 0; k < Row::P; k++)
      if (w.in(lane, k)) acc = fma(w.v[k], g[k], acc);
    constexpr int Q = L == 1 ? 1 : 4;
    for (unsigned j = w.rest(lane); j < (unsigned)w.end; j += Q * L)
#pragma unroll
      for (int q = 0; q < Q; q++)
        if (j + q < (unsigned)w.end) acc = fma(a.val64[j + q], a.x[a.colidx[j + q] - a.f_col], acc);
    acc = lane_sum<L>(acc);
    if (lane == 0) ax[row] = acc;
  }
}

__global__ __launch_bounds__(kBlock) void k_to_f32(const double *__restrict__ a, long long n,
                                                   float *__restrict__ b) {
  for (long long k = (long long)blockIdx.x * kBlock + threadIdx.x; k < n;
       k += (long long)gridDim.x * kBlock)
    b[k] = (float)a[k];
}

// D^-1 of a CSR block's diagonal (duplicates summed; 1 where the diagonal is
// missing or zero).
__global__ __launch_bounds__(kBlock) void k_csr_dinv(long long n_rows, int f_row, int f_col,
                                                     const int *__restrict__ rowptr,
                                                     const int *__restrict__ colidx,
                                                     const double *__restrict__ vals,
                                                     double *__restrict__ dinv) {
  for (long long i = (long long)blockIdx.x * kBlock + threadIdx.x; i < n_rows;
       i += (long long)gridDim.x * kBlock) {
    double d = 0.0;
    for (int j = rowptr[i]; j < rowptr[i + 1]; j++)
      if (colidx[j] - f_col == i + f_row - f_col) d += vals[j];
    dinv[i] = d != 0.0 ? 1.0 / d : 1.0;
  }
}

unsigned sgrid(long long n) {
  long long g = (n + kBlock - 1) / kBlock;
  return (unsigned)std::max<long long>(1, std::min<long long>(g, 65536));
}

template <typename T>
struct Buf {
  T *p = nullptr;
  size_t n = 0;
  // grows only; a reallocation waits for the device first (work in flight
  // may still read the old buffer)
  int ensure(size_t count) {
    if (count <= n && p) return TBSLA_HIP_SUCCESS;
    if (p) {
      (void)hipDeviceSynchronize();
      device_free(p);
    }
    p = nullptr;
    n = 0;
    TBSLA_TRY(device_alloc((void **)&p, std::max<size_t>(count, 1) * sizeof(T)));
    n = count;
    return TBSLA_HIP_SUCCESS;
  }
  void release() {
    if (p) device_free(p);
    p = nullptr;
    n = 0;
  }
};

// What a captured graph bakes in besides the argument block's address: the
// launch plan (kernel variants, grid, iteration indices).  Pointers are not
// part of it -- every kernel reads them from the argument block at run time.
struct GraphKey {
  int L, pre, mixed, replace, batch, nblocks, verify, dia, gdia, two, multi;
  bool operator==(const GraphKey &o) const {
    return L == o.L && pre == o.pre && mixed == o.mixed && replace == o.replace &&
           batch == o.batch && nblocks == o.nblocks && verify == o.verify && dia == o.dia &&
           gdia == o.gdia && two == o.two && multi == o.multi;
  }
};

}  // namespace

// Work vectors, partials, the argument block and graphs kept by a matrix
// handle between solves.
struct CgCache {
  int device = 0;
  Buf<double> b, x, r0, r1, p0, p1, z, ap, t64, dinv, ax;
  Buf<float> t32;
  Buf<double> ppap, prr0, prr1, prz0, prz1;
  Buf<CgSeg> seg;  // a batch's systems
  Buf<int> block_seg;
  // stand-ins for A's or G^T's entry arrays when they hold no entry: one
  // column index (the block's first column) and one zero value
  Buf<int> dummy_i;
  Buf<double> dummy_d;
  // the kernels' argument block (one CgBlock, allocated once and never moved:
  // captured graphs name it) and its pinned staging copy
  Buf<CgBlock> args;
  CgBlock *h_args = nullptr;
  CgCom *h_com = nullptr;  // pinned status copies (2)
  int *h_probe = nullptr;  // pinned: G's probe rows (extents, columns) and the dia check
  hipEvent_t ev[2] = {nullptr, nullptr};
  hipStream_t own = nullptr;  // used when the caller passes the null stream
  // FP32 copy of A's values for the mixed form, made from the handle uid
  // at values version ver; kept with the cache (which a destroyed handle
  // leaves to the next), so a new matrix of the same size allocates nothing
  float *a_v32 = nullptr;
  size_t a_v32_len = 0;
  unsigned long long a_v32_uid = 0, a_v32_ver = 0;
  // FP32 copy of A's diagonal layout, made from the layout build dv32_build
  // (ids are unique in the process; a layout is rebuilt when values change)
  float *dv32 = nullptr;
  size_t dv32_len = 0;
  unsigned long long dv32_build = 0;
  // factor G in its CSR form: G^T's rows (when not given) and FP32 copies,
  // remade on every call (G may have been rewritten in place)
  int *t_rp = nullptr, *t_ci = nullptr;
  double *t_v64 = nullptr;
  float *g_v32 = nullptr, *t_v32 = nullptr;
  size_t f32_len = 0;
  // factor G on diagonals: offsets, slots (FP64 or FP32), the check flag
  Buf<int> gdoff;
  int host_gdoff[8] = {};
  Buf<double> gd64;
  Buf<float> gd32;
  Buf<int> gbad;
  // instantiated graphs, one set per launch plan, most recently used first:
  // exec[0] a plain batch, exec[1] a batch ending with a replacement step
  struct GraphSet {
    GraphKey key;
    hipGraphExec_t exec[2] = {nullptr, nullptr};
    void destroy() {
      for (auto &x : exec)
        if (x) {
          (void)hipGraphExecDestroy(x);
          x = nullptr;
        }
    }
  };
  static constexpr size_t kGraphSets = 8;
  std::vector<GraphSet> graphs;
  std::vector<CgSeg> host_seg;
  std::vector<int> host_blocks;

  void drop_factor() {
    device_free(t_rp);
    device_free(t_ci);
    device_free(t_v64);
    device_free(g_v32);
    device_free(t_v32);
    t_rp = t_ci = nullptr;
    t_v64 = nullptr;
    g_v32 = t_v32 = nullptr;
    f32_len = 0;
  }
  ~CgCache() {
    (void)hipDeviceSynchronize();
    for (auto &g : graphs) g.destroy();
    Buf<double> *bufs[] = {&b, &x, &r0, &r1, &p0, &p1, &z, &ap, &t64, &dinv, &ax,
                           &ppap, &prr0, &prr1, &prz0, &prz1, &gd64};
    for (auto *q : bufs) q->release();
    t32.release();
    gd32.release();
    seg.release();
    block_seg.release();
    dummy_i.release();
    dummy_d.release();
    gdoff.release();
    gbad.release();
    args.release();
    if (h_args) (void)hipHostFree(h_args);
    if (h_com) (void)hipHostFree(h_com);
    if (h_probe) (void)hipHostFree(h_probe);
    for (auto &e : ev)
      if (e) (void)hipEventDestroy(e);
    if (own) (void)hipStreamDestroy(own);
    drop_factor();
    device_free(a_v32);
    device_free(dv32);
  }
};

// Caches of destroyed handles, kept for the next handles' solves: their
// stream, events, pinned status words, work vectors and instantiated graphs
// are reused (creating them costs 1-2 ms per new matrix, a third of a 64^3
// solve).  At most kSpareCaches, per device, under a mutex; never freed at
// process exit (the runtime may be gone by then).  A reused cache's graphs
// name only its own argument block, so they serve the next handle as they
// are.
constexpr size_t kSpareCaches = 2;

std::mutex &spare_mutex() {
  static std::mutex *mu = new std::mutex;
  return *mu;
}
std::vector<CgCache *> &spare_caches() {
  static auto *v = new std::vector<CgCache *>;
  return *v;
}

CgCache *take_cache() {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) dev = 0;
  {
    std::lock_guard<std::mutex> g(spare_mutex());
    auto &v = spare_caches();
    for (size_t k = v.size(); k-- > 0;) {
      if (v[k]->device == dev) {
        CgCache *c = v[k];
        v.erase(v.begin() + (long)k);
        return c;
      }
    }
  }
  CgCache *c = new CgCache();
  c->device = dev;
  return c;
}

void cg_cache_release(tbsla_hip_matrix_s *m) {
  if (!m->cg_cache) return;
  CgCache *c = static_cast<CgCache *>(m->cg_cache);
  m->cg_cache = nullptr;
  if (c->own) (void)hipStreamSynchronize(c->own);
  c->drop_factor();  // arrays derived from the old factor
  {
    std::lock_guard<std::mutex> g(spare_mutex());
    if (spare_caches().size() < kSpareCaches) {
      spare_caches().push_back(c);
      return;
    }
  }
  delete c;
}

namespace {

struct Plan {
  int L, pre, mixed, replace, verify, stall;
  bool dia;   // K1 reads A's diagonal layout
  int dkd;    // its kernel's diagonals: 3, 5 or 7, or 0 for any number
  bool sym;   // and those below the main one read as their mirror images
  bool two;   // K1 in two passes (k_cg_pnew, then k_cg_ap) on A's CSR rows
  bool gdia;  // M = G G^T applied from G's diagonals
  int gkd;    // their kernels' capacity: 4 or 8 diagonals
  bool wide;  // vectors or G's diagonals of 4 GiB or more (64-bit offsets)
  long long n;
  int nblocks;
  int multi;             // a batch of systems
  const CgBlock *args;  // device argument block
  hipStream_t s;
};

template <int L, bool MIX, bool ZBUF>
void launch_k1(const Plan &p, int par, int check, int check_only) {
  if (!p.two) {
    k_cg_spmv_p<L, MIX, ZBUF><<<p.nblocks, kBlock, 0, p.s>>>(p.args, p.multi, par, check, check_only);
    return;
  }
  k_cg_pnew<ZBUF><<<p.nblocks, kBlock, 0, p.s>>>(p.args, p.multi, par, check, check_only);
  if (!check_only) k_cg_ap<L, MIX><<<p.nblocks, kBlock, 0, p.s>>>(p.args, p.multi, par);
}

template <int KD, bool SYM>
void launch_k1_dia(const Plan &p, bool zbuf, int par, int check, int check_only) {
  const int g = p.nblocks;
  if (p.mixed) {
    if (zbuf) k_cg_spmv_dia<true, true, KD, SYM><<<g, kBlock, 0, p.s>>>(p.args, p.multi, par, check, check_only);
    else k_cg_spmv_dia<true, false, KD, SYM><<<g, kBlock, 0, p.s>>>(p.args, p.multi, par, check, check_only);
  } else {
    if (zbuf) k_cg_spmv_dia<false, true, KD, SYM><<<g, kBlock, 0, p.s>>>(p.args, p.multi, par, check, check_only);
    else k_cg_spmv_dia<false, false, KD, SYM><<<g, kBlock, 0, p.s>>>(p.args, p.multi, par, check, check_only);
  }
}

template <int L>
void launch_k1_l(const Plan &p, int par, int check, int check_only) {
  const bool zbuf = p.pre != 0;
  if (p.dia) {
    switch (p.dkd + (p.sym ? 10 : 0)) {
      case 3: launch_k1_dia<3, false>(p, zbuf, par, check, check_only); break;
      case 5: launch_k1_dia<5, false>(p, zbuf, par, check, check_only); break;
      case 7: launch_k1_dia<7, false>(p, zbuf, par, check, check_only); break;
      case 13: launch_k1_dia<3, true>(p, zbuf, par, check, check_only); break;
      case 15: launch_k1_dia<5, true>(p, zbuf, par, check, check_only); break;
      case 17: launch_k1_dia<7, true>(p, zbuf, par, check, check_only); break;
      default: launch_k1_dia<0, false>(p, zbuf, par, check, check_only); break;
    }
    return;
  }
  if (p.mixed) {
    if (zbuf) launch_k1<L, true, true>(p, par, check, check_only);
    else launch_k1<L, true, false>(p, par, check, check_only);
  } else {
    if (zbuf) launch_k1<L, false, true>(p, par, check, check_only);
    else launch_k1<L, false, false>(p, par, check, check_only);
  }
}

void launch_k1_any(const Plan &p, int par, int check, int check_only) {
  switch (p.L) {
    case 1: launch_k1_l<1>(p, par, check, check_only); break;
    case 2: launch_k1_l<2>(p, par, check, check_only); break;
    case 4: launch_k1_l<4>(p, par, check, check_only); break;
    case 8: launch_k1_l<8>(p, par, check, check_only); break;
    case 16: launch_k1_l<16>(p, par, check, check_only); break;
    case 32: launch_k1_l<32>(p, par, check, check_only); break;
    default: launch_k1_l<64>(p, par, check, check_only); break;
  }
}

template <bool WIDE>
void launch_k2_gdia(const Plan &p, int par, int count) {
  const int g = p.nblocks;
  if (p.gkd == 4) {
    if (p.mixed) k_cg_update_gdia<true, 4, WIDE><<<g, kBlock, 0, p.s>>>(p.args, p.multi, par, count);
    else k_cg_update_gdia<false, 4, WIDE><<<g, kBlock, 0, p.s>>>(p.args, p.multi, par, count);
  } else {
    if (p.mixed) k_cg_update_gdia<true, 8, WIDE><<<g, kBlock, 0, p.s>>>(p.args, p.multi, par, count);
    else k_cg_update_gdia<false, 8, WIDE><<<g, kBlock, 0, p.s>>>(p.args, p.multi, par, count);
  }
}

void launch_k2(const Plan &p, int par, int count) {
  const int g = p.nblocks;
  if (p.pre == 0) {
    if (p.mixed) k_cg_update<0, true><<<g, kBlock, 0, p.s>>>(p.args, p.multi, par, count);
    else k_cg_update<0, false><<<g, kBlock, 0, p.s>>>(p.args, p.multi, par, count);
  } else if (p.pre == 1) {
    if (p.mixed) k_cg_update<1, true><<<g, kBlock, 0, p.s>>>(p.args, p.multi, par, count);
    else k_cg_update<1, false><<<g, kBlock, 0, p.s>>>(p.args, p.multi, par, count);
  } else if (p.gdia) {
    if (p.wide) launch_k2_gdia<true>(p, par, count);
    else launch_k2_gdia<false>(p, par, count);
  } else {
    if (p.mixed) k_cg_update<2, true><<<g, kBlock, 0, p.s>>>(p.args, p.multi, par, count);
    else k_cg_update<2, false><<<g, kBlock, 0, p.s>>>(p.args, p.multi, par, count);
  }
}

template <bool WIDE>
void launch_gz_gdia(const Plan &p, int par, int mode) {
  const int g = p.nblocks;
  if (p.gkd == 4) {
    if (p.mixed) k_cg_gz_gdia<true, 4, WIDE><<<g, kBlock, 0, p.s>>>(p.args, p.multi, par, mode);
    else k_cg_gz_gdia<false, 4, WIDE><<<g, kBlock, 0, p.s>>>(p.args, p.multi, par, mode);
  } else {
    if (p.mixed) k_cg_gz_gdia<true, 8, WIDE><<<g, kBlock, 0, p.s>>>(p.args, p.multi, par, mode);
    else k_cg_gz_gdia<false, 8, WIDE><<<g, kBlock, 0, p.s>>>(p.args, p.multi, par, mode);
  }
}

void launch_gz(const Plan &p, int par, int mode) {
  if (p.gdia) {
    if (p.wide) launch_gz_gdia<true>(p, par, mode);
    else launch_gz_gdia<false>(p, par, mode);
  } else {
    if (p.mixed) k_cg_gz<true><<<p.nblocks, kBlock, 0, p.s>>>(p.args, p.multi, par, mode);
    else k_cg_gz<false><<<p.nblocks, kBlock, 0, p.s>>>(p.args, p.multi, par, mode);
  }
}

void launch_gtr(const Plan &p, int par, int mode) {
  if (p.gdia) {
    if (p.mixed) k_cg_gtr_gdia<true><<<p.nblocks, kBlock, 0, p.s>>>(p.args, p.multi, par, mode);
    else k_cg_gtr_gdia<false><<<p.nblocks, kBlock, 0, p.s>>>(p.args, p.multi, par, mode);
  } else {
    if (p.mixed) k_cg_gtr<true><<<p.nblocks, kBlock, 0, p.s>>>(p.args, p.multi, par, mode);
    else k_cg_gtr<false><<<p.nblocks, kBlock, 0, p.s>>>(p.args, p.multi, par, mode);
  }
}

void launch_residual(const Plan &p, int use_ax, int par, int mode, int zero_x) {
  if (p.pre == 1) k_cg_residual<1><<<p.nblocks, kBlock, 0, p.s>>>(p.args, p.multi, use_ax, par, mode, zero_x);
  else if (p.pre == 0) k_cg_residual<0><<<p.nblocks, kBlock, 0, p.s>>>(p.args, p.multi, use_ax, par, mode, zero_x);
  else k_cg_residual<2><<<p.nblocks, kBlock, 0, p.s>>>(p.args, p.multi, use_ax, par, mode, zero_x);
}

// ax = A x with the FP64 matrix, for the systems the mode selects
void launch_ax(const Plan &p, int par, int mode) {
  switch (p.L) {
    case 1: k_cg_ax<1><<<p.nblocks, kBlock, 0, p.s>>>(p.args, p.multi, par, mode); break;
    case 2: k_cg_ax<2><<<p.nblocks, kBlock, 0, p.s>>>(p.args, p.multi, par, mode); break;
    case 4: k_cg_ax<4><<<p.nblocks, kBlock, 0, p.s>>>(p.args, p.multi, par, mode); break;
    case 8: k_cg_ax<8><<<p.nblocks, kBlock, 0, p.s>>>(p.args, p.multi, par, mode); break;
    case 16: k_cg_ax<16><<<p.nblocks, kBlock, 0, p.s>>>(p.args, p.multi, par, mode); break;
    case 32: k_cg_ax<32><<<p.nblocks, kBlock, 0, p.s>>>(p.args, p.multi, par, mode); break;
    default: k_cg_ax<64><<<p.nblocks, kBlock, 0, p.s>>>(p.args, p.multi, par, mode); break;
  }
}

// r = b - A x (FP64), then z = M r for the systems the mode selects
void true_residual(const Plan &p, int par, int mode) {
  launch_ax(p, par, mode);
  launch_residual(p, 1, par, mode, 0);
  if (p.pre == 2) {
    launch_gtr(p, par, mode);
    launch_gz(p, par, mode);
  }
}

// iteration i (global): K1 (tested when i > 0), K2, K3; then, after every
// replace_every-th iteration (i a multiple of it), the true FP64 residual
// replaces the recurrence's.  tail: also settle the systems waiting for
// their true-residual test (a replacement step does it anyway: the same
// FP64 product serves both), so they wait at most one batch, without a host
// round trip.
void enqueue_iteration(const Plan &p, int i, bool tail) {
  const int par = i & 1;
  launch_k1_any(p, par, i > 0, 0);
  const bool replace = p.replace > 0 && i > 0 && i % p.replace == 0;
  launch_k2(p, par, i > 0);
  // a replacement step recomputes z from the true residual: no K3 of its own
  if (replace) true_residual(p, par, kAfterIter);
  else if (p.pre == 2) launch_gz(p, par, kAfterIter);
  if (p.verify && (replace || tail)) {
    true_residual(p, par, kVerify);
    k_cg_vcheck<<<p.nblocks, kBlock, 0, p.s>>>(p.args, p.multi, (i + 1) & 1);
  }
}

// G's diagonals for the diagonal form of M = G G^T: the offsets of the
// entries of kProbeRows rows spread over the block (at most 8 distinct, all
// <= 0: G lower triangular), then every entry placed on one of them.  *ndg: the count of
// diagonals, or 0 (G is then applied from its CSR rows) when the probe or
// the placement fails.
int build_gdia(CgCache &c, const tbsla_hip_matrix_s *G, bool mixed, hipStream_t s, int *ndg_out) {
  *ndg_out = 0;
  const long long n = G->ln_row;
  if (n < 1 || G->stored < 1) return TBSLA_HIP_SUCCESS;
  constexpr int kMaxDiag = 8;
  if (!c.h_probe)
    TBSLA_HIP_CHECK(hipHostMalloc((void **)&c.h_probe, 1024 * sizeof(int), hipHostMallocDefault));
  int *h = c.h_probe;
  TBSLA_TRY(c.gbad.ensure(kProbeRows * 9 + 1));
  k_g_probe<<<1, kProbeRows, 0, s>>>(n, G->f_col, G->rowptr, G->colidx, c.gbad.p + 1);
  TBSLA_HIP_LAUNCH_CHECK();
  TBSLA_HIP_CHECK(hipMemcpyAsync(h, c.gbad.p + 1, kProbeRows * 9 * sizeof(int),
                                 hipMemcpyDeviceToHost, s));
  TBSLA_HIP_CHECK(hipStreamSynchronize(s));
  std::vector<int> off;
  for (int k = 0; k < kProbeRows; k++) {
    const int cnt = h[k * 9];
    if (cnt < 0 || cnt > kMaxDiag) return TBSLA_HIP_SUCCESS;
    for (int j = 0; j < cnt; j++) {
      const int o = h[k * 9 + 1 + j];
      if (o > 0) return TBSLA_HIP_SUCCESS;
      if (std::find(off.begin(), off.end(), o) == off.end()) off.push_back(o);
    }
  }
  if (off.empty() || off.size() > (size_t)kMaxDiag) return TBSLA_HIP_SUCCESS;
  std::sort(off.begin(), off.end());
  const int ndg = (int)off.size();
  const size_t slots = (size_t)((n + kWave - 1) / kWave) * kWave * ndg;
  TBSLA_TRY(c.gdoff.ensure(kMaxDiag));
  static_assert(kMaxDiag <= sizeof c.host_gdoff / sizeof(int), "offsets at hand");
  for (int k = 0; k < ndg; k++) h[kProbeRows * 9 + k] = c.host_gdoff[k] = off[k];
  TBSLA_HIP_CHECK(hipMemcpyAsync(c.gdoff.p, h + kProbeRows * 9, ndg * sizeof(int),
                                 hipMemcpyHostToDevice, s));
  TBSLA_HIP_CHECK(hipMemsetAsync(c.gbad.p, 0, sizeof(int), s));
  if (mixed) {
    TBSLA_TRY(c.gd32.ensure(slots));
    TBSLA_HIP_CHECK(hipMemsetAsync(c.gd32.p, 0, slots * sizeof(float), s));
    k_g_to_dia<float><<<sgrid(n), kBlock, 0, s>>>(n, G->f_col, G->f_row, G->rowptr, G->colidx,
                                                  G->values, c.gdoff.p, ndg, c.gd32.p, c.gbad.p);
  } else {
    TBSLA_TRY(c.gd64.ensure(slots));
    TBSLA_HIP_CHECK(hipMemsetAsync(c.gd64.p, 0, slots * sizeof(double), s));
    k_g_to_dia<double><<<sgrid(n), kBlock, 0, s>>>(n, G->f_col, G->f_row, G->rowptr, G->colidx,
                                                   G->values, c.gdoff.p, ndg, c.gd64.p, c.gbad.p);
  }
  TBSLA_HIP_LAUNCH_CHECK();
  TBSLA_HIP_CHECK(hipMemcpyAsync(h + kProbeRows * 9 + kMaxDiag, c.gbad.p, sizeof(int),
                                 hipMemcpyDeviceToHost, s));
  TBSLA_HIP_CHECK(hipStreamSynchronize(s));
  if (!h[kProbeRows * 9 + kMaxDiag]) *ndg_out = ndg;
  return TBSLA_HIP_SUCCESS;
}

}  // namespace

// The solver behind tbsla_hip_cg and tbsla_hip_cg_batched.
int cg_solve_on(tbsla_hip_matrix_s *m, int nsys, const int *h_rows, const int *h_active,
                const double *d_rhs, double *d_x, const tbsla_hip_cg_options &o,
                tbsla_hip_cg_result *res, hipStream_t s);

// The null stream cannot be captured into a graph: a solve asked for on it
// runs on a stream of the handle's own (default priority), ordered after
// the null stream's earlier work; it is synchronised on return.
int cg_solve(tbsla_hip_matrix_s *m, int nsys, const int *h_rows, const int *h_active,
             const double *d_rhs, double *d_x, const tbsla_hip_cg_options &o,
             tbsla_hip_cg_result *res, hipStream_t s) {
  if (s != nullptr) return cg_solve_on(m, nsys, h_rows, h_active, d_rhs, d_x, o, res, s);
  if (!m->cg_cache) m->cg_cache = take_cache();
  CgCache &c = *static_cast<CgCache *>(m->cg_cache);
  if (!c.own) TBSLA_HIP_CHECK(hipStreamCreateWithFlags(&c.own, hipStreamNonBlocking));
  TBSLA_HIP_CHECK(hipDeviceSynchronize());  // earlier null-stream work
  return cg_solve_on(m, nsys, h_rows, h_active, d_rhs, d_x, o, res, c.own);
}

int cg_solve_on(tbsla_hip_matrix_s *m, int nsys, const int *h_rows, const int *h_active,
                const double *d_rhs, double *d_x, const tbsla_hip_cg_options &o,
                tbsla_hip_cg_result *res, hipStream_t s) {
  if (m->format != TBSLA_HIP_CSR) return fail(TBSLA_HIP_ERR_UNSUPPORTED, "CG needs a CSR block");
  if (m->ln_row != m->ln_col || m->f_row != m->f_col)
    return fail(TBSLA_HIP_ERR_INVALID, "CG needs a square diagonal block");
  const long long n = m->ln_row;
  if (nsys < 1 || h_rows[0] != 0 || h_rows[nsys] != n)
    return fail(TBSLA_HIP_ERR_INVALID, "system row offsets must cover the block");
  for (int k = 0; k < nsys; k++)
    if (h_rows[k + 1] <= h_rows[k]) return fail(TBSLA_HIP_ERR_INVALID, "empty system");
  if (o.preconditioner < TBSLA_HIP_PRECOND_NONE || o.preconditioner > TBSLA_HIP_PRECOND_FACTORED)
    return fail(TBSLA_HIP_ERR_UNSUPPORTED, "unknown preconditioner");
  if (o.precision != TBSLA_HIP_CG_FP64 && o.precision != TBSLA_HIP_CG_MIXED)
    return fail(TBSLA_HIP_ERR_UNSUPPORTED, "unknown precision");
  if (o.factor_form < TBSLA_HIP_FACTOR_AUTO || o.factor_form > TBSLA_HIP_FACTOR_DIAGONALS)
    return fail(TBSLA_HIP_ERR_INVALID, "unknown factor_form");
  tbsla_hip_matrix_s *G = o.factor;
  const int pre = o.preconditioner;
  if (pre == TBSLA_HIP_PRECOND_FACTORED) {
    if (!G || G->format != TBSLA_HIP_CSR || G->ln_row != n || G->ln_col != n ||
        G->f_row != m->f_row || G->f_col != m->f_col)
      return fail(TBSLA_HIP_ERR_INVALID, "factor G must be a CSR block of the matrix's shape");
    tbsla_hip_matrix_s *GT = o.factor_t;
    if (GT && (GT->format != TBSLA_HIP_CSR || GT->ln_row != n || GT->stored != G->stored))
      return fail(TBSLA_HIP_ERR_INVALID, "factor_t must be the CSR transpose of the factor");
  }
  const bool mixed = o.precision == TBSLA_HIP_CG_MIXED;
  const int max_it = o.max_iterations;
  if (max_it < 0) return fail(TBSLA_HIP_ERR_INVALID, "max_iterations < 0");
  if (o.spmv_passes < 0 || o.spmv_passes > 2)
    return fail(TBSLA_HIP_ERR_INVALID, "spmv_passes must be 0, 1 or 2");
  if (o.max_blocks_per_system < 0 || o.max_blocks_per_system > kMaxBlocksPerSystem)
    return fail(TBSLA_HIP_ERR_INVALID, "max_blocks_per_system must be 0..1024");
  // workgroups per system: the dot-product partials every workgroup of a
  // system reads grow with their square, which a lone system's parallelism
  // pays for and a batch's does not.  A lone system: one workgroup per 512
  // rows, 256 to 1024 (at 64^3, 512 workgroups beat 1024 and 256)
  const long long lone = std::min<long long>(kMaxBlocksPerSystem,
                                             std::max<long long>(256, n / kRowsPerBlockLone));
  const long long cap = o.max_blocks_per_system > 0 ? o.max_blocks_per_system
                        : nsys > 1                  ? kBatchBlocksPerSystem
                                                    : lone;

  if (!m->cg_cache) m->cg_cache = take_cache();
  CgCache &c = *static_cast<CgCache *>(m->cg_cache);

  // lanes per row of the iteration's SpMV: a power of two near an eighth of
  // the mean row length (rows are short in the SPD problems CG serves; one
  // lane per row lets a workgroup cover its rows in one pass)
  int L = o.lanes_per_row;
  if (L <= 0) {
    const double mean = n > 0 ? (double)m->stored / n : 1.0;
    L = 1;
    while (L < 64 && L < mean / 8) L <<= 1;
  }
  if (L < 1 || L > 64 || (L & (L - 1))) return fail(TBSLA_HIP_ERR_INVALID, "lanes_per_row");

  // workgroup layout: a workgroup covers whole passes of kBlock / L rows (one
  // pass when the system allows), at most kMaxBlocksPerSystem per system
  std::vector<CgSeg> &hs = c.host_seg;
  std::vector<int> &hb = c.host_blocks;
  hs.assign(nsys, CgSeg{});
  hb.clear();
  const long long pass_rows = kBlock / L;
  // A batch (or the same cap asked for, so that a system alone and in a batch
  // is laid out alike): at least kBlock rows per workgroup, a row per thread in
  // K2 and in the first pass of K1.  96 systems of 4,096 to 65,536 rows, L = 8:
  // 96 rows a workgroup left five threads in eight idle there (over a solve K1a
  // took 40 and K2 54 us on average, 21 and 28 so).
  const bool batch_layout = o.max_blocks_per_system > 0
                                ? o.max_blocks_per_system <= kBatchBlocksPerSystem
                                : nsys > 1;
  const long long min_rpb = batch_layout ? kBlock : pass_rows;
  for (int k = 0; k < nsys; k++) {
    const long long rows = h_rows[k + 1] - h_rows[k];
    long long rpb = std::max<long long>(min_rpb, (rows + cap - 1) / cap);
    rpb = (rpb + pass_rows - 1) / pass_rows * pass_rows;
    const int nb = (int)((rows + rpb - 1) / rpb);
    CgSeg &S = hs[k];
    S.row0 = h_rows[k];
    S.row1 = h_rows[k + 1];
    S.blk0 = (int)hb.size();
    S.blk1 = S.blk0 + nb;
    S.rpb = (int)rpb;
    S.done = (h_active && !h_active[k]) ? kInactive : kRunning;
    for (int i = 0; i < nb; i++) hb.push_back(k);
  }
  const int nblocks = (int)hb.size();
  int nactive = 0;
  for (auto &S : hs) nactive += S.done != kInactive;

  // buffers
  Buf<double> *vecs[] = {&c.b, &c.x, &c.r0, &c.r1, &c.p0, &c.p1, &c.z, &c.ap, &c.ax};
  for (auto *v : vecs) TBSLA_TRY(v->ensure((size_t)n));
  Buf<double> *parts[] = {&c.ppap, &c.prr0, &c.prr1, &c.prz0, &c.prz1};
  for (auto *v : parts) TBSLA_TRY(v->ensure((size_t)nblocks));
  const bool multi = nsys > 1;
  if (multi) TBSLA_TRY(c.seg.ensure(nsys));
  TBSLA_TRY(c.args.ensure(1));
  if (multi) TBSLA_TRY(c.block_seg.ensure(nblocks));
  if (!c.h_com) TBSLA_HIP_CHECK(hipHostMalloc((void **)&c.h_com, 2 * sizeof(CgCom), hipHostMallocDefault));
  if (!c.h_args) TBSLA_HIP_CHECK(hipHostMalloc((void **)&c.h_args, sizeof(CgBlock), hipHostMallocDefault));
  for (auto &e : c.ev)
    if (!e) TBSLA_HIP_CHECK(hipEventCreateWithFlags(&e, hipEventDisableTiming));
  if (pre == TBSLA_HIP_PRECOND_JACOBI) TBSLA_TRY(c.dinv.ensure((size_t)n));
  if (mixed) {
    const size_t need = (size_t)std::max(m->stored, 1LL);
    if (c.a_v32_len < need) {
      TBSLA_HIP_CHECK(hipStreamSynchronize(s));
      device_free(c.a_v32);
      c.a_v32 = nullptr;
      c.a_v32_len = 0;
      TBSLA_TRY(device_alloc((void **)&c.a_v32, need * 4));
      c.a_v32_len = need;
      c.a_v32_uid = 0;
    }
    if (c.a_v32_uid != m->uid || c.a_v32_ver != m->values_version) {
      if (m->stored > 0) {
        k_to_f32<<<sgrid(m->stored), kBlock, 0, s>>>(m->values, m->stored, c.a_v32);
        TBSLA_HIP_LAUNCH_CHECK();
      }
      c.a_v32_uid = m->uid;
      c.a_v32_ver = m->values_version;
    }
  }
  // M = G G^T: from G's diagonals when its entries lie on at most 8 of
  // offset <= 0 (a stencil factor; no column indices read), else from the
  // CSR rows of G and G^T
  bool gdia = false;
  int gndiag = 0;
  if (pre == TBSLA_HIP_PRECOND_FACTORED) {
    if (mixed) TBSLA_TRY(c.t32.ensure((size_t)n));
    else TBSLA_TRY(c.t64.ensure((size_t)n));
    if (o.factor_form != TBSLA_HIP_FACTOR_ROWS) {
      TBSLA_TRY(build_gdia(c, G, mixed, s, &gndiag));
      gdia = gndiag > 0;
      if (!gdia && o.factor_form == TBSLA_HIP_FACTOR_DIAGONALS)
        return fail(TBSLA_HIP_ERR_UNSUPPORTED,
                    "factor G is not held on at most 8 diagonals of offset <= 0");
    }
    if (!gdia) {
      // the transpose and the FP32 copies are rebuilt on every call (G may
      // have been rewritten in place since the last solve)
      tbsla_hip_matrix_s *GT = o.factor_t;
      if (!GT) {
        TBSLA_HIP_CHECK(hipStreamSynchronize(s));
        device_free(c.t_rp);
        device_free(c.t_ci);
        device_free(c.t_v64);
        c.t_rp = c.t_ci = nullptr;
        c.t_v64 = nullptr;
        TBSLA_TRY(csr_transpose_arrays(G, &c.t_rp, &c.t_ci, &c.t_v64, s));
      }
      if (mixed) {
        if (c.f32_len < (size_t)std::max(G->stored, 1LL)) {
          TBSLA_HIP_CHECK(hipStreamSynchronize(s));
          device_free(c.g_v32);
          device_free(c.t_v32);
          c.g_v32 = c.t_v32 = nullptr;
          c.f32_len = 0;
          TBSLA_TRY(device_alloc((void **)&c.g_v32, (size_t)std::max(G->stored, 1LL) * 4));
          TBSLA_TRY(device_alloc((void **)&c.t_v32, (size_t)std::max(G->stored, 1LL) * 4));
          c.f32_len = (size_t)std::max(G->stored, 1LL);
        }
        if (G->stored > 0) {
          k_to_f32<<<sgrid(G->stored), kBlock, 0, s>>>(G->values, G->stored, c.g_v32);
          k_to_f32<<<sgrid(G->stored), kBlock, 0, s>>>(GT ? GT->values : c.t_v64, G->stored,
                                                       c.t_v32);
          TBSLA_HIP_LAUNCH_CHECK();
        }
      }
    }
  }

  CgArgs a{};
  a.rowptr = m->rowptr;
  a.colidx = m->colidx;
  a.val64 = m->values;
  a.val32 = mixed ? c.a_v32 : nullptr;
  a.f_col = m->f_col;
  if (pre == TBSLA_HIP_PRECOND_FACTORED) {
    if (gdia) {
      a.gdoff = c.gdoff.p;
      a.gd64 = c.gd64.p;
      a.gd32 = c.gd32.p;
      a.gndiag = gndiag;
      for (int k = 0; k < 8; k++) a.gdoff8[k] = c.host_gdoff[std::min(k, gndiag - 1)];
    } else {
      a.g_rp = G->rowptr;
      a.g_ci = G->colidx;
      a.g_v64 = G->values;
      a.g_v32 = c.g_v32;
      a.t_rp = o.factor_t ? o.factor_t->rowptr : c.t_rp;
      a.t_ci = o.factor_t ? o.factor_t->colidx : c.t_ci;
      a.t_v64 = o.factor_t ? o.factor_t->values : c.t_v64;
      a.t_v32 = c.t_v32;
    }
  }
  a.dinv = c.dinv.p;
  a.b = c.b.p;
  a.x = c.x.p;
  a.r[0] = c.r0.p;
  a.r[1] = c.r1.p;
  a.p[0] = c.p0.p;
  a.p[1] = c.p1.p;
  a.z = c.z.p;
  a.ap = c.ap.p;
  a.ax = c.ax.p;
  a.t64 = c.t64.p;
  a.t32 = c.t32.p;
  a.ppap = c.ppap.p;
  a.prr[0] = c.prr0.p;
  a.prr[1] = c.prr1.p;
  a.prz[0] = c.prz0.p;
  a.prz[1] = c.prz1.p;
  a.seg = multi ? c.seg.p : &c.args.p->seg;
  a.com = &c.args.p->com;
  a.block_seg = c.block_seg.p;
  a.verify = (mixed || o.replace_every > 0) ? 1 : 0;
  a.stall_window = o.stall_window;
  a.ncol = (int)m->ln_col;
  // A in the diagonal layout with no remote entries: K1 reads its diagonals
  const int *d_off = nullptr, *h_off = nullptr;
  const double *d_v = nullptr;
  int ndiag = 0, symmetric = 0;
  long long dv_len = 0;
  unsigned long long build = 0;
  const bool dia = split_diag_only(m, &d_off, &h_off, &d_v, &ndiag, &dv_len, &build, &symmetric) && m->ln_col > 0;
  // K1 on CSR rows in two passes: asked for, or picked for large blocks,
  // whose gathers of z and p miss the caches (a random column then costs
  // one line fill instead of two)
  const bool two = !dia && (o.spmv_passes == 2 ||
                            (o.spmv_passes == 0 && m->stored >= kTwoPassEntries));
  if (dia) {
    a.doff = d_off;
    std::copy_n(h_off, std::min(ndiag, 8), a.doff8);
    a.dv64 = d_v;
    a.ndiag = ndiag;
    if (mixed) {
      if (c.dv32_len < (size_t)dv_len) {
        TBSLA_HIP_CHECK(hipStreamSynchronize(s));
        device_free(c.dv32);
        c.dv32 = nullptr;
        c.dv32_len = 0;
        TBSLA_TRY(device_alloc((void **)&c.dv32, (size_t)dv_len * 4));
        c.dv32_len = (size_t)dv_len;
        c.dv32_build = 0;
      }
      if (c.dv32_build != build) {
        k_to_f32<<<sgrid(dv_len), kBlock, 0, s>>>(d_v, dv_len, c.dv32);
        TBSLA_HIP_LAUNCH_CHECK();
        c.dv32_build = build;
      }
      a.dv32 = c.dv32;
    }
  }
  // the prefetches of K1 and K2 read entry 0 of A's and G^T's arrays even
  // when they hold none: a one-entry stand-in then (never used otherwise)
  if (!c.dummy_i.p) {
    TBSLA_TRY(c.dummy_i.ensure(1));
    TBSLA_TRY(c.dummy_d.ensure(1));
    const double zero = 0.0;
    TBSLA_HIP_CHECK(hipMemcpy(c.dummy_d.p, &zero, sizeof zero, hipMemcpyHostToDevice));
  }
  a.a_nnz = (int)std::max(m->stored, 1LL);
  if (m->stored == 0) {
    a.colidx = c.dummy_i.p;
    a.val64 = c.dummy_d.p;
    a.val32 = (const float *)c.dummy_d.p;
  }
  if (pre == TBSLA_HIP_PRECOND_FACTORED && !gdia) {
    a.g_nnz = (int)std::max(G->stored, 1LL);
    if (G->stored == 0) {
      a.g_ci = c.dummy_i.p;
      a.g_v64 = c.dummy_d.p;
      a.g_v32 = (const float *)c.dummy_d.p;
      a.t_ci = c.dummy_i.p;
      a.t_v64 = c.dummy_d.p;
      a.t_v32 = (const float *)c.dummy_d.p;
    }
  }

  Plan p;
  p.L = L;
  p.pre = pre;
  p.mixed = mixed;
  p.replace = std::max(0, o.replace_every);
  p.verify = a.verify;
  p.stall = o.stall_window;
  p.dia = dia;
  const long long most = 1LL << 32;
  const bool narrow_a = (n + kWave) * std::max(ndiag, 1) * 8 < most;
  p.dkd = dia && narrow_a && (ndiag == 3 || ndiag == 5 || ndiag == 7) ? ndiag : 0;
  p.sym = p.dkd > 0 && symmetric;
  p.wide = (n + kWave) * std::max(gndiag, 1) * 8 >= most;
  p.two = two;
  p.gdia = gdia;
  p.gkd = gndiag <= 4 ? 4 : 8;
  p.n = n;
  p.nblocks = nblocks;
  p.multi = multi ? 1 : 0;
  p.args = c.args.p;
  p.s = s;

  // upload the argument block (from its pinned copy: the stream's earlier
  // work has finished with the previous contents, see the end of the solve),
  // layout, inputs, start
  TBSLA_HIP_CHECK(hipStreamSynchronize(s));
  *c.h_args = CgBlock{a, hs[0], CgCom{}};
  const int fcol = m->f_col;
  TBSLA_HIP_CHECK(hipMemcpyAsync(c.args.p, c.h_args, sizeof(CgBlock), hipMemcpyHostToDevice, s));
  TBSLA_HIP_CHECK(hipMemcpyAsync(c.dummy_i.p, &fcol, sizeof fcol, hipMemcpyHostToDevice, s));
  if (multi) {
    TBSLA_HIP_CHECK(hipMemcpyAsync(c.seg.p, hs.data(), sizeof(CgSeg) * nsys, hipMemcpyHostToDevice, s));
    TBSLA_HIP_CHECK(hipMemcpyAsync(c.block_seg.p, hb.data(), sizeof(int) * nblocks, hipMemcpyHostToDevice, s));
  }

  TBSLA_HIP_CHECK(hipMemcpyAsync(c.b.p, d_rhs, (size_t)n * 8, hipMemcpyDeviceToDevice, s));
  // x of inactive systems stays as given; active ones start at 0 unless the
  // caller's x is the initial guess
  TBSLA_HIP_CHECK(hipMemcpyAsync(c.x.p, d_x, (size_t)n * 8, hipMemcpyDeviceToDevice, s));
  if (pre == TBSLA_HIP_PRECOND_JACOBI)
    k_csr_dinv<<<sgrid(n), kBlock, 0, s>>>(n, m->f_row, m->f_col, m->rowptr, m->colidx, m->values,
                                          c.dinv.p);
  // A x by the engine's own rows: a system alone and in a batch starts alike
  if (o.use_initial_guess) launch_ax(p, 0, kStart);
  launch_residual(p, o.use_initial_guess ? 1 : 0, 0, kStart, o.use_initial_guess ? 0 : 1);
  if (pre == TBSLA_HIP_PRECOND_FACTORED) {
    launch_gtr(p, 0, kStart);
    launch_gz(p, 0, kStart);
  }
  // The reference clamps both divisors at an absolute 1e-10 (CG.cpp:35,63,69),
  // which stalls the iteration once r.r drops below it; it is kept for the
  // reference's own setting (absolute test, FP64, no preconditioner) and
  // otherwise replaced by a guard against exact zero unless set explicitly.
  const bool reference_setting = !o.relative && !mixed && pre == TBSLA_HIP_PRECOND_NONE;
  const double near_zero = o.near_zero > 0 ? o.near_zero
                           : (o.near_zero < 0 ? 1e-300 : (reference_setting ? kNearZero : 1e-300));
  k_cg_start<<<nblocks, kBlock, 0, s>>>(p.args, p.multi, o.tolerance, o.relative, near_zero);
  TBSLA_HIP_LAUNCH_CHECK();

  // Graph batches of B iterations starting at 1 + tB (B even, so every
  // node's iteration parity is fixed): variant 0 without a replacement
  // step, variant 1 whose last iteration (a multiple of replace_every) has
  // one.  B: 16, or the largest even divisor of replace_every up to 16.
  int B = 0;
  if (o.graph_batch >= 0) {
    B = o.graph_batch > 0 ? o.graph_batch : 16;
    if (p.replace > 0) {
      B = 0;
      for (int d = 2; d <= 16; d += 2)
        if (p.replace % d == 0) B = d;
    }
    if (B % 2) B = 0;
  }
  int it = 0;  // next global iteration to enqueue
  if (max_it > 0) {
    enqueue_iteration(p, 0, false);
    it = 1;
  }
  GraphKey key{};
  key.L = p.L;
  key.pre = pre;
  key.mixed = mixed;
  key.replace = p.replace;
  key.batch = B;
  key.nblocks = nblocks;
  key.multi = p.multi;
  key.verify = p.verify;
  key.dia = p.dia ? 1 + p.dkd + (p.sym ? 10 : 0) : 0;
  key.gdia = p.gdia ? p.gkd + (p.wide ? 16 : 0) : 0;
  key.two = p.two ? 1 : 0;
  // the graph set of this plan, captured and instantiated once; the least
  // recently used set is destroyed when kGraphSets are held (the stream is
  // idle between solves, so no set is in flight then)
  CgCache::GraphSet *gs = nullptr;
  if (B > 0) {
    size_t pos = c.graphs.size();
    for (size_t q = 0; q < c.graphs.size(); q++)
      if (c.graphs[q].key == key) {
        pos = q;
        break;
      }
    if (pos == c.graphs.size()) {
      const int variants = p.replace > 0 ? 2 : 1;
      CgCache::GraphSet fresh;
      fresh.key = key;
      for (int v = 0; v < variants; v++) {
        // variant v: iterations 1..B; with v == 1 the last one replaces (its
        // index is taken as a multiple of replace_every of the same parity)
        hipGraph_t graph = nullptr;
        hipError_t e = hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal);
        if (e == hipSuccess) {
          for (int k = 0; k < B; k++) {
            const bool last = k == B - 1;
            enqueue_iteration(p, (v == 1 && last) ? B * p.replace : 1 + k, false);
          }
          e = hipStreamEndCapture(s, &graph);
        }
        if (e == hipSuccess) e = hipGraphInstantiate(&fresh.exec[v], graph, nullptr, nullptr, 0);
        if (graph) (void)hipGraphDestroy(graph);
        if (e != hipSuccess) {
          fresh.destroy();  // no partial set is ever kept
          return fail(TBSLA_HIP_ERR_HIP, std::string("graph capture: ") + hipGetErrorString(e));
        }
      }
      if (c.graphs.size() == CgCache::kGraphSets) {
        c.graphs.back().destroy();
        c.graphs.pop_back();
      }
      c.graphs.insert(c.graphs.begin(), fresh);
    } else if (pos != 0) {
      CgCache::GraphSet moved = c.graphs[pos];
      c.graphs.erase(c.graphs.begin() + (long)pos);
      c.graphs.insert(c.graphs.begin(), moved);
    }
    gs = &c.graphs.front();
  }
  const int poll_every = B > 0 ? B : 16;

  // main loop: one batch in flight, status polled from pinned copies.
  // Graph batches start at iterations 1 + kB; direct launches only for the
  // tail (or when no graph is used).
  int batches = 0;
  bool finished = false;
  // settle waiting systems after a batch (a replacement step does): a lone
  // system's batches leave that out while its residual, by its decay over the last
  // batch, is more than three batches from the threshold (five kernels that find
  // nothing to do: 30 of 455 us a batch at 10^6 rows, mixed, factored).  Were it
  // to get there sooner, the status of that batch would tell.  The batch then in
  // flight finds it waiting and does nothing, so that batch is taken back: the
  // iterations are numbered, and end at max_it, as if it had been settled at once.
  bool near = true;
  bool left_out[2] = {false, false};  // of the batch behind each status copy
  double ratio = 0.0;
  while (it < max_it && !finished) {
    const int slot = batches & 1;
    left_out[slot] = false;
    if (B > 0 && it + B <= max_it) {
      const int last = it + B - 1;  // the batch's last iteration
      const bool rep = p.replace > 0 && last % p.replace == 0;
      TBSLA_HIP_CHECK(hipGraphLaunch(gs->exec[rep ? 1 : 0], s));
      // only a whole batch can be taken back: one comes after
      left_out[slot] = p.verify && !rep && !near && it + 2 * B <= max_it;
      if (p.verify && !rep && !left_out[slot]) {
        true_residual(p, last & 1, kVerify);
        k_cg_vcheck<<<nblocks, kBlock, 0, s>>>(p.args, p.multi, (last + 1) & 1);
      }
      it += B;
    } else {
      const int stop = std::min(max_it, it + poll_every);
      for (; it < stop; it++) enqueue_iteration(p, it, it == stop - 1);
    }
    TBSLA_HIP_LAUNCH_CHECK();
    TBSLA_HIP_CHECK(hipMemcpyAsync(c.h_com + slot, a.com, sizeof(CgCom), hipMemcpyDeviceToHost, s));
    TBSLA_HIP_CHECK(hipEventRecord(c.ev[slot], s));
    if (batches > 0) {
      const int prev = slot ^ 1;
      TBSLA_HIP_CHECK(hipEventSynchronize(c.ev[prev]));
      const CgCom h = c.h_com[prev];
      if (h.npending > 0 && p.verify) {
        if (left_out[prev]) {
          it -= B;
          left_out[slot] = false;  // settled here
        }
        true_residual(p, 0, kVerify);
        k_cg_vcheck<<<nblocks, kBlock, 0, s>>>(p.args, p.multi, it);
        TBSLA_HIP_LAUNCH_CHECK();
      }
      if (h.ndone >= nactive) finished = true;
      const double decay = std::max(ratio / h.ratio, 1.0);
      near = multi || !(ratio > 0 && h.ratio > 4 * decay * decay * decay);
      ratio = h.ratio;
    }
    batches++;
  }
  TBSLA_HIP_CHECK(hipStreamSynchronize(s));
  CgCom h{};
  TBSLA_HIP_CHECK(hipMemcpy(&h, a.com, sizeof h, hipMemcpyDeviceToHost));
  if (h.ndone < nactive) {
    // the final test after the last iteration (CG.cpp:66-72), then the
    // true residual of systems whose recurrence converged
    if (max_it > 0) launch_k1_any(p, it & 1, 1, 1);
    if (p.verify) {
      true_residual(p, 0, kVerify);
      k_cg_vcheck<<<nblocks, kBlock, 0, s>>>(p.args, p.multi, it);
    }
    TBSLA_HIP_LAUNCH_CHECK();
  }
  TBSLA_HIP_CHECK(hipMemcpyAsync(d_x, c.x.p, (size_t)n * 8, hipMemcpyDeviceToDevice, s));
  TBSLA_HIP_CHECK(hipMemcpyAsync(hs.data(), a.seg, sizeof(CgSeg) * nsys, hipMemcpyDeviceToHost, s));
  TBSLA_HIP_CHECK(hipMemcpyAsync(&h, a.com, sizeof h, hipMemcpyDeviceToHost, s));
  TBSLA_HIP_CHECK(hipStreamSynchronize(s));
  int dev = 0, khz = 0;
  (void)hipGetDevice(&dev);
  (void)hipDeviceGetAttribute(&khz, hipDeviceAttributeWallClockRate, dev);
  for (int k = 0; k < nsys; k++) {
    const CgSeg &S = hs[k];
    tbsla_hip_cg_result &r = res[k];
    r.iterations = S.iters;
    r.res_norm = S.rnorm;
    r.status = S.done == kConverged ? TBSLA_HIP_CG_CONVERGED
               : S.done == kBreakdown ? TBSLA_HIP_CG_BREAKDOWN
               : S.done == kInactive  ? TBSLA_HIP_CG_INACTIVE
                                      : TBSLA_HIP_CG_MAX_ITERATIONS;
    r.time_us = (S.t_done > 0 && khz > 0) ? (double)(S.t_done - h.t0) * 1000.0 / khz : -1.0;
  }
  return TBSLA_HIP_SUCCESS;
}

}  // namespace tbsla_hip

using namespace tbsla_hip;

extern "C" int tbsla_hip_cg(tbsla_hip_matrix_t m, const double *d_rhs, double *d_x,
                            const tbsla_hip_cg_options *opt, int *nb_iterations,
                            double *res_norm, void *stream) {
  if (!m || !d_rhs || !d_x) return fail(TBSLA_HIP_ERR_INVALID, "null argument");
  tbsla_hip_cg_options o{};
  o.max_iterations = 10000;
  o.tolerance = 1.0e-10;  // CG.cpp:34
  if (opt) o = *opt;
  const int rows[2] = {0, m->ln_row};
  if (m->ln_row < 1) return fail(TBSLA_HIP_ERR_INVALID, "empty block");
  tbsla_hip_cg_result r{};
  TBSLA_TRY(cg_solve(m, 1, rows, nullptr, d_rhs, d_x, o, &r, static_cast<hipStream_t>(stream)));
  if (nb_iterations) *nb_iterations = r.iterations;
  if (res_norm) *res_norm = r.res_norm;
  if (r.status == TBSLA_HIP_CG_BREAKDOWN)
    return fail(TBSLA_HIP_ERR_BREAKDOWN, "CG breakdown (r.z <= 0, non-finite, or no progress)");
  return TBSLA_HIP_SUCCESS;
}

extern "C" int tbsla_hip_cg_batched(tbsla_hip_matrix_t m, int nsys, const int *h_row_offsets,
                                    const int *h_active, const double *d_rhs, double *d_x,
                                    const tbsla_hip_cg_options *opt,
                                    tbsla_hip_cg_result *h_results, void *stream) {
  if (!m || !h_row_offsets || !d_rhs || !d_x || !h_results || nsys < 1)
    return fail(TBSLA_HIP_ERR_INVALID, "null argument");
  tbsla_hip_cg_options o{};
  o.max_iterations = 10000;
  o.tolerance = 1.0e-10;
  if (opt) o = *opt;
  return cg_solve(m, nsys, h_row_offsets, h_active, d_rhs, d_x, o, h_results,
                  static_cast<hipStream_t>(stream));
}
