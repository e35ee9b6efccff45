// Internal launchers of the HIP kernels (host-callable, stream-ordered).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace tcx {

constexpr int kModeAssign = 0;
constexpr int kModeNcc = 1;
constexpr int kModeOwn = 2;
// assign in place of the pruned search: as there, pairs of series without a
// finite norm and such centroids have no distance (label 0, INFINITY, the first
// lag), and an all-zero centroid is at distance 1 of both series of any other
// pair
constexpr int kModeSearch = 3;

struct SbdArgs {
  const float* x = nullptr;      // [n][m] series
  long n = 0;
  int m = 0;
  int k = 0;                     // centroids (assign) or y rows (ncc)
  const float2* cspec = nullptr; // [k][F] lane-strided spectra
  const float* cnorm = nullptr;  // [k]
  const float2* tw = nullptr;    // [F] exp(-2 pi i q / F)
  int rev = 0;                   // 1: k-Shape lag order
  int* label = nullptr;          // required (assign), may be NULL (own)
  float* dist = nullptr;
  int* shift = nullptr;
  float* dmat = nullptr;
  int* changed = nullptr;
  float* ncc_out = nullptr;
  const int* fixed_label = nullptr;  // own: the centroid of each series
  // centroids split into this many chunks over the grid (sbd_chunks); assign
  // with more than one also needs the chunk results, [chunks][n] each
  int chunks = 1;
  float* part_dist = nullptr;
  int* part_label = nullptr;
  int* part_shift = nullptr;
  int cus = 0;                   // compute units of the device
  const int* skip = nullptr;     // assign: nothing is done when *skip (may be NULL)
};

// largest supported FFT length (m <= 4096)
constexpr int kMaxFft = 8192;

hipError_t launch_znorm(float* x, long rows, int m, int ddof, hipStream_t st);
// Twiddle table (F entries) of the length-F transform, host side.
void fft_twiddle_table(int F, float2* out);
// bmag (may be NULL): rows (bound_rows(rows) x bound_kpad(F), fragment
// order) of |Y[f]| / |y| for f <= F/2, zero padded, as IEEE binary16 bits
// rounded up (the centroid operand of launch_bounds).
hipError_t launch_spectra(int F, const float* y, int rows, int m, const float2* tw,
                          float2* spec, float* norms, int* zero, float* mag, uint16_t* bmag,
                          hipStream_t st);

// Exact pruned assignment (bound-and-prune on the spectra), k <= kPruneMaxK.
constexpr int kPruneMaxK = 1024;
constexpr int kLdsBytes = 160 * 1024;  // LDS of one workgroup on gfx950
// Largest k the pruned assignment takes at FFT length F (LDS-bound).
int prune_max_k(int F);
// Columns of a series' bound row (launch_series_spec's xm): F/2+1
// magnitudes padded to a multiple of 16 (the bound product's K step).
__host__ __device__ constexpr int bound_kpad(int F) { return ((F / 2 + 1) + 15) & ~15; }
// Bound rows are IEEE binary16 values in MFMA fragment order: the 16 x 16
// block of rows 16 b .. 16 b + 15 and columns 16 s .. 16 s + 15 is 256
// consecutive values, element (r, c) at 4 (r + 16 (c / 4)) + c % 4, so that
// lane l of a wave reads its operand of v_mfma_f32_16x16x16_f16 (row l % 16,
// columns 4 (l / 16) .. + 3) as the l-th 8-byte vector of the block.  Rows
// are padded to a multiple of 16.
__host__ __device__ constexpr long bound_frag(long row, int f, int kpad) {
  return (((row >> 4) * (kpad >> 4) + (f >> 4)) * 64 + (row & 15) + 16 * ((f & 15) >> 2)) * 4 +
         (f & 3);
}
__host__ __device__ constexpr long bound_rows(long rows) { return (rows + 15) & ~15L; }
// The count of inverse transforms is spread over kEvalSlots counters of a
// 128-byte line each (the sum counts).  One counter took 10 ns per wave, one
// wave after the other, which the kernel waited for: fit of ten iterations
// n=100000 m=512 k=16 9030 us with one, 8420 now, 64 uneven jobs at once 66 and
// 62 ms.
constexpr int kEvalSlots = 16, kEvalStride = 128 / sizeof(unsigned long long);
constexpr size_t kEvalBytes = 128 * kEvalSlots;
inline unsigned long long eval_sum(const void* counters) {
  unsigned long long s = 0;
  for (int i = 0; i < kEvalSlots; ++i)
    s += static_cast<const unsigned long long*>(counters)[i * kEvalStride];
  return s;
}

struct PruneArgs {
  const float* x = nullptr;
  const float2* xs = nullptr;    // per-series half spectra [n][F/2+1] (may be NULL: from x)
  const float* xn = nullptr;     // per-series norms (with xs)
  const float* ub = nullptr;     // per-series bounds [n][ub_ld] of launch_bounds (with xs)
  int ub_ld = 0;
  long n = 0;
  long npairs = 0;               // pairs of order[] (or ceil(n/2) without order)
  int m = 0, k = 0;
  const float2* cspec = nullptr;
  const float* cmag = nullptr;   // |C| in the spectrum layout
  const float* cnorm = nullptr;
  const float2* tw = nullptr;
  int rev = 0;
  const int* order = nullptr;    // 2*npairs row indices, -1 = hole (may be NULL)
  int* label = nullptr;
  float* dist = nullptr;
  int* shift = nullptr;
  int* changed = nullptr;
  unsigned long long* evals = nullptr;  // inverse transforms run, kEvalSlots counters (may be NULL)
  const int* skip = nullptr;     // nothing is done when *skip (may be NULL)
  int cus = 0;                   // compute units of the device
};
hipError_t launch_assign_prune(int F, const PruneArgs& a, hipStream_t st);
// Half spectra X_r[0 .. F/2] of every row and the row norms (k_series_spec);
// with xm (may be NULL) also the bound rows (bound_rows(n) x bound_kpad(F),
// fragment order, binary16 rounded up): weight_f |X_r[f]| / |x_r|, weight 2
// for 0 < f < F/2, zero padded.
hipError_t launch_series_spec(int F, const float* x, long n, int m, const float2* tw, float2* xs,
                              float* xn, uint16_t* xm, hipStream_t st);
// ub[i][j] = sum_f xm[i][f] cm[j][f] / F (cm: launch_spectra's bmag rows),
// i < n, j < k, row stride ld >= k: the pruned assignment's bounds
// (k_bounds).  Both operands are rounded up, so ub is never below the
// product of the FP32 magnitudes.
hipError_t launch_bounds(int F, const uint16_t* xm, long n, const uint16_t* cm, int k, float* ub,
                         int ld, hipStream_t st);
hipError_t launch_sbd(int F, int mode, const SbdArgs& a, hipStream_t st);
// Chunks the centroids of n series are worth splitting into (1: none); merge:
// the merge of the chunk results is to be paid for (by all distances, which the
// unsplit kernel gives as well).
int sbd_chunks(int F, long n, int k, int cus, bool merge);
// Shifts each row in place by the lag of its largest NCC with one centroid
// (spectrum, norm and all-zero flag given; an all-zero one changes nothing).
hipError_t launch_align(int F, float* x, long n, int m, const float2* cspec, const float* cnorm,
                        const int* czero, const float2* tw, int rev, hipStream_t st);
hipError_t configure_sbd_kernels();

// ------------------------------------------------------------ extraction
constexpr int kGroupChunk = 512;  // rows per grouping block
constexpr int kPackPad = 64;       // cluster segments padded to this many columns
constexpr int kSyrkTile = 256;     // panel rows are padded to a multiple of this
constexpr int kSyrkSub = 128;      // S block edge (one wave)

// The packed panel Y (time t x packed column p, BF16 hi and lo parts) is
// stored in MFMA operand order: chunk (c = p / 16, r = t / 32) holds 512
// values at element offset (c * panel_blocks(m) + r) * 512, value (t, p) at
// ((t % 32) + 32 * ((p / 8) % 2)) * 8 + p % 8 inside it.  Rows run to a
// multiple of kSyrkTile, rows t >= m are zero.
__host__ __device__ constexpr int panel_blocks(int m) {
  return (m + kSyrkTile - 1) / kSyrkTile * (kSyrkTile / 32);
}

// A work item of S = Y^T Y (grouped executor): one kSyrkSub block of S_j
// (one wave) over a packed column range.
struct SyrkItem {
  int cluster;
  int ti, tj;         // block row and column (ti <= tj)
  int part;           // index of this item's partial
  long p0, p1;        // packed column range [p0, p1), multiples of 16
};

// A kSyrkSub block of S_j and its K-chunk partials.
struct SyrkTile {
  int cluster;
  int ti, tj;
  int part0, nparts;  // partials part0 .. part0+nparts-1, summed in order
};

// A (cluster, K chunk) group of the single fit's S = Y^T Y: the upper
// triangle of kSyrkSub blocks of S_j (row-major order) over the packed
// columns [p0, p1); block u's partial is part + u * stride.
struct SyrkGroup {
  int part, stride;
  long p0, p1;        // multiples of 16
};

// A cluster of the single fit with partials: block u of S_j sums the
// nparts partials from part0 + u * nparts on, in order.
struct SyrkCluster {
  int cluster, part0, nparts;
};
struct SyrkPlanHead {
  int ngroups, nclusters;  // clusters: those with members
};
constexpr int kSyrkMinSteps = 16;  // 16-column steps of a K chunk, at least
int syrk_max_groups(int m, int cus);  // groups of one round of the device

struct PowerInfo {
  double lambda;
  int steps;
  int converged;
  int fallback;
  int flipped;
  int zero;           // power iteration hit M v = 0 (NaN path, zero centroid)
  int empty;
};

hipError_t launch_fill_int(int* p, long count, int value, hipStream_t st);
// Grouping by the key label * B + bin(dist) (see k_group_count): bins per
// cluster for n rows and k clusters, 1 without distances or for large k.
constexpr int kGroupBins = 64;
constexpr long kGroupMaxBlkKeys = 32L << 20;  // per-block key counts kept (ints)
int group_bins(long n, int k, bool have_dist);
hipError_t launch_group_count(const int* label, long n, int k, const float* dist, int B,
                              int* blk_count, int* minrow, int* bad, hipStream_t st);
hipError_t launch_group_scan(int nblk, int k, int B, const int* blk_count, int* blk_base,
                             int* kcounts, int* counts, long* offsets, long* koff,
                             hipStream_t st);
hipError_t launch_group_place(const int* label, long n, int k, const float* dist, int B,
                              const int* blk_base, const long* koff, int* perm, hipStream_t st);
// FP64 (sum, sum of squares) of every row.
hipError_t launch_row_stats(const float* x, long rows, int m, double2* stats, hipStream_t st);
// True when launch_align_pack reads per-row sums (launch_row_stats) for
// this m; otherwise `stats` may be NULL.
bool align_pack_uses_row_stats(int m);
hipError_t launch_align_pack(const float* x, int m, const int* perm, long n_pad,
                             const long* offsets, const int* minrow, int k, const int* shift,
                             const int* czero, const double2* stats, int cus, uint16_t* yhi,
                             uint16_t* ylo, float* a0, hipStream_t st);
// Single fit: blocks of k_syrk for ngroups groups (each group's waves on
// one XCD), the launch over the groups, and the reduction of the clusters'
// kSyrkSub x kSyrkSub partials into S.
long syrk_blocks(int m, int ngroups);
// The first kRefineStatusInts ints of a refinement's status zeroed, minrow
// INT_MAX, perm -1.
constexpr int kRefineStatusInts = (kEvalBytes + 256) / sizeof(int);
hipError_t launch_refine_init(int* status, int* minrow, int k, int* perm, long n_pad,
                              hipStream_t st);
// The plan of S from the clusters' sizes on the device.
hipError_t launch_syrk_plan(const long* offsets, const int* counts, int m, int k, int cus,
                            SyrkPlanHead* head, SyrkGroup* groups, SyrkCluster* clusters,
                            hipStream_t st);
// max_groups, max_clusters: at least the plan's counts (the grid's size).
hipError_t launch_syrk(const SyrkGroup* groups, const SyrkPlanHead* head, int max_groups,
                       const uint16_t* yhi, const uint16_t* ylo, int m, int split, float* part,
                       hipStream_t st);
hipError_t launch_syrk_reduce(const SyrkCluster* clusters, const SyrkPlanHead* head,
                              int max_clusters, const float* part, int m, float* S,
                              hipStream_t st);
// redo (may be NULL): set to 1 when a cluster failed its tests and
// defer_fallback left it to the caller.
hipError_t launch_power(const float* S, int m, int k, const int* counts, const float* a0,
                        uint64_t seed, int iter, int max_steps, double tol, const double* vin,
                        const double* svin, const double* rsum, const int* steps_in,
                        const int* conv_in, int eig_mode, const int* mask, int defer_fallback,
                        float* c_out, PowerInfo* info, int* redo, hipStream_t st);

// Lanczos evaluation of the power iterate M^I v0 (one block per cluster).
// Lanczos evaluation of the power iterate (one step = two launches).
constexpr int kLanczosMax = 128;
struct LzState {
  double sigma;                   // 1^T S 1
  double alpha[kLanczosMax + 1];  // tridiagonal T: diagonal
  double beta[kLanczosMax + 1];   // off-diagonal, beta[l] = T[l][l-1]
  double y[kLanczosMax];          // T^I e1 / |T^I e1| at the last check
  int it;                         // index of the newest basis vector
  int len;                        // steps done
  int prev_len;                   // len at the last check
  int conv;                       // accepted
  int done;                       // finished (accepted, breakdown or cap)
};
// Fused single-launch form (one block per cluster, for small m).
constexpr int kFusedLanczosMaxM = 768;
// Acceptance of the Lanczos evaluation of M^I v0: y = T_j^I e1 is formed at
// j = kLzFirstCheck and every kLzCheckEvery steps after, and accepted when
// it moved by <= kLzPowerTol since the previous check.  For a geometric
// convergence rate rho per step the accepted y is then within about
// rho^4 / (1 - rho^4) * kLzPowerTol of the limit.  S itself, in FP32 from
// split-BF16 products, leaves the centroids about 2e-6 (relative L2) from
// the FP64 oracle's at n=100000, m=512, k=16; 1e-7 leaves that and the SBD
// error unchanged (1e-9 needed 28 steps there, 1e-7 needs 24).
constexpr int kLzFirstCheck = 12;
constexpr int kLzCheckEvery = 4;
constexpr double kLzPowerTol = 1e-7;
__host__ __device__ constexpr bool lz_power_check(int len) {
  return len >= kLzFirstCheck && len % kLzCheckEvery == 0;
}

// Lanczos with G blocks per cluster in one launch (members exchange through
// device-scope memory and wait for each other, so all k*G blocks must be
// resident at once).  Used for m > kLzMultiMaxM when the plan fits, and for
// 512 < m <= 640 where it holds every cluster and plan_lz_multi needs several
// launches.
constexpr int kLzCoopMinM = 256;
constexpr int kLzCoopMaxR = 64;   // rows of S per member
constexpr int kLzCoopMaxG = 64;   // members per cluster
constexpr int kLzCoopMaxM = kLzCoopMaxR * kLzCoopMaxG;
constexpr size_t kLzCoopSLdsBytes = 96 * 1024;  // S rows kept in LDS up to this size
constexpr size_t kLzCoopLdsMax = 160 * 1024;    // LDS of one CU
struct LzCoopPlan {
  int G = 0, R = 0, nb = 0;  // members per cluster, rows per member, blocks
  bool s_lds = false;
  size_t lds = 0;            // dynamic LDS bytes per block
  long xch_len = 0;          // exchange words per cluster
  int form = 0;              // k_lz_multi's register split
  int per = 0;               // clusters of one of its launches
};
// Bytes of the exchange and failure words of k clusters, at most.
inline size_t lz_xch_bound(int m, int k) {
  const size_t words = 2 * (2 * (size_t)kLzCoopMaxG * (kLanczosMax + 2) + (size_t)m) + kLzCoopMaxG;
  return 8 * (size_t)k * words + 4 * ((size_t)k + 1);
}
// False when m, k or the device do not allow every member to be resident.
bool plan_lz_coop(int m, int k, int cus, LzCoopPlan* p);
// xch: k * p.xch_len words and fails: k words, zero when first used; gen:
// launch generation, 1 <= gen < kLzCoopMaxGen, different from every earlier
// launch on the same buffers since they were zeroed.  timeout: wall-clock
// ticks a member waits for the others.
constexpr uint32_t kLzCoopMaxGen = 1u << 22;
hipError_t launch_lz_coop(const LzCoopPlan& p, const float* S, int m, int k, const int* counts,
                          uint64_t seed, int iter, int I, double lz_tol, uint64_t* xch,
                          uint32_t* fails, uint32_t gen, long long timeout, double* vout,
                          double* rout, int* steps_out, int* conv_out, hipStream_t st);
// The same with one exchange per step and the rows of S in registers
// (k_lz_multi; S v written too, Q: (kLanczosMax + 1) x m per cluster for basis
// rows past those in LDS), for kLzResMaxD < m <= kLzMultiMaxM, p.per clusters
// per launch: here the k <= p.per from j0 on (S to conv_out are those of cluster
// 0, xch and fails of this launch).
constexpr int kLzMultiMaxM = 1024;
bool plan_lz_multi(int m, int k, int cus, LzCoopPlan* p);
hipError_t launch_lz_multi(const LzCoopPlan& p, const float* S, int m, int j0, int k,
                           const int* counts,
                           uint64_t seed, int iter, int I, double lz_tol, double* Q,
                           uint64_t* xch, uint32_t* fails, uint32_t gen, long long timeout,
                           double* vout, double* svout, double* rout, int* steps_out,
                           int* conv_out, hipStream_t st);
hipError_t launch_power_lanczos(const float* S, int m, int k, const int* counts, uint64_t seed,
                                int iter, int I, double lz_tol, double* Q, double* vout,
                                double* rout, int* steps_out, int* conv_out, hipStream_t st);
hipError_t launch_cluster_matvec(const float* S, int m, int k, const double* x, long xstride,
                                 double* y, const LzState* state, hipStream_t st);
// mask (may be NULL): clusters to run; others are left done.
hipError_t launch_lz_setup(int m, int k, const int* counts, const int* mask, uint64_t seed,
                           int iter, const double* rbuf, double* Q, LzState* state,
                           hipStream_t st);
// mode 0: power iterate M^I v0; mode 1: top eigenvector of M (tol on the
// Ritz residual relative to the Ritz value).
hipError_t launch_lz_step(int m, int k, int mode, int I, double lz_tol, const double* rbuf,
                          const double* wbuf, double* Q, LzState* state, hipStream_t st);
hipError_t launch_lz_finish(int m, int k, const int* counts, const double* Q,
                            const LzState* state, double* vout, int* steps_out, int* conv_out,
                            hipStream_t st);
hipError_t configure_extract_kernels();

// ----------------------------------------------------- grouped launches
// One launch runs a kernel's body for many independent jobs (the fits of a
// batch): job j owns the blocks [first[j], first[j+1]) of the grid and runs
// them as blocks 0 .. first[j+1] - first[j] - 1 of a launch of its own, so a
// job's results do not depend on the other jobs of the launch.  `jobs` and
// `first` are device arrays (njobs entries, njobs + 1 prefix values).
struct GroupTable {
  const void* jobs = nullptr;  // device array of the kernel's job struct
  const int* first = nullptr;  // device prefix of blocks per job
  int njobs = 0;
  int blocks = 0;              // first[njobs]
  size_t lds = 0;              // dynamic LDS of the launch (largest job's)
};

struct FillSeg {  // p[0 .. count) = value
  int* p;
  long count;
  int value;
};
hipError_t launch_fill_segs(const FillSeg* segs, int nseg, long max_count, hipStream_t st);

struct ZnormJob {
  float* x;
  long rows;
  int m, ddof;
};
// Rows of every job z-normalized, jobs in groups by znorm_form: 0 the three
// passes (m > 4096), else the 16-byte vectors per lane (1: 16 lanes per row),
// negative with a tail for rows that are no whole aligned vectors.
hipError_t launch_znorm_group(const GroupTable& g, int form, hipStream_t st);
int znorm_form(const float* x, int m);  // form of launch_znorm for these rows
long znorm_blocks(int form, long rows);
long row_stats_blocks(long rows);

struct SeriesSpecJob {
  const float* x;
  long n;
  int m;
  float2* xs;
  float* xn;
  uint16_t* xm;
};
long series_spec_blocks(int F, long n);
hipError_t launch_series_spec_group(int F, const GroupTable& g, const float2* tw, hipStream_t st);

struct SpectraJob {
  const float* y;
  int rows, m;
  float2* spec;
  float* norms;
  int* zero;
  float* mag;
  uint16_t* bmag;
};
long spectra_blocks(int F, long rows);
hipError_t launch_spectra_group(int F, const GroupTable& g, const float2* tw, hipStream_t st);

struct BoundsJob {
  const uint16_t* xm;
  long n;
  const uint16_t* cm;
  int k, ld;
  float* ub;
};
// Bound-product kernel form for (F, k): 0..4; blocks of a job of n rows.
int bounds_form(int F, int k);
long bounds_blocks(int form, long n);
hipError_t launch_bounds_group(int F, int form, const GroupTable& g, hipStream_t st);

struct PruneJob {
  const float* x;
  const float2* xs;
  const float* xn;
  const float* ub;
  int ub_ld;
  long n, npairs;
  int m, k;
  const float2* cspec;
  const float* cmag;
  const float* cnorm;
  int rev;
  const int* order;
  int* label;
  float* dist;
  int* shift;
  int* changed;
  unsigned long long* evals;  // kEvalSlots counters
  const long* npad;  // may be NULL; else npairs = *npad / 2, read on the device
};
long prune_blocks(int F, long npairs, int k, long n);  // grid cap tuned per (F, k, n)
size_t prune_lds(int F, int k);
hipError_t launch_assign_prune_group(int F, const GroupTable& g, const float2* tw, hipStream_t st);

struct GroupCountJob {
  const int* label;
  long n;
  int k;
  const float* dist;
  int B;
  int* blk_count;
  int* minrow;
  int lds_min;
  int* bad;
};
size_t group_count_lds(int k, int B, int* lds_min);
hipError_t launch_group_count_group(const GroupTable& g, hipStream_t st);

struct GroupScanJob {
  int nrowblk, K;
  const int* blk_count;
  int* blk_base;
  int* counts;
};
hipError_t launch_group_scan_group(const GroupTable& g, hipStream_t st);

struct GroupOffsetsJob {
  int k, B;
  const int* kcounts;
  int* counts;
  long* offsets;
  long* koff;
};
hipError_t launch_group_offsets_group(const GroupTable& g, hipStream_t st);

struct GroupPlaceJob {
  const int* label;
  long n;
  int k;
  const float* dist;
  int B;
  const int* blk_base;
  const long* koff;
  int* perm;
};
size_t group_place_lds(int k, int B);
hipError_t launch_group_place_group(const GroupTable& g, hipStream_t st);

struct RowStatsJob {
  const float* x;
  long rows;
  int m;
  double2* stats;
};
hipError_t launch_row_stats_group(const GroupTable& g, hipStream_t st);

struct AlignPackJob {
  const float* x;
  int m;
  const int* perm;
  long n_pad;
  const long* offsets;
  const int* minrow;
  int k;
  const int* shift;
  const int* czero;
  const double2* stats;
  uint16_t* yhi;
  uint16_t* ylo;
  float* a0;
};
// Align + pack form for m: R = 16, 32, 64 (rows staged in LDS) or 0 (from
// HBM with per-row sums, m > 1024); columns per block; dynamic LDS bytes.
int align_pack_form(int m);
long align_pack_cols(int form);
size_t align_pack_lds(int form, int m);
hipError_t launch_align_pack_group(int form, const GroupTable& g, hipStream_t st);

// S = Y^T Y of many jobs: one item (tile) per block, the job's panels,
// length and partials from syrk_jobs[job].
struct SyrkJob {
  const uint16_t* yhi;
  const uint16_t* ylo;
  int m;
  float* part;
  float* S;
};
struct GroupSyrkItem {
  int job;
  SyrkItem it;
};
struct GroupSyrkTile {
  int job;
  SyrkTile t;
};
hipError_t launch_syrk_group(const SyrkJob* jobs, const GroupSyrkItem* items, int nitems,
                             int split, hipStream_t st);
hipError_t launch_syrk_reduce_group(const SyrkJob* jobs, const GroupSyrkTile* tiles,
                                    int ntiles, hipStream_t st);

// Gram form of thin clusters (segment nd < m, nd <= kGramMaxND, m <=
// kGramMaxM): G = Yc Yc^T in 64 x 64 tiles (the diagonal ones also form
// the start u0 = Yc v0), the Lanczos stage on G, and the map back to
// v = Yc^T g, M v = Yc^T h.  One item or job per block.
constexpr int kGramMaxM = 4096;
constexpr int kGramMaxND = 2048;
struct GramItem {
  const uint16_t* yhi;
  const uint16_t* ylo;
  float* G;  // n x n, row stride n
  long p0;   // first packed column of the cluster (multiple of 64)
  int m, nd, n, ti, tj;  // segment nd (multiple of 64), members n (<= nd)
  // diagonal tiles also form the start u0 = Yc v0 of their 64 members
  // (u0 NULL: not this tile), v0 = power_v0(seed, iter, cluster, .)
  double* u0;
  uint64_t seed;
  int iter, cluster;
};
struct GramVecJob {  // the map back of one thin cluster
  const uint16_t* yhi;
  const uint16_t* ylo;
  long p0;
  int m, nd, n;
  const double* g;    // g (n)
  const double* h;    // h (n; may be sv: read before sv is written)
  double* v;          // m
  double* sv;         // M v (m)
  double* r;          // zeros (m)
};
struct GramLzJob {
  const float* G;
  int nd, I;
  const double* u0;
  double* Q;
  double* g;
  double* h;
  int* steps;
  int* conv;
};
hipError_t launch_gram_tiles(const GramItem* items, int nitems, hipStream_t st);
size_t gram_map_lds(int m, int nd);
size_t gram_lanczos_lds(int nd);
hipError_t launch_gram_lanczos(const GramLzJob* jobs, int njobs, size_t lds, double lz_tol,
                               hipStream_t st);
hipError_t launch_gram_map(const GramVecJob* jobs, int njobs, size_t lds, hipStream_t st);

// Resident Lanczos for orders d <= kLzResMaxD: one block per cluster, the
// matrix in registers (k_lz_res).  S form: M = P S P from power_v0, v =
// M^I v0, h = S v, r = S 1.  Gram form: no centring, start vstart, v =
// S^I vstart / |.|, h = S v.
constexpr int kLzResMaxD = 256;
struct LzResJob {
  const float* S;  // d x d, row stride d
  int d, gram, I;
  uint64_t seed;
  int iter, cluster;
  const double* vstart;  // Gram form
  double* Q;             // (kLanczosMax + 1) x d: basis rows past those in LDS
  double* v;
  double* r;             // S form
  double* h;
  int* steps;
  int* conv;
};
// Register split by order: 0 up to 64, 1 up to 128, 2 up to 256.
int lz_res_form(int d);
hipError_t launch_lz_res_group(const LzResJob* jobs, int njobs, int form, double lz_tol,
                               hipStream_t st);
hipError_t launch_lz_res(const float* S, int m, int k, const int* counts, uint64_t seed, int iter,
                         int I, double lz_tol, double* Q, double* vout, double* svout,
                         double* rout, int* steps_out, int* conv_out, hipStream_t st);

struct ClusterMatvecJob {
  const float* S;
  int m, k;
  const double* x;
  long xstride;
  double* y;
  const LzState* state;
};
long cluster_matvec_blocks(int m, int k);
hipError_t launch_cluster_matvec_group(const GroupTable& g, hipStream_t st);

struct LzJob {  // k_lz_setup / k_lz_step / k_lz_finish of one job
  int m;
  const int* counts;
  const int* mask;
  uint64_t seed;
  int iter, I;
  const double* rbuf;
  const double* wbuf;
  double* Q;
  LzState* state;
  double* vout;
  int* steps_out;
  int* conv_out;
  int* done_out;  // may be NULL: per-cluster copy of state.done (one readback)
};
size_t lz_step_lds(int m);
hipError_t launch_lz_setup_group(const GroupTable& g, hipStream_t st);
hipError_t launch_lz_step_group(const GroupTable& g, int mode, double lz_tol, hipStream_t st);
hipError_t launch_lz_finish_group(const GroupTable& g, hipStream_t st);

struct PowerJob {
  const float* S;
  int m;
  const int* counts;
  const float* a0;
  uint64_t seed;
  int iter, max_steps;
  double tol;
  const double* vin;
  const double* svin;
  const double* rsum;
  const int* steps_in;
  const int* conv_in;
  int eig_mode;
  const int* mask;
  int defer_fallback;
  float* c_out;
  PowerInfo* info;
};
hipError_t launch_power_group(const GroupTable& g, hipStream_t st);
size_t power_lds(int m);

}  // namespace tcx
