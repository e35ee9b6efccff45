// SBD kernels: z-normalization, centroid spectra, the fused
// FFT -> conj-multiply -> inverse FFT -> max-over-lags -> argmin assignment,
// the materialized NCC and the alignment.
//
// Layout: series are rows of a row-major FP32 [n][m] matrix.  A spectrum is
// F complex values stored lane-strided ([s][lane], s < P, lane < L) so that
// the lane group that produced it reads it back with coalesced loads.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <type_traits>

#include "tcx_device.hpp"
#include "tcx_internal.hpp"
#include "tcx_kernels.hpp"

namespace tcx {

// ---------------------------------------------------------------- z-norm
// One wave per row, FP64 accumulation of mean and of the centred sum of
// squares; (x - mean) / sqrt(ss / (m - ddof)), NaN -> 0 (nan_to_num).
// Semantics of zscore, Code/test/test_timesC.py:42-52.
__device__ __forceinline__ void znorm_body(const int bid, const int nblk,
    float* __restrict__ x, long rows,
                                               int m, int ddof) {
  const int lane = threadIdx.x & (kWave - 1);
  const long row = (long)bid * 4 + (threadIdx.x >> 6);
  if (row >= rows) return;
  float* r = x + row * (long)m;
  double s = 0.0;
  for (int t = lane; t < m; t += kWave) s += (double)r[t];
  s = wave_sum_f64(s);
  const double mean = s / (double)m;
  double ss = 0.0;
  for (int t = lane; t < m; t += kWave) {
    double d = (double)r[t] - mean;
    ss += d * d;
  }
  ss = wave_sum_f64(ss);
  const double sd = sqrt(ss / (double)(m - ddof));
  for (int t = lane; t < m; t += kWave) {
    double v = ((double)r[t] - mean) / sd;
    float f;
    if (isnan(v))
      f = 0.f;
    else if (isinf(v))
      f = v > 0 ? 3.402823466e38f : -3.402823466e38f;
    else
      f = (float)v;
    r[t] = f;
  }
}

__global__ __launch_bounds__(256) void k_znorm(float* __restrict__ x, long rows,
                                               int m, int ddof) {
  znorm_body(blockIdx.x, gridDim.x, x, rows, m, ddof);
}

// (v - mean) / sd of a row as a float: the residual step makes q the
// division's quotient (Markstein) where the row's sd is in a range in which
// nothing over- or underflows and nothing is NaN (kFast); else the division
// with nan_to_num.
template <bool kFast>
__device__ __forceinline__ float znorm_value(float v, double mean, double sd, double rsd) {
  const double d = (double)v - mean;
  if constexpr (kFast) {
    const double q = d * rsd;
    return (float)__builtin_fma(__builtin_fma(-q, sd, d), rsd, q);
  }
  const double w = d / sd;
  return isnan(w) ? 0.f : (isinf(w) ? (w > 0 ? 3.402823466e38f : -3.402823466e38f) : (float)w);
}

// The same with the row read once into registers, for m <= 4 G NV: lane l of
// the row's G lanes holds the 16-byte vectors l, l + G, ... and one of the m %
// 4 values after the last (kTail: rows that start at any float; without it
// the rows are whole aligned vectors); the sums are the same two-pass FP64
// sums in another order.  HBM bound; 16 lanes per row up to m = 128, where a
// wave per row leaves most of its lanes idle.  Times of a call (14 us of it
// the launch and the wait), before: rows that are no whole aligned vectors in
// three passes, a wave per row, the division: n=60000 m=365 65 -> 40 us, n=
// 30000 m=1001 91 -> 48 us (5.0 TB/s), n=100000 m=128 55 -> 28 us, m=37 43 ->
// 24 us.
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef f32x4 f32x4_u __attribute__((aligned(4)));
template <int G, bool kTail, int NV>
__device__ __forceinline__ void znorm_v_body(const int bid, const int nblk,
    float* __restrict__ x, long rows, int m, int ddof) {
  using vec = std::conditional_t<kTail, f32x4_u, f32x4>;
  const int lane = threadIdx.x & (G - 1);
  const long row = (long)bid * (256 / G) + threadIdx.x / G;
  if (row >= rows) return;
  float* r = x + row * (long)m;
  vec* rv = reinterpret_cast<vec*>(r);
  const int nv = m >> 2, tail = kTail ? m & 3 : 0;
  f32x4 v[NV];
#pragma unroll
  for (int u = 0; u < NV; ++u) {
    const int i = lane + G * u;
    v[u] = i < nv ? rv[i] : f32x4{0.f, 0.f, 0.f, 0.f};
  }
  float vt = 0.f;
  if (kTail && lane < tail) vt = r[4 * nv + lane];
  auto sum = [](double t) { return G == kWave ? wave_sum_f64(t) : row16_sum_f64(t); };
  double s = (double)vt;
#pragma unroll
  for (int u = 0; u < NV; ++u)
    s += ((double)v[u].x + (double)v[u].y) + ((double)v[u].z + (double)v[u].w);
  s = sum(s);
  const double mean = s / (double)m;
  double ss = 0.0;
  if (kTail && lane < tail) ss = ((double)vt - mean) * ((double)vt - mean);
#pragma unroll
  for (int u = 0; u < NV; ++u) {
    if (lane + G * u < nv) {
      const double a = (double)v[u].x - mean, b = (double)v[u].y - mean;
      const double c = (double)v[u].z - mean, d = (double)v[u].w - mean;
      ss += (a * a + b * b) + (c * c + d * d);
    }
  }
  ss = sum(ss);
  const double sd = sqrt(ss / (double)(m - ddof));
  const double rsd = 1.0 / sd;
  auto write = [&](auto fast) {
    auto z = [&](float e) { return znorm_value<decltype(fast)::value>(e, mean, sd, rsd); };
#pragma unroll
    for (int u = 0; u < NV; ++u) {
      const int i = lane + G * u;
      if (i < nv) rv[i] = f32x4{z(v[u].x), z(v[u].y), z(v[u].z), z(v[u].w)};
    }
    if (kTail && lane < tail) r[4 * nv + lane] = z(vt);
  };
  if (__all(sd > 1e-100 && sd < 1e100))  // over the wave's rows; false for NaN
    write(std::true_type{});
  else
    write(std::false_type{});
}

template <int G, bool kTail, int NV>
__global__ __launch_bounds__(256) void k_znorm_v(float* __restrict__ x, long rows, int m,
                                                 int ddof) {
  znorm_v_body<G, kTail, NV>(blockIdx.x, gridDim.x, x, rows, m, ddof);
}

// ------------------------------------------------------------- spectra
// Forward FFT of each row (zero padded to F, imaginary part 0), stored
// lane-strided, plus the row's L2 norm, an all-zero flag and (mag != NULL)
// the spectrum's magnitudes lane-major: |X[lane + L*s]| at lane*P + s, so a
// lane reads its values as 16-byte vectors.
template <int F>
__device__ __forceinline__ void spectra_body(const int bid, const int nblk,
    const float* __restrict__ y, int rows, int m, const float2* __restrict__ twg,
    float2* __restrict__ spec, float* __restrict__ norms, int* __restrict__ zero,
    float* __restrict__ mag, uint16_t* __restrict__ bmag) {
  using G = FftGeom<F>;
  constexpr int L = G::L, P = G::P;
  extern __shared__ float2 smem[];
  float2* tw = smem;
  float* red = reinterpret_cast<float*>(smem + fft_tw_lds<F>() + G::kGroups * fft_buf_len<F>());
  for (int i = threadIdx.x; i < fft_tw_lds<F>(); i += blockDim.x) tw[i] = twg[i];
  __syncthreads();
  const int g = threadIdx.x / L, lane = threadIdx.x % L;
  float2* buf = smem + fft_tw_lds<F>() + g * fft_buf_len<F>();
  for (int row = bid * G::kGroups + g; row < rows; row += nblk * G::kGroups) {
    const float* yr = y + (long)row * m;
    float2 v[P];
    float ss = 0.f;
    int nz = 0;
#pragma unroll
    for (int s = 0; s < P; ++s) {
      int t = lane + L * s;
      float a = t < m ? yr[t] : 0.f;
      v[s] = make_float2(a, 0.f);
      ss += a * a;
      nz |= (a != 0.f);
    }
    ss = group_sum<L>(ss, red);
    float fnz = group_sum<L>((float)nz, red);
    fft<F, L, false>(v, buf, tw, twg, lane);
    float2* o = spec + (long)row * F;
#pragma unroll
    for (int s = 0; s < P; ++s) o[s * L + lane] = v[s];
    if (mag) {
      float* mo = mag + (long)row * F + lane * P;
#pragma unroll
      for (int s = 0; s < P; ++s) mo[s] = sqrtf(v[s].x * v[s].x + v[s].y * v[s].y);
    }
    if (bmag) {  // bound operand row: |C[f]| / |c| for f <= F/2, zero padded
      constexpr int KP = bound_kpad(F);
      const float rn = ss > 0.f ? 1.f / sqrtf(ss) : 0.f;
#pragma unroll
      for (int s = 0; s < P; ++s) {
        const int f = lane + L * s;
        if (f <= F / 2)
          bmag[bound_frag(row, f, KP)] = f16_bits_up(sqrtf(v[s].x * v[s].x + v[s].y * v[s].y) * rn);
      }
      for (int f = F / 2 + 1 + lane; f < KP; f += L) bmag[bound_frag(row, f, KP)] = 0;
    }
    if (lane == 0) {
      norms[row] = sqrtf(ss);
      if (zero) zero[row] = fnz == 0.f;
    }
  }
}

template <int F>
__global__ __launch_bounds__(FftGeom<F>::kBlock) void k_spectra(
    const float* __restrict__ y, int rows, int m, const float2* __restrict__ twg,
    float2* __restrict__ spec, float* __restrict__ norms, int* __restrict__ zero,
    float* __restrict__ mag, uint16_t* __restrict__ bmag) {
  spectra_body<F>(blockIdx.x, gridDim.x, y, rows, m, twg, spec, norms, zero, mag, bmag);
}

// ------------------------------------------------ fused SBD / assignment
// Two series share one complex transform: z = x_a + i x_b.  For centroid j
// with spectrum C_j, ifft(FFT(z) conj(C_j)) = cc_a + i cc_b, the two
// circular cross-correlations of length F (F >= 2m-1, so no aliasing).
// ASSIGN: per series keep the centroid with the smallest
//   dist = 1 - (max_lag cc / F) / (|x| |c_j|)       (first argmin)
// and the lag key of its maximum (first argmax), test_timesC.py:258-260.
// SEARCH: ASSIGN with the pruned search's results where a norm is no number,
// zero or past the range.
// OWN: the same of one given centroid per series (fixed_label): at most two
// inverse transforms per pair.
// NCC: write cc / F / (|x| |y|) for all 2m-1 lags (ncc.cuh:467-517 layout
// out[x][y][lag]).
// blockIdx.y is a chunk of kc centroids; with several chunks ASSIGN and SEARCH write
// each chunk's result at y * n (k_split_min then takes the first smallest).

// z / d where r = 1 / d: the residual step makes the quotient the division's
// (Markstein) as long as nothing overflows and the residual is exact: the
// exponents of quotient and denominator sum to -103 or more.
__device__ __forceinline__ float div_by(float z, float d, float r) {
  const float q = z * r;
  return __builtin_fmaf(__builtin_fmaf(-q, d, z), r, q);
}

template <int F, int MODE, bool kFew>
__global__ __launch_bounds__(FftGeom<F>::kBlock, kFew ? 2 : FftGeom<F>::kMinWavesDense) void k_sbd(
    const float* __restrict__ x, long n, int m, int k, int kc,
    const float2* __restrict__ cspec, const float* __restrict__ cnorm,
    const float2* __restrict__ twg, int rev, int* __restrict__ label,
    float* __restrict__ dist, int* __restrict__ shift, float* __restrict__ dmat,
    int* __restrict__ changed, float* __restrict__ ncc_out,
    const int* __restrict__ fixed_label, const int* __restrict__ skip) {
  using G = FftGeom<F>;
  constexpr int L = G::L, P = G::P;
  extern __shared__ float2 smem[];
  if (MODE == kModeAssign && skip && *skip) return;
  float2* tw = smem;
  float* red = reinterpret_cast<float*>(smem + fft_tw_lds<F>() + G::kGroups * fft_buf_len<F>());
  for (int i = threadIdx.x; i < fft_tw_lds<F>(); i += blockDim.x) tw[i] = twg[i];
  __syncthreads();
  const int g = threadIdx.x / L, lane = threadIdx.x % L;
  float2* buf = smem + fft_tw_lds<F>() + g * fft_buf_len<F>();
  const long npairs = (n + 1) / 2;
  const int nlag = 2 * m - 1;
  const int j0 = blockIdx.y * kc, j1 = j0 + kc < k ? j0 + kc : k;
  for (long pr = (long)blockIdx.x * G::kGroups + g; pr < npairs;
       pr += (long)gridDim.x * G::kGroups) {
    const long ia = 2 * pr, ib = 2 * pr + 1;
    const bool hasb = ib < n;
    const float* xa = x + ia * (long)m;
    const float* xb = x + (hasb ? ib : ia) * (long)m;
    float2 zx[P];
    float sa = 0.f, sb = 0.f;
    const int ml = opaque(m);
#pragma unroll
    for (int s = 0; s < P; ++s) {
      int t = lane + L * s;
      float a = t < ml ? xa[t] : 0.f;
      float b = (hasb && t < ml) ? xb[t] : 0.f;
      zx[s] = make_float2(a, b);
      sa += a * a;
      sb += b * b;
    }
    sa = group_sum<L>(sa, red);
    sb = group_sum<L>(sb, red);
    float na = sqrtf(sa), nb = sqrtf(sb);
    if (MODE == kModeSearch && !(sa < INFINITY || (hasb && sb < INFINITY)))
      na = nb = NAN;  // no distance
    fft<F, L, false>(zx, buf, tw, twg, lane);

    float bestA = INFINITY, bestB = INFINITY;
    int labA = 0, labB = 0, keyA = 0, keyB = 0;
    int fixA = -1, fixB = -1, e0 = j0, e1 = j1;
    if constexpr (MODE == kModeOwn) {  // a label outside [0, k) is left to the caller
      fixA = fixed_label[ia];
      fixB = hasb ? fixed_label[ib] : fixA;
      if (fixA < 0 || fixA >= k) fixA = -1;
      if (fixB < 0 || fixB >= k) fixB = -1;
      e0 = fixA >= 0 ? 0 : 1;
      e1 = fixB >= 0 && fixB != fixA ? 2 : 1;
    }
    for (int e = e0; e < e1; ++e) {
      const int j = MODE == kModeOwn ? (e == 0 ? fixA : fixB) : e;
      const float2* cj = cspec + (long)j * F;
      float2 z[P];
#pragma unroll
      for (int s = 0; s < P; ++s) z[s] = cj[s * L + lane];
      // all of the spectrum in flight at once: without the barrier the compiler
      // may load and multiply one value after the other, a latency each (NCC at
      // F = 512 and 1024: n=700 m=301 k=12 38.3 us, 34.8 with it).  With 128
      // registers the values would spill
      if constexpr ((F <= 1024 || kFew) && MODE != kModeOwn) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int s = 0; s < P; ++s) z[s] = cmulc(zx[s], z[s]);
      fft<F, L, true>(z, buf, tw, twg, lane);
      const float cn = cnorm[j];
      const float dena = na * cn, denb = nb * cn;
      if constexpr (MODE != kModeNcc) {
        float va, vb;
        int ka, kb;
        lag_max<F, L, P>(z, hasb, rev, lane, m, red, va, ka, vb, kb);
        // den == 0: NumPy divides by inf, every lag is 0, argmax is index 0
        float da = 1.f, db = 1.f;
        if (dena != 0.f) da = 1.f - (va / (float)F) / dena; else ka = 0;
        if (denb != 0.f) db = 1.f - (vb / (float)F) / denb; else kb = 0;
        if constexpr (MODE == kModeSearch) {
          if (cn == 0.f && (na == na || nb == nb)) {
            da = db = 1.f;
            ka = kb = 0;
          } else if (!(cn < INFINITY)) {
            da = db = INFINITY;
          }
        }
        if (MODE == kModeOwn ? (j == fixA) : (da < bestA)) { bestA = da; labA = j; keyA = ka; }
        if (MODE == kModeOwn ? (j == fixB) : (db < bestB)) { bestB = db; labB = j; keyB = kb; }
        if (MODE == kModeAssign && dmat && lane == 0) {
          dmat[ia * k + j] = da;
          if (hasb) dmat[ib * k + j] = db;
        }
      } else {
        const float sca = dena != 0.f ? 1.f : 0.f, scb = denb != 0.f ? 1.f : 0.f;
        const float dA = dena != 0.f ? dena : 1.f, dB = denb != 0.f ? denb : 1.f;
        float* oa = ncc_out + (ia * (long)k + j) * nlag;
        float* ob = ncc_out + (ib * (long)k + j) * nlag;
        const int mo = opaque(m);
        auto write = [&](auto quot) {
#pragma unroll
          for (int s = 0; s < P; ++s) {
            const int key = lag_key(lane + L * s, mo, F, 0);
            if (key >= 0) {
              oa[key] = sca * quot(z[s].x / (float)F, 0);
              if (hasb) ob[key] = scb * quot(z[s].y / (float)F, 1);
            }
          }
        };
        // In this range of the denominators nothing overflows (z / F is at most
        // about the denominator), and the residual, a multiple of 2^-46 times the
        // powers of two in quotient and denominator, is exact but for quotients
        // below 2^-77, whose last bit may differ from the division's
        if (fminf(dA, dB) > 0x1p-26f && fmaxf(dA, dB) < 0x1p50f) {
          const float rA = 1.f / dA, rB = 1.f / dB;
          write([&](float v, int b) { return b ? div_by(v, dB, rB) : div_by(v, dA, rA); });
        } else {
          write([&](float v, int b) { return v / (b ? dB : dA); });
        }
      }
    }
    if constexpr (MODE != kModeNcc) {
      if (lane == 0) {
        const long o = (long)blockIdx.y * n;
        if (changed && label[ia] != labA) *changed = 1;
        if (label) label[o + ia] = labA;
        if (dist) dist[o + ia] = bestA;
        // (1 - m) first: OWN's key of a series without a distance is INT_MAX,
        // a shift past the row
        if (shift) shift[o + ia] = keyA + (1 - m);
        if (hasb) {
          if (changed && label[ib] != labB) *changed = 1;
          if (label) label[o + ib] = labB;
          if (dist) dist[o + ib] = bestB;
          if (shift) shift[o + ib] = keyB + (1 - m);
        }
      }
    }
  }
}

// The chunk results [chunks][n] of k_sbd to one: the first smallest distance
// in chunk order, as one pass over all centroids keeps it.
__global__ __launch_bounds__(256) void k_split_min(
    const float* __restrict__ pdist, const int* __restrict__ plabel,
    const int* __restrict__ pshift, long n, int m, int chunks, int* __restrict__ label,
    float* __restrict__ dist, int* __restrict__ shift) {
  const long i = (long)blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  float best = INFINITY;
  int lab = 0, sh = 1 - m;
  for (int c = 0; c < chunks; ++c) {
    const float d = pdist[c * n + i];
    const int l = plabel[c * n + i], s = pshift[c * n + i];
    if (d < best) {
      best = d;
      lab = l;
      sh = s;
    }
  }
  label[i] = lab;
  if (dist) dist[i] = best;
  if (shift) shift[i] = sh;
}

// The first N (<= P) magnitudes of a lane from its lane-major row segment
// (16-byte aligned, P a multiple of 4): N/4 vector loads and a scalar tail.
template <int P, int N>
__device__ __forceinline__ void load_mag(const float* __restrict__ src, float (&out)[N]) {
  static_assert(P % 4 == 0 && N <= P, "lane-major magnitudes");
#pragma unroll
  for (int i = 0; i + 4 <= N; i += 4) {
    const float4 q = *reinterpret_cast<const float4*>(src + i);
    out[i] = q.x;
    out[i + 1] = q.y;
    out[i + 2] = q.z;
    out[i + 3] = q.w;
  }
#pragma unroll
  for (int i = N / 4 * 4; i < N; ++i) out[i] = src[i];
}

// ------------------------------------------- pruned assignment (exact)
// For every centroid j the lag maximum of the correlation is bounded by the
// spectra:  max_l cc[l] = max_l (1/F) |sum_f X_f conj(C_f) e^{2 pi i f l/F}|
// <= (1/F) sum_f |X_f| |C_f|,  so  dist_j >= lb_j = 1 - ub_j  with
// ub_j = sum_f |X_f||C_f| / (F |x| |c_j|).  Per pair of series the
// centroids are evaluated (inverse FFT, exact distance) in decreasing
// order of their bound; a centroid whose lower bound (with a rounding
// margin) exceeds the best exact distance found cannot be the argmin and
// is skipped.  Ties keep NumPy's first-index rule.  The result equals the
// dense kernel's; the pair's two series share each evaluated transform.
// |X_a|, |X_b| come from the packed transform Z = FFT(x_a + i x_b):
// X_a = (Z_f + conj(Z_{F-f}))/2, X_b = (Z_f - conj(Z_{F-f}))/(2i).
// order (may be NULL): row indices to pair up, -1 = hole; rows with the
// same previous label are adjacent there, so both series of a pair tend to
// share their candidates.
constexpr float kUbRel = 1e-4f;   // rounding margin of the bound
constexpr float kUbAbs = 1e-5f;

// a' + b' after v_permlane16_swap (O = 16: odd rows of a with even rows of
// b) or v_permlane32_swap (O = 32: upper half of a with lower half of b).
template <int O>
__device__ __forceinline__ float swap_sum(float a, float b) {
  static_assert(O == 16 || O == 32, "row or half swap");
  if constexpr (O == 16) {
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false,
                                                    false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
  } else {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false,
                                                    false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
  }
}

// Reduce-scatter of the CNT values v[0..CNT) of every lane over a group of
// L lanes (one wave or less): at lane-bit O a lane keeps the lower or upper
// half of its values (by that bit) plus the partner's matching half; once a
// single value is left the remaining levels are plain butterfly sums.
// Afterwards a lane holds the group sums of values base .. base + CNT/L - 1
// (one value when CNT <= L).
template <int CNT, int O, int L, int N>
__device__ __forceinline__ void reduce_scatter(float (&v)[N], int lane, int& base) {
  if constexpr (O >= 1) {
    const bool up = (lane & O) != 0;
    if constexpr (O >= 16) {
      // rows of 16 (O = 16) or halves of 32 (O = 32) swapped between two
      // registers a, b: afterwards a lane without bit O holds its own a and
      // its partner's a, a lane with bit O its partner's b and its own b, so
      // the sum of the two is each lane's kept half plus the partner's
      if constexpr (CNT > 1) {
        constexpr int HF = CNT / 2;
#pragma unroll
        for (int i = 0; i < HF; ++i) v[i] = swap_sum<O>(v[i], v[i + HF]);
        if (up) base += HF;
        reduce_scatter<HF, O / 2, L>(v, lane, base);
      } else {
        v[0] = swap_sum<O>(v[0], v[0]);
        reduce_scatter<1, O / 2, L>(v, lane, base);
      }
    } else {
      // partner by DPP: lane ^ 1, lane ^ 2, the 8-lane mirror (bit 2 flips),
      // the 16-lane mirror (bit 3 flips); each pairs the two halves of the
      // current subgroup one to one
      constexpr int CTRL = O == 1 ? 0xB1 : O == 2 ? 0x4E : O == 4 ? 0x141 : 0x140;
      if constexpr (CNT > 1) {
        constexpr int HF = CNT / 2;
#pragma unroll
        for (int i = 0; i < HF; ++i) {
          const float send = up ? v[i] : v[i + HF];
          const float keep = up ? v[i + HF] : v[i];
          v[i] = keep + dpp_f32<CTRL>(send);
        }
        if (up) base += HF;
        reduce_scatter<HF, O / 2, L>(v, lane, base);
      } else {
        v[0] += dpp_f32<CTRL>(v[0]);
        reduce_scatter<1, O / 2, L>(v, lane, base);
      }
    }
  }
}

// Partner values of the packed spectrum Z = FFT(x_a + i x_b) held
// lane-strided (Z[lane + L*s] in zx[s]): for s <= P/2, (px[s], py[s]) =
// Z[F - f] with f = lane + L*s, from lane' = (L - lane) % L, s' = P-1-s
// (lane 0: s' = (P - s) % P).  Then X_a[f] = (Z[f] + conj(Z[F-f])) / 2 and
// X_b[f] = (Z[f] - conj(Z[F-f])) / (2i).  Groups wider than a wave exchange
// through `buf` (LDS) between barriers.
template <int F, int L, int P>
__device__ __forceinline__ void partner_half(const float2 (&zx)[P], float2* buf, int lane,
                                             float (&px)[P / 2 + 1], float (&py)[P / 2 + 1]) {
  constexpr int H = P / 2;
  const int pl = (L - lane) & (L - 1);
  if constexpr (L > kWave) {
#pragma unroll
    for (int s = 0; s < P; ++s) buf[lds_pad(lane + L * s)] = zx[s];
    __syncthreads();
  }
#pragma unroll
  for (int s = 0; s <= H; ++s) {
    if constexpr (L > kWave) {
      const float2 q = buf[lds_pad(pl + L * (P - 1 - s))];
      px[s] = q.x;
      py[s] = q.y;
    } else {
      px[s] = __shfl(zx[P - 1 - s].x, pl, L);
      py[s] = __shfl(zx[P - 1 - s].y, pl, L);
    }
    if (lane == 0) {
      px[s] = zx[(P - s) & (P - 1)].x;
      py[s] = zx[(P - s) & (P - 1)].y;
    }
  }
  if constexpr (L > kWave) __syncthreads();  // reads done before buf is reused
}

// Half spectra of every series, once per fit (the series do not change
// between iterations): row r holds X_r[f] for f = 0 .. F/2 (F/2 + 1 values,
// X_r[F-f] = conj(X_r[f])), and xn[r] = |x_r|.  Rows are transformed in
// natural pairs packed as x_a + i x_b and split with partner_half.
template <int F>
__device__ __forceinline__ void series_spec_body(const int bid, const int nblk,
    const float* __restrict__ x, long n, int m, const float2* __restrict__ twg,
    float2* __restrict__ xs, float* __restrict__ xn, uint16_t* __restrict__ xm) {
  using G = FftGeom<F>;
  constexpr int L = G::L, P = G::P, H = P / 2;
  constexpr long HS = F / 2 + 1;
  extern __shared__ float2 smem[];
  float2* tw = smem;
  float* red = reinterpret_cast<float*>(smem + fft_tw_lds<F>() + G::kGroups * fft_buf_len<F>());
  for (int i = threadIdx.x; i < fft_tw_lds<F>(); i += blockDim.x) tw[i] = twg[i];
  __syncthreads();
  const int g = threadIdx.x / L, lane = threadIdx.x % L;
  float2* buf = smem + fft_tw_lds<F>() + g * fft_buf_len<F>();
  const long npairs = (n + 1) / 2;
  for (long pr = (long)bid * G::kGroups + g; pr < npairs;
       pr += (long)nblk * G::kGroups) {
    const long ia = 2 * pr, ib = 2 * pr + 1;
    const bool hasb = ib < n;
    const float* xa = x + ia * (long)m;
    const float* xb = x + (hasb ? ib : ia) * (long)m;
    float2 zx[P];
    float sa = 0.f, sb = 0.f;
    const int ml = opaque(m);
#pragma unroll
    for (int s = 0; s < P; ++s) {
      const int t = lane + L * s;
      const float a = t < ml ? xa[t] : 0.f;
      const float b = (hasb && t < ml) ? xb[t] : 0.f;
      zx[s] = make_float2(a, b);
      sa += a * a;
      sb += b * b;
    }
    sa = group_sum<L>(sa, red);
    sb = group_sum<L>(sb, red);
    if (lane == 0) {
      xn[ia] = sqrtf(sa);
      if (hasb) xn[ib] = sqrtf(sb);
    }
    fft<F, L, false>(zx, buf, tw, twg, lane);
    float px[H + 1], py[H + 1];
    partner_half<F, L, P>(zx, buf, lane, px, py);
    float2* oa = xs + ia * HS;
    float2* ob = xs + ib * HS;
    // bound rows: weight * |X_f| / |x|, weight 2 inside, 1 at f = 0, F/2
    // (the 1/F is applied to the product)
    constexpr int KP = bound_kpad(F);
    const float ra = sa > 0.f ? 1.f / sqrtf(sa) : 0.f;
    const float rb = sb > 0.f ? 1.f / sqrtf(sb) : 0.f;
#pragma unroll
    for (int s = 0; s <= H; ++s) {
      const int f = lane + L * s;
      if (s < H || lane == 0) {  // f < F/2, or f = F/2
        const int fo = s < H ? f : F / 2;
        const float2 A = make_float2(0.5f * (zx[s].x + px[s]), 0.5f * (zx[s].y - py[s]));
        const float2 B = make_float2(0.5f * (zx[s].y + py[s]), 0.5f * (px[s] - zx[s].x));
        oa[fo] = A;
        if (hasb) ob[fo] = B;
        if (xm) {
          const float w = (fo == 0 || fo == F / 2) ? 1.f : 2.f;
          xm[bound_frag(ia, fo, KP)] = f16_bits_up(w * sqrtf(A.x * A.x + A.y * A.y) * ra);
          if (hasb) xm[bound_frag(ib, fo, KP)] = f16_bits_up(w * sqrtf(B.x * B.x + B.y * B.y) * rb);
        }
      }
    }
    if (xm)
      for (int f = F / 2 + 1 + lane; f < KP; f += L) {  // padding of the K dimension
        xm[bound_frag(ia, f, KP)] = 0;
        if (hasb) xm[bound_frag(ib, f, KP)] = 0;
      }
  }
}

template <int F>
__global__ __launch_bounds__(FftGeom<F>::kBlock, FftGeom<F>::kMinWaves) void k_series_spec(
    const float* __restrict__ x, long n, int m, const float2* __restrict__ twg,
    float2* __restrict__ xs, float* __restrict__ xn, uint16_t* __restrict__ xm) {
  series_spec_body<F>(blockIdx.x, gridDim.x, x, n, m, twg, xs, xn, xm);
}

// ------------------------------------------ bounds of the pruned assignment
// ub[i][j] = sum_f xm[i][f] cm[j][f] / F for every series i and centroid j:
// the bounds k_assign_prune otherwise forms per pair, as one product of the
// per-fit magnitude rows xm (k_series_spec) and the centroids' rows cm =
// |C_j[f]| / |c_j| (k_spectra), both binary16 rounded up in fragment order
// (bound_frag), on v_mfma_f32_16x16x16_f16 with FP32 accumulation (the
// products of two binary16 values are exact in FP32).  A wave computes 16
// series x 16 centroids per tile and NT tiles per pass over its rows of xm;
// for the 16 columns of a step lane l reads the l-th 8-byte vector of the
// fragment block of each operand (one contiguous 512 B per wave).  Result
// element (i, j) is in lane j + 16 (i / 4), register i % 4.  Rows past n (or
// centroids past k) in the last block are computed from whatever the
// padding holds and never stored: a result element depends on its own row
// and column only.
typedef _Float16 bound_h4 __attribute__((ext_vector_type(4)));
typedef float bound_f4 __attribute__((ext_vector_type(4)));
template <int NT, int MT, int NS>
__device__ __forceinline__ void bounds_body(const int bid, const int nblk,
    const uint16_t* __restrict__ xm, long n, int kpad,
                                                const uint16_t* __restrict__ cm, int k, int ld,
                                                float scale, float* __restrict__ ub) {
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  const long blk0 = ((long)bid * 4 + wid) * MT;  // first 16-row block of the wave
  if (blk0 * 16 >= n) return;
  const long nrb = (n + 15) >> 4;  // row blocks of 16
  const int r = lane & 15, kq = lane >> 4;
  const int nsteps = kpad >> 4;
  const bound_h4* xa[MT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    const long b = blk0 + mt < nrb ? blk0 + mt : blk0;  // blocks past n: computed, not stored
    xa[mt] = reinterpret_cast<const bound_h4*>(xm) + b * nsteps * 64 + lane;
  }
  for (int t0 = 0; t0 * 16 < k; t0 += NT) {
    bound_f4 acc[MT][NT];
    const bound_h4* cb[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const int jt = (t0 + t) * 16 < k ? t0 + t : t0;  // tiles past k: computed, not stored
      cb[t] = reinterpret_cast<const bound_h4*>(cm) + (long)jt * nsteps * 64 + lane;
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) acc[mt][t] = bound_f4{0.f, 0.f, 0.f, 0.f};
    }
    for (int s0 = 0; s0 < nsteps; s0 += NS) {
      bound_h4 a[MT][NS], bv[NT][NS];
#pragma unroll
      for (int u = 0; u < NS; ++u) {
        const int s = s0 + u < nsteps ? s0 + u : nsteps - 1;  // clamped, dropped below
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) a[mt][u] = xa[mt][(long)s * 64];
#pragma unroll
        for (int t = 0; t < NT; ++t) bv[t][u] = cb[t][(long)s * 64];
      }
#pragma unroll
      for (int u = 0; u < NS; ++u) {
        if (s0 + u < nsteps) {  // uniform
#pragma unroll
          for (int mt = 0; mt < MT; ++mt)
#pragma unroll
            for (int t = 0; t < NT; ++t)
              acc[mt][t] =
                  __builtin_amdgcn_mfma_f32_16x16x16f16(a[mt][u], bv[t][u], acc[mt][t], 0, 0, 0);
        }
      }
    }
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        const int j = (t0 + t) * 16 + r;
        if (j >= k) continue;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const long i = (blk0 + mt) * 16 + 4 * kq + q;
          if (i < n) ub[i * ld + j] = acc[mt][t][q] * scale;
        }
      }
  }
}

template <int NT, int MT, int NS>
__global__ __launch_bounds__(256) void k_bounds(const uint16_t* __restrict__ xm, long n, int kpad,
                                                const uint16_t* __restrict__ cm, int k, int ld,
                                                float scale, float* __restrict__ ub) {
  bounds_body<NT, MT, NS>(blockIdx.x, gridDim.x, xm, n, kpad, cm, k, ld, scale, ub);
}

// Bounds of every centroid for one series pair (group of L lanes) from the
// weighted half-spectrum magnitudes ma, mb: ub = sum_f |X_f| |C_f| /
// (F |x| |c|), written to ubs[0, k) (series a) and ubs[k, 2k) (series b).
template <int F, int L, int P>
__device__ __forceinline__ void prune_bounds(const float* ma, const float* mb, float na, float nb,
                                             const float* __restrict__ cmag,
                                             const float* __restrict__ cnorm, int k, int lane,
                                             float* red, float* ubs) {
  constexpr int H = P / 2;
  if constexpr (L <= kWave) {
    // KC centroids at a time; the 2*KC per-lane partial sums are reduced
    // by a reduce-scatter over the L lanes (each level halves the values
    // a lane keeps)
    constexpr int KC = 4;
    for (int j0 = 0; j0 < k; j0 += KC) {
      float v[2 * KC];
#pragma unroll
      for (int c = 0; c < KC; ++c) {
        float aa = 0.f, ab = 0.f;
        if (j0 + c < k) {
          float cv[H + 1];
          load_mag<P, H + 1>(cmag + (long)(j0 + c) * F + lane * P, cv);
#pragma unroll
          for (int s = 0; s <= H; ++s) {
            aa += ma[s] * cv[s];
            ab += mb[s] * cv[s];
          }
        }
        v[c] = aa;
        v[KC + c] = ab;
      }
      int base = 0;
      reduce_scatter<2 * KC, L / 2, L>(v, lane, base);
      constexpr int kHeld = 2 * KC >= L ? 2 * KC / L : 1;
#pragma unroll
      for (int i = 0; i < kHeld; ++i) {
        const int idx = base + i, ser = idx / KC, jj = j0 + idx % KC;
        if (jj < k) {
          const float den = (ser ? nb : na) * cnorm[jj];
          ubs[ser * k + jj] = den != 0.f ? (v[i] / (float)F) / den : 0.f;
        }
      }
    }
  } else {
    for (int j = 0; j < k; ++j) {
      float cv[H + 1];
      load_mag<P, H + 1>(cmag + (long)j * F + lane * P, cv);
      float aa = 0.f, ab = 0.f;
#pragma unroll
      for (int s = 0; s <= H; ++s) {
        aa += ma[s] * cv[s];
        ab += mb[s] * cv[s];
      }
      aa = group_sum<L>(aa, red);
      ab = group_sum<L>(ab, red);
      if (lane == 0) {
        const float cn = cnorm[j];
        const float dena = na * cn, denb = nb * cn;
        ubs[j] = dena != 0.f ? (aa / (float)F) / dena : 0.f;
        ubs[k + j] = denb != 0.f ? (ab / (float)F) / denb : 0.f;
      }
    }
  }
}

// Launch geometry of the pruned assignment (that of the dense kernel).
template <int F>
struct PruneGeom {
  static constexpr int L = FftGeom<F>::L;
  static constexpr int kBlock = FftGeom<F>::kBlock;
  static constexpr int kGroups = kBlock / L;
  static constexpr int kMinWaves = FftGeom<F>::kMinWaves;
};

template <int F, bool kPre>
__device__ __forceinline__ void assign_prune_body(const int bid, const int nblk,
    const float* __restrict__ x, const float2* __restrict__ xs, const float* __restrict__ xn,
    const float* __restrict__ ubg, int ub_ld, long n, long npairs, int m, int k,
    const float2* __restrict__ cspec, const float* __restrict__ cmag,
    const float* __restrict__ cnorm, const float2* __restrict__ twg, int rev,
    const int* __restrict__ order, int* __restrict__ label, float* __restrict__ dist,
    int* __restrict__ shift, int* __restrict__ changed, unsigned long long* __restrict__ evals) {
  using G = PruneGeom<F>;
  constexpr int L = G::L, P = FftGeom<F>::P;
  constexpr bool kTG = kPre ? F > 1024 : F >= 1024;
  extern __shared__ float2 smem[];
  float2* tw = smem;
  float* red = reinterpret_cast<float*>(smem + fft_tw_lds<F, kTG>() + G::kGroups * fft_buf_len<F>());
  float* ubs_all = red + 64;
  for (int i = threadIdx.x; i < fft_tw_lds<F, kTG>(); i += blockDim.x) tw[i] = twg[i];
  __syncthreads();
  const int g = threadIdx.x / L, lane = threadIdx.x % L;
  float2* buf = smem + fft_tw_lds<F, kTG>() + g * fft_buf_len<F>();
  float* ubs = ubs_all + (long)g * 2 * k;  // [0,k): series a, [k,2k): series b
  unsigned my_evals = 0;
  for (long pr = (long)bid * G::kGroups + g; pr < npairs;
       pr += (long)nblk * G::kGroups) {
    long ia = order ? order[2 * pr] : 2 * pr;
    long ib = order ? (2 * pr + 1 < 2 * npairs ? order[2 * pr + 1] : -1) : 2 * pr + 1;
    if (ia >= n) ia = -1;
    if (ib >= n) ib = -1;
    if (ia < 0) {
      ia = ib;
      ib = -1;
    }
    if (ia < 0) continue;  // hole pair (uniform for the group)
    const bool hasb = ib >= 0;
    // packed spectrum zx[s] = Z[lane + L*s], Z = X_a + i X_b; without the
    // per-fit data also the weighted half-spectrum magnitudes ma, mb
    // (f = lane + L*s for s < P/2, f = F/2 at lane 0, s = P/2; weight 2
    // inside, 1 at f = 0 and f = F/2) for the bounds
    constexpr int H = P / 2;
    float2 zx[P];
    float na, nb;
    if constexpr (kPre) {
      // from the per-fit half spectra: X[f] for f <= F/2, conj(X[F-f]) above
      constexpr long HS = F / 2 + 1;
      // lane bases: f = lane + L*s below F/2 and F - f above, so that every
      // load is a base plus an immediate offset
      const float2* pa = xs + ia * HS + lane;
      const float2* pb = xs + (hasb ? ib : ia) * HS + lane;
      const float2* qa = xs + ia * HS + (F - L * H) - lane;
      const float2* qb = xs + (hasb ? ib : ia) * HS + (F - L * H) - lane;
      na = xn[ia];
      nb = hasb ? xn[ib] : 0.f;
      // all loads of the pair in flight at once (one latency per pair)
      auto assemble = [&](int s) {
        float2 A, B;
        if (s < H) {
          A = pa[L * s];
          B = hasb ? pb[L * s] : make_float2(0.f, 0.f);
        } else {
          const float2 a2 = qa[-L * (s - H)];
          const float2 b2 = hasb ? qb[-L * (s - H)] : make_float2(0.f, 0.f);
          A = make_float2(a2.x, -a2.y);
          B = make_float2(b2.x, -b2.y);
        }
        zx[s] = make_float2(A.x - B.y, A.y + B.x);
      };
#pragma unroll
      for (int s = 0; s < P; ++s) assemble(s);
      // the bounds, computed for every series by k_bounds
      for (int j = lane; j < k; j += L) {
        ubs[j] = ubg[ia * ub_ld + j];
        ubs[k + j] = hasb ? ubg[ib * ub_ld + j] : 0.f;
      }
    } else {
      const float* xa = x + ia * (long)m;
      const float* xb = x + (hasb ? ib : ia) * (long)m;
      float sa = 0.f, sb = 0.f;
    const int ml = opaque(m);
#pragma unroll
      for (int s = 0; s < P; ++s) {
        const int t = lane + L * s;
        const float a = t < ml ? xa[t] : 0.f;
        const float b = (hasb && t < ml) ? xb[t] : 0.f;
        zx[s] = make_float2(a, b);
        sa += a * a;
        sb += b * b;
      }
      sa = group_sum<L>(sa, red);
      sb = group_sum<L>(sb, red);
      na = sqrtf(sa);
      nb = sqrtf(sb);
      fft<F, L, false, kTG>(zx, buf, tw, twg, lane);
      // |X_a[f]| = |Z[f] + conj(Z[F-f])| / 2, |X_b[f]| = |Z[f] - conj(Z[F-f])| / 2
      float px[H + 1], py[H + 1];
      float ma[H + 1], mb[H + 1];
      partner_half<F, L, P>(zx, buf, lane, px, py);
#pragma unroll
      for (int s = 0; s <= H; ++s) {
        const float ar = zx[s].x + px[s], ai = zx[s].y - py[s];
        const float br = zx[s].x - px[s], bi = zx[s].y + py[s];
        const float wgt = s == H ? (lane == 0 ? 0.5f : 0.f) : ((s == 0 && lane == 0) ? 0.5f : 1.f);
        ma[s] = wgt * sqrtf(ar * ar + ai * ai);
        mb[s] = wgt * sqrtf(br * br + bi * bi);
      }
      prune_bounds<F, L, P>(ma, mb, na, nb, cmag, cnorm, k, lane, red, ubs);
    }
    group_sync<L>();
    float bestA = INFINITY, bestB = hasb ? INFINITY : -INFINITY;
    int labA = 0, labB = 0, keyA = 0, keyB = 0;
    // groups of whole waves with k <= 64: centroid j's two bounds stay in the
    // registers of lane j of every wave (-1: evaluated), the next candidate
    // is a wave max and a ballot, the same in every wave
    const bool inreg = L >= kWave && k <= kWave;  // uniform
    const int wl = lane & (kWave - 1);
    float myA = -1.f, myB = -1.f;
    if (inreg && wl < k) {
      myA = ubs[wl];
      myB = ubs[k + wl];
    }
    for (int round = 0; round < k; ++round) {
      // candidate with the largest bound among centroids that can still win
      float sc = -INFINITY;
      int cj = 0x7fffffff;
      if (inreg) {
        const bool oka = (myA >= 0.f) & (1.f - (myA * (1.f + kUbRel) + kUbAbs) <= bestA);
        const bool okb = (myB >= 0.f) & (1.f - (myB * (1.f + kUbRel) + kUbAbs) <= bestB);
        float v = oka ? myA : -INFINITY;
        v = okb ? fmaxf(v, myB) : v;
        sc = wave_max(v);
        if (sc > -INFINITY) cj = __builtin_ctzll(__ballot(v == sc));  // first j on ties
      } else {
        for (int j = lane; j < k; j += L) {  // j increases: strict '>' keeps the first
          const float ua = ubs[j], ub = ubs[k + j];
          const bool oka = (ua >= 0.f) & (1.f - (ua * (1.f + kUbRel) + kUbAbs) <= bestA);
          const bool okb = (ub >= 0.f) & (1.f - (ub * (1.f + kUbRel) + kUbAbs) <= bestB);
          float v = oka ? ua : -INFINITY;
          v = okb ? fmaxf(v, ub) : v;
          const bool take = v > sc;
          sc = take ? v : sc;
          cj = take ? j : cj;
        }
        group_argmax<L>(sc, cj, red);
      }
      if (!(sc > -INFINITY)) break;
      const int j = cj;
      if (inreg) {
        if (wl == j) {
          myA = -1.f;  // evaluated
          myB = -1.f;
        }
      } else {
        group_sync<L>();
        if (lane == 0) {
          ubs[j] = -1.f;  // evaluated
          ubs[k + j] = -1.f;
        }
      }
      const float cn = cnorm[j];
      const float dena = na * cn, denb = nb * cn;
      float da = 1.f, db = 1.f;
      int ka = 0, kb = 0;
      if (cn != 0.f) {
        ++my_evals;
        const float2* cjs = cspec + (long)j * F;
        float2 z[P];
#pragma unroll
        for (int s = 0; s < P; ++s) z[s] = cmulc(zx[s], cjs[s * L + lane]);
        fft<F, L, true, kTG>(z, buf, tw, twg, lane);
        float va, vb;
        lag_max<F, L, P>(z, hasb, rev, lane, m, red, va, ka, vb, kb);
        if (dena != 0.f) da = 1.f - (va / (float)F) / dena; else ka = 0;
        if (denb != 0.f) db = 1.f - (vb / (float)F) / denb; else kb = 0;
      }
      if (da < bestA || (da == bestA && j < labA)) { bestA = da; labA = j; keyA = ka; }
      if (hasb && (db < bestB || (db == bestB && j < labB))) { bestB = db; labB = j; keyB = kb; }
      if (!inreg) group_sync<L>();  // ubs of the evaluated centroid is written
    }
    group_sync<L>();  // ubs is rewritten by the next pair
    if (lane == 0) {
      if (changed && label[ia] != labA) *changed = 1;
      label[ia] = labA;
      if (dist) dist[ia] = bestA;
      if (shift) shift[ia] = keyA + 1 - m;
      if (hasb) {
        if (changed && label[ib] != labB) *changed = 1;
        label[ib] = labB;
        if (dist) dist[ib] = bestB;
        if (shift) shift[ib] = keyB + 1 - m;
      }
    }
  }
  if (evals) {  // one add per wave (a group of several waves: of its first)
    unsigned v = lane == 0 ? my_evals : 0;
#pragma unroll
    for (int o = L; o < kWave; o *= 2) v += __shfl_xor(v, o);
    if (threadIdx.x % (L < kWave ? kWave : L) == 0 && v)
      atomicAdd(evals + (bid % kEvalSlots) * kEvalStride, (unsigned long long)v);
  }
}

template <int F, bool kPre, bool kFew>
__global__ __launch_bounds__(PruneGeom<F>::kBlock, kFew    ? 2
                                                   : kPre ? FftGeom<F>::kMinWaves
                                                          : FftGeom<F>::kMinWavesPrune)
void k_assign_prune(
    const float* __restrict__ x, const float2* __restrict__ xs, const float* __restrict__ xn,
    const float* __restrict__ ubg, int ub_ld, long n, long npairs, int m, int k,
    const float2* __restrict__ cspec, const float* __restrict__ cmag,
    const float* __restrict__ cnorm, const float2* __restrict__ twg, int rev,
    const int* __restrict__ order, int* __restrict__ label, float* __restrict__ dist,
    int* __restrict__ shift, int* __restrict__ changed, unsigned long long* __restrict__ evals,
    const int* __restrict__ skip) {
  if (skip && *skip) return;
  assign_prune_body<F, kPre>(blockIdx.x, gridDim.x, x, xs, xn, ubg, ub_ld, n, npairs, m, k, cspec, cmag, cnorm, twg, rev, order, label, dist, shift, changed, evals);
}

// ------------------------------------------------------------- alignment
// Each series against one centroid, shifted in place by the lag of its
// largest NCC with zero fill (out[t] = in[t - s], 0 outside; roll_zeropad,
// test_timesC.py:55-77), nothing for an all-zero centroid: one kernel forms
// the pair's correlation, its lags (the search's, bit for bit) and the shifted
// rows, which it reads again from L2.  Bound by the two transforms.  With
// the shifts through memory, the bounds of a search over one centroid and a
// second kernel to shift the rows, n=12000 m=700 took 143 us, 95 now.
template <int F>
__global__ __launch_bounds__(FftGeom<F>::kBlock, FftGeom<F>::kMinWaves) void k_align(
    float* x, long n, int m, const float2* __restrict__ cspec, const float* __restrict__ cnorm,
    const int* __restrict__ czero, const float2* __restrict__ twg, int rev) {
  using G = FftGeom<F>;
  constexpr int L = G::L, P = G::P;
  extern __shared__ float2 smem[];
  if (*czero) return;
  float2* tw = smem;
  float* red = reinterpret_cast<float*>(smem + fft_tw_lds<F>() + G::kGroups * fft_buf_len<F>());
  for (int i = threadIdx.x; i < fft_tw_lds<F>(); i += blockDim.x) tw[i] = twg[i];
  __syncthreads();
  const int g = threadIdx.x / L, lane = threadIdx.x % L;
  float2* buf = smem + fft_tw_lds<F>() + g * fft_buf_len<F>();
  const long npairs = (n + 1) / 2;
  for (long pr = (long)blockIdx.x * G::kGroups + g; pr < npairs;
       pr += (long)gridDim.x * G::kGroups) {
    const bool hasb = 2 * pr + 1 < n;
    float* xa = x + 2 * pr * (long)m;
    float* xb = hasb ? xa + m : xa;
    float2 z[P];
    float sa = 0.f, sb = 0.f;
    const int ml = opaque(m);
#pragma unroll
    for (int s = 0; s < P; ++s) {
      int t = lane + L * s;
      float a = t < ml ? xa[t] : 0.f;
      float b = (hasb && t < ml) ? xb[t] : 0.f;
      z[s] = make_float2(a, b);
      sa += a * a;
      sb += b * b;
    }
    sa = group_sum<L>(sa, red);
    sb = group_sum<L>(sb, red);
    fft<F, L, false>(z, buf, tw, twg, lane);
#pragma unroll
    for (int s = 0; s < P; ++s) z[s] = cmulc(z[s], cspec[s * L + lane]);
    fft<F, L, true>(z, buf, tw, twg, lane);
    float va, vb;
    int ka, kb;
    lag_max<F, L, P>(z, hasb, rev, lane, m, red, va, ka, vb, kb);
    // index 0, the argmax of an all-zero or all-NaN row, where a norm is zero or
    // past the range or the distance is no number (lag_max then has no lag), as
    // the search over centroids leaves it
    const float cn = cnorm[0];
    auto key = [&](float ss, float v, int k) {
      const float den = sqrtf(ss) * cn;
      return ss < INFINITY && cn < INFINITY && den != 0.f && 1.f - (v / (float)F) / den < INFINITY
                 ? k : 0;
    };
    ka = key(sa, va, ka);
    kb = key(sb, vb, kb);
    const int ha = ka + 1 - m, hb = kb + 1 - m;
    const int mo = opaque(m);
#pragma unroll
    for (int s = 0; s < P; ++s) {
      const int pa = lane + L * s - ha, pb = lane + L * s - hb;
      z[s].x = (unsigned)pa < (unsigned)mo ? xa[pa] : 0.f;
      z[s].y = (unsigned)pb < (unsigned)mo ? xb[pb] : 0.f;
    }
    group_sync<L>();  // both rows read before they are overwritten
    const int mw = opaque(m);
#pragma unroll
    for (int s = 0; s < P; ++s) {
      const int t = lane + L * s;
      if (t < mw) {
        xa[t] = z[s].x;
        if (hasb) xb[t] = z[s].y;
      }
    }
  }
}

// --------------------------------------------------------- grouped forms
// The kernels above for many jobs in one launch (GroupTable): each block
// finds its job and runs the body as that job's block bid of nblk.
#define TCX_GROUP_JOB(T)                                                       \
  const int gj_ = group_job(first, njobs, blockIdx.x);                         \
  const T a = jobs[gj_];                                                       \
  const int bid = blockIdx.x - first[gj_], nblk = first[gj_ + 1] - first[gj_];

__global__ __launch_bounds__(256) void k_znorm_group(const ZnormJob* __restrict__ jobs,
                                                     const int* __restrict__ first, int njobs) {
  TCX_GROUP_JOB(ZnormJob)
  znorm_body(bid, nblk, a.x, a.rows, a.m, a.ddof);
}

template <int G, bool kTail, int NV>
__global__ __launch_bounds__(256) void k_znorm_v_group(const ZnormJob* __restrict__ jobs,
                                                       const int* __restrict__ first, int njobs) {
  TCX_GROUP_JOB(ZnormJob)
  znorm_v_body<G, kTail, NV>(bid, nblk, a.x, a.rows, a.m, a.ddof);
}

template <int F>
__global__ __launch_bounds__(FftGeom<F>::kBlock) void k_spectra_group(
    const SpectraJob* __restrict__ jobs, const int* __restrict__ first, int njobs,
    const float2* __restrict__ twg) {
  TCX_GROUP_JOB(SpectraJob)
  spectra_body<F>(bid, nblk, a.y, a.rows, a.m, twg, a.spec, a.norms, a.zero, a.mag, a.bmag);
}

template <int F>
__global__ __launch_bounds__(FftGeom<F>::kBlock, FftGeom<F>::kMinWaves) void k_series_spec_group(
    const SeriesSpecJob* __restrict__ jobs, const int* __restrict__ first, int njobs,
    const float2* __restrict__ twg) {
  TCX_GROUP_JOB(SeriesSpecJob)
  series_spec_body<F>(bid, nblk, a.x, a.n, a.m, twg, a.xs, a.xn, a.xm);
}

template <int NT, int MT, int NS>
__global__ __launch_bounds__(256) void k_bounds_group(const BoundsJob* __restrict__ jobs,
                                                      const int* __restrict__ first, int njobs,
                                                      int kpad, float scale) {
  TCX_GROUP_JOB(BoundsJob)
  bounds_body<NT, MT, NS>(bid, nblk, a.xm, a.n, kpad, a.cm, a.k, a.ld, scale, a.ub);
}

template <int F>
__global__ __launch_bounds__(PruneGeom<F>::kBlock, PruneGeom<F>::kMinWaves) void k_assign_prune_group(
    const PruneJob* __restrict__ jobs, const int* __restrict__ first, int njobs,
    const float2* __restrict__ twg) {
  TCX_GROUP_JOB(PruneJob)
  const long npairs = a.npad ? *a.npad / 2 : a.npairs;  // the grid covers the largest count
  assign_prune_body<F, true>(bid, nblk, a.x, a.xs, a.xn, a.ub, a.ub_ld, a.n, npairs, a.m, a.k,
                             a.cspec, a.cmag, a.cnorm, twg, a.rev, a.order, a.label, a.dist,
                             a.shift, a.changed, a.evals);
}

// ---------------------------------------------------------------- launchers
template <int F>
static size_t sbd_smem() {
  using G = FftGeom<F>;
  return sizeof(float2) * (fft_tw_lds<F>() + G::kGroups * fft_buf_len<F>()) + sizeof(float) * 64;
}

template <int F>
static hipError_t launch_spectra_F(const float* y, int rows, int m, const float2* tw,
                                   float2* spec, float* norms, int* zero, float* mag,
                                   uint16_t* bmag, hipStream_t st) {
  using G = FftGeom<F>;
  int blocks = (rows + G::kGroups - 1) / G::kGroups;
  if (blocks < 1) blocks = 1;
  if (blocks > 4096) blocks = 4096;
  hipLaunchKernelGGL((k_spectra<F>), dim3(blocks), dim3(G::kBlock), sbd_smem<F>(), st, y,
                     rows, m, tw, spec, norms, zero, mag, bmag);
  return hipGetLastError();
}

// Chunks of centroids (blockIdx.y) that fill the device when the pairs alone
// do not: as many as keep at most three waves per SIMD busy.  merge: the chunk
// results take k_split_min, a launch of about 2 us more, which fewer transforms
// than `least` saved per pair do not pay (all distances whole and in chunks:
// n=1 m=12 k=2 17.6, 18.9 us, k=4 20.3, 19.2; n=9000 m=24 k=4 21.8, 23.3; n=3000
// m=50 k=2 20.6, 21.8).  With more than a wave per SIMD in the pairs alone, the
// chunks' own forward transforms cost what they save unless there are some more
// centroids (n=9000 m=60 k=4 24.8, 26.1, n=3000 m=400 k=2 29.5, 30.9).
template <int F>
static int sbd_chunks_F(long npairs, int k, int cus, bool merge) {
  using G = FftGeom<F>;
  const long blocks = (npairs + G::kGroups - 1) / G::kGroups;
  const long waves = blocks * (G::kBlock / kWave);
  // at F = 8192 two per SIMD: one block of the two-wave form per CU
  long c = (F > 4096 ? 8L : 12L) * cus / (waves > 0 ? waves : 1);
  if (c > k) c = k;
  if (c < 2) return 1;
  const long kc = (k + c - 1) / c;
  const int least = F <= 16 || (F <= 64 && npairs > 2048) ? 6 : (F <= 128 ? 3 : 1);
  if (merge && k - kc < least) return 1;
  if (waves > 4L * cus && k < (F <= 128 ? 6 : 3)) return 1;
  return (int)((k + kc - 1) / kc);
}

// Whether a launch has at most two waves per SIMD in all.
template <int F>
static bool few_waves(long blocks, int cus) {
  return blocks * (FftGeom<F>::kBlock / kWave) <= 8L * cus;
}

template <int F, int MODE>
static hipError_t launch_sbd_F(const SbdArgs& a, hipStream_t st) {
  using G = FftGeom<F>;
  long npairs = (a.n + 1) / 2;
  long blocks = (npairs + G::kGroups - 1) / G::kGroups;
  if (blocks < 1) blocks = 1;
  if (blocks > 8192) blocks = 8192;
  const bool split = (MODE == kModeAssign || MODE == kModeSearch) && a.chunks > 1;
  if (split && a.changed) return hipErrorInvalidValue;
  const int chunks = MODE == kModeOwn || a.chunks < 1 ? 1 : a.chunks;
  if (split && (!a.part_dist || !a.part_label || !a.part_shift)) return hipErrorInvalidValue;
  const int kc = (a.k + chunks - 1) / chunks;
  constexpr bool kFew = FftGeom<F>::kFewDense && MODE != kModeOwn;
  auto* kernel = kFew && few_waves<F>(blocks * chunks, a.cus) ? k_sbd<F, MODE, kFew>
                                                              : k_sbd<F, MODE, false>;
  hipLaunchKernelGGL(kernel, dim3((unsigned)blocks, (unsigned)chunks), dim3(G::kBlock),
                     sbd_smem<F>(), st, a.x, a.n, a.m, a.k, kc, a.cspec, a.cnorm, a.tw, a.rev,
                     split ? a.part_label : a.label, split ? a.part_dist : a.dist,
                     split ? a.part_shift : a.shift, a.dmat, split ? nullptr : a.changed,
                     a.ncc_out, a.fixed_label, a.skip);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess || !split) return e;
  hipLaunchKernelGGL(k_split_min, dim3((unsigned)((a.n + 255) / 256)), dim3(256), 0, st,
                     a.part_dist, a.part_label, a.part_shift, a.n, a.m, chunks, a.label, a.dist,
                     a.shift);
  return hipGetLastError();
}

template <int F, bool TG = (F > 1024)>
static size_t prune_smem(int k) {
  using G = PruneGeom<F>;
  return sizeof(float2) * (fft_tw_lds<F, TG>() + G::kGroups * fft_buf_len<F>()) +
         sizeof(float) * 64 + sizeof(float) * 2 * (size_t)k * G::kGroups;
}

// Largest k whose per-group bound lists fit the LDS of one workgroup.
template <int F>
static int prune_max_k_F() {
  const size_t fixed = prune_smem<F>(0);
  const size_t per_k = sizeof(float) * 2 * PruneGeom<F>::kGroups;
  const size_t fit = fixed < (size_t)kLdsBytes ? ((size_t)kLdsBytes - fixed) / per_k : 0;
  return fit < (size_t)kPruneMaxK ? (int)fit : kPruneMaxK;
}

template <int F>
static hipError_t launch_prune_F(const PruneArgs& a, hipStream_t st) {
  using G = PruneGeom<F>;
  const int tuned = tuned_prune_cap(F, a.k, a.n);  // the grid changes no result
  const long cap = tuned > 0 ? tuned : 8192;
  long blocks = (a.npairs + G::kGroups - 1) / G::kGroups;
  if (blocks < 1) blocks = 1;
  if (blocks > cap) blocks = cap;
  const bool pre = a.xs && a.ub;
  constexpr bool kTG = F >= 1024;  // as in the body
  constexpr bool kFew = FftGeom<F>::kFewPrune;
  auto* kernel = pre                                   ? k_assign_prune<F, true, false>
                 : kFew && few_waves<F>(blocks, a.cus) ? k_assign_prune<F, false, kFew>
                                                       : k_assign_prune<F, false, false>;
  const size_t smem = pre ? prune_smem<F>(a.k) : prune_smem<F, kTG>(a.k);
  hipLaunchKernelGGL(kernel, dim3((unsigned)blocks), dim3(G::kBlock), smem, st, a.x,
                     pre ? a.xs : nullptr, pre ? a.xn : nullptr, pre ? a.ub : nullptr,
                     pre ? a.ub_ld : 0, a.n, a.npairs, a.m, a.k, a.cspec, a.cmag, a.cnorm, a.tw,
                     a.rev, a.order, a.label, a.dist, a.shift, a.changed, a.evals, a.skip);
  return hipGetLastError();
}

template <int F>
static hipError_t launch_series_spec_F(const float* x, long n, int m, const float2* tw,
                                       float2* xs, float* xn, uint16_t* xm, hipStream_t st) {
  using G = FftGeom<F>;
  long blocks = ((n + 1) / 2 + G::kGroups - 1) / G::kGroups;
  if (blocks < 1) blocks = 1;
  if (blocks > 8192) blocks = 8192;
  hipLaunchKernelGGL((k_series_spec<F>), dim3((unsigned)blocks), dim3(G::kBlock), sbd_smem<F>(),
                     st, x, n, m, tw, xs, xn, xm);
  return hipGetLastError();
}

// Host: the twiddle table of the length-F transform in the layout the
// Stockham passes read (tw_offset).
void fft_twiddle_table(int F, float2* out) {
  const int P = F / fft_lanes(F);
  const double two_pi = 6.283185307179586476925286766559;
  for (int ns = 1; ns < F;) {
    const int R = F / ns < P ? F / ns : P;
    if (ns > 1) {
      const int off = tw_offset(F, P, ns);
      for (int r = 1; r < R; ++r)
        for (int kk = 0; kk < ns; ++kk) {
          const double a = two_pi * (double)r * (double)kk / ((double)ns * (double)R);
          out[off + (r - 1) * ns + kk] = make_float2((float)std::cos(a), (float)-std::sin(a));
        }
    }
    ns *= R;
  }
}

#define TCX_FOR_EACH_F(X) \
  X(4) X(8) X(16) X(32) X(64) X(128) X(256) X(512) X(1024) X(2048) X(4096) X(8192)

hipError_t launch_spectra(int F, const float* y, int rows, int m, const float2* tw,
                          float2* spec, float* norms, int* zero, float* mag, uint16_t* bmag,
                          hipStream_t st) {
  switch (F) {
#define X(FF) \
  case FF:    \
    return launch_spectra_F<FF>(y, rows, m, tw, spec, norms, zero, mag, bmag, st);
    TCX_FOR_EACH_F(X)
#undef X
    default:
      return hipErrorInvalidValue;
  }
}

int prune_max_k(int F) {
  switch (F) {
#define X(FF) \
  case FF:    \
    return prune_max_k_F<FF>();
    TCX_FOR_EACH_F(X)
#undef X
    default:
      return 0;
  }
}

hipError_t launch_series_spec(int F, const float* x, long n, int m, const float2* tw, float2* xs,
                              float* xn, uint16_t* xm, hipStream_t st) {
  if (n <= 0) return hipSuccess;
  switch (F) {
#define X(FF) \
  case FF:    \
    return launch_series_spec_F<FF>(x, n, m, tw, xs, xn, xm, st);
    TCX_FOR_EACH_F(X)
#undef X
    default:
      return hipErrorInvalidValue;
  }
}

hipError_t launch_bounds(int F, const uint16_t* xm, long n, const uint16_t* cm, int k, float* ub,
                         int ld, hipStream_t st) {
  if (n <= 0 || k <= 0) return hipSuccess;
  if (ld < k || F < 2) return hipErrorInvalidValue;
  const int kpad = bound_kpad(F);
  const float scale = 1.f / (float)F;  // a power of two: exact
  // MT row blocks of 16 per wave share each centroid operand load, NS
  // steps of 16 columns in flight per batch (for one centroid tile the
  // whole row up to 33 steps: F <= 1024 in one batch); 4 waves per block
  auto grid = [&](int mt) { return dim3((unsigned)((n + 64L * mt - 1) / (64L * mt))); };
  const int nsteps = kpad >> 4;
  if (k <= 16 && nsteps <= 9)
    hipLaunchKernelGGL((k_bounds<1, 1, 9>), grid(1), dim3(256), 0, st, xm, n, kpad, cm, k, ld,
                       scale, ub);
  else if (k <= 16 && nsteps <= 17)
    hipLaunchKernelGGL((k_bounds<1, 1, 17>), grid(1), dim3(256), 0, st, xm, n, kpad, cm, k, ld,
                       scale, ub);
  else if (k <= 16)
    hipLaunchKernelGGL((k_bounds<1, 1, 33>), grid(1), dim3(256), 0, st, xm, n, kpad, cm, k, ld,
                       scale, ub);
  else if (k <= 32)
    hipLaunchKernelGGL((k_bounds<2, 2, 11>), grid(2), dim3(256), 0, st, xm, n, kpad, cm, k, ld,
                       scale, ub);
  else
    hipLaunchKernelGGL((k_bounds<4, 1, 11>), grid(1), dim3(256), 0, st, xm, n, kpad, cm, k, ld,
                       scale, ub);
  return hipGetLastError();
}

hipError_t launch_assign_prune(int F, const PruneArgs& a, hipStream_t st) {
  if (a.k > prune_max_k(F)) return hipErrorInvalidValue;
  switch (F) {
#define X(FF) \
  case FF:    \
    return launch_prune_F<FF>(a, st);
    TCX_FOR_EACH_F(X)
#undef X
    default:
      return hipErrorInvalidValue;
  }
}

hipError_t launch_sbd(int F, int mode, const SbdArgs& a, hipStream_t st) {
  switch (F) {
#define X(FF)                                                           \
  case FF:                                                              \
    return mode == kModeAssign   ? launch_sbd_F<FF, kModeAssign>(a, st) \
           : mode == kModeOwn    ? launch_sbd_F<FF, kModeOwn>(a, st)    \
           : mode == kModeSearch ? launch_sbd_F<FF, kModeSearch>(a, st) \
                                 : launch_sbd_F<FF, kModeNcc>(a, st);
    TCX_FOR_EACH_F(X)
#undef X
    default:
      return hipErrorInvalidValue;
  }
}

int sbd_chunks(int F, long n, int k, int cus, bool merge) {
  switch (F) {
#define X(FF) \
  case FF:    \
    return sbd_chunks_F<FF>((n + 1) / 2, k, cus, merge);
    TCX_FOR_EACH_F(X)
#undef X
    default:
      return 1;
  }
}

// Kernels whose dynamic LDS exceeds the default per-launch limit.
hipError_t configure_sbd_kernels() {
  hipError_t e = hipSuccess;
#define X(FF)                                                                                 \
  if (e == hipSuccess)                                                                        \
    e = hipFuncSetAttribute((const void*)k_sbd<FF, kModeAssign, false>,                       \
                            hipFuncAttributeMaxDynamicSharedMemorySize, (int)sbd_smem<FF>()); \
  if (e == hipSuccess)                                                                        \
    e = hipFuncSetAttribute((const void*)k_sbd<FF, kModeNcc, false>,                          \
                            hipFuncAttributeMaxDynamicSharedMemorySize, (int)sbd_smem<FF>()); \
  if (e == hipSuccess)                                                                        \
    e = hipFuncSetAttribute((const void*)k_sbd<FF, kModeOwn, false>,                          \
                            hipFuncAttributeMaxDynamicSharedMemorySize, (int)sbd_smem<FF>()); \
  if (e == hipSuccess)                                                                        \
    e = hipFuncSetAttribute((const void*)k_sbd<FF, kModeSearch, false>,                       \
                            hipFuncAttributeMaxDynamicSharedMemorySize, (int)sbd_smem<FF>()); \
  if (e == hipSuccess)                                                                        \
    e = hipFuncSetAttribute((const void*)k_sbd<FF, kModeAssign, FftGeom<FF>::kFewDense>,      \
                            hipFuncAttributeMaxDynamicSharedMemorySize, (int)sbd_smem<FF>()); \
  if (e == hipSuccess)                                                                        \
    e = hipFuncSetAttribute((const void*)k_sbd<FF, kModeSearch, FftGeom<FF>::kFewDense>,      \
                            hipFuncAttributeMaxDynamicSharedMemorySize, (int)sbd_smem<FF>()); \
  if (e == hipSuccess)                                                                        \
    e = hipFuncSetAttribute((const void*)k_sbd<FF, kModeNcc, FftGeom<FF>::kFewDense>,         \
                            hipFuncAttributeMaxDynamicSharedMemorySize, (int)sbd_smem<FF>()); \
  if (e == hipSuccess)                                                                        \
    e = hipFuncSetAttribute((const void*)k_align<FF>,                                         \
                            hipFuncAttributeMaxDynamicSharedMemorySize, (int)sbd_smem<FF>()); \
  if (e == hipSuccess)                                                                        \
    e = hipFuncSetAttribute((const void*)k_spectra<FF>,                                       \
                            hipFuncAttributeMaxDynamicSharedMemorySize, (int)sbd_smem<FF>()); \
  if (e == hipSuccess)                                                                        \
    e = hipFuncSetAttribute((const void*)k_assign_prune<FF, false, false>,                    \
                            hipFuncAttributeMaxDynamicSharedMemorySize,                       \
                            (int)prune_smem<FF>(prune_max_k_F<FF>()));                        \
  if (e == hipSuccess)                                                                        \
    e = hipFuncSetAttribute((const void*)k_assign_prune<FF, true, false>,                     \
                            hipFuncAttributeMaxDynamicSharedMemorySize,                       \
                            (int)prune_smem<FF>(prune_max_k_F<FF>()));                        \
  if (e == hipSuccess)                                                                        \
    e = hipFuncSetAttribute((const void*)k_assign_prune<FF, false, FftGeom<FF>::kFewPrune>,   \
                            hipFuncAttributeMaxDynamicSharedMemorySize,                       \
                            (int)prune_smem<FF>(prune_max_k_F<FF>()));                        \
  if (e == hipSuccess)                                                                        \
    e = hipFuncSetAttribute((const void*)k_series_spec<FF>,                                   \
                            hipFuncAttributeMaxDynamicSharedMemorySize, (int)sbd_smem<FF>()); \
  if (e == hipSuccess)                                                                        \
    e = hipFuncSetAttribute((const void*)k_series_spec_group<FF>,                             \
                            hipFuncAttributeMaxDynamicSharedMemorySize, (int)sbd_smem<FF>()); \
  if (e == hipSuccess)                                                                        \
    e = hipFuncSetAttribute((const void*)k_spectra_group<FF>,                                 \
                            hipFuncAttributeMaxDynamicSharedMemorySize, (int)sbd_smem<FF>()); \
  if (e == hipSuccess)                                                                        \
    e = hipFuncSetAttribute((const void*)k_assign_prune_group<FF>,                            \
                            hipFuncAttributeMaxDynamicSharedMemorySize,                       \
                            (int)prune_smem<FF>(prune_max_k_F<FF>()));
  TCX_FOR_EACH_F(X)
#undef X
  return e;
}

// The form of a z-norm: 0, three passes over the row (longer than a wave
// holds); else the vectors a lane holds (1: 16 lanes per row with up to two,
// for rows of at most 128 values), negative with the tail.
int znorm_form(const float* x, int m) {
  if (m > 4096) return 0;
  int nv = 1;
  if (m > 128)
    for (nv = 2; 4 * kWave * nv < m;) nv *= 2;
  return (m & 3) == 0 && (reinterpret_cast<uintptr_t>(x) & 15) == 0 ? nv : -nv;
}

long znorm_blocks(int form, long rows) {
  const long per = form == 1 || form == -1 ? 16 : 4;
  return (rows + per - 1) / per;
}

#define TCX_FOR_EACH_ZNORM(X)                                                         \
  X(1, 16, false, 2) X(2, 64, false, 2) X(4, 64, false, 4) X(8, 64, false, 8)         \
  X(16, 64, false, 16) X(-1, 16, true, 2) X(-2, 64, true, 2) X(-4, 64, true, 4)       \
  X(-8, 64, true, 8) X(-16, 64, true, 16)

hipError_t launch_znorm(float* x, long rows, int m, int ddof, hipStream_t st) {
  if (rows <= 0) return hipSuccess;
  const int form = znorm_form(x, m);
  const dim3 grid((unsigned)znorm_blocks(form, rows));
  switch (form) {
#define X(FORM, G, TAIL, NV)                                                                     \
  case FORM:                                                                                     \
    hipLaunchKernelGGL((k_znorm_v<G, TAIL, NV>), grid, dim3(256), 0, st, x, rows, m, ddof);      \
    break;
    TCX_FOR_EACH_ZNORM(X)
#undef X
    default:
      hipLaunchKernelGGL(k_znorm, grid, dim3(256), 0, st, x, rows, m, ddof);
  }
  return hipGetLastError();
}

// ------------------------------------------------ grouped-form launchers
hipError_t launch_znorm_group(const GroupTable& g, int form, hipStream_t st) {
  if (g.blocks <= 0) return hipSuccess;
  const ZnormJob* j = static_cast<const ZnormJob*>(g.jobs);
  switch (form) {
    case 0:
      hipLaunchKernelGGL(k_znorm_group, dim3(g.blocks), dim3(256), 0, st, j, g.first, g.njobs);
      break;
#define X(FORM, G, TAIL, NV)                                                                     \
  case FORM:                                                                                     \
    hipLaunchKernelGGL((k_znorm_v_group<G, TAIL, NV>), dim3(g.blocks), dim3(256), 0, st, j,       \
                       g.first, g.njobs);                                                        \
    break;
    TCX_FOR_EACH_ZNORM(X)
#undef X
    default:
      return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

template <int F>
static long groups_blocks(long units) {  // launch_spectra_F / launch_*_F block counts
  long b = (units + FftGeom<F>::kGroups - 1) / FftGeom<F>::kGroups;
  return b < 1 ? 1 : b;
}

long series_spec_blocks(int F, long n) {
  switch (F) {
#define X(FF) \
  case FF:    \
    return std::min(groups_blocks<FF>((n + 1) / 2), 8192L);
    TCX_FOR_EACH_F(X)
#undef X
    default:
      return 0;
  }
}

long spectra_blocks(int F, long rows) {
  switch (F) {
#define X(FF) \
  case FF:    \
    return std::min(groups_blocks<FF>(rows), 4096L);
    TCX_FOR_EACH_F(X)
#undef X
    default:
      return 0;
  }
}

long prune_blocks(int F, long npairs, int k, long n) {
  const int tuned = tuned_prune_cap(F, k, n);  // the grid changes no result
  const long cap = tuned > 0 ? tuned : 8192;
  switch (F) {
#define X(FF)                                                                   \
  case FF: {                                                                    \
    long b = (npairs + PruneGeom<FF>::kGroups - 1) / PruneGeom<FF>::kGroups;     \
    return b < 1 ? 1 : (b > cap ? cap : b);                                     \
  }
    TCX_FOR_EACH_F(X)
#undef X
    default:
      return 0;
  }
}

size_t prune_lds(int F, int k) {
  switch (F) {
#define X(FF) \
  case FF:    \
    return prune_smem<FF>(k);
    TCX_FOR_EACH_F(X)
#undef X
    default:
      return 0;
  }
}

hipError_t launch_series_spec_group(int F, const GroupTable& g, const float2* tw, hipStream_t st) {
  if (g.blocks <= 0) return hipSuccess;
  const SeriesSpecJob* j = static_cast<const SeriesSpecJob*>(g.jobs);
  switch (F) {
#define X(FF)                                                                                    \
  case FF:                                                                                       \
    hipLaunchKernelGGL((k_series_spec_group<FF>), dim3(g.blocks), dim3(FftGeom<FF>::kBlock),      \
                       sbd_smem<FF>(), st, j, g.first, g.njobs, tw);                            \
    break;
    TCX_FOR_EACH_F(X)
#undef X
    default:
      return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

hipError_t launch_spectra_group(int F, const GroupTable& g, const float2* tw, hipStream_t st) {
  if (g.blocks <= 0) return hipSuccess;
  const SpectraJob* j = static_cast<const SpectraJob*>(g.jobs);
  switch (F) {
#define X(FF)                                                                                    \
  case FF:                                                                                       \
    hipLaunchKernelGGL((k_spectra_group<FF>), dim3(g.blocks), dim3(FftGeom<FF>::kBlock),          \
                       sbd_smem<FF>(), st, j, g.first, g.njobs, tw);                            \
    break;
    TCX_FOR_EACH_F(X)
#undef X
    default:
      return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

// The forms of launch_bounds: 0 <1,1,9>, 1 <1,1,17>, 2 <1,1,33> (k <= 16),
// 3 <2,2,11> (k <= 32), 4 <4,1,11>.
int bounds_form(int F, int k) {
  const int nsteps = bound_kpad(F) >> 4;
  if (k <= 16) return nsteps <= 9 ? 0 : (nsteps <= 17 ? 1 : 2);
  return k <= 32 ? 3 : 4;
}

long bounds_blocks(int form, long n) {
  const long mt = form == 3 ? 2 : 1;
  return (n + 64 * mt - 1) / (64 * mt);
}

hipError_t launch_bounds_group(int F, int form, const GroupTable& g, hipStream_t st) {
  if (g.blocks <= 0) return hipSuccess;
  const BoundsJob* j = static_cast<const BoundsJob*>(g.jobs);
  const int kpad = bound_kpad(F);
  const float scale = 1.f / (float)F;
  switch (form) {
    case 0:
      hipLaunchKernelGGL((k_bounds_group<1, 1, 9>), dim3(g.blocks), dim3(256), 0, st, j, g.first,
                         g.njobs, kpad, scale);
      break;
    case 1:
      hipLaunchKernelGGL((k_bounds_group<1, 1, 17>), dim3(g.blocks), dim3(256), 0, st, j, g.first,
                         g.njobs, kpad, scale);
      break;
    case 2:
      hipLaunchKernelGGL((k_bounds_group<1, 1, 33>), dim3(g.blocks), dim3(256), 0, st, j, g.first,
                         g.njobs, kpad, scale);
      break;
    case 3:
      hipLaunchKernelGGL((k_bounds_group<2, 2, 11>), dim3(g.blocks), dim3(256), 0, st, j, g.first,
                         g.njobs, kpad, scale);
      break;
    case 4:
      hipLaunchKernelGGL((k_bounds_group<4, 1, 11>), dim3(g.blocks), dim3(256), 0, st, j, g.first,
                         g.njobs, kpad, scale);
      break;
    default:
      return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

hipError_t launch_assign_prune_group(int F, const GroupTable& g, const float2* tw,
                                     hipStream_t st) {
  if (g.blocks <= 0) return hipSuccess;
  const PruneJob* j = static_cast<const PruneJob*>(g.jobs);
  switch (F) {
#define X(FF)                                                                                    \
  case FF:                                                                                       \
    if (g.lds > prune_smem<FF>(prune_max_k_F<FF>())) return hipErrorInvalidValue;                \
    hipLaunchKernelGGL((k_assign_prune_group<FF>), dim3(g.blocks), dim3(PruneGeom<FF>::kBlock),   \
                       g.lds, st, j, g.first, g.njobs, tw);                                     \
    break;
    TCX_FOR_EACH_F(X)
#undef X
    default:
      return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

template <int F>
static hipError_t launch_align_F(float* x, long n, int m, const float2* cspec, const float* cnorm,
                                 const int* czero, const float2* tw, int rev, hipStream_t st) {
  using G = FftGeom<F>;
  const long blocks = std::min(groups_blocks<F>((n + 1) / 2), 8192L);
  hipLaunchKernelGGL((k_align<F>), dim3((unsigned)blocks), dim3(G::kBlock), sbd_smem<F>(), st, x,
                     n, m, cspec, cnorm, czero, tw, rev);
  return hipGetLastError();
}

hipError_t launch_align(int F, float* x, long n, int m, const float2* cspec, const float* cnorm,
                        const int* czero, const float2* tw, int rev, hipStream_t st) {
  if (n <= 0) return hipSuccess;
  switch (F) {
#define X(FF) \
  case FF:    \
    return launch_align_F<FF>(x, n, m, cspec, cnorm, czero, tw, rev, st);
    TCX_FOR_EACH_F(X)
#undef X
    default:
      return hipErrorInvalidValue;
  }
}

}  // namespace tcx
