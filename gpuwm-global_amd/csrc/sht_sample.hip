// Spectral fields evaluated at arbitrary points (reference
// spectral/sampling.py:382-515: sample_scalar, sample_gradient, sample_wind).
//
// Per order m a field's amplitude at a point is a sum over degrees of
// coefficient times basis value, turned by e^{i m lambda} and added into the
// output.  The amplitudes of 16 PT points and 16 CT columns (real and
// imaginary parts of 8 fields each) are one wavefront's tiles of
//     A (points x 4 degrees) B (4 degrees x columns)
// on v_mfma_f64_16x16x4_f64 (v_mfma_f32_16x16x4_f32 for the float32 sampler),
// four degrees of one order per step.  The basis is generated as it is used:
// a lane runs the normalized associated-Legendre recurrence of its point in
// FP64 (reference legendre.py:86-146, the reference's operand order in every
// expression but the derivative's division, see rd below; this file is
// compiled with -ffp-contract=off), four degrees a step, and hands them over
// in A's layout through the wavefront's LDS.  No basis cube is stored (the
// reference's device path materialises a (2K x points) basis per point chunk,
// 8 bytes of HBM traffic per value).
//
// Bound: the FP64 matrix pipe, whose peak equals the vector peak; what the
// former kernel (lane = two points, coefficients by scalar loads) lacked was
// operands, since a scalar load feeds one wavefront's multiply-adds and waits
// for all loads at once.  Here a coefficient is loaded once per lane for PT
// MFMAs and a basis value feeds CT.  T383, 30,000 points: 40 fields 11.25 ->
// 7.10 ms in float64 (51 TFLOP/s; 62 is what a large FP64 matrix product
// reaches), 9.18 -> 4.74 ms in float32 (bound by the FP64 recurrence); 3 fields
// at 300 points 2.84 -> 0.73 ms.
// Gradients and winds run the derivative's recurrence beside two MFMAs a value
// (nine FP64 operations, not four), so there it counts as much: lanes that
// share a point form the derivative of one degree each, the last odd column
// tile runs alone, and one column tile of many points takes four point tiles,
// whose lanes share no point.  Gradients, T383, 30,000 points, former kernel ->
// every lane all derivatives and no tile alone -> here: 40 fields float64 19.9
// -> 19.2 -> 16.1 ms, float32 19.6 -> 14.4 -> 12.1; 8 fields float64 4.26 ->
// 4.76 -> 3.86; T127, 20 fields 1.40 -> 1.61 -> 1.31, 8 fields 0.51 -> 0.62 ->
// 0.53.
//
// Precision: F32 = false accumulates in FP64; F32 = true rounds each basis
// value to fp32 and accumulates an order's terms in fp32 before the FP64 sum
// (the reference's "float32" sampler, sampling.py:30-44).
#include "sht_kernels.h"

#include <math.h>

#include <algorithm>
#include <type_traits>

namespace sht {

// Packed triangle index of (n, m), order-major (reference sampling.py:72-80).
__device__ __forceinline__ long long tri_index(int T, int n, int m) {
  return (long long)m * (T + 1) - ((long long)m * (m - 1)) / 2 + (n - m);
}

// (count, T+1, T+1) complex64 [n, m] -> (K, ldc) complex, fields fastest:
// complex128 for the float64 sampler, complex64 for the float32 one; columns
// past the live fields are zero.  Winds: column 2l is psi and 2l + 1 chi of
// level l, from vorticity / divergence by the inverse Laplacian.
__global__ void sample_pack_kernel(SamplePackArgs a) {
  const int T1 = a.T + 1;
  const long long total = (long long)a.ldc * T1 * T1;
  for (long long e = blockIdx.x * (long long)blockDim.x + threadIdx.x; e < total;
       e += (long long)gridDim.x * blockDim.x) {
    const int m = (int)(e % T1);
    const int n = (int)((e / T1) % T1);
    const int col = (int)(e / ((long long)T1 * T1));
    if (m > n) continue;
    float2 v = make_float2(0.f, 0.f);
    if (a.wind) {
      // the inverse Laplacian in the arithmetic of the spectral operator
      // kernel (c / lambda_n in fp32, lambda_n = -n(n+1)/a^2 rounded once),
      // so psi and chi are inverse_laplacian's bits
      const int level = col >> 1;
      if (level < a.count && n > 0) {
        const float2* src = (col & 1) ? a.in1 : a.in0;
        const float2 c = src[((size_t)level * T1 + n) * T1 + m];
        const float eig = (float)(-((double)n * ((double)n + 1.0)) / (a.radius * a.radius));
        v = make_float2(c.x / eig, c.y / eig);
      }
    } else if (col < a.count) {
      v = a.in0[((size_t)col * T1 + n) * T1 + m];
    }
    const long long o = tri_index(a.T, n, m) * a.ldc + col;
    if (a.f64) static_cast<double2*>(a.out)[o] = make_double2(v.x, v.y);
    else static_cast<float2*>(a.out)[o] = v;
  }
}

typedef double d4 __attribute__((ext_vector_type(4)));
typedef float f4 __attribute__((ext_vector_type(4)));
template <bool F32>
struct SampleAcc {
  using T = typename std::conditional<F32, float, double>::type;
  using D = typename std::conditional<F32, f4, d4>::type;
};
__device__ __forceinline__ void sample_mfma(d4& acc, double a, double b) {
  acc = __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, acc, 0, 0, 0);
}
__device__ __forceinline__ void sample_mfma(f4& acc, float a, float b) {
  acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, acc, 0, 0, 0);
}

// The outputs of one point from its two sums (s0: values, or zonal sums
// d/dlambda; s1: meridional sums d/dphi).  KIND 0: the field; 1: east and
// north derivatives per metre; 2: u and v from column pairs (psi, chi):
// u = -north(psi) + east(chi), v = east(psi) + north(chi) (reference
// sampling.py:481-515).
template <int KIND>
__device__ __forceinline__ void sample_store(int col, int p, int npts, int nout, double s0,
                                             double s1, double s0b, double s1b, double radius,
                                             double coslat, double* out0, double* out1) {
  if constexpr (KIND == 0) {
    if (col < nout) out0[(size_t)col * npts + p] = s0;
  } else if constexpr (KIND == 1) {
    if (col < nout) {
      out0[(size_t)col * npts + p] = s0 / (radius * coslat);
      out1[(size_t)col * npts + p] = s1 / radius;
    }
  } else {
    const int level = col >> 1;
    if (level < nout) {
      const double east_scale = radius * coslat;
      const double psi_e = s0 / east_scale, psi_n = s1 / radius;
      const double chi_e = s0b / east_scale, chi_n = s1b / radius;
      out0[(size_t)level * npts + p] = -psi_n + chi_e;
      out1[(size_t)level * npts + p] = psi_e + chi_n;
    }
  }
}

// One wavefront: 16 PT points x CT column tiles (8 fields each) x one part of
// the order range (orders mcut[r] .. mcut[r+1]-1, cut so the parts hold equal
// shares of the triangle); the four wavefronts of a block take neighbouring
// points and read the same coefficients.  With one part the outputs are
// stored; with several the two raw sums per (column, point) go to part r of
// `partial` and sample_reduce_kernel adds the parts in order.  An output's
// arithmetic depends on neither PT, CT nor its neighbours.
// MFMA operands: lane l = (g = l / 16, q = l % 16); A holds point q of the
// tile at degree n0 + g, B degree n0 + g at column q; accumulator register i
// is point g + 4 i (FP64) or 4 g + i (fp32) at column q.
template <int PT, int KIND, bool F32>
struct SampleShared {
  static constexpr int NP = 16 * PT;            // points of a wavefront
  static constexpr int NB = KIND != 0 ? 2 : 1;  // bases: P, dP/dphi
  // per wavefront: basis values [2 buffers][P, dP][degree][point], then
  // cos and sin of the order's phase per point
  typename SampleAcc<F32>::T A[4][2][NB][4][NP];
  double E[4][2][NP];
};

template <int PT, int CT, int KIND, bool F32>
__device__ __forceinline__ void sample_tiles(
    SampleShared<PT, KIND, F32>& sh, int ct0,
    const typename SampleAcc<F32>::T* __restrict__ coef, const double* __restrict__ rec,
    const double* __restrict__ diag, const double* __restrict__ sin_lat,
    const double* __restrict__ cos_lat, const double* __restrict__ lon, const SampleCuts& cuts,
    int T, int npts, int ldc, int nout, double radius, double* __restrict__ out0,
    double* __restrict__ out1, double* __restrict__ partial) {
  using Acc = typename SampleAcc<F32>::T;
  using D = typename SampleAcc<F32>::D;
  constexpr bool GRAD = KIND != 0;
  constexpr int NP = 16 * PT, NB = GRAD ? 2 : 1;
  auto& sA = sh.A;
  auto& sE = sh.E;
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int g = lane >> 4, q = lane & 15;
  const int p0 = ((int)blockIdx.x * 4 + wv) * NP;
  if (p0 >= npts) return;  // wave-uniform; no block barrier in this kernel
  const int r = blockIdx.z;
  const int m0 = cuts.m[r], m1 = cuts.m[r + 1];
  const long long K = (long long)(T + 1) * (T + 2) / 2;
  const double* rec_a = rec;
  const double* rec_b = rec + K;
  const double* rec_c = rec + 2 * K;
  const double* diag_f = diag;
  const double* diag_g = diag + (T + 1);
  const double pi = 3.14159265358979323846;

  // the recurrence of point lane % NP (every 64 / NP-th lane the same one)
  const int mine = lane % NP;
  const int pp = min(p0 + mine, npts - 1);  // past the end: a real point
  const double x = sin_lat[pp], lam = lon[pp];
  const double root = sqrt(fmax(0.0, 1.0 - x * x));
  // dP = root (n x P - c P_{n-1}) / (x^2 - 1): the division by the point's
  // constant (x^2 - 1) is one multiplication by rd = root / (x^2 - 1), one
  // rounding more than the reference's form and ~10 FP64 instructions less
  // per (n, m) step
  const double rd = GRAD ? root / (x * x - 1.0) : 0.0;
  double dg = 1.0 / sqrt(4.0 * pi);
  for (int mm = 1; mm <= m0; ++mm) dg = diag_f[mm] * root * dg;  // P_{m0 m0}

  double o[NB][PT][CT][4];
#pragma unroll
  for (int b = 0; b < NB; ++b)
#pragma unroll
    for (int t = 0; t < PT; ++t)
#pragma unroll
      for (int c = 0; c < CT; ++c)
#pragma unroll
        for (int i = 0; i < 4; ++i) o[b][t][c][i] = 0.0;

  const size_t row = 2 * (size_t)ldc;  // values of one packed (n, m)
  for (int m = m0; m < m1; ++m) {
    const long long k0 = tri_index(T, m, m);
    const int len = T + 1 - m;  // degrees
    const Acc* cp = coef + ((size_t)k0 + g) * row + 16 * ct0 + q;  // degree m + g
    D acc[NB][PT][CT];
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
      for (int t = 0; t < PT; ++t)
#pragma unroll
        for (int c = 0; c < CT; ++c) acc[b][t][c] = D{0, 0, 0, 0};
    // degrees m + j + g of the step at j; past T the order's last row, taken
    // as 0 by `tail` steps
    auto load_b = [&](Acc(&v)[CT], int j) {
      const Acc* at = cp + (long long)(min(j + g, len - 1) - g) * (long long)row;
#pragma unroll
      for (int c = 0; c < CT; ++c) v[c] = at[16 * c];
    };
    double prev = 0.0, prev2 = 0.0;  // P of the two degrees before
    // basis values of the step at j into buffer `buf`; FIRST: j = 0, whose
    // degrees m and m + 1 have their own rules; TAIL: degrees past T are 0
    auto basis = [&](auto FIRST, auto TAIL, int j, int buf) {
      constexpr bool first = decltype(FIRST)::value, tail = decltype(TAIL)::value;
      // the lanes that share a point form its four values of P each, and
      // between them those of dP and the LDS writes
      constexpr int SHARE = 64 / NP, EACH = 4 / SHARE;
      const int part = lane / NP;
      double P[4], rc[EACH];
      double ra[4], rb[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const long long k = k0 + (tail ? min(j + u, len - 1) : j + u);
        ra[u] = rec_a[k];
        rb[u] = rec_b[k];
      }
      if constexpr (GRAD)
#pragma unroll
        for (int e = 0; e < EACH; ++e) {
          const int u = (SHARE > 1 ? part * EACH : 0) + e;
          rc[e] = rec_c[k0 + (tail ? min(j + u, len - 1) : j + u)];
        }
      double below = prev;  // P one degree below this lane's first
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        double v;
        if (first && u == 0) v = dg;
        else if (first && u == 1) v = diag_g[m] * x * dg;
        else v = ra[u] * (x * prev - rb[u] * prev2);
        if constexpr (GRAD)
          if (u > 0 && u % EACH == 0) below = part * EACH == u ? prev : below;
        prev2 = prev;
        prev = v;
        P[u] = tail && j + u >= len ? 0.0 : v;
      }
#pragma unroll
      for (int e = 0; e < EACH; ++e) {
        double v = P[e];
#pragma unroll
        for (int h = 1; h < SHARE; ++h) v = part == h ? P[h * EACH + e] : v;
        sA[wv][buf][0][part * EACH + e][mine] = (Acc)v;
        if constexpr (GRAD) {
          // at degree m the second term is 0 (rec_c and P below); past T the
          // basis value is 0 and so is the derivative
          const int u = (SHARE > 1 ? part * EACH : 0) + e;
          double d = rd * ((double)(m + j + u) * x * v - rc[e] * below);
          if (first && u == 0 && m == 0) d = 0.0;
          if (tail) d = j + u < len ? d : 0.0;
          sA[wv][buf][NB - 1][part * EACH + e][mine] = (Acc)d;
          below = v;
        }
      }
    };
    auto lds_sync = [] {  // this wavefront's LDS accesses, in order
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    };
    // one step: the A fragments of `buf`, its coefficients v; the next step's
    // basis values and the coefficients two steps ahead are started before
    // the MFMAs.  TAIL: this step or the next may pass T.
    auto step = [&](Acc(&v)[CT], int j, int buf, auto TAIL) {
      Acc a[NB][PT], b[CT];
#pragma unroll
      for (int s = 0; s < NB; ++s)
#pragma unroll
        for (int t = 0; t < PT; ++t) a[s][t] = sA[wv][buf][s][g][16 * t + q];
#pragma unroll
      for (int c = 0; c < CT; ++c) {
        b[c] = v[c];
        if (decltype(TAIL)::value) b[c] = j + g < len ? b[c] : Acc(0);
      }
      load_b(v, j + 8);
      basis(std::false_type{}, TAIL, j + 4, buf ^ 1);
      lds_sync();
#pragma unroll
      for (int s = 0; s < NB; ++s)
#pragma unroll
        for (int t = 0; t < PT; ++t)
#pragma unroll
          for (int c = 0; c < CT; ++c) sample_mfma(acc[s][t][c], a[s][t], b[c]);
    };
    Acc v0[CT], v1[CT];
    load_b(v0, 0);
    load_b(v1, 4);
    basis(std::true_type{}, std::true_type{}, 0, 0);
    lds_sync();
    int j = 0;
    for (; j + 12 <= len; j += 8) {  // both steps and the basis values after them whole
      step(v0, j, 0, std::false_type{});
      step(v1, j + 4, 1, std::false_type{});
    }
    for (int buf = 0; j < len; j += 4, buf ^= 1) {  // at most three steps
      step(v0, j, buf, std::true_type{});
#pragma unroll
      for (int c = 0; c < CT; ++c) {
        const Acc y = v0[c];
        v0[c] = v1[c];
        v1[c] = y;
      }
    }
    // the order is complete: turn its amplitudes by e^{i m lambda}.  The real
    // column of a field takes cos (for d/dlambda: -m sin), the imaginary one
    // -sin (-m cos); the two are added at the end.
    const double mult = m == 0 ? 1.0 : 2.0;
    {
      double sm, cm;
      sincos((double)m * lam, &sm, &cm);
      sE[wv][0][mine] = mult * cm;
      sE[wv][1][mine] = mult * sm;
    }
    lds_sync();
    const bool im = q & 1;
#pragma unroll
    for (int t = 0; t < PT; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int at = 16 * t + (F32 ? 4 * g + i : g + 4 * i);
        const double cm = sE[wv][0][at], sm = sE[wv][1][at];
        const double w = im ? -sm : cm;
        if constexpr (KIND == 0) {
#pragma unroll
          for (int c = 0; c < CT; ++c) o[0][t][c][i] = fma((double)acc[0][t][c][i], w, o[0][t][c][i]);
        } else {
          const double wz = -(double)m * (im ? cm : sm);
#pragma unroll
          for (int c = 0; c < CT; ++c) {
            o[0][t][c][i] = fma((double)acc[0][t][c][i], wz, o[0][t][c][i]);
            o[NB - 1][t][c][i] = fma((double)acc[NB - 1][t][c][i], w, o[NB - 1][t][c][i]);
          }
        }
      }
    lds_sync();  // the phases are read before the next order's land
    if (m + 1 <= T) dg = diag_f[m + 1] * root * dg;
  }

  // real and imaginary shares meet; lane pair (2 f, 2 f + 1) of a tile is field f
  const size_t plane = (size_t)ldc * npts;
#pragma unroll
  for (int t = 0; t < PT; ++t)
#pragma unroll
    for (int c = 0; c < CT; ++c)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        double s0 = o[0][t][c][i], s1 = GRAD ? o[NB - 1][t][c][i] : 0.0;
        s0 += __shfl_xor(s0, 1);
        if constexpr (GRAD) s1 += __shfl_xor(s1, 1);
        const int p = p0 + 16 * t + (F32 ? 4 * g + i : g + 4 * i);
        const int col = 8 * (ct0 + c) + (q >> 1);
        const bool ok = p < npts && !(q & 1);
        if (gridDim.z > 1) {
          // raw sums of this part: partial[r][col][p], then [R + r] for the second
          if (ok) {
            partial[(size_t)r * plane + (size_t)col * npts + p] = s0;
            if constexpr (GRAD)
              partial[(size_t)(gridDim.z + r) * plane + (size_t)col * npts + p] = s1;
          }
          continue;
        }
        double s0b = 0.0, s1b = 0.0;
        if constexpr (KIND == 2) {  // the level's chi, two lanes on
          s0b = __shfl_xor(s0, 2);
          s1b = __shfl_xor(s1, 2);
        }
        if (ok && !(KIND == 2 && (q & 2)))
          sample_store<KIND>(col, p, npts, nout, s0, s1, s0b, s1b, radius,
                             KIND == 0 ? 0.0 : cos_lat[p], out0, out1);
      }
}

template <int PT, int CT, int KIND, bool F32>
__global__ void __launch_bounds__(256, 2) sample_kernel(
    const typename SampleAcc<F32>::T* __restrict__ coef, const double* __restrict__ rec,
    const double* __restrict__ diag, const double* __restrict__ sin_lat,
    const double* __restrict__ cos_lat, const double* __restrict__ lon, SampleCuts cuts, int T,
    int npts, int ldc, int nout, double radius, double* __restrict__ out0,
    double* __restrict__ out1, double* __restrict__ partial) {
  __shared__ SampleShared<PT, KIND, F32> sh;
  const int tiles = ldc / 8, ct0 = (int)blockIdx.y * CT;
  if constexpr (KIND != 0 && CT == 2) {
    if (ct0 + CT > tiles) {  // block-uniform: one tile is left
      sample_tiles<PT, 1, KIND, F32>(sh, ct0, coef, rec, diag, sin_lat, cos_lat, lon, cuts, T,
                                     npts, ldc, nout, radius, out0, out1, partial);
      return;
    }
  }
  // the last group of column tiles starts early enough to be whole: its first
  // tiles may be another group's too, with the same bits
  sample_tiles<PT, CT, KIND, F32>(sh, min(ct0, tiles - CT), coef, rec, diag, sin_lat, cos_lat, lon,
                                  cuts, T, npts, ldc, nout, radius, out0, out1, partial);
}

// Adds the R parts' sums of each (column, point) in part order and stores
// the outputs; one thread per (column or column pair, point).
template <int KIND>
__global__ void sample_reduce_kernel(const double* __restrict__ partial, int nparts, int ldc,
                                     int npts, int nout, double radius,
                                     const double* __restrict__ cos_lat, double* out0,
                                     double* out1) {
  constexpr int STRIDE = KIND == 2 ? 2 : 1;
  const long long total = (long long)(ldc / STRIDE) * npts;
  const size_t plane = (size_t)ldc * npts;
  for (long long e = blockIdx.x * (long long)blockDim.x + threadIdx.x; e < total;
       e += (long long)gridDim.x * blockDim.x) {
    const int p = (int)(e % npts);
    const int col = (int)(e / npts) * STRIDE;
    if ((KIND == 2 ? col >> 1 : col) >= nout) continue;
    double s[4] = {0.0, 0.0, 0.0, 0.0};  // s0, s1 of col; s0, s1 of col + 1 (winds)
    for (int r = 0; r < nparts; ++r) {
      const size_t o = (size_t)r * plane + (size_t)col * npts + p;
      s[0] += partial[o];
      if (KIND != 0) s[1] += partial[(size_t)nparts * plane + o];
      if (KIND == 2) {
        s[2] += partial[o + npts];
        s[3] += partial[(size_t)nparts * plane + o + npts];
      }
    }
    sample_store<KIND>(col, p, npts, nout, s[0], s[1], s[2], s[3], radius,
                       KIND == 0 ? 0.0 : cos_lat[p], out0, out1);
  }
}

}  // namespace sht

extern "C" hipError_t sht_launch_sample_pack(const sht::SamplePackArgs* a, hipStream_t s) {
  const long long total = (long long)a->ldc * (a->T + 1) * (a->T + 1);
  if (total <= 0) return hipSuccess;
  long long blocks = (total + 255) / 256;
  if (blocks > 65536) blocks = 65536;
  hipLaunchKernelGGL(sht::sample_pack_kernel, dim3((unsigned)blocks), dim3(256), 0, s, *a);
  return hipGetLastError();
}

namespace {

template <int PT, int CT, int KIND, bool F32>
hipError_t launch_sample_tile(const sht::SampleArgs& a, hipStream_t s) {
  const int tiles = a.ldc / 8;
  if (tiles < CT) return hipErrorInvalidValue;  // the first column would be negative
  const dim3 g((unsigned)((a.npts + 64 * PT - 1) / (64 * PT)), (unsigned)((tiles + CT - 1) / CT),
               (unsigned)a.cuts.parts);
  hipLaunchKernelGGL((sht::sample_kernel<PT, CT, KIND, F32>), g, dim3(256), 0, s,
                     static_cast<const typename sht::SampleAcc<F32>::T*>(a.coef), a.rec, a.diag,
                     a.sin_lat, a.cos_lat, a.lon, a.cuts, a.T, a.npts, a.ldc, a.nout, a.radius,
                     a.out0, a.out1, a.partial);
  return hipGetLastError();
}

// The tile of a wavefront.  Two point tiles and as many column tiles as the
// registers of two wavefronts per SIMD hold (five for values, two for the two
// bases of gradients and winds) feed the most MFMAs per basis value and
// coefficient; fewer points or columns take smaller tiles, so that the launch
// still has a wavefront for each of the chip's 1024 SIMDs.  One column tile of
// derivatives takes four point tiles from two wavefronts per SIMD up.  ct is the
// even share of the column tiles between the groups, so it is never above their
// number: a group wider than all of them would begin at a negative column.
struct SampleTile {
  int pt, ct;
};
SampleTile sample_tile(int kind, int ldc, int npts, int parts) {
  const long long most = kind == 0 ? 5 : 2, tiles = ldc / 8;
  const long long groups = (tiles + most - 1) / most;
  const int ct = (int)((tiles + groups - 1) / groups);
  const long long waves2 = ((long long)npts + 31) / 32 * groups * parts;
  const long long waves1 = ((long long)npts + 15) / 16 * groups * parts;
  const long long waves4 = ((long long)npts + 63) / 64 * groups * parts;
  if (kind != 0 && ct == 1 && waves4 >= 2048) return {4, 1};
  if (waves2 >= 2048 || (waves2 >= 1024 && ct >= 2)) return {2, ct};
  if (waves1 >= 1024 && ct >= 2) return {1, ct};
  return {1, 1};
}

template <int KIND, bool F32>
hipError_t launch_sample_kind(const sht::SampleArgs& a, hipStream_t s) {
  const SampleTile t = sample_tile(KIND, a.ldc, a.npts, a.cuts.parts);
#define SHT_TILE(PT, CT) \
  if (t.pt == PT && t.ct == CT) return launch_sample_tile<PT, CT, KIND, F32>(a, s)
  SHT_TILE(1, 1);
  SHT_TILE(1, 2);
  SHT_TILE(2, 1);
  SHT_TILE(2, 2);
  if constexpr (KIND == 0) {
    SHT_TILE(1, 3);
    SHT_TILE(1, 4);
    SHT_TILE(1, 5);
    SHT_TILE(2, 3);
    SHT_TILE(2, 4);
    SHT_TILE(2, 5);
  } else {
    SHT_TILE(4, 1);
  }
#undef SHT_TILE
  return hipErrorInvalidValue;
}

}  // namespace

extern "C" void sht_sample_tile(int kind, int ldc, int npts, int parts, int* pt, int* ct) {
  const SampleTile t = sample_tile(kind, ldc, npts, parts);
  *pt = t.pt;
  *ct = t.ct;
}

extern "C" hipError_t sht_launch_sample(const sht::SampleArgs* a, hipStream_t s) {
  if (a->npts <= 0 || a->ldc <= 0) return hipSuccess;
  const int R = a->cuts.parts;
  if (a->ldc % 8 || R < 1 || R > sht::kSampleMaxParts || (R > 1 && !a->partial))
    return hipErrorInvalidValue;
  hipError_t le = hipErrorInvalidValue;
  if (a->kind == 0) le = a->f32 ? launch_sample_kind<0, true>(*a, s) : launch_sample_kind<0, false>(*a, s);
  else if (a->kind == 1) le = a->f32 ? launch_sample_kind<1, true>(*a, s) : launch_sample_kind<1, false>(*a, s);
  else le = a->f32 ? launch_sample_kind<2, true>(*a, s) : launch_sample_kind<2, false>(*a, s);
  if (le != hipSuccess) return le;
  hipError_t e = hipGetLastError();
  if (e != hipSuccess || R == 1) return e;
  const int stride = a->kind == 2 ? 2 : 1;
  long long blocks = ((long long)(a->ldc / stride) * a->npts + 255) / 256;
  if (blocks > 65536) blocks = 65536;
#define SHT_REDUCE(KIND)                                                                       \
  hipLaunchKernelGGL(sht::sample_reduce_kernel<KIND>, dim3((unsigned)blocks), dim3(256), 0, s,  \
                     a->partial, R, a->ldc, a->npts, a->nout, a->radius, a->cos_lat, a->out0, \
                     a->out1)
  if (a->kind == 0) SHT_REDUCE(0);
  else if (a->kind == 1) SHT_REDUCE(1);
  else SHT_REDUCE(2);
#undef SHT_REDUCE
  return hipGetLastError();
}
