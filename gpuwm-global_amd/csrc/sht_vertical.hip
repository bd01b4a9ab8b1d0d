// The semi-implicit vertical-mode operators on spectral columns (reference
// semi_implicit.py: VerticalModeSemiImplicit.linear_tendencies :796-813,
// half_apply :845-878, apply :887-919 and solve_shifted :921-959, with
// _finish :815-843).
//
// Every (n, m) column couples the L divergence levels and the L+1
// thermodynamic rows x = [theta, ln ps] through the constant vertical
// matrices B (L x L+1), C (L+1 x L), M (L x L) and per-degree matrices:
//   mode 0 (solve_shifted, apply): forcing = D + k2_n (s_bx B x + s_md M D);
//           d = H_n forcing; x' = x + s_c C (s_cd D + s_cn d)
//   mode 1 (linear_tendencies):    d = s_bx k2_n B x; x' = s_c C D
//   mode 2 (half_apply):           d = P_D D + Q_D (k2_n B x);
//                                  x' = P_x x + Q_x (C D)
// In modes 0 and 2 degree zero passes through (d(0,0) = D(0,0), x'(0,0) =
// x(0,0)), and every output is projected (zero above the triangle, m = 0
// real).  solve_shifted is s_bx = s_c = tau w, s_md = s_cd = 0, s_cn = 1;
// apply is s_bx = s_c = dt, s_md = -alpha (1 - alpha) dt^2, s_cd = 1 - alpha,
// s_cn = alpha.
//
// Each product is a small GEMM (levels x levels against levels x orders of
// one degree) on v_mfma_f32_16x16x4_f32, and a whole column operator is a
// chain of them that never leaves the registers of one wavefront:
//   * a wavefront holds 16 orders of one degree, every level, as two column
//     tiles (real and imaginary parts);
//   * lane l = (g = l / 16, q = l % 16) holds, of order q, at register r of
//     tile t the place 16 t + 4 g + r.  That is the MFMA's accumulator layout
//     (row 4 g + r of a 16-row tile, column q), and with the k index of step
//     (t, r) taken as that place it is its B operand layout too, so a
//     product's result is the next product's operand as it stands;
//   * the A operand of the four steps of one k tile is then four consecutive
//     matrix values of one row, a 16-byte LDS read;
//   * place 16 t + 4 g + r holds level 16 t + 4 r + g, so that the steps of
//     the last tile past the last level are whole steps, and are left out;
//   * a level of 16 orders is 128 contiguous bytes in memory.
// The matrices sit in LDS, zero padded to whole tiles.
//
// Bound: the phases of a wavefront in turn, its loads, its MFMAs (their time
// at full rate is a third of the call at 40 levels) and its stores; with every
// MFMA taken out the solve is 32 us, near the HBM time of its planes.
// Measured at T383 (former form, matrix rows against register columns by fma
// -> here; us a call, events around many; by card): 40 levels solve 79 ->
// 47-50, apply 100 -> 56-60, tendencies 47 -> 37-39, half map 215 -> 76-80; 64
// levels here 116, 139, 85 and 200.  A wavefront of 8 orders (real and
// imaginary parts in one tile, six wavefronts per SIMD instead of four) takes
// 66 and 101 us for solve and half map: its loads and stores are 64-byte
// pieces.
#include <algorithm>

#include "sht_kernels.h"

namespace sht {

typedef __attribute__((ext_vector_type(4))) float v4f;

// One column set: tile t, part c (0 real, 1 imaginary), register r.
template <int NT>
struct Cols {
  v4f v[NT][2];
};

template <int NT>
__device__ __forceinline__ Cols<NT> col_zero() {
  Cols<NT> o;
#pragma unroll
  for (int t = 0; t < NT; ++t) o.v[t][0] = o.v[t][1] = v4f{0.f, 0.f, 0.f, 0.f};
  return o;
}

// out + A b over `rtiles` row tiles and the first `len` levels of b; A in LDS,
// row stride LD floats.
template <int NT, int LD>
__device__ __forceinline__ Cols<NT> col_product(const float* A, const Cols<NT>& b, int rtiles,
                                                int len, int lane, Cols<NT> out) {
  const float* mine = A + (lane & 15) * LD + 4 * (lane >> 4);
#pragma unroll
  for (int kt = 0; kt < NT; ++kt) {
    if (16 * kt >= len) break;  // uniform
    v4f a[NT];
#pragma unroll
    for (int rt = 0; rt < NT; ++rt) a[rt] = *reinterpret_cast<const v4f*>(mine + 16 * rt * LD + 16 * kt);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      if (kt + 1 >= NT - 1 && 16 * kt + 4 * r >= len) break;  // uniform: past the last level
#pragma unroll
      for (int rt = 0; rt < NT; ++rt) {
        if (rt + 1 == NT && rt >= rtiles) continue;  // only the last tile can be past the rows
#pragma unroll
        for (int c = 0; c < 2; ++c)
          out.v[rt][c] =
              __builtin_amdgcn_mfma_f32_16x16x4f32(a[rt][r], b.v[kt][c][r], out.v[rt][c], 0, 0, 0);
      }
    }
  }
  return out;
}

// x + s y, elementwise.
template <int NT>
__device__ __forceinline__ Cols<NT> col_axpy(const Cols<NT>& x, float s, const Cols<NT>& y) {
  Cols<NT> o;
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int c = 0; c < 2; ++c)
#pragma unroll
      for (int r = 0; r < 4; ++r) o.v[t][c][r] = fmaf(s, y.v[t][c][r], x.v[t][c][r]);
  return o;
}
template <int NT>
__device__ __forceinline__ Cols<NT> col_scale(float s, const Cols<NT>& x) {
  Cols<NT> o;
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int c = 0; c < 2; ++c) o.v[t][c] = x.v[t][c] * s;
  return o;
}

// x with the places of levels `len` and up zero.  The matrices' padding is
// zero, but times an infinite value of the operand it leaves NaN in a
// product's padding, which the next product would spread over the column
// unless `len` fills its steps of four.
template <int NT>
__device__ __forceinline__ Cols<NT> col_trim(Cols<NT> x, int len, int g) {
  if (len % 4 == 0) return x;  // uniform
#pragma unroll
  for (int r = 0; r < 4; ++r)  // only the last tile has any
#pragma unroll
    for (int c = 0; c < 2; ++c)
      x.v[NT - 1][c][r] = 16 * (NT - 1) + 4 * r + g < len ? x.v[NT - 1][c][r] : 0.f;
  return x;
}

// The level at row or column place p of a staged matrix: place 16 t + 4 g + r
// holds level 16 t + 4 r + g.
__device__ __forceinline__ int level_at(int p) {
  return (p & ~15) + 4 * (p & 3) + ((p >> 2) & 3);
}
constexpr int vertical_ld(int nt) { return 16 * nt + 4; }  // 16-byte rows, spread over the banks
template <int NT>
constexpr int vertical_slot() { return 16 * NT * vertical_ld(NT); }  // floats of one matrix

// NT = ceil((L + 1) / 16) tiles.  A block is one degree and 16 orders per
// wavefront; the orders of one degree (which share its matrices) are
// neighbours in launch order.  Two blocks per CU (128 VGPRs) where the mode
// fits them: the tendencies also at four tiles, at the price of 8 spilled
// registers (50 levels, 139 against 128 VGPRs: T255 35.2 -> 31.0 us, T383
// 59.4 -> 52.0).
template <int NT, int MODE>
__global__ void __launch_bounds__(512, NT <= 3 || (NT == 4 && MODE == 1) ? 4 : 2) vertical_kernel(VerticalArgs a) {
  constexpr int LD = vertical_ld(NT), SLOT = vertical_slot<NT>();
  extern __shared__ float smem[];
  const int L = a.nlev, L1 = a.nlev + 1, T1 = a.T + 1;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, nw = blockDim.x >> 6;
  const int per = (T1 + 16 * nw - 1) / (16 * nw);  // blocks per degree
  // the longest degrees first; a degree's blocks start at another place each
  // time, since launch position j runs on XCD j % 8: with `per` and 8 not
  // coprime, some XCDs would get the blocks above the triangle throughout
  const int n = a.T - (int)blockIdx.x / per;
  const int first = ((int)blockIdx.x % per + n) % per * nw * 16;  // the block's first order
  const int m0 = first + 16 * w;
  const int g = lane >> 4, m = m0 + (lane & 15);
  const bool live = m < T1, in_tri = live && m <= n;
  const size_t plane = (size_t)T1 * T1;
  const size_t at = (size_t)n * T1 + m, at_in = (size_t)n * T1 + min(m, n);

  // ---- the columns: off-triangle orders and levels past the end are zero ----
  auto load_levels = [&](const float2* f) {
    Cols<NT> o;
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int lev = 16 * t + 4 * r + g;
        const float2 x = f[(size_t)min(lev, L - 1) * plane + at_in];
        const bool ok = in_tri && lev < L;
        o.v[t][0][r] = ok ? x.x : 0.f;
        o.v[t][1][r] = ok ? x.y : 0.f;
      }
    return o;
  };
  auto store_level = [&](float2* f, int lev, float re, float im) {
    if (live && lev < L)
      f[(size_t)lev * plane + at] = make_float2(in_tri ? re : 0.f, in_tri && m > 0 ? im : 0.f);
  };
  auto store_levels = [&](float2* f, const Cols<NT>& o) {
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) store_level(f, 16 * t + 4 * r + g, o.v[t][0][r], o.v[t][1][r]);
  };
  // row L of a thermodynamic column is ln ps: lane group L % 4,
  // register (L / 4) % 4 of tile L / 16
  auto store_x = [&](const Cols<NT>& o) {
    store_levels(a.theta_out, o);
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (live && 16 * t + 4 * r + g == L)
          a.lnps_out[at] = make_float2(in_tri ? o.v[t][0][r] : 0.f,
                                       in_tri && m > 0 ? o.v[t][1][r] : 0.f);
  };

  if (first > n) {  // block-uniform: no order in the triangle
    const Cols<NT> z = col_zero<NT>();
    store_levels(a.d_out, z);
    store_x(z);
    return;
  }

  Cols<NT> x = load_levels(a.theta);
  Cols<NT> D = load_levels(a.div);
  {
    const float2 ps = a.lnps[at_in];
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (in_tri && 16 * t + 4 * r + g == L) {
          x.v[t][0][r] = ps.x;
          x.v[t][1][r] = ps.y;
        }
  }

  // ---- the matrices: slots B, C, then [M,] H_n or P_D, Q_D, P_x, Q_x ----
  // (a wavefront takes whole rows, four rows' loads in flight)
  auto stage = [&](int slot, const float* src, int rows, int len) {
    float* dst = smem + (size_t)slot * SLOT;
    for (int r0 = w; r0 < 16 * NT; r0 += 4 * nw)
#pragma unroll
      for (int c0 = 0; c0 < LD; c0 += 64) {
        const int c = c0 + lane, jc = level_at(c);
        float v[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const int jr = level_at(r0 + u * nw);
          const bool ok = jr < rows && jc < len && c < 16 * NT;
          v[u] = src[ok ? jr * len + jc : 0];
          v[u] = ok ? v[u] : 0.f;
        }
#pragma unroll
        for (int u = 0; u < 4; ++u)
          if (r0 + u * nw < 16 * NT && c < LD) dst[(r0 + u * nw) * LD + c] = v[u];
      }
  };
  stage(0, a.b_matrix, L, L1);
  stage(1, a.c_matrix, L1, L);
  const bool with_m = MODE == 0 && a.m_matrix != nullptr;
  if constexpr (MODE == 0) {
    stage(2, a.inverse + (size_t)n * L * L, L, L);
    if (with_m) stage(3, a.m_matrix, L, L);
  } else if constexpr (MODE == 2) {
    const size_t dn = (size_t)n * L * L, xn = (size_t)n * L1 * L1;
    stage(2, a.p_d + dn, L, L);
    stage(3, a.q_d + dn, L, L);
    stage(4, a.p_x + xn, L1, L1);
    stage(5, a.q_x + xn, L1, L1);
  }
  const float k2 = a.k2[n];
  __syncthreads();
  if (m0 > n) {  // wave-uniform: nothing of the triangle (no barrier below)
    store_levels(a.d_out, col_zero<NT>());
    store_x(col_zero<NT>());
    return;
  }

  const int tl = (L + 15) / 16;  // tiles of L levels; NT of L + 1 rows
  auto mul_add = [&](int slot, const Cols<NT>& b, int rtiles, int len, const Cols<NT>& to) {
    return col_product<NT, LD>(smem + (size_t)slot * SLOT, b, rtiles, len, lane, to);
  };
  auto mul = [&](int slot, const Cols<NT>& b, int rtiles, int len) {
    return mul_add(slot, b, rtiles, len, col_zero<NT>());
  };
  const bool pin = n == 0 && m == 0 && MODE != 1;
  auto pinned = [&](const Cols<NT>& o, const Cols<NT>& as) {
    Cols<NT> p;
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int c = 0; c < 2; ++c) p.v[t][c] = pin ? as.v[t][c] : o.v[t][c];
    return p;
  };
  const Cols<NT> bx = mul(0, x, tl, L1);
  if constexpr (MODE == 1) {
    store_levels(a.d_out, col_scale(a.s_bx * k2, bx));
    store_x(col_scale(a.s_c, mul(1, D, NT, L)));
  } else if constexpr (MODE == 0) {
    Cols<NT> f = col_axpy(D, k2 * a.s_bx, bx);
    if (with_m) f = col_axpy(f, k2 * a.s_md, mul(3, D, tl, L));
    const Cols<NT> d = col_trim(mul(2, col_trim(f, L, g), tl, L), L, g);
    store_levels(a.d_out, pinned(d, D));
    const Cols<NT> u = col_axpy(col_scale(a.s_cd, D), a.s_cn, d);
    store_x(pinned(col_axpy(x, a.s_c, mul(1, u, NT, L)), x));
  } else {
    store_levels(a.d_out,
                 pinned(mul_add(3, col_trim(col_scale(k2, bx), L, g), tl, L,
                                     mul(2, D, tl, L)), D));
    // P_x x and Q_x (C D) apart, added once.  Carried on in P_x x's
    // accumulators, each of the small product's terms is rounded at its size:
    // 1.6 times the error of theta and ln ps.  The divergence's two products
    // are of a size, and one accumulation is as exact as two.
    const Cols<NT> qx = mul(5, col_trim(mul(1, D, NT, L), L1, g), NT, L1);
    store_x(pinned(col_axpy(mul(4, x, NT, L1), 1.f, qx), x));
  }
}

}  // namespace sht

namespace {

template <int NT, int MODE>
hipError_t launch_vertical(const sht::VerticalArgs& a, hipStream_t s) {
  const int slots = MODE == 0 ? (a.m_matrix ? 4 : 3) : MODE == 1 ? 2 : 6;
  const size_t lds = (size_t)slots * sht::vertical_slot<NT>() * sizeof(float);
  const int T1 = a.T + 1;
  // Wavefronts (16 orders each) per block: eight, which share one copy of the
  // matrices, or as many as the degree has orders for.  At T383, 40 levels:
  // four take 52 (solve) and 90 us (half map), eight 52 and 82 on the same
  // card; five or six spread unevenly over a CU's four SIMDs (62-73 us).  From 32 levels on, also eight where a degree has fewer
  // orders (T <= 63): the others only stage, most of the time of such a launch
  // (half map, T31: 40 levels 24.3 -> 19.0 us a call, 64 levels 53.9 -> 32.5).
  const int waves = T1 <= 64 && NT >= 3 ? 8 : std::min(8, (T1 + 15) / 16);
  const int per = (T1 + 16 * waves - 1) / (16 * waves);
  const void* k = reinterpret_cast<const void*>(sht::vertical_kernel<NT, MODE>);
  hipError_t e = hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  if (e != hipSuccess) return e;
  sht::VerticalArgs copy = a;
  void* args[] = {&copy};
  return hipLaunchKernel(k, dim3((unsigned)(T1 * per)), dim3(64 * waves), args, lds, s);
}

template <int NT>
hipError_t launch_tiles(const sht::VerticalArgs& a, hipStream_t s) {
  return a.mode == 0   ? launch_vertical<NT, 0>(a, s)
         : a.mode == 1 ? launch_vertical<NT, 1>(a, s)
                       : launch_vertical<NT, 2>(a, s);
}

}  // namespace

extern "C" hipError_t sht_launch_vertical_solve(const sht::VerticalArgs* a, hipStream_t s) {
  if (a->nlev < 1 || a->nlev > sht::kMaxLevels || a->mode < 0 || a->mode > 2)
    return hipErrorInvalidValue;
  switch ((a->nlev + 16) / 16) {  // ceil((nlev + 1) / 16)
    case 1: return launch_tiles<1>(*a, s);
    case 2: return launch_tiles<2>(*a, s);
    case 3: return launch_tiles<3>(*a, s);
    case 4: return launch_tiles<4>(*a, s);
    default: return launch_tiles<5>(*a, s);
  }
}
