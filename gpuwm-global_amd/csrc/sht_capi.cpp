// C ABI of the spherical-harmonic transform engine (include/arwen_sht.h).
//
// A plan owns one truncation's device state: Gauss nodes and weights, the
// three Legendre tables in both GEMM layouts, the FFT twiddles and the
// per-row scale vectors.  A batch owns the workspaces, the grouped-GEMM work
// list of its jobs and, once captured, a hipGraph of its launches.
#include "arwen_sht.h"

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstring>
#include <list>
#include <memory>
#include <mutex>
#include <queue>
#include <string>
#include <tuple>
#include <vector>

#include "sht_kernels.h"
#include "sht_static.h"

namespace {

thread_local std::string g_error;

struct Failure {
  int code;
};

[[noreturn]] void fail(int code, const std::string& msg) {
  g_error = msg;
  throw Failure{code};
}

void hip_check(hipError_t e, const char* what) {
  if (e != hipSuccess) {
    fail(e == hipErrorOutOfMemory ? ARWEN_SHT_ENOMEM : ARWEN_SHT_EHIP,
         std::string(what) + ": " + hipGetErrorString(e));
  }
}

template <class F>
int guarded(F&& f) {
  try {
    f();
    return ARWEN_SHT_OK;
  } catch (const Failure& x) {
    return x.code;
  } catch (const std::bad_alloc&) {
    g_error = "host allocation failed";
    return ARWEN_SHT_ENOMEM;
  } catch (...) {
    g_error = "unexpected C++ exception";
    return ARWEN_SHT_EHIP;
  }
}

// Set-up work of a single operation's first call goes to the caller's stream
// (zero fills and uploads ordered before its kernels, no device-wide wait);
// null elsewhere.  The host copies of what is uploaded there live in
// g_setup_keep until the owner takes them.
thread_local hipStream_t g_setup_stream = nullptr;
thread_local std::vector<std::vector<char>>* g_setup_keep = nullptr;

// Owning device buffer.
struct DevBuf {
  void* p = nullptr;
  size_t bytes = 0;
  DevBuf() = default;
  explicit DevBuf(size_t n, bool zero = true) { alloc(n, zero); }
  void alloc(size_t n, bool zero = true) {
    release();
    bytes = n;
    if (n == 0) return;
    hip_check(hipMalloc(&p, n), "hipMalloc");
    if (zero) {
      if (g_setup_stream)
        hip_check(hipMemsetAsync(p, 0, n, g_setup_stream), "hipMemsetAsync");
      else
        hip_check(hipMemset(p, 0, n), "hipMemset");
    }
  }
  void release() {
    if (p) (void)hipFree(p);
    p = nullptr;
    bytes = 0;
  }
  void swap(DevBuf& o) {
    std::swap(p, o.p);
    std::swap(bytes, o.bytes);
  }
  ~DevBuf() { release(); }
  DevBuf(const DevBuf&) = delete;
  DevBuf& operator=(const DevBuf&) = delete;
  template <class T>
  T* as() const {
    return static_cast<T*>(p);
  }
};

template <class T>
void upload(DevBuf& buf, const std::vector<T>& host) {
  buf.alloc(host.size() * sizeof(T), false);
  if (host.empty()) return;
  const size_t n = host.size() * sizeof(T);
  if (g_setup_stream && g_setup_keep) {
    // the copy may still be pending when this returns: copy from a kept buffer
    g_setup_keep->emplace_back(reinterpret_cast<const char*>(host.data()),
                               reinterpret_cast<const char*>(host.data()) + n);
    hip_check(hipMemcpyAsync(buf.p, g_setup_keep->back().data(), n, hipMemcpyHostToDevice,
                             g_setup_stream),
              "hipMemcpyAsync H2D");
  } else {
    hip_check(hipMemcpy(buf.p, host.data(), n, hipMemcpyHostToDevice), "hipMemcpy H2D");
  }
}

// Passes of the row FFT kernels for scalar fields: primes above 13 first,
// largest first (the first pass of such a radix shares its sums between outputs
// and has no twiddles), then the radices 2..16 of least modelled cost.  A pass costs its
// LDS round trip (~100 wave instructions) plus, per round of 64 butterflies,
// ~20 R for addresses, twiddles and LDS accesses and its DFT (direct for 5,
// 7, 11, 13, ~5 R log2 R otherwise); with N = 1152 this takes 12 x 12 x 8
// over 4 x 4 x 4 x 2 x 3 x 3.
// Rounding: fewer passes round less, direct sums of 5..13 a little more.  In a
// float32 emulation over 345 row lengths the FFT's rms error is 0.92 of the
// passes 4, 2, 3 and direct sums' at the median and 1.08 at most (above 1.0 at
// 21 lengths; no other order of the same radices does better).  On the device,
// whole transforms: inverse 0.98 at the median, 1.02 at most; forward 0.97 and
// 1.08.
double pass_cost(int n, int r) {
  const int rounds = (n / r + 63) / 64;
  double dft = 5.0 * r * std::log2((double)r);
  for (int p : {5, 7, 11, 13})
    if (r % p == 0) dft += (r / p) * 2.0 * (p - 1) * (p - 1);
  return 100.0 + rounds * (20.0 * r + dft);
}

void best_passes(int n, int rest, int largest, std::vector<int>& now, double cost,
                 std::vector<int>& best, double& least) {
  if (cost >= least) return;
  if (rest == 1) {
    best = now;
    least = cost;
    return;
  }
  for (int r = largest; r >= 2; --r) {
    if (rest % r) continue;
    now.push_back(r);
    best_passes(n, rest / r, r, now, cost + pass_cost(n, r), best, least);
    now.pop_back();
  }
}

std::vector<int> factor_radices(int n) {
  std::vector<int> r;
  int rest = n;
  for (int p = 2; p <= rest; ++p)
    while (rest % p == 0) {
      if (p > 13) r.insert(r.begin(), p);
      rest /= p;
    }
  int smooth = n;
  for (int p : r) smooth /= p;
  std::vector<int> now, best;
  double least = 1e300;
  best_passes(n, smooth, 16, now, 0.0, best, least);
  r.insert(r.end(), best.begin(), best.end());
  return r;
}

// Passes for the vector operators' rows: fours, a two, threes and the other
// primes in rising order.
std::vector<int> plain_radices(int n) {
  std::vector<int> r;
  while (n % 4 == 0) { r.push_back(4); n /= 4; }
  for (int p = 2; n > 1; ++p)
    while (n % p == 0) { r.push_back(p); n /= p; }
  return r;
}

}  // namespace

enum TableKind { kP = 0, kD = 1, kPm = 2 };

struct arwen_sht_batch;

struct arwen_sht_plan {
  int device = 0;
  int T = 0, nlat = 0, nlon = 0, JH = 0, JHP = 0, MB = 0;
  double radius = 0;
  int precision = 0;
  std::vector<int> koff;  // 2(T+1)+1 entries
  long long tab_elems = 0;
  int ldp = 0;            // packed floats per column
  int ldw = 0;            // waist floats per column
  std::vector<double> mu, w;
  DevBuf d_mu, d_w, d_koff, d_tw;
  DevBuf tab_syn[3], tab_ana[3];
  DevBuf scale_fold, scale_fold_vec, scale_fold_vec_cos, scale_one, scale_inv_a, scale_inv_acos;
  DevBuf scale_waist, scale_waist_vec;  // 2 pi w (x 1/a): folds of a reference waist (already / nlon)
  DevBuf sample_rec, sample_diag;       // point sampler recurrence tables, built on first use
  // vector operators' FP64 low orders m < m0: FP64 twiddles, per-row FP64
  // scales and the FP64 tables of those orders (kinds dP/dphi and P m / cos)
  int m0 = 0;
  DevBuf d_tw64;
  // FP64 row scales of the recurrence form (every order of u and v):
  // fold 2 pi w / (a nlon cos(phi)), unfold 1 / (a cos(phi))
  DevBuf scale_fold_vec64_cos, scale_inv_acos64;
  DevBuf low_syn[3], low_ana[3];
  sht::FftPlan fft{};
  // single-operation batches by (op, count, stream), most recent first
  std::list<std::pair<std::tuple<int, int, void*>, arwen_sht_batch*>> cache;
  std::mutex cache_mu;
  ~arwen_sht_plan();

  int kp(int m, int p) const { return koff[2 * m + p + 1] - koff[2 * m + p]; }
  size_t table_bytes() const {
    size_t per = precision == ARWEN_SHT_FP32 ? 4 : 6;
    size_t low = 0;
    for (int k = 0; k < 3; ++k) low += low_syn[k].bytes + low_ana[k].bytes;
    return 6 * (size_t)tab_elems * per + low;
  }
  const void* table(int kind, bool syn, long long* piece) const {
    *piece = tab_elems;
    return syn ? tab_syn[kind].p : tab_ana[kind].p;
  }
};

namespace {

void build_sample_tables(arwen_sht_plan* P);

void build_plan(arwen_sht_plan* P, const arwen_sht_plan_desc* d) {
  if (!d) fail(ARWEN_SHT_EINVAL, "plan descriptor is NULL");
  const int T = d->truncation;
  if (T < 1) fail(ARWEN_SHT_EINVAL, "truncation must be >= 1, got " + std::to_string(T));
  if (d->nlat < T + 1)
    fail(ARWEN_SHT_EINVAL, "nlat=" + std::to_string(d->nlat) + " is too small for T" +
                               std::to_string(T) + "; need at least " + std::to_string(T + 1));
  if (d->nlon % 2 || d->nlon < 2 * T + 2)
    fail(ARWEN_SHT_EINVAL, "nlon must be even and >= 2T+2, got " + std::to_string(d->nlon));
  if (!(d->radius_m > 0) || !std::isfinite(d->radius_m))
    fail(ARWEN_SHT_EINVAL, "radius_m must be finite and positive");
  if (d->precision != ARWEN_SHT_FP32 && d->precision != ARWEN_SHT_BF16X3 &&
      d->precision != ARWEN_SHT_BF16X6)
    fail(ARWEN_SHT_EINVAL, "precision must be ARWEN_SHT_FP32, _BF16X3 or _BF16X6");
  if ((d->sin_lat == nullptr) != (d->weights == nullptr))
    fail(ARWEN_SHT_EINVAL, "sin_lat and weights must be given together");
  hip_check(hipGetDevice(&P->device), "hipGetDevice");
  P->T = T;
  P->nlat = d->nlat;
  P->nlon = d->nlon;
  P->radius = d->radius_m;
  P->precision = d->precision;
  P->JH = (d->nlat + 1) / 2;
  P->JHP = SHT_ROUND_UP(P->JH, sht::kPad);
  P->MB = (T + 1 + sht::kMT - 1) / sht::kMT;
  // blocks hold degrees m..T+1: the vector operators' recurrence form
  // contracts the basis one degree past the truncation (the other operations
  // leave that row zero in their data and ignore it in their results)
  P->koff.assign(2 * (T + 1) + 1, 0);
  for (int m = 0; m <= T; ++m)
    for (int p = 0; p < 2; ++p)
      P->koff[2 * m + p + 1] = P->koff[2 * m + p] + sht::k_padded(T + 1, m, p);
  P->ldp = P->koff.back();
  P->tab_elems = (long long)P->ldp * P->JHP;
  P->ldw = P->MB * 2 * P->JHP * sht::kMT;

  // Nodes and weights.
  P->mu.resize(P->nlat);
  P->w.resize(P->nlat);
  P->d_mu.alloc(P->nlat * sizeof(double), false);
  P->d_w.alloc(P->nlat * sizeof(double), false);
  if (d->sin_lat) {
    for (int j = 0; j < P->nlat; ++j) {
      P->mu[j] = d->sin_lat[j];
      P->w[j] = d->weights[j];
    }
    for (int j = 0; j < P->nlat; ++j)
      if (P->mu[j] != -P->mu[P->nlat - 1 - j])
        fail(ARWEN_SHT_EINVAL, "sin_lat must be ascending and symmetric about the equator");
    hip_check(hipMemcpy(P->d_mu.p, P->mu.data(), P->nlat * 8, hipMemcpyHostToDevice), "copy mu");
    hip_check(hipMemcpy(P->d_w.p, P->w.data(), P->nlat * 8, hipMemcpyHostToDevice), "copy w");
  } else {
    hip_check(sht_launch_gauss_newton(P->nlat, P->d_mu.as<double>(), P->d_w.as<double>(), 0),
              "gauss_newton launch");
    hip_check(hipMemcpy(P->mu.data(), P->d_mu.p, P->nlat * 8, hipMemcpyDeviceToHost), "read mu");
    hip_check(hipMemcpy(P->w.data(), P->d_w.p, P->nlat * 8, hipMemcpyDeviceToHost), "read w");
  }
  upload(P->d_koff, P->koff);

  // FP64 vector orders (resolved below once the FFT path is known).
  if (d->fp64_orders < -1)
    fail(ARWEN_SHT_EINVAL, "fp64_orders must be -1 (default), 0 or positive, got " +
                               std::to_string(d->fp64_orders));
  {
    const int L = sht_fft_wave_L(P->nlon);
    const bool wave = L && sht_fold64_lds_bytes(P->nlon) <= 160 * 1024;
    int m0 = d->fp64_orders;
    if (m0 < 0) m0 = P->precision == ARWEN_SHT_FP32 ? 0 : sht::kMT * ((T + 1 + 191) / 192);
    m0 = SHT_ROUND_UP(m0, sht::kMT);
    P->m0 = wave ? std::min(m0, P->MB * sht::kMT) : 0;
  }

  // Legendre tables.
  sht::TableOut out{};
  out.elems = P->tab_elems;
  const bool fp32 = P->precision == ARWEN_SHT_FP32;
  for (int k = 0; k < 3; ++k) {
    size_t bytes = (size_t)P->tab_elems * (fp32 ? 4 : 6);
    P->tab_syn[k].alloc(bytes, true);
    P->tab_ana[k].alloc(bytes, true);
    if (fp32) {
      out.f32_syn[k] = P->tab_syn[k].as<float>();
      out.f32_ana[k] = P->tab_ana[k].as<float>();
    } else {
      out.bf_syn[k] = P->tab_syn[k].as<unsigned short>();
      out.bf_ana[k] = P->tab_ana[k].as<unsigned short>();
    }
  }
  if (P->m0 > 0) {
    // the basis over degrees m..T+1 in both layouts (the recurrence form in FP64)
    const size_t low_bytes = (size_t)P->m0 * (T + 2) * P->JHP * sizeof(double);
    P->low_syn[kP].alloc(low_bytes, true);
    P->low_ana[kP].alloc(low_bytes, true);
    out.f64_low_syn[kP] = P->low_syn[kP].as<double>();
    out.f64_low_ana[kP] = P->low_ana[kP].as<double>();
    out.low_m0 = P->m0;
  }
  hip_check(sht_launch_legendre_tables(T, P->nlat, P->JH, P->JHP, P->d_mu.as<double>(),
                                       P->d_koff.as<int>(), &out, 0),
            "legendre_tables launch");

  // FFT plan.
  P->fft.N = P->nlon;
  for (auto* passes : {&P->fft.scalar, &P->fft.vector}) {
    const bool direct = passes == &P->fft.vector;
    const std::vector<int> rad = direct ? plain_radices(P->nlon) : factor_radices(P->nlon);
    if ((int)rad.size() > sht::kMaxStages) fail(ARWEN_SHT_EINVAL, "nlon has too many factors");
    passes->n = (int)rad.size();
    passes->direct = direct;
    for (size_t s = 0; s < rad.size(); ++s) passes->radix[s] = rad[s];
  }
  std::vector<float2> tw(P->nlon);
  for (int k = 0; k < P->nlon; ++k) {
    double ang = -2.0 * M_PI * (double)k / (double)P->nlon;
    tw[k] = make_float2((float)std::cos(ang), (float)std::sin(ang));
  }
  upload(P->d_tw, tw);
  P->fft.tw = P->d_tw.as<float2>();
  if (P->m0 > 0) {
    std::vector<double2> tw64(P->nlon);
    for (int k = 0; k < P->nlon; ++k) {
      const double ang = -2.0 * M_PI * (double)k / (double)P->nlon;
      tw64[k] = make_double2(std::cos(ang), std::sin(ang));
    }
    upload(P->d_tw64, tw64);
    P->fft.tw64 = P->d_tw64.as<double2>();
  }
  {
    int lds_max = 65536;
    (void)hipDeviceGetAttribute(&lds_max, hipDeviceAttributeMaxSharedMemoryPerBlock, P->device);
    // the longest row a plan takes: 32 bytes of LDS per longitude
    if ((size_t)P->nlon * 4 * sizeof(float2) > (size_t)lds_max)
      fail(ARWEN_SHT_EINVAL, "nlon=" + std::to_string(P->nlon) + " needs more LDS than the device has");
    hip_check(sht_fft_allow_lds((size_t)lds_max), "FFT LDS attribute");
    if (P->m0 > 0) hip_check(sht_low_allow_lds((size_t)lds_max), "low-order LDS attribute");
    // wave-resident FFTs (N = 64 L) when their LDS fits the device
    const int L = sht_fft_wave_L(P->nlon);
    P->fft.wave_L = (L && sht_fft_wave_lds_bytes(P->nlon, 1) <= (size_t)lds_max) ? L : 0;
  }

  // Per folded-row scales.
  std::vector<float> sf(P->JHP, 0.f), sfv(P->JHP, 0.f), one(P->JHP, 1.f), inva(P->JHP, 0.f);
  std::vector<float> invacos(P->JHP, 0.f), sfvc(P->JHP, 0.f);
  std::vector<float> sw(P->JHP, 0.f), swv(P->JHP, 0.f);
  for (int i = 0; i < P->JH; ++i) {
    const int jn = P->nlat - 1 - i;
    double wq = P->w[jn];
    if (jn == i) wq *= 0.5;  // the equator row is its own mirror
    sf[i] = (float)(2.0 * M_PI * wq / P->nlon);
    sfv[i] = (float)(2.0 * M_PI * wq / (P->radius * P->nlon));
    sw[i] = (float)(2.0 * M_PI * wq);
    swv[i] = (float)(2.0 * M_PI * wq / P->radius);
    inva[i] = (float)(1.0 / P->radius);
    const double mu = P->mu[jn];
    invacos[i] = (float)(1.0 / (P->radius * std::sqrt(std::max(0.0, 1.0 - mu * mu))));
    sfvc[i] = (float)(2.0 * M_PI * wq / (P->radius * P->nlon) /
                      std::sqrt(std::max(0.0, 1.0 - mu * mu)));
  }
  upload(P->scale_fold, sf);
  upload(P->scale_fold_vec, sfv);
  upload(P->scale_fold_vec_cos, sfvc);
  upload(P->scale_waist, sw);
  upload(P->scale_waist_vec, swv);
  upload(P->scale_one, one);
  upload(P->scale_inv_a, inva);
  upload(P->scale_inv_acos, invacos);
  if (P->m0 > 0) {

    std::vector<double> sfvc64(P->JHP, 0.0), invac64(P->JHP, 0.0);
    for (int i = 0; i < P->JH; ++i) {
      const int jn = P->nlat - 1 - i;
      double wq = P->w[jn];
      if (jn == i) wq *= 0.5;
      const double mu = P->mu[jn];
      const double cosl = std::sqrt(std::max(0.0, 1.0 - mu * mu));
      sfvc64[i] = 2.0 * M_PI * wq / (P->radius * P->nlon) / cosl;
      invac64[i] = 1.0 / (P->radius * cosl);
    }
    upload(P->scale_fold_vec64_cos, sfvc64);
    upload(P->scale_inv_acos64, invac64);
  }
  // the point sampler's recurrence coefficients, so that sampling allocates nothing
  build_sample_tables(P);
  // this device's copy of arwen_sht_sample_static's array, resolved once
  hip_check(sht_static_setup(P->device), "static sampler workspace");
  hip_check(hipDeviceSynchronize(), "plan build");
}

}  // namespace

// ---------------------------------------------------------------------------
// Batches
// ---------------------------------------------------------------------------

// One work group of the grouped GEMM before it is cut into panels: up to kMT
// consecutive orders of one job and one output parity, with one or two
// segments (table kind, data) accumulated into the same output.
struct HostGroup {
  int nseg = 0, N = 0, mcount = 0;
  const char* A[2][sht::kMT] = {};  // table block of (seg, order), tiled layout
  int K[2][sht::kMT] = {};          // k extent: SYN degrees KP(m, p); ANA JHP
  int Arows[2][sht::kMT] = {};      // rows of the table block: SYN JHP; ANA KP(m, q)
  const char* B[2][sht::kMT] = {};  // SYN packed block of (seg, order); ANA waist block of seg
  float* C[sht::kMT] = {};          // SYN C[0] = waist block; ANA packed block of the order
  int R[sht::kMT] = {};             // output rows per order (SYN JHP; ANA KP(m, q))
  int cmap[2] = {0, 0};             // B column map per segment (GemmStep::cmap)
  int bcs = 0, ccs = 0;             // column strides (floats)
  long long piece_bytes = 0;        // table piece stride (split modes)
  size_t esz = 4;                   // table element bytes (4 fp32, 2 bf16 pieces); data are fp32
};

// Device work lists of one GEMM direction, built for one column tile and grid.
struct GemmLists {
  DevBuf panels, steps, items;
  int nitems = 0, nsteps = 0;
  int bn = 0;
  int slots = 0;  // the grid asked for
  int grid = 0;   // workgroups launched (at most `slots`)
  void swap(GemmLists& o) {
    panels.swap(o.panels);
    steps.swap(o.steps);
    items.swap(o.items);
    std::swap(nitems, o.nitems);
    std::swap(nsteps, o.nsteps);
    std::swap(bn, o.bn);
    std::swap(slots, o.slots);
    std::swap(grid, o.grid);
  }
};

struct JobState {
  arwen_sht_job job;
  DevBuf packed_a;            // synthesis input (packed coefficients)
  DevBuf waist_a, waist_b;    // synthesis output (b: gradient north) / analysis input
  DevBuf packed_out;          // analysis output
  DevBuf low;                 // vector jobs: FP64 low waist [level][u|v][m < m0][p][i]
  DevBuf low_ab;              // vordiv_from_uv: FP64 A, B [level][A|B][n < T+2][m < m0]
  int ncols = 0;
};

struct arwen_sht_batch {
  int device = 0;
  int precision = 0;
  std::vector<std::vector<char>> setup_keep;  // host sources of stream-ordered uploads
  std::vector<std::unique_ptr<JobState>> jobs;
  std::vector<sht::PackArgs> packs;
  std::vector<sht::UnfoldArgs> unfolds;
  std::vector<sht::FoldArgs> folds;
  std::vector<sht::UnpackArgs> unpacks;
  std::vector<sht::WaistUnfoldArgs> waist_unfolds;  // synthesis into a reference waist
  std::vector<sht::WaistFoldArgs> waist_folds;      // analysis from a reference waist
  std::vector<sht::LowSynArgs> low_syns;            // vector jobs' FP64 low orders
  std::vector<sht::LowAnaArgs> low_anas;
  bool single = false;  // one operation of a plan's cache: may take the few-column kernels
  std::vector<std::pair<sht::SmallSynArgs, int>> small_syns;  // and the jobs of each
  std::vector<sht::SmallAnaArgs> small_anas;
  std::vector<HostGroup> groups[2];  // GEMM work groups per direction (0 SYN, 1 ANA)
  GemmLists lists[2];
  arwen_sht_gemm_config config{{32, 32}, {0, 0}, 1};
  double legendre_flops = 0, fft_bytes = 0;
  double low_flops = 0;  // the part of legendre_flops the FP64 low-order kernels do
  hipGraph_t graph = nullptr;
  hipGraphExec_t exec = nullptr;
  ~arwen_sht_batch() {
    if (exec) (void)hipGraphExecDestroy(exec);
    if (graph) (void)hipGraphDestroy(graph);
  }
};

arwen_sht_plan::~arwen_sht_plan() {
  for (auto& e : cache) delete e.second;
}

namespace {

bool is_synthesis(int op) {
  return (op >= ARWEN_SHT_OP_SYNTHESIS && op <= ARWEN_SHT_OP_UV_FROM_VORDIV) ||
         (op >= ARWEN_SHT_OP_SYNTHESIS_TO_WAIST && op <= ARWEN_SHT_OP_MERIDIONAL_TO_WAIST) ||
         op == ARWEN_SHT_OP_SYNTHESIS_GRADIENT;
}
bool to_waist(int op) {
  return op >= ARWEN_SHT_OP_SYNTHESIS_TO_WAIST && op <= ARWEN_SHT_OP_MERIDIONAL_TO_WAIST;
}
bool from_waist(int op) {
  return op == ARWEN_SHT_OP_ANALYSIS_FROM_WAIST || op == ARWEN_SHT_OP_VORDIV_FROM_WAIST ||
         op == ARWEN_SHT_OP_DIVERGENCE_FROM_WAIST;
}

constexpr int kXcds = 8;  // MI355X: 8 XCDs x 32 CUs

// Column tile of a new batch's direction: 64 columns where the launch is bound
// by table reads and has enough of the larger tiles, else 32.  A tile reads
// its table fragments through L1 once for its columns, so 64 halve that
// traffic; they cost residency (two blocks per CU, not three) and padding.
// They also come in generations of 512, which a launch of few does not fill.
// What counts of the padding is what 64-column tiles have more of than
// 32-column ones (80 columns: 128 against 96).  A call, us, 32 against 64
// columns (64-column items, padded columns over the 32-column tiles'):
//   bf16x6 synthesis  T383 60 fields (1152, 1) 114 : 103, 40 (1152, 1.33) 78.0 :
//     78.3, gradients of 40 (2304, 1.33) 184 : 174, wind 40 levels (1692, 1.2)
//     204 : 194; T287 wind 40 levels (1296, 1.2) 132 : 126; gradients of 40
//     fields (1.33), T191 on 576 longitudes (1152) 90.3 : 96.3, T255 on 768
//     (1536) 131 : 126; T255 60 fields (512, 1) 46.1 : 46.5
//   bf16x6 analysis   T383 20 fields (384, 1) 49.9 : 47.0, vorticity, divergence
//     40 levels (1128, 1.2) 205 : 195, 24 (752, 1.33) 141 : 136; T223 60 levels
//     (640, 1) 129 : 120; T255 on 768 longitudes 40 levels (558, 1.2) 142 : 145
//   fp32 synthesis    T383 gradients of 32 fields (1152, 1) 136 : 131, of 40
//     (2304, 1.33) 178 : 185; T255 gradients of 64 (1024, 1) 112 : 109; T191 on
//     576 longitudes, 20 MB of tables, wind 64 levels (1152, 1) 132 : 135
//   fp32 analysis     T383 64 fields (774, 1) 118 : 118, 128 125 : 115 (kernel)
// so: tables from half of the eight 4 MB L2s up; in the split modes, with no
// more padding about as many items as run together, with more of it more than
// two generations (synthesis) or 700 (analysis); in FP32, whose MFMA time
// weighs more, two generations (and tables of 24 MB) or four and hardly any
// padding at all.  Over 2,336 calls of T106 to T383 this is 0.1% above the
// better of the two at the mean and at most 4% above 32 columns.
int default_cols(int dir, const std::vector<HostGroup>& groups, int precision) {
  const bool split = precision != ARWEN_SHT_FP32;
  long long tiles = 0, used = 0, wide = 0, narrow = 0, table = 0;
  const int pieces = split ? (precision == ARWEN_SHT_BF16X6 ? 3 : 2) : 1;
  for (const HostGroup& g : groups) {
    int rows = 0;
    for (int z = 0; z < g.mcount; ++z) rows = std::max(rows, g.R[z]);
    const long long panels = (rows + sht::kGemmBM - 1) / sht::kGemmBM, nt = (g.N + 63) / 64;
    tiles += panels * nt;
    used += panels * g.N;
    wide += panels * nt * 64;
    narrow += panels * ((g.N + 31) / 32) * 32;
    for (int sg = 0; sg < g.nseg; ++sg)
      for (int z = 0; z < g.mcount; ++z)
        table += (long long)g.K[sg][z] * g.Arows[sg][z] * (long long)g.esz * pieces;
  }
  const bool same = 50 * wide <= 51 * narrow;  // hardly more padding than 32-column tiles
  const bool fits =
      !split     ? 10 * wide <= 11 * used &&
                       (dir == 0 ? tiles >= 1024 && table >= (24ll << 20) : tiles > 2047)
      : dir == 0 ? (same && tiles >= 512) || (4 * wide <= 5 * narrow && tiles >= 1200) ||
                       (3 * wide <= 4 * narrow && tiles >= 1300)
                 : (same && tiles >= 380) || (3 * wide <= 4 * used && tiles >= 700);
  return fits && table >= (16ll << 20) ? 64 : 32;
}

// Persistent grid of direction d; 0 in the config = the workgroups that are
// resident together (256 CUs).
int gemm_slots(const arwen_sht_gemm_config& c, int d) {
  return c.grid[d] > 0 ? c.grid[d] : 256 * sht::gemm_blocks_per_cu(c.cols[d]);
}

// Cuts the work groups of one direction into panels (group x 64-row tile),
// their k-step lists and (panel, column tile) work items, and deals the items
// to `slots` persistent workgroups.
// Workgroups are dispatched round-robin over the 8 XCDs, and the grid is a
// multiple of 8, so workgroup b runs on XCD b % 8.  Every work item of one
// group (same orders, same tables, same data columns) goes to one XCD, where
// its tiles run side by side and share that XCD's L2; groups are balanced
// over the XCDs longest first, and an XCD's items go, in that order, each to
// its workgroup with the least work so far.  A workgroup walks its own queue,
// so it knows its next item early enough to load it ahead.
// The time of an item: its steps, and kItemSteps more for its stores and its
// change-over (measured at T383 with 32-column tiles: 0.8 us a step, 1.6 us
// of stores).
constexpr int kItemSteps = 2;

void build_lists(int dir, const std::vector<HostGroup>& groups, int bn, int slots,
                 GemmLists& out) {
  const int TR = sht::kGemmBM;
  std::vector<sht::GemmPanel> panels;
  std::vector<sht::GemmStep> steps;
  std::vector<long long> gwork(groups.size(), 0);
  std::vector<std::vector<sht::GemmItem>> per_group(groups.size());
  for (size_t gid = 0; gid < groups.size(); ++gid) {
    const HostGroup& g = groups[gid];
    int Rmax = 0;
    for (int z = 0; z < g.mcount; ++z) Rmax = std::max(Rmax, g.R[z]);
    for (int r0 = 0; r0 < Rmax; r0 += TR) {
      sht::GemmPanel pn{};
      sht::GemmItem it{};
      it.step0 = (int)steps.size();
      it.N = g.N;
      it.bcs = g.bcs;
      it.piece_bytes = g.piece_bytes;
      pn.ccs = g.ccs;
      for (int z = 0; z < sht::kMT; ++z) {
        pn.rows[z] = z < g.mcount ? std::max(0, std::min(TR, g.R[z] - r0)) : 0;
        if (dir == 0)
          pn.c[z] = z == 0 ? (unsigned long long)(g.C[0] + (size_t)r0 * sht::kMT) : 0ull;
        else
          pn.c[z] = z < g.mcount ? (unsigned long long)(g.C[z] + r0) : 0ull;
      }
      for (int sg = 0; sg < g.nseg; ++sg) {
        int kmax = 0;
        for (int z = 0; z < g.mcount; ++z) kmax = std::max(kmax, g.K[sg][z]);
        // every k-chunk is a trip of kMT steps, step z for order z (the
        // kernel fixes each step's order at compile time); an order that
        // does not reach this chunk or row tile gets a null step (extent 0:
        // its loads return zeros).  ANA: the chunk's B tile, shared by the
        // orders, comes with step 0.
        for (int k0 = 0; k0 < kmax; k0 += 32) {
          for (int z = 0; z < sht::kMT; ++z) {
            sht::GemmStep st{};
            st.z = z;
            st.cmap = g.cmap[sg];
            const bool live = z < g.mcount && k0 < g.K[sg][z] &&
                              (dir == 0 || g.Arows[sg][z] > r0);
            if (live) {
              const int chunk_rows = g.Arows[sg][z];
              st.a = (unsigned long long)(g.A[sg][z] +
                                          ((size_t)k0 * chunk_rows + (size_t)r0 * 32) * g.esz);
              st.a_bytes = (unsigned)(std::min(TR, chunk_rows - r0) * 32 * g.esz);
            } else {
              st.a = (unsigned long long)g.A[sg][0];
            }
            if (dir == 0) {
              st.b = (unsigned long long)(live ? g.B[sg][z] + (size_t)k0 * sizeof(float)
                                               : g.B[sg][0]);
              st.b_klen = live ? g.K[sg][z] - k0 : 0;
            } else if (z == 0) {
              st.b = (unsigned long long)(g.B[sg][0] + (size_t)k0 * sht::kMT * sizeof(float));
              st.b_klen = g.K[sg][0] - k0;
            }
            steps.push_back(st);
          }
        }
      }
      it.nsteps = (int)steps.size() - it.step0;
      bool any = false;
      for (int e = it.step0; e < (int)steps.size(); ++e) any = any || steps[e].a_bytes > 0;
      if (!any) {  // nothing reaches this row tile
        steps.resize(it.step0);
        continue;
      }
      if (it.nsteps + sht::kGemmNulls > sht::kGemmMaxSteps)
        fail(ARWEN_SHT_EINVAL, "truncation too large for the GEMM step list (" +
                                   std::to_string(it.nsteps) + " steps in one panel, at most " +
                                   std::to_string(sht::kGemmMaxSteps - sht::kMT) + ")");
      // null steps: the kernel's loads run ahead of the list's end
      sht::GemmStep null{};
      null.a = steps[it.step0].a;
      null.b = steps[it.step0].b ? steps[it.step0].b : steps[it.step0].a;
      for (int e = 0; e < sht::kGemmNulls; ++e) steps.push_back(null);
      panels.push_back(pn);
      it.panel = (int)panels.size();
      for (it.c0 = 0; it.c0 < g.N; it.c0 += bn) {
        gwork[gid] += it.nsteps + kItemSteps;
        per_group[gid].push_back(it);
      }
    }
  }
  const int nx = kXcds;
  std::vector<int> order(groups.size());
  for (size_t g = 0; g < order.size(); ++g) order[g] = (int)g;
  std::stable_sort(order.begin(), order.end(), [&](int a, int b) { return gwork[a] > gwork[b]; });
  std::vector<long long> load(nx, 0);
  std::vector<std::vector<sht::GemmItem>> lists(nx);
  for (int g : order) {
    if (per_group[g].empty()) continue;
    const int x = (int)(std::min_element(load.begin(), load.end()) - load.begin());
    load[x] += gwork[g];
    lists[x].insert(lists[x].end(), per_group[g].begin(), per_group[g].end());
  }
  size_t longest = 0;
  for (auto& l : lists) longest = std::max(longest, l.size());
  // workgroups per XCD; a launch takes at least one each
  const int per_xcd = (int)std::max<size_t>(1, std::min<size_t>(slots / nx, longest));
  std::vector<std::vector<sht::GemmItem>> queues((size_t)per_xcd * nx);
  for (int x = 0; x < nx; ++x) {
    using Slot = std::pair<long long, int>;  // work so far, workgroup of the XCD
    std::priority_queue<Slot, std::vector<Slot>, std::greater<Slot>> free;
    for (int b = 0; b < per_xcd; ++b) free.push({0, b});
    for (const sht::GemmItem& it : lists[x]) {
      const Slot sl = free.top();
      free.pop();
      queues[(size_t)sl.second * nx + x].push_back(it);
      free.push({sl.first + it.nsteps + kItemSteps, sl.second});
    }
  }
  longest = 0;
  for (auto& q : queues) longest = std::max(longest, q.size());
  std::vector<sht::GemmItem> t(longest * queues.size());  // zero = none
  for (size_t b = 0; b < queues.size(); ++b)
    for (size_t k = 0; k < queues[b].size(); ++k) t[k * queues.size() + b] = queues[b][k];
  // the kernel addresses the lists with 32-bit byte offsets, the items up to
  // four of a queue ahead (past the list: none)
  if (std::max(steps.size(), t.size() + 4 * queues.size()) >=
      (size_t(1) << 32) / sizeof(sht::GemmStep))
    fail(ARWEN_SHT_EINVAL, "too many operations for one GEMM work list");
  upload(out.panels, panels);
  upload(out.steps, steps);
  upload(out.items, t);
  out.nitems = (int)t.size();
  out.nsteps = (int)steps.size();
  out.bn = bn;
  out.slots = slots;
  out.grid = (int)queues.size();
}

const char* table_block(const arwen_sht_plan* P, int kind, bool syn, int m, int p,
                        long long* piece_bytes, size_t* esz) {
  long long piece;
  const char* base = static_cast<const char*>(P->table(kind, syn, &piece));
  *esz = P->precision == ARWEN_SHT_FP32 ? 4 : 2;
  *piece_bytes = piece * (long long)*esz;
  return base + (size_t)P->koff[2 * m + p] * P->JHP * *esz;
}

// Element offset of the waist block (m-tile of m, parity p) within a column,
// layout W[c][m/kMT][p][i][m%kMT].
size_t waist_offset(const arwen_sht_plan* P, int m, int p) {
  return ((size_t)((m / sht::kMT) * 2 + p) * P->JHP) * sht::kMT;
}

// Column maps of the vector operators' second data arrangement (see
// GemmStep::cmap): synthesis [i chi, i psi] = [-a3, a2, a1, -a0] of the packed
// [-psi, chi]; analysis [U, -V] = [a3, -a2, -a1, a0] of the waist [iV, iU].
constexpr int kMapSynVec = 1 | (1 << 1) | (1 << 4);
constexpr int kMapAnaVec = 1 | (1 << 2) | (1 << 3);

// GEMM data operand (fp32 in every precision mode; the split modes cut it
// into bf16 pieces as it enters the GEMM's LDS tiles).
struct DataRef {
  const char* base;
};

// Synthesis group: segments (table kind, parity, packed data, column map).
struct SynSeg {
  int kind;
  int pflip;  // data/table parity = q ^ pflip
  DataRef packed;
  int cmap;
};

void add_syn_group(std::vector<HostGroup>& b, const arwen_sht_plan* P, int mb, int q, int ncols,
                   float* waist, const SynSeg* segs, int nseg) {
  HostGroup g;
  g.nseg = nseg;
  g.N = ncols;
  g.mcount = std::min(sht::kMT, P->T + 1 - mb * sht::kMT);
  g.ccs = P->ldw;
  g.bcs = P->ldp;
  g.C[0] = waist + waist_offset(P, mb * sht::kMT, q);
  for (int sg = 0; sg < nseg; ++sg) g.cmap[sg] = segs[sg].cmap;
  for (int mm = 0; mm < g.mcount; ++mm) {
    const int m = mb * sht::kMT + mm;
    g.R[mm] = P->JHP;
    for (int sg = 0; sg < nseg; ++sg) {
      const int p = q ^ segs[sg].pflip;
      g.A[sg][mm] = table_block(P, segs[sg].kind, true, m, p, &g.piece_bytes, &g.esz);
      g.Arows[sg][mm] = P->JHP;
      g.B[sg][mm] = segs[sg].packed.base + (size_t)P->koff[2 * m + p] * sizeof(float);
      g.K[sg][mm] = P->kp(m, p);
    }
  }
  b.push_back(g);
}

// Analysis group: segments (table kind, waist parity flip, waist, column map).
struct AnaSeg {
  int kind;
  int pflip;
  DataRef waist;
  int cmap;
};

void add_ana_group(std::vector<HostGroup>& b, const arwen_sht_plan* P, int mb, int q, int ncols,
                   float* packed_out, const AnaSeg* segs, int nseg) {
  HostGroup g;
  g.nseg = nseg;
  g.N = ncols;
  g.mcount = std::min(sht::kMT, P->T + 1 - mb * sht::kMT);
  g.ccs = P->ldp;
  g.bcs = P->ldw;
  for (int sg = 0; sg < nseg; ++sg) {
    g.B[sg][0] = segs[sg].waist.base +
                 waist_offset(P, mb * sht::kMT, q ^ segs[sg].pflip) * sizeof(float);
    g.cmap[sg] = segs[sg].cmap;
  }
  for (int mm = 0; mm < g.mcount; ++mm) {
    const int m = mb * sht::kMT + mm;
    g.R[mm] = P->kp(m, q);
    g.C[mm] = packed_out + P->koff[2 * m + q];
    for (int sg = 0; sg < nseg; ++sg) {
      g.A[sg][mm] = table_block(P, segs[sg].kind, false, m, q, &g.piece_bytes, &g.esz);
      g.Arows[sg][mm] = P->kp(m, q);
      g.K[sg][mm] = P->JHP;
    }
  }
  b.push_back(g);
}

// Whether a single operation takes the few-column kernels (small_*_kernel):
// the scalar operations, while their time stays below the grouped path's.
// That grows with the fields and, through the gathers and the k chain of one
// wavefront, with the square (synthesis) or the cube (analysis, whose results
// leave in 8-byte pieces) of K = ceil((T+1)/64) k-chunks.  A batch keeps the
// grouped path whatever its jobs' sizes: there one launch serves all jobs of a
// direction, and the lines below were measured for calls of one job.  GPU time of a call
// either side of the lines, grouped -> few-column, us (float32; bf16x6 alike):
//   synthesis, fields K^2 <= 72:   T127 16 fields 17.1 -> 13.1, T255 4 21.8 ->
//     17.7, T383 2 31.8 -> 28.9
//   two contractions, <= 36:       T255 2 fields 38.0 -> 36.6, 4 39.1 -> 39.6;
//     T383 1 58.5 -> 54.7
//   analysis, fields K^3 <= 100, and 256 up to 16 fields (bf16x6): T127 16
//     fields 17.3 -> 14.3; T191 8 17.0 -> 16.1, 16 19.7 -> 23.8; T255 4
//     19.1 -> 18.1, 8 20.8 -> 21.0; T383 1 29.6 -> 27.7, 4 31.3 -> 33.6;
//     T511 1 50.3 -> 56.2
bool small_job(const arwen_sht_batch* B, const arwen_sht_job& J) {
  if (!B->single || J.op == ARWEN_SHT_OP_UV_FROM_VORDIV || J.op == ARWEN_SHT_OP_VORDIV_FROM_UV ||
      J.op == ARWEN_SHT_OP_VORDIV_FROM_WAIST || J.op == ARWEN_SHT_OP_DIVERGENCE_FROM_WAIST)
    return false;
  const long long K = (J.plan->T + 64) / 64, n = J.count;
  if (!is_synthesis(J.op)) return n * K * K * K <= (n <= 16 ? 256 : 100);
  const bool two = J.op == ARWEN_SHT_OP_GRADIENT || J.op == ARWEN_SHT_OP_SYNTHESIS_GRADIENT;
  return n * K * K <= (two ? 36 : 72);
}

// One job's share of a batch.  prepare: allocate its workspaces, add its
// grouped-GEMM work groups and its algorithmic work (once, at batch
// creation); always: append its launch arguments, which carry the caller's
// buffers (so a single-operation batch is rebound to new buffers without
// allocating).  The work groups reference only workspaces and tables.
void setup_job(arwen_sht_batch* B, JobState* js, bool prepare) {
  auto& syn = B->groups[0];
  auto& ana = B->groups[1];
  const arwen_sht_job& J = js->job;
  const arwen_sht_plan* P = J.plan;
  const int n = J.count;
  const int T = P->T;
  const bool vec = J.op == ARWEN_SHT_OP_UV_FROM_VORDIV || J.op == ARWEN_SHT_OP_VORDIV_FROM_UV ||
                   J.op == ARWEN_SHT_OP_VORDIV_FROM_WAIST;
  const bool sgrad = J.op == ARWEN_SHT_OP_SYNTHESIS_GRADIENT;
  const double pcf = 4.0 * (P->nlat / 2.0) * (T + 1.0) * (T + 2.0) / 2.0;  // FLOP per PC
  // the orders m < m0 of that (vector jobs in the split modes: FP64 kernels)
  const double pcf_low =
      4.0 * (P->nlat / 2.0) * (P->m0 * (T + 1.0) - P->m0 * (P->m0 - 1.0) / 2.0);
  // the first order tile's share (orders m < 4), four contractions per level
  // there in the plain FP32 recurrence form
  const double pcf_t0 = 4.0 * (P->nlat / 2.0) * (sht::kMT * (T + 1.0) - sht::kMT * (sht::kMT - 1.0) / 2.0);
  const double fftb = 4.0 * P->nlat * P->nlon + 8.0 * P->nlat * (T + 1.0);
  if (n == 0) return;
  if (is_synthesis(J.op)) {
    // ---- pack ----
    const int ncol = vec ? 4 : 2;
    js->ncols = ncol * n;
    const bool small = small_job(B, J);
    if (prepare && !small) js->packed_a.alloc((size_t)js->ncols * P->ldp * 4);
    if (prepare) js->waist_a.alloc((size_t)js->ncols * P->ldw * 4);
    const bool grad = J.op == ARWEN_SHT_OP_GRADIENT;
    if ((grad || sgrad) && prepare) js->waist_b.alloc((size_t)js->ncols * P->ldw * 4);
    sht::PackArgs pa{};
    pa.koff = P->d_koff.as<int>();
    pa.T = T;
    pa.mtiles = (T + 1 + 31) / 32;
    pa.job.in0 = static_cast<const float2*>(J.in0);
    pa.job.in1 = static_cast<const float2*>(J.in1);
    pa.job.out0 = js->packed_a.as<float>();
    pa.job.nfields = n;
    pa.job.col0 = 0;
    pa.job.ldp = P->ldp;
    pa.job.radius = (float)P->radius;
    // u, v with FP64 low orders: the orders m >= m0 in the recurrence form;
    // without them (plain FP32) on a wave-resident grid: the recurrence form
    // from m = 4 on, the first order tile in the two-segment form
    const bool low = J.op == ARWEN_SHT_OP_UV_FROM_VORDIV && P->m0 > 0;
    const bool recp = J.op == ARWEN_SHT_OP_UV_FROM_VORDIV && P->m0 == 0 && P->fft.wave_L > 0;
    pa.job.mode = (J.op == ARWEN_SHT_OP_ZONAL_DERIVATIVE || J.op == ARWEN_SHT_OP_ZONAL_TO_WAIST)
                      ? sht::kIM
                  : low || recp                      ? sht::kVectorRec
                  : vec                              ? sht::kVector
                  : (J.flags & ARWEN_SHT_JOB_INVLAP) ? sht::kInvLap
                                                     : sht::kPlain;
    pa.job.off00 = static_cast<const float2*>(J.coeff_offset);
    pa.job.m0 = low ? P->m0 : 0;
    pa.job.mdp = recp ? sht::kMT : 0;
    if (!small) {
      B->packs.push_back(pa);
    } else {
      // table kind and output of each contraction (dP/dphi flips the parity)
      const bool merid = J.op == ARWEN_SHT_OP_MERIDIONAL_DERIVATIVE ||
                         J.op == ARWEN_SHT_OP_MERIDIONAL_TO_WAIST;
      const int kinds[2] = {merid ? kD : grad ? kPm : kP, kD};
      const int njobs = grad || sgrad ? 2 : 1;
      sht::SmallSynArgs sa{};
      sa.in = pa.job.in0;
      sa.off00 = pa.job.off00;
      sa.koff = pa.koff;
      for (int k = 0; k < njobs; ++k) {
        sa.table[k] = P->table(kinds[k], true, &sa.piece);
        sa.waist[k] = (k == 0 ? js->waist_a : js->waist_b).as<float>();
        sa.pflip[k] = kinds[k] == kD ? 1 : 0;
      }
      sa.T = T;
      sa.JHP = P->JHP;
      sa.ldw = P->ldw;
      sa.nfields = n;
      sa.mode = pa.job.mode;
      sa.radius = pa.job.radius;
      B->small_syns.emplace_back(sa, njobs);
    }
    // ---- FP64 low orders of u, v (orders m < m0) ----
    if (low) {
      if (prepare) js->low.alloc((size_t)n * 2 * P->m0 * 2 * P->JHP * sizeof(double2));
      sht::LowSynArgs ls{};
      ls.vort = static_cast<const float2*>(J.in0);
      ls.div = static_cast<const float2*>(J.in1);
      ls.p = P->low_syn[kP].as<double>();
      ls.low = js->low.as<double2>();
      ls.radius = P->radius;
      ls.T = T;
      ls.JH = P->JH;
      ls.JHP = P->JHP;
      ls.m0 = P->m0;
      ls.nlev = n;
      B->low_syns.push_back(ls);
    }
    // ---- grouped GEMM: one group per (m-tile, output parity) ----
    const DataRef pk{js->packed_a.as<char>()};
    for (int mb = low ? P->m0 / sht::kMT : 0; prepare && !small && mb < P->MB; ++mb)
      for (int q = 0; q < 2; ++q) {
        if (low || (recp && mb >= 1)) {
          // recurrence form: a cos(phi) [u, v] = P [U, V] (pack_vector_rec_kernel)
          SynSeg sg[1] = {{kP, 0, pk, 0}};
          add_syn_group(syn, P, mb, q, js->ncols, js->waist_a.as<float>(), sg, 1);
        } else if (J.op == ARWEN_SHT_OP_UV_FROM_VORDIV) {
          // U,V = -dP/dphi (psi) + i P m/cos (chi), i P m/cos (psi) + dP/dphi (chi):
          // dP/dphi flips the parity, so its segment reads the other parity.
          SynSeg sg[2] = {{kD, 1, pk, 0}, {kPm, 0, pk, kMapSynVec}};
          add_syn_group(syn, P, mb, q, js->ncols, js->waist_a.as<float>(), sg, 2);
        } else if (J.op == ARWEN_SHT_OP_MERIDIONAL_DERIVATIVE ||
                   J.op == ARWEN_SHT_OP_MERIDIONAL_TO_WAIST) {
          SynSeg sg[1] = {{kD, 1, pk, 0}};
          add_syn_group(syn, P, mb, q, js->ncols, js->waist_a.as<float>(), sg, 1);
        } else if (grad) {
          SynSeg se[1] = {{kPm, 0, pk, 0}};
          add_syn_group(syn, P, mb, q, js->ncols, js->waist_a.as<float>(), se, 1);
          SynSeg sn[1] = {{kD, 1, pk, 0}};
          add_syn_group(syn, P, mb, q, js->ncols, js->waist_b.as<float>(), sn, 1);
        } else if (sgrad) {  // the basis waist feeds the grid and (times i m) the east
          SynSeg sp[1] = {{kP, 0, pk, 0}};
          add_syn_group(syn, P, mb, q, js->ncols, js->waist_a.as<float>(), sp, 1);
          SynSeg sn[1] = {{kD, 1, pk, 0}};
          add_syn_group(syn, P, mb, q, js->ncols, js->waist_b.as<float>(), sn, 1);
        } else {  // SYNTHESIS, ZONAL_DERIVATIVE and their waist forms
          SynSeg sg[1] = {{kP, 0, pk, 0}};
          add_syn_group(syn, P, mb, q, js->ncols, js->waist_a.as<float>(), sg, 1);
        }
      }
    // algorithmic FLOPs: one plane contraction per table application
    {
      double pcs = (J.op == ARWEN_SHT_OP_UV_FROM_VORDIV) ? 4.0 * n
                   : (grad || sgrad)                     ? 2.0 * n
                                                         : 1.0 * n;
      if (prepare && low) {  // two per level: the GEMM above m0, the FP64 kernel below
        B->legendre_flops += 2.0 * n * pcf;
        B->low_flops += 2.0 * n * pcf_low;
      } else if (prepare && recp) {  // four per level in the first order tile, two above
        B->legendre_flops += 2.0 * n * pcf + 2.0 * n * pcf_t0;
      } else if (prepare) {
        B->legendre_flops += pcs * pcf;
      }
    }
    // ---- inverse FFTs ----
    auto unfold = [&](const DevBuf& waist, void* grid, int col0, int fstride, const DevBuf& sc,
                      int imul, int post_exp = 0) {
      sht::UnfoldArgs ua{};
      ua.fft = P->fft;
      ua.T = T;
      ua.nlat = P->nlat;
      ua.JH = P->JH;
      ua.JHP = P->JHP;
      ua.job.waist = waist.as<float>();
      ua.job.grid = static_cast<float*>(grid);
      ua.job.rowscale = sc.as<float>();
      ua.job.nfields = n;
      ua.job.col0 = col0;
      ua.job.fstride = fstride;
      ua.job.ldw = P->ldw;
      ua.job.imul = imul;
      ua.job.post_exp = post_exp;
      if (low) {  // FP64 unfold; orders m < m0 from the low waist of u (col0 0) or v
        const int f = col0 == 0 ? 0 : 1;
        ua.job.f64 = 1;
        ua.job.low = js->low.as<double2>() + (size_t)f * P->m0 * 2 * P->JHP;
        ua.job.low_stride = 2 * P->m0 * 2 * P->JHP;
        // both parts in the recurrence form: a cos(phi) (u, v)
        ua.job.rowscale64 = P->scale_inv_acos64.as<double>();
        ua.job.rowscale64_hi = P->scale_inv_acos64.as<double>();
        ua.job.m0 = P->m0;
      }
      B->unfolds.push_back(ua);
      if (prepare) B->fft_bytes += n * fftb;
    };
    if (to_waist(J.op)) {
      // the reference's waist (*lead, nlat, T+1): north = E + O, south = E - O
      sht::WaistUnfoldArgs wu{};
      wu.waist = js->waist_a.as<float>();
      wu.out = static_cast<float2*>(J.out0);
      wu.T = T;
      wu.nlat = P->nlat;
      wu.JH = P->JH;
      wu.JHP = P->JHP;
      wu.ldw = P->ldw;
      wu.nfields = n;
      wu.col0 = 0;
      wu.fstride = 2;
      B->waist_unfolds.push_back(wu);
    } else if (J.op == ARWEN_SHT_OP_UV_FROM_VORDIV) {
      unfold(js->waist_a, J.out0, 0, 4, P->scale_inv_a, 0);
      unfold(js->waist_a, J.out1, 2, 4, P->scale_inv_a, 0);
      for (size_t k = B->unfolds.size() - 2; k < B->unfolds.size(); ++k)
        B->unfolds[k].job.wind = 1;
      if (recp)  // the recurrence form's orders: a cos(phi) (u, v)
        for (size_t k = B->unfolds.size() - 2; k < B->unfolds.size(); ++k) {
          B->unfolds[k].job.rowscale_hi = P->scale_inv_acos.as<float>();
          B->unfolds[k].job.m_hi = sht::kMT;
        }
    } else if (grad) {
      unfold(js->waist_a, J.out0, 0, 2, P->scale_inv_a, 1);
      unfold(js->waist_b, J.out1, 0, 2, P->scale_inv_a, 0);
    } else if (sgrad) {
      unfold(js->waist_a, J.out0, 0, 2, P->scale_one, 0);
      unfold(js->waist_a, J.out1, 0, 2, P->scale_inv_acos, 2);  // i m / (a cos)
      unfold(js->waist_b, J.out2, 0, 2, P->scale_inv_a, 0);
    } else {
      unfold(js->waist_a, J.out0, 0, 2, P->scale_one, 0, (J.flags & ARWEN_SHT_JOB_EXP) ? 1 : 0);
    }
  } else {
    // ---- FFT + fold ----
    const bool divw = J.op == ARWEN_SHT_OP_DIVERGENCE_FROM_WAIST;
    const int ncol = vec ? 4 : 2;
    js->ncols = ncol * n;
    if (prepare) js->waist_a.alloc((size_t)js->ncols * P->ldw * 4);
    if (prepare && divw) js->waist_b.alloc((size_t)js->ncols * P->ldw * 4);
    const bool small = small_job(B, J);
    if (prepare && !small) js->packed_out.alloc((size_t)js->ncols * P->ldp * 4);
    if (from_waist(J.op)) {
      // a reference waist (*lead, nlat, T+1), already divided by nlon
      sht::WaistFoldArgs wf{};
      wf.w0 = static_cast<const float2*>(J.in0);
      wf.w1 = static_cast<const float2*>(J.in1);
      wf.waist = js->waist_a.as<float>();
      wf.waist1 = divw ? js->waist_b.as<float>() : nullptr;
      wf.rowscale = (vec || divw) ? P->scale_waist_vec.as<float>() : P->scale_waist.as<float>();
      wf.T = T;
      wf.nlat = P->nlat;
      wf.JH = P->JH;
      wf.JHP = P->JHP;
      wf.ldw = P->ldw;
      wf.nfields = n;
      wf.col0 = 0;
      wf.vector = divw ? 2 : vec ? 1 : 0;
      B->waist_folds.push_back(wf);
    }
    sht::FoldArgs fa{};
    fa.fft = P->fft;
    fa.T = T;
    fa.nlat = P->nlat;
    fa.JH = P->JH;
    fa.JHP = P->JHP;
    fa.job.grid0 = static_cast<const float*>(J.in0);
    fa.job.grid1 = static_cast<const float*>(J.in1);
    fa.job.waist0 = js->waist_a.as<float>();
    fa.job.rowscale = vec ? P->scale_fold_vec.as<float>() : P->scale_fold.as<float>();
    fa.job.nfields = n;
    fa.job.col0 = 0;
    fa.job.ldw = P->ldw;
    fa.job.vector = vec ? 1 : 0;
    fa.job.fstride = ncol;
    fa.job.goff = J.grid_offset;
    const bool low = J.op == ARWEN_SHT_OP_VORDIV_FROM_UV && P->m0 > 0;
    // without FP64 low orders (plain FP32) on a wave-resident grid: the
    // recurrence form from m = 4 on, its weights 1/cos(phi) in the fold
    const bool recp = J.op == ARWEN_SHT_OP_VORDIV_FROM_UV && P->m0 == 0 && P->fft.wave_L > 0;
    if (recp) {
      fa.job.rowscale_hi = P->scale_fold_vec_cos.as<float>();
      fa.job.m_hi = sht::kMT;
    }
    if (low) {
      // FP64 folds of u and v, one field each: i U to level columns 2, 3 and
      // i V to 0, 1 (the [iV, iU] arrangement), orders m < m0 also in FP64
      if (prepare) js->low.alloc((size_t)n * 2 * P->m0 * 2 * P->JHP * sizeof(double2));
      for (int f = 0; f < 2; ++f) {
        sht::FoldArgs fh = fa;
        fh.job.grid0 = static_cast<const float*>(f == 0 ? J.in0 : J.in1);
        fh.job.grid1 = nullptr;
        fh.job.vector = 0;
        fh.job.col0 = f == 0 ? 2 : 0;
        fh.job.fstride = 4;
        fh.job.low = js->low.as<double2>() + (size_t)f * P->m0 * 2 * P->JHP;
        fh.job.low_stride = 2 * P->m0 * 2 * P->JHP;
        // both parts in the recurrence form: weights 2 pi w / (a nlon cos(phi))
        fh.job.rowscale64 = P->scale_fold_vec64_cos.as<double>();
        fh.job.rowscale64_hi = P->scale_fold_vec64_cos.as<double>();
        fh.job.m0 = P->m0;
        B->folds.push_back(fh);
      }
      if (prepare) B->fft_bytes += 2.0 * n * fftb;
      if (prepare) js->low_ab.alloc((size_t)n * P->m0 * 2 * (T + 2) * sizeof(double2));
      sht::LowAnaArgs la{};
      la.low = js->low.as<double2>();
      la.p = P->low_ana[kP].as<double>();
      la.ab = js->low_ab.as<double2>();
      la.vort = static_cast<float2*>(J.out0);
      la.div = static_cast<float2*>(J.out1);
      la.T = T;
      la.JH = P->JH;
      la.JHP = P->JHP;
      la.m0 = P->m0;
      la.nlev = n;
      B->low_anas.push_back(la);
    } else if (!from_waist(J.op)) {
      if (vec && !P->fft.wave_L) {
        // one component per launch: i U to level columns 2, 3, i V to 0, 1
        for (int f = 0; f < 2; ++f) {
          sht::FoldArgs fh = fa;
          fh.job.grid0 = static_cast<const float*>(f == 0 ? J.in0 : J.in1);
          fh.job.grid1 = nullptr;
          fh.job.vector = 0;
          fh.job.imul = 1;
          fh.job.col0 = f == 0 ? 2 : 0;
          B->folds.push_back(fh);
        }
      } else {
        B->folds.push_back(fa);
      }
      if (prepare) B->fft_bytes += (vec ? 2.0 : 1.0) * n * fftb;
    }
    const DataRef wst{js->waist_a.as<char>()};
    for (int mb = low ? P->m0 / sht::kMT : 0; prepare && !small && mb < P->MB; ++mb)
      for (int q = 0; q < 2; ++q) {
        if (low || (recp && mb >= 1)) {
          // recurrence form: [iB, iA] = P^T [iV, iU] / cos(phi); unpack_vector_rec_kernel
          AnaSeg sg[1] = {{kP, 0, wst, 0}};
          add_ana_group(ana, P, mb, q, js->ncols, js->packed_out.as<float>(), sg, 1);
        } else if (vec) {
          // zeta, D = Pm^T [iV, iU]_q + dP^T [U, -V]_{1-q}
          AnaSeg sg[2] = {{kPm, 0, wst, 0}, {kD, 1, wst, kMapAnaVec}};
          add_ana_group(ana, P, mb, q, js->ncols, js->packed_out.as<float>(), sg, 2);
        } else if (divw) {
          // D = Pm^T (iU)_q + dP^T (-V)_{1-q}
          AnaSeg sg[2] = {{kPm, 0, wst, 0}, {kD, 1, DataRef{js->waist_b.as<char>()}, 0}};
          add_ana_group(ana, P, mb, q, js->ncols, js->packed_out.as<float>(), sg, 2);
        } else {
          AnaSeg sg[1] = {{kP, 0, wst, 0}};
          add_ana_group(ana, P, mb, q, js->ncols, js->packed_out.as<float>(), sg, 1);
        }
      }
    if (prepare && low) {  // two per level: the GEMM above m0, the FP64 kernel below
      B->legendre_flops += 2.0 * n * pcf;
      B->low_flops += 2.0 * n * pcf_low;
    } else if (prepare && recp) {  // four per level in the first order tile, two above
      B->legendre_flops += 2.0 * n * pcf + 2.0 * n * pcf_t0;
    } else if (prepare) {
      B->legendre_flops += (vec ? 4.0 : divw ? 2.0 : 1.0) * n * pcf;
    }
    if (small) {
      sht::SmallAnaArgs sa{};
      sa.waist = js->waist_a.as<float>();
      sa.table = P->table(kP, false, &sa.piece);
      sa.koff = P->d_koff.as<int>();
      sa.out = static_cast<float2*>(J.out0);
      sa.off00 = static_cast<const float2*>(J.coeff_offset);
      sa.T = T;
      sa.JHP = P->JHP;
      sa.ldw = P->ldw;
      sa.nfields = n;
      B->small_anas.push_back(sa);
      return;
    }
    sht::UnpackArgs ua{};
    ua.koff = P->d_koff.as<int>();
    ua.T = T;
    ua.tiles = (T + 1 + 31) / 32;
    ua.job.in = js->packed_out.as<float>();
    ua.job.out0 = static_cast<float2*>(J.out0);
    ua.job.out1 = static_cast<float2*>(J.out1);
    ua.job.nfields = n;
    ua.job.col0 = 0;
    ua.job.ldp = P->ldp;
    ua.job.vector = vec ? 1 : 0;
    ua.job.m0 = low ? P->m0 : 0;
    ua.job.rec = low || recp ? 1 : 0;
    ua.job.mdp = recp ? sht::kMT : 0;
    ua.job.off00 = vec ? nullptr : static_cast<const float2*>(J.coeff_offset);
    B->unpacks.push_back(ua);
  }
}

// The launch arguments of every job, rebuilt from the jobs' current buffers.
void bind_jobs(arwen_sht_batch* B) {
  B->packs.clear();
  B->unfolds.clear();
  B->folds.clear();
  B->unpacks.clear();
  B->waist_unfolds.clear();
  B->waist_folds.clear();
  B->low_syns.clear();
  B->low_anas.clear();
  B->small_syns.clear();
  B->small_anas.clear();
  for (auto& js : B->jobs) setup_job(B, js.get(), false);
}

// What a job may hold, whatever its plan.
void check_job(const arwen_sht_job& J, int j) {
  if (J.count < 0) fail(ARWEN_SHT_EINVAL, "job count must be >= 0");
  const bool vec = J.op == ARWEN_SHT_OP_UV_FROM_VORDIV || J.op == ARWEN_SHT_OP_VORDIV_FROM_UV ||
                   J.op == ARWEN_SHT_OP_VORDIV_FROM_WAIST;
  const bool sgrad = J.op == ARWEN_SHT_OP_SYNTHESIS_GRADIENT;
  const bool two_out = vec || J.op == ARWEN_SHT_OP_GRADIENT || sgrad;
  const bool two_in = vec || J.op == ARWEN_SHT_OP_DIVERGENCE_FROM_WAIST;
  if (J.op < ARWEN_SHT_OP_SYNTHESIS || J.op > ARWEN_SHT_OP_DIVERGENCE_FROM_WAIST)
    fail(ARWEN_SHT_EINVAL, "unknown op " + std::to_string(J.op));
  if (J.count > 0 && (!J.in0 || !J.out0 || (two_in && !J.in1) || (two_out && !J.out1) ||
                      (sgrad && !J.out2)))
    fail(ARWEN_SHT_EINVAL, "job " + std::to_string(j) + " is missing a buffer");
  if (J.flags & ~(ARWEN_SHT_JOB_EXP | ARWEN_SHT_JOB_INVLAP))
    fail(ARWEN_SHT_EINVAL, "job " + std::to_string(j) + " has unknown flags");
  if ((J.flags & ARWEN_SHT_JOB_EXP) && J.op != ARWEN_SHT_OP_SYNTHESIS)
    fail(ARWEN_SHT_EINVAL, "ARWEN_SHT_JOB_EXP applies to ARWEN_SHT_OP_SYNTHESIS only");
  if ((J.flags & ARWEN_SHT_JOB_INVLAP) && (J.op != ARWEN_SHT_OP_SYNTHESIS || J.coeff_offset))
    fail(ARWEN_SHT_EINVAL,
         "ARWEN_SHT_JOB_INVLAP applies to ARWEN_SHT_OP_SYNTHESIS without a coeff_offset");
  if (J.grid_offset && J.op != ARWEN_SHT_OP_ANALYSIS)
    fail(ARWEN_SHT_EINVAL, "grid_offset applies to ARWEN_SHT_OP_ANALYSIS only");
  if (J.coeff_offset && J.op != ARWEN_SHT_OP_ANALYSIS && J.op != ARWEN_SHT_OP_SYNTHESIS &&
      !sgrad)
    fail(ARWEN_SHT_EINVAL,
         "coeff_offset applies to ARWEN_SHT_OP_ANALYSIS, _SYNTHESIS and _SYNTHESIS_GRADIENT only");
}

void plan_batch(arwen_sht_batch* B, const arwen_sht_job* jobs, int njobs) {
  if (njobs <= 0 || !jobs) fail(ARWEN_SHT_EINVAL, "a batch needs at least one job");
  hip_check(hipGetDevice(&B->device), "hipGetDevice");
  B->precision = jobs[0].plan ? jobs[0].plan->precision : 0;
  for (int j = 0; j < njobs; ++j) {
    const arwen_sht_job& J = jobs[j];
    const arwen_sht_plan* P = J.plan;
    if (!P) fail(ARWEN_SHT_EINVAL, "job " + std::to_string(j) + " has no plan");
    if (P->precision != B->precision)
      fail(ARWEN_SHT_EINVAL, "all plans of a batch must share one precision");
    if (P->device != B->device)
      fail(ARWEN_SHT_EINVAL, "job " + std::to_string(j) + "'s plan belongs to another device");
    check_job(J, j);
    auto js = std::make_unique<JobState>();
    js->job = J;
    setup_job(B, js.get(), true);
    B->jobs.push_back(std::move(js));
  }
  for (int d = 0; d < 2; ++d) {
    B->config.cols[d] = default_cols(d, B->groups[d], B->precision);
    build_lists(d, B->groups[d], B->config.cols[d], gemm_slots(B->config, d), B->lists[d]);
  }
  if (!g_setup_stream) hip_check(hipDeviceSynchronize(), "batch setup");
}

// plan_batch with its zero fills and uploads on `s`, before whatever the
// caller queues there next; nothing waits for them on the host.
void plan_batch_on(arwen_sht_batch* B, const arwen_sht_job* jobs, int njobs, hipStream_t s) {
  struct Scope {
    Scope(hipStream_t st, std::vector<std::vector<char>>* keep) {
      g_setup_stream = st;
      g_setup_keep = keep;
    }
    ~Scope() {
      g_setup_stream = nullptr;
      g_setup_keep = nullptr;
    }
  } scope(s, &B->setup_keep);
  plan_batch(B, jobs, njobs);
}

hipError_t launch_gemm(const arwen_sht_batch* B, int d, hipStream_t s) {
  const GemmLists& L = B->lists[d];
  sht::GemmLaunch g{};
  g.mode = B->precision;
  g.dir = d;
  g.bn = L.bn;
  g.acc2 = B->config.split_acc;
  g.panels = L.panels.as<sht::GemmPanel>();
  g.steps = L.steps.as<sht::GemmStep>();
  g.items = L.items.as<sht::GemmItem>();
  g.nitems = L.nitems;
  g.nsteps = L.nsteps;
  g.grid = L.grid;
  return sht_launch_legendre_gemm(&g, s);
}

// Phases of a batch run, in order; `ev` (optional) gets one event before
// each phase and one after the last.
// pack, synthesis GEMM, its FP64 low orders, inverse FFT, forward FFT, analysis
// GEMM, its FP64 low orders, unpack
constexpr int kPhases = 8;

void run_batch(arwen_sht_batch* B, hipStream_t s, hipEvent_t* ev = nullptr) {
  int dev;
  hip_check(hipGetDevice(&dev), "hipGetDevice");
  if (dev != B->device) fail(ARWEN_SHT_EINVAL, "batch used on a device other than its own");
  auto mark = [&](int k) {
    if (ev) hip_check(hipEventRecord(ev[k], s), "hipEventRecord");
  };
  mark(0);
  for (auto& a : B->packs) hip_check(sht_launch_pack(&a, s), "pack launch");
  mark(1);
  hip_check(launch_gemm(B, 0, s), "synthesis GEMM launch");
  for (auto& a : B->small_syns)
    hip_check(sht_launch_small_synthesis(&a.first, B->precision, a.second, s),
              "few-column synthesis launch");
  mark(2);
  for (auto& a : B->low_syns) hip_check(sht_launch_low_synthesis(&a, s), "low-order synthesis launch");
  mark(3);
  for (auto& a : B->unfolds) hip_check(sht_launch_irfft_unfold(&a, s), "irfft launch");
  for (auto& a : B->waist_unfolds) hip_check(sht_launch_waist_unfold(&a, s), "waist unfold launch");
  mark(4);
  for (auto& a : B->folds) hip_check(sht_launch_rfft_fold(&a, s), "rfft launch");
  for (auto& a : B->waist_folds) hip_check(sht_launch_waist_fold(&a, s), "waist fold launch");
  mark(5);
  hip_check(launch_gemm(B, 1, s), "analysis GEMM launch");
  for (auto& a : B->small_anas)
    hip_check(sht_launch_small_analysis(&a, B->precision, s), "few-column analysis launch");
  mark(6);
  for (auto& a : B->low_anas) hip_check(sht_launch_low_analysis(&a, s), "low-order analysis launch");
  mark(7);
  for (auto& a : B->unpacks) hip_check(sht_launch_unpack(&a, s), "unpack launch");
  mark(8);
}

void drop_graph(arwen_sht_batch* B) {
  if (B->exec) {
    (void)hipGraphExecDestroy(B->exec);
    B->exec = nullptr;
  }
  if (B->graph) {
    (void)hipGraphDestroy(B->graph);
    B->graph = nullptr;
  }
}

void apply_config(arwen_sht_batch* B, const arwen_sht_gemm_config& c) {
  for (int d = 0; d < 2; ++d) {
    if (c.cols[d] != 32 && c.cols[d] != 64 && c.cols[d] != 96)
      fail(ARWEN_SHT_EINVAL, "cols must be 32, 64 or 96");
    // the 96-column tile has no split accumulators; in the split modes it
    // would change results, so it is offered only where they are off
    if (c.cols[d] == 96 && c.split_acc && B->precision != ARWEN_SHT_FP32)
      fail(ARWEN_SHT_EINVAL, "cols 96 needs split_acc = 0 in the split-BF16 modes");
    if (c.grid[d] < 0) fail(ARWEN_SHT_EINVAL, "grid must be >= 0");
  }
  if (c.split_acc != 0 && c.split_acc != 1) fail(ARWEN_SHT_EINVAL, "split_acc must be 0 or 1");
  // the lists are rebuilt while no launch of this batch is in flight
  hip_check(hipDeviceSynchronize(), "config change");
  drop_graph(B);
  // both are there before either replaces the old ones: a failure leaves the
  // batch as it was
  GemmLists fresh[2];
  bool change[2];
  for (int d = 0; d < 2; ++d) {
    change[d] = B->lists[d].bn != c.cols[d] || B->lists[d].slots != gemm_slots(c, d);
    if (change[d]) build_lists(d, B->groups[d], c.cols[d], gemm_slots(c, d), fresh[d]);
  }
  for (int d = 0; d < 2; ++d)
    if (change[d]) B->lists[d].swap(fresh[d]);
  B->config = c;
  hip_check(hipDeviceSynchronize(), "config upload");
}

// A single operation runs as a one-job batch kept by the plan per (op,
// count, stream): its workspaces and GEMM work lists depend on those only, so
// a later call with other buffers rebinds the launch arguments on the host
// and launches, with no allocation and no synchronization.  The first call of
// a key allocates, then zero-fills and uploads on the caller's stream ahead
// of its kernels (no host wait); at most kSingleCache keys are kept, and
// evicting one waits for its stream.  Calls of one plan on one stream share
// that key's workspaces in stream order.
constexpr size_t kSingleCache = 16;

int single_job(arwen_sht_plan* P, const arwen_sht_job& job, void* stream) {
  return guarded([&] {
    if (!P) fail(ARWEN_SHT_EINVAL, "plan is NULL");
    const int op = job.op, count = job.count;
    if (count < 0) fail(ARWEN_SHT_EINVAL, "count must be >= 0");
    if (count == 0) return;
    check_job(job, 0);  // every call: a kept batch takes this one's buffers and flags
    std::lock_guard<std::mutex> lock(P->cache_mu);
    const auto key = std::make_tuple(op, count, stream);
    arwen_sht_batch* B = nullptr;
    for (auto it = P->cache.begin(); it != P->cache.end(); ++it) {
      if (it->first == key) {
        B = it->second;
        P->cache.splice(P->cache.begin(), P->cache, it);
        break;
      }
    }
    arwen_sht_job J = job;
    J.plan = P;
    if (!B) {
      auto nb = std::make_unique<arwen_sht_batch>();
      nb->single = true;
      plan_batch_on(nb.get(), &J, 1, static_cast<hipStream_t>(stream));
      B = nb.release();
      P->cache.push_front({key, B});
      while (P->cache.size() > kSingleCache) {
        auto& victim = P->cache.back();
        hip_check(hipStreamSynchronize(static_cast<hipStream_t>(std::get<2>(victim.first))),
                  "single-operation cache eviction");
        delete victim.second;
        P->cache.pop_back();
      }
    } else {
      B->jobs[0]->job = J;
      bind_jobs(B);
    }
    run_batch(B, static_cast<hipStream_t>(stream));
  });
}

int single_op(arwen_sht_plan* P, int op, const void* in0, const void* in1, void* out0,
              void* out1, int count, void* stream) {
  arwen_sht_job J{};
  J.op = op;
  J.count = count;
  J.in0 = in0;
  J.in1 = in1;
  J.out0 = out0;
  J.out1 = out1;
  return single_job(P, J, stream);
}

}  // namespace

// ---------------------------------------------------------------------------
// Exported C ABI
// ---------------------------------------------------------------------------
extern "C" {

const char* arwen_sht_last_error(void) { return g_error.c_str(); }

int arwen_sht_plan_create(const arwen_sht_plan_desc* desc, arwen_sht_plan** out) {
  return guarded([&] {
    if (!out) fail(ARWEN_SHT_EINVAL, "out is NULL");
    *out = nullptr;
    auto P = std::make_unique<arwen_sht_plan>();
    build_plan(P.get(), desc);
    *out = P.release();
  });
}

int arwen_sht_plan_destroy(arwen_sht_plan* plan) {
  return guarded([&] {
    if (!plan) return;
    (void)hipDeviceSynchronize();
    delete plan;
  });
}

int arwen_sht_plan_grid(const arwen_sht_plan* P, double* sin_lat, double* weights) {
  return guarded([&] {
    if (!P) fail(ARWEN_SHT_EINVAL, "plan is NULL");
    if (sin_lat) std::memcpy(sin_lat, P->mu.data(), P->nlat * sizeof(double));
    if (weights) std::memcpy(weights, P->w.data(), P->nlat * sizeof(double));
  });
}

size_t arwen_sht_plan_table_bytes(const arwen_sht_plan* P) { return P ? P->table_bytes() : 0; }

int arwen_sht_plan_fp64_orders(const arwen_sht_plan* P) { return P ? P->m0 : 0; }

int arwen_sht_gauss_nodes(int nlat, double* sin_lat, double* weights) {
  return guarded([&] {
    if (nlat < 1) fail(ARWEN_SHT_EINVAL, "nlat must be >= 1, got " + std::to_string(nlat));
    if (!sin_lat || !weights) fail(ARWEN_SHT_EINVAL, "sin_lat and weights are required");
    DevBuf mu((size_t)nlat * 8, false), w((size_t)nlat * 8, false);
    hip_check(sht_launch_gauss_newton(nlat, mu.as<double>(), w.as<double>(), 0),
              "gauss_newton launch");
    hip_check(hipMemcpy(sin_lat, mu.p, (size_t)nlat * 8, hipMemcpyDeviceToHost), "read nodes");
    hip_check(hipMemcpy(weights, w.p, (size_t)nlat * 8, hipMemcpyDeviceToHost), "read weights");
  });
}

int arwen_sht_plan_table_f64(const arwen_sht_plan* P, int kind, double* out) {
  return guarded([&] {
    if (!P || !out) fail(ARWEN_SHT_EINVAL, "plan and out are required");
    if (kind < 0 || kind > 2) fail(ARWEN_SHT_EINVAL, "kind must be 0 (P), 1 (dP) or 2 (P*m/cos)");
    DevBuf tab((size_t)P->tab_elems * 8, true);
    sht::TableOut t{};
    t.elems = P->tab_elems;
    t.f64_syn[kind] = tab.as<double>();
    hip_check(sht_launch_legendre_tables(P->T, P->nlat, P->JH, P->JHP, P->d_mu.as<double>(),
                                         P->d_koff.as<int>(), &t, 0),
              "legendre_tables launch");
    std::vector<double> h(P->tab_elems);
    hip_check(hipMemcpy(h.data(), tab.p, h.size() * 8, hipMemcpyDeviceToHost), "read table");
    const int T1 = P->T + 1;
    std::fill(out, out + (size_t)T1 * T1 * P->JH, 0.0);
    for (int m = 0; m <= P->T; ++m)
      for (int n = m; n <= P->T; ++n) {
        const int p = (n - m) & 1, idx = (n - m) >> 1;
        const size_t base = (size_t)P->koff[2 * m + p] * P->JHP;
        for (int i = 0; i < P->JH; ++i)
          out[((size_t)m * T1 + n) * P->JH + i] = h[base + (size_t)i * P->kp(m, p) + idx];
      }
  });
}

int arwen_sht_synthesis_to_waist(arwen_sht_plan* P, const void* coeff, void* waist, int count,
                                 int kind, void* s) {
  if (kind < 0 || kind > 2)
    return guarded([&] {
      fail(ARWEN_SHT_EINVAL, "waist kind must be 0 (basis), 1 (basis after i*m) or 2 (dP/dphi), got " +
                                 std::to_string(kind));
    });
  const int op = kind == 0   ? ARWEN_SHT_OP_SYNTHESIS_TO_WAIST
                 : kind == 1 ? ARWEN_SHT_OP_ZONAL_TO_WAIST
                             : ARWEN_SHT_OP_MERIDIONAL_TO_WAIST;
  return single_op(P, op, coeff, nullptr, waist, nullptr, count, s);
}

int arwen_sht_analysis_from_waist(arwen_sht_plan* P, const void* waist, void* coeff, int count,
                                  void* s) {
  return single_op(P, ARWEN_SHT_OP_ANALYSIS_FROM_WAIST, waist, nullptr, coeff, nullptr, count, s);
}

int arwen_sht_divergence_from_waist(arwen_sht_plan* P, const void* uw, const void* vw, void* div,
                                    int count, void* s) {
  return single_op(P, ARWEN_SHT_OP_DIVERGENCE_FROM_WAIST, uw, vw, div, nullptr, count, s);
}

int arwen_sht_vordiv_from_waist(arwen_sht_plan* P, const void* uw, const void* vw, void* vort,
                                void* div, int count, void* s) {
  return single_op(P, ARWEN_SHT_OP_VORDIV_FROM_WAIST, uw, vw, vort, div, count, s);
}

namespace {
int waist_rows(arwen_sht_plan* P, const float* rows_in, float* rows_out, const void* waist_in,
               void* waist_out, int nlead, int nrows, int row0, void* stream, bool to_rows) {
  return guarded([&] {
    if (!P) fail(ARWEN_SHT_EINVAL, "plan is NULL");
    if (nlead < 0 || nrows < 0) fail(ARWEN_SHT_EINVAL, "nlead and nrows must be >= 0");
    if (row0 < 0 || row0 + nrows > P->nlat)
      fail(ARWEN_SHT_EINVAL, "rows [" + std::to_string(row0) + ", " + std::to_string(row0 + nrows) +
                                 ") are outside the waist's " + std::to_string(P->nlat) +
                                 " latitudes");
    if ((long long)nlead * nrows == 0) return;
    if ((long long)nlead * nrows > (long long)INT32_MAX / 64)
      fail(ARWEN_SHT_EINVAL, "nlead x nrows is too large for one call");
    if ((to_rows && (!waist_in || !rows_out)) || (!to_rows && (!rows_in || !waist_out)))
      fail(ARWEN_SHT_EINVAL, "a buffer is NULL");
    int dev;
    hip_check(hipGetDevice(&dev), "hipGetDevice");
    if (dev != P->device) fail(ARWEN_SHT_EINVAL, "plan used on a device other than its own");
    sht::WaistRowsArgs a{};
    a.fft = P->fft;
    a.T = P->T;
    a.nlat = P->nlat;
    a.rows_in = rows_in;
    a.rows_out = rows_out;
    a.waist_in = static_cast<const float2*>(waist_in);
    a.waist_out = static_cast<float2*>(waist_out);
    a.nlead = nlead;
    a.nrows = nrows;
    a.row0 = row0;
    hipStream_t st = static_cast<hipStream_t>(stream);
    hip_check(to_rows ? sht_launch_rows_from_waist(&a, st) : sht_launch_waist_from_rows(&a, st),
              to_rows ? "rows_from_waist launch" : "waist_from_rows launch");
  });
}
}  // namespace

int arwen_sht_waist_from_rows(arwen_sht_plan* P, const float* rows, void* waist, int nlead,
                              int nrows, int row0, void* s) {
  return waist_rows(P, rows, nullptr, nullptr, waist, nlead, nrows, row0, s, false);
}

int arwen_sht_rows_from_waist(arwen_sht_plan* P, const void* waist, float* rows, int nlead,
                              int nrows, int row0, void* s) {
  return waist_rows(P, nullptr, rows, waist, nullptr, nlead, nrows, row0, s, true);
}

int arwen_sht_analysis(arwen_sht_plan* P, const float* grid, void* coeff, int count, void* s) {
  return single_op(P, ARWEN_SHT_OP_ANALYSIS, grid, nullptr, coeff, nullptr, count, s);
}
int arwen_sht_synthesis(arwen_sht_plan* P, const void* coeff, float* grid, int count, void* s) {
  return single_op(P, ARWEN_SHT_OP_SYNTHESIS, coeff, nullptr, grid, nullptr, count, s);
}
int arwen_sht_zonal_derivative(arwen_sht_plan* P, const void* coeff, float* grid, int count,
                               void* s) {
  return single_op(P, ARWEN_SHT_OP_ZONAL_DERIVATIVE, coeff, nullptr, grid, nullptr, count, s);
}
int arwen_sht_meridional_derivative(arwen_sht_plan* P, const void* coeff, float* grid,
                                    int count, void* s) {
  return single_op(P, ARWEN_SHT_OP_MERIDIONAL_DERIVATIVE, coeff, nullptr, grid, nullptr, count,
                   s);
}
int arwen_sht_gradient(arwen_sht_plan* P, const void* coeff, float* east, float* north,
                       int count, void* s) {
  return single_op(P, ARWEN_SHT_OP_GRADIENT, coeff, nullptr, east, north, count, s);
}
int arwen_sht_synthesis_gradient(arwen_sht_plan* P, const void* coeff, float* grid, float* east,
                                 float* north, int count, void* s) {
  arwen_sht_job J{};
  J.op = ARWEN_SHT_OP_SYNTHESIS_GRADIENT;
  J.count = count;
  J.in0 = coeff;
  J.out0 = grid;
  J.out1 = east;
  J.out2 = north;
  return single_job(P, J, s);
}

int arwen_sht_analysis_about(arwen_sht_plan* P, const float* grid, void* coeff, int count,
                             const float* grid_offset, const void* coeff_offset, void* s) {
  arwen_sht_job J{};
  J.op = ARWEN_SHT_OP_ANALYSIS;
  J.count = count;
  J.in0 = grid;
  J.out0 = coeff;
  J.grid_offset = grid_offset;
  J.coeff_offset = coeff_offset;
  return single_job(P, J, s);
}

int arwen_sht_synthesis_about(arwen_sht_plan* P, const void* coeff, float* grid, int count,
                              const void* coeff_offset, int flags, void* s) {
  arwen_sht_job J{};
  J.op = ARWEN_SHT_OP_SYNTHESIS;
  J.count = count;
  J.in0 = coeff;
  J.out0 = grid;
  J.coeff_offset = coeff_offset;
  J.flags = flags;
  return single_job(P, J, s);
}

int arwen_sht_uv_from_vordiv(arwen_sht_plan* P, const void* vort, const void* div, float* u,
                             float* v, int count, void* s) {
  return single_op(P, ARWEN_SHT_OP_UV_FROM_VORDIV, vort, div, u, v, count, s);
}
int arwen_sht_vordiv_from_uv(arwen_sht_plan* P, const float* u, const float* v, void* vort,
                             void* div, int count, void* s) {
  return single_op(P, ARWEN_SHT_OP_VORDIV_FROM_UV, u, v, vort, div, count, s);
}

int arwen_sht_spectral_op(arwen_sht_plan* P, int op, const void* in, void* out, int count,
                          void* s) {
  return guarded([&] {
    if (!P) fail(ARWEN_SHT_EINVAL, "plan is NULL");
    if (op < 0 || op > 2) fail(ARWEN_SHT_EINVAL, "op must be 0 (project), 1 or 2");
    if (count < 0) fail(ARWEN_SHT_EINVAL, "count must be >= 0");
    if (count == 0) return;
    if (!in || !out) fail(ARWEN_SHT_EINVAL, "in and out are required");
    long long total = (long long)count * (P->T + 1) * (P->T + 1);
    hip_check(sht_launch_spectral_elementwise(static_cast<const float2*>(in),
                                              static_cast<float2*>(out), total, P->T, op,
                                              (float)P->radius, static_cast<hipStream_t>(s)),
              "spectral op launch");
  });
}

namespace {
// Sampler field columns are padded to one 8-field MFMA column tile; a
// wavefront takes several, never more than there are (sht_sample_tile).
constexpr int kSampleColPad = 8;

int sample_columns(int count, int kind) {
  const long long cols = (kind == 2 ? 2LL : 1LL) * count;
  return (int)((cols + kSampleColPad - 1) / kSampleColPad * kSampleColPad);
}

// The point sampler's recurrence coefficients per packed (n, m) and per order,
// with the reference's numpy expressions (sampling.py:83-112) in double.
void build_sample_tables(arwen_sht_plan* P) {
  const int T = P->T;
  const long long K = (long long)(T + 1) * (T + 2) / 2;
  std::vector<double> rec(3 * K, 0.0), diag(2 * (T + 1), 0.0);
  long long k = 0;
  for (int m = 0; m <= T; ++m)
    for (int n = m; n <= T; ++n, ++k) {
      const double nn = n, mm2 = (double)((long long)m * m), nm2 = (double)((long long)n * n - (long long)m * m);
      if (n >= m + 2) {
        rec[k] = std::sqrt((4.0 * nn * nn - 1.0) / nm2);
        rec[K + k] = std::sqrt(((nn - 1.0) * (nn - 1.0) - mm2) / (4.0 * (nn - 1.0) * (nn - 1.0) - 1.0));
      }
      if (n > m) rec[2 * K + k] = std::sqrt(nm2 * (2.0 * nn + 1.0) / (2.0 * nn - 1.0));
    }
  for (int m = 1; m <= T; ++m) diag[m] = -std::sqrt((2 * m + 1) / (2.0 * m));
  for (int m = 0; m <= T; ++m) diag[T + 1 + m] = std::sqrt((double)(2 * m + 3));
  // both uploads succeed before the plan holds either (the sampler checks both)
  DevBuf r, dg;
  upload(r, rec);
  upload(dg, diag);
  P->sample_rec.swap(r);
  P->sample_diag.swap(dg);
}
}  // namespace

// Order-range parts per (point block, field tile): a function of T only, so
// a point's arithmetic never depends on how many points share a launch.
sht::SampleCuts sample_cuts(int T) {
  sht::SampleCuts c{};
  c.parts = std::max(1, std::min(sht::kSampleMaxParts, (T + 1) / 16));
  const long long K = (long long)(T + 1) * (T + 2) / 2;
  c.m[0] = 0;
  long long acc = 0;
  int r = 1;
  for (int m = 0; m <= T && r < c.parts; ++m) {
    acc += T + 1 - m;  // entries of orders 0..m
    if (acc * c.parts >= (long long)r * K) c.m[r++] = m + 1;
  }
  for (; r < c.parts; ++r) c.m[r] = c.m[r - 1] + 1;  // not reached for T >= 15
  c.m[c.parts] = T + 1;
  return c;
}

size_t arwen_sht_sample_workspace_bytes(const arwen_sht_plan* P, int count, int kind,
                                        int npoints) {
  if (!P || count < 0 || kind < 0 || kind > 2 || npoints < 0) return 0;
  const long long K = (long long)(P->T + 1) * (P->T + 2) / 2;
  const int ldc = sample_columns(count, kind);
  const int R = sample_cuts(P->T).parts;
  size_t bytes = (size_t)K * ldc * sizeof(double2);  // packed coefficients, either precision
  // per-part raw sums: one plane per part for values, two for derivatives
  if (R > 1) bytes += (size_t)(kind == 0 ? 1 : 2) * R * ldc * (size_t)npoints * sizeof(double);
  return bytes;
}

namespace {
// The sampler's argument checks; returns false when there is nothing to do.
bool sample_checks(const arwen_sht_plan* P, const void* in0, const void* in1, int count,
                   const double* sin_lat, const double* cos_lat, const double* lon_rad,
                   int npoints, int kind, int precision, const double* out0, const double* out1) {
  if (!P) fail(ARWEN_SHT_EINVAL, "plan is NULL");
  if (kind < 0 || kind > 2)
    fail(ARWEN_SHT_EINVAL, "sample kind must be 0 (values), 1 (gradient) or 2 (wind), got " +
                               std::to_string(kind));
  if (precision != 0 && precision != 1)
    fail(ARWEN_SHT_EINVAL, "sample precision must be 0 (float64) or 1 (float32), got " +
                               std::to_string(precision));
  if (count < 0 || npoints < 0) fail(ARWEN_SHT_EINVAL, "count and npoints must be >= 0");
  if ((long long)count * npoints == 0) return false;
  if (!in0 || (kind == 2 && !in1)) fail(ARWEN_SHT_EINVAL, "an input field is NULL");
  if (!sin_lat || !lon_rad || (kind != 0 && !cos_lat))
    fail(ARWEN_SHT_EINVAL, "a point coordinate array is NULL");
  if (!out0 || (kind != 0 && !out1)) fail(ARWEN_SHT_EINVAL, "an output is NULL");
  int dev;
  hip_check(hipGetDevice(&dev), "hipGetDevice");
  if (dev != P->device) fail(ARWEN_SHT_EINVAL, "plan used on a device other than its own");
  if (!P->sample_rec.p || !P->sample_diag.p)
    fail(ARWEN_SHT_EHIP, "the plan's sampler tables are missing");
  return true;
}

// The pack and sampler launches with the workspace at `workspace` (at least
// arwen_sht_sample_workspace_bytes of the call); allocates nothing.
void sample_launch(arwen_sht_plan* P, const void* in0, const void* in1, int count,
                   const double* sin_lat, const double* cos_lat, const double* lon_rad,
                   int npoints, int kind, int precision, void* workspace, double* out0,
                   double* out1, hipStream_t st);
}  // namespace

int arwen_sht_sample_static(arwen_sht_plan* P, const void* in0, const void* in1, int count,
                            const double* sin_lat, const double* cos_lat, const double* lon_rad,
                            int npoints, int kind, int precision, double* out0, double* out1,
                            void* s) {
  return guarded([&] {
    if (!sample_checks(P, in0, in1, count, sin_lat, cos_lat, lon_rad, npoints, kind, precision,
                       out0, out1))
      return;
    const size_t need = arwen_sht_sample_workspace_bytes(P, count, kind, npoints);
    if (need > ARWEN_SHT_SAMPLE_STATIC_BYTES)
      fail(ARWEN_SHT_EINVAL, "the sample needs a " + std::to_string(need) +
                                 "-byte workspace, more than the static array's " +
                                 std::to_string((size_t)ARWEN_SHT_SAMPLE_STATIC_BYTES) +
                                 " bytes: use arwen_sht_sample or fewer points");
    void* scratch = sht_static_scratch(P->device);
    if (!scratch) fail(ARWEN_SHT_EHIP, "the static sampler workspace of this device is unresolved");
    sample_launch(P, in0, in1, count, sin_lat, cos_lat, lon_rad, npoints, kind, precision,
                  scratch, out0, out1, static_cast<hipStream_t>(s));
  });
}

int arwen_sht_sample(arwen_sht_plan* P, const void* in0, const void* in1, int count,
                     const double* sin_lat, const double* cos_lat, const double* lon_rad,
                     int npoints, int kind, int precision, void* workspace,
                     size_t workspace_bytes, double* out0, double* out1, void* s) {
  return guarded([&] {
    if (!sample_checks(P, in0, in1, count, sin_lat, cos_lat, lon_rad, npoints, kind, precision,
                       out0, out1))
      return;
    const size_t need = arwen_sht_sample_workspace_bytes(P, count, kind, npoints);
    if (!workspace || workspace_bytes < need)
      fail(ARWEN_SHT_EINVAL, "sample workspace must hold " + std::to_string(need) + " bytes");
    sample_launch(P, in0, in1, count, sin_lat, cos_lat, lon_rad, npoints, kind, precision,
                  workspace, out0, out1, static_cast<hipStream_t>(s));
  });
}

namespace {
void sample_launch(arwen_sht_plan* P, const void* in0, const void* in1, int count,
                   const double* sin_lat, const double* cos_lat, const double* lon_rad,
                   int npoints, int kind, int precision, void* workspace, double* out0,
                   double* out1, hipStream_t st) {
  {
    const int ldc = sample_columns(count, kind);
    sht::SamplePackArgs pa{};
    pa.in0 = static_cast<const float2*>(in0);
    pa.in1 = static_cast<const float2*>(in1);
    pa.out = workspace;
    pa.f64 = precision == 0 ? 1 : 0;
    pa.radius = (double)(float)P->radius;  // the spectral operator kernel's lambda_n
    pa.T = P->T;
    pa.count = count;
    pa.ldc = ldc;
    pa.wind = kind == 2 ? 1 : 0;
    hip_check(sht_launch_sample_pack(&pa, st), "sample pack launch");
    sht::SampleArgs a{};
    a.coef = workspace;
    a.rec = P->sample_rec.as<double>();
    a.diag = P->sample_diag.as<double>();
    a.sin_lat = sin_lat;
    a.cos_lat = cos_lat ? cos_lat : sin_lat;  // unread for values
    a.lon = lon_rad;
    a.out0 = out0;
    a.out1 = out1 ? out1 : out0;  // unwritten for values
    a.cuts = sample_cuts(P->T);
    const long long K = (long long)(P->T + 1) * (P->T + 2) / 2;
    a.partial = a.cuts.parts > 1
                    ? reinterpret_cast<double*>(static_cast<char*>(workspace) +
                                                (size_t)K * ldc * sizeof(double2))
                    : nullptr;
    a.radius = P->radius;
    a.T = P->T;
    a.npts = npoints;
    a.ldc = ldc;
    a.nout = count;
    a.kind = kind;
    a.f32 = precision;
    hip_check(sht_launch_sample(&a, st), "sample launch");
  }
}
}  // namespace

int arwen_sht_vertical_solve(arwen_sht_plan* P, int nlev, const void* div, const void* theta,
                             const void* lnps, const float* b_matrix, const float* c_matrix,
                             const float* m_matrix, const float* inverse, const float* k2,
                             float s_bx, float s_md, float s_c, float s_cd, float s_cn,
                             void* div_out, void* theta_out, void* lnps_out, void* s) {
  return guarded([&] {
    if (!P) fail(ARWEN_SHT_EINVAL, "plan is NULL");
    if (nlev < 1 || nlev > sht::kMaxLevels)
      fail(ARWEN_SHT_EINVAL, "nlev must be in 1.." + std::to_string(sht::kMaxLevels) + ", got " +
                                 std::to_string(nlev));
    if (!div || !theta || !lnps || !div_out || !theta_out || !lnps_out)
      fail(ARWEN_SHT_EINVAL, "a spectral input or output is NULL");
    if (!b_matrix || !c_matrix || !inverse || !k2)
      fail(ARWEN_SHT_EINVAL, "b_matrix, c_matrix, inverse and k2 are required");
    if (s_md != 0.f && !m_matrix) fail(ARWEN_SHT_EINVAL, "s_md != 0 needs m_matrix");
    int dev;
    hip_check(hipGetDevice(&dev), "hipGetDevice");
    if (dev != P->device) fail(ARWEN_SHT_EINVAL, "plan used on a device other than its own");
    sht::VerticalArgs a{};
    a.div = static_cast<const float2*>(div);
    a.theta = static_cast<const float2*>(theta);
    a.lnps = static_cast<const float2*>(lnps);
    a.b_matrix = b_matrix;
    a.c_matrix = c_matrix;
    a.m_matrix = s_md != 0.f ? m_matrix : nullptr;
    a.inverse = inverse;
    a.k2 = k2;
    a.d_out = static_cast<float2*>(div_out);
    a.theta_out = static_cast<float2*>(theta_out);
    a.lnps_out = static_cast<float2*>(lnps_out);
    a.s_bx = s_bx;
    a.s_md = s_md;
    a.s_c = s_c;
    a.s_cd = s_cd;
    a.s_cn = s_cn;
    a.T = P->T;
    a.nlev = nlev;
    a.mode = 0;
    hip_check(sht_launch_vertical_solve(&a, static_cast<hipStream_t>(s)), "vertical solve launch");
  });
}

namespace {
void vertical_common(arwen_sht_plan* P, int nlev, const void* div, const void* theta,
                     const void* lnps, const float* b, const float* c, const float* k2,
                     void* div_out, void* theta_out, void* lnps_out, sht::VerticalArgs& a) {
  if (!P) fail(ARWEN_SHT_EINVAL, "plan is NULL");
  if (nlev < 1 || nlev > sht::kMaxLevels)
    fail(ARWEN_SHT_EINVAL, "nlev must be in 1.." + std::to_string(sht::kMaxLevels) + ", got " +
                               std::to_string(nlev));
  if (!div || !theta || !lnps || !div_out || !theta_out || !lnps_out)
    fail(ARWEN_SHT_EINVAL, "a spectral input or output is NULL");
  if (!b || !c || !k2) fail(ARWEN_SHT_EINVAL, "b_matrix, c_matrix and k2 are required");
  int dev;
  hip_check(hipGetDevice(&dev), "hipGetDevice");
  if (dev != P->device) fail(ARWEN_SHT_EINVAL, "plan used on a device other than its own");
  a.div = static_cast<const float2*>(div);
  a.theta = static_cast<const float2*>(theta);
  a.lnps = static_cast<const float2*>(lnps);
  a.b_matrix = b;
  a.c_matrix = c;
  a.k2 = k2;
  a.d_out = static_cast<float2*>(div_out);
  a.theta_out = static_cast<float2*>(theta_out);
  a.lnps_out = static_cast<float2*>(lnps_out);
  a.T = P->T;
  a.nlev = nlev;
}
}  // namespace

int arwen_sht_vertical_tendencies(arwen_sht_plan* P, int nlev, const void* div, const void* theta,
                                  const void* lnps, const float* b_matrix, const float* c_matrix,
                                  const float* k2, float weight, void* div_out, void* theta_out,
                                  void* lnps_out, void* s) {
  return guarded([&] {
    sht::VerticalArgs a{};
    vertical_common(P, nlev, div, theta, lnps, b_matrix, c_matrix, k2, div_out, theta_out,
                    lnps_out, a);
    a.s_bx = weight;
    a.s_c = weight;
    a.mode = 1;
    hip_check(sht_launch_vertical_solve(&a, static_cast<hipStream_t>(s)),
              "vertical tendencies launch");
  });
}

int arwen_sht_vertical_half_apply(arwen_sht_plan* P, int nlev, const void* div, const void* theta,
                                  const void* lnps, const float* b_matrix, const float* c_matrix,
                                  const float* p_d, const float* q_d, const float* p_x,
                                  const float* q_x, const float* k2, void* div_out,
                                  void* theta_out, void* lnps_out, void* s) {
  return guarded([&] {
    sht::VerticalArgs a{};
    vertical_common(P, nlev, div, theta, lnps, b_matrix, c_matrix, k2, div_out, theta_out,
                    lnps_out, a);
    if (!p_d || !q_d || !p_x || !q_x) fail(ARWEN_SHT_EINVAL, "the four half maps are required");
    a.p_d = p_d;
    a.q_d = q_d;
    a.p_x = p_x;
    a.q_x = q_x;
    a.mode = 2;
    hip_check(sht_launch_vertical_solve(&a, static_cast<hipStream_t>(s)), "half map launch");
  });
}

int arwen_sht_batch_create(const arwen_sht_job* jobs, int njobs, arwen_sht_batch** out) {
  return guarded([&] {
    if (!out) fail(ARWEN_SHT_EINVAL, "out is NULL");
    *out = nullptr;
    auto B = std::make_unique<arwen_sht_batch>();
    plan_batch(B.get(), jobs, njobs);
    *out = B.release();
  });
}

int arwen_sht_batch_destroy(arwen_sht_batch* B) {
  return guarded([&] {
    if (!B) return;
    (void)hipDeviceSynchronize();
    delete B;
  });
}

int arwen_sht_batch_run(arwen_sht_batch* B, void* stream) {
  return guarded([&] {
    if (!B) fail(ARWEN_SHT_EINVAL, "batch is NULL");
    run_batch(B, static_cast<hipStream_t>(stream));
  });
}

int arwen_sht_batch_capture(arwen_sht_batch* B, void* stream) {
  return guarded([&] {
    if (!B) fail(ARWEN_SHT_EINVAL, "batch is NULL");
    if (B->exec) return;
    hipStream_t s = static_cast<hipStream_t>(stream);
    bool own = false;
    if (s == nullptr) {  // the null stream cannot be captured
      hip_check(hipStreamCreate(&s), "hipStreamCreate");
      own = true;
    }
    hip_check(hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal), "begin capture");
    try {
      run_batch(B, s);
    } catch (...) {
      hipGraph_t g;
      (void)hipStreamEndCapture(s, &g);
      if (g) (void)hipGraphDestroy(g);
      if (own) (void)hipStreamDestroy(s);
      throw;
    }
    hip_check(hipStreamEndCapture(s, &B->graph), "end capture");
    hip_check(hipGraphInstantiate(&B->exec, B->graph, nullptr, nullptr, 0), "graph instantiate");
    if (own) (void)hipStreamDestroy(s);
  });
}

int arwen_sht_batch_launch(arwen_sht_batch* B, void* stream) {
  int rc = arwen_sht_batch_capture(B, stream);
  if (rc != ARWEN_SHT_OK) return rc;
  return guarded([&] {
    hip_check(hipGraphLaunch(B->exec, static_cast<hipStream_t>(stream)), "graph launch");
  });
}

int arwen_sht_batch_profile(arwen_sht_batch* B, void* stream, int reps, double* ms) {
  return guarded([&] {
    if (!B || !ms) fail(ARWEN_SHT_EINVAL, "batch and ms are required");
    if (reps < 1) fail(ARWEN_SHT_EINVAL, "reps must be >= 1");
    hipStream_t s = static_cast<hipStream_t>(stream);
    std::vector<hipEvent_t> ev((size_t)(kPhases + 1) * reps, nullptr);
    for (auto& e : ev) hip_check(hipEventCreate(&e), "hipEventCreate");
    try {
      for (int r = 0; r < reps; ++r) run_batch(B, s, &ev[(size_t)r * (kPhases + 1)]);
      hip_check(hipEventSynchronize(ev.back()), "hipEventSynchronize");
      for (int k = 0; k < kPhases; ++k) ms[k] = 0.0;
      for (int r = 0; r < reps; ++r)
        for (int k = 0; k < kPhases; ++k) {
          float t = 0.f;
          hip_check(hipEventElapsedTime(&t, ev[(size_t)r * (kPhases + 1) + k],
                                        ev[(size_t)r * (kPhases + 1) + k + 1]),
                    "hipEventElapsedTime");
          ms[k] += t / reps;
        }
    } catch (...) {
      for (auto& e : ev) (void)hipEventDestroy(e);
      throw;
    }
    for (auto& e : ev) (void)hipEventDestroy(e);
  });
}


int arwen_sht_batch_get_config(const arwen_sht_batch* B, arwen_sht_gemm_config* out) {
  return guarded([&] {
    if (!B || !out) fail(ARWEN_SHT_EINVAL, "batch and out are required");
    *out = B->config;
  });
}

int arwen_sht_batch_set_config(arwen_sht_batch* B, const arwen_sht_gemm_config* config) {
  return guarded([&] {
    if (!B || !config) fail(ARWEN_SHT_EINVAL, "batch and config are required");
    apply_config(B, *config);
  });
}

int arwen_sht_batch_autotune(arwen_sht_batch* B, void* stream, int reps,
                             arwen_sht_gemm_config* out) {
  return guarded([&] {
    if (!B) fail(ARWEN_SHT_EINVAL, "batch is NULL");
    if (reps < 1) fail(ARWEN_SHT_EINVAL, "reps must be >= 1");
    hipStream_t s = static_cast<hipStream_t>(stream);
    hipEvent_t e0, e1;
    hip_check(hipEventCreate(&e0), "hipEventCreate");
    hip_check(hipEventCreate(&e1), "hipEventCreate");
    arwen_sht_gemm_config best = B->config;
    try {
      // Each direction is timed on its own, over every column tile and grid;
      // the operands are the batch's own work buffers (their contents do not
      // change the timing).  The split-accumulator choice is a precision
      // setting and is kept as configured; the 96-column tile, which has no
      // split accumulators, is a candidate only where they are off.
      const bool wide = B->precision == ARWEN_SHT_FP32 || !B->config.split_acc;
      const std::vector<int> cols = wide ? std::vector<int>{32, 64, 96} : std::vector<int>{32, 64};
      // one generation of resident blocks, or more, whose shorter queues the
      // hardware deals as blocks end: best where the launch is long (bf16x6,
      // 96 columns, synthesis + analysis ms at 0 / 2048 / 8192 / 32768: 32 x
      // T383 4.85 / 5.29 / 5.08 / 4.57; 4 x T767 + 8 x T383 + 16 x T127 5.08 /
      // 5.22 / 4.78 / 4.78; T767 1.11 / 1.06 / 1.10 / 1.10)
      const int grids[5] = {0, 256 * 8, 256 * 16, 256 * 32, 256 * 128};
      for (int d = 0; d < 2; ++d) {
        if (B->lists[d].nitems == 0) continue;
        float best_ms = 0.f;
        for (int bn : cols) {
          int timed = -1;  // workgroups of the last launch timed
          for (int gr : grids) {
            arwen_sht_gemm_config c = best;
            c.cols[d] = bn;
            c.grid[d] = gr;
            apply_config(B, c);
            if (B->lists[d].grid == timed) continue;  // a queue for each item already
            timed = B->lists[d].grid;
            hip_check(launch_gemm(B, d, s), "autotune warm-up");
            hip_check(hipEventRecord(e0, s), "hipEventRecord");
            for (int r = 0; r < reps; ++r) hip_check(launch_gemm(B, d, s), "autotune launch");
            hip_check(hipEventRecord(e1, s), "hipEventRecord");
            hip_check(hipEventSynchronize(e1), "hipEventSynchronize");
            float ms = 0.f;
            hip_check(hipEventElapsedTime(&ms, e0, e1), "hipEventElapsedTime");
            if (best_ms == 0.f || ms < best_ms) {
              best_ms = ms;
              best.cols[d] = bn;
              best.grid[d] = gr;
            }
          }
        }
      }
      apply_config(B, best);
    } catch (...) {
      (void)hipEventDestroy(e0);
      (void)hipEventDestroy(e1);
      throw;
    }
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    if (out) *out = best;
  });
}

int arwen_sht_batch_work(const arwen_sht_batch* B, double* flops, double* bytes,
                         double* low_flops) {
  return guarded([&] {
    if (!B) fail(ARWEN_SHT_EINVAL, "batch is NULL");
    if (flops) *flops = B->legendre_flops;
    if (bytes) *bytes = B->fft_bytes;
    if (low_flops) *low_flops = B->low_flops;
  });
}

}  // extern "C"
