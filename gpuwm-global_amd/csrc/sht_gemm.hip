// Grouped Legendre GEMM over the triangular m-schedule (one persistent launch
// per direction).
//
// Every Legendre contraction of a batch is a list of work items: a panel (a
// group of up to kMT = 4 consecutive orders m of one job and one output
// parity, times one 64-row tile) and a first column (BN = 32, 64 or 96
// columns per item; 96 has no split accumulators).  Per order m the group holds
//     C_m[r][c] = sum_seg sum_k A_seg,m[r][k] * B_seg,m[k][c]
// with A a Legendre table block and B a data block; two segments express the
// vector operators (P*m/cos and dP/dphi against differently arranged data) as
// one accumulation.  The host lists each panel's k-steps (one order, 32 k) in
// execution order, with byte addresses and valid extents, so the kernel does
// no schedule arithmetic: panels come in through the scalar cache, step
// descriptors and tiles through bounds-checked buffer loads (reads past an
// extent return 0, which is also how row and column edges are handled).
//
// A step may read its B columns through a map (reverse each group of four,
// negate some of them): the vector operators' second arrangement of the data
// is such a map of the first, so only one copy is stored.
//
// Block tile 64 x BN, four wavefronts of 16 rows x BN (16x16 MFMA blocks).
// Each wavefront loads its own table fragments (16 rows x 32 k per piece)
// from the tiled table straight into registers: no table tile passes through
// LDS.  Only the data tile B, which all four wavefronts read, is staged in
// LDS (SYN: two buffers, one per step; ANA: one k-chunk, resident for its
// trip of four steps).
//
// Pipeline: four register stages (step j's tiles sit in stage j % 4, its
// order within the trip).  While the wavefronts run step j's MFMAs, the
// loads of steps j+1, j+2 and j+3 are in flight (the loop is bound by memory
// latency otherwise).  SYN writes step j+1's B to the other LDS buffer and
// one barrier ends the step; ANA needs barriers only where its resident B
// tile changes.  The panel's step descriptors sit in LDS for the whole tile,
// so no memory load other than the tiles is waited on inside the loop.
//
// A workgroup's items follow each other without a gap: the host deals each
// workgroup its queue, an item's LDS list ends with the next item's first
// three steps (null steps, extent 0, where there is none), so the last trip's
// loads are the next item's, and they are in flight while the outputs are
// stored.  The split synthesis is bound by what it moves (12 KB of table per
// step reach each block's registers through L1, for the tables once from
// memory) and by the loads' latency, not by its MFMAs: with every MFMA
// replaced by one vector operation on its operands it takes the same time
// (T383 wind, 160 columns, 64-column tiles: 62.4 against 62.2 us).  The same
// launch and its analysis took 69.4 / 77.5 us with a prologue of 4-5 us per
// tile (panel, list, first tiles, each waited on) and list order, 66.6 / 72.0
// us from the queues on the same card; 96-column analysis 78.4 -> 69.5 us.
//
// LDS B tiles are unpadded rows of 32 k, one row per column (128 bytes fp32,
// 64 bytes per bf16 piece), whose 16-byte chunks are XOR-swizzled by row, so
// that the MFMA fragment reads (16 columns x one chunk) and the tile writes
// are free of bank conflicts (measured).
//
// SYN (synthesis): rows = folded latitudes, k = degrees, C = waist
//   W[c][m/4][p][i][m%4].  Each lane keeps four order accumulators (4
//   latitudes x 4 orders = 64 contiguous bytes of the waist); the tile is
//   transposed through LDS so that stores write whole column runs.
// ANA (analysis): rows = degrees, k = folded latitudes.  The waist puts the
//   four orders of one latitude side by side, so one B tile (32 latitudes x
//   BN columns x 4 orders) is loaded once per k-chunk and serves the steps
//   of all four orders; steps flagged with a B extent start a new k-chunk.
//
// Precision modes:
//   FP32   v_mfma_f32_16x16x4_f32, fp32 tables and data.
//   BF16X3 v_mfma_f32_16x16x32_bf16 on hi+lo pieces: a0b0 + a0b1 + a1b0.
//   BF16X6 three pieces each: a0b0 + (a0b1 + a1b0) + (a0b2 + a1b1 + a2b0),
//          every term down to 2^-16 relative.  With ACC2 the five small
//          products accumulate apart from a0b0 and are added at the end.
// Tables are split once on the device from FP64 (sht_tables.hip); the data
// stay fp32 in memory and are split as their tile is written to LDS.  Each
// piece is the round-to-nearest-even bf16 of what the previous pieces leave.
// Lane l of a
// 16x16 MFMA: (l & 15) is the row/column and (l >> 4) selects the k chunk;
// A and B use the same k mapping.
#include <algorithm>
#include <type_traits>

#include "sht_kernels.h"

namespace sht {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(4))) unsigned int u32x4;
typedef __attribute__((ext_vector_type(2))) unsigned int u32x2;

// Address spaces of the device pass (the host pass only parses the kernels).
#if defined(__HIP_DEVICE_COMPILE__)
#define SHT_CONST __attribute__((address_space(4)))   // scalar-cache loads
#define SHT_GLOBAL __attribute__((address_space(1)))  // global (not flat) stores
#else
#define SHT_CONST
#define SHT_GLOBAL
#endif

constexpr int kBK = 32;  // k per step
constexpr unsigned kRsrcWord3 = 0x00020000u;  // raw buffer, 32-bit data format

// A step descriptor as loaded by every lane (two 16-byte vector loads); the
// fields are uniform and move to scalar registers with readfirstlane.
struct GemmDesc {
  u32x4 lo, hi;  // {a lo, a hi, b lo, b hi}, {a_bytes, b_klen, z, cmap}
  __device__ __forceinline__ GemmStep scalar() const {
    auto rfl = [](unsigned v) { return (unsigned)__builtin_amdgcn_readfirstlane((int)v); };
    GemmStep s;
    s.a = ((unsigned long long)rfl(lo[1]) << 32) | rfl(lo[0]);
    s.b = ((unsigned long long)rfl(lo[3]) << 32) | rfl(lo[2]);
    s.a_bytes = rfl(hi[0]);
    s.b_klen = (int)rfl(hi[1]);
    s.z = (int)rfl(hi[2]);
    s.cmap = (int)rfl(hi[3]);
    return s;
  }
};

struct GemmWork {
  const GemmPanel* panels;
  const GemmStep* steps;
  const GemmItem* items;
  int nitems, nsteps;  // entries of items and steps
};

// A work item as every lane loads it (16-byte vectors); uniform fields.
struct GemmItemRaw {
  u32x4 lo, hi;
  __device__ __forceinline__ GemmItem scalar() const {
    auto rfl = [](unsigned v) { return (unsigned)__builtin_amdgcn_readfirstlane((int)v); };
    GemmItem t;
    t.panel = (int)rfl(lo[0]);
    t.c0 = (int)rfl(lo[1]);
    t.step0 = (int)rfl(lo[2]);
    t.nsteps = (int)rfl(lo[3]);
    t.N = (int)rfl(hi[0]);
    t.bcs = (int)rfl(hi[1]);
    t.piece_bytes = (long long)(((unsigned long long)rfl(hi[3]) << 32) | rfl(hi[2]));
    return t;
  }
};

__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_rsrc(unsigned long long addr,
                                                            unsigned bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(reinterpret_cast<void*>(addr), 0, (int)bytes,
                                           (int)kRsrcWord3);
}
__device__ __forceinline__ u32x4 load16(__amdgpu_buffer_rsrc_t r, unsigned off) {
  return __builtin_amdgcn_raw_buffer_load_b128(r, (int)off, 0, 0);
}

// 16-byte chunk swizzle of an LDS row: fp32 rows have 8 chunks, bf16 rows 4.
// Chosen by measurement on gfx950 (SQ_LDS_BANK_CONFLICT over the exact
// fragment-read and tile-write patterns of this kernel): both the 16-row x
// one-chunk fragment reads and the whole-row writes are conflict-free.
template <bool F32>
__device__ __forceinline__ int swz(int row, int chunk) {
  if constexpr (F32) return chunk ^ ((row >> 1) & 7);
  else return chunk ^ ((row >> 1) & 3);
}

template <int MODE, int DIR, int BN>
struct GemmCfg {
  static constexpr bool F32 = MODE == kFP32;
  static constexpr int NP = F32 ? 1 : (MODE == kBF16X6 ? 3 : 2);  // stored pieces
  static constexpr int ESZ = F32 ? 4 : 2;   // element bytes of tables and data
  static constexpr int ROWB = kBK * ESZ;    // bytes of one row of a 32-k tile
  static constexpr int BZ = DIR == 0 ? 1 : kMT;
  static constexpr int NB = BN / 16;        // 16-column MFMA blocks per wavefront
  static constexpr int B_TILE = BZ * BN * ROWB;        // LDS bytes per piece
  static constexpr int B_BUFS = DIR == 0 ? 2 : 1;      // ANA keeps one k-chunk resident
  // register stage, in 16-byte registers per lane: the wavefront's own A
  // fragments (16 rows x 32 k: one register per bf16 piece, two for fp32),
  // loaded straight from the tiled table; the thread's share of the B tile,
  // fp32 (split into pieces when written to LDS).
  static constexpr int A_REGS = F32 ? 2 : NP;
  static constexpr int B_REGS = BZ * BN * kBK * 4 / (256 * 16);
  static_assert(B_REGS >= 1, "tile shape");
};

// Four fp32 values as `np` bf16 piece vectors (each the round-to-nearest-even
// bf16 of what the previous pieces leave; the residuals are exact in fp32).
// Pairs are converted together (v_cvt_pk_bf16_f32); a packed pair's values
// return to fp32 as its low half shifted up and its high half masked.
__device__ __forceinline__ void split4(const float (&x)[4], int np, u32x2 (&out)[3]) {
  typedef __attribute__((ext_vector_type(2))) float f2;
  typedef __attribute__((ext_vector_type(2))) __bf16 b2;
  f2 r[2] = {f2{x[0], x[1]}, f2{x[2], x[3]}};
#pragma unroll
  for (int pc = 0; pc < 3; ++pc) {
    if (pc >= np) break;
    unsigned w[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      w[h] = __builtin_bit_cast(unsigned, __builtin_convertvector(r[h], b2));
      if (pc + 1 < np) {
        r[h][0] -= __uint_as_float(w[h] << 16);
        r[h][1] -= __uint_as_float(w[h] & 0xFFFF0000u);
      }
    }
    out[pc] = u32x2{w[0], w[1]};
  }
}

template <int MODE>
__device__ __forceinline__ void mfma_step(f32x4& acc, f32x4& acc2, const u32x4 (&a)[3],
                                          const u32x4 (&b)[3]) {
#define SHT_MFMA_BF(ACC, X, Y)                                                                 \
  ACC = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, X),                \
                                                __builtin_bit_cast(bf16x8, Y), ACC, 0, 0, 0)
  if constexpr (MODE == kFP32) {
    // a[0], b[0] hold k chunk kg, a[1], b[1] chunk kg + 4 (4 floats each)
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int s = 0; s < 4; ++s)
        acc = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(a[h][s]),
                                                   __uint_as_float(b[h][s]), acc, 0, 0, 0);
  } else {
    if constexpr (MODE == kBF16X6) {
      SHT_MFMA_BF(acc2, a[2], b[0]);
      SHT_MFMA_BF(acc2, a[1], b[1]);
      SHT_MFMA_BF(acc2, a[0], b[2]);
    }
    SHT_MFMA_BF(acc2, a[1], b[0]);
    SHT_MFMA_BF(acc2, a[0], b[1]);
    SHT_MFMA_BF(acc, a[0], b[0]);
  }
#undef SHT_MFMA_BF
}

// 32-column tiles fit three workgroups per CU (<= 168 VGPRs), 64- and 96-column
// ones two (the 96-column analysis tile's LDS, B tile plus step list, is exactly
// half of the CU's 160 KB in bf16x6).
template <int MODE, int DIR, int BN, bool ACC2>
__global__ void __launch_bounds__(256, gemm_blocks_per_cu(BN)) legendre_gemm_kernel(GemmWork w) {
  using C = GemmCfg<MODE, DIR, BN>;
  constexpr bool F32 = C::F32;
  constexpr int NP = C::NP, ROWB = C::ROWB, NB = C::NB;
  __shared__ __attribute__((aligned(16))) unsigned char sB[C::B_BUFS][NP * C::B_TILE];
  // the current panel's step list, the next item's first steps (kGemmNulls)
  // and the item after that one
  __shared__ u32x4 sDesc[2 * kGemmMaxSteps];

  const SHT_CONST GemmPanel* panels = (const SHT_CONST GemmPanel*)w.panels;

  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6;
  const int li = lane & 15, kg = lane >> 4;
  const int arow = 16 * wave + li;  // the row of this lane's A fragment

  // this workgroup's items: list positions blockIdx.x + k gridDim.x (none past
  // the list)
  int pos = blockIdx.x;
  auto load_item = [&](int at) {
    GemmItem it = ((const SHT_CONST GemmItem*)w.items)[min(at, w.nitems - 1)];
    if (at >= w.nitems) it.panel = 0;
    return it;
  };
  GemmItem cur = load_item(pos), nxt = load_item(pos + (int)gridDim.x),
           nn = load_item(pos + 2 * (int)gridDim.x);
  if (cur.panel == 0) return;  // block-uniform
  GemmPanel P = panels[cur.panel - 1];

  // An item's LDS list: entries 2 j, 2 j + 1 = step j; from j = nsteps the
  // first kGemmNulls steps of the item `after` it (its own null steps where
  // there is none), then the item at list position `at3` (zeros = none past
  // the list).  At most 512 16-byte entries.  load_list takes a thread's first
  // entry and the item's two, without branches; put_list writes them, and
  // loads and writes the second entry of a list of more than 256.
  const __amdgpu_buffer_rsrc_t srs =
      make_rsrc(reinterpret_cast<unsigned long long>(w.steps), (unsigned)w.nsteps * 32u);
  const __amdgpu_buffer_rsrc_t irs =
      make_rsrc(reinterpret_cast<unsigned long long>(w.items), (unsigned)w.nitems * 32u);
  constexpr unsigned kNoRead = ~15u;  // past every extent: 0, and no memory access
  auto list_entry = [&](int q, const GemmItem& it, const GemmItem& after) {
    const int n2 = 2 * it.nsteps;
    const int own = 2 * it.step0, tail = (after.panel ? 2 * after.step0 : own + n2) - n2;
    const unsigned off = (unsigned)(q + (q < n2 ? own : tail)) * 16u;
    return load16(srs, q < n2 + 2 * kGemmNulls ? off : kNoRead);
  };
  auto load_list = [&](u32x4(&e)[2], const GemmItem& it, const GemmItem& after, int at3) {
    int tl = threadIdx.x;
    asm volatile("" : "+v"(tl));  // formed per item, not held across the loop
    e[0] = list_entry(tl, it, after);
    e[1] = load16(irs, tl < 2 ? (unsigned)at3 * 32u + (unsigned)tl * 16u : kNoRead);
  };
  auto put_list = [&](const u32x4(&e)[2], const GemmItem& it, const GemmItem& after) {
    int tl = threadIdx.x;
    asm volatile("" : "+v"(tl));
    const int n = 2 * (it.nsteps + kGemmNulls);
    if (tl < n) sDesc[tl] = e[0];
    if (tl < 2) sDesc[n + tl] = e[1];
    if (n > 256 && tl + 256 < n) sDesc[tl + 256] = list_entry(tl + 256, it, after);
  };

  // ---- register stages and their loads: step j's tiles sit in stage j % 4
  // (its order within the trip), so loads run three steps ahead.  ANA loads B
  // once per trip (one stage). ----
  constexpr int kStages = kMT;
  constexpr int kBStages = DIR == 0 ? kStages : 1;
  u32x4 ra[kStages][C::A_REGS], rb[kBStages][C::B_REGS];
  int nsteps = cur.nsteps;
  auto fetch_desc = [&](int j) {
    const int e = 2 * min(j, nsteps + kGemmNulls - 1);
    return GemmDesc{sDesc[e], sDesc[e + 1]};
  };
  // what a step's loads need of its item
  struct Cols {
    long long piece_bytes;
    unsigned long long coloff;
    int ncol, bcs;
  };
  auto cols_of = [](const GemmItem& it) {
    return Cols{it.piece_bytes, (unsigned long long)it.c0 * it.bcs * 4,  // fp32 data
                min(BN, it.N - it.c0), it.bcs};
  };
  Cols in = cols_of(cur);  // of the item whose steps are being loaded
  // WITH_B: the step may carry a B tile (SYN: every step; ANA: the first
  // step of each k-chunk, position 0 of a trip of kMT steps)
  auto issue = [&](u32x4(&A)[C::A_REGS], u32x4(&B)[C::B_REGS], const GemmStep& s,
                   auto WITH_B) {
    // A: this lane's fragment of each piece, 16 bytes (bf16: k chunk kg of
    // row arow; fp32: chunks kg and kg + 4); rows past a_bytes read 0
#pragma unroll
    for (int pc = 0; pc < NP; ++pc) {
      const __amdgpu_buffer_rsrc_t r =
          make_rsrc(s.a + (unsigned long long)(pc * in.piece_bytes), s.a_bytes);
      if constexpr (F32) {
        A[0] = load16(r, (unsigned)(arow * ROWB + kg * 16));
        A[1] = load16(r, (unsigned)(arow * ROWB + (kg + 4) * 16));
      } else {
        A[pc] = load16(r, (unsigned)(arow * ROWB + kg * 16));
      }
    }
    const int rev = (s.cmap & 1) ? 3 : 0;
    if constexpr (DIR == 0) {
      // packed fp32 columns, k contiguous: a thread takes 4 k of one column
      int ext = (in.ncol - 1) * in.bcs + s.b_klen;
      asm volatile("" : "+s"(ext));  // a select, not a branch across the step's loads
      const unsigned bytes = s.b_klen > 0 ? (unsigned)ext * 4u : 0u;
      const __amdgpu_buffer_rsrc_t r = make_rsrc(s.b + in.coloff, bytes);
#pragma unroll
      for (int u = 0; u < C::B_REGS; ++u) {
        const int q = tid + 256 * u;
        const int col = q >> 3;
        B[u] = load16(r, (unsigned)((col ^ rev) * in.bcs * 4 + (q & 7) * 16));
      }
    } else if constexpr (decltype(WITH_B)::value) {
      // k-chunk of the fp32 waist: per column 32 latitudes x 4 orders; a
      // thread takes 4 latitudes (a quad, 64 bytes) of one column
      int ext = (in.ncol - 1) * in.bcs + s.b_klen * kMT;
      asm volatile("" : "+s"(ext));
      const unsigned bytes = s.b_klen > 0 ? (unsigned)ext * 4u : 0u;
      const __amdgpu_buffer_rsrc_t r = make_rsrc(s.b + in.coloff, bytes);
#pragma unroll
      for (int u = 0; u < BN / 32; ++u) {
        const int q = tid + 256 * u;
        const int col = q >> 3, quad = q & 7;
        const unsigned off = (unsigned)((col ^ rev) * in.bcs * 4 + quad * 64);
#pragma unroll
        for (int h = 0; h < 4; ++h) B[u * 4 + h] = load16(r, off + 16u * h);
      }
    }
  };
  // B stage -> LDS (split into pieces in the bf16 modes); `cmap` bits 1..4
  // negate columns 0..3 of each group of four
  auto put_b = [&](const u32x4(&B)[C::B_REGS], int buf, int cmap) {
    auto flip_of = [&](int col) { return ((cmap >> (1 + (col & 3))) & 1) ? 0x80000000u : 0u; };
    if constexpr (DIR == 0) {
#pragma unroll
      for (int u = 0; u < C::B_REGS; ++u) {
        const int q = tid + 256 * u;
        const int col = q >> 3, ch = q & 7;  // 4 k starting at 4 ch
        const u32x4 v = B[u] ^ flip_of(col);
        unsigned char* row = &sB[buf][col * ROWB];
        if constexpr (F32) {
          *reinterpret_cast<u32x4*>(row + swz<true>(col, ch) * 16) = v;
        } else {
          const float x[4] = {__uint_as_float(v[0]), __uint_as_float(v[1]),
                              __uint_as_float(v[2]), __uint_as_float(v[3])};
          u32x2 pcs[3];
          split4(x, NP, pcs);
#pragma unroll
          for (int pc = 0; pc < NP; ++pc)
            *reinterpret_cast<u32x2*>(row + pc * C::B_TILE + swz<false>(col, ch >> 1) * 16 +
                                      (ch & 1) * 8) = pcs[pc];
        }
      }
    } else {
      (void)buf;
#pragma unroll
      for (int u = 0; u < BN / 32; ++u) {
        const int q = tid + 256 * u;
        const int col = q >> 3, quad = q & 7;
        const unsigned flip = flip_of(col);
        const u32x4* v = &B[u * 4];  // v[h] = latitude 4 quad + h, four orders
#pragma unroll
        for (int z = 0; z < kMT; ++z) {
          unsigned char* row = &sB[0][(z * BN + col) * ROWB];
          const u32x4 wv = u32x4{v[0][z], v[1][z], v[2][z], v[3][z]} ^ flip;
          if constexpr (F32) {
            *reinterpret_cast<u32x4*>(row + swz<true>(col, quad) * 16) = wv;
          } else {
            const float x[4] = {__uint_as_float(wv[0]), __uint_as_float(wv[1]),
                                __uint_as_float(wv[2]), __uint_as_float(wv[3])};
            u32x2 pcs[3];
            split4(x, NP, pcs);
#pragma unroll
            for (int pc = 0; pc < NP; ++pc)
              *reinterpret_cast<u32x2*>(row + pc * C::B_TILE + swz<false>(col, quad >> 1) * 16 +
                                        (quad & 1) * 8) = pcs[pc];
          }
        }
      }
    }
  };

  f32x4 acc[kMT][NB], acc2[kMT][NB];

  // B fragments of a step's column block nb from LDS buffer `buf`
  auto fragment = [&](int buf, auto ZC, int nb, u32x4(&bf)[3]) {
    const int bbuf = DIR == 0 ? buf : 0;
    constexpr int bz = DIR == 0 ? 0 : decltype(ZC)::value;
    const int col = nb * 16 + li;
    const unsigned char* base = &sB[bbuf][(bz * BN + col) * ROWB];
    if constexpr (F32) {
#pragma unroll
      for (int h = 0; h < 2; ++h)
        bf[h] = *reinterpret_cast<const u32x4*>(base + swz<true>(col, kg + 4 * h) * 16);
    } else {
#pragma unroll
      for (int pc = 0; pc < NP; ++pc)
        bf[pc] = *reinterpret_cast<const u32x4*>(base + pc * C::B_TILE + swz<false>(col, kg) * 16);
    }
  };
  // one step into the accumulators of order Z: A fragments from register
  // stage Z, B fragments from LDS buffer `buf` (kEarly: block 0's already in bf)
  constexpr bool kEarly = DIR == 0 || F32;
  auto compute = [&](int buf, auto ZC, u32x4(&bf)[3]) {
    constexpr int Z = decltype(ZC)::value;
    u32x4 af[3];
#pragma unroll
    for (int r = 0; r < C::A_REGS; ++r) af[r] = ra[Z][r];
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
      if (nb > 0 || !kEarly) fragment(buf, ZC, nb, bf);
      if constexpr (ACC2) mfma_step<MODE>(acc[Z][nb], acc2[Z][nb], af, bf);
      else mfma_step<MODE>(acc[Z][nb], acc[Z][nb], af, bf);
    }
  };

  // ---- the first item's prologue: steps 0, 1 and 2 in flight, step 0's B
  // in LDS buffer 0 ----
  // q1, q2, q3: steps j+1, j+2, j+3 (scalar) at the start of step j; dn:
  // the raw descriptor of step j+4, fetched one step ahead.
  GemmStep q1, q2, q3;
  GemmDesc dn;
  u32x4 list[2];
  load_list(list, cur, nxt, pos + 3 * (int)gridDim.x);
  put_list(list, cur, nxt);
  __syncthreads();
  {
    const GemmStep s0 = fetch_desc(0).scalar();
    q1 = fetch_desc(1).scalar();
    q2 = fetch_desc(2).scalar();
    issue(ra[0], rb[0], s0, std::true_type{});
    issue(ra[1], rb[DIR == 0 ? 1 : 0], q1, std::integral_constant<bool, DIR == 0>{});
    issue(ra[2], rb[DIR == 0 ? 2 : 0], q2, std::integral_constant<bool, DIR == 0>{});
    q3 = fetch_desc(3).scalar();
    dn = fetch_desc(4);
    put_b(rb[0], 0, s0.cmap);
  }
  __syncthreads();

  for (;;) {
    const int c0 = cur.c0, ncol = in.ncol;
#pragma unroll
    for (int a = 0; a < kMT; ++a)
#pragma unroll
      for (int n = 0; n < NB; ++n) {
        acc[a][n] = f32x4{0.f, 0.f, 0.f, 0.f};
        acc2[a][n] = f32x4{0.f, 0.f, 0.f, 0.f};
      }

    // ---- main loop: trips of kMT steps, one per order Z of the panel (the
    // host pads every k-chunk to kMT steps), so each step's accumulators,
    // register stage and LDS buffer are fixed at compile time ----
    // The last trip loads the next item's first three steps (the list goes on
    // with them), so an item begins with its tiles in flight.
    int next_cmap = 0;  // of the next item's step 0 (ANA)
    auto body = [&](auto ZC, int j, bool last) {
      constexpr int Z = decltype(ZC)::value;
      constexpr int s = Z & 1;               // LDS buffer of step j's B (SYN)
      constexpr int R3 = (Z + 3) % kStages;  // register stage (= trip position) of step j+3
      constexpr int R1 = (Z + 1) % kStages;  // register stage of step j+1
      // the first fragments' LDS reads go ahead of the loads' issue (the split
      // analysis, whose registers are full, leaves the order to the compiler)
      u32x4 bf[3];
      if constexpr (kEarly) {
        fragment(s, ZC, 0, bf);
        __builtin_amdgcn_sched_barrier(0);
      }
      issue(ra[R3], rb[DIR == 0 ? R3 : 0], q3, std::integral_constant<bool, DIR == 0 || R3 == 0>{});
      const GemmStep q4 = dn.scalar();
      dn = fetch_desc(j + 5);
      compute(s, ZC, bf);
      if constexpr (DIR == 0) {
        // step j+1's B goes to the other buffer; the barrier orders it before
        // step j+1 reads it and after every read of this buffer two steps ago
        // (in the split modes after the MFMAs: among them, its wait for the
        // loads would stall them; FP32's MFMAs are long, and its tile goes
        // between them: launches of one item a workgroup 1-3% faster)
        if constexpr (!F32) __builtin_amdgcn_sched_barrier(0);
        put_b(rb[R1], s ^ 1, q1.cmap);
        __syncthreads();
      } else if constexpr (R1 == 0) {
        // ANA: the resident B tile changes with the next trip
        next_cmap = q1.cmap;
        if (!last) {
          __syncthreads();  // every wavefront is done with it
          put_b(rb[0], 0, q1.cmap);
          __syncthreads();
        }
      }
      q1 = q2;
      q2 = q3;
      q3 = q4;
    };
    static_assert(kMT == 4, "trip of four steps");
    GemmItem n3{};
    for (int j = 0; j < nsteps; j += kMT) {
      const bool last = j + kMT >= nsteps;
      body(std::integral_constant<int, 0>{}, j, last);
      if (last && nxt.panel) {
        in = cols_of(nxt);
        // the item after the next two, which this list ends with: read here,
        // where barriers still lie between it and any wavefront's put_list
        // (SYN: the ends of the next three steps; ANA: the epilogue's)
        const int e = 2 * (nsteps + kGemmNulls);
        n3 = GemmItemRaw{sDesc[e], sDesc[e + 1]}.scalar();
      }
      body(std::integral_constant<int, 1>{}, j + 1, last);
      body(std::integral_constant<int, 2>{}, j + 2, last);
      body(std::integral_constant<int, 3>{}, j + 3, last);
    }
    if (nxt.panel) load_list(list, nxt, nn, pos + 4 * (int)gridDim.x);

    // ---- epilogue: this lane holds rows 16 wave + 4 kg + q (q < 4) of
    // column 16 nb + li.  The thread index is made opaque, so that nothing
    // derived from it here is formed before the loop and held across it. ----
    int te = threadIdx.x;
    asm volatile("" : "+v"(te));
    const int elane = te & 63, ewave = te >> 6, eli = te & 15, ekg = elane >> 4;
    auto wave_lds_sync = [] {  // this wavefront's LDS accesses, in order
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    };
    if constexpr (DIR == 0) {
      // A elane's four rows x four orders are 64 contiguous bytes of the
      // waist, and the four lanes of a column 256.  Each column block passes
      // through the wavefront's own LDS area, transposed, so that a store
      // instruction writes four whole 256-byte column runs rather than 16-byte
      // pieces of sixteen columns (measured: ~10 us of a T383 synthesis).
      // each wavefront's 16 rows x 16 columns of 4-order values (rows padded
      // to 17 against bank conflicts); declared here, so the analysis
      // instantiations keep their LDS budget
      __shared__ f32x4 sOut[4 * 16 * 17];
      f32x4* mine = sOut + ewave * 16 * 17;
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          f32x4 o;
#pragma unroll
          for (int zz = 0; zz < kMT; ++zz) {
            f32x4 v = acc[zz][nb];
            if constexpr (!F32 && ACC2) v = v + acc2[zz][nb];
            o[zz] = v[q];
          }
          mine[eli * 17 + 4 * ekg + q] = o;
        }
        wave_lds_sync();
        const int r = elane & 15, row = 16 * ewave + r;
#pragma unroll
        for (int tt = 0; tt < 4; ++tt) {  // columns 4 tt + elane / 16 of the block, row r
          const int cl = 4 * tt + (elane >> 4), col = nb * 16 + cl;
          const f32x4 o = mine[cl * 17 + r];
          if (col < ncol && row < P.rows[0])
            *reinterpret_cast<SHT_GLOBAL f32x4*>(reinterpret_cast<SHT_GLOBAL float*>(P.c[0]) +
                                                 (long long)(c0 + col) * P.ccs +
                                                 (long long)row * kMT) = o;
        }
        wave_lds_sync();  // the area is read before the next block lands
      }
    } else {
      // rows row..row+3 of one order are 16 contiguous bytes of the packed
      // output, a column's 64 rows (four wavefronts) 256: per order, the
      // block's tile passes through LDS (the B tile's space, free after the
      // loop) so that a store instruction writes four whole column runs
      // (measured: FP32 analysis with 32-column tiles 187 -> 171 us at T383)
      constexpr int CS = 68;  // floats per staged column: 64 rows + pad
      static_assert(BN * CS * 4 <= C::B_BUFS * NP * C::B_TILE, "staging fits the B tile");
      float* stage = reinterpret_cast<float*>(&sB[0][0]);
#pragma unroll
      for (int zz = 0; zz < kMT; ++zz) {
        __syncthreads();  // the B tile (or the previous order's stage) is consumed
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
          f32x4 v = acc[zz][nb];
          if constexpr (!F32 && ACC2) v = v + acc2[zz][nb];
          *reinterpret_cast<f32x4*>(stage + (nb * 16 + eli) * CS + 16 * ewave + 4 * ekg) = v;
        }
        __syncthreads();
        const int r4 = 4 * (elane & 15);
#pragma unroll
        for (int tt = 0; tt < BN / 16; ++tt) {  // columns 4 (ewave + 4 tt) + elane / 16
          const int col = 4 * (ewave + 4 * tt) + (elane >> 4);
          const f32x4 o = *reinterpret_cast<const f32x4*>(stage + col * CS + r4);
          if (col < ncol && r4 < P.rows[zz])
            *reinterpret_cast<SHT_GLOBAL f32x4*>(reinterpret_cast<SHT_GLOBAL float*>(P.c[zz]) +
                                                 (long long)(c0 + col) * P.ccs + r4) = o;
        }
      }
    }
    if (nxt.panel == 0) break;  // block-uniform
    cur = nxt;
    P = panels[cur.panel - 1];
    nxt = nn;
    nn = n3;
    pos += gridDim.x;
    nsteps = cur.nsteps;
    if constexpr (DIR == 1) {
      __syncthreads();  // the staged outputs are read: sB is free
      put_b(rb[0], 0, next_cmap);
    }
    // every wavefront has passed its last reads of the old list: they precede
    // the barrier that ends the loop (SYN) or those of the epilogue (ANA)
    put_list(list, cur, nxt);
    __syncthreads();
    q1 = fetch_desc(1).scalar();
    q2 = fetch_desc(2).scalar();
    q3 = fetch_desc(3).scalar();
    dn = fetch_desc(4);
  }
}

// ---------------------------------------------------------------------------
// Few columns: contraction straight from and to the boundary layout
// ---------------------------------------------------------------------------
// A single operation on a few fields is bound by latency: of its launches
// (pack, grouped GEMM, FFTs) the GEMM walks up to 24 dependent steps in its
// longest panels (four orders after each other) behind a chain of list and
// descriptor loads, and pack and unpack are a launch each.  Here a wavefront
// takes one order alone (a block the four orders of an m-tile, so that the
// waist is written in 16-byte pieces), addresses follow from the indices, and
// the data operand is gathered from, and the result scattered to, the
// (n, m) arrays, so pack and unpack disappear.  Every output runs the same
// MFMAs in the same order as the grouped GEMM's (two accumulators in the
// split modes), so the bits are the same.
// No LDS in the loop: lane (li, kg) gathers its own B fragment, 8 values of
// column li, once for all of the wavefront's RT row tiles; the next k-chunk's
// gathers and table fragments are in flight behind the current one's MFMAs.
// Measured (GPU time of a whole call): one field's synthesis at T63 13.3 ->
// 6.9 us, T127 15.6 -> 8.4, T255 21.0 -> 13.4; its analysis 11.4 -> 7.2,
// 13.6 -> 8.8, 18.3 -> 17.2.

// B fragment of 32 k for this lane from its values x[j], in the layout of
// mfma_step (fp32: x[4 h + s] at k = 16 h + 4 kg + s; bf16: x[j] at
// k = 8 kg + j).
template <int MODE>
__device__ __forceinline__ void small_fragment(const float (&x)[8], u32x4 (&b)[3]) {
  if constexpr (MODE == kFP32) {
#pragma unroll
    for (int h = 0; h < 2; ++h)
      b[h] = u32x4{__float_as_uint(x[4 * h]), __float_as_uint(x[4 * h + 1]),
                   __float_as_uint(x[4 * h + 2]), __float_as_uint(x[4 * h + 3])};
  } else {
    constexpr int NP = MODE == kBF16X6 ? 3 : 2;
    u32x2 lo[3], hi[3];
    const float a[4] = {x[0], x[1], x[2], x[3]}, c[4] = {x[4], x[5], x[6], x[7]};
    split4(a, NP, lo);
    split4(c, NP, hi);
#pragma unroll
    for (int pc = 0; pc < NP; ++pc) b[pc] = u32x4{lo[pc][0], lo[pc][1], hi[pc][0], hi[pc][1]};
  }
}
// k within its 32-chunk of value j of lane group kg
template <int MODE>
__device__ __forceinline__ int small_k(int j, int kg) {
  return MODE == kFP32 ? 16 * (j >> 2) + 4 * kg + (j & 3) : 8 * kg + j;
}
// A fragments of one 16-row tile and k-chunk: `tile` = row 0 of the tile in
// the tiled table (bytes), rows of 32 k.
template <int MODE>
__device__ __forceinline__ void small_table(const char* tile, long long piece_bytes, int li, int kg,
                                            u32x4 (&a)[3]) {
  if constexpr (MODE == kFP32) {
    a[0] = *reinterpret_cast<const u32x4*>(tile + li * 128 + kg * 16);
    a[1] = *reinterpret_cast<const u32x4*>(tile + li * 128 + (kg + 4) * 16);
  } else {
#pragma unroll
    for (int pc = 0; pc < (MODE == kBF16X6 ? 3 : 2); ++pc)
      a[pc] = *reinterpret_cast<const u32x4*>(tile + pc * piece_bytes + li * 64 + kg * 16);
  }
}

// The k loop of both directions: nch chunks; load(k) gives this lane's stored
// data value at k, shape(k, v) the operand value from it (apart, so that a
// chunk's loads are all in flight before the first is used), table(ch, rt)
// the first row of a tile.
template <int MODE, int RT, class Load, class Shape, class Table>
__device__ __forceinline__ void small_contract(f32x4 (&acc)[RT], int nch, int kg, int li,
                                               long long piece_bytes, Load&& load, Shape&& shape,
                                               Table&& table) {
  f32x4 acc2[RT];
#pragma unroll
  for (int rt = 0; rt < RT; ++rt) acc[rt] = acc2[rt] = f32x4{0.f, 0.f, 0.f, 0.f};
  float x[8];
  u32x4 a[RT][3];
  auto fetch = [&](int ch) {
#pragma unroll
    for (int j = 0; j < 8; ++j) x[j] = load(32 * ch + small_k<MODE>(j, kg));
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) small_table<MODE>(table(ch, rt), piece_bytes, li, kg, a[rt]);
  };
  if (nch > 0) fetch(0);
  for (int ch = 0; ch < nch; ++ch) {
    u32x4 b[3], c[RT][3];
#pragma unroll
    for (int j = 0; j < 8; ++j) x[j] = shape(32 * ch + small_k<MODE>(j, kg), x[j]);
    small_fragment<MODE>(x, b);
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
      for (int pc = 0; pc < 3; ++pc) c[rt][pc] = a[rt][pc];
    if (ch + 1 < nch) fetch(ch + 1);
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
      if constexpr (MODE == kFP32) mfma_step<MODE>(acc[rt], acc[rt], c[rt], b);
      else mfma_step<MODE>(acc[rt], acc2[rt], c[rt], b);
    }
  }
  if constexpr (MODE != kFP32)
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) acc[rt] = acc[rt] + acc2[rt];
}

// Synthesis: grid (m-tile, output parity, row group) x column group (8
// fields) x job.
template <int MODE, int RT>
__global__ void __launch_bounds__(256) small_synthesis_kernel(SmallSynArgs a) {
  constexpr int ESZ = MODE == kFP32 ? 4 : 2;
  __shared__ float sOut[16 * 17 * 4];  // [column][row, padded][order]
  const int lane = threadIdx.x & 63, z = threadIdx.x >> 6;
  const int li = lane & 15, kg = lane >> 4;
  const int rg = (int)blockIdx.x % a.rgroups, q = (int)blockIdx.x / a.rgroups % 2;
  const int mb = (int)blockIdx.x / a.rgroups / 2;
  const int job = blockIdx.z, T1 = a.T + 1;
  const int m = mb * kMT + z, p = q ^ a.pflip[job];
  const int kc = m <= a.T ? (a.T - m - p) / 2 + (a.T >= m + p ? 1 : 0) : 0;  // degrees m + p + 2 k
  const int f = (int)blockIdx.y * 8 + (li >> 1), part = li & 1;
  const bool live = f < a.nfields;
  const float* in = reinterpret_cast<const float*>(a.in + (size_t)min(f, a.nfields - 1) * T1 * T1);
  const int comp = a.mode == kIM ? part ^ 1 : part;
  const double a2 = (double)a.radius * (double)a.radius;
  auto load = [&](int k) {
    return in[2 * ((size_t)min(m + p + 2 * k, a.T) * T1 + m) + comp];
  };
  const float im = a.mode == kIM ? (part ? (float)m : -(float)m) : 1.f;  // x * 1 = x exactly
  const bool inv = a.mode == kInvLap;
  const float2 off = a.off00 && m == 0 ? a.off00[min(f, a.nfields - 1)] : make_float2(0.f, 0.f);
  const float add = part ? off.y : off.x;
  auto shape = [&](int k, float v) {
    const int n = m + p + 2 * k;
    v *= im;
    if (inv) {  // the spectral inverse Laplacian's own arithmetic
      const float eig = (float)(-((double)n * ((double)n + 1.0)) / a2);
      v = n >= 1 && !(m == 0 && part) ? v / eig : 0.f;
    }
    if (a.off00 && n == 0) v += add;
    return live && k < kc ? v : 0.f;
  };
  const char* tab = static_cast<const char*>(a.table[job]) +
                    (size_t)a.koff[2 * min(m, a.T) + p] * a.JHP * ESZ;
  const int r0 = rg * RT * 16;
  f32x4 acc[RT];
  small_contract<MODE, RT>(acc, (kc + 31) / 32, kg, li, a.piece * ESZ, load, shape, [&](int ch, int rt) {
    return tab + ((size_t)ch * a.JHP + min(r0 + 16 * rt, a.JHP - 16)) * 32 * ESZ;
  });
  const int col = threadIdx.x >> 4, row = threadIdx.x & 15, c = (int)blockIdx.y * 16 + col;
#pragma unroll
  for (int rt = 0; rt < RT; ++rt) {
#pragma unroll
    for (int r = 0; r < 4; ++r) sOut[(li * 17 + 4 * kg + r) * 4 + z] = acc[rt][r];
    __syncthreads();
    if (c < 2 * a.nfields && r0 + 16 * rt < a.JHP)
      *reinterpret_cast<f32x4*>(a.waist[job] + (size_t)c * a.ldw +
                                ((size_t)(mb * 2 + q) * a.JHP + r0 + 16 * rt + row) * kMT) =
          *reinterpret_cast<const f32x4*>(&sOut[(col * 17 + row) * 4]);
    __syncthreads();
  }
}

// Analysis: grid (m-tile, parity, row group of degrees) x column group.  The
// block of row group 0 also writes the zeros above the triangle of its orders
// and parity.
template <int MODE, int RT>
__global__ void __launch_bounds__(256) small_analysis_kernel(SmallAnaArgs a) {
  constexpr int ESZ = MODE == kFP32 ? 4 : 2;
  const int lane = threadIdx.x & 63, z = threadIdx.x >> 6;
  const int li = lane & 15, kg = lane >> 4;
  const int rg = (int)blockIdx.x % a.rgroups, q = (int)blockIdx.x / a.rgroups % 2;
  const int mb = (int)blockIdx.x / a.rgroups / 2;
  const int T1 = a.T + 1;
  const int m = mb * kMT + z;
  const size_t plane = (size_t)T1 * T1;
  const int f = (int)blockIdx.y * 8 + (li >> 1), part = li & 1;
  if (rg == 0) {  // degrees n < 4 mb + zz of the orders 4 mb + zz, (n - m) mod 2 = q
    const int nmax = min(mb * kMT + kMT - 1, T1);
    for (int e = threadIdx.x; e < nmax * 32; e += 256) {
      const int zz = e & 3, ff = (int)blockIdx.y * 8 + ((e >> 2) & 7), n = e >> 5;
      const int mm = mb * kMT + zz;
      if (n < mm && mm <= a.T && ((mm - n) & 1) == q && ff < a.nfields)
        a.out[(size_t)ff * plane + (size_t)n * T1 + mm] = make_float2(0.f, 0.f);
    }
  }
  const int kq = m <= a.T ? (a.T - m - q) / 2 + (a.T >= m + q ? 1 : 0) : 0;  // rows m + q + 2 r
  const int r0 = rg * RT * 16;
  if (r0 >= kq) return;  // wave-uniform, and no barrier below
  const int KP = a.koff[2 * m + q + 1] - a.koff[2 * m + q];
  const char* tab = static_cast<const char*>(a.table) + (size_t)a.koff[2 * m + q] * a.JHP * ESZ;
  const float* W = a.waist + (size_t)min(2 * f + part, 2 * a.nfields - 1) * a.ldw +
                   (size_t)(mb * 2 + q) * a.JHP * kMT + z;
  f32x4 acc[RT];
  small_contract<MODE, RT>(
      acc, a.JHP / 32, kg, li, a.piece * ESZ, [&](int k) { return W[(size_t)k * kMT]; },
      [](int, float v) { return v; },
      [&](int ch, int rt) {
        return tab + ((size_t)ch * KP + min(r0 + 16 * rt, KP - 16)) * 32 * ESZ;
      });
  if (f >= a.nfields) return;
  float* out = reinterpret_cast<float*>(a.out + (size_t)f * plane) + part;
#pragma unroll
  for (int rt = 0; rt < RT; ++rt)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int row = r0 + 16 * rt + 4 * kg + r, n = m + q + 2 * row;
      if (row >= kq) continue;
      float v = m == 0 && part ? 0.f : acc[rt][r];
      if (a.off00 && n == 0) {  // m = 0 as well
        const float2 d = a.off00[f];
        v += part ? d.y : d.x;
      }
      out[2 * ((size_t)n * T1 + m)] = v;
    }
}

}  // namespace sht

namespace {

template <int MODE, int DIR>
hipError_t launch_mode(const sht::GemmWork& w, int bn, int acc2, dim3 g, hipStream_t s) {
  const dim3 b(256);
  constexpr bool kSplit = MODE != sht::kFP32;
  if (bn == 96) {
    // no split accumulators: 96 columns leave no registers for them
    hipLaunchKernelGGL((sht::legendre_gemm_kernel<MODE, DIR, 96, false>), g, b, 0, s, w);
  } else if (bn == 64) {
    if (kSplit && acc2)
      hipLaunchKernelGGL((sht::legendre_gemm_kernel<MODE, DIR, 64, kSplit>), g, b, 0, s, w);
    else
      hipLaunchKernelGGL((sht::legendre_gemm_kernel<MODE, DIR, 64, false>), g, b, 0, s, w);
  } else {
    if (kSplit && acc2)
      hipLaunchKernelGGL((sht::legendre_gemm_kernel<MODE, DIR, 32, kSplit>), g, b, 0, s, w);
    else
      hipLaunchKernelGGL((sht::legendre_gemm_kernel<MODE, DIR, 32, false>), g, b, 0, s, w);
  }
  return hipGetLastError();
}

template <int DIR>
hipError_t launch_dir(int mode, const sht::GemmWork& w, int bn, int acc2, dim3 g,
                      hipStream_t s) {
  switch (mode) {
    case sht::kFP32: return launch_mode<sht::kFP32, DIR>(w, bn, acc2, g, s);
    case sht::kBF16X3: return launch_mode<sht::kBF16X3, DIR>(w, bn, acc2, g, s);
    case sht::kBF16X6: return launch_mode<sht::kBF16X6, DIR>(w, bn, acc2, g, s);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace

extern "C" hipError_t sht_launch_legendre_gemm(const sht::GemmLaunch* L, hipStream_t s) {
  if (L->nitems <= 0) return hipSuccess;
  if (L->bn != 32 && L->bn != 64 && L->bn != 96) return hipErrorInvalidValue;
  if (L->bn == 96 && L->acc2 && L->mode != sht::kFP32) return hipErrorInvalidValue;
  const sht::GemmWork w{L->panels, L->steps, L->items, L->nitems, L->nsteps};
  const dim3 g(L->grid);
  return L->dir == 0 ? launch_dir<0>(L->mode, w, L->bn, L->acc2, g, s)
                     : launch_dir<1>(L->mode, w, L->bn, L->acc2, g, s);
}

namespace {

// Synthesis row tiles per wavefront: as many as still leave the chip two blocks per CU
// (more tiles per gathered data fragment), at most 4.
int small_row_tiles(int blocks_of_one, int tiles) {
  int rt = 4;
  while (rt > 1 && (rt > tiles || blocks_of_one / rt < 512)) rt /= 2;
  return rt;
}

template <int MODE>
void launch_small_syn(const sht::SmallSynArgs& a, int rt, dim3 g, hipStream_t s) {
  if (rt == 4) hipLaunchKernelGGL((sht::small_synthesis_kernel<MODE, 4>), g, dim3(256), 0, s, a);
  else if (rt == 2) hipLaunchKernelGGL((sht::small_synthesis_kernel<MODE, 2>), g, dim3(256), 0, s, a);
  else hipLaunchKernelGGL((sht::small_synthesis_kernel<MODE, 1>), g, dim3(256), 0, s, a);
}
template <int MODE>
void launch_small_ana(const sht::SmallAnaArgs& a, int rt, dim3 g, hipStream_t s) {
  if (rt == 4) hipLaunchKernelGGL((sht::small_analysis_kernel<MODE, 4>), g, dim3(256), 0, s, a);
  else hipLaunchKernelGGL((sht::small_analysis_kernel<MODE, 2>), g, dim3(256), 0, s, a);
}

}  // namespace

extern "C" hipError_t sht_launch_small_synthesis(const sht::SmallSynArgs* a, int mode, int njobs,
                                                 hipStream_t s) {
  if (a->nfields <= 0) return hipSuccess;
  const int MB = (a->T + sht::kMT) / sht::kMT, tiles = a->JHP / 16, cg = (a->nfields + 7) / 8;
  const int rt = small_row_tiles(MB * 2 * tiles * cg * njobs, tiles);
  sht::SmallSynArgs b = *a;
  b.rgroups = (tiles + rt - 1) / rt;
  const dim3 g((unsigned)(MB * 2 * b.rgroups), (unsigned)cg, (unsigned)njobs);
  switch (mode) {
    case sht::kFP32: launch_small_syn<sht::kFP32>(b, rt, g, s); break;
    case sht::kBF16X3: launch_small_syn<sht::kBF16X3>(b, rt, g, s); break;
    case sht::kBF16X6: launch_small_syn<sht::kBF16X6>(b, rt, g, s); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

extern "C" hipError_t sht_launch_small_analysis(const sht::SmallAnaArgs* a, int mode,
                                                hipStream_t s) {
  if (a->nfields <= 0) return hipSuccess;
  const int MB = (a->T + sht::kMT) / sht::kMT, tiles = (a->T / 2 + 16) / 16, cg = (a->nfields + 7) / 8;
  // Row tiles per wavefront: four share one gathered data fragment where the
  // rows are many or the fields spread the gathers over more lines, else two
  // (more wavefronts).  Two against four, us a call (bf16x6): T127 8 fields
  // 13.2 : 14.2, T191 1 field 12.2 : 13.0, 4 15.4 : 14.5, T255 1 15.4 : 15.8,
  // 4 19.8 : 18.1, T383 1 29.9 : 27.7.
  const int rt = tiles >= 6 && std::min(a->nfields, 8) * tiles * tiles >= 128 ? 4 : 2;
  sht::SmallAnaArgs b = *a;
  b.rgroups = (tiles + rt - 1) / rt;
  const dim3 g((unsigned)(MB * 2 * b.rgroups), (unsigned)cg);
  switch (mode) {
    case sht::kFP32: launch_small_ana<sht::kFP32>(b, rt, g, s); break;
    case sht::kBF16X3: launch_small_ana<sht::kBF16X3>(b, rt, g, s); break;
    case sht::kBF16X6: launch_small_ana<sht::kBF16X6>(b, rt, g, s); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}
