// vh_mm.hip -- matrix products of any size (bf16 and fp32) that the large-tile
// kernels of vh_dense.hip and vh_dense_f32.hip do not fill the chip with, or whose
// rows they cannot load.
//
// C[M][N] = A . B (+ bias[N]); A is [M][K] or, "MN-major", [K][M]; B is [N][K] or
// [K][N].  What bounds these products is not the matrix cores: 16 blocks of 256
// CUs (256 x 784 -> 512 fp32: 43 us on 64 x 128 tiles), or operands whose rows are
// not 16-byte aligned and were gathered element by element (K = 2001: 70 - 95 us a
// product that takes 17 on whole units).  So
//  * tiles are 32 x 32 to 64 x 64 (bf16: to 128 x 128), two to five blocks a CU; the
//    four waves of a block of the smaller ones split K (KS groups of waves, every KS-th
//    stage each, added in group order), and what is still short is split over blocks
//    (fp32 partials, added in split order by mm_reduce_kernel); a cost model of the
//    tiles picks both (mm_plan);
//  * operands whose rows are not whole 16-byte units are first copied to padded
//    rows (mm_pad_kernel: both operands in one launch); the products then copy
//    whole units straight into LDS (vh_tiles.hpp).
// A Linear layer's two gradients go in one launch, the bias gradient as column
// sums of the staged dY tiles.
#include "vh_kernels.hpp"
#include "vh_tiles.hpp"

namespace vh {

namespace {

using namespace tiles;

struct MmArgs {
  const void *a, *b;
  void* c;           // [M][ldc], or fp32 partials [split][M][N]
  const void* bias;  // [N] or nullptr
  void* colsum;      // [N] (element type, one split) or fp32 [split][N], or nullptr: column sums of B
  int M, N, K, lda, ldb, ldc;
  int a_bytes, b_bytes, c_bytes;
  int tiles_m, tiles_n, splits, per;  // stages per split
  int cs_shift;      // column sums: 4 << cs_shift columns per block (ColSum)
};

// One BM x BN tile (logical block lb).  S: NB LDS stages.
template <typename T, int BM, int BN, int WM, int WN, int NB, bool AT, bool BT, bool CS>
__device__ __forceinline__ void mm_tile(const MmArgs& g, const int lb, u32x4g* S) {
  using ST = typename Elem<T>::storage;
  using G = GT<T>;
  using TA = MnTile<T, BM>;
  using TB = MnTile<T, BN>;
  constexpr int ES = G::ES, UE = G::UE, BK = G::BK, FM = WM / 32, FN = WN / 32, NWN = BN / WN;
  constexpr int WPG = (BM / WM) * (BN / WN), KS = 4 / WPG;  // waves per group, groups
  constexpr int AC = BM / 8 / WPG, BC = BN / 8 / WPG, GS = (BM + BN) * 8;  // copies per wave; units per group
  static_assert(WPG * KS == 4 && AC >= 1 && BC >= 1, "four waves");

  const int nt = g.tiles_m * g.tiles_n, z = lb / nt, tl = lb - z * nt;
  // column-major groups of 8 row tiles: a group shares its B panel in L2
  const int grp8 = tl / (8 * g.tiles_n), gm = min(g.tiles_m - grp8 * 8, 8), ing = tl - grp8 * 8 * g.tiles_n;
  const int tm = grp8 * 8 + ing % gm, tn = ing / gm, m0 = tm * BM, n0 = tn * BN;
  const int kb = z * g.per * BK, ke = min(g.K, kb + g.per * BK);
  const int nst = (ke - kb + BK - 1) / BK;

  const int tid = threadIdx.x, lane = tid & 63, row_l = lane & 31, half_l = lane >> 5;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6), grp = wv / WPG, wave = wv % WPG;
  const int wm = (wave / NWN) * WM, wn = (wave % NWN) * WN;

  // copy instruction c = wave + WPG i of an operand: byte offset of this lane's unit
  // in stage 0, and the k (K-major: of the unit; MN-major: row) it stands for
  struct Unit {
    int off, k;
  };
  auto unit = [&](auto MN, auto TILE, int rows, int r0, int ld, int c) {
    using Tl = decltype(TILE);
    Unit u;
    if constexpr (decltype(MN)::value) {
      const int kr = Tl::krow(Tl::RPI * c + lane / Tl::UR);
      const int col = r0 + ((lane % Tl::UR) ^ Tl::swz(kr)) * UE;
      u.k = kr;
      u.off = col < rows ? (kr * ld + col) * ES : kOORg;
    } else {
      const int r = 8 * c + (lane >> 3), ku = (lane & 7) ^ ((r >> 1) & 7);
      u.k = ku * UE;
      u.off = r0 + r < rows ? ((r0 + r) * ld + ku * UE) * ES : kOORg;
    }
    return u;
  };
  Unit ua[AC], ub[BC];
#pragma unroll
  for (int i = 0; i < AC; ++i) ua[i] = unit(std::integral_constant<bool, AT>{}, TA{}, g.M, m0, g.lda, wave + WPG * i);
#pragma unroll
  for (int i = 0; i < BC; ++i) ub[i] = unit(std::integral_constant<bool, BT>{}, TB{}, g.N, n0, g.ldb, wave + WPG * i);
  const __amdgpu_buffer_rsrc_t ar = rsrc_g(g.a, g.a_bytes), br = rsrc_g(g.b, g.b_bytes);
  const int astep = AT ? g.lda * ES : ES, bstep = BT ? g.ldb * ES : ES;  // bytes per k
  auto issue = [&](u32x4g* st, int sk) {
    const int k0 = kb + (sk * KS + grp) * BK;  // this group's stage
    const uint32_t la = lds_byte_addr(st) + grp * GS * 16;
    // k at or past the end of the split: out of every range (sign bit)
    const int ask = (int)((uint32_t)k0 * astep), bsk = (int)((uint32_t)k0 * bstep), left = ke - 1 - k0;
#pragma unroll
    for (int i = 0; i < AC; ++i)
      lds_copy16(ar, (ua[i].off + ask) | ((left - ua[i].k) & kOORg), 0, la + (wave + WPG * i) * 1024);
#pragma unroll
    for (int i = 0; i < BC; ++i)
      lds_copy16(br, (ub[i].off + bsk) | ((left - ub[i].k) & kOORg), 0,
                 la + BM * 128 + (wave + WPG * i) * 1024);
  };

  struct Frags {
    typename G::frag a[FM], b[FN];
  };
  auto read = [&](const u32x4g* st, int kk, Frags& q) {
    const char* at = reinterpret_cast<const char*>(st + grp * GS);
    const char* bt = at + BM * 128;
    if constexpr (AT) {
      read_mn<T, BM, FM>(at, wm, kk, lane, q.a);
    } else {
#pragma unroll
      for (int i = 0; i < FM; ++i) q.a[i] = read_k<T>(at, wm + 32 * i, kk, lane);
    }
    if constexpr (BT) {
      read_mn<T, BN, FN>(bt, wn, kk, lane, q.b);
    } else {
#pragma unroll
      for (int j = 0; j < FN; ++j) q.b[j] = read_k<T>(bt, wn + 32 * j, kk, lane);
    }
  };
  f32x16 acc[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j) acc[i][j] = f32x16{};
  Totals<T, FM, FN> tot;
  tot.init();
  auto mma = [&](const Frags& q) { mma_all<FM, FN>(acc, q.a, q.b); };

  // column sums (B MN-major): the blocks of one column tile share its columns
  ColSum<T, BN, KS> cs;
  if constexpr (CS) cs.init(g.colsum != nullptr, tm, g.cs_shift);

  // the loop of vh_gather.hip: copies of the next NB-1 stages in flight, reads of the
  // next step ahead of the MFMAs of this one
  Frags fa, fb;
  const int ns = (nst + KS - 1) / KS;
#pragma unroll
  for (int i = 0; i < NB - 1; ++i)
    if (i < ns) issue(S + i * KS * GS, i);
  stage_sync<NB, AC + BC>(ns - 1);
  read(S, 0, fa);
  for_stages<NB>(ns, [&](auto BUF, int s) {
    constexpr int B = decltype(BUF)::value;
    const u32x4g* cur = S + B * KS * GS;
    const u32x4g* nxt = S + (B + 1) % NB * KS * GS;
    if (s + NB - 1 < ns) issue(S + (B + NB - 1) % NB * KS * GS, s + NB - 1);
    if constexpr (CS) {
      if (cs.on) cs.stage(reinterpret_cast<const char*>(cur) + BM * 128, GS * 16, s);
    }
#pragma unroll
    for (int kk = 1; kk < 4; kk += 2) {
      read(cur, kk, fb);
      __builtin_amdgcn_sched_barrier(0);
      mma(fa);
      __builtin_amdgcn_sched_barrier(0);
      if (kk + 1 < 4) {
        read(cur, kk + 1, fa);
      } else if (s + 1 < ns) {
        stage_sync<NB, AC + BC>(ns - 2 - s);
        read(nxt, 0, fa);
      }
      __builtin_amdgcn_sched_barrier(0);
      mma(fb);
      __builtin_amdgcn_sched_barrier(0);
    }
    tot.template stage<B>(acc);
  });
  tot.finish(acc);

  float* red = reinterpret_cast<float*>(S);
  if constexpr (CS) {
    if (cs.on)
      cs.finish(red, [&](int col, float t) {
        const int n = n0 + col;
        if (n >= g.N) return;
        if (g.splits > 1)
          reinterpret_cast<float*>(g.colsum)[(size_t)z * g.N + n] = t;
        else
          reinterpret_cast<ST*>(g.colsum)[n] = Elem<T>::from_f32(t);
      });
  }
  if constexpr (KS > 1) {  // the groups' sums, added in group order
    constexpr int TILE = FM * FN * 1024;
    static_assert((KS - 1) * WPG * TILE * 4 <= KS * GS * 16, "group sums exceed a stage");
    __syncthreads();
    if (grp > 0) {
#pragma unroll
      for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j)
#pragma unroll
          for (int v = 0; v < 16; ++v)
            red[((grp - 1) * WPG + wave) * TILE + ((i * FN + j) * 16 + v) * 64 + lane] = acc[i][j][v];
    }
    __syncthreads();
    if (grp > 0) return;
#pragma unroll
    for (int q = 0; q < KS - 1; ++q)
#pragma unroll
      for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j)
#pragma unroll
          for (int v = 0; v < 16; ++v) acc[i][j][v] += red[(q * WPG + wave) * TILE + ((i * FN + j) * 16 + v) * 64 + lane];
  }

  // epilogue: lanes walk columns
  const bool part = g.splits > 1;
  const ST* bias = reinterpret_cast<const ST*>(g.bias);
  const __amdgpu_buffer_rsrc_t cr = rsrc_g(g.c, g.c_bytes);
  const int es = part ? 4 : ES, ld = part ? g.N : g.ldc, zoff = part ? z * g.M * g.N * 4 : 0;
#pragma unroll
  for (int j = 0; j < FN; ++j) {
    const int col = n0 + wn + (BT ? mn_spread<T, FN>(j, row_l) : 32 * j + row_l);
    const float bv = bias && col < g.N ? Elem<T>::to_f32(bias[col]) : 0.f;
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const int e = (v >> 2) * 8 + half_l * 4 + (v & 3);
        const int row = m0 + wm + (AT ? mn_spread<T, FM>(i, e) : 32 * i + e);
        const int o = row < g.M && col < g.N ? zoff + (row * ld + col) * es : kOORg;
        const float r = acc[i][j][v] + bv;
        if (ES == 2 && !part)
          __builtin_amdgcn_raw_buffer_store_b16(__builtin_bit_cast(uint16_t, (__bf16)r), cr, o, 0, 0);
        else
          __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, r), cr, o, 0, 0);
      }
  }
}

template <int BM, int BN, int WM, int WN>
constexpr int mm_stage() {  // units
  return 4 / ((BM / WM) * (BN / WN)) * (BM + BN) * 8;
}

template <typename T, int BM, int BN, int WM, int WN, int NB, bool AT, bool BT>
__global__ __launch_bounds__(256) void mm_kernel(MmArgs g) {
  __shared__ __attribute__((aligned(16))) u32x4g S[NB * mm_stage<BM, BN, WM, WN>()];
  mm_tile<T, BM, BN, WM, WN, NB, AT, BT, AT && BT>(g, xcd_block(gridDim.x), S);
}

// Linear's dX (K-major x K-major) and dW (MN-major x MN-major, with the bias
// gradient) in one launch: blocks 0 .. t0-1 take dX's tiles, the rest dW's.
template <typename T, int BM, int BN, int WM, int WN>
__global__ __launch_bounds__(256) void mm_pair_kernel(MmArgs g0, MmArgs g1) {
  __shared__ __attribute__((aligned(16))) u32x4g S[2 * mm_stage<BM, BN, WM, WN>()];
  const int t0 = g0.tiles_m * g0.tiles_n * g0.splits, h = blockIdx.x;
  if (h < t0)
    mm_tile<T, BM, BN, WM, WN, 2, false, false, false>(g0, xcd_map(h, t0), S);
  else
    mm_tile<T, BM, BN, WM, WN, 2, true, true, true>(g1, xcd_map(h - t0, g1.tiles_m * g1.tiles_n * g1.splits), S);
}

// Split products: C (+ bias) and the column sums from the fp32 partials, in split
// order; blocks b0 .. take a second product's (the pair's dW), ..
struct MmReduce {
  const float *part, *cpart;
  void *c, *colsum;
  const void* bias;
  int M, N, ldc, splits, nb, nbc;  // blocks of C and of the column sums
  FastDiv fN;
};
template <typename T>
__global__ __launch_bounds__(256) void mm_reduce_kernel(MmReduce r0, MmReduce r1) {
  using ST = typename Elem<T>::storage;
  const bool first = (int)blockIdx.x < r0.nb + r0.nbc;
  const MmReduce& r = first ? r0 : r1;
  const int b = (int)blockIdx.x - (first ? 0 : r0.nb + r0.nbc);
  const ST* bias = reinterpret_cast<const ST*>(r.bias);
  if (b < r.nb)
    reduce_splits_block(r.part, r.splits, (long)r.M * r.N,
                        [&](long i, float v) {
                          uint32_t row, col;
                          r.fN.divmod((uint32_t)i, row, col);
                          if (bias) v += Elem<T>::to_f32(bias[col]);
                          reinterpret_cast<ST*>(r.c)[(size_t)row * r.ldc + col] = Elem<T>::from_f32(v);
                        },
                        b, r.nb);
  else
    reduce_splits_block(r.cpart, r.splits, r.N,
                        [&](long i, float v) { reinterpret_cast<ST*>(r.colsum)[i] = Elem<T>::from_f32(v); }, b - r.nb, r.nbc);
}

// Rows of `cols` elements copied to rows of whole 16-byte units (zeros past the
// end): one unit per thread, a wave's loads contiguous but for the row ends.
struct PadSeg {
  const void* src;
  void* dst;
  long total;  // units
  int cols, ld, upr;
  FastDiv fupr;
};
template <typename T>
__global__ __launch_bounds__(256) void mm_pad_kernel(PadSeg p0, PadSeg p1, int b0) {
  using ST = typename Elem<T>::storage;
  constexpr int UE = GT<T>::UE;
  const PadSeg& p = (int)blockIdx.x < b0 ? p0 : p1;
  const long id = (long)((int)blockIdx.x < b0 ? blockIdx.x : blockIdx.x - b0) * 256 + threadIdx.x;
  if (id >= p.total) return;
  uint32_t row, u;
  p.fupr.divmod((uint32_t)id, row, u);
  const ST* s = reinterpret_cast<const ST*>(p.src) + (size_t)row * p.ld + u * UE;
  uint4 q;
  if ((int)(u + 1) * UE <= p.cols) {
    __builtin_memcpy(&q, s, 16);  // one load at the element's alignment
  } else {
    ST v[UE];
#pragma unroll
    for (int j = 0; j < UE; ++j) v[j] = (int)u * UE + j < p.cols ? s[j] : (ST)0;
    __builtin_memcpy(&q, v, 16);
  }
  reinterpret_cast<uint4*>(p.dst)[id] = q;
}

// ---------------------------------------------------------------- host side
size_t align256(size_t b) { return (b + 255) & ~size_t(255); }

// What a tile costs, us: `alone`, a pass of the wave groups over their stages by a
// block that has its CU to itself; `busy`, the same as a share of a CU full of blocks;
// both larger by a fraction where operand rows do not start on 128-byte lines (every
// copy of a row then reads two); `ends`, prologue and epilogue, in passes; `fit`, the
// blocks that fit a CU.  Fitted to 2600 timings of all tiles and splits over 130
// products of 1 .. 8192 rows (K to 65536); the plan it picks takes 1.01 - 1.06 times
// the best one's time in the mean.
struct TileCost {
  int bm, bn, ks, fit;
  float alone, busy, busy_off, ends, alone_off;
};
template <typename T>
constexpr int mm_tiles() {  // fp32 gains nothing above 64 x 64 (4096^3: 978 us, 970 on 64 x 128)
  return GT<T>::ES == 2 ? 5 : 3;
}
template <typename T>
const TileCost* mm_costs(bool at) {
  static constexpr TileCost b16[] = {{64, 64, 1, 5, .25f, .196f, .20f, 2.0f, .25f},
                                     {32, 64, 2, 3, .25f, .232f, .20f, 2.2f, .26f},
                                     {32, 32, 4, 2, .40f, .325f, .11f, 2.0f, .26f},
                                     {64, 128, 1, 3, .27f, .307f, .21f, 2.5f, .29f},
                                     {128, 128, 1, 2, .42f, .471f, 0.f, 5.6f, .24f}};
  // MN-major A and B: bound by their transposing reads
  static constexpr TileCost b16t[] = {{64, 64, 1, 5, .48f, .200f, .30f, 2.0f, .35f},
                                      {32, 64, 2, 3, .40f, .300f, .25f, 2.0f, .30f},
                                      {32, 32, 4, 2, .60f, .480f, .10f, 2.0f, .30f},
                                      {64, 128, 1, 3, .55f, .305f, .25f, 2.7f, .15f},
                                      {128, 128, 1, 2, .74f, .520f, 0.f, 3.3f, .07f}};
  static constexpr TileCost f32[] = {{64, 64, 1, 5, .58f, .512f, .02f, 2.0f, 0.f},
                                     {32, 64, 2, 3, .58f, .585f, .02f, 2.0f, .02f},
                                     {32, 32, 4, 2, .75f, .630f, .05f, 2.5f, .15f}};
  return GT<T>::ES == 4 ? f32 : at ? b16t : b16;
}

constexpr size_t kMostWs = (size_t)1 << 30;  // workspace of a call
constexpr float kSplitUs = 4.f;  // of the reduction's launch

// Tile and K splits of a product, or of a Linear layer's pair in one launch.
struct MmPlan {
  TileCost t;
  int per[2], splits[2];  // stages per split
  float us;
};
template <typename T>
MmPlan mm_plan(const DenseProblem* p, int np) {
  constexpr int BK = GT<T>::BK, ES = GT<T>::ES;
  MmPlan best{};
  best.us = 1e30f;
  long stages[2] = {0, 0}, deepest = 0;
  bool off = false;
  for (int i = 0; i < np; ++i) {
    stages[i] = ((long)p[i].K + BK - 1) / BK;
    deepest = std::max(deepest, stages[i]);
    off = off || (long)p[i].lda * ES % 128 || (long)p[i].ldb * ES % 128;
  }
  const TileCost* costs = mm_costs<T>(p[np - 1].at);
  // (sizes of tiles and groups are powers of two: no divisions without splits, the plan of
  // a small call takes 0.1 us)
  auto consider = [&](const TileCost& t, int s) -> long {
    const long cap = s > 1 ? (deepest + s - 1) / s : deepest;
    // every split computes at least two passes of each wave group: its copies cover
    // nothing otherwise
    if (s > 1 && cap < 2 * t.ks) return 1L << 30;
    const int lm = __builtin_ctz(t.bm), ln = __builtin_ctz(t.bn), lk = __builtin_ctz(t.ks);
    MmPlan m{t, {0, 0}, {1, 1}, 0.f};
    long blocks = 0, longest = 0;
    float work = 0.f;
    for (int i = 0; i < np; ++i) {
      long tiles = (((long)p[i].M + t.bm - 1) >> lm) * (((long)p[i].N + t.bn - 1) >> ln), per = stages[i];
      if (per > cap) {
        const long n = std::min(256L, (per + cap - 1) / cap);
        per = (per + n - 1) / n;
        m.splits[i] = (int)((stages[i] + per - 1) / per);
        if (tiles > 256) return 1L << 30;
        tiles *= m.splits[i];
        // partials: written and read at 6 TB/s
        m.us += (float)m.splits[i] * (float)p[i].M * (float)p[i].N * 1.33e-6f;
      }
      m.per[i] = (int)per;
      const long passes = (per + t.ks - 1) >> lk;
      blocks += tiles;
      longest = std::max(longest, passes);
      work += (float)tiles * ((float)passes + t.ends);
    }
    if (m.splits[0] > 1 || m.splits[1] > 1) m.us += kSplitUs;
    const float alone = t.alone * (off ? 1.f + t.alone_off : 1.f), busy = t.busy * (off ? 1.f + t.busy_off : 1.f);
    const long rounds = (blocks + 255) >> 8;   // blocks on the fullest CU
    const float mean = work / (float)blocks;   // passes of a block
    float deep;                                // a block's share of the CU's time
    if (rounds <= t.fit)
      deep = busy * (float)rounds;
    else if (rounds <= 2 * t.fit)  // what does not fit starts when the first blocks end, all about together
      deep = busy * (float)t.fit + std::max(alone, busy * (float)(rounds - t.fit));
    else
      deep = busy * (float)blocks / 256.f + .5f * alone;
    m.us += std::max(alone * ((float)longest + t.ends), deep * mean);
    if (m.us < best.us) best = m;
    return blocks;
  };
  constexpr int nt = mm_tiles<T>();
  long blocks[nt];
  for (int k = 0; k < nt; ++k) blocks[k] = consider(costs[k], 1);
  // A split pays for its reduction where the grid leaves room (fp32 512 x 512 x 8192: 52
  // -> 43 us at 16 splits, 64 x 2048 x 2048: 14.8 -> 12.5) or one product of a pair has
  // few deep blocks (Linear 16384 x 64 -> 64 backward, one tile of dW: 112 -> 14).
  for (int k = 0; k < 3 && best.us > 2 * kSplitUs; ++k)
    for (int s = 2; s <= 256; s += std::max(1, s / 4))
      if (consider(costs[k], s) > blocks[k] + 2048) break;
  return best;
}

// An operand with its rows as whole 16-byte units: stored rows (K-major: M or N;
// MN-major: K) of `cols` elements.
struct Opnd {
  const void* p;
  int rows, cols, ld, ldp;  // ldp: the padded copy's pitch, 0 if none is needed
  size_t bytes;             // of the copy
};
template <typename T>
Opnd opnd(const void* p, int rows, int cols, int ld) {
  constexpr int UE = GT<T>::UE;
  Opnd o{p, rows, cols, ld, 0, 0};
  if (cols % UE || ld % UE || ((uintptr_t)p & 15)) {
    o.ldp = (cols + UE - 1) / UE * UE;
    o.bytes = align256((size_t)rows * o.ldp * GT<T>::ES);
  }
  return o;
}

// Products that the implicit GEMM (element-wise gathers, no copies) computes sooner:
// an operand's rows need a copy, and
//  * the product is over in less than the copy's launch (us here and there: bf16 30 x 139
//    x 38 8.5 and 10.0; fp32 10 x 55 x 9 8.3 and 9.1; but 298 x 9 x 254 21.7 and 9.1), or
//    K is so short that the copy doubles the traffic (fp32 4766 x 89 x 9: 7.7 and 9.3; 7028 x
//    657 x 4 11.9 and 9.3);
//  * it reads a long operand once, by many blocks or with K split: of few rows (fp32 3 x
//    1274 x 11586 24.7 and 37, 42 x 1817 x 4365 24.3 and 29.1; 62 x 1002 x 945, 16 tiles of a K
//    not split there, 44 and 13), or few columns of an MN-major A (fp32 15665 x 31 x 14088
//    347 and 505).  bf16 gathers of K-major rows are slow (35 x 2764 x 4314 39 and 20), those
//    of an MN-major B ahead at 3 x 1490 x 5800 (15.8 and 24) and 48 x 3511 x 9048 (32 and 38),
//    not at 56 x 10447 x 1455 (31 and 23); of both operands MN-major at 35 x 2764 x 4314 (19.7
//    and 21.6), not at 18 x 220 x 71840 (74 and 32).
template <typename T>
bool mm_generic(const DenseProblem& q, const Opnd& a, const Opnd& b, bool alone) {
  if (!a.ldp && !b.ldp) return false;
  const double mnk = (double)q.M * q.N * q.K;
  constexpr bool b16 = GT<T>::ES == 2;
  if (alone && ((q.K <= (b16 ? 160 : 96) && mnk <= 5e5) || (q.K <= 24 && mnk <= 1.5e7 && !q.at))) return true;
  const bool wide = q.M <= (b16 ? 64 : 96);
  const int len = wide ? q.N : q.M;  // it is read by len / 64 tiles at once, or split
  if ((q.K < 1024 && (b16 || len < 8192)) || (!wide && (q.N > 64 || !q.at))) return false;
  const Opnd& o = wide ? b : a;
  if (!o.ldp || (q.at && (b16 || !wide) && len < (b16 ? 1500 : 1000))) return false;
  const double bytes = (double)o.rows * o.cols * GT<T>::ES;
  if (q.at || !b16) return bytes > (wide && !b16 ? 2e6 : 8e6);
  return q.bt && bytes > (q.M <= 16 ? 14e6 : 40e6);
}

struct MmLayout {
  Opnd a[2], b[2];
  MmArgs g[2];
  TileCost t;
  size_t part[2], cpart[2], copies, bytes;
  float us;
  bool shared;
};

template <typename T>
bool mm_layout(const DenseProblem* p, int np, const void* bias, MmLayout& l) {
  constexpr int ES = GT<T>::ES;
  l.bytes = 0;
  for (int i = 0; i < np; ++i)
    if (std::min({p[i].M, p[i].N, p[i].K}) <= 0 || std::max({p[i].M, p[i].N, p[i].K}) > (1 << 30) ||
        (p[i].at && !p[i].bt))
      return false;
  const MmPlan m = mm_plan<T>(p, np);
  l.t = m.t;
  l.us = m.us;
  long blocks = 0;
  for (int i = 0; i < np; ++i) {
    const DenseProblem& q = p[i];
    l.a[i] = opnd<T>(q.a, q.at ? q.K : q.M, q.at ? q.M : q.K, q.lda);
    l.b[i] = opnd<T>(q.b, q.bt ? q.K : q.N, q.bt ? q.N : q.K, q.ldb);
    if (mm_generic<T>(q, l.a[i], l.b[i], np == 1)) return false;
    MmArgs& g = l.g[i];
    g = MmArgs{};
    g.M = q.M;
    g.N = q.N;
    g.K = q.K;
    g.lda = l.a[i].ldp ? l.a[i].ldp : q.lda;
    g.ldb = l.b[i].ldp ? l.b[i].ldp : q.ldb;
    g.ldc = q.ldc;
    g.c = q.c;
    g.bias = bias;
    g.colsum = q.colsum;
    const long tm = ((long)q.M + m.t.bm - 1) / m.t.bm, tn = ((long)q.N + m.t.bn - 1) / m.t.bn;
    blocks += tm * tn * m.splits[i];
    if (blocks > (1L << 30)) return false;
    g.tiles_m = (int)tm;
    g.tiles_n = (int)tn;
    g.per = m.per[i];
    g.splits = m.splits[i];
    g.cs_shift = colsum_shift(g.tiles_m, l.t.bn);
    // with slack: a stage's addresses run past the last row
    const long ab = ((long)l.a[i].rows + 64) * g.lda * ES, bb = ((long)l.b[i].rows + 64) * g.ldb * ES;
    const long cb = (long)q.M * q.ldc * ES, pb = g.splits > 1 ? (long)g.splits * q.M * q.N * 4 : 0;
    if (std::max({ab, bb, cb, pb, (long)q.M * q.N}) > kMaxBytesG) return false;
    // bytes of the operand as stored: the last row may end before its pitch
    g.a_bytes = (int)(((long)l.a[i].rows - 1) * g.lda * ES + (l.a[i].ldp ? l.a[i].ldp : l.a[i].cols) * ES);
    g.b_bytes = (int)(((long)l.b[i].rows - 1) * g.ldb * ES + (l.b[i].ldp ? l.b[i].ldp : l.b[i].cols) * ES);
    g.c_bytes = (int)(pb ? pb : ((long)q.M - 1) * q.ldc * ES + (long)q.N * ES);
    l.part[i] = l.bytes;
    l.bytes += align256((size_t)pb);
    l.cpart[i] = l.bytes;
    if (pb && q.colsum) l.bytes += align256((size_t)g.splits * q.N * 4);
  }
  // one copy of dY, the rows of dX's A and the k rows of dW's B
  l.shared = np == 2 && l.b[1].p == l.a[0].p && l.b[1].rows == l.a[0].rows && l.b[1].cols == l.a[0].cols;
  l.copies = l.bytes;
  for (int i = 0; i < np; ++i) l.bytes += l.a[i].bytes + (i == 1 && l.shared ? 0 : l.b[i].bytes);
  return l.bytes <= kMostWs;
}

template <typename T, int BM, int BN, int WM, int WN>
void mm_launch(const MmArgs* g, int np, bool at, bool bt, hipStream_t st) {
  const unsigned n = (unsigned)(g[0].tiles_m * g[0].tiles_n * g[0].splits);
  if (np == 2) {
    const unsigned n1 = (unsigned)(g[1].tiles_m * g[1].tiles_n * g[1].splits);
    mm_pair_kernel<T, BM, BN, WM, WN><<<dim3(n + n1), 256, 0, st>>>(g[0], g[1]);
    return;
  }
  // A third stage where the grid leaves room for it, from 12 stages on (bf16 900 x 600
  // x 2000, 10 stages: 8.0 us on two, 8.3 on three; 700 x 3000 x 500: 23.6 and 17.5).
  // MN-major x MN-major tiles are bound by their transposing reads and lose as often
  // as they gain (271 x 2368 x 3200: 24.3 and 26.3; 1400^3: 16.9 and 15.9): two.
  if constexpr (GT<T>::ES == 2) {
    if (!at && g[0].per >= 12 && third_stage(BM, BN, 4 / ((BM / WM) * (BN / WN)), n)) {
      if (bt)
        mm_kernel<T, BM, BN, WM, WN, 3, false, true><<<dim3(n), 256, 0, st>>>(g[0]);
      else
        mm_kernel<T, BM, BN, WM, WN, 3, false, false><<<dim3(n), 256, 0, st>>>(g[0]);
      return;
    }
  }
  if (at && bt)
    mm_kernel<T, BM, BN, WM, WN, 2, true, true><<<dim3(n), 256, 0, st>>>(g[0]);
  else if (bt)
    mm_kernel<T, BM, BN, WM, WN, 2, false, true><<<dim3(n), 256, 0, st>>>(g[0]);
  else
    mm_kernel<T, BM, BN, WM, WN, 2, false, false><<<dim3(n), 256, 0, st>>>(g[0]);
}

template <typename T>
int mm_run_t(const DenseProblem* p, int np, const void* bias, WsGet get, hipStream_t st) {
  MmLayout l;
  if (!mm_layout<T>(p, np, bias, l)) return VH_ERR_UNSUPPORTED;
  void* wsp = nullptr;
  if (l.bytes) {
    const int r = get(st, l.bytes, &wsp);
    if (r != VH_OK) return r;
  }
  char* ws = static_cast<char*>(wsp);
  size_t at = l.copies;
  PadSeg seg[4];
  int ns = 0;
  auto place = [&](const Opnd& o) -> const void* {
    if (!o.ldp) return o.p;
    PadSeg& s = seg[ns++];
    s.src = o.p;
    s.dst = ws + at;
    s.cols = o.cols;
    s.ld = o.ld;
    s.upr = o.ldp / GT<T>::UE;
    s.total = (long)o.rows * s.upr;
    s.fupr = FastDiv((uint32_t)s.upr);
    at += o.bytes;
    return s.dst;
  };
  for (int i = 0; i < np; ++i) {
    l.g[i].a = place(l.a[i]);
    l.g[i].b = i == 1 && l.shared ? l.g[0].a : place(l.b[i]);
  }
  for (int i = 0; i < ns; i += 2) {
    PadSeg none{};
    none.fupr = FastDiv(1);
    const PadSeg& s1 = i + 1 < ns ? seg[i + 1] : none;
    const long b0 = (seg[i].total + 255) / 256, b1 = (s1.total + 255) / 256;
    mm_pad_kernel<T><<<dim3((unsigned)(b0 + b1)), 256, 0, st>>>(seg[i], s1, (int)b0);
    VH_LAUNCH_CHECK();
  }
  MmReduce r[2] = {};
  int nb = 0;
  for (int i = 0; i < np; ++i) {
    MmArgs& g = l.g[i];
    if (g.splits <= 1) continue;
    r[i].part = reinterpret_cast<float*>(ws + l.part[i]);
    r[i].c = g.c;
    r[i].bias = g.bias;
    r[i].M = g.M;
    r[i].N = g.N;
    r[i].ldc = g.ldc;
    r[i].splits = g.splits;
    r[i].nb = reduce_splits_grid((long)g.M * g.N);
    r[i].fN = FastDiv((uint32_t)g.N);
    g.c = ws + l.part[i];
    g.bias = nullptr;
    if (g.colsum) {
      r[i].cpart = reinterpret_cast<float*>(ws + l.cpart[i]);
      r[i].colsum = g.colsum;
      r[i].nbc = reduce_splits_grid(g.N);
      g.colsum = ws + l.cpart[i];
    }
    nb += r[i].nb + r[i].nbc;
  }
  const bool ta = p[0].at, tb = p[0].bt;
  if constexpr (GT<T>::ES == 2) {
    if (l.t.bm == 128) mm_launch<T, 128, 128, 64, 64>(l.g, np, ta, tb, st);
    if (l.t.bm == 64 && l.t.bn == 128) mm_launch<T, 64, 128, 32, 64>(l.g, np, ta, tb, st);
  }
  if (l.t.bm == 64 && l.t.bn == 64) mm_launch<T, 64, 64, 32, 32>(l.g, np, ta, tb, st);
  if (l.t.bm == 32 && l.t.bn == 64) mm_launch<T, 32, 64, 32, 32>(l.g, np, ta, tb, st);
  if (l.t.bm == 32 && l.t.bn == 32) mm_launch<T, 32, 32, 32, 32>(l.g, np, ta, tb, st);
  VH_LAUNCH_CHECK();
  if (nb) {
    mm_reduce_kernel<T><<<dim3((unsigned)nb), 256, 0, st>>>(r[0], r[1]);
    VH_LAUNCH_CHECK();
  }
  return VH_OK;
}

}  // namespace

bool mm_info(int dt, const DenseProblem* p, int np, MmInfo* o) {
  MmLayout l;
  if (!(dt == VH_BF16 ? mm_layout<bf16>(p, np, nullptr, l) : mm_layout<float>(p, np, nullptr, l))) return false;
  *o = MmInfo{l.t.bm, l.t.bn, l.t.fit, {l.g[0].splits, np > 1 ? l.g[1].splits : 0}, {l.g[0].per, np > 1 ? l.g[1].per : 0}, l.bytes, l.us};
  return true;
}

int mm_run(int dt, const DenseProblem* p, int np, const void* bias, WsGet get, hipStream_t st) {
  return dt == VH_BF16 ? mm_run_t<bf16>(p, np, bias, get, st) : mm_run_t<float>(p, np, bias, get, st);
}

}  // namespace vh
