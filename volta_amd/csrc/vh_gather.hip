// vh_gather.hip -- convolutions of any geometry as implicit GEMMs over
// channels-last copies (bf16 and fp32), for gfx950 MFMA.
//
// A convolution pass whose shape fits none of the specialised kernels (odd
// widths, strides, fp32) spends its time on the gather: in NCHW the values an
// MFMA operand needs -- consecutive channels of one position -- lie a plane
// apart, so every 16-byte LDS unit takes 4 or 8 scalar loads with their own
// bounds checks, and the matrix cores wait (measured: 70-90 TFLOP/s bf16, 60-70
// of 157 fp32).  Here one pass over the tensor (gather_prep_kernel) first writes
// it as [N][Hp][Wp][Cp]: channels last, padded to whole 16-byte units, with the
// convolution's zero border in place.  After it
//  * every operand unit is 16 contiguous, aligned bytes: it goes from global
//    memory straight into LDS (buffer_load_dwordx4 ... lds), no registers;
//  * a unit's address is base(position) + offset(tap, channel unit): no bounds
//    checks, whatever the stride and padding.
// The copy costs one read and one write of the tensor; the product reads it once
// per tap (mostly from L2) and row of tiles.
//
// gather_conv_kernel: D[o][position], forward and (one stride phase at a time,
// every phase a stride-1 convolution over its own taps) input gradient; weights
// re-laid out to [m][tap][Cp] by the same prep launch.
// gather_wgrad_kernel: D[o][(tap, c)] summed over positions: both operands are
// rows of positions, so the k index is the slow one of both tiles; bf16
// fragments come from transposing LDS reads (ds_read_b64_tr_b16), fp32 ones from
// 4-byte reads.  Split over positions, fp32 partials added in a fixed order by
// gather_wgrad_reduce_kernel.
#include "vh_kernels.hpp"
#include "vh_tiles.hpp"

namespace vh {

namespace {

using namespace tiles;

constexpr int kMaxPhases = 16;
constexpr int kLaunchPhases = 4;  // stride 2 in one launch, its arguments below 600 bytes

// ---------------------------------------------------------------- preparation
// One tensor copied from [N][C][H][W] to [N][Hp][Wp][Cp] with (padT, padL) zero
// rows and columns before it (rows and columns past Hp / Wp are dropped).
struct PackSeg {
  const void* src;
  void* dst;
  int C, H, W, Cp, Hp, Wp, padT, padL;
  int src_bytes, npos, ncg;  // npos = N*Hp*Wp; channel groups of GROUP channels
  FastDiv fHpWp, fWp, fcg;
};

// The weights [O][C][KH][KW] as rows [phase][m] of 16-byte channel units, padded
// to whole stages with zeros: transposed = 0: m = o, units of channels; 1 (input
// gradient): m = c, units of output channels, taps of the phase in reverse order.
// Order of the product's k index (units): chunks of 8 channel units, in each the
// taps, so that a stage is one tap of one chunk and the R*S stages that read the
// same values of the other operand follow each other (its lines stay in L1 / L2;
// tap-major, 9 passes over all channels, ran at L2-miss rate: 3x3 384->128 @32
// bf16 72 us); the last chunk holds the CU % 8 units left.
struct WeightSeg {
  const void* src;
  void* dst;
  int O, C, KH, KW, transposed, CU;
  int sh, sw, ph, pw;            // input gradient: strides and padding (phase of a tap)
  int nph;
  int units, total;              // copied units of all phases; with the row tails
  FastDiv fRS, fM, fKW;
  // per phase (a * sw + b): dst offset in units, units per row, taps, tap columns; rows < 0: no such phase
  int off[kMaxPhases], row_units[kMaxPhases], taps[kMaxPhases], cols[kMaxPhases];
};

struct PrepArgs {
  PackSeg p[2];
  WeightSeg w;
  int b0, b1, b2;  // blocks of p[0], p[0..1], p[0..1] and w
};

// A wave copies 64 positions x 64 bytes of channels: a lane loads its position's
// channels one by one (64 neighbouring positions per load), then the wave's 16-byte
// units change lanes through LDS so that a store covers 64 contiguous bytes of 16
// positions (stored by their own lanes they would be 64 scattered 16-byte pieces).
// Slot of unit u of position l: u ^ ((l >> 2) & 3), conflict-free both ways.
template <typename T>
__device__ __forceinline__ void pack_block(const PackSeg& s, int blk, uint4* lds) {
  using ST = typename Elem<T>::storage;
  constexpr int ES = GT<T>::ES, UE = GT<T>::UE, GROUP = 64 / ES;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  uint32_t pt, cg;
  s.fcg.divmod((uint32_t)(blk * 4 + wave), pt, cg);
  const int pos = (int)pt * 64 + lane, c0 = (int)cg * GROUP;
  if ((int)pt * 64 >= s.npos) return;
  uint32_t n, hw, h, w;
  s.fHpWp.divmod((uint32_t)min(pos, s.npos - 1), n, hw);
  s.fWp.divmod(hw, h, w);
  const int hi = (int)h - s.padT, wi = (int)w - s.padL, HW = s.H * s.W;
  const bool in = pos < s.npos && (unsigned)hi < (unsigned)s.H && (unsigned)wi < (unsigned)s.W;
  const int voff = in ? ((int)n * s.C * HW + hi * s.W + wi) * ES : kOORg;
  const __amdgpu_buffer_rsrc_t r = rsrc_g(s.src, s.src_bytes);
  ST v[GROUP];
#pragma unroll
  for (int j = 0; j < GROUP; ++j) {
    const int c = c0 + j;
    if constexpr (ES == 2)
      v[j] = c < s.C ? __builtin_amdgcn_raw_buffer_load_b16(r, voff, c * HW * ES, 0) : (ST)0;
    else
      v[j] = c < s.C ? __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, voff, c * HW * ES, 0)) : 0.f;
  }
  uint4* t = lds + wave * 256;
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    uint4 q;
    __builtin_memcpy(&q, v + u * UE, 16);
    t[lane * 4 + (u ^ ((lane >> 2) & 3))] = q;
  }
  __builtin_amdgcn_wave_barrier();  // a wave's own LDS operations complete in order
  ST* d = reinterpret_cast<ST*>(s.dst) + c0 + (lane & 3) * UE;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int l = 16 * i + (lane >> 2), q = (int)pt * 64 + l;
    const uint4 o = t[l * 4 + ((lane & 3) ^ ((l >> 2) & 3))];
    if (q < s.npos && c0 + (lane & 3) * UE < s.Cp) *reinterpret_cast<uint4*>(d + (size_t)q * s.Cp) = o;
  }
}

// One 16-byte unit per thread: (channel unit, m, tap) with the tap fastest, so
// that a wave's loads run along the stored (channel, tap) index.
template <typename T>
__device__ __forceinline__ void weight_block(const WeightSeg& s, int blk) {
  using ST = typename Elem<T>::storage;
  constexpr int UE = GT<T>::UE;
  const int id = blk * 256 + threadIdx.x;
  if (id >= s.total) return;
  uint4* dst = reinterpret_cast<uint4*>(s.dst);
  const int RS = s.KH * s.KW, M = s.transposed ? s.C : s.O, KC = s.transposed ? s.O : s.C;
  if (id >= s.units) {  // the zero tail of row m of a phase
    int t = id - s.units;
    for (int f = 0; f < s.nph; ++f) {
      const int tail = s.row_units[f] - s.taps[f] * s.CU, cnt = tail * M;
      if (s.off[f] < 0) continue;
      if (t < cnt) {
        const int m = t / tail, u = t - m * tail;
        dst[(size_t)s.off[f] + (size_t)m * s.row_units[f] + s.taps[f] * s.CU + u] = make_uint4(0, 0, 0, 0);
        return;
      }
      t -= cnt;
    }
    return;
  }
  uint32_t q, tap, cu, m;
  s.fRS.divmod((uint32_t)id, q, tap);
  s.fM.divmod(q, cu, m);
  const ST* src = reinterpret_cast<const ST*>(s.src);
  ST v[UE];
#pragma unroll
  for (int j = 0; j < UE; ++j) {
    const int kc = (int)cu * UE + j;
    const size_t idx = s.transposed ? ((size_t)kc * s.C + m) * RS + tap : ((size_t)m * s.C + kc) * RS + tap;
    v[j] = kc < KC ? src[idx] : (ST)0;
  }
  int f = 0, t = (int)tap;
  if (s.transposed) {
    uint32_t kh, kw;
    s.fKW.divmod(tap, kh, kw);
    // the phase whose input rows this tap reaches: a = (kh - ph) mod sh
    const int i = (int)kh / s.sh, j = (int)kw / s.sw;
    int a = ((int)kh - s.ph) % s.sh, b = ((int)kw - s.pw) % s.sw;
    a += a < 0 ? s.sh : 0;
    b += b < 0 ? s.sw : 0;
    f = a * s.sw + b;
    if (s.off[f] < 0) return;  // fewer input rows or columns than the stride: no such phase
    t = s.taps[f] - 1 - (i * s.cols[f] + j);
  }
  uint4 o;
  __builtin_memcpy(&o, v, 16);
  const int full = s.CU & ~7, c = (int)cu;
  const int ku = c < full ? (c & ~7) * s.taps[f] + t * 8 + (c & 7) : full * s.taps[f] + t * (s.CU - full) + c - full;
  dst[(size_t)s.off[f] + (size_t)m * s.row_units[f] + ku] = o;
}

template <typename T>
__global__ __launch_bounds__(256) void gather_prep_kernel(PrepArgs a) {
  __shared__ uint4 lds[4 * 256];
  const int b = blockIdx.x;
  if (b < a.b0)
    pack_block<T>(a.p[0], b, lds);
  else if (b < a.b1)
    pack_block<T>(a.p[1], b - a.b0, lds);
  else
    weight_block<T>(a.w, b - a.b1);
}

// ---------------------------------------------------------------- forward, input gradient
// One stride phase (the forward pass is a single one): positions (n, i, j) of an
// Hc x Wc grid, reading x at rows i*sh + r (+ the phase's offset, in off0).
struct ConvPhase {
  int w_off, w_bytes;   // weights of the phase: byte offset, size
  int nst, units, full; // stages, channel units of all taps, those of whole chunks
  int off0;             // byte offset of tap 0 of position (0, 0)
  int N;                // positions
  int sub_a, sub_b;     // output position (osh*i + sub_a, osw*j + sub_b)
  FastDiv fHW, fW, fT, fS;  // by positions per image and row, taps, tap columns
};

struct ConvArgs {
  const char* w;
  const void* x;
  void* y;
  const void* bias;
  const void* mask;
  int M, tiles_m, full, x_bytes, y_bytes;  // full: channel units in whole chunks of 8
  int img, rowb, colb;   // bytes between images, input rows and columns of x
  int sh, sw, act;       // act: 0 none, 1 ReLU, 2 zero where mask <= 0
  int OH, OW, osh, osw;  // output extents and strides
  int nph, tiles;
  FastDiv ftail;         // by the channel units of the last chunk
  ConvPhase ph[kLaunchPhases];
};

// Tile BM x BN, four waves of WM x WN, NB LDS stages of 128 bytes per row: row r
// of 8 units, slot t holds k unit t ^ ((r >> 1) & 7), so that a fragment read (16
// lanes = 16 rows of one unit) is spread over all banks.  Copy instruction c
// brings rows 8c .. 8c+7, a lane's k unit depends on c's parity.
// A tile of fewer than four waves' WM x WN is computed by KS groups of waves that
// take every KS-th stage each (their sums added in group order at the end): for
// grids of few positions, which larger tiles would leave on a part of the CUs.
template <typename T, int BM, int BN, int WM, int WN, int NB>
__global__ __launch_bounds__(256) void gather_conv_kernel(ConvArgs g) {
  using ST = typename Elem<T>::storage;
  using G = GT<T>;
  using Frag = typename G::frag;
  constexpr int ES = G::ES, FM = WM / 32, FN = WN / 32, NWN = BN / WN;
  constexpr int WPG = (BM / WM) * (BN / WN), KS = 4 / WPG;  // waves per group, groups
  constexpr int AC = BM / 8 / WPG, BC = BN / 8 / WPG;       // copy instructions per wave and stage
  static_assert(WPG * KS == 4, "four waves");
  constexpr int STAGE = KS * (BM + BN) * 8;
  __shared__ __attribute__((aligned(16))) u32x4g S[NB * STAGE];

  // consecutive tiles on one XCD (the grid is a multiple of 8): the m-tiles of one
  // position tile share its gathered rows in that L2, and so do its stride phases,
  // whose interleaved stores meet there again
  const int lb = xcd_map(blockIdx.x, gridDim.x);
  if (lb >= g.tiles) return;
  const int tn = lb / (g.tiles_m * g.nph), in = lb - tn * g.tiles_m * g.nph;
  const int f = in / g.tiles_m;
  const ConvPhase p = g.ph[f];
  const int m0 = (in - f * g.tiles_m) * BM, n0 = tn * BN;
  if (n0 >= p.N) return;

  const int tid = threadIdx.x, lane = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6), grp = wv / WPG, wave = wv % WPG;
  const int wm = (wave / NWN) * WM, wn = (wave % NWN) * WN;
  const int l8 = lane >> 3;
  // k unit in copy instruction wave + WPG i: the parity is the wave's, or i's if WPG = 1
  auto unit0 = [&](int i) { return (lane & 7) ^ (((WPG == 1 ? i : wave) & 1) * 4 + (l8 >> 1)); };

  int aoff[AC], boff[BC];
#pragma unroll
  for (int i = 0; i < AC; ++i) aoff[i] = ((m0 + 8 * (wave + WPG * i) + l8) * p.nst * 8 + unit0(i)) * 16;
#pragma unroll
  for (int i = 0; i < BC; ++i) {
    const int pos = n0 + 8 * (wave + WPG * i) + l8;
    uint32_t n, hw, h, w;
    p.fHW.divmod((uint32_t)min(pos, p.N - 1), n, hw);
    p.fW.divmod(hw, h, w);
    boff[i] = pos < p.N ? (int)n * g.img + (int)h * g.sh * g.rowb + (int)w * g.sw * g.colb + p.off0 : kOORg;
  }
  const __amdgpu_buffer_rsrc_t ar = rsrc_g(g.w + p.w_off, p.w_bytes), br = rsrc_g(g.x, g.x_bytes);
  auto issue = [&](u32x4g* st, int sk) {
    const int s = sk * KS + grp;  // this group's stage
    const uint32_t la = lds_byte_addr(st) + grp * (BM + BN) * 128;
    const int ask = s * 128;
#pragma unroll
    for (int i = 0; i < AC; ++i)
      lds_copy16(ar, KS == 1 || s < p.nst ? aoff[i] : kOORg, ask, la + (wave + WPG * i) * 1024);
    // this lane's unit of the stage: its tap and channel unit
    auto tap_off = [&](int ku0) {
      const int ku = s * 8 + ku0;
      uint32_t tap, cu, r, c;
      if (s * 8 < p.full) {  // a whole chunk: the stage is one tap of it
        uint32_t chunk;
        p.fT.divmod((uint32_t)s, chunk, tap);
        cu = chunk * 8 + ku0;
      } else {
        g.ftail.divmod((uint32_t)(ku - p.full), tap, cu);
        cu += g.full;
      }
      p.fS.divmod(tap, r, c);
      // past the last unit: out of every range (sign bit)
      return ((int)r * g.rowb + (int)c * g.colb + (int)cu * 16) | ((p.units - 1 - ku) & kOORg);
    };
    const int off0 = tap_off(unit0(0)), off1 = WPG == 1 ? tap_off(unit0(1)) : off0;
#pragma unroll
    for (int i = 0; i < BC; ++i)
      lds_copy16(br, boff[i] + (i & 1 ? off1 : off0), 0, la + BM * 128 + (wave + WPG * i) * 1024);
  };

  const int row_l = lane & 31, half_l = lane >> 5;
  struct Frags {
    Frag a[FM], b[FN];
  };
  auto read = [&](const u32x4g* st, int kk, Frags& q) {
    const char* at = reinterpret_cast<const char*>(st) + grp * (BM + BN) * 128;
#pragma unroll
    for (int i = 0; i < FM; ++i) q.a[i] = read_k<T>(at, wm + 32 * i, kk, lane);
#pragma unroll
    for (int j = 0; j < FN; ++j) q.b[j] = read_k<T>(at + BM * 128, wn + 32 * j, kk, lane);
  };
  f32x16 acc[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j) acc[i][j] = f32x16{};
  Totals<T, FM, FN> tot;
  tot.init();
  auto mma = [&](const Frags& q) { mma_all<FM, FN>(acc, q.a, q.b); };

  // stage s sits in buffer s % NB; fa holds its first step on entry.  The copies
  // of stage s+NB-1 go into the buffer whose stage s-1 every wave finished reading
  // before the last barrier.  The reads of step k+1 are kept ahead of the
  // MFMAs of step k (left alone the compiler sinks them to their use, and every
  // step waits for LDS).
  Frags fa, fb;
  const int nst = (p.nst + KS - 1) / KS;
#pragma unroll
  for (int i = 0; i < NB - 1; ++i)
    if (i < nst) issue(S + i * STAGE, i);
  stage_sync<NB, AC + BC>(nst - 1);
  read(S, 0, fa);
  for_stages<NB>(nst, [&](auto BUF, int s) {
    constexpr int B = decltype(BUF)::value;
    const u32x4g* cur = S + B * STAGE;
    const u32x4g* nxt = S + (B + 1) % NB * STAGE;
    if (s + NB - 1 < nst) issue(S + (B + NB - 1) % NB * STAGE, s + NB - 1);
#pragma unroll
    for (int kk = 1; kk < 4; kk += 2) {
      read(cur, kk, fb);
      __builtin_amdgcn_sched_barrier(0);
      mma(fa);
      __builtin_amdgcn_sched_barrier(0);
      if (kk + 1 < 4) {
        read(cur, kk + 1, fa);
      } else if (s + 1 < nst) {
        stage_sync<NB, AC + BC>(nst - 2 - s);
        read(nxt, 0, fa);
      }
      __builtin_amdgcn_sched_barrier(0);
      mma(fb);
      __builtin_amdgcn_sched_barrier(0);
    }
    tot.template stage<B>(acc);
  });
  tot.finish(acc);

  if constexpr (KS > 1) {  // the groups' sums, added in group order
    float* red = reinterpret_cast<float*>(S);
    constexpr int TILE = FM * FN * 1024;
    static_assert((KS - 1) * WPG * TILE * 4 <= STAGE * 16, "group sums exceed a stage");
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
          for (int v = 0; v < 16; ++v)
            acc[i][j][v] += red[(q * WPG + wave) * TILE + ((i * FN + j) * 16 + v) * 64 + lane];
  }

  // epilogue: (+ bias), ReLU or mask, one rounding; lanes walk positions
  const __amdgpu_buffer_rsrc_t yr = rsrc_g(g.y, g.y_bytes);
  const int plane = g.OH * g.OW * ES;
  int voff[FN];
#pragma unroll
  for (int j = 0; j < FN; ++j) {
    const int pos = n0 + wn + 32 * j + row_l;
    uint32_t n, hw, h, w;
    p.fHW.divmod((uint32_t)min(pos, p.N - 1), n, hw);
    p.fW.divmod(hw, h, w);
    voff[j] = pos < p.N ? (int)n * g.M * plane + (((int)h * g.osh + p.sub_a) * g.OW + (int)w * g.osw + p.sub_b) * ES +
                              half_l * 4 * plane
                        : kOORg;
  }
  auto row_of = [&](int i, int v) { return m0 + wm + 32 * i + (v >> 2) * 8 + (v & 3); };  // + 4 * half_l
  uint32_t keep[FM][FN];  // bit v: mask > 0; read before the first store
  if (g.act == 2) {
    const __amdgpu_buffer_rsrc_t mr = rsrc_g(g.mask, g.y_bytes);
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int j = 0; j < FN; ++j) {
        keep[i][j] = 0;
#pragma unroll
        for (int v = 0; v < 16; ++v) {
          const int row = row_of(i, v), o = row + 4 * half_l < g.M ? voff[j] : kOORg;
          float m;
          if constexpr (ES == 2)
            m = bf16_to_f32(__builtin_amdgcn_raw_buffer_load_b16(mr, o, row * plane, 0));
          else
            m = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(mr, o, row * plane, 0));
          keep[i][j] |= (m > 0.f ? 1u : 0u) << v;
        }
      }
  }
  const ST* bias = reinterpret_cast<const ST*>(g.bias);
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      const int row = row_of(i, v);
      const bool ok = row + 4 * half_l < g.M;
      const float bv = bias && ok ? Elem<T>::to_f32(bias[row + 4 * half_l]) : 0.f;
#pragma unroll
      for (int j = 0; j < FN; ++j) {
        float r = acc[i][j][v] + bv;
        if (g.act == 1) r = fmaxf(r, 0.f);
        if (g.act == 2 && !((keep[i][j] >> v) & 1)) r = 0.f;
        const int o = ok ? voff[j] : kOORg;
        if constexpr (ES == 2)
          __builtin_amdgcn_raw_buffer_store_b16(Elem<T>::from_f32(r), yr, o, row * plane, 0);
        else
          __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, r), yr, o, row * plane, 0);
      }
    }
}

// ---------------------------------------------------------------- weight gradient
struct WgradArgs {
  const void* dy;  // [N][..][..][Op] (base already at position (0, 0, 0))
  const void* x;   // [N][Hp][Wp][Cp]
  float* part;     // [split][O][RS * Cp]
  float* dbpart;   // [split][O] or nullptr
  int O, NC, K;    // rows, columns (RS * Cp), positions
  int tiles_m, tiles_n, per;  // stages per split
  int add;         // onto the partials of the images before these
  int dy_bytes, x_bytes;
  int dimg, drow, dcol;       // bytes between images, rows and columns of dy
  int ximg, xrow, xcol;       // the same of x, per output row / column (strides applied)
  int trow, tcol;             // bytes between tap rows and columns
  int cs_shift;               // bias gradient: 4 << cs_shift columns of o per block (ColSum)
  FastDiv fPQ, fQ, fCU, fS;
};

template <typename T, int BM, int BN, int WM, int WN>
__global__ __launch_bounds__(256) void gather_wgrad_kernel(WgradArgs g) {
  using G = GT<T>;
  using TA = MnTile<T, BM>;
  using TB = MnTile<T, BN>;
  constexpr int UE = G::UE, BK = G::BK, FM = WM / 32, FN = WN / 32, NWN = BN / WN;
  constexpr int A_UNITS = BK * TA::UR, B_UNITS = BK * TB::UR;
  constexpr int AC = BM / 32, BC = BN / 32;  // copy instructions per wave and stage
  static_assert((BM / WM) * (BN / WN) == 4, "four waves");
  __shared__ __attribute__((aligned(16))) u32x4g S0[A_UNITS + B_UNITS];
  __shared__ __attribute__((aligned(16))) u32x4g S1[A_UNITS + B_UNITS];

  // the tiles of one split share its positions: consecutive on one XCD
  const int nt = g.tiles_m * g.tiles_n;
  const int lb = xcd_map(blockIdx.x, gridDim.x);
  const int z = lb / nt, tl = lb - z * nt;
  const int kb = z * g.per * BK, ke = min(g.K, kb + g.per * BK);
  if (kb >= ke) return;
  const int tm = tl % g.tiles_m, m0 = tm * BM, tn = tl / g.tiles_m, n0 = tn * BN;

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = (wave / NWN) * WM, wn = (wave % NWN) * WN;

  // this lane's k row of copy instruction wave + 4 i, and its column unit (the same
  // for every i: 4 instructions are a multiple of the swizzle's period)
  auto akr = [&](int i) { return TA::krow(TA::RPI * (wave + 4 * i) + lane / TA::UR); };
  auto bkr = [&](int i) { return TB::krow(TB::RPI * (wave + 4 * i) + lane / TB::UR); };
  const int au = m0 / UE + ((lane % TA::UR) ^ TA::swz(akr(0))), bu = n0 / UE + ((lane % TB::UR) ^ TB::swz(bkr(0)));
  const int acol = au * 16 < g.dcol ? au * 16 : kOORg;  // dcol = bytes of a dy position
  uint32_t tap, cu, r, c;
  g.fCU.divmod((uint32_t)bu, tap, cu);
  g.fS.divmod(tap, r, c);
  const int bcol = bu * UE < g.NC ? (int)r * g.trow + (int)c * g.tcol + (int)cu * 16 : kOORg;
  const __amdgpu_buffer_rsrc_t ar = rsrc_g(g.dy, g.dy_bytes), br = rsrc_g(g.x, g.x_bytes);
  auto issue = [&](u32x4g* st, int k0) {
    const uint32_t la = lds_byte_addr(st);
    auto place = [&](int k, int img, int row, int col) {
      uint32_t n, pq, p, q;
      g.fPQ.divmod((uint32_t)min(k, g.K - 1), n, pq);
      g.fQ.divmod(pq, p, q);
      return k < ke ? (int)n * img + (int)p * row + (int)q * col : kOORg;
    };
#pragma unroll
    for (int i = 0; i < AC; ++i)
      lds_copy16(ar, place(k0 + akr(i), g.dimg, g.drow, g.dcol) + acol, 0, la + (wave + 4 * i) * 1024);
#pragma unroll
    for (int i = 0; i < BC; ++i)
      lds_copy16(br, place(k0 + bkr(i), g.ximg, g.xrow, g.xcol) + bcol, 0,
                 la + A_UNITS * 16 + (wave + 4 * i) * 1024);
  };

  const int row_l = lane & 31, half_l = lane >> 5;
  struct Frags {
    typename G::frag a[FM], b[FN];
  };
  auto read = [&](const u32x4g* st, int kk, Frags& q) {
    const char* at = reinterpret_cast<const char*>(st);
    read_mn<T, BM, FM>(at, wm, kk, lane, q.a);
    read_mn<T, BN, FN>(at + A_UNITS * 16, wn, kk, lane, q.b);
  };
  f32x16 acc[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j) acc[i][j] = f32x16{};
  Totals<T, FM, FN> tot;
  tot.init();
  auto mma = [&](const Frags& q) { mma_all<FM, FN>(acc, q.a, q.b); };

  // bias gradient: the blocks of one m-tile share its BM columns of o
  ColSum<T, BM, 1> cs;
  cs.init(g.dbpart != nullptr, tn, g.cs_shift);

  Frags fa, fb;
  const int nst = (ke - kb + BK - 1) / BK;
  issue(S0, kb);
  gather_sync();
  read(S0, 0, fa);
  auto body = [&](auto BUF, int s) {
    constexpr int B = decltype(BUF)::value;
    u32x4g* cur = B == 0 ? S0 : S1;
    u32x4g* nxt = B == 0 ? S1 : S0;
    if (s + 1 < nst) issue(nxt, kb + (s + 1) * BK);
    if (cs.on) cs.stage(reinterpret_cast<const char*>(cur), 0, s);
#pragma unroll
    for (int kk = 1; kk < 4; kk += 2) {
      read(cur, kk, fb);
      __builtin_amdgcn_sched_barrier(0);
      mma(fa);
      __builtin_amdgcn_sched_barrier(0);
      if (kk + 1 < 4) {
        read(cur, kk + 1, fa);
      } else if (s + 1 < nst) {
        gather_sync();
        read(nxt, 0, fa);
      }
      __builtin_amdgcn_sched_barrier(0);
      mma(fb);
      __builtin_amdgcn_sched_barrier(0);
    }
    tot.template stage<B>(acc);
  };
  int s = 0;
  for (; s + 1 < nst; s += 2) {
    body(std::integral_constant<int, 0>{}, s);
    body(std::integral_constant<int, 1>{}, s + 1);
  }
  if (s < nst) body(std::integral_constant<int, 0>{}, s);
  tot.finish(acc);

#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      const int row = m0 + wm + mn_spread<T, FM>(i, (v >> 2) * 8 + half_l * 4 + (v & 3));
      if (row < g.O) {
        float* d = g.part + ((size_t)z * g.O + row) * g.NC;
#pragma unroll
        for (int j = 0; j < FN; ++j) {
          const int col = n0 + wn + mn_spread<T, FN>(j, row_l);
          if (col < g.NC) d[col] = g.add ? d[col] + acc[i][j][v] : acc[i][j][v];
        }
      }
    }
  if (cs.on)
    cs.finish(reinterpret_cast<float*>(S0), [&](int col, float t) {
      float* d = g.dbpart + (size_t)z * g.O + m0 + col;
      if (m0 + col < g.O) *d = g.add ? *d + t : t;
    });
}

// dW[o][c][tap] and db[o] from the splits' partials [split][o][tap][Cp], added in
// a fixed order.  Few splits: block (o, 64 channels), in split order, through LDS
// so that the store is contiguous.
template <typename T>
__global__ __launch_bounds__(256) void gather_wgrad_reduce_kernel(const float* __restrict__ part,
                                                                  const float* __restrict__ dbpart, void* dw, void* db,
                                                                  int O, int C, int Cp, int RS, int splits) {
  using ST = typename Elem<T>::storage;
  extern __shared__ float tile[];  // [RS][65]
  const int o = blockIdx.x, c0 = blockIdx.y * 64, nc = min(64, C - c0);
  const size_t NC = (size_t)RS * Cp, slab = NC * O;
  for (int i = threadIdx.x; i < RS * 64; i += 256) {
    const int rs = i >> 6, cl = i & 63;
    float t = 0.f;
    if (cl < nc) {
      const float* q = part + (size_t)o * NC + (size_t)rs * Cp + c0 + cl;
#pragma unroll 8
      for (int z = 0; z < splits; ++z) t += q[z * slab];
    }
    tile[rs * 65 + cl] = t;
  }
  __syncthreads();
  ST* d = reinterpret_cast<ST*>(dw) + ((size_t)o * C + c0) * RS;
  for (int i = threadIdx.x; i < nc * RS; i += 256) {
    const int cl = i / RS, rs = i - cl * RS;
    d[i] = Elem<T>::from_f32(tile[rs * 65 + cl]);
  }
  if (db && blockIdx.y == 0 && threadIdx.x == 0) {
    float t = 0.f;
    for (int z = 0; z < splits; ++z) t += dbpart[(size_t)z * O + o];
    reinterpret_cast<ST*>(db)[o] = Elem<T>::from_f32(t);
  }
}

// Many splits of few weights: float4 quads of one (o, tap), the splits dealt to
// 2^lg_g groups of threads (blocks nb .. take the bias gradient).
template <typename T>
__global__ __launch_bounds__(256) void gather_wgrad_reduce_vec4_kernel(const float* __restrict__ part,
                                                                       const float* __restrict__ dbpart, void* dw,
                                                                       void* db, int O, int C, FastDiv fCp, FastDiv fRS,
                                                                       int splits, int lg_g, int nb) {
  using ST = typename Elem<T>::storage;
  if ((int)blockIdx.x >= nb) {  // a wave per output, its lanes' sums added in pairs
    const int o = ((int)blockIdx.x - nb) * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    float t = 0.f;
    for (int z = lane; z < splits && o < O; z += 64) t += dbpart[(size_t)z * O + o];
    for (int d = 1; d < 64; d <<= 1) t += __shfl_xor(t, d, 64);
    if (lane == 0 && o < O) reinterpret_cast<ST*>(db)[o] = Elem<T>::from_f32(t);
    return;
  }
  const int RS = (int)fRS.d;
  reduce_splits_vec4_block(
      part, splits, (long)O * RS * fCp.d, lg_g,
      [&](long i, float v) {
        uint32_t ot, c, o, tap;
        fCp.divmod((uint32_t)i, ot, c);
        fRS.divmod(ot, o, tap);
        if ((int)c < C) reinterpret_cast<ST*>(dw)[((size_t)o * C + c) * RS + tap] = Elem<T>::from_f32(v);
      },
      (int)blockIdx.x, nb);
}

// ---------------------------------------------------------------- host side
int round_up(long v, int m) { return (int)((v + m - 1) / m * m); }
size_t align256(size_t b) { return (b + 255) & ~size_t(255); }

template <typename T>
long pack_bytes(int N, int Hp, int Wp, int Cp) {
  return (long)N * Hp * Wp * Cp * GT<T>::ES;
}

template <typename T>
PackSeg pack_seg(const void* src, void* dst, int N, int C, int H, int W, int Cp, int Hp, int Wp, int padT, int padL) {
  constexpr int GROUP = 64 / GT<T>::ES;
  PackSeg s{};
  s.src = src;
  s.dst = dst;
  s.C = C;
  s.H = H;
  s.W = W;
  s.Cp = Cp;
  s.Hp = Hp;
  s.Wp = Wp;
  s.padT = padT;
  s.padL = padL;
  s.src_bytes = (int)((long)N * C * H * W * GT<T>::ES);
  s.npos = N * Hp * Wp;
  s.ncg = (Cp + GROUP - 1) / GROUP;
  s.fHpWp = FastDiv((uint32_t)(Hp * Wp));
  s.fWp = FastDiv((uint32_t)Wp);
  s.fcg = FastDiv((uint32_t)s.ncg);
  return s;
}

int pack_blocks(const PackSeg& s) { return (int)(((long)(s.npos + 63) / 64 * s.ncg + 3) / 4); }

template <typename T>
int launch_prep(PrepArgs& a, int npack, bool weights, hipStream_t st) {
  a.b0 = npack > 0 ? pack_blocks(a.p[0]) : 0;
  a.b1 = a.b0 + (npack > 1 ? pack_blocks(a.p[1]) : 0);
  a.b2 = a.b1 + (weights ? (a.w.total + 255) / 256 : 0);
  gather_prep_kernel<T><<<dim3((unsigned)a.b2), 256, 0, st>>>(a);
  VH_LAUNCH_CHECK();
  return VH_OK;
}

// A pass: its arguments and all its phases.
struct ConvPlan {
  ConvArgs a;
  ConvPhase ph[kMaxPhases];
  int nph;
};

template <typename T, int BM, int BN, int WM, int WN>
int launch_conv_tile(ConvPlan& p, hipStream_t st) {
  constexpr bool b16 = GT<T>::ES == 2, three = b16 && BM * BN < 128 * 128;  // (256 tiles of 128 x 128: never picked)
  ConvArgs& a = p.a;
  a.tiles_m = (a.M + BM - 1) / BM;
  for (int f0 = 0; f0 < p.nph; f0 += kLaunchPhases) {
    a.nph = std::min(kLaunchPhases, p.nph - f0);
    a.tiles = 0;
    for (int f = 0; f < a.nph; ++f) {
      a.ph[f] = p.ph[f0 + f];
      a.tiles = std::max(a.tiles, (a.ph[f].N + BN - 1) / BN);
    }
    a.tiles *= a.tiles_m * a.nph;
    const dim3 grid((unsigned)((a.tiles + 7) / 8 * 8));
    if (three && third_stage(BM, BN, 4 / ((BM / WM) * (BN / WN)), a.tiles))
      gather_conv_kernel<T, BM, BN, WM, WN, three ? 3 : 2><<<grid, 256, 0, st>>>(a);
    else
      gather_conv_kernel<T, BM, BN, WM, WN, 2><<<grid, 256, 0, st>>>(a);
    VH_LAUNCH_CHECK();
  }
  return VH_OK;
}

// The tile, by its cost: rounds of 256 blocks, each of the tile's weight (tile_cost,
// vh_tiles.hpp).  Measured over 31 shapes of each type (3x3, 32 .. 512
// channels, 1.5k .. 1M positions); it finds the fastest or one within 7 %, e.g. us on
// 64 x 64, 32 x 64 (K in two groups of waves), 32 x 32 (four):
//   fp32 217 -> 224 @11 N=8:     47.5  31.6  23.4
//   fp32 128 -> 128 @28x29 N=16: 50.7  56.1  61.9
//   bf16 64 -> 64 @28x29 N=16:   12.6  11.4  14.8
// and on 128 x 128, 64 x 128, 64 x 64:
//   bf16 3x3 s2 64 -> 128 @56:   28.2  32.4  29.7
//   bf16 96 -> 144 @35x27 N=32:  26.0  24.6  29.5
// fp32 gains nothing from tiles above 64 x 64: five blocks a CU cover each other's
// copies and stores.  Deep bf16 products of one or two blocks a CU split K over two
// groups of waves on the 64 x 64 tile (256 @14x15 N=32: 30.6 -> 26.3; shallow ones
// lose to the extra sum, 64 channels 13.8 -> 14.3).
struct ConvTile {
  int bm, bn, ks;
};
template <typename T>
ConvTile pick_conv(const ConvPlan& a) {
  constexpr bool b16 = GT<T>::ES == 2;
  static constexpr int tile[][2] = {{64, 64}, {32, 128}, {32, 64}, {32, 32}, {64, 128}, {128, 128}};
  long n = 0;
  int nst = 0;
  for (int f = 0; f < a.nph; ++f) {
    n += a.ph[f].N;
    nst = std::max(nst, a.ph[f].nst);
  }
  const int M = a.a.M;
  const long g64 = (long)((M + 63) / 64) * ((n + 63) / 64);
  int best = 0;
  float least = 1e30f;
  for (int k = 0; k < (b16 ? 6 : 4); ++k) {
    const long g = (long)((M + tile[k][0] - 1) / tile[k][0]) * ((n + tile[k][1] - 1) / tile[k][1]);
    const float cost = tile_cost<T>(tile[k][0], tile[k][1], nst, g);
    if (cost < least) {
      least = cost;
      best = k;
    }
  }
  const int ks = b16 && best == 0 && g64 <= 512 && nst >= 16 ? 2 : best == 2 ? 2 : best == 3 ? 4 : 1;
  return {tile[best][0], tile[best][1], ks};
}

template <typename T>
int launch_conv(ConvPlan& a, hipStream_t st) {
  const ConvTile t = pick_conv<T>(a);
  if constexpr (GT<T>::ES == 2) {
    if (t.bm == 128) return launch_conv_tile<T, 128, 128, 64, 64>(a, st);
    if (t.bm == 64 && t.bn == 128) return launch_conv_tile<T, 64, 128, 32, 64>(a, st);
    if (t.bm == 64 && t.ks == 2) return launch_conv_tile<T, 64, 64, 64, 32>(a, st);
  }
  if (t.bm == 32 && t.bn == 128) return launch_conv_tile<T, 32, 128, 32, 32>(a, st);
  if (t.bm == 32 && t.bn == 64) return launch_conv_tile<T, 32, 64, 32, 32>(a, st);
  if (t.bm == 32) return launch_conv_tile<T, 32, 32, 32, 32>(a, st);
  return launch_conv_tile<T, 64, 64, 32, 32>(a, st);
}

struct Geo {
  int Cp, Op, Hp, Wp;              // x copy: channels, padded extents
  int Pp, Qp, dT, dL;              // dy copy: padded extents, zero rows and columns before it
};

template <typename T>
bool make_geo(const ConvGeom& g, Geo& o) {
  constexpr int UE = GT<T>::UE;
  o.Cp = round_up(g.C, UE);
  o.Op = round_up(g.O, UE);
  const long Hp = (long)(g.P - 1) * g.sh + g.R, Wp = (long)(g.Q - 1) * g.sw + g.S;
  if (std::max(Hp, Wp) > (1 << 30) || std::max(g.ph, g.pw) > (1 << 30)) return false;
  o.Hp = (int)Hp;
  o.Wp = (int)Wp;
  // dy rows that the input-gradient phases reach: i + (a + ph) / sh - t
  int lo_h = 0, hi_h = g.P - 1, lo_w = 0, hi_w = g.Q - 1;
  auto reach = [](int in, int s, int p, int k, int& lo, int& hi) {
    for (int a = 0; a < s && a < in; ++a) {
      const int k0 = (a + p) % s, taps = k0 < k ? (k - k0 + s - 1) / s : 0;
      if (!taps) continue;
      const int off = (a + p - k0) / s, n = (in - a + s - 1) / s;
      lo = std::min(lo, off - (taps - 1));
      hi = std::max(hi, off + n - 1);
    }
  };
  reach(g.H, g.sh, g.ph, g.R, lo_h, hi_h);
  reach(g.W, g.sw, g.pw, g.S, lo_w, hi_w);
  o.dT = -lo_h;
  o.dL = -lo_w;
  o.Pp = hi_h - lo_h + 1;
  o.Qp = hi_w - lo_w + 1;
  const long ES = GT<T>::ES;
  for (long b : {(long)g.N * g.C * g.H * g.W * ES, (long)g.N * g.O * g.P * g.Q * ES, (long)g.N * o.Hp * o.Wp * o.Cp * ES,
                 (long)g.N * o.Pp * o.Qp * o.Op * ES, (long)(g.O + 128) * (g.R * g.S + 1) * (o.Cp + 64) * ES,
                 (long)(g.C + 128) * (g.R * g.S + 1) * (o.Op + 64) * ES})
    if (b > kMaxBytesG) return false;
  return true;
}

// Phases of the input gradient with taps, in (a, b) order.
struct DPhase {
  int a, b, Hc, Wc, Rc, Sc, offa, offb;
};
int dgrad_phase_list(const ConvGeom& g, DPhase* ph) {
  int n = 0;
  for (int a = 0; a < g.sh; ++a)
    for (int b = 0; b < g.sw; ++b) {
      DPhase& f = ph[n++];
      f.a = a;
      f.b = b;
      f.Hc = a < g.H ? (g.H - a + g.sh - 1) / g.sh : 0;
      f.Wc = b < g.W ? (g.W - b + g.sw - 1) / g.sw : 0;
      const int kh0 = (a + g.ph) % g.sh, kw0 = (b + g.pw) % g.sw;
      f.Rc = kh0 < g.R ? (g.R - kh0 + g.sh - 1) / g.sh : 0;
      f.Sc = kw0 < g.S ? (g.S - kw0 + g.sw - 1) / g.sw : 0;
      f.offa = (a + g.ph - kh0) / g.sh;
      f.offb = (b + g.pw - kw0) / g.sw;
    }
  return n;
}

struct WgradPlan {
  int splits, per;
};

// 64 x 64 tiles, positions split for about four blocks a CU (measured on 13 shapes
// of each type against 64 x 128, 128 x 64 and 128 x 128 tiles at one to four blocks
// a CU: best or within 3 % on all; on few weights the larger tiles' zero padding
// and partials cost up to 2x).  A split costs a write and a read of its partial
// tile: at least 4 stages each, 8 once every CU has a block (217 -> 224 channels at
// 8 x 11 x 11 positions, fp32: 32.2 -> 25 us).
template <typename T>
WgradPlan wgrad_plan(const ConvGeom& g, const Geo& o) {
  constexpr int BK = GT<T>::BK;
  WgradPlan p;
  const long tiles = (long)((g.O + 63) / 64) * ((g.R * g.S * o.Cp + 63) / 64);
  const long stages = ((long)g.N * g.P * g.Q + BK - 1) / BK;
  long want = std::min(std::max<long>(1, 1024 / tiles), std::max<long>(1, stages / 4));
  if (tiles * want > 256) want = std::max<long>((256 + tiles - 1) / tiles, std::min(want, stages / 8));
  p.per = (int)((stages + want - 1) / want);
  p.splits = (int)((stages + p.per - 1) / p.per);
  return p;
}

// Workspace of a call: the copies of x and dy, the weights, the partials.
struct Layout {
  size_t x = 0, dy = 0, w = 0, part = 0, bytes = 0;
};  // for the images of one chunk

template <typename T>
bool make_layout(const GatherCall& c, const Geo& o, const WgradPlan& wg, Layout& l) {
  const ConvGeom& g = c.g;
  constexpr int UE = GT<T>::UE;
  auto take = [&](size_t b) {
    const size_t at = l.bytes;
    l.bytes += align256(b);
    return at;
  };
  if (c.y || c.dw) l.x = take((size_t)pack_bytes<T>(g.N, o.Hp, o.Wp, o.Cp));
  if (c.dx) l.dy = take((size_t)pack_bytes<T>(g.N, o.Pp, o.Qp, o.Op));
  else if (c.dw) l.dy = take((size_t)pack_bytes<T>(g.N, g.P, g.Q, o.Op));
  if (c.y) l.w = take((size_t)g.O * ((g.R * g.S * o.Cp / UE + 7) / 8) * 128);
  if (c.dx) {
    if (c.y || g.sh * g.sw > kMaxPhases) return false;
    DPhase ph[kMaxPhases];
    const int n = dgrad_phase_list(g, ph);
    size_t wu = 1;
    for (int f = 0; f < n; ++f) wu += (size_t)g.C * ((ph[f].Rc * ph[f].Sc * (o.Op / UE) + 7) / 8) * 8;
    l.w = take(wu * 16);
  }
  if (c.dw) l.part = take((size_t)wg.splits * g.O * (g.R * g.S * o.Cp + 1) * sizeof(float));
  return true;
}

template <typename T>
void conv_args(ConvPlan& plan, WeightSeg& s, const GatherCall& c, const Geo& o, char* ws, const Layout& l) {
  constexpr int ES = GT<T>::ES, UE = GT<T>::UE;
  const ConvGeom& g = c.g;
  ConvArgs& a = plan.a;
  const int RS = g.R * g.S;
  s.src = c.w;
  s.dst = ws + l.w;
  s.O = g.O;
  s.C = g.C;
  s.KH = g.R;
  s.KW = g.S;
  s.fRS = FastDiv((uint32_t)RS);
  s.fKW = FastDiv((uint32_t)g.S);
  a.w = ws + l.w;
  a.bias = c.bias;
  if (c.y) {
    const int CU = o.Cp / UE, units = RS * CU, nst = (units + 7) / 8;
    s.CU = CU;
    s.sh = s.sw = s.nph = 1;
    s.units = g.O * units;
    s.total = g.O * nst * 8;
    s.row_units[0] = nst * 8;
    s.taps[0] = RS;
    s.cols[0] = g.S;
    s.fM = FastDiv((uint32_t)g.O);
    a.x = ws + l.x;
    a.y = c.y;
    a.M = g.O;
    a.full = CU & ~7;
    a.x_bytes = (int)pack_bytes<T>(g.N, o.Hp, o.Wp, o.Cp);
    a.y_bytes = (int)((long)g.N * g.O * g.P * g.Q * ES);
    a.colb = o.Cp * ES;
    a.rowb = o.Wp * a.colb;
    a.img = o.Hp * a.rowb;
    a.sh = g.sh;
    a.sw = g.sw;
    a.act = c.act;
    a.OH = g.P;
    a.OW = g.Q;
    a.osh = a.osw = 1;
    plan.nph = 1;
    a.ftail = FastDiv((uint32_t)std::max(1, CU & 7));
    ConvPhase& p = plan.ph[0];
    p.w_bytes = g.O * nst * 128;
    p.nst = nst;
    p.units = units;
    p.full = RS * a.full;
    p.fT = FastDiv((uint32_t)RS);
    p.N = g.N * g.P * g.Q;
    p.fHW = FastDiv((uint32_t)(g.P * g.Q));
    p.fW = FastDiv((uint32_t)g.Q);
    p.fS = FastDiv((uint32_t)g.S);
    return;
  }
  const int CU = o.Op / UE;
  DPhase ph[kMaxPhases];
  const int n = dgrad_phase_list(g, ph);
  s.transposed = 1;
  s.CU = CU;
  s.sh = g.sh;
  s.sw = g.sw;
  s.ph = g.ph;
  s.pw = g.pw;
  s.nph = n;
  s.units = g.C * RS * CU;
  s.fM = FastDiv((uint32_t)g.C);
  a.x = ws + l.dy;
  a.y = c.dx;
  a.mask = c.mask;
  a.act = c.mask ? 2 : 0;
  a.M = g.C;
  a.full = CU & ~7;
  a.x_bytes = (int)pack_bytes<T>(g.N, o.Pp, o.Qp, o.Op);
  a.y_bytes = (int)((long)g.N * g.C * g.H * g.W * ES);
  a.colb = o.Op * ES;
  a.rowb = o.Qp * a.colb;
  a.img = o.Pp * a.rowb;
  a.sh = a.sw = 1;
  a.OH = g.H;
  a.OW = g.W;
  a.osh = g.sh;
  a.osw = g.sw;
  a.ftail = FastDiv((uint32_t)std::max(1, CU & 7));
  int off = 0, tails = 0;
  for (int f = 0; f < n; ++f) {
    const DPhase& q = ph[f];
    const int taps = q.Rc * q.Sc, units = taps * CU, nst = (units + 7) / 8;
    const bool live = q.Hc > 0 && q.Wc > 0;
    s.off[f] = live ? off : -1;
    s.row_units[f] = nst * 8;
    s.taps[f] = taps;
    s.cols[f] = std::max(1, q.Sc);
    if (!live) continue;
    tails += g.C * (nst * 8 - units);
    ConvPhase& p = plan.ph[plan.nph++];
    p.w_off = off * 16;
    p.w_bytes = g.C * nst * 128;
    p.nst = nst;
    p.units = units;
    p.full = taps * a.full;
    p.fT = FastDiv((uint32_t)std::max(1, taps));
    p.off0 = (q.offa - (q.Rc - 1) + o.dT) * a.rowb + (q.offb - (q.Sc - 1) + o.dL) * a.colb;
    p.N = g.N * q.Hc * q.Wc;
    p.sub_a = q.a;
    p.sub_b = q.b;
    p.fHW = FastDiv((uint32_t)(q.Hc * q.Wc));
    p.fW = FastDiv((uint32_t)q.Wc);
    p.fS = FastDiv((uint32_t)std::max(1, q.Sc));
    off += g.C * nst * 8;
  }
  s.total = s.units + tails;
}

// The partials of one chunk's images (the first: add false), and after the last chunk
// their sums.
template <typename T>
int run_wgrad(const GatherCall& c, const Geo& o, const WgradPlan& p, char* ws, const Layout& l, bool add, bool last,
              hipStream_t st) {
  constexpr int ES = GT<T>::ES, UE = GT<T>::UE;
  const ConvGeom& g = c.g;
  // the copy of dy has the input gradient's border when both are computed
  const int Pd = c.dx ? o.Pp : g.P, Qd = c.dx ? o.Qp : g.Q, dT = c.dx ? o.dT : 0, dL = c.dx ? o.dL : 0;
  WgradArgs a{};
  a.dcol = o.Op * ES;
  a.drow = Qd * a.dcol;
  a.dimg = Pd * a.drow;
  const long skip = (long)dT * a.drow + (long)dL * a.dcol;
  a.dy = ws + l.dy + skip;
  a.dy_bytes = (int)(pack_bytes<T>(g.N, Pd, Qd, o.Op) - skip);
  a.x = ws + l.x;
  a.x_bytes = (int)pack_bytes<T>(g.N, o.Hp, o.Wp, o.Cp);
  a.O = g.O;
  a.NC = g.R * g.S * o.Cp;
  a.K = g.N * g.P * g.Q;
  a.part = reinterpret_cast<float*>(ws + l.part);
  a.dbpart = c.db ? a.part + (size_t)p.splits * g.O * a.NC : nullptr;
  a.tiles_m = (g.O + 63) / 64;
  a.tiles_n = (a.NC + 63) / 64;
  a.per = p.per;
  a.add = add;
  a.tcol = o.Cp * ES;
  a.trow = o.Wp * a.tcol;
  a.xcol = g.sw * a.tcol;
  a.xrow = g.sh * a.trow;
  a.ximg = o.Hp * a.trow;
  a.cs_shift = colsum_shift(a.tiles_n, 64);
  a.fPQ = FastDiv((uint32_t)(g.P * g.Q));
  a.fQ = FastDiv((uint32_t)g.Q);
  a.fCU = FastDiv((uint32_t)(o.Cp / UE));
  a.fS = FastDiv((uint32_t)g.S);
  const dim3 grid((unsigned)(a.tiles_m * a.tiles_n * p.splits));
  gather_wgrad_kernel<T, 64, 64, 32, 32><<<grid, 256, 0, st>>>(a);
  VH_LAUNCH_CHECK();
  if (!last) return VH_OK;
  const int RS = g.R * g.S;
  if (p.splits > 8) {
    const int lg = reduce_vec4_lg_groups(p.splits), nb = reduce_vec4_grid((long)g.O * a.NC, lg);
    const int ndb = c.db ? (g.O + 3) / 4 : 0;
    gather_wgrad_reduce_vec4_kernel<T><<<dim3((unsigned)(nb + ndb)), 256, 0, st>>>(
        a.part, a.dbpart, c.dw, c.db, g.O, g.C, FastDiv((uint32_t)o.Cp), FastDiv((uint32_t)RS), p.splits, lg, nb);
  } else {
    gather_wgrad_reduce_kernel<T><<<dim3((unsigned)g.O, (unsigned)((g.C + 63) / 64)), 256, (size_t)RS * 65 * sizeof(float),
                                    st>>>(a.part, a.dbpart, c.dw, c.db, g.O, g.C, o.Cp, RS, p.splits);
  }
  VH_LAUNCH_CHECK();
  return VH_OK;
}

// A call's workspace is bounded, so that no stream holds copies of whole large tensors,
// by what the allocation-free entry point has (it then runs the same kernels).  More
// images are taken in equal chunks, each with its own copies; the partials of the
// weight gradient add up over them.  Eight chunks of 64 MiB had cost a 1x1 128 -> 256 @64
// N=64 fp32 backward 730 us where two take 500.
struct CallPlan {
  Geo o;
  Layout l;
  WgradPlan wg;
  int images;  // per chunk
};

template <typename T>
bool plan_call(const GatherCall& c, CallPlan& p) {
  // more than 64 taps: beyond the reduction's LDS tile
  if (c.g.N <= 0 || c.g.R * c.g.S > 64 || !make_geo<T>(c.g, p.o)) return false;
  GatherCall part = c;
  auto fits = [&](int images) {
    part.g.N = p.images = images;
    p.l = Layout{};
    p.wg = wgrad_plan<T>(part.g, p.o);
    return make_layout<T>(part, p.o, p.wg, p.l) && p.l.bytes <= kGatherMostWs;
  };
  if (fits(c.g.N)) return true;
  if (!fits(1)) return false;
  int lo = 1, hi = c.g.N;  // lo fits, hi does not
  while (hi - lo > 1) {
    const int mid = lo + (hi - lo) / 2;
    (fits(mid) ? lo : hi) = mid;
  }
  const int chunks = (c.g.N + lo - 1) / lo;
  return fits((c.g.N + chunks - 1) / chunks);
}

template <typename T>
size_t call_ws(const GatherCall& c) {
  CallPlan p;
  return plan_call<T>(c, p) ? p.l.bytes : 0;
}

template <typename T>
int run_call(const GatherCall& c, char* ws, hipStream_t st) {
  CallPlan cp;
  if (!plan_call<T>(c, cp)) return VH_ERR_UNSUPPORTED;
  const Geo& o = cp.o;
  const Layout& l = cp.l;
  const size_t in = (size_t)c.g.C * c.g.H * c.g.W * GT<T>::ES, out = (size_t)c.g.O * c.g.P * c.g.Q * GT<T>::ES;
  auto image = [](const void* p, size_t off) { return p ? static_cast<const char*>(p) + off : nullptr; };
  for (int n0 = 0; n0 < c.g.N; n0 += cp.images) {
    GatherCall d = c;
    d.g.N = std::min(cp.images, c.g.N - n0);
    d.x = image(c.x, n0 * in);
    d.mask = image(c.mask, n0 * in);
    d.dx = const_cast<char*>(image(c.dx, n0 * in));
    d.dy = image(c.dy, n0 * out);
    d.y = const_cast<char*>(image(c.y, n0 * out));
    const ConvGeom& g = d.g;
    PrepArgs pa{};
    ConvPlan a{};
    int np = 0;
    if (d.y || d.dw) pa.p[np++] = pack_seg<T>(d.x, ws + l.x, g.N, g.C, g.H, g.W, o.Cp, o.Hp, o.Wp, g.ph, g.pw);
    if (d.dx)
      pa.p[np++] = pack_seg<T>(d.dy, ws + l.dy, g.N, g.O, g.P, g.Q, o.Op, o.Pp, o.Qp, o.dT, o.dL);
    else if (d.dw)
      pa.p[np++] = pack_seg<T>(d.dy, ws + l.dy, g.N, g.O, g.P, g.Q, o.Op, g.P, g.Q, 0, 0);
    const bool conv = d.y || d.dx;
    if (conv) conv_args<T>(a, pa.w, d, o, ws, l);
    int r = launch_prep<T>(pa, np, conv && n0 == 0, st);
    if (r == VH_OK && conv) r = launch_conv<T>(a, st);
    if (r == VH_OK && d.dw) r = run_wgrad<T>(d, o, cp.wg, ws, l, n0 > 0, n0 + cp.images >= c.g.N, st);
    if (r != VH_OK) return r;
  }
  return VH_OK;
}

// The plan of a call and, of its first chunk, the farthest bytes that the kernels
// address: every one within its buffer.
template <typename T>
bool call_info(const GatherCall& c, GatherInfo& o) {
  constexpr int UE = GT<T>::UE;
  CallPlan cp;
  if (!plan_call<T>(c, cp)) return false;
  GatherCall d = c;
  d.g.N = cp.images;
  PrepArgs pa{};
  ConvPlan a{};
  o = GatherInfo{cp.images, 0, 0, 0, cp.wg.splits, cp.wg.per, cp.l.bytes, true};
  if (c.dw) {
    const long stages = ((long)cp.images * c.g.P * c.g.Q + GT<T>::BK - 1) / GT<T>::BK;
    o.ok = (long)cp.wg.splits * cp.wg.per >= stages && (long)(cp.wg.splits - 1) * cp.wg.per < stages;
  }
  if (!c.y && !c.dx) return true;
  conv_args<T>(a, pa.w, d, cp.o, reinterpret_cast<char*>(256), cp.l);  // (nothing is read)
  const ConvTile t = pick_conv<T>(a);
  o.bm = t.bm;
  o.bn = t.bn;
  o.ks = t.ks;
  const long planes = (long)a.a.OH * a.a.OW * GT<T>::ES;
  for (int f = 0; f < a.nph; ++f) {
    const ConvPhase& p = a.ph[f];
    const long hw = p.fHW.d, wc = p.fW.d, hc = hw / wc, images = p.N / hw, taps = p.fT.d, tc = p.fS.d, tr = taps / tc;
    const long in = (images - 1) * a.a.img + (hc - 1) * a.a.sh * a.a.rowb + (wc - 1) * a.a.sw * a.a.colb + p.off0;
    const long units = (c.y ? cp.o.Cp : cp.o.Op) / UE;
    const long tap = (tr - 1) * a.a.rowb + (tc - 1) * a.a.colb + units * 16;
    const long out = ((images - 1) * a.a.M + a.a.M - 1) * planes +
                     (((hc - 1) * a.a.osh + p.sub_a) * a.a.OW + (wc - 1) * a.a.osw + p.sub_b + 1) * GT<T>::ES;
    const bool live = p.nst > 0;
    o.ok = o.ok && (!live || (p.off0 >= 0 && in + tap <= a.a.x_bytes)) && out <= a.a.y_bytes &&
           (long)a.a.M * p.nst * 128 == p.w_bytes && (long)p.w_off + p.w_bytes <= (long)(cp.l.bytes - cp.l.w) &&
           p.units <= p.nst * 8;
  }
  return true;
}

}  // namespace

size_t gather_ws(int dt, const GatherCall& c) { return dt == VH_BF16 ? call_ws<bf16>(c) : call_ws<float>(c); }

bool gather_info(int dt, const GatherCall& c, GatherInfo* o) {
  return dt == VH_BF16 ? call_info<bf16>(c, *o) : call_info<float>(c, *o);
}

int gather_run(int dt, const GatherCall& c, void* ws, hipStream_t st) {
  return dt == VH_BF16 ? run_call<bf16>(c, static_cast<char*>(ws), st) : run_call<float>(c, static_cast<char*>(ws), st);
}

}  // namespace vh
