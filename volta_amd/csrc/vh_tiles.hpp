// vh_tiles.hpp -- operand tiles of the direct-to-LDS products (vh_gather.hip,
// vh_mm.hip) on gfx950 MFMA: their layouts in LDS and the fragment reads.
//
// A stage holds 128 bytes of k per row of the product (64 k bf16, 32 fp32) of both
// operands, copied by buffer_load_dwordx4 ... lds: the 64 16-byte units of a copy
// instruction land contiguously, so a layout is set by which unit each lane fetches.
//  * K-major tile (R rows x 8 units): slot t of row r holds k unit t ^ ((r >> 1) & 7).
//  * MN-major tile (k rows of R columns, UR units each): slot t of k row kr holds
//    unit t ^ swz(kr).
// A step is 32 bytes of k.  K-major: the lanes of half h (lane / 32) take unit
// 2 kk + h of their row in one 16-byte read -- 8 bf16, or 4 fp32 for four MFMAs of
// 2 k.  MN-major tiles give the same k to the same half.
#pragma once
#include <type_traits>

#include "vh_common.hpp"

namespace vh {

namespace tiles {

typedef unsigned int u32x4g __attribute__((ext_vector_type(4)));
typedef unsigned int u32x2g __attribute__((ext_vector_type(2)));

constexpr int kOORg = (int)0x80000000u;  // buffer offset past every range: loads 0, stores dropped
constexpr long kMaxBytesG = (1L << 31) - 4096;  // tensors are addressed with 32-bit byte offsets

template <typename T>
struct GT {
  static constexpr int ES = sizeof(typename Elem<T>::storage);
  static constexpr int UE = 16 / ES;   // elements per 16-byte unit
  static constexpr int BK = 128 / ES;  // k per stage: 8 units per K-major row
  using frag = std::conditional_t<ES == 2, bf16x8, f32x4>;
};

__device__ __forceinline__ __amdgpu_buffer_rsrc_t rsrc_g(const void* p, int bytes) {
  return __builtin_amdgcn_make_buffer_rsrc((void*)p, (short)0, bytes, 0x00020000);
}

// s_waitcnt vmcnt(0) lgkmcnt(0), then the block barrier
__device__ __forceinline__ void gather_sync() {
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// The same once the oldest stage in flight has landed: NB buffers, COPIES copy
// instructions per wave and stage, `later` stages of the product after that one (the
// last ones are waited for together).
template <int NB, int COPIES>
__device__ __forceinline__ void stage_sync(int later) {
  if (NB > 2 && later >= NB - 2)
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"((NB - 2) * COPIES) : "memory");
  else
    gather_sync();
}

// body(buffer, stage) for stages 0 .. ns-1, the buffers in turn and known to the compiler
template <int NB, typename F>
__device__ __forceinline__ void for_stages(int ns, F body) {
  static_assert(NB == 2 || NB == 3, "buffers");
  int s = 0;
  for (; s + NB - 1 < ns; s += NB) {
    body(std::integral_constant<int, 0>{}, s);
    body(std::integral_constant<int, 1>{}, s + 1);
    if constexpr (NB > 2) body(std::integral_constant<int, 2>{}, s + 2);
  }
  if (s < ns) body(std::integral_constant<int, 0>{}, s);
  if constexpr (NB > 2)
    if (s + 1 < ns) body(std::integral_constant<int, 1>{}, s + 1);
}

// all MFMAs of one fragment step: independent accumulators back to back
template <int FM, int FN>
__device__ __forceinline__ void mma_all(f32x16 (&c)[FM][FN], const bf16x8 (&a)[FM], const bf16x8 (&b)[FN]) {
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j) c[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[i], b[j], c[i][j], 0, 0, 0);
}
template <int FM, int FN>
__device__ __forceinline__ void mma_all(f32x16 (&c)[FM][FN], const f32x4 (&a)[FM], const f32x4 (&b)[FN]) {
#pragma unroll
  for (int t = 0; t < 4; ++t)
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int j = 0; j < FN; ++j) c[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[i][t], b[j][t], c[i][j], 0, 0, 0);
}

// fp32 sums in two levels: an accumulator takes the products of 64 k (two stages),
// then goes into the total and starts again.  The error of a sum grows with the root
// of the additions in a row: one accumulator over all of K was up to 3 times further
// off 64 bits (512 channels 3x3 @7: 5.7e-7; 32768 positions: 1.1e-6) than sums of a
// few hundred; so it is 1.7e-7.  Always after the second buffer, so that the zeros are
// the compiler's and no registers (at the fourth stage, by a test of s: 2.1e-7, 8 - 15 %
// slower): 2048^3 forward and gradients 386 -> 399 us.  bf16 results are rounded at
// 2^-9: one level.
template <typename T, int FM, int FN>
struct Totals {
  static constexpr bool two = GT<T>::ES == 4;
  f32x16 t[two ? FM : 1][two ? FN : 1];
  __device__ __forceinline__ void init() {
    if constexpr (two)
#pragma unroll
      for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) t[i][j] = f32x16{};
  }
  // after the stage in buffer B of two
  template <int B>
  __device__ __forceinline__ void stage(f32x16 (&acc)[FM][FN]) {
    if constexpr (two && B == 1)
#pragma unroll
      for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) {
          t[i][j] += acc[i][j];
          acc[i][j] = f32x16{};
        }
  }
  __device__ __forceinline__ void finish(f32x16 (&acc)[FM][FN]) const {
    if constexpr (two)
#pragma unroll
      for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) acc[i][j] += t[i][j];
  }
};

// Fragment of rows row0 .. +31 of a K-major tile, step kk.
template <typename T>
__device__ __forceinline__ typename GT<T>::frag read_k(const char* tile, int row0, int kk, int lane) {
  const int r = lane & 31;
  return __builtin_bit_cast(typename GT<T>::frag,
                            *reinterpret_cast<const u32x4g*>(tile + (row0 + r) * 128 +
                                                             ((2 * kk + (lane >> 5)) ^ ((r >> 1) & 7)) * 16));
}

// MN-major tile of R columns: copy instruction c brings the k rows (64 / UR) c ..
template <typename T, int R>
struct MnTile {
  static constexpr int ES = GT<T>::ES, UR = R * ES / 16, RPI = 64 / UR;
  // the swizzle puts what the two halves (fp32: k rows 4 apart) or the four k rows
  // of a transposing read (bf16) take onto different banks
  __device__ static int swz(int kr) {
    if (ES == 4) return UR >= 16 ? 8 * ((kr >> 2) & 1) : 0;
    return UR >= 16 ? 4 * (kr & 3) : UR == 8 ? 4 * ((kr >> 1) & 1) : 0;
  }
  // k row held in row pr of the tile: fp32 rows of 128 bytes change places instead
  // of slots (an involution)
  __device__ static int krow(int pr) { return ES == 4 && UR == 8 ? pr ^ ((pr >> 2) & 1) : pr; }
};

// Fragments of F * 32 columns col0 .. of an MN-major tile, step kk.  bf16: fragment
// f is columns 32 f .. 32 f + 31, by transposing reads; fp32 with two fragments:
// the even and the odd columns, one 8-byte read per k (mn_spread).
template <typename T, int R, int F>
__device__ __forceinline__ void read_mn(const char* tile, int col0, int kk, int lane, typename GT<T>::frag (&v)[F]) {
  using Tl = MnTile<T, R>;
  const int row_l = lane & 31, half_l = lane >> 5;
  if constexpr (Tl::ES == 2) {
    typedef short v4i16 __attribute__((ext_vector_type(4)));
    typedef short v8i16 __attribute__((ext_vector_type(8)));
    // k rows 16 kk + 8 half + (lane & 15) / 4 and + 4
    const int kr = 8 * half_l + ((lane & 15) >> 2);
    const int in = (2 * ((lane >> 4) & 1) + ((lane & 3) >> 1)) * 16 + 8 * (lane & 1);
#pragma unroll
    for (int f = 0; f < F; ++f) {
      const __attribute__((address_space(3))) char* q = (const __attribute__((address_space(3))) char*)tile +
                                                        (16 * kk + kr) * Tl::UR * 16 + in +
                                                        (((col0 + 32 * f) >> 3) ^ Tl::swz(kr)) * 16;
      const v4i16 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) v4i16*)q);
      const v4i16 hi =
          __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) v4i16*)(q + 4 * Tl::UR * 16));
      const v8i16 w = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
      v[f] = __builtin_bit_cast(bf16x8, w);
    }
  } else {
    static_assert(F <= 2, "fragments per wave");
    const int col = col0 + F * row_l;
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const int kr = 8 * kk + 4 * half_l + t;
      const char* q = tile + (Tl::krow(kr) * Tl::UR + ((col >> 2) ^ Tl::swz(kr))) * 16 + (col & 3) * 4;
      if constexpr (F == 2) {
        const float2 p = *reinterpret_cast<const float2*>(q);
        v[0][t] = p.x;
        v[1][t] = p.y;
      } else {
        v[0][t] = *reinterpret_cast<const float*>(q);
      }
    }
  }
}

// Row / column of a wave's F * 32 that element e of fragment f of an MN-major
// operand stands for.
template <typename T, int F>
__device__ __forceinline__ int mn_spread(int f, int e) {
  return GT<T>::ES == 4 && F == 2 ? 2 * e + f : 32 * f + e;
}

// Column sums (a bias gradient) of an MN-major operand of R columns from its staged
// tiles, KG of them `group_bytes` apart: of the blocks that share the columns, block
// idx sums 4 << shift of them, a thread 4 columns of every (256 >> shift)-th k row.
// Added in pairs of lanes, then of waves: the rounding stays that of the threads' own
// sums, which start again every 8 stages.
template <typename T, int R, int KG>
struct ColSum {
  using Tl = MnTile<T, R>;
  static constexpr int ES = GT<T>::ES, UE = GT<T>::UE, BK = GT<T>::BK;
  int shift, c0, c, k0;
  bool on;
  float part[4], tot[4];
  __device__ __forceinline__ void init(bool want, int idx, int sh) {
    shift = sh;
    c0 = idx * (4 << sh);
    on = want && c0 < R;
    c = c0 + 4 * ((int)threadIdx.x & ((1 << sh) - 1));
    k0 = (int)threadIdx.x >> sh;
#pragma unroll
    for (int e = 0; e < 4; ++e) part[e] = tot[e] = 0.f;
  }
  __device__ __forceinline__ void stage(const char* tile, int group_bytes, int s) {
    for (int r = k0; r < KG * BK; r += 256 >> shift) {
      const int kr = r % BK;
      const char* q =
          tile + (r / BK) * group_bytes + (Tl::krow(kr) * Tl::UR + ((c / UE) ^ Tl::swz(kr))) * 16 + (c % UE) * ES;
      if constexpr (ES == 2) {
        const u32x2g v = *reinterpret_cast<const u32x2g*>(q);
        part[0] += __builtin_bit_cast(float, v[0] << 16);
        part[1] += __builtin_bit_cast(float, v[0] & 0xffff0000u);
        part[2] += __builtin_bit_cast(float, v[1] << 16);
        part[3] += __builtin_bit_cast(float, v[1] & 0xffff0000u);
      } else {
        const float4 v = *reinterpret_cast<const float4*>(q);
        part[0] += v.x;
        part[1] += v.y;
        part[2] += v.z;
        part[3] += v.w;
      }
    }
    if ((s & 7) == 7) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        tot[e] += part[e];
        part[e] = 0.f;
      }
    }
  }
  // all threads of the block, `on` the same for all; red: 4 * R floats.  out(column
  // of the tile, sum)
  template <typename F>
  __device__ __forceinline__ void finish(float* red, F out) {
    const int tid = threadIdx.x, w = 4 << shift;
#pragma unroll
    for (int e = 0; e < 4; ++e) tot[e] += part[e];
    for (int d = 1 << shift; d < 64; d <<= 1) {
#pragma unroll
      for (int e = 0; e < 4; ++e) tot[e] += __shfl_xor(tot[e], d, 64);
    }
    __syncthreads();
    if ((tid & 63) < (1 << shift)) {
#pragma unroll
      for (int e = 0; e < 4; ++e) red[(tid >> 6) * w + c - c0 + e] = tot[e];
    }
    __syncthreads();
    if (tid < w && c0 + tid < R) out(c0 + tid, (red[tid] + red[w + tid]) + (red[2 * w + tid] + red[3 * w + tid]));
  }
};

// Cost of a convolution of `blocks` tiles over nst stages (matrix products have their
// own, mm_plan): rounds of 256 blocks, each of the tile's weight.
//  * fp32 rounds are their MFMAs: a weight is the stages of one block, plus 3 to 4
//    for its prologue and epilogue (half-size tiles in two K groups: half the
//    stages, slightly longer ones).
//  * bf16: the times of one round relative to 64 x 64 (products, 4096^3: 108, 143, 175, 252,
//    505 us on 128 x 128 .. 32 x 32).  A block alone on a CU cannot cover its
//    copies: less than 1.7 rounds cost as much (2048^3: 30 us on 256 blocks of 128 x
//    128, 24 on 512 of 64 x 128; 1024^3: 22, 9.4, 7.7, 7.0, 11.5).
template <typename T>
float tile_cost(int bm, int bn, int nst, long blocks) {
  const float rounds = (float)((blocks + 255) / 256);
  if (GT<T>::ES == 4) {
    if (bm == 32 && bn == 64) return rounds * (1.05f * (float)((nst + 1) / 2) + 3.5f);
    if (bm == 32 && bn == 32) return rounds * (1.1f * (float)((nst + 3) / 4) + 4.f);
    return rounds * ((float)nst + 3.f);  // 64 x 64, 32 x 128
  }
  const float w = bm == 128 ? 2.46f : bm == 64 ? (bn == 128 ? 1.5f : 1.f) : bn == 128 ? 1.1f : 0.72f;
  // deep products: four K groups shorten the chain (217 -> 224 @11 N=8: 17.4 -> 13.9 us)
  return w * std::max(rounds, bm == 32 && bn == 32 && nst >= 16 ? 1.4f : 1.7f);
}

// Whether a grid of bf16 tiles (ks wave groups) keeps a third stage: the whole grid
// still fits on the 256 CUs at once, 160 KB of LDS each.  Its few blocks cannot cover
// a copy's latency with two (3x3 217 -> 224 @11 N=8: 14.0 -> 12.5 us; 512 -> 512 @7
// N=32: 36.1 -> 30.5); where it takes blocks off a CU it costs more than it gives
// (256 -> 256 @14x15 N=32, 420 blocks in two K groups: 26.4 us on two, 31.2 on three).
// fp32 stages take four times as long to compute: within 2 % on either.
inline bool third_stage(int bm, int bn, int ks, long blocks) {
  return blocks <= 256L * (160 * 1024 / (3 * ks * (bm + bn) * 128));
}

}  // namespace tiles

}  // namespace vh
