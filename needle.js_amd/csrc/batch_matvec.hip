// Matvec of many activation rows on fp16 MFMA for matrices whose scales
// belong to groups of columns: int8 codes with one fp32 scale per group
// (g % 32 == 0), and Cactus-Quant codes with one binary16 norm per group
// (g = 32, 64, 128 or 256).
//
//   Y[b][n] = sum_u s[n][u] * sum_{j < 32} w[n][32 u + j] * x[b][32 u + j]
//
// over 32-column units u, s the scale or norm of the unit's group, w the
// exact code or the codebook value, and for Cactus-Quant x the rotated input
// (prepareCqActivation, backends/cq.ts:30-46).  Workgroup = (64 weight rows,
// 16 a wave) x (16 BS batch rows) x (a slice of k in 256-column chunks): the
// activations of a chunk are rotated (Cactus-Quant), split into fp16 hi + lo
// and written to LDS once for all of the workgroup's weight rows, and every
// weight row is read and widened once for all of its batch rows -- the forms
// with one batch row (or eight) per launch read and decode the matrix again
// for each.  KW groups of four waves take the slice's chunks in turn, each
// with its own LDS buffer, so that a SIMD has another wave to issue from while
// one waits (BS = 1, 4-bit codes: 2.5 us a chunk and workgroup with one group,
// 1.35 with four).
//
// Bound: the vector ALU.  A wave spends about 750 instructions on a chunk at
// BS = 1 with 4-bit codes (300 on the rotation and split of its share of the
// rows, 450 on decoding its 16 weight rows and the scaled sums) against 32
// MFMAs.  Before, the loads did: with 16 consecutive columns a thread and
// codes and norms read by the lane that uses them, a chunk took 20 load
// instructions of up to 64 separate lines; by rows through LDS it takes 8.
// 300 rows x (1536 x 512, 4-bit): 7.5 us (28.8 with a workgroup per batch
// row); 64 rows x (4096 x 4096, int8): 16.8 us (64.6 eight rows a launch).
//
// Split: a chunk's row is scaled by 2^(15 - e), e the exponent of its largest
// magnitude, hi = f16(v), lo = f16(v - hi): v is kept to 2^-23 of itself, and
// to 2^-39 of the chunk's largest where lo is subnormal.  int8 codes are
// exact in fp16; a codebook value is hi + lo too, after a factor that the
// upload picks so that the whole book loses least (nd_split_codebook), and
// all four products are taken.  fp16 products are exact in the fp32
// accumulator.  Each unit has its own accumulator from zero, so that its
// scale multiplies the unit's own dot, as the per-row forms do; chunk sums
// are scaled back (an exact ldexp) and added with Kahan's compensation.
// Cactus-Quant sums, which the split of x has cost bits already, take a
// chunk's units in two chains and the groups' and the scale in 64 bits: 1500 x
// 777, groups of 64, 100 rows: error against 64 bits 1.07e-7 in 2 bits and
// 1.09e-7 ternary, a row at a time 1.14e-7 and 1.11e-7 (1.18e-7 and 1.17e-7
// with one chain and 32 bits).
//
// MFMA operands (16x16x32 f16): A = activations (row = batch row, lane l
// holds row l % 16 and eight k of the unit, block l / 16), B = weights (column
// = weight row l % 16, the same eight k); lane l's accumulator component c is
// batch row 4 (l / 16) + c of weight row l % 16, so a lane needs only its own
// weight row's scales.
#include <cmath>

#include "nd_internal.hpp"
#include "nd_wave.hpp"

namespace {

using nd::codes_to_half;
using nd::float4v;
using nd::half8;
using nd::u32x2;
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef _Float16 half4 __attribute__((ext_vector_type(4)));

constexpr uint32_t kChunk = 256;          // columns per LDS stage
constexpr uint32_t kUnits = kChunk / 32;  // units per stage
constexpr uint32_t kRowH = kChunk + 8;    // halves per LDS row: 16 rows cover all banks
constexpr uint32_t kWaves = 4;            // per group: 64 weight rows
constexpr uint32_t kMaxSlices = 8;
constexpr uint32_t kTernaryBits = 5;


struct BatchArgs {
  const uint8_t* w;      // int8 codes (nd_tile_weights) or packed codes [n][row_bytes]
  const void* s;         // fp32 scales or binary16 norms [n][groups]
  const float* x;
  float* y;
  float* part;           // slice partials and arrival counters (slices > 1)
  uint32_t* counters;
  uint32_t x_stride, y_stride, k, units, groups, unit_shift, row_bytes, row_start, row_count,
      batch, tiles_n, tiles, slices, chunks, units_per_group, xl;
  double out_scale;  // Cactus-Quant: of the sums
  nd_code_planes cb;
};

// Four codes (one per byte, < 16) to four bytes of a 16-entry byte table.
template <int BITS>
__device__ __forceinline__ uint32_t table_bytes(const uint32_t (&tab)[4], uint32_t idx, uint32_t m) {
  if constexpr (BITS == 4) {
    const uint32_t lo = __builtin_amdgcn_perm(tab[1], tab[0], idx);
    const uint32_t hi = __builtin_amdgcn_perm(tab[3], tab[2], idx);
    return (lo & ~m) | (hi & m);
  } else {
    return __builtin_amdgcn_perm(tab[1], tab[0], idx);
  }
}

// Codebook halves of four codes (one per byte of c): hi[2], lo[2], two halves
// a word.
template <int BITS>
__device__ __forceinline__ void decode4(const nd_code_planes& cb, uint32_t c, uint32_t* hi,
                                        uint32_t* lo) {
  uint32_t idx = c, m = 0;
  if constexpr (BITS == 4) {
    // Selector 0x0c gives a zero byte, 0x0d an all-ones one.
    m = __builtin_amdgcn_perm(0u, 0u, 0x0c0c0c0cu | ((c >> 3) & 0x01010101u));
    idx = c & 0x07070707u;
  }
  const uint32_t h0 = table_bytes<BITS>(cb.v[0], idx, m), h1 = table_bytes<BITS>(cb.v[1], idx, m);
  const uint32_t l0 = table_bytes<BITS>(cb.v[2], idx, m), l1 = table_bytes<BITS>(cb.v[3], idx, m);
  hi[0] = __builtin_amdgcn_perm(h1, h0, 0x05010400u);
  hi[1] = __builtin_amdgcn_perm(h1, h0, 0x07030602u);
  lo[0] = __builtin_amdgcn_perm(l1, l0, 0x05010400u);
  lo[1] = __builtin_amdgcn_perm(l1, l0, 0x07030602u);
}

// FORM 0: int8 codes; 2, 3, 4: Cactus-Quant codes of that many bits (ternary
// crumbs are 2).  VEC: float4 loads of x.
template <int FORM, int KW, int BS, bool VEC>
__global__ __launch_bounds__(64 * kWaves * KW) void batch_matvec_kernel(BatchArgs a) {
  constexpr bool kCq = FORM != 0;
  constexpr uint32_t kThreads = 64 * kWaves, kRows = 16 * BS;
  constexpr uint32_t kPassRows = kThreads / 16;  // batch rows staged per pass
  constexpr int kPasses = kRows / kPassRows;
  static_assert(kRows % kPassRows == 0, "the staging divides evenly");
  __shared__ __align__(16) _Float16 s_xb[KW][2][kRows][kRowH];
  __shared__ __align__(16) int s_eb[KW][kRows];
  // Scales of the chunk's units and, for Cactus-Quant, its packed codes (rows
  // padded to 4 words past a multiple of 8 or 16: 16 rows cover all banks).
  constexpr uint32_t kWRows = 16 * kWaves;
  constexpr uint32_t kCodeWords = kCq ? 8 * FORM : 4, kCodeLd = kCodeWords + 4;
  __shared__ __align__(16) uint32_t s_cb[KW][kCq ? kWRows : 1][kCodeLd];
  __shared__ float s_sb[KW][kWRows][kUnits + 1];
  const uint32_t grp = KW > 1 ? __builtin_amdgcn_readfirstlane(threadIdx.x / kThreads) : 0;
  const uint32_t t = KW > 1 ? threadIdx.x % kThreads : threadIdx.x, wave = t >> 6, lane = t & 63;
  auto& s_x = s_xb[grp];
  auto& s_e = s_eb[grp];
  auto& s_c = s_cb[grp];
  auto& s_s = s_sb[grp];
  const uint32_t r16 = lane & 15, kb = lane >> 4;
  // Tile and slice: with slices, every slice of a tile on one XCD (the
  // dispatcher hands workgroup L to XCD L % 8).
  uint32_t tile = blockIdx.x, slice = 0;
  if (a.slices > 1) {
    const uint32_t tpx = (a.tiles + 7) / 8, sl = blockIdx.x >> 3;
    tile = 8 * (sl % tpx) + (blockIdx.x & 7);
    slice = sl / tpx;
    if (tile >= a.tiles) return;
  }
  const uint32_t row0 = (tile % a.tiles_n) * kWRows, b0 = tile / a.tiles_n * kRows;
  // Group grp takes chunks c_begin + grp, + KW, ...; without slices the last
  // round may run past the row (x, codes and scales clamp, as zeros).
  const uint32_t per = a.chunks / a.slices, c_begin = slice * per + grp;
  const uint32_t rounds = (per + KW - 1) / KW;
  const uint32_t row = row0 + 16 * wave + r16;
  const uint32_t wrow = a.row_start + (row < a.row_count ? row : a.row_count - 1);

  // Staging: thread t takes batch row t / 16 of each pass and of the chunk's
  // columns the four pieces of four at sc + piece(q): bits 0, 1, 4 and 7 of
  // the column are in the thread, bits 2, 3, 5 and 6 are its lane's.
  const uint32_t sr = t >> 4, sc = (t & 3) * 4 + (t >> 2 & 3) * 32;
  auto piece = [](uint32_t q) { return 16 * (q & 1) + 128 * (q >> 1); };
  float xv[kPasses][16];
  auto load_x = [&](uint32_t chunk) {
    const uint32_t c0 = chunk * kChunk + sc;
#pragma unroll
    for (int p = 0; p < kPasses; ++p) {
      const uint32_t b = b0 + p * kPassRows + sr;
      const float* xr = a.x + (size_t)(b < a.batch ? b : a.batch - 1) * a.x_stride;
      if constexpr (VEC) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const uint32_t c = c0 + piece(q);
          const float4 f = *reinterpret_cast<const float4*>(xr + (c < a.k ? c : 0));
          xv[p][4 * q] = f.x;
          xv[p][4 * q + 1] = f.y;
          xv[p][4 * q + 2] = f.z;
          xv[p][4 * q + 3] = f.w;
        }
      } else {
        // Rows of any alignment: four words at a time, the last four of the
        // row instead of a piece that runs past it (k >= 4).
        typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const uint32_t c = c0 + piece(q);
          const f32x4u f = *reinterpret_cast<const f32x4u*>(xr + min(c, a.k - 4));
#pragma unroll
          for (int i = 0; i < 4; ++i) xv[p][4 * q + i] = f[i];
        }
      }
    }
  };
  // Weights of a chunk on their way to the products: int8 codes straight to
  // the lane that multiplies them (its weight row's 16 bytes of each unit
  // pair), packed Cactus-Quant codes and the scales by the group's threads
  // in row order, to go through LDS.
  constexpr uint32_t kPieces = kCq ? kWRows * kCodeWords / 4 / kThreads : kUnits / 2;
  constexpr uint32_t kScales = kWRows * kUnits / kThreads;  // per thread
  static_assert(!kCq || kWRows * kCodeWords / 4 % kThreads == 0 || FORM == 3, "whole passes");
  constexpr uint32_t kPieceLoads = FORM == 3 ? 2 : kPieces;  // 3-bit: 1.5 passes
  typedef uint32_t u32x4u __attribute__((ext_vector_type(4), aligned(4)));
  struct Weights {
    u32x4 q[kPieceLoads];
    uint32_t s[kScales];
  };
  auto load_w = [&](Weights& w, uint32_t chunk) {
    const uint32_t u0 = chunk * kUnits;
    if constexpr (!kCq) {
      const uint8_t* base = a.w + nd_tile_row(wrow, a.k) + kb * 256;
#pragma unroll
      for (uint32_t p = 0; p < kUnits / 2; ++p)
        w.q[p] = *reinterpret_cast<const u32x4*>(
            base + (size_t)(u0 + 2 * p < a.units ? u0 / 2 + p : 0) * 1024);
    } else {
      // 16-byte pieces of the rows' chunk; one that starts past the row
      // rereads its start, one that straddles its end runs into the next row
      // or the allocation's slack (both meet zero scales).
      constexpr uint32_t kPr = kCodeWords / 4;  // pieces per row
#pragma unroll
      for (uint32_t p = 0; p < kPieceLoads; ++p) {
        const uint32_t e = min(t + p * kThreads, kWRows * kPr - 1), r = e / kPr, c = e % kPr;
        const uint32_t rr = row0 + r < a.row_count ? row0 + r : a.row_count - 1;
        const uint32_t at = u0 * 4 * FORM + c * 16;
        const u32x4u v = *reinterpret_cast<const u32x4u*>(
            a.w + (size_t)(a.row_start + rr) * a.row_bytes + (at < a.row_bytes ? at : 0));
        w.q[p] = u32x4{v.x, v.y, v.z, v.w};
      }
    }
#pragma unroll
    for (uint32_t p = 0; p < kScales; ++p) {
      const uint32_t e = t + p * kThreads, r = e / kUnits, u = u0 + e % kUnits;
      const uint32_t rr = row0 + r < a.row_count ? row0 + r : a.row_count - 1;
      const size_t at = (size_t)(a.row_start + rr) * a.groups +
                        ((u < a.units ? u : 0) >> a.unit_shift);
      if constexpr (kCq)
        w.s[p] = reinterpret_cast<const uint16_t*>(a.s)[at];
      else
        w.s[p] = reinterpret_cast<const uint32_t*>(a.s)[at];
    }
  };
  // The packed codes and the scales to LDS (units past the row: scale zero).
  auto stage_w = [&](const Weights& w, uint32_t chunk) {
    if constexpr (kCq) {
      constexpr uint32_t kPr = kCodeWords / 4;
#pragma unroll
      for (uint32_t p = 0; p < kPieceLoads; ++p) {
        const uint32_t e = t + p * kThreads;
        if (FORM != 3 || e < kWRows * kPr)
          *reinterpret_cast<u32x4*>(&s_c[e / kPr][e % kPr * 4]) = w.q[p];
      }
    }
#pragma unroll
    for (uint32_t p = 0; p < kScales; ++p) {
      const uint32_t e = t + p * kThreads;
      const float v = kCq ? (float)__builtin_bit_cast(_Float16, (uint16_t)w.s[p])
                          : __uint_as_float(w.s[p]);
      s_s[e / kUnits][e % kUnits] = chunk * kUnits + e % kUnits < a.units ? v : 0.f;
    }
  };
  auto stage = [&](uint32_t chunk) {
    const uint32_t c0 = chunk * kChunk + sc;
#pragma unroll
    for (int p = 0; p < kPasses; ++p) {
      const bool live = b0 + p * kPassRows + sr < a.batch;
      float(&v)[16] = xv[p];
      if constexpr (VEC) {
#pragma unroll
        for (int i = 0; i < 16; ++i) v[i] = live && c0 + piece(i / 4) < a.k ? v[i] : 0.f;
      } else {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          // The piece may have been read `back` columns early.
          const uint32_t c = c0 + piece(q), back = c + 4 > a.k ? c + 4 - a.k : 0;
          const float f[4] = {v[4 * q], v[4 * q + 1], v[4 * q + 2], v[4 * q + 3]};
#pragma unroll
          for (uint32_t i = 0; i < 4; ++i) {
            float y = f[i];
#pragma unroll
            for (uint32_t s = 1; s + i < 4; ++s) y = back == s ? f[i + s] : y;
            v[4 * q + i] = live && c + i < a.k ? y : 0.f;
          }
        }
      }
      if constexpr (kCq) {
        // fastWalshHadamard: strides 1, 2, 16 and 128 in the thread, 4, 8, 32
        // and 64 with the lanes that hold them; the reference's operands, one
        // fp32 add or subtract each (fma(v, -1, other) is other - v).
        auto inner = [&](int st) {
#pragma unroll
          for (int i = 0; i < 16; ++i)
            if ((i & st) == 0) {
              const float l = v[i], r = v[i + st];
              v[i] = l + r;
              v[i + st] = l - r;
            }
        };
        auto cross = [&](auto m) {
          const float sign = (lane & decltype(m)::value) != 0 ? -1.f : 1.f;
#pragma unroll
          for (int i = 0; i < 16; ++i)
            v[i] = fmaf(v[i], sign, nd::lane_xor<decltype(m)::value>(v[i]));
        };
        inner(1);
        inner(2);
        cross(std::integral_constant<int, 1>());
        cross(std::integral_constant<int, 2>());
        inner(4);
        if (a.units_per_group > 1) cross(std::integral_constant<int, 4>());
        if (a.units_per_group > 2) cross(std::integral_constant<int, 8>());
        if (a.units_per_group > 4) inner(8);
      }
      float mx = 0.f;
#pragma unroll
      for (int i = 0; i < 16; ++i) mx = fmaxf(mx, fabsf(v[i]));
      mx = nd::row_max(mx);  // the batch row's 16 threads are one DPP row
      int ex = 0;
      if (mx > 0.f && mx <= 3.4028235e38f) frexpf(mx, &ex);  // mx < 2^ex
      ex = ex < -110 ? -110 : ex;  // 2^(15 - ex) stays finite; lo then ends at 2^-149
      const float down = ldexpf(1.f, 15 - ex);
      if ((t & 15) == 0) s_e[p * kPassRows + sr] = ex - 15;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        half4 hv, lv;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float f = v[4 * q + i] * down;
          const _Float16 hf = (_Float16)f;
          hv[i] = hf;
          lv[i] = (_Float16)(f - (float)hf);
        }
        *reinterpret_cast<half4*>(&s_x[0][p * kPassRows + sr][sc + piece(q)]) = hv;
        *reinterpret_cast<half4*>(&s_x[1][p * kPassRows + sr][sc + piece(q)]) = lv;
      }
    }
  };

  // Cactus-Quant: two chains of four units a chunk instead of one of eight.
  constexpr uint32_t kAcc = kCq ? 2 : 1;
  float4v tot[BS] = {}, comp[BS] = {};
  Weights wn;
  load_x(c_begin);
  load_w(wn, c_begin);
  for (uint32_t i = 0; i < rounds; ++i) {
    const uint32_t c = c_begin + i * KW;
    stage(c);
    stage_w(wn, c);
    const Weights w = wn;
    if (i + 1 < rounds) {
      load_x(c + KW);
      load_w(wn, c + KW);
    }
    nd::lds_barrier();
    float4v acc[kAcc][BS] = {};
    const uint32_t* crow = s_c[kCq ? 16 * wave + r16 : 0];
    u32x2 plo{};  // int8: the pair's second unit, from the permlane swap
#pragma unroll
    for (uint32_t u = 0; u < kUnits; ++u) {
      const float sv = s_s[16 * wave + r16][u];
      half8 wh, wl = {};
      uint32_t kcol = 32 * u + 8 * kb;
      if constexpr (!kCq) {
        // A lane's 16 bytes are half of one unit of the pair; the swaps give
        // every lane eight codes of the first unit (k blocks 0, 2, 1, 3 over
        // the lane blocks) and eight of the second.
        if (u % 2 == 0) {
          const auto lo = __builtin_amdgcn_permlane32_swap(w.q[u / 2].x, w.q[u / 2].z, false, false);
          const auto hi = __builtin_amdgcn_permlane32_swap(w.q[u / 2].y, w.q[u / 2].w, false, false);
          wh = codes_to_half(u32x2{lo[0], hi[0]});
          plo = u32x2{lo[1], hi[1]};
        } else {
          wh = codes_to_half(plo);
        }
        kcol = 32 * u + 8 * (kb == 1 ? 2 : kb == 2 ? 1 : kb);
      } else {
        uint32_t c0, c1;
        if constexpr (FORM == 4) {
          const uint32_t b = crow[4 * u + kb];
          const uint32_t even = b & 0x0f0f0f0fu, odd = (b >> 4) & 0x0f0f0f0fu;
          c0 = __builtin_amdgcn_perm(odd, even, 0x05010400u);
          c1 = __builtin_amdgcn_perm(odd, even, 0x07030602u);
        } else {
          uint32_t b;
          if constexpr (FORM == 3) {  // 24 bits from bit 24 kb, in words 0, 1 or 1, 2
            const uint64_t b64 = ((uint64_t)crow[3 * u + (kb >> 1) + 1] << 32) | crow[3 * u + (kb >> 1)];
            b = (uint32_t)(b64 >> (kb == 0 ? 0 : kb == 1 ? 24 : kb == 2 ? 16 : 40));
          } else {
            b = crow[2 * u + (kb >> 1)] >> (16 * (kb & 1));
          }
          constexpr uint32_t M = (1u << FORM) - 1;
          auto spread = [&](uint32_t v) {
            return (v & M) | ((v >> FORM) & M) << 8 | ((v >> (2 * FORM)) & M) << 16 |
                   ((v >> (3 * FORM)) & M) << 24;
          };
          c0 = spread(b);
          c1 = spread(b >> (4 * FORM));
        }
        u32x4 hw, lw;
        uint32_t h4[4], l4[4];
        decode4<FORM>(a.cb, c0, h4, l4);
        decode4<FORM>(a.cb, c1, h4 + 2, l4 + 2);
        hw = u32x4{h4[0], h4[1], h4[2], h4[3]};
        lw = u32x4{l4[0], l4[1], l4[2], l4[3]};
        wh = __builtin_bit_cast(half8, hw);
        wl = __builtin_bit_cast(half8, lw);
      }
#pragma unroll
      for (int b = 0; b < BS; ++b) {
        const half8 xh = *reinterpret_cast<const half8*>(&s_x[0][16 * b + r16][kcol]);
        const half8 xl = *reinterpret_cast<const half8*>(&s_x[1][16 * b + r16][kcol]);
        float4v d = {0.f, 0.f, 0.f, 0.f};
        if constexpr (kCq) {
          d = __builtin_amdgcn_mfma_f32_16x16x32_f16(xl, wl, d, 0, 0, 0);
          d = __builtin_amdgcn_mfma_f32_16x16x32_f16(xh, wl, d, 0, 0, 0);
        }
        d = __builtin_amdgcn_mfma_f32_16x16x32_f16(xl, wh, d, 0, 0, 0);
        d = __builtin_amdgcn_mfma_f32_16x16x32_f16(xh, wh, d, 0, 0, 0);
#pragma unroll
        for (int i = 0; i < 4; ++i)
          acc[u % kAcc][b][i] = fmaf(sv, d[i], acc[u % kAcc][b][i]);
      }
    }
#pragma unroll
    for (int b = 0; b < BS; ++b) {
      const int4 e4 = *reinterpret_cast<const int4*>(&s_e[16 * b + 4 * kb]);
      const int e[4] = {e4.x, e4.y, e4.z, e4.w};
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const float all = kAcc > 1 ? acc[0][b][q] + acc[kAcc - 1][b][q] : acc[0][b][q];
        const float v = ldexpf(all, e[q]) - comp[b][q], sum = tot[b][q] + v;
        const float lost = (sum - tot[b][q]) - v;
        comp[b][q] = fabsf(sum) <= 3.4028235e38f ? lost : 0.f;  // no inf - inf
        tot[b][q] = sum;
      }
    }
    if (i + 1 < rounds) nd::lds_barrier();  // every wave is done with the chunk
  }
  double wide[kCq ? 4 * BS : 1];
  if constexpr (kCq)
#pragma unroll
    for (int j = 0; j < 4 * BS; ++j) wide[j] = (double)tot[j / 4][j % 4];
  if constexpr (KW > 1) {
    // The groups' sums in group order, through LDS.
    float* red = reinterpret_cast<float*>(&s_xb[0][0][0][0]);
    static_assert((KW - 1) * 4 * BS * kThreads * 4 <= sizeof(s_xb), "the sums fit");
    nd::lds_barrier();
    if (grp > 0)
#pragma unroll
      for (int j = 0; j < 4 * BS; ++j)
        red[((grp - 1) * 4 * BS + j) * kThreads + t] = tot[j / 4][j % 4];
    nd::lds_barrier();
    if (grp == 0)
#pragma unroll
      for (int g = 1; g < KW; ++g)
#pragma unroll
        for (int j = 0; j < 4 * BS; ++j) {
          const float v = red[((g - 1) * 4 * BS + j) * kThreads + t];
          if constexpr (kCq) wide[j] += (double)v;
          else tot[j / 4][j % 4] += v;
        }
  }

  if (a.slices > 1) {
    // Slices: partials stored, the slice counted in once they are complete,
    // and the tile's last slice adds all of them in slice order (the same sum
    // on every run).  See nd_wave.hpp for the scopes.
    constexpr uint32_t kTile = kThreads * 4 * BS;
    float* mine = a.part + ((size_t)tile * a.slices + slice) * kTile;
    if (grp == 0)
#pragma unroll
    for (int b = 0; b < BS; ++b)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        float* at = mine + (4 * b + i) * kThreads + t;
        if (a.xl)
          __hip_atomic_store(at, tot[b][i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        else
          __hip_atomic_store(at, tot[b][i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
    __builtin_amdgcn_s_waitcnt(0);  // every store above has completed
    __syncthreads();
    __shared__ uint32_t s_last;
    uint32_t* counter = a.counters + (size_t)tile * 32;
    if (threadIdx.x == 0)
      s_last = (a.xl ? __hip_atomic_fetch_add(counter, 1u, __ATOMIC_RELAXED,
                                              __HIP_MEMORY_SCOPE_WORKGROUP)
                     : __hip_atomic_fetch_add(counter, 1u, __ATOMIC_RELAXED,
                                              __HIP_MEMORY_SCOPE_AGENT)) == a.slices - 1;
    __syncthreads();
    if (!s_last || grp > 0) return;
    const float* all = a.part + (size_t)tile * a.slices * kTile + t;
    constexpr uint32_t kMax = BS == 4 ? kMaxSlices / 2 : kMaxSlices;  // the launcher's limit
    float pv[kMax][4 * BS];
#pragma unroll
    for (uint32_t z = 0; z < kMax; ++z)
#pragma unroll
      for (int i = 0; i < 4 * BS; ++i)
        pv[z][i] = __hip_atomic_load(all + (size_t)(z < a.slices ? z : 0) * kTile + i * kThreads,
                                     __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
    for (int i = 0; i < 4 * BS; ++i) {
      float sum = pv[0][i];
#pragma unroll
      for (uint32_t z = 1; z < kMax; ++z)
        if (z < a.slices) sum += pv[z][i];
      tot[i / 4][i % 4] = sum;
    }
    if (t == 0) {
      if (a.xl)
        __hip_atomic_store(counter, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
      else
        __hip_atomic_store(counter, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
  }
  if (row >= a.row_count || grp > 0) return;
#pragma unroll
  for (int b = 0; b < BS; ++b)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const uint32_t br = b0 + 16 * b + 4 * kb + i;
      if (br < a.batch)
        a.y[(size_t)br * a.y_stride + row] =
            kCq ? (float)(wide[kCq ? 4 * b + i : 0] * a.out_scale) : tot[b][i];
    }
}

using BatchFn = void (*)(BatchArgs);

struct Tile {
  uint32_t kw, bs;
};

template <int FORM, bool VEC>
BatchFn pick_tile(const Tile& tl) {
  switch (tl.bs * 8 + tl.kw) {
    case 8 + 1: return &batch_matvec_kernel<FORM, 1, 1, VEC>;
    case 8 + 2: return &batch_matvec_kernel<FORM, 2, 1, VEC>;
    case 8 + 4: return &batch_matvec_kernel<FORM, 4, 1, VEC>;
    case 16 + 1: return &batch_matvec_kernel<FORM, 1, 2, VEC>;
    case 16 + 2: return &batch_matvec_kernel<FORM, 2, 2, VEC>;
    case 32 + 1: return &batch_matvec_kernel<FORM, 1, 4, VEC>;
    default: return &batch_matvec_kernel<FORM, 2, 4, VEC>;
  }
}

BatchFn pick(int form, bool vec, const Tile& tl) {
  if (form == 0) return pick_tile<0, true>(tl);
  if (form == 2) return vec ? pick_tile<2, true>(tl) : pick_tile<2, false>(tl);
  if (form == 3) return vec ? pick_tile<3, true>(tl) : pick_tile<3, false>(tl);
  return vec ? pick_tile<4, true>(tl) : pick_tile<4, false>(tl);
}

}  // namespace

// The codebook times a factor as hi/lo fp16 byte planes.  The factor brings
// the largest magnitude to [2^7, 2^8) -- lo stays normal down to 2^-10 of it
// -- and is picked out of 256 in that octave for the smallest squared
// residual of the whole book: a value's residual is the same in every product
// with it, so unlike the activations' it does not average out (ternary books,
// one magnitude, lose nothing; the 3- and 4-bit books measured 5e-8 and 1e-8
// of the result with a power of two, against the 1.2e-7 of fp32 sums).
bool nd_split_codebook(const float* cb, uint32_t bits, nd_code_planes* out, double* factor) {
  const int n = bits == 4 ? 16 : bits == 3 ? 8 : 4;
  double mx = 0.0;
  for (int i = 0; i < n; ++i) {
    if (!std::isfinite(cb[i])) return false;
    mx = std::fmax(mx, std::fabs((double)cb[i]));
  }
  int e = 0;
  if (mx > 0.0) std::frexp(mx, &e);
  if (e > 60 || e < -60) return false;
  auto split = [](double v, _Float16& h, _Float16& l) {
    h = (_Float16)v;
    l = (_Float16)(v - (double)h);
    return v - (double)h - (double)l;
  };
  double best = INFINITY;
  for (int j = 0; j < 256; ++j) {
    const double f = std::ldexp(1.0 + j / 256.0, 7 - e);
    if (j && mx * f >= 256.0) break;
    double lost = 0.0;
    for (int i = 0; i < n; ++i) {
      _Float16 h, l;
      const double r = split(cb[i] * f, h, l) / f;
      lost += r * r;
    }
    if (lost < best) {
      best = lost;
      *factor = f;
    }
  }
  *out = nd_code_planes{};
  for (int i = 0; i < n; ++i) {
    _Float16 h, l;
    split(cb[i] * *factor, h, l);
    const uint16_t hb = __builtin_bit_cast(uint16_t, h), lb = __builtin_bit_cast(uint16_t, l);
    const int w = i / 4, sh = 8 * (i % 4);
    out->v[0][w] |= (uint32_t)(hb & 0xff) << sh;
    out->v[1][w] |= (uint32_t)(hb >> 8) << sh;
    out->v[2][w] |= (uint32_t)(lb & 0xff) << sh;
    out->v[3][w] |= (uint32_t)(lb >> 8) << sh;
  }
  return true;
}

namespace {

// Tile and slices of a launch: the largest batch tile that still gives 160
// workgroups (5/8 of the CUs; 240 tiles of 32 rows against 456 of 16: 8.4 and
// 9.0 us, 80 against 152: 8.0 and 6.2), counting the k slices that `split`
// allows (power-of-two shares of at least two chunks, up to 256 workgroups);
// then as many wave groups as the chunks and LDS allow.
struct Plan {
  Tile tile;
  uint32_t tiles_n, slices, chunks;
  uint64_t tiles;
};

Plan plan_batch(uint32_t width, uint32_t row_count, uint32_t batch, bool split) {
  Plan p{};
  p.chunks = (width + kChunk - 1) / kChunk;
  p.tiles_n = (row_count + 16 * kWaves - 1) / (16 * kWaves);
  for (uint32_t bs = 4; bs >= 1; bs /= 2) {
    if (bs > 1 && 8 * bs >= batch) continue;  // half the tile would be padding
    p.tile.bs = bs;
    p.tiles = (uint64_t)p.tiles_n * ((batch + 16 * bs - 1) / (16 * bs));
    p.slices = 1;
    const uint32_t limit = bs == 4 ? kMaxSlices / 2 : kMaxSlices;
    const size_t tile_bytes = 64 * kWaves * 4 * bs * sizeof(float);
    while (split && p.slices < limit && p.chunks % (4 * p.slices) == 0 &&
           p.tiles * p.slices < 256 && p.tiles <= kMatvecCounters &&
           p.tiles * p.slices * 2 * tile_bytes <= kMatvecPartialBytes)
      p.slices *= 2;
    if (p.tiles * p.slices >= 160) break;
  }
  const uint32_t per = p.chunks / p.slices, most = p.tile.bs > 1 ? 2 : 4;
  p.tile.kw = 1;
  while (p.tile.kw < most && p.tile.kw < per && (p.slices == 1 || per % (2 * p.tile.kw) == 0))
    p.tile.kw *= 2;
  return p;
}

}  // namespace

bool nd_batch_matvec_fits(const nd_mat* m, uint32_t batch) {
  if (batch < 3) return false;
  if (m->bits) return m->g >= 32 && m->g <= kChunk && m->k >= 4 && m->cb_factor > 0.0;
  return m->wt && m->g % 32 == 0 && m->k % 128 == 0;
}

float nd_batch_matvec_us(const nd_mat* m, uint32_t row_count, uint32_t batch) {
  const Plan p = plan_batch(m->kpad, row_count, batch, false);
  const float chunk_us = p.tile.bs == 4 ? 4.4f : p.tile.bs == 2 ? 2.4f : 1.4f;
  const uint32_t chunks = (p.chunks + p.tile.kw - 1) / p.tile.kw * p.tile.kw;  // whole rounds
  return (float)((p.tiles + 255) / 256) * (float)chunks * chunk_us;
}

hipError_t nd_launch_batch_matvec(const nd_mat* m, const float* x, uint32_t batch,
                                  uint32_t x_stride, uint32_t row_start, uint32_t row_count,
                                  float* y, uint32_t y_stride, hipStream_t s, void* split) {
  if (batch == 0 || row_count == 0) return hipSuccess;
  if (!nd_batch_matvec_fits(m, batch)) return hipErrorInvalidValue;
  BatchArgs a{};
  const uint32_t width = m->bits ? m->kpad : m->k;
  a.w = m->bits ? m->packed : reinterpret_cast<const uint8_t*>(m->wt);
  a.s = m->bits ? (const void*)m->norms : (const void*)m->scales;
  a.x = x;
  a.y = y;
  a.x_stride = x_stride;
  a.y_stride = y_stride;
  a.k = m->k;
  a.units = width / 32;
  a.groups = width / m->g;
  while ((32u << a.unit_shift) < m->g) ++a.unit_shift;
  a.row_bytes = m->row_bytes;
  a.row_start = row_start;
  a.row_count = row_count;
  a.batch = batch;
  a.units_per_group = m->g / 32;
  int form = 0;
  if (m->bits) {
    a.cb = m->planes;
    a.out_scale = (double)(float)(1.0 / std::sqrt((double)m->g)) / m->cb_factor;
    form = m->bits == kTernaryBits ? 2 : (int)m->bits;
  }
  const bool vec =
      (m->k & 3) == 0 && (x_stride & 3) == 0 && (reinterpret_cast<uintptr_t>(x) & 15) == 0;
  if (!m->bits && !vec) return hipErrorInvalidValue;
  const Plan p = plan_batch(width, row_count, batch, split != nullptr);
  if (p.tiles > 0x7fffffffu) return hipErrorInvalidValue;
  a.tiles_n = p.tiles_n;
  a.tiles = (uint32_t)p.tiles;
  a.slices = p.slices;
  a.chunks = p.chunks;
  uint32_t grid = a.tiles;
  if (a.slices > 1) {
    a.part = reinterpret_cast<float*>(split);
    a.counters = reinterpret_cast<uint32_t*>(reinterpret_cast<char*>(split) + kMatvecPartialBytes);
    a.xl = nd_xcd_local() ? 1u : 0u;
    grid = (a.tiles + 7) / 8 * 8 * a.slices;
  }
  hipLaunchKernelGGL(pick(form, vec, p.tile), dim3(grid), dim3(64 * kWaves * p.tile.kw), 0, s, a);
  return hipGetLastError();
}
