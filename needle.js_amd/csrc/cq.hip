// Cactus-Quant (CQ2 / CQ3 / CQ4 / ternary) matrices on gfx950: the shipped
// weight format of needle.js (model/cact.ts:61-75, 346-396), multiplied
// without expanding the weights (backends/cq.ts:107-231).
//
// Layout in HBM, as in the archive: packed codes [n][row_bytes] (row_bytes =
// kpad * pb / 8, pb = 2 for ternary records), then binary16 norms
// [n][kpad / g].  Here kpad is the stored width: the archive's (k rounded up
// to the group size g) rounded up to 32 codes, the added codes and their
// groups' norms zero, so every row is whole 32-code units.  The codebook of the matrix's
// width (4, 8 or 16 floats; ternary: 0, +c, 0, -c with c = 1.2240064 /
// sqrt(g)) travels as a kernel argument and is copied to LDS.
//
//  * cq_prepare_kernel: prepareCqActivation (cq.ts:30-46) -- per group the
//    fastWalshHadamard butterflies (cq.ts:8-27) in the reference's stage
//    order with an fp32 result per butterfly, then value * 1/sqrt(g) in
//    float64 with an fp32 store: bit-identical to the reference's Float32Array.
//  * cq_matvec_kernel: thread (sub, u) owns 32-weight unit u of rows row0 +
//    p * rpp + sub; its 32 prepared inputs stay in registers, each row
//    contributes one 8 / 12 / 16-byte load and the unit's binary16 norms;
//    codes index the LDS codebook; fp32 dots per group times the group norm,
//    reduced over the row's threads through LDS and a DPP butterfly.
//  * cq_row_kernel: dequantizeCqRow (cq.ts:243-295): f32(codebook * norm),
//    the same butterflies, f32(value * 1/sqrt(g)); bit-identical.
#include <cmath>

#include "nd_internal.hpp"
#include "nd_wave.hpp"

namespace {

constexpr int kCqThreads = 256;
constexpr uint32_t kTernaryBits = 5;
constexpr double kTernaryCentroid = 1.2240064;  // backends/cq.ts:6

// binary16 bit pattern -> float (float16ToNumber, fp16.ts:5-32; exact).
__device__ __forceinline__ float half_bits_to_float(uint32_t h) {
  return (float)__builtin_bit_cast(_Float16, (uint16_t)h);
}

// Per-group FWHT of v[0, len) in LDS (len = kpad, groups of g): stride 1, 2,
// 4, ... with one butterfly per (pair) and a barrier per stage; each result
// is one fp32 add or subtract, as the reference's Float32Array stores.
__device__ void fwht_groups(float* v, uint32_t len, uint32_t g) {
  for (uint32_t stride = 1; stride < g; stride <<= 1) {
    for (uint32_t i = threadIdx.x; i < len / 2; i += blockDim.x) {
      // Pair i: block of 2*stride, position inside the block's left half.
      const uint32_t block = i / stride, inner = i % stride;
      const uint32_t left = block * 2 * stride + inner, right = left + stride;
      const float a = v[left], b = v[right];
      v[left] = a + b;
      v[right] = a - b;
    }
    __syncthreads();
  }
}

// out[b][0, kpad) = prepareCqActivation(x[b][0, k)) for one batch row per
// workgroup.
__global__ __launch_bounds__(kCqThreads) void cq_prepare_kernel(const float* __restrict__ x,
                                                                uint32_t x_stride, uint32_t k,
                                                                uint32_t kpad, uint32_t g,
                                                                double inverse_root,
                                                                float* __restrict__ out) {
  __shared__ float v[8192];
  const float* xb = x + (size_t)blockIdx.x * x_stride;
  float* ob = out + (size_t)blockIdx.x * kpad;
  for (uint32_t i = threadIdx.x; i < kpad; i += blockDim.x) v[i] = i < k ? xb[i] : 0.f;
  __syncthreads();
  fwht_groups(v, kpad, g);
  for (uint32_t i = threadIdx.x; i < kpad; i += blockDim.x)
    ob[i] = (float)((double)v[i] * inverse_root);
}

// dequantizeCqRow for one row.
struct Codebook {
  float v[16];
};

__device__ __forceinline__ uint32_t code_at(const uint8_t* row, uint32_t c, uint32_t bits) {
  if (bits == 2 || bits == kTernaryBits) return (row[c >> 2] >> ((c & 3) * 2)) & 3u;
  if (bits == 4) return (row[c >> 1] >> ((c & 1) * 4)) & 15u;
  const uint32_t bit = c * 3, at = bit >> 3, shift = bit & 7;
  const uint32_t word = (uint32_t)row[at] | (shift > 5 ? (uint32_t)row[at + 1] << 8 : 0u);
  return (word >> shift) & 7u;
}

__global__ __launch_bounds__(kCqThreads) void cq_row_kernel(
    const uint8_t* __restrict__ packed, const uint16_t* __restrict__ norms, Codebook cb,
    uint32_t k, uint32_t kpad, uint32_t g, uint32_t bits, uint32_t row_bytes, uint32_t row,
    double inverse_root, float* __restrict__ out) {
  __shared__ float v[8192];
  const uint8_t* prow = packed + (size_t)row * row_bytes;
  const uint32_t groups = kpad / g;
  for (uint32_t c = threadIdx.x; c < kpad; c += blockDim.x) {
    const float norm = half_bits_to_float(norms[(size_t)row * groups + c / g]);
    const uint32_t code = code_at(prow, c, bits);
    // Ternary: crumb 3 -> -c, 1 -> +c, 0 and 2 -> 0 (the record's index
    // mapping into Float32Array([-c, 0, c]), cq.ts:259-273); cb holds them
    // by crumb.
    v[c] = cb.v[code] * norm;
  }
  __syncthreads();
  fwht_groups(v, kpad, g);
  for (uint32_t c = threadIdx.x; c < k; c += blockDim.x)
    out[c] = (float)((double)v[c] * inverse_root);
}

// cb.v[i] for i < N by a select tree over the bits of i (constant indices
// only).
template <int N>
__device__ __forceinline__ float pick_code(const Codebook& cb, uint32_t i) {
  float v[N];
#pragma unroll
  for (int j = 0; j < N; ++j) v[j] = cb.v[j];
#pragma unroll
  for (int half = N / 2, bit = 0; half >= 1; half /= 2, ++bit) {
#pragma unroll
    for (int j = 0; j < half; ++j) v[j] = (i >> bit) & 1u ? v[2 * j + 1] : v[2 * j];
  }
  return v[0];
}

// Rotated inputs of unit u (32 consecutive columns) in registers: the
// butterflies of fastWalshHadamard with strides 1 .. GS / 2 inside the unit
// (GS = min(g, 32)), then strides 32, 64, ... as exchanges with the lanes
// holding the group's other units (lane strides 1 .. lanes_per_group / 2).
// Each result is one fp32 add or subtract of the same two operands as the
// reference's; the 1/sqrt(g) factor is left to the caller.
template <int M>
__device__ __forceinline__ void cross_lane_stage(float (&v)[32]) {
  const bool right = (__lane_id() & M) != 0;
#pragma unroll
  for (int i = 0; i < 32; ++i) {
    const float other = nd::lane_xor<M>(v[i]);
    v[i] = right ? other - v[i] : v[i] + other;
  }
}

template <int GS>
__device__ __forceinline__ void rotate_unit(float (&v)[32], uint32_t lanes_per_group) {
#pragma unroll
  for (int st = 1; st < GS; st <<= 1) {
#pragma unroll
    for (int i = 0; i < 32; ++i) {
      if ((i & st) == 0) {
        const float a = v[i], b = v[i + st];
        v[i] = a + b;
        v[i + st] = a - b;
      }
    }
  }
  if (lanes_per_group > 1) cross_lane_stage<1>(v);
  if (lanes_per_group > 2) cross_lane_stage<2>(v);
  if (lanes_per_group > 4) cross_lane_stage<4>(v);
  if (lanes_per_group > 8) cross_lane_stage<8>(v);
  if (lanes_per_group > 16) cross_lane_stage<16>(v);
  if (lanes_per_group > 32) cross_lane_stage<32>(v);
}

// y[b][r] for rows [row_start, row_start + row_count), batch row b =
// blockIdx.y.  Thread (sub, u) owns 32-code unit u of rows row0 + i * rpp +
// sub (i < RACC).  UB = bytes of a unit (8: 2-bit and ternary, 12: 3-bit,
// 16: 4-bit); NG = groups in a unit (1 when g >= 32, else 32 / g).
// ROTATE: x is the raw input [k] and each thread rotates its unit in
// registers (g <= 2048: a group's units sit in one wave); otherwise x holds
// rotated rows [kpad] from cq_prepare_kernel.  VEC: x rows are 16-byte
// aligned with k % 4 == 0 (float4 loads), else scalar loads.  Both load
// unconditionally from clamped addresses and zero what lies past the row.  The weight codes and norms
// are issued first among the HBM loads after x, so the rotation overlaps
// their latency; codes index an LDS copy of the codebook; fp32 dots per
// group times the group norm; row sums through LDS and a DPP butterfly,
// times out_scale (1/sqrt(g) for ROTATE, else 1).
// Codes per table lookup for UB-byte units: entries of kE floats indexed by
// kE packed codes.
constexpr int lookup_codes(int ub) { return ub == 8 ? 4 : 2; }

template <int UB, int NG, int RACC, bool ROTATE, bool VEC>
__global__ __launch_bounds__(kCqThreads) void cq_matvec_kernel(
    const uint8_t* __restrict__ packed, const uint16_t* __restrict__ norms, Codebook cb,
    const float* __restrict__ x, uint32_t x_stride, float* __restrict__ y, uint32_t y_stride,
    uint32_t k, uint32_t kpad, uint32_t g_log2, uint32_t row_bytes, uint32_t row_start,
    uint32_t row_count, uint32_t tpr_log2, uint32_t lanes_per_group, float out_scale) {
  constexpr int kGs = 32 / NG;  // weights per group inside a unit
  // Lookup table in LDS: entry i holds the codebook values of the kE codes
  // packed in index i (kE * bits index bits), one read per kE weights.
  constexpr int kPB = UB / 4;                  // bits per code
  constexpr int kE = lookup_codes(UB);         // codes per lookup
  constexpr int kLB = kPB * kE;                // bits per lookup index
  constexpr int kEntries = 1 << kLB;
  constexpr int kLookups = 32 / kE;            // per unit
  __shared__ __align__(16) float tab[kEntries * kE];
  __shared__ float red[RACC * kCqThreads];
  const uint32_t t = threadIdx.x;
  const uint32_t tpr = 1u << tpr_log2, rpp = kCqThreads >> tpr_log2;
  const uint32_t sub = t >> tpr_log2, u = t & (tpr - 1);
  const uint32_t units = kpad / 32, groups = kpad >> g_log2;
  const bool active = u < units;
  const uint32_t uc = active ? u : 0;
  const uint32_t row0 = blockIdx.x * rpp * RACC;
  const float* xb = x + (size_t)blockIdx.y * x_stride;

  // x first (L2-resident, needed first), then the weights; nothing reads
  // x until the weight loads are issued, so the wait for x leaves them in
  // flight.
  float xv[32];
  const uint32_t c0 = u * 32, lim = ROTATE ? k : kpad;
  if constexpr (VEC) {
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      const uint32_t c = c0 + 4 * q;
      const float4 f = *reinterpret_cast<const float4*>(xb + (c < lim ? c : lim - 4));
      xv[4 * q] = f.x;
      xv[4 * q + 1] = f.y;
      xv[4 * q + 2] = f.z;
      xv[4 * q + 3] = f.w;
    }
  } else {
#pragma unroll
    for (int i = 0; i < 32; ++i) {
      const uint32_t c = c0 + i;
      xv[i] = xb[c < lim ? c : lim - 1];
    }
  }
  __builtin_amdgcn_sched_barrier(0);
  uint32_t raw[RACC][UB / 4];
  uint32_t nb[RACC][(NG + 1) / 2];
#pragma unroll
  for (int r = 0; r < RACC; ++r) {
    const uint32_t row = row0 + r * rpp + sub;
    const uint32_t rr = row_start + (row < row_count ? row : 0);
    const uint32_t* src = reinterpret_cast<const uint32_t*>(packed + (size_t)rr * row_bytes +
                                                            (size_t)uc * UB);
#pragma unroll
    for (int w = 0; w < UB / 4; ++w) raw[r][w] = src[w];
    const uint16_t* nrow = norms + (size_t)rr * groups;
    if constexpr (NG == 1) {
      nb[r][0] = nrow[(uc * 32) >> g_log2];
    } else if constexpr (NG == 2) {
      nb[r][0] = *reinterpret_cast<const uint32_t*>(nrow + uc * 2);
    } else {
      const uint2 v = *reinterpret_cast<const uint2*>(nrow + uc * 4);
      nb[r][0] = v.x;
      nb[r][1] = v.y;
    }
  }
  __builtin_amdgcn_sched_barrier(0);
  // The table, while the loads are in flight.  The codebook is read at
  // constant indices (scalar loads of the kernel arguments) and each entry
  // picked with a select tree: no per-lane loads from the argument segment.
  if (t < (uint32_t)kEntries) {
#pragma unroll
    for (int e = 0; e < kE; ++e)
      tab[t * kE + e] = pick_code<(1 << kPB)>(cb, (t >> (e * kPB)) & ((1u << kPB) - 1));
  }
  // Columns past the row (clamped loads above) read as zero.
#pragma unroll
  for (int i = 0; i < 32; ++i) {
    const uint32_t c = VEC ? c0 + (i & ~3) : c0 + i;
    xv[i] = c < lim ? xv[i] : 0.f;
  }
  if constexpr (ROTATE) rotate_unit<kGs>(xv, lanes_per_group);
  __syncthreads();  // tab

  // Codebook values of row r's 32 codes: kLookups table reads (bits
  // kLB * i .. of the unit's 32 * kPB-bit stream).  Row r + 1's reads are
  // issued before row r's products, so LDS latency overlaps the FMAs.
  auto lookup_row = [&](int r, float (&tv)[32]) {
#pragma unroll
    for (int i = 0; i < kLookups; ++i) {
      const int bit = kLB * i, w = bit >> 5, sh = bit & 31;
      const uint32_t b = sh + kLB <= 32
                             ? (raw[r][w] >> sh) & (kEntries - 1u)
                             : ((raw[r][w] >> sh) | (raw[r][w + 1] << (32 - sh))) & (kEntries - 1u);
      const char* at = reinterpret_cast<const char*>(tab) + b * (kE * 4);
      if constexpr (kE == 4) {
        const float4 f = *reinterpret_cast<const float4*>(at);
        tv[4 * i] = f.x;
        tv[4 * i + 1] = f.y;
        tv[4 * i + 2] = f.z;
        tv[4 * i + 3] = f.w;
      } else if constexpr (kE == 2) {
        const float2 f = *reinterpret_cast<const float2*>(at);
        tv[2 * i] = f.x;
        tv[2 * i + 1] = f.y;
      } else {
        tv[i] = *reinterpret_cast<const float*>(at);
      }
    }
  };
  float acc[RACC];
  float tv[2][32];
  lookup_row(0, tv[0]);
#pragma unroll
  for (int r = 0; r < RACC; ++r) {
    if (r + 1 < RACC) lookup_row(r + 1, tv[(r + 1) & 1]);
    __builtin_amdgcn_sched_barrier(0);
    const float(&v)[32] = tv[r & 1];
    float total = 0.f;
#pragma unroll
    for (int s = 0; s < NG; ++s) {
      float d[kE];
#pragma unroll
      for (int e = 0; e < kE; ++e) d[e] = 0.f;
#pragma unroll
      for (int jj = 0; jj < kGs; ++jj) {
        const int j = s * kGs + jj;
        d[jj % kE] = fmaf(v[j], xv[j], d[jj % kE]);
      }
      float dot = d[0];
      if constexpr (kE >= 2) dot += d[1];
      if constexpr (kE == 4) dot += d[2] + d[3];
      const uint32_t h = NG == 1 ? nb[r][0] : (nb[r][s >> 1] >> (16 * (s & 1))) & 0xFFFFu;
      total = fmaf(half_bits_to_float(h), dot, total);
    }
    acc[r] = active ? total : 0.f;
  }

  // Row sums over the row's tpr threads: red is [RACC][256]; T = 256 /
  // (rpp * RACC) threads per output each add tpr / T = RACC columns, then a
  // T-lane butterfly.
#pragma unroll
  for (int r = 0; r < RACC; ++r) red[r * kCqThreads + t] = acc[r];
  __syncthreads();
  const uint32_t outputs = rpp * RACC;
  const uint32_t T = kCqThreads / outputs;
  const uint32_t o = t / T, part = t % T;
  const uint32_t osub = o / RACC, orr = o % RACC;
  const float* col = red + orr * kCqThreads + osub * tpr;
  float sum = 0.f;
#pragma unroll
  for (int i = 0; i < RACC; ++i) sum += col[part + T * i];
  if (T > 32) sum = nd::sum_xor<32>(sum);
  if (T > 16) sum = nd::sum_xor<16>(sum);
  if (T > 8) sum += nd::lane_xor<8>(sum);
  if (T > 4) sum += nd::lane_xor<4>(sum);
  if (T > 2) sum += nd::lane_xor<2>(sum);
  if (T > 1) sum += nd::lane_xor<1>(sum);
  if (part == 0) {
    const uint32_t row = row0 + orr * rpp + osub;
    if (row < row_count) y[(size_t)blockIdx.y * y_stride + row] = sum * out_scale;
  }
}

// One activation row times a large matrix (g >= 32, at most 64 units a row):
// workgroups that stay for many rows, so that the rotation of x and a wider
// lookup table are set up once.  The table holds a copy of every entry for each
// lane of an LDS access phase (32 copies of 8-byte entries, 16 of 16-byte
// ones), laid out so that a lane's copy lies in banks of its own: a lookup of 64
// random codes takes the minimum of cycles, where the one shared copy of
// cq_matvec_kernel, whose LDS reads bound it, took about three times that.
// Bound by the weights: 32768 x 2048 in 4 bits (38 MB) 8.2 us a call against 10.5,
// of which about 4.3 are the launch's.
// The workgroup rotates x together (4 values a thread, the stages of
// rotate_unit in the same order: the same bits) while the first rows arrive.
// Wave w of the launch takes 64 / tpr rows at a time (tpr threads a row, one
// 32-code unit each), kStreamRows such passes in flight, strided over the rows
// by the launch's waves.  The same fp32 dots per unit, times the norm, as
// cq_matvec_kernel; row sums by a butterfly over the row's lanes.
constexpr uint32_t kStreamThreads = 512;
constexpr int kStreamRows = 4;
static_assert(kStreamThreads * 4 == 64 * 32, "a thread holds 4 of a row's values");

template <int M>
__device__ __forceinline__ void cross_lane_stage4(float (&v)[4]) {
  const bool right = (__lane_id() & M) != 0;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float other = nd::lane_xor<M>(v[i]);
    v[i] = right ? other - v[i] : v[i] + other;
  }
}

template <int UB>
__global__ __launch_bounds__(kStreamThreads) void cq_stream_kernel(
    const uint8_t* __restrict__ packed, const uint16_t* __restrict__ norms, Codebook cb,
    const float* __restrict__ x, bool vec, float* __restrict__ y, uint32_t k, uint32_t units,
    uint32_t groups, uint32_t g_log2, uint32_t row_bytes, uint32_t row_start, uint32_t row_count,
    uint32_t tpr_log2, float out_scale) {
  constexpr int kPB = UB / 4, kE = lookup_codes(UB), kLB = kPB * kE;
  constexpr uint32_t kEntries = 1u << kLB, kCopies = 64 / kE;  // an entry's copies: 64 words
  constexpr int kLookups = 32 / kE, kW = UB / 4;
  // x: 32 floats of a unit at 36 words, so that 16-byte reads of consecutive
  // units cover all banks.
  __shared__ __align__(16) float tab[kEntries * 64];
  __shared__ __align__(16) float sx[64 * 36];
  const uint32_t t = threadIdx.x, lane = t & 63;
  const uint32_t tpr = 1u << tpr_log2, rpw = 64u >> tpr_log2;  // rows a wave pass
  const uint32_t sub = lane >> tpr_log2, u = lane & (tpr - 1);
  const bool active = u < units;
  const uint32_t uc = active ? u : 0;
  const uint32_t wave = blockIdx.x * (kStreamThreads / 64) + __builtin_amdgcn_readfirstlane(t >> 6);
  const uint32_t step = gridDim.x * (kStreamThreads / 64) * rpw;  // rows between a wave's passes
  float v[4];
  if (vec) {
    const float4 f = *reinterpret_cast<const float4*>(x + (4 * t < k ? 4 * t : 0));
    v[0] = f.x;
    v[1] = f.y;
    v[2] = f.z;
    v[3] = f.w;
  } else {
#pragma unroll
    for (uint32_t i = 0; i < 4; ++i) v[i] = x[4 * t + i < k ? 4 * t + i : 0];
  }
  uint32_t raw[kStreamRows][kW], nb[kStreamRows];
  const uint32_t own = wave * rpw;
  // A pass beyond the rows re-reads the wave's first rows: loads without a
  // branch, and no line that many waves would ask for at once.
  auto load = [&](uint32_t first) __attribute__((always_inline)) {
#pragma unroll
    for (int r = 0; r < kStreamRows; ++r) {
      const uint32_t at = first + r * step < row_count ? first + r * step : own;
      const uint32_t row = at + sub;
      const size_t rr = row_start + (row < row_count ? row : row_count - 1);
      const uint32_t* src =
          reinterpret_cast<const uint32_t*>(packed + rr * row_bytes + (size_t)uc * UB);
#pragma unroll
      for (int w = 0; w < kW; ++w) raw[r][w] = __builtin_nontemporal_load(src + w);
      nb[r] = norms[rr * groups + ((uc * 32) >> g_log2)];
    }
  };
  __builtin_amdgcn_sched_barrier(0);
  load(own);
  __builtin_amdgcn_sched_barrier(0);
  // Copy c of entry e at words (e kCopies + c) kE.  Thread t writes the copies of
  // entry t, in an order turned by its lane: a write's lanes lie in different banks.
  for (uint32_t e = t; e < kEntries; e += kStreamThreads) {
    float c[kE];
#pragma unroll
    for (int i = 0; i < kE; ++i)
      c[i] = pick_code<(1 << kPB)>(cb, (e >> (i * kPB)) & ((1u << kPB) - 1));
#pragma unroll
    for (uint32_t q = 0; q < 16; ++q) {
      float4* at = reinterpret_cast<float4*>(tab + e * 64) + ((q + e) & 15);
      if constexpr (kE == 4)
        *at = make_float4(c[0], c[1], c[2], c[3]);
      else
        *at = make_float4(c[0], c[1], c[0], c[1]);
    }
  }
#pragma unroll
  for (uint32_t i = 0; i < 4; ++i) v[i] = 4 * t + i < k ? v[i] : 0.f;
  {
    const float a = v[0] + v[1], b = v[0] - v[1], c = v[2] + v[3], d = v[2] - v[3];
    v[0] = a + c;
    v[1] = b + d;
    v[2] = a - c;
    v[3] = b - d;
  }
  cross_lane_stage4<1>(v);
  cross_lane_stage4<2>(v);
  cross_lane_stage4<4>(v);
  if (g_log2 > 5) cross_lane_stage4<8>(v);
  if (g_log2 > 6) cross_lane_stage4<16>(v);
  if (g_log2 > 7) cross_lane_stage4<32>(v);
  auto word_of = [](uint32_t c) { return (c >> 5) * 36 + (c & 31); };
  *reinterpret_cast<float4*>(sx + word_of(4 * t)) = make_float4(v[0], v[1], v[2], v[3]);
  nd::lds_barrier();
  if (g_log2 > 8) {  // strides 256, 512, 1024: thread t's values are 256 apart
    if (t < 256) {
      float z[8];
#pragma unroll
      for (uint32_t i = 0; i < 8; ++i) z[i] = sx[word_of(t + 256 * i)];
#pragma unroll
      for (uint32_t st = 1; st < 8; st <<= 1) {
        if ((256u * st) >> g_log2) continue;
#pragma unroll
        for (uint32_t i = 0; i < 8; ++i) {
          if ((i & st) == 0) {
            const float a = z[i], b = z[i + st];
            z[i] = a + b;
            z[i + st] = a - b;
          }
        }
      }
#pragma unroll
      for (uint32_t i = 0; i < 8; ++i) sx[word_of(t + 256 * i)] = z[i];
    }
    nd::lds_barrier();
  }
  float xv[32];
#pragma unroll
  for (int q = 0; q < 8; ++q) {
    const float4 f = *reinterpret_cast<const float4*>(sx + u * 36 + 4 * q);
    xv[4 * q] = f.x;
    xv[4 * q + 1] = f.y;
    xv[4 * q + 2] = f.z;
    xv[4 * q + 3] = f.w;
  }

  const char* mine = reinterpret_cast<const char*>(tab) + (lane % kCopies) * (kE * 4);
  auto row_of = [&](const uint32_t (&codes)[kW], uint32_t norm, uint32_t row)
      __attribute__((always_inline)) {
    float d[kE];
#pragma unroll
    for (int e = 0; e < kE; ++e) d[e] = 0.f;
#pragma unroll
    for (int i = 0; i < kLookups; ++i) {
      const int bit = kLB * i, w = bit >> 5, sh = bit & 31;
      uint32_t b = codes[w] >> sh;
      if constexpr (32 % kLB != 0) {
        if (sh + kLB > 32) b |= codes[w + 1] << (32 - sh);
      }
      const char* at = mine + (b & (kEntries - 1u)) * 256u;
      if constexpr (kE == 4) {
        const float4 f = *reinterpret_cast<const float4*>(at);
        d[0] = fmaf(f.x, xv[4 * i], d[0]);
        d[1] = fmaf(f.y, xv[4 * i + 1], d[1]);
        d[2] = fmaf(f.z, xv[4 * i + 2], d[2]);
        d[3] = fmaf(f.w, xv[4 * i + 3], d[3]);
      } else {
        const float2 f = *reinterpret_cast<const float2*>(at);
        d[0] = fmaf(f.x, xv[2 * i], d[0]);
        d[1] = fmaf(f.y, xv[2 * i + 1], d[1]);
      }
    }
    float dot = d[0] + d[1];
    if constexpr (kE == 4) dot += d[2] + d[3];
    float sum = active ? half_bits_to_float(norm) * dot : 0.f;
    if (tpr > 32) sum = nd::sum_xor<32>(sum);
    if (tpr > 16) sum = nd::sum_xor<16>(sum);
    sum += nd::lane_xor<8>(sum);
    sum += nd::lane_xor<4>(sum);
    sum += nd::lane_xor<2>(sum);
    sum += nd::lane_xor<1>(sum);
    if (u == 0 && row < row_count) y[row] = sum * out_scale;
  };
  for (uint32_t first = own; first < row_count; first += kStreamRows * step) {
    uint32_t cur[kStreamRows][kW], cn[kStreamRows];
#pragma unroll
    for (int r = 0; r < kStreamRows; ++r) {
#pragma unroll
      for (int w = 0; w < kW; ++w) cur[r][w] = raw[r][w];
      cn[r] = nb[r];
    }
    if (first + kStreamRows * step < row_count) load(first + kStreamRows * step);
    if (first + (kStreamRows - 1) * step < row_count) {
#pragma unroll
      for (int r = 0; r < kStreamRows; ++r) row_of(cur[r], cn[r], first + r * step + sub);
    } else {
#pragma unroll
      for (int r = 0; r < kStreamRows; ++r) {
        if (first + r * step >= row_count) break;
        row_of(cur[r], cn[r], first + r * step + sub);
      }
    }
  }
}

using CqStreamFn = void (*)(const uint8_t*, const uint16_t*, Codebook, const float*, bool, float*,
                            uint32_t, uint32_t, uint32_t, uint32_t, uint32_t, uint32_t, uint32_t,
                            uint32_t, float);

CqStreamFn pick_stream(const nd_mat* m) {
  return m->bits == 4   ? &cq_stream_kernel<16>
         : m->bits == 3 ? &cq_stream_kernel<12>
                        : &cq_stream_kernel<8>;
}

Codebook codebook_of(const nd_mat* m) {
  Codebook c{};
  for (int i = 0; i < 16; ++i) c.v[i] = m->cb[i];
  return c;
}

using CqFn = void (*)(const uint8_t*, const uint16_t*, Codebook, const float*, uint32_t, float*,
                      uint32_t, uint32_t, uint32_t, uint32_t, uint32_t, uint32_t, uint32_t,
                      uint32_t, uint32_t, float);

constexpr int kRacc = 8;  // rows per thread: rpp * 8 <= 256 outputs per workgroup
constexpr uint32_t kMaxRotateGroup = 2048;  // 64 lanes of 32 codes
constexpr uint32_t kStreamBlocks = 512;     // two to a CU (64 KB of table each)
constexpr uint64_t kStreamUnits = 131072;

template <int UB, int RACC, bool ROTATE, bool VEC>
CqFn pick_ng(uint32_t g) {
  return g >= 32   ? &cq_matvec_kernel<UB, 1, RACC, ROTATE, VEC>
         : g == 16 ? &cq_matvec_kernel<UB, 2, RACC, ROTATE, VEC>
                   : &cq_matvec_kernel<UB, 4, RACC, ROTATE, VEC>;
}

template <int RACC, bool ROTATE, bool VEC>
CqFn pick_w(const nd_mat* m) {
  return m->bits == 4   ? pick_ng<16, RACC, ROTATE, VEC>(m->g)
         : m->bits == 3 ? pick_ng<12, RACC, ROTATE, VEC>(m->g)
                        : pick_ng<8, RACC, ROTATE, VEC>(m->g);
}

// kRacc rows per thread, or one when kRacc would give the launch fewer than
// 256 workgroups (small matrices: more workgroups, each on fewer rows) and a
// row has at most 64 units.
template <bool ROTATE, bool VEC>
CqFn pick(const nd_mat* m, uint32_t racc) {
  return racc == 1 ? pick_w<1, ROTATE, VEC>(m) : pick_w<kRacc, ROTATE, VEC>(m);
}

}  // namespace

// Geometry checks happened at upload (bits, g a power of two >= 8 with g
// dividing kpad, kpad <= 8192, kpad % 32 == 0).  Rotated inputs are kpad
// wide; columns from k on are zero before the rotation.
hipError_t nd_launch_cq_prepare(const nd_mat* m, const float* x, uint32_t batch, uint32_t x_stride,
                                float* prepared, hipStream_t s) {
  if (batch == 0) return hipSuccess;
  hipLaunchKernelGGL(cq_prepare_kernel, dim3(batch), dim3(kCqThreads), 0, s, x, x_stride, m->k,
                     m->kpad, m->g, 1.0 / std::sqrt((double)m->g), prepared);
  return hipGetLastError();
}

// y[b][r - row_start] for b < batch from x [batch][x_stride].  Groups of
// up to 2048 are rotated inside the matvec (one launch); wider groups are
// rotated by cq_prepare_kernel into `prepared` (kCqPreparedRows rows of
// kCqMaxKpad floats), kCqPreparedRows batch rows at a time.
hipError_t nd_launch_cq_matvec(const nd_mat* m, const float* x, uint32_t batch, uint32_t x_stride,
                               float* prepared, uint32_t row_start, uint32_t row_count, float* y,
                               uint32_t y_stride, hipStream_t s) {
  if (row_count == 0 || batch == 0) return hipSuccess;
  const uint32_t units = m->kpad / 32;
  uint32_t tpr_log2 = 3;  // at least 8 threads per row: rpp * kRacc <= 256 outputs
  while ((1u << tpr_log2) < units) ++tpr_log2;
  const uint32_t rpp = kCqThreads >> tpr_log2;
  // One row per thread keeps a row's threads in one wave (the row sum's
  // butterfly spans T = tpr lanes): rows of at most 64 units.
  const uint32_t racc =
      tpr_log2 <= 6 && (uint64_t)((row_count + rpp * kRacc - 1) / (rpp * kRacc)) * batch < 256
          ? 1u
          : kRacc;
  const uint32_t blocks = (row_count + rpp * racc - 1) / (rpp * racc);
  const bool vec = (m->k & 3) == 0 && (x_stride & 3) == 0 &&
                   (reinterpret_cast<uintptr_t>(x) & 15) == 0;
  if (nd_batch_matvec_fits(m, batch)) {
    // The batched form when it should be a tenth faster: a round of 256
    // workgroups here takes about 1.6 us at kRacc rows a thread and 0.6 at
    // one, 3.3 times that with scalar loads of x (measured at 1536 x 512, 512
    // x 512, 8192 x 512, 4096 x 1024, 16384 x 2048, 4096 x 4096 and 300 x 777,
    // 2 to 300 batch rows: the faster form, or one within a tenth of it, at
    // every point).
    const uint64_t rounds = ((uint64_t)blocks * batch + 255) / 256;
    const float here = (float)rounds * (racc == 1 ? 0.6f : 1.6f) * (vec ? 1.f : 3.3f);
    if (nd_batch_matvec_us(m, row_count, batch) < 0.9f * here)
      return nd_launch_batch_matvec(m, x, batch, x_stride, row_start, row_count, y, y_stride, s,
                                    nullptr);
  }
  uint32_t g_log2 = 0;
  while ((1u << g_log2) < m->g) ++g_log2;
  const uint32_t lanes_per_group = m->g > 32 ? m->g / 32 : 1;
  // The streaming form from 131072 units (8192 x 512: level at 4.9 us, 4096 x
  // 2048: 7.0 against 4.8, 32768 x 2048: 10.5 against 8.2 in 4 bits and 10.7
  // against 8.1 in 2; below, 4096 x 512: 4.7 against 4.9), when the row's threads
  // are at least two thirds in use or x needs scalar loads, which it makes once a
  // workgroup (32768 x 300, 10 of 16: 5.1 against 5.3; 40001 x 777: 13.9 against
  // 7.5).
  uint32_t row_log2 = 4;  // its row sum spans at least 16 lanes
  while ((1u << row_log2) < units) ++row_log2;
  if (batch == 1 && m->g >= 32 && units > 8 && units <= 64 &&
      (uint64_t)row_count * units >= kStreamUnits && (!vec || units * 3 >= 2u << row_log2)) {
    const uint32_t rows_per_block = (kStreamThreads >> row_log2);
    const uint32_t want = (row_count + rows_per_block - 1) / rows_per_block;
    hipLaunchKernelGGL(pick_stream(m), dim3(want < kStreamBlocks ? want : kStreamBlocks),
                       dim3(kStreamThreads), 0, s, m->packed, m->norms, codebook_of(m), x, vec, y,
                       m->k, units, m->kpad >> g_log2, g_log2, m->row_bytes, row_start, row_count,
                       row_log2, (float)(1.0 / std::sqrt((double)m->g)));
    return hipGetLastError();
  }
  if (m->g <= kMaxRotateGroup) {
    const CqFn f = vec ? pick<true, true>(m, racc) : pick<true, false>(m, racc);
    hipLaunchKernelGGL(f, dim3(blocks, batch), dim3(kCqThreads), 0, s, m->packed,
                       m->norms, codebook_of(m), x, x_stride, y, y_stride, m->k, m->kpad, g_log2,
                       m->row_bytes, row_start, row_count, tpr_log2, lanes_per_group,
                       (float)(1.0 / std::sqrt((double)m->g)));
    return hipGetLastError();
  }
  for (uint32_t b0 = 0; b0 < batch; b0 += kCqPreparedRows) {
    const uint32_t nb = batch - b0 < kCqPreparedRows ? batch - b0 : kCqPreparedRows;
    hipError_t e = nd_launch_cq_prepare(m, x + (size_t)b0 * x_stride, nb, x_stride, prepared, s);
    if (e != hipSuccess) return e;
    const CqFn f = pick<false, true>(m, racc);
    hipLaunchKernelGGL(f, dim3(blocks, nb), dim3(kCqThreads), 0, s, m->packed,
                       m->norms, codebook_of(m), prepared, m->kpad, y + (size_t)b0 * y_stride,
                       y_stride, m->k, m->kpad, g_log2, m->row_bytes, row_start, row_count,
                       tpr_log2, 1u, 1.0f);
    e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

hipError_t nd_launch_cq_row(const nd_mat* m, uint32_t row, float* out, hipStream_t s) {
  const double inverse_root = 1.0 / std::sqrt((double)m->g);
  Codebook cb = codebook_of(m);
  if (m->bits == kTernaryBits) {  // Float32Array([-c, 0, c]) with c = 1.2240064 * 1/sqrt(g)
    const float c = (float)(kTernaryCentroid * inverse_root);
    cb.v[0] = 0.f;
    cb.v[1] = c;
    cb.v[2] = 0.f;
    cb.v[3] = -c;
  }
  hipLaunchKernelGGL(cq_row_kernel, dim3(1), dim3(kCqThreads), 0, s, m->packed, m->norms, cb,
                     m->k, m->kpad, m->g, m->bits, m->row_bytes, row, inverse_root, out);
  return hipGetLastError();
}
