// BLASST tile-skip simulator kernels (gfx950).
//
// The reference simulator (blasst_skip.py:389-654) measures FP8 fake quant +
// whole-tile BLASST skipping on 128-query x 128-key tiles with per-head static
// FP8 scales.  Its semantics, restated here:
//
//   per-head quant    scale_h = max(amax_h / 448, FLT_MIN); deq = e4m3(x / scale) * scale
//                     (blasst_skip.py:278-297)
//   scores            s = (q . k) * sm_scale in fp32 over operands already rounded
//                     to the matmul dtype (blasst_skip.py:477-480, 499-500)
//   block statistics  bmax_j = max over the 128 keys of block j; running max
//                     rm_j = max(rm_{j-1}, bmax_j); final max M = rm_last
//   rungs             exact: p = exp(s - M)                          (:484-491)
//                     online: w = exp(s - rm_j) * exp(rm_j - M)      (:502-519)
//                     static P: pq = e4m3(exp(s - rm_j) * 256) / 256, numerator
//                     pq * exp(rm_j - M), denominator the unquantised w (:526-570)
//                     PV operands rounded to the matmul dtype, fp32 sums
//   tile predicate    tile_margin_j = max over the tile's 128 rows of (bmax_j - rm_j);
//                     keep_j = tile_margin_j >= log(threshold); a tile keeping no
//                     block keeps the first block of largest max-over-rows bmax
//                     (blasst_skip.py:375-386, 584-619)
//
// With bf16 matmul operands the scan and the rungs run on the matrix cores
// (further down).  fp32 operands stay on the kernels here:
//
// Work decomposition: one wave per 64 / LPR query rows of one head, LPR =
// D / 64 lanes per row, each holding 64 dimensions of the row's q and output
// in registers; the lanes of a row read the same key rows at a time, four
// keys' dot products as four independent chains.  The online and static-P
// rungs form each key block's scores once, in the block-max pass, and keep
// them in LDS (32 KB per wave at D = 64, 16 KB at D = 128) for the
// accumulation pass.  Tile statistics are combined across the waves of a
// 128-row tile by ordered-integer atomicMax.
#include <algorithm>

#include "lbfq_common.h"
#include "../../include/lbfq.h"

using namespace lbfq;

namespace {

constexpr int kTileQ = 128;  // query tile / key block (QUERY_TILE, KEY_BLOCK)
constexpr float kDenomFloor = 1e-30f;

__device__ __forceinline__ uint32_t ordered_bits(float f) {
  const uint32_t u = __float_as_uint(f);
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}
__device__ __forceinline__ float from_ordered_bits(uint32_t u) {
  return __uint_as_float((u & 0x80000000u) ? (u & 0x7fffffffu) : ~u);
}
__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
  for (int m = 1; m < 64; m <<= 1) v = fmaxf(v, __shfl_xor(v, m, 64));
  return v;
}
__device__ __forceinline__ float round_bf16(float v) { return bf16_bits_to_f32(f32_to_bf16_bits(v)); }

// ---- per-head static FP8 fake quant --------------------------------------------
template <int DT>
__global__ void __launch_bounds__(256) head_amax_kernel(const void* x, int64_t S, int64_t H, int64_t D,
                                                        uint32_t* amax_bits) {
  const int64_t h = blockIdx.y;
  float m = 0.0f;
  for (int64_t e = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x; e < S * D;
       e += static_cast<int64_t>(gridDim.x) * 256) {
    const int64_t s = e / D, d = e - s * D;
    m = fmaxf(m, fabsf(load_as_f32(x, (s * H + h) * D + d, DT)));
  }
  m = wave_max(m);
  if ((threadIdx.x & 63) == 0) atomicMax(amax_bits + h, __float_as_uint(m));  // m >= 0
}

template <int DT>
__global__ void __launch_bounds__(256) head_quant_kernel(const void* x, int64_t n, int64_t H, int64_t D,
                                                         const uint32_t* amax_bits, float* deq, float* deq_mm,
                                                         int mm_bf16, float* scale_out,
                                                         unsigned long long* counts, double* sqerr) {
  unsigned long long sat = 0, uf = 0;
  double sq = 0.0;
  for (int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x; i < n;
       i += static_cast<int64_t>(gridDim.x) * 256) {
    const int64_t h = (i / D) % H;
    const float sc = fmaxf(__uint_as_float(amax_bits[h]) / kFp8Max, 1.17549435e-38f);
    const float xf = load_as_f32(x, i, DT);
    const float scaled = xf / sc;
    const float q = e4m3_decode(e4m3_encode(scaled));
    const float dq = q * sc;
    if (deq) deq[i] = dq;
    if (deq_mm) deq_mm[i] = mm_bf16 ? round_bf16(dq) : dq;
    sat += fabsf(scaled) > kFp8Max ? 1ull : 0ull;
    uf += (q == 0.0f && scaled != 0.0f) ? 1ull : 0ull;
    const double e = static_cast<double>(dq) - static_cast<double>(xf);
    sq += e * e;
  }
  if (blockIdx.x == 0 && threadIdx.x < H && scale_out)
    scale_out[threadIdx.x] = fmaxf(__uint_as_float(amax_bits[threadIdx.x]) / kFp8Max, 1.17549435e-38f);
#pragma unroll
  for (int m = 1; m < 64; m <<= 1) {
    sat += __shfl_xor(sat, m, 64);
    uf += __shfl_xor(uf, m, 64);
    sq += __shfl_xor(sq, m, 64);
  }
  if ((threadIdx.x & 63) == 0) {
    atomicAdd(counts + 0, sat);
    atomicAdd(counts + 1, uf);
    atomicAdd(sqerr, sq);
  }
}

// ---- scores of one row against key rows ---------------------------------------
// A row's D dimensions are split over LPR = D / 64 lanes (lane l holds
// row l % (64 / LPR), dimensions [l / (64 / LPR) * 64, + 64)), so a lane keeps
// 64 q and 64 output values and D = 128 runs more than one wave per SIMD.
// Each lane's partial dot product is a chain in dimension order; the LPR
// partials are then added (partner lanes l and l ^ 32 form the same sum).
template <int D>
struct Split {
  static constexpr int LPR = D / 64;     // lanes per row
  static constexpr int DL = D / LPR;     // dimensions per lane
  static constexpr int RPW = 64 / LPR;   // rows per wave
};

template <int DL, int LPR>
__device__ __forceinline__ float row_sum(float acc) {
  // lanes l, l ^ (64 / LPR), ... hold the partials of one row; every one of
  // them forms the same sum (pairwise, commutative at each step)
#pragma unroll
  for (int m = 64 / LPR; m < 64; m <<= 1) acc += __shfl_xor(acc, m, 64);
  return acc;
}

template <int DL, int LPR>
__device__ __forceinline__ float dot_part(const float (&q)[DL], const float* krow, float sm_scale) {
  float acc = 0.0f;
#pragma unroll
  for (int d = 0; d < DL; d += 4) {
    const float4 k4 = *reinterpret_cast<const float4*>(krow + d);
    acc = fmaf(q[d], k4.x, acc);
    acc = fmaf(q[d + 1], k4.y, acc);
    acc = fmaf(q[d + 2], k4.z, acc);
    acc = fmaf(q[d + 3], k4.w, acc);
  }
  return row_sum<DL, LPR>(acc) * sm_scale;
}

// dot_part for four consecutive keys (rows `stride` floats apart): four
// independent chains, each in the order of dot_part.
template <int DL, int LPR>
__device__ __forceinline__ void dot_part4(const float (&q)[DL], const float* krow, int64_t stride, float sm_scale,
                                          float (&s)[4]) {
  float a[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int d = 0; d < DL; d += 4) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float4 k4 = *reinterpret_cast<const float4*>(krow + i * stride + d);
      a[i] = fmaf(q[d], k4.x, a[i]);
      a[i] = fmaf(q[d + 1], k4.y, a[i]);
      a[i] = fmaf(q[d + 2], k4.z, a[i]);
      a[i] = fmaf(q[d + 3], k4.w, a[i]);
    }
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    s[i] = row_sum<DL, LPR>(a[i]) * sm_scale;
  }
}

// Pass 1: per row the final max; per (tile, key block) the max over the tile's
// rows of bmax_j - rm_j and of bmax_j.  A workgroup is one 128-row query tile
// (128 / (64 / LPR) waves); 32-key slices of K are staged in LDS, double
// buffered, and every wave reads its key rows from there (the two lane
// halves of a D = 128 wave read two addresses: broadcast reads).
constexpr int kScanKeys = 32;  // keys per staged slice

template <int D>
__global__ void __launch_bounds__(256) scan_kernel(const float* q, const float* k, int64_t S, int64_t H,
                                                   float sm_scale, float* final_max, uint32_t* tile_margin,
                                                   uint32_t* tile_bmax) {
  using SP = Split<D>;
  constexpr int DL = SP::DL, NWV = kTileQ / SP::RPW, NT = 64 * NWV;
  constexpr int F4 = kScanKeys * D / 4 / NT;  // float4 per thread per slice
  __shared__ __align__(16) float ks[2][kScanKeys * D];
  const int64_t h = blockIdx.y;
  const int wave = threadIdx.x / 64, lane = threadIdx.x % 64;
  const int r = lane % SP::RPW, part = lane / SP::RPW;
  const int64_t row = static_cast<int64_t>(blockIdx.x) * kTileQ + wave * SP::RPW + r;
  const int64_t nb = S / kTileQ, mt = blockIdx.x;
  float qr[DL];
#pragma unroll
  for (int d = 0; d < DL; d += 4) {
    const float4 v = *reinterpret_cast<const float4*>(q + (row * H + h) * D + part * DL + d);
    qr[d] = v.x; qr[d + 1] = v.y; qr[d + 2] = v.z; qr[d + 3] = v.w;
  }
  // slice n covers keys [32 n, 32 n + 32); thread chunk i is float4 (tid + NT i)
  // of the slice, key (tid + NT i) / (D / 4)
  typedef float f32x4 __attribute__((ext_vector_type(4)));
  f32x4 kreg[F4];
  const int64_t nslice = S / kScanKeys;
#pragma unroll
  for (int i = 0; i < F4; ++i) {
    const int c = threadIdx.x + NT * i, kk = c / (D / 4), c4 = c % (D / 4);
    kreg[i] = *reinterpret_cast<const f32x4*>(k + (static_cast<int64_t>(kk) * H + h) * D + 4 * c4);
  }
#pragma unroll
  for (int i = 0; i < F4; ++i) *reinterpret_cast<f32x4*>(&ks[0][4 * (threadIdx.x + NT * i)]) = kreg[i];
  __syncthreads();
  float rm = -INFINITY, bmax = -INFINITY;
  for (int64_t n = 0; n < nslice; ++n) {
    {  // slice n + 1 (slice n again after the last), in flight during slice n
      const int64_t key0 = (n + 1 < nslice ? n + 1 : n) * kScanKeys;
#pragma unroll
      for (int i = 0; i < F4; ++i) {
        const int c = threadIdx.x + NT * i, kk = c / (D / 4), c4 = c % (D / 4);
        kreg[i] = *reinterpret_cast<const f32x4*>(k + ((key0 + kk) * H + h) * D + 4 * c4);
      }
    }
    const float* kb = &ks[n & 1][part * DL];
    for (int kk = 0; kk < kScanKeys; kk += 4) {
      float s4[4];
      dot_part4<DL, SP::LPR>(qr, kb + kk * D, D, sm_scale, s4);
#pragma unroll
      for (int i = 0; i < 4; ++i) bmax = fmaxf(bmax, s4[i]);
    }
    if ((n + 1) % (kTileQ / kScanKeys) == 0) {  // the end of key block j
      const int64_t j = n / (kTileQ / kScanKeys);
      rm = fmaxf(rm, bmax);
      const float tm = wave_max(bmax - rm), tb = wave_max(bmax);
      if (lane == 0) {
        const int64_t o = (h * (S / kTileQ) + mt) * nb + j;
        atomicMax(tile_margin + o, ordered_bits(tm));
        atomicMax(tile_bmax + o, ordered_bits(tb));
      }
      bmax = -INFINITY;
    }
    // into the buffer every wave finished reading a slice ago (unread after the last)
#pragma unroll
    for (int i = 0; i < F4; ++i) *reinterpret_cast<f32x4*>(&ks[(n + 1) & 1][4 * (threadIdx.x + NT * i)]) = kreg[i];
    __syncthreads();
  }
  if (part == 0) final_max[h * S + row] = rm;
}

// Tile keep masks for T thresholds, with the empty-tile safeguard.
__global__ void __launch_bounds__(256) keep_kernel(const uint32_t* tile_margin, const uint32_t* tile_bmax,
                                                   int64_t HM, int64_t nb, const float* log_thr, int T,
                                                   uint8_t* keep, unsigned long long* counts) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (i >= HM * T) return;
  const int t = static_cast<int>(i / HM);
  const int64_t hm = i - static_cast<int64_t>(t) * HM;
  const float lt = log_thr[t];
  uint8_t* kp = keep + i * nb;
  const uint32_t* mp = tile_margin + hm * nb;
  const uint32_t* bp = tile_bmax + hm * nb;
  int64_t kept = 0, best = 0;
  float bestv = -INFINITY;
  for (int64_t j = 0; j < nb; ++j) {
    const bool kj = from_ordered_bits(mp[j]) >= lt;
    kp[j] = kj ? 1 : 0;
    kept += kj ? 1 : 0;
    const float bv = from_ordered_bits(bp[j]);
    if (bv > bestv) { bestv = bv; best = j; }
  }
  unsigned long long forced = 0;
  if (kept == 0) {
    kp[best] = 1;
    kept = 1;
    forced = 1;
  }
  atomicAdd(counts + 2 * t, static_cast<unsigned long long>(nb - kept));
  if (forced) atomicAdd(counts + 2 * t + 1, forced);
}

// Pass 2: one rung (exact / online / static P with a tile keep mask).
template <int D, int MODE>
__global__ void __launch_bounds__(64) attend_kernel(const float* q, const float* k, const float* v, int64_t S,
                                                    int64_t H, float sm_scale, int round_p, const float* final_max,
                                                    const uint8_t* keep, float* out, float* dropped,
                                                    unsigned long long* p_counts, double* p_sqerr) {
  using SP = Split<D>;
  constexpr int DL = SP::DL, RPW = SP::RPW;
  // the block's scores of the wave's rows (column r), formed in the block-max
  // pass and read back by the lanes of the same row in the accumulation pass
  __shared__ float sc[MODE != 0 ? kTileQ * RPW : 1];
  const int64_t h = blockIdx.y;
  const int r = threadIdx.x % RPW, part = threadIdx.x / RPW;
  const int64_t row = static_cast<int64_t>(blockIdx.x) * RPW + r;
  const int64_t nb = S / kTileQ, mt = row / kTileQ;
  const int64_t dofs = part * DL;  // this lane's dimensions of q, v and the output row
  float qr[DL], acc[DL];
#pragma unroll
  for (int d = 0; d < DL; d += 4) {
    const float4 x = *reinterpret_cast<const float4*>(q + (row * H + h) * D + dofs + d);
    qr[d] = x.x; qr[d + 1] = x.y; qr[d + 2] = x.z; qr[d + 3] = x.w;
    acc[d] = acc[d + 1] = acc[d + 2] = acc[d + 3] = 0.0f;
  }
  const float fm = final_max[h * S + row];
  const uint8_t* kr = keep ? keep + (h * (S / kTileQ) + mt) * nb : nullptr;
  float den = 0.0f, tot_l = 0.0f, drop_l = 0.0f, rm = -INFINITY;
  unsigned long long uf = 0, cnt = 0;
  double sq = 0.0;
  for (int64_t j = 0; j < nb; ++j) {
    const bool kj = kr ? kr[j] != 0 : true;
    float rescale = 1.0f;
    if (MODE != 0) {
      float bmax = -INFINITY;
      for (int kk = 0; kk < kTileQ; kk += 4) {
        const int64_t key = j * kTileQ + kk;
        float s4[4];
        dot_part4<DL, SP::LPR>(qr, k + (key * H + h) * D + dofs, H * D, sm_scale, s4);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          sc[(kk + i) * RPW + r] = s4[i];  // the LPR lanes of a row store the same value
          bmax = fmaxf(bmax, s4[i]);
        }
      }
      rm = fmaxf(rm, bmax);
      rescale = expf(rm - fm);
    }
    // a skipped block adds nothing; its unquantised mass is still needed for
    // the dropped-mass diagnostic and the P statistics cover all blocks
    if (!kj && !dropped && !p_counts) continue;
    float lb = 0.0f;
    for (int kk = 0; kk < kTileQ; ++kk) {
      const int64_t key = j * kTileQ + kk;
      const float s =
          MODE != 0 ? sc[kk * RPW + r] : dot_part<DL, SP::LPR>(qr, k + (key * H + h) * D + dofs, sm_scale);
      float pw;
      if (MODE == 0) {
        const float p = expf(s - fm);
        den += p;
        pw = p;
      } else {
        const float on = expf(s - rm);
        const float w = on * rescale;
        if (MODE == 1) {
          den += w;
          pw = w;
        } else {
          lb += w;
          const float scaled = on * 256.0f;
          const float pq = e4m3_decode(e4m3_encode(scaled)) * (1.0f / 256.0f);
          if (p_counts && part == 0) {  // once per row
            uf += (pq == 0.0f && scaled != 0.0f) ? 1ull : 0ull;
            cnt += 1;
            const double e = static_cast<double>(pq) - static_cast<double>(on);
            sq += e * e;
          }
          pw = pq * rescale;
        }
      }
      if (!kj) continue;
      if (round_p) pw = round_bf16(pw);
      const float* vrow = v + (key * H + h) * D + dofs;
#pragma unroll
      for (int d = 0; d < DL; d += 4) {
        const float4 v4 = *reinterpret_cast<const float4*>(vrow + d);
        acc[d] = fmaf(pw, v4.x, acc[d]);
        acc[d + 1] = fmaf(pw, v4.y, acc[d + 1]);
        acc[d + 2] = fmaf(pw, v4.z, acc[d + 2]);
        acc[d + 3] = fmaf(pw, v4.w, acc[d + 3]);
      }
    }
    if (MODE == 2) {
      if (kj) den += lb;
      tot_l += lb;
      if (!kj) drop_l += lb;
    }
  }
  const float dn = MODE == 2 ? fmaxf(den, kDenomFloor) : den;
  float* orow = out + (row * H + h) * D + dofs;
#pragma unroll
  for (int d = 0; d < DL; d += 4) {
    float4 o;
    o.x = acc[d] / dn; o.y = acc[d + 1] / dn; o.z = acc[d + 2] / dn; o.w = acc[d + 3] / dn;
    *reinterpret_cast<float4*>(orow + d) = o;
  }
  if (MODE == 2 && dropped && part == 0) dropped[h * S + row] = drop_l / fmaxf(tot_l, kDenomFloor);
  if (MODE == 2 && p_counts) {
#pragma unroll
    for (int m = 1; m < 64; m <<= 1) {
      uf += __shfl_xor(uf, m, 64);
      cnt += __shfl_xor(cnt, m, 64);
      sq += __shfl_xor(sq, m, 64);
    }
    if (threadIdx.x == 0) {
      atomicAdd(p_counts + 0, uf);
      atomicAdd(p_counts + 1, cnt);
      atomicAdd(p_sqerr, sq);
    }
  }
}

// ---- bf16 operands: the matrix-core kernels ------------------------------------------
// With matmul_dtype bf16 every operand of both products is a bf16 value, so the
// 32x32x16 bf16 MFMA forms the same products with fp32 accumulation.  Operands
// are laid out head-major once, q and k as (H, S, D) rows and v transposed,
// (H, D, S), and the scan and each rung run as flash-style kernels over
// 128-key blocks.
//
// One wave owns 32 query rows; lane (li, g) = (lane % 32, lane / 32) holds row
// li and, of each 32-key group, keys 8 (r / 4) + 4 g + r % 4 (r = 0..15: the
// accumulator layout of S^T = K Q^T).  Eight waves share each staged block.  P
// feeds the product O^T = V^T P^T from the score registers: its k-step j of a
// group contracts the keys of registers 8 j .. 8 j + 7, which the staged V^T
// rows hold next to each other (keys 0-3, 8-11, 4-7, 12-15 of a 16-key run).
// The row's final max is known from the scan, so nothing is rescaled.
//
// At 8 heads x 16384 x 128 (0.55 TFLOP a product) the scan takes 0.51 ms, the
// exact and online rungs 1.40 and 1.47, static P 1.73 (2.4 with its statistics,
// whose squared errors are fp64): 1.1 PFLOP/s in the scan, which the MFMAs and
// their LDS reads bound, and 0.6-0.8 in the rungs, which the exponentials and
// conversions bound. The fp32 kernels, bound by FMA issue, took 11, 57, 57
// and 70 ms on the same operands.
//
// The weights are formed from differences of the unscaled scores, which lie
// close together and so differ without a rounding, with sm log2 e as the
// exponent's factor: a score scaled first is off by 2^-24 of itself, as much as
// the products' own error. Mean error of a head against 64-bit arithmetic, 6000
// heads of 1024 and 2048 tokens x 128: 9.2e-6 in the bf16 rung (the fp32 kernels
// 9.2e-6), 9.3e-6 (9.4e-6) with FP8 operands and 1.9e-5 (2.0e-5) with FP8 P;
// scaled first 9.4e-6, 9.6e-6 and 2.0e-5. The FP8 P that round the other way, of
// 3.7e9: 17.5e3 (18.8e3; scaled first 19.1e3).
typedef float v16f __attribute__((ext_vector_type(16)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));

constexpr int kMmWaves = 8, kMmThreads = 64 * kMmWaves, kMmRows = 32 * kMmWaves;

__device__ __forceinline__ v16f mfma_bf16(const u32x4& a, const u32x4& b, const v16f& c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0,
                                                 0);
}
__device__ __forceinline__ uint32_t pack_bf16(float a, float b) {
  const f32x2 v = {a, b};
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2));
}
// v is in a register here: the work that produces it cannot be put off
// (the host pass type-checks device code too and has no "v" registers)
template <typename T>
__device__ __forceinline__ void pin(T& v) {
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile("" : "+v"(v));
#endif
}
// max / sum over the two lanes of a row (v_permlane32_swap: (v[l], v[l ^ 32]) in one order or the other)
__device__ __forceinline__ float pair_max(float v) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float pair_add(float v) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// F exp(c x / log2 e) for x <= 0, c = hi + lo > 0 and F a power of two: exp2 of the
// rounded product x hi, corrected to first order for what the rounding and c's
// low part leave out (v_exp_f32 is good to 1 ulp, the rounded product alone is
// off by |x c| 2^-24).
struct ExpFactor {
  float hi, lo;
};
// log2 e, and sm log2 e for differences of unscaled scores
constexpr ExpFactor kLog2e = {1.44269502f, 1.92596303e-8f};
__device__ __forceinline__ ExpFactor exp_factor(float sm) {
  const double c = static_cast<double>(sm) * 1.4426950408889634;
  const float hi = static_cast<float>(c);
  return {hi, static_cast<float>(c - static_cast<double>(hi))};
}
template <int F>
__device__ __forceinline__ float exp_scaled(float x, ExpFactor c) {
  constexpr float kLn2 = 0.693147182f;
  const float t = x * c.hi;
  const float lo = fmaf(x, c.lo, fmaf(x, c.hi, -t));
  const float e = __builtin_amdgcn_exp2f(t) * static_cast<float>(F);
  const float r = fmaf(e, lo * kLn2, e);
  return e == 0.0f ? 0.0f : r;  // x = -inf: lo is not a number
}

// Staged blocks of 128 keys: K rows (pitch KP bytes) and V^T rows (pitch VP),
// 16 bytes past a multiple of 128 so that the rows a ds_read_b128 phase
// touches fall on distinct banks.
template <int D, bool WITH_V>
struct MmStage {
  static constexpr int KP = 2 * D + 16;
  static constexpr int VP = 2 * kTileQ + 16;
  static constexpr int KBYTES = kTileQ * KP;
  static constexpr int BUF = KBYTES + (WITH_V ? D * VP : 0);
  static constexpr int CH = kTileQ * D / 8 / kMmThreads;  // 16-byte chunks per thread, of K and of V^T
};

template <int D, bool WITH_V>
__device__ __forceinline__ void mm_load(const uint16_t* k, const uint16_t* vt, int64_t S, int64_t key0, int tid,
                                        u32x4 (&kr)[MmStage<D, WITH_V>::CH], u32x4 (&vr)[MmStage<D, WITH_V>::CH]) {
#pragma unroll
  for (int i = 0; i < MmStage<D, WITH_V>::CH; ++i) {
    const int c = tid + kMmThreads * i;
    kr[i] = *reinterpret_cast<const u32x4*>(k + key0 * D + 8 * c);
    if constexpr (WITH_V) vr[i] = *reinterpret_cast<const u32x4*>(vt + (c / 16) * S + key0 + 8 * (c % 16));
  }
}
template <int D, bool WITH_V>
__device__ __forceinline__ void mm_store(uint8_t* buf, int tid, const u32x4 (&kr)[MmStage<D, WITH_V>::CH],
                                         const u32x4 (&vr)[MmStage<D, WITH_V>::CH]) {
  using St = MmStage<D, WITH_V>;
#pragma unroll
  for (int i = 0; i < St::CH; ++i) {
    const int c = tid + kMmThreads * i;
    *reinterpret_cast<u32x4*>(buf + (c / (D / 8)) * St::KP + 16 * (c % (D / 8))) = kr[i];
    if constexpr (WITH_V) {
      const int row = c / 16, kc = c % 16;  // keys 16 (kc / 2) + 8 (kc % 2) + [0, 8)
      uint8_t* p = buf + St::KBYTES + row * St::VP + 2 * (16 * (kc >> 1) + 4 * (kc & 1));
      *reinterpret_cast<u32x2*>(p) = vr[i].xy;
      *reinterpret_cast<u32x2*>(p + 16) = vr[i].zw;
    }
  }
}
// S^T of 32-key group kb of the staged block
template <int D, bool WITH_V>
__device__ __forceinline__ v16f mm_scores(const uint8_t* buf, int kb, int li, int g, const u32x4 (&q)[D / 16]) {
  const uint8_t* krow = buf + (32 * kb + li) * MmStage<D, WITH_V>::KP + 16 * g;
  v16f s;
#pragma unroll
  for (int r = 0; r < 16; ++r) s[r] = 0.0f;
#pragma unroll
  for (int ks = 0; ks < D / 16; ++ks) s = mfma_bf16(*reinterpret_cast<const u32x4*>(krow + 32 * ks), q[ks], s);
  return s;
}
__device__ __forceinline__ float max16(const v16f& s) {
  float m = fmaxf(s[0], s[1]);
#pragma unroll
  for (int r = 2; r < 16; ++r) m = fmaxf(m, s[r]);
  return m;
}
// the work item of this workgroup: consecutive ones of a head on one XCD
__device__ __forceinline__ void mm_item(int nqb, int& h, int& qb) {
  const int n = gridDim.x;
  int w = blockIdx.x;
  if ((n & 7) == 0) w = (w & 7) * (n >> 3) + (w >> 3);
  h = w / nqb;
  qb = w - h * nqb;
}

// Pass 1 on the matrix cores (the statistics of scan_kernel); bound by the MFMAs.
template <int D>
__global__ void __launch_bounds__(kMmThreads, 2) scan_mm_kernel(const uint16_t* q, const uint16_t* k, int64_t S,
                                                                float sm_scale, float* final_max,
                                                                uint32_t* tile_margin, uint32_t* tile_bmax) {
  using St = MmStage<D, false>;
  __shared__ __align__(16) uint8_t lds[2 * St::BUF];
  const int nqb = static_cast<int>((S + kMmRows - 1) / kMmRows);
  int h, qb;
  mm_item(nqb, h, qb);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, li = lane & 31, g = lane >> 5;
  const int64_t row0 = static_cast<int64_t>(qb) * kMmRows + wave * 32;
  const bool live = row0 < S;  // S is a multiple of 128: a wave's rows are all inside or all outside
  const int64_t row = (live ? row0 : 0) + li;
  const int64_t nb = S / kTileQ;
  const uint16_t* kh = k + static_cast<int64_t>(h) * S * D;
  u32x4 qop[D / 16];
#pragma unroll
  for (int ks = 0; ks < D / 16; ++ks)
    qop[ks] = *reinterpret_cast<const u32x4*>(q + (static_cast<int64_t>(h) * S + row) * D + 16 * ks + 8 * g);
  u32x4 kr[St::CH], vr[St::CH];
  mm_load<D, false>(kh, nullptr, S, 0, tid, kr, vr);
  mm_store<D, false>(lds, tid, kr, vr);
  __syncthreads();
  float rm = -INFINITY;
  for (int64_t j = 0; j < nb; ++j) {
    const uint8_t* buf = lds + (j & 1) * St::BUF;
    mm_load<D, false>(kh, nullptr, S, (j + 1 < nb ? j + 1 : j) * kTileQ, tid, kr, vr);
    float m = -INFINITY;
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) m = fmaxf(m, max16(mm_scores<D, false>(buf, kb, li, g, qop)));
    const float bmax = pair_max(m) * sm_scale;  // sm_scale > 0: the max of the scaled scores
    rm = fmaxf(rm, bmax);
    const float tm = wave_max(bmax - rm), tb = wave_max(bmax);
    if (lane == 0 && live) {
      const int64_t o = (static_cast<int64_t>(h) * nb + row0 / kTileQ) * nb + j;
      atomicMax(tile_margin + o, ordered_bits(tm));
      atomicMax(tile_bmax + o, ordered_bits(tb));
    }
    mm_store<D, false>(lds + ((j + 1) & 1) * St::BUF, tid, kr, vr);  // idle after the last block
    __syncthreads();
  }
  if (live && g == 0) final_max[static_cast<int64_t>(h) * S + row] = rm;
}

// Pass 2 on the matrix cores: one rung, as attend_kernel.  Two waves per SIMD
// (one workgroup per CU): the softmax of one overlaps the products of the other.
template <int D, int MODE, bool STATS>
__global__ void __launch_bounds__(kMmThreads, 2)
    attend_mm_kernel(const uint16_t* q, const uint16_t* k, const uint16_t* vt, int64_t S, int64_t H, float sm_scale,
                     const float* final_max, const uint8_t* keep, float* out, float* dropped,
                     unsigned long long* p_counts, double* p_sqerr) {
  using St = MmStage<D, true>;
  constexpr int NDB = D / 32;
  __shared__ __align__(16) uint8_t lds[2 * St::BUF];
  const int nqb = static_cast<int>((S + kMmRows - 1) / kMmRows);
  int h, qb;
  mm_item(nqb, h, qb);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, li = lane & 31, g = lane >> 5;
  const int64_t row0 = static_cast<int64_t>(qb) * kMmRows + wave * 32;
  const bool live = row0 < S;
  const int64_t row = (live ? row0 : 0) + li;
  const int64_t nb = S / kTileQ;
  const uint16_t* kh = k + static_cast<int64_t>(h) * S * D;
  const uint16_t* vh = vt + static_cast<int64_t>(h) * S * D;
  u32x4 qop[D / 16];
#pragma unroll
  for (int ks = 0; ks < D / 16; ++ks)
    qop[ks] = *reinterpret_cast<const u32x4*>(q + (static_cast<int64_t>(h) * S + row) * D + 16 * ks + 8 * g);
  const float fm = final_max[static_cast<int64_t>(h) * S + row];
  const uint8_t* kp = keep ? keep + (static_cast<int64_t>(h) * nb + (live ? row0 : 0) / kTileQ) * nb : nullptr;
  v16f acc[NDB];
#pragma unroll
  for (int db = 0; db < NDB; ++db)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[db][r] = 0.0f;
  // den, tot_l, drop_l: this lane's keys; the lane pair's are added at the end
  float den = 0.0f, tot_l = 0.0f, drop_l = 0.0f, mu = -INFINITY;  // mu: the running max, unscaled
  const ExpFactor ef = exp_factor(sm_scale);
  unsigned uf = 0;  // at most 64 keys of S / 128 blocks
  double sq = 0.0;
  u32x4 kr[St::CH], vr[St::CH];
  mm_load<D, true>(kh, vh, S, 0, tid, kr, vr);
  mm_store<D, true>(lds, tid, kr, vr);
  __syncthreads();
  for (int64_t j = 0; j < nb; ++j) {
    const uint8_t* buf = lds + (j & 1) * St::BUF;
    const bool kj = kp ? kp[j] != 0 : true;  // wave-uniform
    v16f s[4];
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) s[kb] = mm_scores<D, true>(buf, kb, li, g, qop);
    mm_load<D, true>(kh, vh, S, (j + 1 < nb ? j + 1 : j) * kTileQ, tid, kr, vr);
    float rescale = 1.0f;
    if constexpr (MODE != 0) {
      const float m = fmaxf(fmaxf(max16(s[0]), max16(s[1])), fmaxf(max16(s[2]), max16(s[3])));
      mu = fmaxf(mu, pair_max(m));
      rescale = exp_scaled<1>(mu * sm_scale - fm, kLog2e);
    }
    // a skipped block adds nothing; its unquantised mass is still needed for
    // the dropped-mass diagnostic and the P statistics cover all blocks
    if (kj || dropped || STATS) {
      float lb = 0.0f;
      uint32_t w[4][2][4];  // P as bf16 pairs: w[kb][jj][i] holds registers 8 jj + 2 i and + 1 of group kb
      // rescale / 256, and 1 / 256: powers of two aside, the factors of attend_kernel
      const float rs = rescale * (1.0f / 256.0f);
#pragma unroll
      for (int kb = 0; kb < 4; ++kb) {
#pragma unroll
        for (int r = 0; r < 16; r += 2) {
          float p[2];
          if constexpr (MODE == 2) {
            float x[2], sc[2];  // the unscaled difference to the running max, 256 exp of the scaled one
#pragma unroll
            for (int e = 0; e < 2; ++e) {
              x[e] = s[kb][r + e] - mu;
              sc[e] = exp_scaled<256>(x[e], ef);
              lb += sc[e];
            }
            const int code = __builtin_amdgcn_cvt_pk_fp8_f32(sc[0], sc[1], 0, false);
            const f32x2 dq = __builtin_amdgcn_cvt_pk_f32_fp8(code, false);
#pragma unroll
            for (int e = 0; e < 2; ++e) {
              const float d = fminf(dq[e], 480.0f);  // what the software codec decodes a NaN's code to
              if constexpr (STATS) {
                const float on = sc[e] * (1.0f / 256.0f), err = d * (1.0f / 256.0f) - on;  // exact difference
                // exp(x) > 0 down to the smallest denormal, below what v_exp_f32 returns
                uf += static_cast<unsigned>(d == 0.0f) & static_cast<unsigned>(x[e] * sm_scale > -103.972077f);
                sq += static_cast<double>(err) * static_cast<double>(err);
              }
              p[e] = d * rs;
            }
          } else {
#pragma unroll
            for (int e = 0; e < 2; ++e) {
              if constexpr (MODE == 1) p[e] = exp_scaled<1>(s[kb][r + e] - mu, ef) * rescale;
              else p[e] = exp_scaled<1>(fmaf(s[kb][r + e], sm_scale, -fm), kLog2e);
              lb += p[e];
            }
          }
          w[kb][r / 8][(r % 8) / 2] = pack_bf16(p[0], p[1]);
          // eight keys at a time: more in flight does not fit 256 registers
          if (MODE == 2 && r % 8 == 6) {
#pragma unroll
            for (int i = 0; i < 4; ++i) pin(w[kb][r / 8][i]);
            pin(lb);
            if constexpr (STATS) {
              pin(uf);
              pin(sq);
            }
            __builtin_amdgcn_sched_barrier(0);
          }
        }
      }
      if constexpr (MODE == 2) {
        lb *= rs;
        if (kj) den += lb;
        tot_l += lb;
        if (!kj) drop_l += lb;
      } else {
        den += lb;
      }
      if (kj) {
        const uint8_t* vb = buf + St::KBYTES + li * St::VP + 16 * g;
#pragma unroll
        for (int kb = 0; kb < 4; ++kb)
#pragma unroll
          for (int jj = 0; jj < 2; ++jj) {
            const u32x4 pb = {w[kb][jj][0], w[kb][jj][1], w[kb][jj][2], w[kb][jj][3]};
#pragma unroll
            for (int db = 0; db < NDB; ++db)
              acc[db] = mfma_bf16(*reinterpret_cast<const u32x4*>(vb + 32 * db * St::VP + 32 * (2 * kb + jj)), pb,
                                  acc[db]);
          }
      }
    }
    mm_store<D, true>(lds + ((j + 1) & 1) * St::BUF, tid, kr, vr);  // idle after the last block
    __syncthreads();
  }
  if (!live) return;
  den = pair_add(den);
  const float dn = MODE == 2 ? fmaxf(den, kDenomFloor) : den;
  float* orow = out + (row * H + h) * D;
#pragma unroll
  for (int db = 0; db < NDB; ++db)
#pragma unroll
    for (int r4 = 0; r4 < 4; ++r4)
      *reinterpret_cast<float4*>(orow + 32 * db + 8 * r4 + 4 * g) =
          make_float4(acc[db][4 * r4] / dn, acc[db][4 * r4 + 1] / dn, acc[db][4 * r4 + 2] / dn,
                      acc[db][4 * r4 + 3] / dn);
  if constexpr (MODE == 2) {
    if (dropped) {
      const float d = pair_add(drop_l) / fmaxf(pair_add(tot_l), kDenomFloor);
      if (g == 0) dropped[static_cast<int64_t>(h) * S + row] = d;
    }
    if constexpr (STATS) {
      unsigned long long n_uf = uf;
#pragma unroll
      for (int m = 1; m < 64; m <<= 1) {
        n_uf += __shfl_xor(n_uf, m, 64);
        sq += __shfl_xor(sq, m, 64);
      }
      if (lane == 0) {
        atomicAdd(p_counts + 0, n_uf);
        atomicAdd(p_counts + 1, static_cast<unsigned long long>(32 * S));
        atomicAdd(p_sqerr, sq);
      }
    }
  }
}

// Largest |x| of each head (fp32 bits, zeroed before).  A workgroup reads whole
// rows; the D / 8 lanes of a head's piece fold theirs before one LDS atomic.
template <int DT, int D>
__global__ void __launch_bounds__(256) head_amax_rows_kernel(const void* x, int64_t S, int64_t H, uint32_t* amax_bits) {
  __shared__ uint32_t top[256];
  const int per_row = static_cast<int>(H) * (D / 8);
  top[threadIdx.x] = 0u;
  __syncthreads();
  const int64_t rows = (S + gridDim.x - 1) / gridDim.x, r0 = rows * blockIdx.x;
  const int64_t r1 = r0 + rows < S ? r0 + rows : S;
  const int64_t e1 = r1 * per_row;
  for (int64_t e0 = r0 * per_row; e0 < e1; e0 += 256) {
    const int64_t e = e0 + threadIdx.x;
    float m = 0.0f;
    if (e < e1) {
#pragma unroll
      for (int i = 0; i < 8; ++i) m = fmaxf(m, fabsf(load_as_f32(x, 8 * e + i, DT)));
    }
#pragma unroll
    for (int o = 1; o < D / 8; o <<= 1) m = fmaxf(m, __shfl_xor(m, o, 64));
    if (e < e1 && threadIdx.x % (D / 8) == 0) atomicMax(&top[(e / (D / 8)) % H], __float_as_uint(m));  // m >= 0
  }
  __syncthreads();
  for (int h = threadIdx.x; h < H; h += 256) atomicMax(amax_bits + h, top[h]);
}

// One operand for the matrix-core kernels: x (S, H, D) of dtype DT, rounded to
// bf16 (amax_bits null) or fake-quantised per head first (the arithmetic and
// statistics of head_quant_kernel), as (H, S, D) rows or transposed (H, D, S).
// A workgroup takes 64 rows of one head; the transpose goes through LDS.
template <int DT, int D, bool TR>
__global__ void __launch_bounds__(256) mm_operand_kernel(const void* x, int64_t S, int64_t H, const uint32_t* amax_bits,
                                                         uint16_t* out, float* scale_out, unsigned long long* counts,
                                                         double* sqerr) {
  constexpr int PITCH = 64 + 4;  // V^T rows in LDS, in values
  __shared__ uint16_t tr[TR ? D * PITCH : 1];
  const int64_t h = blockIdx.x % H, s0 = (blockIdx.x / H) * 64;
  const bool quant = amax_bits != nullptr;
  const float sc = quant ? fmaxf(__uint_as_float(amax_bits[h]) / kFp8Max, 1.17549435e-38f) : 1.0f;
  if (quant && scale_out && s0 == 0 && threadIdx.x == 0) scale_out[h] = sc;
  unsigned sat = 0, uf = 0;
  double sq = 0.0;
  for (int e = threadIdx.x; e < 64 * (D / 8); e += 256) {
    const int r = e / (D / 8), d0 = 8 * (e % (D / 8));
    if (s0 + r >= S) break;
    uint32_t w[4];
#pragma unroll
    for (int i = 0; i < 8; i += 2) {
      float v[2];
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        const float xf = load_as_f32(x, ((s0 + r) * H + h) * D + d0 + i + k, DT);
        v[k] = xf;
        if (quant) {
          const float scaled = xf / sc;
          const float q = e4m3_decode(e4m3_encode(scaled));
          v[k] = q * sc;
          sat += fabsf(scaled) > kFp8Max ? 1u : 0u;
          uf += (q == 0.0f && scaled != 0.0f) ? 1u : 0u;
          const double err = static_cast<double>(v[k]) - static_cast<double>(xf);
          sq += err * err;
        }
      }
      w[i / 2] = pack_bf16(as_f32(v[0]), as_f32(v[1]));
    }
    if constexpr (TR) {
#pragma unroll
      for (int i = 0; i < 8; ++i) tr[(d0 + i) * PITCH + r] = static_cast<uint16_t>(w[i / 2] >> (16 * (i & 1)));
    } else {
      *reinterpret_cast<uint4*>(out + (h * S + s0 + r) * D + d0) = make_uint4(w[0], w[1], w[2], w[3]);
    }
  }
  if constexpr (TR) {
    __syncthreads();
    const int n = S - s0 < 64 ? static_cast<int>(S - s0) : 64;  // a multiple of 8: S is one of 128
    for (int e = threadIdx.x; e < D * 8; e += 256) {
      const int d = e / 8, k0 = 8 * (e % 8);
      if (k0 >= n) continue;
      const uint16_t* p = tr + d * PITCH + k0;
      const u32x2 a = *reinterpret_cast<const u32x2*>(p), b = *reinterpret_cast<const u32x2*>(p + 4);
      *reinterpret_cast<uint4*>(out + (h * D + d) * S + s0 + k0) = make_uint4(a.x, a.y, b.x, b.y);
    }
  }
  if (quant) {
    unsigned long long n_sat = sat, n_uf = uf;
#pragma unroll
    for (int m = 1; m < 64; m <<= 1) {
      n_sat += __shfl_xor(n_sat, m, 64);
      n_uf += __shfl_xor(n_uf, m, 64);
      sq += __shfl_xor(sq, m, 64);
    }
    if ((threadIdx.x & 63) == 0) {
      if (n_sat) atomicAdd(counts + 0, n_sat);
      if (n_uf) atomicAdd(counts + 1, n_uf);
      atomicAdd(sqerr, sq);
    }
  }
}

__global__ void fill_kernel(uint32_t* p, int64_t n, uint32_t v) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (i < n) p[i] = v;
}

}  // namespace

extern "C" int lbfq_head_fp8_quant(const void* x, int dtype, int64_t S, int64_t H, int64_t D, float* deq,
                                   float* deq_mm, int mm_bf16, float* scale, uint32_t* amax_ws,
                                   int64_t* counts, double* sqerr, lbfq_stream_t stream) {
  LBFQ_CHECK_ARG(x && amax_ws && counts && sqerr, "head_fp8_quant: null pointer");
  LBFQ_CHECK_ARG(dtype == kF32 || dtype == kF16 || dtype == kBF16, "head_fp8_quant: unsupported dtype %d", dtype);
  LBFQ_CHECK_ARG(S > 0 && H > 0 && D > 0 && H <= 256, "head_fp8_quant: bad shape");
  hipStream_t st = static_cast<hipStream_t>(stream);
  hipLaunchKernelGGL(fill_kernel, dim3(static_cast<unsigned>((H + 255) / 256)), dim3(256), 0, st, amax_ws, H, 0u);
  const unsigned gx = static_cast<unsigned>(std::min<int64_t>((S * D + 255) / 256, 1024));
  const int64_t n = S * H * D;
  const unsigned gq = static_cast<unsigned>(std::min<int64_t>((n + 255) / 256, 8192));
  auto* cnt = reinterpret_cast<unsigned long long*>(counts);
#define LBFQ_HQ(DT)                                                                                            \
  do {                                                                                                         \
    hipLaunchKernelGGL(head_amax_kernel<DT>, dim3(gx, static_cast<unsigned>(H)), dim3(256), 0, st, x, S, H, D, \
                       amax_ws);                                                                               \
    hipLaunchKernelGGL(head_quant_kernel<DT>, dim3(gq), dim3(256), 0, st, x, n, H, D, amax_ws, deq, deq_mm,    \
                       mm_bf16, scale, cnt, sqerr);                                                            \
  } while (0)
  if (dtype == kF32) LBFQ_HQ(kF32);
  else if (dtype == kF16) LBFQ_HQ(kF16);
  else LBFQ_HQ(kBF16);
#undef LBFQ_HQ
  LBFQ_LAUNCH_CHECK("head_fp8_quant");
  return 0;
}

extern "C" int lbfq_blasst_scan(const float* q, const float* k, int64_t S, int64_t H, int64_t D, float sm_scale,
                                float* final_max, uint32_t* tile_margin, uint32_t* tile_bmax,
                                lbfq_stream_t stream) {
  LBFQ_CHECK_ARG(q && k && final_max && tile_margin && tile_bmax, "blasst_scan: null pointer");
  LBFQ_CHECK_ARG(D == 64 || D == 128, "blasst_scan: D must be 64 or 128");
  LBFQ_CHECK_ARG(S > 0 && S % kTileQ == 0, "blasst_scan: S must be a positive multiple of %d", kTileQ);
  LBFQ_CHECK_ARG(H > 0 && H < 65536, "blasst_scan: bad H");
  hipStream_t st = static_cast<hipStream_t>(stream);
  const int64_t nt = H * (S / kTileQ) * (S / kTileQ);
  const uint32_t neg_inf = 0x007fffffu;  // ordered bits of -inf
  hipLaunchKernelGGL(fill_kernel, dim3(static_cast<unsigned>((nt + 255) / 256)), dim3(256), 0, st, tile_margin, nt,
                     neg_inf);
  hipLaunchKernelGGL(fill_kernel, dim3(static_cast<unsigned>((nt + 255) / 256)), dim3(256), 0, st, tile_bmax, nt,
                     neg_inf);
  if (D == 128)
    hipLaunchKernelGGL(scan_kernel<128>, dim3(static_cast<unsigned>(S / kTileQ), static_cast<unsigned>(H)),
                       dim3(64 * kTileQ / Split<128>::RPW), 0, st, q, k, S, H, sm_scale, final_max, tile_margin,
                       tile_bmax);
  else
    hipLaunchKernelGGL(scan_kernel<64>, dim3(static_cast<unsigned>(S / kTileQ), static_cast<unsigned>(H)),
                       dim3(64 * kTileQ / Split<64>::RPW), 0, st, q, k, S, H, sm_scale, final_max, tile_margin,
                       tile_bmax);
  LBFQ_LAUNCH_CHECK("blasst_scan");
  return 0;
}

extern "C" int lbfq_blasst_keep(const uint32_t* tile_margin, const uint32_t* tile_bmax, int64_t H, int64_t S,
                                const float* log_thresholds, int T, uint8_t* keep, int64_t* counts,
                                lbfq_stream_t stream) {
  LBFQ_CHECK_ARG(tile_margin && tile_bmax && log_thresholds && keep && counts, "blasst_keep: null pointer");
  LBFQ_CHECK_ARG(T > 0 && S > 0 && S % kTileQ == 0 && H > 0, "blasst_keep: bad shape");
  const int64_t hm = H * (S / kTileQ), nb = S / kTileQ;
  const int64_t n = hm * T;
  hipLaunchKernelGGL(keep_kernel, dim3(static_cast<unsigned>((n + 255) / 256)), dim3(256), 0,
                     static_cast<hipStream_t>(stream), tile_margin, tile_bmax, hm, nb, log_thresholds, T, keep,
                     reinterpret_cast<unsigned long long*>(counts));
  LBFQ_LAUNCH_CHECK("blasst_keep");
  return 0;
}

extern "C" int lbfq_blasst_attend(const lbfq_blasst_attend_params* p, lbfq_stream_t stream) {
  LBFQ_CHECK_ARG(p && p->q && p->k && p->v && p->final_max && p->out, "blasst_attend: null pointer");
  LBFQ_CHECK_ARG(p->D == 64 || p->D == 128, "blasst_attend: D must be 64 or 128");
  LBFQ_CHECK_ARG(p->S > 0 && p->S % kTileQ == 0, "blasst_attend: S must be a positive multiple of %d", kTileQ);
  LBFQ_CHECK_ARG(p->mode >= 0 && p->mode <= 2, "blasst_attend: mode must be 0, 1 or 2");
  LBFQ_CHECK_ARG(p->mode == 2 || (!p->keep && !p->dropped && !p->p_counts),
                 "blasst_attend: keep masks, dropped mass and P statistics need mode 2");
  LBFQ_CHECK_ARG(!p->p_counts || p->p_sqerr, "blasst_attend: p_counts needs p_sqerr");
  hipStream_t st = static_cast<hipStream_t>(stream);
  auto* pc = reinterpret_cast<unsigned long long*>(p->p_counts);
#define LBFQ_ATT(DD, MM)                                                                                          \
  hipLaunchKernelGGL((attend_kernel<DD, MM>), dim3(static_cast<unsigned>(p->S / Split<DD>::RPW),                 \
                     static_cast<unsigned>(p->H)), dim3(64), 0, st, p->q, p->k, p->v, p->S, p->H, p->sm_scale, \
                     p->round_p_bf16, p->final_max, p->keep, p->out, p->dropped, pc, p->p_sqerr)
  if (p->D == 128) {
    if (p->mode == 0) LBFQ_ATT(128, 0);
    else if (p->mode == 1) LBFQ_ATT(128, 1);
    else LBFQ_ATT(128, 2);
  } else {
    if (p->mode == 0) LBFQ_ATT(64, 0);
    else if (p->mode == 1) LBFQ_ATT(64, 1);
    else LBFQ_ATT(64, 2);
  }
#undef LBFQ_ATT
  LBFQ_LAUNCH_CHECK("blasst_attend");
  return 0;
}

extern "C" int lbfq_blasst_operand_bf16(const void* x, int dtype, int64_t S, int64_t H, int64_t D, int quantise,
                                        int transposed, uint16_t* out, float* scale, uint32_t* amax_ws,
                                        int64_t* counts, double* sqerr, lbfq_stream_t stream) {
  LBFQ_CHECK_ARG(x && out, "blasst_operand_bf16: null pointer");
  LBFQ_CHECK_ARG(!quantise || (amax_ws && counts && sqerr), "blasst_operand_bf16: missing statistics");
  LBFQ_CHECK_ARG(dtype == kF32 || dtype == kF16 || dtype == kBF16, "blasst_operand_bf16: unsupported dtype %d", dtype);
  LBFQ_CHECK_ARG(D == 64 || D == 128, "blasst_operand_bf16: D must be 64 or 128");
  LBFQ_CHECK_ARG(S > 0 && S % kTileQ == 0, "blasst_operand_bf16: S must be a positive multiple of %d", kTileQ);
  LBFQ_CHECK_ARG(H > 0 && (!quantise || H <= 256) && H * (S / 64) < (1ll << 31), "blasst_operand_bf16: bad H");
  hipStream_t st = static_cast<hipStream_t>(stream);
  auto* cnt = reinterpret_cast<unsigned long long*>(counts);
  const unsigned gx = static_cast<unsigned>(std::min<int64_t>(S, 1024)), go = static_cast<unsigned>(H * (S / 64));
  if (quantise)
    hipLaunchKernelGGL(fill_kernel, dim3(1), dim3(256), 0, st, amax_ws, H, 0u);
  const uint32_t* am = quantise ? amax_ws : nullptr;
#define LBFQ_OP(DT, DD)                                                                                             \
  do {                                                                                                              \
    if (quantise) hipLaunchKernelGGL((head_amax_rows_kernel<DT, DD>), dim3(gx), dim3(256), 0, st, x, S, H, amax_ws); \
    if (transposed)                                                                                                 \
      hipLaunchKernelGGL((mm_operand_kernel<DT, DD, true>), dim3(go), dim3(256), 0, st, x, S, H, am, out, scale, cnt, \
                         sqerr);                                                                                    \
    else                                                                                                            \
      hipLaunchKernelGGL((mm_operand_kernel<DT, DD, false>), dim3(go), dim3(256), 0, st, x, S, H, am, out, scale,    \
                         cnt, sqerr);                                                                               \
  } while (0)
#define LBFQ_OPD(DT) \
  if (D == 128) LBFQ_OP(DT, 128); else LBFQ_OP(DT, 64)
  if (dtype == kF32) { LBFQ_OPD(kF32); } else if (dtype == kF16) { LBFQ_OPD(kF16); } else { LBFQ_OPD(kBF16); }
#undef LBFQ_OPD
#undef LBFQ_OP
  LBFQ_LAUNCH_CHECK("blasst_operand_bf16");
  return 0;
}

extern "C" int lbfq_blasst_scan_bf16(const uint16_t* q, const uint16_t* k, int64_t S, int64_t H, int64_t D,
                                     float sm_scale, float* final_max, uint32_t* tile_margin, uint32_t* tile_bmax,
                                     lbfq_stream_t stream) {
  LBFQ_CHECK_ARG(q && k && final_max && tile_margin && tile_bmax, "blasst_scan_bf16: null pointer");
  LBFQ_CHECK_ARG(D == 64 || D == 128, "blasst_scan_bf16: D must be 64 or 128");
  LBFQ_CHECK_ARG(S > 0 && S % kTileQ == 0, "blasst_scan_bf16: S must be a positive multiple of %d", kTileQ);
  LBFQ_CHECK_ARG(sm_scale > 0.0f, "blasst_scan_bf16: sm_scale must be positive");
  const int64_t nqb = (S + kMmRows - 1) / kMmRows;
  LBFQ_CHECK_ARG(H > 0 && H < 65536 && H * nqb < (1ll << 31), "blasst_scan_bf16: bad H");
  hipStream_t st = static_cast<hipStream_t>(stream);
  const int64_t nt = H * (S / kTileQ) * (S / kTileQ);
  const uint32_t neg_inf = 0x007fffffu;  // ordered bits of -inf
  const dim3 gf(static_cast<unsigned>((nt + 255) / 256)), grid(static_cast<unsigned>(H * nqb));
  hipLaunchKernelGGL(fill_kernel, gf, dim3(256), 0, st, tile_margin, nt, neg_inf);
  hipLaunchKernelGGL(fill_kernel, gf, dim3(256), 0, st, tile_bmax, nt, neg_inf);
  if (D == 128)
    hipLaunchKernelGGL(scan_mm_kernel<128>, grid, dim3(kMmThreads), 0, st, q, k, S, sm_scale, final_max, tile_margin,
                       tile_bmax);
  else
    hipLaunchKernelGGL(scan_mm_kernel<64>, grid, dim3(kMmThreads), 0, st, q, k, S, sm_scale, final_max, tile_margin,
                       tile_bmax);
  LBFQ_LAUNCH_CHECK("blasst_scan_bf16");
  return 0;
}

extern "C" int lbfq_blasst_attend_bf16(const uint16_t* q, const uint16_t* k, const uint16_t* v_t, int64_t S, int64_t H,
                                       int64_t D, float sm_scale, int mode, const float* final_max,
                                       const uint8_t* keep, float* out, float* dropped, int64_t* p_counts,
                                       double* p_sqerr, lbfq_stream_t stream) {
  LBFQ_CHECK_ARG(q && k && v_t && final_max && out, "blasst_attend_bf16: null pointer");
  LBFQ_CHECK_ARG(D == 64 || D == 128, "blasst_attend_bf16: D must be 64 or 128");
  LBFQ_CHECK_ARG(S > 0 && S % kTileQ == 0, "blasst_attend_bf16: S must be a positive multiple of %d", kTileQ);
  LBFQ_CHECK_ARG(sm_scale > 0.0f, "blasst_attend_bf16: sm_scale must be positive");
  LBFQ_CHECK_ARG(mode >= 0 && mode <= 2, "blasst_attend_bf16: mode must be 0, 1 or 2");
  LBFQ_CHECK_ARG(mode == 2 || (!keep && !dropped && !p_counts),
                 "blasst_attend_bf16: keep masks, dropped mass and P statistics need mode 2");
  LBFQ_CHECK_ARG(!p_counts || p_sqerr, "blasst_attend_bf16: p_counts needs p_sqerr");
  const int64_t nqb = (S + kMmRows - 1) / kMmRows;
  LBFQ_CHECK_ARG(H > 0 && H < 65536 && H * nqb < (1ll << 31), "blasst_attend_bf16: bad H");
  hipStream_t st = static_cast<hipStream_t>(stream);
  auto* pc = reinterpret_cast<unsigned long long*>(p_counts);
  const dim3 grid(static_cast<unsigned>(H * nqb));
#define LBFQ_ATT(DD, MM, ST)                                                                                        \
  hipLaunchKernelGGL((attend_mm_kernel<DD, MM, ST>), grid, dim3(kMmThreads), 0, st, q, k, v_t, S, H, sm_scale,      \
                     final_max, keep, out, dropped, pc, p_sqerr)
#define LBFQ_ATT_D(DD)                       \
  do {                                       \
    if (mode == 0) LBFQ_ATT(DD, 0, false);   \
    else if (mode == 1) LBFQ_ATT(DD, 1, false); \
    else if (pc) LBFQ_ATT(DD, 2, true);      \
    else LBFQ_ATT(DD, 2, false);             \
  } while (0)
  if (D == 128) LBFQ_ATT_D(128);
  else LBFQ_ATT_D(64);
#undef LBFQ_ATT_D
#undef LBFQ_ATT
  LBFQ_LAUNCH_CHECK("blasst_attend_bf16");
  return 0;
}
