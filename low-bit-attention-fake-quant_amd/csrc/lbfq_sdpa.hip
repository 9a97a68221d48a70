// Path A of fake_quant_attention (p_requant=False, attention.py:245-321 of the
// reference) on gfx950: attention over the dequantised Q/K/V, probabilities
// not quantised.
//
// lbfq_sdpa_dequant turns the E4M3 codes of the prepass into the SDPA dtype
// exactly as the reference's dequantisers do (dtype(code * scale),
// quant_triton.py:81-109/180-198/275-298/373-396), adding the V block means
// in that dtype (attention.py:281-286).  lbfq_sdpa_fwd is a flash-style
// attention over those tensors on the 32x32x16 bf16 / fp16 MFMA with fp32
// accumulation:
//
//   no Q smoothing (qk_bias == NULL): SDPA with P in fp32 (attention.py:289-294,
//     "P stays in FP32"): one online-softmax pass; P enters the PV product as
//     two SDPA-dtype terms, its rounding and the (exact) rounding residual
//     rounded once more, i.e. with ~16 of fp32's 24 significant bits;
//   Q smoothing: s = dtype(q_deq . k_deq) * sm_scale + qm[g] . K_s * sm_scale,
//     P = dtype(softmax(s)), O = P V (attention.py:296-319).  Two passes over
//     the keys: the first forms each row's max and sum, the second rounds the
//     normalised P to the SDPA dtype -- the value the reference rounds --
//     before the PV product.  The correction comes in log2 units from lbfq_qmk.
//
// Work decomposition: one wave = 32 queries of one (b, h), NW waves per
// workgroup, 64-key tiles: NW = 8 (256 queries, one workgroup per CU, two
// waves per SIMD) when that makes at least 256 workgroups, else 4 (128
// queries, two workgroups per CU).  The workgroup's threads load each K and
// V^T tile from global memory one tile ahead and stage it in a double-buffered
// LDS area that all its waves read (one barrier per tile).  Scores are
// computed transposed, S^T = K Q^T: lane (i, g) = (lane % 32, lane / 32)
// holds query i and, of each 32-key block, the accumulator rows
// 8 (r / 4) + 4 g + r % 4 (r = 0..15).  K row i of a block is key key_of(i), so
// that those rows are keys 16 (r / 8) + 8 g + r % 8.  The PV product
// O^T = V^T P^T consumes P in that layout: its k-step j of a block contracts
// the keys of registers 8 j .. 8 j + 7, for lane group g the eight consecutive
// keys 16 j + 8 g + {0..7}, one 16-byte piece of a V^T row.
#include <cmath>

#include "lbfq_common.h"
#include "../../include/lbfq.h"

using namespace lbfq;

namespace {

typedef float v16f __attribute__((ext_vector_type(16)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));


constexpr float kLog2e = 1.4426950408889634f;

// C (32x32) += A (32x16) B (16x32): lane (i, g) supplies A[i][8g..8g+7] and
// B[8g..8g+7][i] as 8 packed 16-bit values.
template <int DT>
__device__ __forceinline__ v16f mfma16(const uint4& a, const uint4& b, const v16f& c) {
  if constexpr (DT == kBF16)
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c,
                                                    0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c,
                                                   0, 0, 0);
}

template <int DT>
__device__ __forceinline__ uint32_t to_bits(float x) {
  if constexpr (DT == kBF16) return f32_to_bf16_bits(x);
  else return f32_to_f16_bits(x);
}
template <int DT>
__device__ __forceinline__ float from_bits(uint32_t x) {
  if constexpr (DT == kBF16) return bf16_bits_to_f32(static_cast<uint16_t>(x));
  else return f16_bits_to_f32(static_cast<uint16_t>(x));
}
template <int DT>
__device__ __forceinline__ float round_dt(float x) { return from_bits<DT>(to_bits<DT>(x)); }

// 2^(e - 127) for an E8M0 byte (e = 0 is the subnormal 2^-127)
__device__ __forceinline__ float e8m0_to_f32(uint32_t e) {
  return __uint_as_float(e ? (e << 23) : 0x00400000u);
}

// The four E4M3 codes of a word as fp32 (exact).
__device__ __forceinline__ void decode4(uint32_t w, float* x) {
  x[0] = __builtin_amdgcn_cvt_f32_fp8(static_cast<int>(w), 0);
  x[1] = __builtin_amdgcn_cvt_f32_fp8(static_cast<int>(w), 1);
  x[2] = __builtin_amdgcn_cvt_f32_fp8(static_cast<int>(w), 2);
  x[3] = __builtin_amdgcn_cvt_f32_fp8(static_cast<int>(w), 3);
}

// dtype(code * scale) as the reference's dequantisers round it: the fp32
// product, then RNE (as_f32 keeps the compiler from rounding the exact
// product to fp16 in one step).
template <int DT>
__device__ __forceinline__ uint32_t dequant_bits(float x, float sc) {
  return to_bits<DT>(as_f32(x * sc));
}

__device__ __forceinline__ float xor32_max(float v) { return fmaxf(v, __shfl_xor(v, 32, 64)); }
__device__ __forceinline__ float xor32_add(float v) { return v + __shfl_xor(v, 32, 64); }

struct SdpaArgs {
  int H, S, P;
  float sml2;  // sm_scale * log2(e)
  const uint16_t* q;
  const uint16_t* k;
  const uint16_t* v_t;
  const float* bias;  // (B,H,G,P) log2 units, or null
  int G, q_group;
  void* out;
  int out_dtype;
  const int32_t* out_row_map;
};

// LDS staging of one 64-key tile, shared by the workgroup's waves and
// double-buffered: the K rows (D bf16 each, pitch KP bytes) and the V^T rows
// (64 keys each, pitch VP bytes).  The pitches are 16 bytes past a multiple of
// 128 so that the eight rows one ds_read_b128 phase touches fall on distinct
// banks.
template <int D>
struct Stage {
  static constexpr int KP = 2 * D + 16;
  static constexpr int VP = 2 * 64 + 16;
  static constexpr int KBYTES = 64 * KP;
  static constexpr int BUF = KBYTES + D * VP;
};
// The copies of a tile per thread of an NW-wave workgroup.
template <int D, int NW>
struct Copy {
  static constexpr int T = 64 * NW;           // threads per workgroup
  static constexpr int KCH = 64 * D / 8 / T;  // 16-byte K chunks per thread
  static constexpr int VCH = D * 8 / T;       // 16-byte V^T chunks per thread
};

// global -> registers: the thread's K and V^T chunks of the tile at key0
template <int D, int NW, bool WITH_V>
__device__ __forceinline__ void stage_load(const uint16_t* kbase, const uint16_t* vbase, int P, int key0, int tid,
                                           u32x4 (&kr)[Copy<D, NW>::KCH], u32x4 (&vr)[Copy<D, NW>::VCH]) {
  using C = Copy<D, NW>;
  constexpr int CPR = D / 8;  // K chunks per row
#pragma unroll
  for (int i = 0; i < C::KCH; ++i) {
    const int c = tid + C::T * i, row = c / CPR, col = c % CPR;
    kr[i] = *reinterpret_cast<const u32x4*>(kbase + static_cast<size_t>(key0 + row) * D + 8 * col);
  }
  if constexpr (WITH_V) {
#pragma unroll
    for (int i = 0; i < C::VCH; ++i) {
      const int c = tid + C::T * i, row = c >> 3, kc = c & 7;
      vr[i] = *reinterpret_cast<const u32x4*>(vbase + static_cast<size_t>(row) * P + key0 + 8 * kc);
    }
  }
}

// registers -> LDS buffer
template <int D, int NW, bool WITH_V>
__device__ __forceinline__ void stage_store(uint8_t* buf, int tid, const u32x4 (&kr)[Copy<D, NW>::KCH],
                                            const u32x4 (&vr)[Copy<D, NW>::VCH]) {
  using C = Copy<D, NW>;
  constexpr int CPR = D / 8;
#pragma unroll
  for (int i = 0; i < C::KCH; ++i) {
    const int c = tid + C::T * i, row = c / CPR, col = c % CPR;
    *reinterpret_cast<u32x4*>(buf + row * Stage<D>::KP + 16 * col) = kr[i];
  }
  if constexpr (WITH_V) {
#pragma unroll
    for (int i = 0; i < C::VCH; ++i) {
      const int c = tid + C::T * i, row = c >> 3, kc = c & 7;
      *reinterpret_cast<u32x4*>(buf + Stage<D>::KBYTES + row * Stage<D>::VP + 16 * kc) = vr[i];
    }
  }
}

// Key of K row i of a 32-key block (bits 2 and 3 of i exchanged).
__device__ __forceinline__ int key_of(int i) { return (i & 0x13) | ((i & 4) << 1) | ((i & 8) >> 1); }

// S^T of the staged tile for the lane's query: two 32-key blocks
template <int D, int DT>
__device__ __forceinline__ void scores(const uint8_t* buf, int li, int g, const uint4 (&qop)[D / 16], v16f (&s)[2]) {
  constexpr int NKS = D / 16;
#pragma unroll
  for (int kb = 0; kb < 2; ++kb) {
    const uint8_t* krow = buf + (32 * kb + key_of(li)) * Stage<D>::KP + 16 * g;
    uint4 kop[NKS];
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks) kop[ks] = *reinterpret_cast<const uint4*>(krow + 32 * ks);
#pragma unroll
    for (int r = 0; r < 16; ++r) s[kb][r] = 0.0f;
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks) s[kb] = mfma16<DT>(kop[ks], qop[ks], s[kb]);
  }
}

// log2-unit scores of the lane's 32 keys (register r of block kb is key
// key0 + 32 kb + 16 (r / 8) + 8 g + r % 8); in the tile that holds key S - 1,
// keys >= S are set to -inf.  brow: the correction of the tile's keys for the lane's query
template <bool BIAS, int DT, bool FENCE = true, bool MASK = true>
__device__ __forceinline__ void to_log2(const v16f (&s)[2], int key0, int g, int S, float sml2, const float* brow,
                                        float (&u)[32]) {
  if constexpr (BIAS) {
#pragma unroll
    for (int kb = 0; kb < 2; ++kb) {
#pragma unroll
      for (int q4 = 0; q4 < 4; ++q4) {
        const float4 bv = *reinterpret_cast<const float4*>(brow + 32 * kb + 16 * (q4 >> 1) + 8 * g + 4 * (q4 & 1));
        const float bb[4] = {bv.x, bv.y, bv.z, bv.w};
#pragma unroll
        for (int e = 0; e < 4; ++e)  // the main term rounded to DT first
          u[16 * kb + 4 * q4 + e] = fmaf(round_dt<DT>(s[kb][4 * q4 + e]), sml2, bb[e]);
      }
      // the second block's correction loads stay behind the first block's use
      // (all eight in flight at once took the kernel past 256 VGPRs)
      if constexpr (FENCE) __builtin_amdgcn_sched_barrier(0);
    }
  } else {
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
      for (int r = 0; r < 16; ++r) u[16 * kb + r] = s[kb][r] * sml2;
  }
  if (MASK && key0 + 64 > S) {
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
      for (int r = 0; r < 16; ++r)
        if (key0 + 32 * kb + 16 * (r >> 3) + 8 * g + (r & 7) >= S) u[16 * kb + r] = -INFINITY;
  }
}

// Two fp32 values rounded (RNE) to the SDPA dtype and packed into one word,
// low half the first: one packed conversion.
template <int DT>
__device__ __forceinline__ uint32_t pack2(float a, float b) {
  const f32x2 v = {a, b};
  if constexpr (DT == kBF16) return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2));
  else return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, f16x2));
}
// The two halves of a packed word as fp32 (exact).
template <int DT>
__device__ __forceinline__ float lo_of(uint32_t w) { return from_bits<DT>(w & 0xffffu); }
template <int DT>
__device__ __forceinline__ float hi_of(uint32_t w) {
  if constexpr (DT == kBF16) return __uint_as_float(w & 0xffff0000u);
  else return from_bits<DT>(w >> 16);
}

// The lane's 32 P values (score layout) as packed SDPA-dtype pairs:
// w[kb][j][k] holds registers 16 kb + 8 j + 2 k and + 1.
template <int DT>
__device__ __forceinline__ void pack(const float (&p)[32], uint32_t (&w)[2][2][4]) {
#pragma unroll
  for (int kb = 0; kb < 2; ++kb)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const int r = 16 * kb + 8 * j + 2 * k;
        w[kb][j][k] = pack2<DT>(p[r], p[r + 1]);
      }
}

// P as its SDPA-dtype rounding (whi) plus the rounding's exact residual,
// rounded once more (wlo): p = hi + lo to ~16 significant bits.
template <int DT>
__device__ __forceinline__ void pack_split(const float (&p)[32], uint32_t (&whi)[2][2][4], uint32_t (&wlo)[2][2][4]) {
  pack<DT>(p, whi);
#pragma unroll
  for (int kb = 0; kb < 2; ++kb)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const int r = 16 * kb + 8 * j + 2 * k;
        const uint32_t h = whi[kb][j][k];
        wlo[kb][j][k] = pack2<DT>(p[r] - lo_of<DT>(h), p[r + 1] - hi_of<DT>(h));  // exact differences
      }
}

// O^T (D x 32 queries) += V^T (D x 64 keys) P^T for the staged tile
template <int D, int DT>
__device__ __forceinline__ void pv(const uint8_t* buf, int li, int g, const uint32_t (&w)[2][2][4],
                                   v16f (&acc)[D / 32]) {
  const uint8_t* vb = buf + Stage<D>::KBYTES + li * Stage<D>::VP + 16 * g;
#pragma unroll
  for (int kb = 0; kb < 2; ++kb) {
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const uint4 pb = make_uint4(w[kb][j][0], w[kb][j][1], w[kb][j][2], w[kb][j][3]);
#pragma unroll
      for (int db = 0; db < D / 32; ++db) {
        const uint4 va = *reinterpret_cast<const uint4*>(vb + 32 * db * Stage<D>::VP + 32 * (2 * kb + j));
        acc[db] = mfma16<DT>(va, pb, acc[db]);
      }
    }
  }
}

// Element offset of query qi's output row (its original position).
template <int D>
__device__ __forceinline__ size_t out_base(const SdpaArgs& a, int bh, int qi) {
  const int b = bh / a.H, h = bh - b * a.H;
  const int orow = a.out_row_map ? a.out_row_map[static_cast<size_t>(bh) * a.S + qi] : qi;
  return ((static_cast<size_t>(b) * a.S + orow) * a.H + h) * D;
}

// Four outputs: rounded to the SDPA dtype (the reference's output), then to the caller's dtype.
template <int DT>
__device__ __forceinline__ void store_out(const SdpaArgs& a, size_t at, const float (&v)[4]) {
  float o[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) o[k] = round_dt<DT>(v[k]);
  if (a.out_dtype == kF32) {
    *reinterpret_cast<float4*>(reinterpret_cast<float*>(a.out) + at) = make_float4(o[0], o[1], o[2], o[3]);
    return;
  }
  uint32_t wv[2];
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    const uint32_t lo16 = a.out_dtype == kBF16 ? f32_to_bf16_bits(o[2 * k]) : f32_to_f16_bits(o[2 * k]);
    const uint32_t hi16 = a.out_dtype == kBF16 ? f32_to_bf16_bits(o[2 * k + 1]) : f32_to_f16_bits(o[2 * k + 1]);
    wv[k] = lo16 | (hi16 << 16);
  }
  *reinterpret_cast<uint2*>(reinterpret_cast<uint16_t*>(a.out) + at) = make_uint2(wv[0], wv[1]);
}

// BLDS (qm groups of >= 32 queries, so a wave's queries lie in at most two):
// the correction rows of the tile are staged next to it, one value per lane and
// row, and read back as LDS broadcasts (8 heads x 32760 x 128: 7.73 -> 7.49 ms).
// Smaller groups read them from global memory, eight loads a tile whose latency
// nothing hides.
template <int D, bool BIAS, bool BLDS, int DT, int NW>
__global__ void __launch_bounds__(NW * 64, 2) sdpa_fwd_kernel(const SdpaArgs a) {
  constexpr int NKS = D / 16, NDB = D / 32;
  using St = Stage<D>;
  __shared__ __align__(16) uint8_t lds[2 * St::BUF];
  __shared__ __align__(16) float bias_s[BLDS ? 2 : 1][BLDS ? NW : 1][2][BLDS ? 64 : 1];
  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6;
  const int li = lane & 31, g = lane >> 5;
  constexpr int QB = 32 * NW;  // queries per workgroup
  const int nqb = (a.P + QB - 1) / QB;
  const int bh = blockIdx.x / nqb, qb = blockIdx.x - bh * nqb;
  const int S = a.S, P = a.P;
  // every wave takes part in the staging and the barriers; a wave whose rows
  // are all padding (rows [S, P) of q are zero; rows past the pitch read the
  // last one) computes and stores nothing
  const int qi = qb * QB + wave * 32 + li;

  uint4 qop[NKS];
  {
    const uint16_t* qrow = a.q + (static_cast<size_t>(bh) * P + (qi < P ? qi : P - 1)) * D + 8 * g;
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks) qop[ks] = *reinterpret_cast<const uint4*>(qrow + 16 * ks);
  }
  const float* brow = nullptr;         // the lane's correction row
  const float *b0 = nullptr, *b1 = nullptr;  // the rows of the wave's first and last query
  int bsel = 0;                        // which of the two is the lane's
  if constexpr (BIAS) {
    auto row_of = [&](int q) {
      int grp = (q < S ? q : S - 1) / a.q_group;
      grp = grp < a.G ? grp : a.G - 1;
      return a.bias + (static_cast<size_t>(bh) * a.G + grp) * P;
    };
    brow = row_of(qi);
    const int q0 = __builtin_amdgcn_readfirstlane(qb * QB + wave * 32);
    b0 = row_of(q0);
    b1 = row_of(q0 + 31);
    bsel = brow == b0 ? 0 : 1;
  }
  float br0 = 0.0f, br1 = 0.0f;  // the next tile's correction of key `lane`, rows b0 and b1
  auto bias_load = [&](int key0) {
    if constexpr (BLDS) {
      br0 = b0[key0 + lane];
      br1 = b1[key0 + lane];
    }
  };
  auto bias_store = [&](int slot) {
    if constexpr (BLDS) {
      bias_s[slot][wave][0][lane] = br0;
      bias_s[slot][wave][1][lane] = br1;
    }
  };
  auto bias_tile = [&](int t) -> const float* {
    if constexpr (BLDS) return bias_s[t & 1][wave][bsel];
    else return brow + 64 * t;
  };
  const uint16_t* kbase = a.k + static_cast<size_t>(bh) * P * D;
  const uint16_t* vbase = a.v_t + static_cast<size_t>(bh) * D * P;
  const int nt = (S + 63) / 64;
  u32x4 kr[Copy<D, NW>::KCH], vr[Copy<D, NW>::VCH];

  v16f acc[NDB];
#pragma unroll
  for (int db = 0; db < NDB; ++db)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[db][r] = 0.0f;

  float inv_l = 1.0f;
  if constexpr (BIAS) {
    // pass 1: the row's max and sum (each lane over its own keys, merged at the end)
    float m = -INFINITY, l = 0.0f;
    stage_load<D, NW, false>(kbase, vbase, P, 0, tid, kr, vr);
    bias_load(0);
    stage_store<D, NW, false>(lds, tid, kr, vr);
    bias_store(0);
    stage_load<D, NW, false>(kbase, vbase, P, nt > 1 ? 64 : 0, tid, kr, vr);
    stage_store<D, NW, false>(lds + St::BUF, tid, kr, vr);
    __syncthreads();
    v16f s0[2], s1[2];
    scores<D, DT>(lds, li, g, qop, s0);
    __syncthreads();
    // one tile: its softmax sums beside the products of the next, whose K is
    // staged already (past the last tile they are not used), an MFMA to every 12
    // VALU instructions: 8 heads x 32760 x 128 7.49 -> 7.20 ms.  The same in pass 2
    // gained nothing more, and with four waves it spills.
    auto step = [&](int t, const v16f (&s)[2], v16f (&sn)[2], auto MASK) {
      stage_load<D, NW, false>(kbase, vbase, P, 64 * (t + 2 < nt ? t + 2 : nt - 1), tid, kr, vr);
      bias_load(64 * (t + 1 < nt ? t + 1 : t));
      scores<D, DT>(lds + ((t + 1) & 1) * St::BUF, li, g, qop, sn);
      float u[32];
      to_log2<true, DT, false, MASK>(s, 64 * t, g, S, a.sml2, bias_tile(t), u);
      float tmax = u[0];
#pragma unroll
      for (int j = 1; j < 32; ++j) tmax = fmaxf(tmax, u[j]);
      const float m_new = fmaxf(m, tmax);
      const float ms = m_new == -INFINITY ? 0.0f : m_new;  // a lane whose keys so far are all masked
      float sum = 0.0f;
#pragma unroll
      for (int j = 0; j < 32; ++j) sum += __builtin_amdgcn_exp2f(u[j] - ms);
      l = l * __builtin_amdgcn_exp2f(m - ms) + sum;
      m = m_new;
      if constexpr (!MASK) {
#pragma unroll
        for (int i = 0; i < 2 * NKS; ++i) {
          __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
          __builtin_amdgcn_sched_group_barrier(0x002, 12, 0);
        }
      }
      stage_store<D, NW, false>(lds + (t & 1) * St::BUF, tid, kr, vr);
      bias_store((t + 1) & 1);
      __syncthreads();
    };
    int t = 0;
    for (; t + 2 < nt; t += 2) {
      step(t, s0, s1, std::false_type{});
      step(t + 1, s1, s0, std::false_type{});
    }
    step(t, s0, s1, std::true_type{});
    if (t + 1 < nt) step(t + 1, s1, s0, std::true_type{});
    const float mo = __shfl_xor(m, 32, 64), lo = __shfl_xor(l, 32, 64);
    const float mrow = fmaxf(m, mo);  // finite: key 0 is valid
    const float inv = 1.0f / (l * __builtin_amdgcn_exp2f(m - mrow) + lo * __builtin_amdgcn_exp2f(mo - mrow));
    // pass 2: P = dtype(exp2(u - max) / sum), O = P V
    stage_load<D, NW, true>(kbase, vbase, P, 0, tid, kr, vr);
    bias_load(0);
    stage_store<D, NW, true>(lds, tid, kr, vr);
    bias_store(0);
    __syncthreads();
    for (int t = 0; t < nt; ++t) {
      const uint8_t* buf = lds + (t & 1) * St::BUF;
      v16f s[2];
      scores<D, DT>(buf, li, g, qop, s);
      stage_load<D, NW, true>(kbase, vbase, P, 64 * (t + 1 < nt ? t + 1 : t), tid, kr, vr);
      bias_load(64 * (t + 1 < nt ? t + 1 : t));
      float u[32];
      to_log2<true, DT>(s, 64 * t, g, S, a.sml2, bias_tile(t), u);
#pragma unroll
      for (int j = 0; j < 32; ++j) u[j] = __builtin_amdgcn_exp2f(u[j] - mrow) * inv;
      uint32_t w[2][2][4];
      pack<DT>(u, w);
      pv<D, DT>(buf, li, g, w, acc);
      stage_store<D, NW, true>(lds + ((t + 1) & 1) * St::BUF, tid, kr, vr);  // idle after the last tile
      bias_store((t + 1) & 1);
      __syncthreads();
    }
  } else {
    // online softmax; P as its SDPA-dtype rounding plus the rounded residual
    float m = -INFINITY, l = 0.0f;
    stage_load<D, NW, true>(kbase, vbase, P, 0, tid, kr, vr);
    stage_store<D, NW, true>(lds, tid, kr, vr);
    __syncthreads();
    for (int t = 0; t < nt; ++t) {
      const uint8_t* buf = lds + (t & 1) * St::BUF;
      v16f s[2];
      scores<D, DT>(buf, li, g, qop, s);
      stage_load<D, NW, true>(kbase, vbase, P, 64 * (t + 1 < nt ? t + 1 : t), tid, kr, vr);
      float u[32];
      to_log2<false, DT>(s, 64 * t, g, S, a.sml2, nullptr, u);
      float tmax = u[0];
#pragma unroll
      for (int j = 1; j < 32; ++j) tmax = fmaxf(tmax, u[j]);
      const float m_new = fmaxf(m, xor32_max(tmax));  // finite: key 64 t is valid
      const float alpha = __builtin_amdgcn_exp2f(m - m_new);  // 0 on the first tile
      m = m_new;
      float sum = 0.0f;
#pragma unroll
      for (int j = 0; j < 32; ++j) {
        u[j] = __builtin_amdgcn_exp2f(u[j] - m_new);
        sum += u[j];
      }
      l = l * alpha + sum;
      if (__any(alpha != 1.0f)) {
#pragma unroll
        for (int db = 0; db < NDB; ++db)
#pragma unroll
          for (int r = 0; r < 16; ++r) acc[db][r] *= alpha;
      }
      uint32_t whi[2][2][4], wlo[2][2][4];
      pack_split<DT>(u, whi, wlo);
      pv<D, DT>(buf, li, g, whi, acc);
      pv<D, DT>(buf, li, g, wlo, acc);
      stage_store<D, NW, true>(lds + ((t + 1) & 1) * St::BUF, tid, kr, vr);  // idle after the last tile
      __syncthreads();
    }
    inv_l = 1.0f / xor32_add(l);
  }

  if (qi >= S) return;
  const size_t obase = out_base<D>(a, bh, qi);
#pragma unroll
  for (int db = 0; db < NDB; ++db) {
#pragma unroll
    for (int r4 = 0; r4 < 4; ++r4) {
      float o[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) o[k] = acc[db][4 * r4 + k] * inv_l;
      store_out<DT>(a, obase + 32 * db + 8 * r4 + 4 * g, o);
    }
  }
}

// Small problems: too few 32-query waves to occupy the chip, each a serial
// chain over all its tiles.  Here a workgroup is 32 queries, and its NW waves
// take every NW-th 64-key tile each, reading their operands straight from
// memory (nothing is shared), with the tile's K and V^T loads issued together.
// The partial results meet in LDS: without a correction each wave's row max,
// sum and accumulator, rescaled to the common max; with one, the first pass's
// max and sum meet before the second, which then rounds the same normalised P
// as sdpa_fwd_kernel, and only accumulators are added.
template <int D, bool BIAS, int DT, int NW>
__global__ void __launch_bounds__(NW * 64, 2) sdpa_split_kernel(const SdpaArgs a) {
  constexpr int NKS = D / 16, NDB = D / 32;
  __shared__ __align__(16) float acc_s[NW][D / 4][32][4];  // [wave][4 dims][query]
  __shared__ float m_s[NW][32], l_s[NW][32];
  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int li = lane & 31, g = lane >> 5;
  const int S = a.S, P = a.P;
  const int nqb = (S + 31) / 32;
  const int bh = blockIdx.x / nqb, qb = blockIdx.x - bh * nqb;
  const int qi = qb * 32 + li;  // below the pitch, a multiple of 128
  uint4 qop[NKS];
  {
    const uint16_t* qrow = a.q + (static_cast<size_t>(bh) * P + qi) * D + 8 * g;
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks) qop[ks] = *reinterpret_cast<const uint4*>(qrow + 16 * ks);
  }
  const float* brow = nullptr;
  if constexpr (BIAS) {
    int grp = (qi < S ? qi : S - 1) / a.q_group;
    grp = grp < a.G ? grp : a.G - 1;
    brow = a.bias + (static_cast<size_t>(bh) * a.G + grp) * P;
  }
  const uint16_t* kbase = a.k + static_cast<size_t>(bh) * P * D + key_of(li) * D + 8 * g;
  const uint16_t* vbase = a.v_t + static_cast<size_t>(bh) * D * P + static_cast<size_t>(li) * P + 8 * g;
  const int nt = (S + 63) / 64;
  // V^T operand of k-step j of key block kb, rows 32 db + li
  auto v_load = [&](int t, uint4 (&vr)[2][2][NDB]) {
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int db = 0; db < NDB; ++db)
          vr[kb][j][db] = *reinterpret_cast<const uint4*>(vbase + static_cast<size_t>(32 * db) * P + 64 * t + 32 * kb + 16 * j);
  };
  auto tile_scores = [&](int t, v16f (&s)[2]) {
    uint4 kr[2][NKS];
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
      for (int ks = 0; ks < NKS; ++ks)
        kr[kb][ks] = *reinterpret_cast<const uint4*>(kbase + static_cast<size_t>(64 * t + 32 * kb) * D + 16 * ks);
#pragma unroll
    for (int kb = 0; kb < 2; ++kb) {
#pragma unroll
      for (int r = 0; r < 16; ++r) s[kb][r] = 0.0f;
#pragma unroll
      for (int ks = 0; ks < NKS; ++ks) s[kb] = mfma16<DT>(kr[kb][ks], qop[ks], s[kb]);
    }
  };
  v16f acc[NDB];
#pragma unroll
  for (int db = 0; db < NDB; ++db)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[db][r] = 0.0f;
  auto pv_tile = [&](const uint4 (&vr)[2][2][NDB], const uint32_t (&w)[2][2][4]) {
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const uint4 pb = make_uint4(w[kb][j][0], w[kb][j][1], w[kb][j][2], w[kb][j][3]);
#pragma unroll
        for (int db = 0; db < NDB; ++db) acc[db] = mfma16<DT>(vr[kb][j][db], pb, acc[db]);
      }
  };
  float m = -INFINITY, l = 0.0f;  // this wave's tiles; with a correction, this lane's keys of them
  float scale = 1.0f;             // of this wave's accumulator in the sum over waves
  if constexpr (BIAS) {
    for (int t = wave; t < nt; t += NW) {
      v16f s[2];
      tile_scores(t, s);
      float u[32];
      to_log2<true, DT>(s, 64 * t, g, S, a.sml2, brow + 64 * t, u);
      float tmax = u[0];
#pragma unroll
      for (int j = 1; j < 32; ++j) tmax = fmaxf(tmax, u[j]);
      const float m_new = fmaxf(m, tmax);
      const float ms = m_new == -INFINITY ? 0.0f : m_new;  // a lane whose keys so far are all masked
      float sum = 0.0f;
#pragma unroll
      for (int j = 0; j < 32; ++j) sum += __builtin_amdgcn_exp2f(u[j] - ms);
      l = l * __builtin_amdgcn_exp2f(m - ms) + sum;
      m = m_new;
    }
    // the lane pair, then the waves: a wave without tiles, or a pair whose keys
    // are all masked, has m = -inf and l = 0
    const float mo = __shfl_xor(m, 32, 64), lo = __shfl_xor(l, 32, 64);
    const float mp = fmaxf(m, mo), mps = mp == -INFINITY ? 0.0f : mp;
    const float lp = l * __builtin_amdgcn_exp2f(m - mps) + lo * __builtin_amdgcn_exp2f(mo - mps);
    if (g == 0) { m_s[wave][li] = mp; l_s[wave][li] = lp; }
    __syncthreads();
    float mrow = -INFINITY;
#pragma unroll
    for (int w = 0; w < NW; ++w) mrow = fmaxf(mrow, m_s[w][li]);  // finite: key 0 is valid
    float lrow = 0.0f;
#pragma unroll
    for (int w = 0; w < NW; ++w) lrow += l_s[w][li] * __builtin_amdgcn_exp2f(m_s[w][li] - mrow);
    const float inv = 1.0f / lrow;
    for (int t = wave; t < nt; t += NW) {
      uint4 vr[2][2][NDB];
      v_load(t, vr);
      v16f s[2];
      tile_scores(t, s);
      float u[32];
      to_log2<true, DT>(s, 64 * t, g, S, a.sml2, brow + 64 * t, u);
#pragma unroll
      for (int j = 0; j < 32; ++j) u[j] = __builtin_amdgcn_exp2f(u[j] - mrow) * inv;
      uint32_t w[2][2][4];
      pack<DT>(u, w);
      pv_tile(vr, w);
    }
  } else {
    for (int t = wave; t < nt; t += NW) {
      uint4 vr[2][2][NDB];
      v_load(t, vr);
      v16f s[2];
      tile_scores(t, s);
      float u[32];
      to_log2<false, DT>(s, 64 * t, g, S, a.sml2, nullptr, u);
      float tmax = u[0];
#pragma unroll
      for (int j = 1; j < 32; ++j) tmax = fmaxf(tmax, u[j]);
      const float m_new = fmaxf(m, xor32_max(tmax));
      const float ms = m_new == -INFINITY ? 0.0f : m_new;  // the wave's products so far all overflowed
      const float alpha = __builtin_amdgcn_exp2f(m - ms);  // 0 on the wave's first tile
      m = m_new;
      float sum = 0.0f;
#pragma unroll
      for (int j = 0; j < 32; ++j) {
        u[j] = __builtin_amdgcn_exp2f(u[j] - ms);
        sum += u[j];
      }
      l = l * alpha + sum;
      if (__any(alpha != 1.0f)) {
#pragma unroll
        for (int db = 0; db < NDB; ++db)
#pragma unroll
          for (int r = 0; r < 16; ++r) acc[db][r] *= alpha;
      }
      uint32_t whi[2][2][4], wlo[2][2][4];
      pack_split<DT>(u, whi, wlo);
      pv_tile(vr, whi);
      pv_tile(vr, wlo);
    }
    const float lp = xor32_add(l);
    if (g == 0) { m_s[wave][li] = m; l_s[wave][li] = lp; }
    __syncthreads();
    float mrow = -INFINITY;
#pragma unroll
    for (int w = 0; w < NW; ++w) mrow = fmaxf(mrow, m_s[w][li]);  // finite: wave 0 holds key 0
    float lrow = 0.0f;
#pragma unroll
    for (int w = 0; w < NW; ++w) lrow += l_s[w][li] * __builtin_amdgcn_exp2f(m_s[w][li] - mrow);
    scale = __builtin_amdgcn_exp2f(m - mrow) / lrow;  // 0 for a wave without tiles
  }
#pragma unroll
  for (int db = 0; db < NDB; ++db)
#pragma unroll
    for (int r4 = 0; r4 < 4; ++r4)
      *reinterpret_cast<float4*>(&acc_s[wave][8 * db + 2 * r4 + g][li][0]) =
          make_float4(acc[db][4 * r4] * scale, acc[db][4 * r4 + 1] * scale, acc[db][4 * r4 + 2] * scale,
                      acc[db][4 * r4 + 3] * scale);
  __syncthreads();
  // four dimensions of a query per thread, summed over the waves
  for (int e = tid; e < 8 * D; e += NW * 64) {
    const int q = e % 32, d4 = e / 32, qq = qb * 32 + q;
    if (qq >= S) continue;
    float o[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      const float4 v = *reinterpret_cast<const float4*>(&acc_s[w][d4][q][0]);
      o[0] += v.x; o[1] += v.y; o[2] += v.z; o[3] += v.w;
    }
    store_out<DT>(a, out_base<D>(a, bh, qq) + 4 * d4, o);
  }
}

// ---- dequantisation into the SDPA dtype -----------------------------------------

// Q or K codes (BH, P, D) -> (BH, P, D): rows < S dtype(code * scale), rows >= S zero.
// 8 elements per thread.  qk_mx 0: scale (BH, S / blk) fp32 per blk rows;
// 1: scale (BH, P, D / blk) E8M0 per blk columns.
template <int DT>
__device__ __forceinline__ void qk_dequant(int64_t t, const uint8_t* codes, int qk_mx, const void* scale, int blk,
                                           int64_t BH, int S, int P, int D, uint16_t* out) {
  const int per_row = D / 8;
  if (t >= BH * P * per_row) return;
  const int c8 = static_cast<int>(t % per_row);
  const int64_t rowi = t / per_row;  // bh * P + r
  const int r = static_cast<int>(rowi % P);
  const int64_t bh = rowi / P;
  uint4 o = make_uint4(0, 0, 0, 0);
  if (r < S) {
    float sc;
    if (qk_mx) sc = e8m0_to_f32(reinterpret_cast<const uint8_t*>(scale)[rowi * (D / blk) + (8 * c8) / blk]);
    else sc = reinterpret_cast<const float*>(scale)[bh * (S / blk) + r / blk];
    const uint2 c = reinterpret_cast<const uint2*>(codes)[t];
    float x[8];
    decode4(c.x, x);
    decode4(c.y, x + 4);
    uint32_t w[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) w[k] = dequant_bits<DT>(x[2 * k], sc) | (dequant_bits<DT>(x[2 * k + 1], sc) << 16);
    o = make_uint4(w[0], w[1], w[2], w[3]);
  }
  reinterpret_cast<uint4*>(out)[t] = o;
}

// V^T codes (BH, D, P) -> (BH, D, P): keys < S dtype(dtype(code * scale) + dtype(alpha)),
// keys >= S zero.  8 keys per thread.  v_kind 0: scale (BH, D) fp32; 1: (BH, S / vb)
// fp32; 2: (BH, S / vb, D) E8M0.  alpha: (BH, S / vsb, D) fp32 or null.
template <int DT>
__device__ __forceinline__ void v_dequant_t(int64_t t, const uint8_t* codes_t, int v_kind, const void* scale, int vb,
                                            const float* alpha, int vsb, int64_t BH, int S, int P, int D,
                                            uint16_t* out) {
  const int per_row = P / 8;
  if (t >= BH * D * per_row) return;
  const int k0 = 8 * static_cast<int>(t % per_row);
  const int64_t rowi = t / per_row;  // bh * D + d
  const int d = static_cast<int>(rowi % D);
  const int64_t bh = rowi / D;
  uint4 o = make_uint4(0, 0, 0, 0);
  if (k0 < S) {
    const uint2 c = reinterpret_cast<const uint2*>(codes_t)[t];
    const int nvb = v_kind ? S / vb : 1, nvsb = alpha ? S / vsb : 1;
    // the blocks of keys k0 .. k0 + 7, advanced as the keys cross a boundary
    int sb = v_kind ? k0 / vb : 0, sb_next = v_kind ? (sb + 1) * vb : 0;
    int ab = alpha ? k0 / vsb : 0, ab_next = alpha ? (ab + 1) * vsb : 0;
    float x8[8];
    decode4(c.x, x8);
    decode4(c.y, x8 + 4);
    uint32_t hv[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int k = k0 + e;
      if (v_kind && k >= sb_next) { ++sb; sb_next += vb; }
      if (alpha && k >= ab_next) { ++ab; ab_next += vsb; }
      hv[e] = 0u;
      if (k < S) {
        float sc;
        if (v_kind == 0) sc = reinterpret_cast<const float*>(scale)[rowi];
        else if (v_kind == 1) sc = reinterpret_cast<const float*>(scale)[bh * nvb + sb];
        else sc = e8m0_to_f32(reinterpret_cast<const uint8_t*>(scale)[(bh * nvb + sb) * D + d]);
        uint32_t bits = dequant_bits<DT>(x8[e], sc);
        if (alpha) {
          bits = to_bits<DT>(as_f32(from_bits<DT>(bits) + round_dt<DT>(alpha[(bh * nvsb + ab) * D + d])));
        }
        hv[e] = bits;
      }
    }
    o = make_uint4(hv[0] | (hv[1] << 16), hv[2] | (hv[3] << 16), hv[4] | (hv[5] << 16), hv[6] | (hv[7] << 16));
  }
  reinterpret_cast<uint4*>(out)[t] = o;
}

// Q, K and V^T (grid y: 0, 1, 2; all three have B H P D elements) in one
// launch: a small call is bound by its launches (2 x 1024 x 64: a whole call takes
// 72 us with three here and three more for the Q and K codes and the table of V
// maxima, 60 with one of each kind).
template <int DT>
__global__ void sdpa_dequant_kernel(const lbfq_sdpa_dequant_params p, int64_t BH, int S, int P, int D) {
  const int64_t t = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (blockIdx.y == 2)
    v_dequant_t<DT>(t, p.v_codes_t, p.v_kind, p.v_scale, p.v_block, p.v_alpha, p.v_smooth_block, BH, S, P, D,
                    static_cast<uint16_t*>(p.v_t_out));
  else
    qk_dequant<DT>(t, blockIdx.y ? p.k_codes : p.q_codes, p.qk_mx, blockIdx.y ? p.k_scale : p.q_scale, p.qk_block, BH,
                   S, P, D, static_cast<uint16_t*>(blockIdx.y ? p.k_out : p.q_out));
}

}  // namespace

extern "C" int lbfq_sdpa_dequant(const lbfq_sdpa_dequant_params* p, lbfq_stream_t stream) {
  LBFQ_CHECK_ARG(p, "lbfq_sdpa_dequant: null params");
  LBFQ_CHECK_ARG(p->D == 64 || p->D == 128, "lbfq_sdpa_dequant: D must be 64 or 128");
  LBFQ_CHECK_ARG(p->B > 0 && p->H > 0 && p->S > 0 && p->s_pitch >= p->S && p->s_pitch % 128 == 0,
                 "lbfq_sdpa_dequant: s_pitch must be >= S and a multiple of 128");
  LBFQ_CHECK_ARG(p->s_pitch < (int64_t{1} << 30) && p->B * p->H * p->s_pitch * p->D / 8 < (int64_t{1} << 39),
                 "lbfq_sdpa_dequant: problem too large");
  LBFQ_CHECK_ARG(p->q_codes && p->k_codes && p->v_codes_t && p->q_scale && p->k_scale && p->v_scale,
                 "lbfq_sdpa_dequant: missing codes or scales");
  LBFQ_CHECK_ARG(p->q_out && p->k_out && p->v_t_out, "lbfq_sdpa_dequant: missing output");
  LBFQ_CHECK_ARG(p->sdpa_dtype == kBF16 || p->sdpa_dtype == kF16, "lbfq_sdpa_dequant: the SDPA dtype is bf16 or fp16");
  LBFQ_CHECK_ARG(p->qk_mx ? (p->qk_block >= 8 && p->qk_block <= p->D && (p->qk_block & (p->qk_block - 1)) == 0)
                          : (p->qk_block > 0 && p->S % p->qk_block == 0),
                 "lbfq_sdpa_dequant: bad Q/K block %d", p->qk_block);
  LBFQ_CHECK_ARG(p->v_kind >= 0 && p->v_kind <= 2, "lbfq_sdpa_dequant: bad v_kind %d", p->v_kind);
  LBFQ_CHECK_ARG(p->v_kind == 0 || (p->v_block > 0 && p->S % p->v_block == 0), "lbfq_sdpa_dequant: bad V block %d",
                 p->v_block);
  LBFQ_CHECK_ARG(!p->v_alpha || (p->v_smooth_block > 0 && p->S % p->v_smooth_block == 0),
                 "lbfq_sdpa_dequant: bad V smoothing block %d", p->v_smooth_block);
  hipStream_t st = static_cast<hipStream_t>(stream);
  const int64_t BH = p->B * p->H;
  const int S = static_cast<int>(p->S), P = static_cast<int>(p->s_pitch), D = static_cast<int>(p->D);
  const dim3 grid(static_cast<unsigned>((BH * P * (D / 8) + 255) / 256), 3), block(256);
  if (p->sdpa_dtype == kBF16)
    hipLaunchKernelGGL(sdpa_dequant_kernel<kBF16>, grid, block, 0, st, *p, BH, S, P, D);
  else
    hipLaunchKernelGGL(sdpa_dequant_kernel<kF16>, grid, block, 0, st, *p, BH, S, P, D);
  LBFQ_LAUNCH_CHECK("lbfq_sdpa_dequant");
  return 0;
}

// Up to this many 32-query waves (a quarter of the SIMDs) a problem runs
// sdpa_split_kernel.  Its workgroups each read all of their head's K and V^T,
// so past that the shared tiles win again.  us, shared tiles -> split:
//                      waves   plain           with Q smoothing
//   2 x 1024 x 64         64   20.9 ->  11.8   39.6 ->  18.0
//   2 x 1024 x 128        64   33.0 ->  20.1   41.2 ->  29.8
//   1 x 8192 x 128       256  225   -> 128    310   -> 201
//   4 x 2048 x 128       256   61.1 ->  36.5   82.7 ->  54.6
//   8 x 2048 x 128       512   62.2 ->  94     78.6 -> 133
constexpr int64_t kSplitWaves = 256;

extern "C" int lbfq_sdpa_fwd(const lbfq_sdpa_params* p, lbfq_stream_t stream) {
  LBFQ_CHECK_ARG(p, "lbfq_sdpa_fwd: null params");
  LBFQ_CHECK_ARG(p->D == 64 || p->D == 128, "lbfq_sdpa_fwd: D must be 64 or 128");
  LBFQ_CHECK_ARG(p->B > 0 && p->H > 0 && p->S > 0 && p->s_pitch >= p->S && p->s_pitch % 128 == 0,
                 "lbfq_sdpa_fwd: s_pitch must be >= S and a multiple of 128");
  LBFQ_CHECK_ARG(p->s_pitch < (int64_t{1} << 30) && p->B * p->H * (p->s_pitch / 128) < (int64_t{1} << 31),
                 "lbfq_sdpa_fwd: problem too large");
  LBFQ_CHECK_ARG(p->q && p->k && p->v_t && p->out, "lbfq_sdpa_fwd: missing tensor");
  LBFQ_CHECK_ARG(p->sdpa_dtype == kBF16 || p->sdpa_dtype == kF16, "lbfq_sdpa_fwd: the SDPA dtype is bf16 or fp16");
  LBFQ_CHECK_ARG(p->out_dtype >= kF32 && p->out_dtype <= kBF16, "lbfq_sdpa_fwd: bad output dtype %d", p->out_dtype);
  LBFQ_CHECK_ARG(!p->qk_bias || (p->groups > 0 && p->q_group > 0), "lbfq_sdpa_fwd: bad qm groups");
  SdpaArgs a{};
  a.H = static_cast<int>(p->H);
  a.S = static_cast<int>(p->S);
  a.P = static_cast<int>(p->s_pitch);
  a.sml2 = p->sm_scale * kLog2e;
  a.q = static_cast<const uint16_t*>(p->q);
  a.k = static_cast<const uint16_t*>(p->k);
  a.v_t = static_cast<const uint16_t*>(p->v_t);
  a.bias = p->qk_bias;
  a.G = p->qk_bias ? static_cast<int>(p->groups) : 1;
  a.q_group = p->qk_bias ? p->q_group : 1;
  a.out = p->out;
  a.out_dtype = p->out_dtype;
  a.out_row_map = p->out_row_map;
  // eight-wave workgroups (256 queries, one per CU) where there are enough of
  // them to fill the chip; four-wave ones (two per CU) for small problems
  const int64_t nwg8 = p->B * p->H * ((p->s_pitch + 255) / 256);
  const bool w8 = nwg8 >= 256;
  const dim3 grid(static_cast<unsigned>(w8 ? nwg8 : p->B * p->H * (p->s_pitch / 128))), block(w8 ? 512 : 256);
  hipStream_t st = static_cast<hipStream_t>(stream);
  const bool bias = p->qk_bias != nullptr, bf = p->sdpa_dtype == kBF16;
  // few 32-query waves: eight waves share one's keys (kSplitWaves below)
  const int64_t nw32 = p->B * p->H * ((p->S + 31) / 32);
  if (nw32 <= kSplitWaves && p->S > 64) {
    const dim3 gs(static_cast<unsigned>(nw32)), bs(512);
#define LBFQ_SP(DD, BI)                                                                            \
  do {                                                                                             \
    if (bf) hipLaunchKernelGGL((sdpa_split_kernel<DD, BI, kBF16, 8>), gs, bs, 0, st, a);           \
    else hipLaunchKernelGGL((sdpa_split_kernel<DD, BI, kF16, 8>), gs, bs, 0, st, a);               \
  } while (0)
    if (p->D == 128) { if (bias) LBFQ_SP(128, true); else LBFQ_SP(128, false); }
    else { if (bias) LBFQ_SP(64, true); else LBFQ_SP(64, false); }
#undef LBFQ_SP
    LBFQ_LAUNCH_CHECK("lbfq_sdpa_fwd (split)");
    return 0;
  }
  const bool blds = bias && p->q_group >= 32;
#define LBFQ_SD(DD, BI, BL, DT)                                                             \
  do {                                                                                      \
    if (w8) hipLaunchKernelGGL((sdpa_fwd_kernel<DD, BI, BL, DT, 8>), grid, block, 0, st, a); \
    else hipLaunchKernelGGL((sdpa_fwd_kernel<DD, BI, BL, DT, 4>), grid, block, 0, st, a);    \
  } while (0)
#define LBFQ_SD_DT(DD, BI, BL) \
  if (bf) LBFQ_SD(DD, BI, BL, kBF16); else LBFQ_SD(DD, BI, BL, kF16)
#define LBFQ_SD_BI(DD)                                                                                     \
  if (blds) { LBFQ_SD_DT(DD, true, true); } else if (bias) { LBFQ_SD_DT(DD, true, false); } \
  else { LBFQ_SD_DT(DD, false, false); }
  if (p->D == 128) { LBFQ_SD_BI(128) } else { LBFQ_SD_BI(64) }
#undef LBFQ_SD_BI
#undef LBFQ_SD_DT
#undef LBFQ_SD
  LBFQ_LAUNCH_CHECK("lbfq_sdpa_fwd");
  return 0;
}
