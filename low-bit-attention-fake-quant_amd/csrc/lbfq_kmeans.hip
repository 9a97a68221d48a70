// Token k-means reorder for the Q / V reorder (gfx950).
//
// Replaces flash-kmeans batch_kmeans_Euclid (called at kmeans.py:78-81 of the
// reference) and the stable argsort / inverse scatter (kmeans.py:84-87).
// Deterministic Lloyd specification shared with the CPU oracle:
//   init   : centroid j = token j*stride + mix(seed, bh, j) % stride,
//            stride = S / K, mix = splitmix64 finaliser;
//   assign : cn_j = sum_d fmaf(c, c), dot_j = sum_d fmaf(x, c) sequential in d,
//            score_j = fmaf(-2, dot_j, cn_j), first minimum wins;
//   update : fp64 sums per 1024-token chunk in token order, chunks added in
//            order, c = (float)(sum / count), empty clusters keep c;
//   labels : those of the last assign of `iters` rounds.
// A slice whose assignment leaves every label as it was has converged: its
// later rounds would recompute the same centroids and labels exactly, so its
// workgroups skip them (a per-slice flag on the device, no host round trip).
// Within a slice that still moves, most of a round repeats the previous one:
// a token whose label cannot have changed (distance bounds, below) is not read
// again by the assignment, and a chunk whose sums are exact in fp64 is updated
// by the tokens that moved instead of being summed anew.  Both leave every
// label and centroid bit as the rounds above define them.
// The order is a stable counting sort of the labels (argsort stable=True).
#include <mutex>
#include <type_traits>
#include "lbfq_common.h"
#include "../../include/lbfq.h"

using namespace lbfq;

namespace {

constexpr int kChunk = 1024;
constexpr int kMaxD = 128;
constexpr int kMaxKAssign = 64;   // centroids held in LDS by the assign kernel

__device__ __forceinline__ uint64_t kmix(uint64_t seed, uint64_t bh, uint64_t K, uint64_t j) {
  uint64_t z = seed + 0x9E3779B97F4A7C15ull * (bh * K + j + 1ull);
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  return z ^ (z >> 31);
}

// State carried from round to round (all null where the workspace has no room for it).
struct Track {
  float2* ul;           // [BH][S]: distance bounds of each token when it was last assigned (assign_settle)
  float* cum;           // [BH][K]: path length of each centroid so far
  float* delta;         // [BH][K]: its last step
  float* cum_max;       // [2][BH]: sum over the rounds of the longest step, slot it % 2 read by round it
  int32_t* touched;     // [BH][K]: an update changed the cluster's sums since the last centroid pass
  int32_t* exact;       // [BH][nchunk]: every fp64 sum over the chunk's values is exact
  uint8_t* part_label;  // [BH][S]: the labels that the chunk's partial sums stand for
};

__global__ void km_init_kernel(const void* x, int dt, int64_t S, int64_t H, int64_t D, int K, uint64_t seed,
                               float* cent, float* cum) {
  const int64_t bh = blockIdx.x / K;
  const int j = blockIdx.x % K;
  const int64_t b = bh / H, h = bh % H;
  const int64_t stride = S / K;
  const int64_t idx = j * stride + static_cast<int64_t>(kmix(seed, bh, K, j) % static_cast<uint64_t>(stride));
  const int d = threadIdx.x;
  if (d < D) cent[(bh * K + j) * D + d] = load_as_f32(x, ((b * S + idx) * H + h) * D + d, dt);
  if (cum && d == 0) cum[bh * K + j] = 0.0f;
}

// the larger of two finite numbers in one instruction (fmaxf of values the
// compiler cannot trace quiets both first; callers test for NaN themselves)
__device__ __forceinline__ float vmax(float a, float b) { return __builtin_amdgcn_fmed3f(a, b, 3.402823466e38f); }

typedef float v16f __attribute__((ext_vector_type(16)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));

// 8 consecutive elements of dtype DT: as loaded, and as fp32
typedef uint16_t u16x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x1 __attribute__((ext_vector_type(1)));
template <int DT>
struct Raw8 {
  uint4 r[DT == kF32 ? 2 : 1];
  // magnitudes of a word's values: bits without the sign, two 16-bit values side by side
  using Mag = std::conditional_t<DT == kF32, u32x1, u16x2>;
  static __device__ __forceinline__ void range_word(uint32_t w, Mag& big, Mag& small) {
    const Mag a = __builtin_bit_cast(Mag, w & (DT == kF32 ? 0x7fffffffu : 0x7fff7fffu));
    big = __builtin_elementwise_max(big, a);
    const Mag one = 1;
    small = __builtin_elementwise_min(small, static_cast<Mag>(a - one));  // 0 - 1 wraps to the top
  }
  // fold the 8 values into the largest magnitude and the smallest nonzero one, minus 1
  __device__ __forceinline__ void range(Mag& big, Mag& small) const {
#pragma unroll
    for (int k = 0; k < (DT == kF32 ? 2 : 1); ++k) {
      range_word(r[k].x, big, small);
      range_word(r[k].y, big, small);
      range_word(r[k].z, big, small);
      range_word(r[k].w, big, small);
    }
  }
  static __device__ __forceinline__ uint32_t widest(Mag m, bool largest) {
    if constexpr (DT == kF32) return m[0];
    else return largest ? (m[0] > m[1] ? m[0] : m[1]) : (m[0] < m[1] ? m[0] : m[1]);
  }
  __device__ __forceinline__ void load(const void* x, int64_t idx) {
    const uint4* p = reinterpret_cast<const uint4*>(static_cast<const uint8_t*>(x) + idx * (DT == kF32 ? 4 : 2));
    r[0] = p[0];
    if constexpr (DT == kF32) r[1] = p[1];
  }
  __device__ __forceinline__ void to_f32(float (&v)[8]) const {
    const uint32_t w[4] = {r[0].x, r[0].y, r[0].z, r[0].w};
    if constexpr (DT == kF32) {
      const uint32_t w1[4] = {r[1].x, r[1].y, r[1].z, r[1].w};
#pragma unroll
      for (int k = 0; k < 4; ++k) { v[k] = __uint_as_float(w[k]); v[4 + k] = __uint_as_float(w1[k]); }
    } else {
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const uint16_t lo = static_cast<uint16_t>(w[k] & 0xffffu), hi = static_cast<uint16_t>(w[k] >> 16);
        if constexpr (DT == kBF16) { v[2 * k] = bf16_bits_to_f32(lo); v[2 * k + 1] = bf16_bits_to_f32(hi); }
        else { v[2 * k] = f16_bits_to_f32(lo); v[2 * k + 1] = f16_bits_to_f32(hi); }
      }
    }
  }
};

template <int DT>
__device__ __forceinline__ void load8(const void* x, int64_t idx, float (&v)[8]) {
  Raw8<DT> r;
  r.load(x, idx);
  r.to_f32(v);
}

// v = hi + lo + r with hi = bf16(v), lo = bf16(v - hi), |r| <= 2^-18 |v|
// (v - hi is exact; both roundings to nearest)
__device__ __forceinline__ void split8(const float (&v)[8], bf16x8& hi, bf16x8& lo) {
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    hi[i] = static_cast<__bf16>(v[i]);
    lo[i] = static_cast<__bf16>(v[i] - static_cast<float>(hi[i]));
  }
}

// ---- assignment ------------------------------------------------------------------
// The labels of the specification (first minimum of fmaf(-2, dot_j, cn_j) over
// sequential fp32 FMA chains), found on the matrix cores and settled exactly
// where they cannot decide.
//
// A wave takes 32 tokens.  v_mfma_f32_32x32x16_bf16 forms
// a_j = dot_j - cn_j / 2 for 32 centroids at a time (rows: centroids, read as
// hi / lo bf16 pairs from LDS; columns: tokens, straight from global memory --
// bf16 tokens are exact, fp16 / fp32 ones are split in hi + lo as well).  The
// largest a_j belongs to the smallest score.  With X = |x|_2 and
// C = max_j |c_j|_2 (so sum_d |x_d c_d| <= X C), the errors of a_j are at most
//   the specification's own chain    2^-17 X C       (128 FMA roundings)
//   its last rounding                2^-24 (X C + C^2 / 2)
//   operands split in two            2^-18 X C       (3 * 2^-18 X C when x is split too: the
//                                                     residuals of both and the lo * lo term)
//   accumulation                     2^-20 (X C + C^2 / 2) per MFMA: 16, or 24 with x split
//   the centroid's number            2^-17 (X C + C^2 / 2): it replaces a_j's last six bits,
//                                    so that the largest a_j names its centroid
// the accumulation at twice the largest error of an MFMA measured on a gfx950
// relative to the magnitudes it adds (2^-21.4 over operands of mixed magnitude,
// 2^-23 over operands of one).  Twice their sum is below 1.25 * 2^-14 X C +
// 2^-15 C^2 (2^-13 and 2^-14 with x split): two centroids whose a_j are further
// apart than that gap are in the specification's order.  A token with another
// centroid within the gap of its best -- or with a gap that is not finite, as
// any non-finite or overflowing product makes it -- is settled by the
// specification itself.  Where two centroids are near, the usual case,
// the token waits for the end of the segment: there a wave runs the FMA chains
// of 32 waiting tokens, one lane for each of their two centroids (a chain is
// ~4000 cycles of latency; run where each token turned up, one or two of 32,
// they doubled the kernel's time).  Any more, and one lane per centroid runs
// the chains at once.
//
// At 40 x 32768 x 128 bf16 (335 MB, 62 us as reads alone in this pattern) the
// first round takes 112 us with 32 clusters, and a full one 108 to 122 with 64;
// one token per lane against LDS broadcasts, bound by its FMA issue, took 196
// and 345.  The rest is latency before the first tokens (centroids, bounds,
// lists), and that is what a late round with few open tokens takes: 28 us there,
// 13 at 12 x 8192.  A step issues three VALU instructions per centroid and token
// pair of lanes (number in, second, first); with separate passes for the
// maximum, the near mask and the runner-up it issued eight and took 15% longer
// with 64 clusters.
constexpr int kAsgWaves = 8;
constexpr int kAsgThreads = 64 * kAsgWaves;
constexpr int kSlab = 32 * kAsgWaves;  // tokens per slab: one 32-token step of each wave
constexpr int kSeg = 8;                // slabs of a segment at most

// Below every a_j where c2max is finite: |c_j|^2 < 1e38 then, and a finite gap
// bounds x.c by X C < 2^64, so a_j > -0.51e38.  From 1e38 on c2max is infinite,
// no gap is finite and every token takes the full settle.
constexpr float kNeverWins = -1e38f;

template <int D, int MB>
struct AssignLds {
  static constexpr int P = D + 4;  // row pitch of the fp32 centroids: float4 reads of 16 rows hit distinct banks
  uint4 part[2][D / 16][MB][64];   // hi / lo operands, as the lanes read them
  float cent[32 * MB * P];
  float cn[32 * MB];
  float a0[32 * MB];               // -cn / 2, the MFMA accumulators' start; kNeverWins for rows that never win
  float c2max;                     // >= max_j |c_j|^2; infinity from -kNeverWins on, or if a centroid is not finite
  uint64_t twins;                  // centroids that a later row repeats
};

// The largest of the lanes' values, which are not negative; infinity if one is not finite.
__device__ __forceinline__ float wave_top(float v) {
  v = v < INFINITY ? v : INFINITY;
#pragma unroll
  for (int m = 1; m < 64; m <<= 1) v = fmaxf(v, __shfl_xor(v, m, 64));
  return v;
}

// The centroids of slice bh into LDS: fp32 rows, hi / lo MFMA operands and the
// norms (the specification's chain).  Rows K .. 32 MB - 1 are zero with norm
// +inf, so they never win; nor does a row that repeats an earlier one bit by
// bit, as its scores are the earlier row's and the first minimum wins.  Repeats
// are what a padded sequence brings (its pad tokens are one row, and an initial
// centroid is every S / K-th token): left in, they tie in every round, and each
// pad token takes the full settle: a round over 8 x 512 x 128 with 140 tokens of
// padding took 50 us with 32 clusters and 97 with 64, against 11 and 14 here.
template <int D, int MB>
__device__ __forceinline__ void assign_fill(AssignLds<D, MB>& lds, const float* cent, int K) {
  using L = AssignLds<D, MB>;
  constexpr int C8 = D / 8;
  for (int e = threadIdx.x; e < 32 * MB * C8; e += kAsgThreads) {
    const int j = e / C8, c8 = e % C8;
    float v[8] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
    if (j < K) load8<kF32>(cent, j * D + 8 * c8, v);
    float4* row = reinterpret_cast<float4*>(lds.cent + j * L::P + 8 * c8);
    row[0] = make_float4(v[0], v[1], v[2], v[3]);
    row[1] = make_float4(v[4], v[5], v[6], v[7]);
    bf16x8 hi, lo;
    split8(v, hi, lo);
    lds.part[0][c8 / 2][j / 32][j % 32 + 32 * (c8 & 1)] = __builtin_bit_cast(uint4, hi);
    lds.part[1][c8 / 2][j / 32][j % 32 + 32 * (c8 & 1)] = __builtin_bit_cast(uint4, lo);
  }
  __syncthreads();
  if (threadIdx.x < 64) {  // one wave
    const int j = threadIdx.x < 32 * MB ? threadIdx.x : 0;
    const uint4* row = reinterpret_cast<const uint4*>(lds.cent + j * L::P);
    float acc = 0.0f;
#pragma unroll 8
    for (int i = 0; i < D / 4; ++i) {
      const float4 v = __builtin_bit_cast(float4, row[i]);
      acc = fmaf(v.x, v.x, acc);
      acc = fmaf(v.y, v.y, acc);
      acc = fmaf(v.z, v.z, acc);
      acc = fmaf(v.w, v.w, acc);
    }
    const bool real = static_cast<int>(threadIdx.x) < K;
    // the first row of this norm, then whether all of it is the same
    const int bits = __float_as_int(acc);
    int first = j;
    for (int jo = K - 1; jo >= 0; --jo) first = __builtin_amdgcn_readlane(bits, jo) == bits && jo < first ? jo : first;
    bool repeat = real && first < j;
    if (__any(repeat)) {
      const uint4* row0 = reinterpret_cast<const uint4*>(lds.cent + first * L::P);
      uint32_t diff = 0u;
#pragma unroll 8
      for (int i = 0; i < D / 4; ++i) {
        const uint4 v = row[i], v0 = row0[i];
        diff |= (v.x ^ v0.x) | (v.y ^ v0.y) | (v.z ^ v0.z) | (v.w ^ v0.w);
      }
      repeat = repeat && diff == 0u;
    }
    uint64_t twins = 0ull;
    for (uint64_t m = __ballot(repeat); m; m &= m - 1)
      twins |= 1ull << __builtin_amdgcn_readlane(first, __builtin_ctzll(m));
    float c2max = wave_top(real ? acc : 0.0f);
    c2max = c2max < -kNeverWins ? c2max : INFINITY;
    if (threadIdx.x < 32 * MB) {
      lds.cn[j] = real && !repeat ? acc : INFINITY;
      lds.a0[j] = real && !repeat ? -0.5f * acc : kNeverWins;
    }
    if (threadIdx.x == 0) {
      lds.c2max = c2max;
      lds.twins = twins;
    }
  }
  __syncthreads();
}

// v of lane l ^ 32, on the VALU (v_permlane32_swap exchanges the upper half of
// its first operand with the lower half of its second)
__device__ __forceinline__ uint32_t from_pair(uint32_t v, int g) {
  const auto r = __builtin_amdgcn_permlane32_swap(v, v, false, false);
  return g ? r[0] : r[1];
}
__device__ __forceinline__ float from_pair(float v, int g) {
  return __uint_as_float(from_pair(__float_as_uint(v), g));
}

// The specification for one token (its row at element x0) per PER lanes: lane
// j of the group runs centroid j's chain; returns the label in every lane of
// the group.  A NaN score never wins, and if nothing does the label is 0.
template <int D, int DT, int MB>
__device__ __forceinline__ int assign_exact(const AssignLds<D, MB>& lds, const void* x, int64_t x0, int lane) {
  constexpr int PER = 32 * MB;
  const int j = lane % PER;
  const float* c = lds.cent + j * AssignLds<D, MB>::P;
  float dot = 0.0f;
#pragma unroll 1
  for (int d = 0; d < D; d += 8) {
    float xv[8];
    load8<DT>(x, x0 + d, xv);
    const float4 c0 = *reinterpret_cast<const float4*>(c + d), c1 = *reinterpret_cast<const float4*>(c + d + 4);
    dot = fmaf(xv[0], c0.x, dot);
    dot = fmaf(xv[1], c0.y, dot);
    dot = fmaf(xv[2], c0.z, dot);
    dot = fmaf(xv[3], c0.w, dot);
    dot = fmaf(xv[4], c1.x, dot);
    dot = fmaf(xv[5], c1.y, dot);
    dot = fmaf(xv[6], c1.z, dot);
    dot = fmaf(xv[7], c1.w, dot);
  }
  float sc = fmaf(-2.0f, dot, lds.cn[j]);
  int best = j;
  if (!(sc < INFINITY)) { sc = INFINITY; best = 0; }
#pragma unroll
  for (int m = 1; m < PER; m <<= 1) {
    const float so = __shfl_xor(sc, m, 64);
    const int bo = __shfl_xor(best, m, 64);
    if (so < sc || (so == sc && bo < best)) { sc = so; best = bo; }
  }
  return best;
}

// The specification between centroids j0 < j1 of a token: lane l runs the chain
// of j0 and lane l ^ 32 that of j1 (j: this lane's); both return the label.
// The token's gap is finite, so both rows are real ones (kNeverWins) and both
// scores are finite.
template <int D, int DT, int MB>
__device__ __forceinline__ int assign_pair(const AssignLds<D, MB>& lds, const void* x, int64_t x0, int j) {
  const float* c = lds.cent + j * AssignLds<D, MB>::P;
  float dot = 0.0f;
#pragma unroll 4
  for (int d = 0; d < D; d += 8) {
    float xv[8];
    load8<DT>(x, x0 + d, xv);
    const float4 c0 = *reinterpret_cast<const float4*>(c + d), c1 = *reinterpret_cast<const float4*>(c + d + 4);
    dot = fmaf(xv[0], c0.x, dot);
    dot = fmaf(xv[1], c0.y, dot);
    dot = fmaf(xv[2], c0.z, dot);
    dot = fmaf(xv[3], c0.w, dot);
    dot = fmaf(xv[4], c1.x, dot);
    dot = fmaf(xv[5], c1.y, dot);
    dot = fmaf(xv[6], c1.z, dot);
    dot = fmaf(xv[7], c1.w, dot);
  }
  const float sc = fmaf(-2.0f, dot, lds.cn[j]);
  const float so = __shfl_xor(sc, 32, 64);
  const int jo = __shfl_xor(j, 32, 64);
  return so < sc || (so == sc && jo < j) ? jo : j;
}

// ---- distance bounds (Hamerly, "Making k-means even faster", SDM 2010) -------------
// With every assignment a token keeps u >= |x - c_label| and
// l <= min over the other centroids of |x - c_j|.  A later round's centroids
// lie at most their path length away, so with cum[j] the length of centroid
// j's path and cmax the sum over the rounds of the longest step,
//   |x - c_label| <= u + (cum[label] - cum[label] then),
//   |x - c_j|     >= l - (cmax - cmax then);
// u - cum and l + cmax are what is stored.  While the squared distances stay
// further apart than twice the error of the specification's fp32 scores
// (2^-16 X C + 2^-17 C^2 each, X <= u + C), the label is what the
// specification would choose again, and the token's row is not read.  All
// roundings are taken outwards by 2^-18 relative, 50 times their size; the sums
// over the rounds, however many, are rounded up as they grow (add_up), so that
// no difference of two of them is short of the path between.
constexpr float kOut = 0x1p-18f;

// a + b or more, for a, b >= 0 (a step below half a last bit of the path so far counts too)
__device__ __forceinline__ float add_up(float a, float b) {
  const float s = a + b;
  return fmaf(s, 0x1p-22f, s);
}

// label still certain: (st.x, st.y) the stored pair, cum and cmax of now, c >= max_j |c_j|
__device__ __forceinline__ bool bounds_hold(float2 st, float cum, float cmax, float c) {
  const float u = st.x + cum + kOut * (fabsf(st.x) + cum);
  const float l = st.y - cmax - kOut * (fabsf(st.y) + cmax);
  const float thr = 0x1p-14f * (u + c) * c + 0x1p-15f * c * c + 0x1p-120f;
  return l > u && (l - u) * (l + u) > thr;  // false for NaN
}

// Grid: any number of workgroups; each takes a contiguous share of the
// BH * ceil(S / kSlab) slabs (two workgroups per CU and equal shares: no
// partial last wave of workgroups), up to kSeg slabs of one slice at a time,
// refilling LDS when the slice changes.  From the second round on it first
// lists the segment's tokens whose bounds no longer hold, and its waves take
// 32 of the list at a time.
// prev_changed: the flags of the previous round (NULL in the first round);
// changed: this round's flags, set to 1 for a slice in which some label
// changed.  They are zero on entry from the second round on; in the first
// round every label counts as changed, so every slice's flag is written.
// it: the round.
template <int D, int DT, int MB>
__global__ void __launch_bounds__(kAsgThreads, 4)
    km_assign_kernel(const void* x, int64_t BH, int64_t S, int64_t H, int K, const float* cent, int32_t* labels,
                     const int32_t* prev_changed, int32_t* changed, const Track tr, int it) {
  constexpr int NKS = D / 16;
  constexpr bool XSPLIT = DT != kBF16;
  constexpr float kGapXC = XSPLIT ? 0x1p-13f : 1.25f * 0x1p-14f, kGapCC = XSPLIT ? 0x1p-14f : 0x1p-15f;
  __shared__ AssignLds<D, MB> lds;
  __shared__ float cum_s[32 * MB];
  __shared__ uint16_t list_s[kSeg * kSlab];  // the segment's tokens to assign
  __shared__ uint32_t pend_s[kSeg * kSlab];  // tokens between two centroids: token | j0 << 16 | j1 << 24
  __shared__ int nlist_s, npend_s;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int li = lane & 31, g = lane >> 5;
  const uint64_t lt_mask = lane == 0 ? 0ull : (~0ull >> (64 - lane));
  const int64_t nslab = (S + kSlab - 1) / kSlab, total = BH * nslab;
  const int64_t w0 = total * blockIdx.x / gridDim.x, w1 = total * (blockIdx.x + 1) / gridDim.x;
  const bool filter = tr.ul && prev_changed;
  int64_t cur = -1;
  float c2max = 0.0f, cmax = 0.0f;  // >= max_j |c_j|^2; the slice's cum_max of this round
  uint64_t twins = 0ull;
  for (int64_t w = w0; w < w1;) {
    const int64_t bh = w / nslab, s_in = w - bh * nslab;
    int64_t ns = w1 - w < kSeg ? w1 - w : kSeg;
    ns = nslab - s_in < ns ? nslab - s_in : ns;
    w += ns;
    if (prev_changed && prev_changed[bh] == 0) continue;  // converged slice (uniform per workgroup)
    if (bh != cur) {
      if (cur >= 0) __syncthreads();  // every wave is done with the previous slice's centroids
      assign_fill<D, MB>(lds, cent + bh * K * D, K);
      cur = bh;
      c2max = lds.c2max;
      twins = lds.twins;
      if (tr.ul) {
        if (static_cast<int>(threadIdx.x) < K) cum_s[threadIdx.x] = tr.cum[bh * K + threadIdx.x];
        cmax = 0.0f;
        if (prev_changed)
          cmax = add_up(tr.cum_max[(it & 1) * BH + bh], wave_top(lane < K ? tr.delta[bh * K + lane] : 0.0f));
        if (s_in == 0 && threadIdx.x == 0) tr.cum_max[((it + 1) & 1) * BH + bh] = cmax;
        __syncthreads();
      }
    }
    const int64_t base = s_in * kSlab;  // the segment's first token
    const int n = static_cast<int>(S - base < ns * kSlab ? S - base : ns * kSlab);
    int32_t* const lab = labels + bh * S + base;
    int nl = n;  // tokens to assign
    __syncthreads();  // every wave is done with the previous lists
    if (threadIdx.x == 0) { nlist_s = 0; npend_s = 0; }
    __syncthreads();
    if (filter) {
      const float c = 1.001f * sqrtf(c2max);
      const float2* ul = tr.ul + bh * S + base;
      // kLd tokens' loads in flight per thread
      constexpr int kLd = 4;
      for (int i0 = 0; i0 < n; i0 += kLd * kAsgThreads) {
        float2 st[kLd];
        int lb[kLd];
#pragma unroll
        for (int q = 0; q < kLd; ++q) {
          int i = i0 + q * kAsgThreads + static_cast<int>(threadIdx.x);
          i = i < n ? i : n - 1;
          st[q] = ul[i];
          lb[q] = lab[i];
        }
#pragma unroll
        for (int q = 0; q < kLd; ++q) {
          const int i = i0 + q * kAsgThreads + static_cast<int>(threadIdx.x);
          const bool need = i < n && !bounds_hold(st[q], cum_s[lb[q]], cmax, c);
          const uint64_t m = __ballot(need);
          int at = 0;
          if (lane == 0 && m) at = atomicAdd(&nlist_s, __popcll(m));
          at = __builtin_amdgcn_readfirstlane(at);
          if (need) list_s[at + __popcll(m & lt_mask)] = static_cast<uint16_t>(i);
        }
      }
      __syncthreads();
      nl = nlist_s;
    }
    const int64_t b = bh / H, h = bh - b * H;
    const int64_t xseg = ((b * S + base) * H + h) * D;
    // token operands: lane (li, g) holds dimensions 16 ks + 8 g + [0, 8) of its
    // token.  The next step's are loaded once this step's MFMAs have read them;
    // tokens that are split (fp16, fp32) GK k-steps at a time as they are used,
    // to stay under 128 registers.
    constexpr bool AHEAD = !XSPLIT;
    constexpr int GK = AHEAD ? NKS : DT == kF16 || MB == 1 ? NKS / 2 : 2;
    Raw8<DT> raw[GK];
    auto token_of = [&](int p0) -> int {
      const int p = p0 + li < nl ? p0 + li : nl - 1;  // lanes past the end repeat the last token
      return filter ? list_s[p] : p;
    };
    auto load_raw = [&](int i, int k0) {
      const int64_t x0 = xseg + static_cast<int64_t>(i) * H * D;
#pragma unroll
      for (int q = 0; q < GK; ++q) raw[q].load(x, x0 + 16 * (k0 + q) + 8 * g);
    };
    bool moved = false;
    int p0 = wave * 32;
    int i = p0 < nl ? token_of(p0) : 0;
    if (AHEAD && p0 < nl) load_raw(i, 0);
    while (p0 < nl) {
      // the centroid operands are read from LDS in every step: kept in registers
      // across steps they do not fit
      asm volatile("" ::: "memory");
      const bool valid = p0 + li < nl;
      float xx = 0.0f;
      v16f a[MB];
#pragma unroll
      for (int m = 0; m < MB; ++m)
#pragma unroll
        for (int r = 0; r < 16; ++r) a[m][r] = lds.a0[32 * m + 8 * (r >> 2) + 4 * g + (r & 3)];
#pragma unroll 1
      for (int k0 = 0; k0 < NKS; k0 += GK) {
        if constexpr (!AHEAD) load_raw(i, k0);
#pragma unroll
        for (int q = 0; q < GK; ++q) {
          const int ks = k0 + q;
          bf16x8 xh, xl;
          if constexpr (XSPLIT) {
            float v[8];
            raw[q].to_f32(v);
            split8(v, xh, xl);
#pragma unroll
            for (int e = 0; e < 8; ++e) xx = fmaf(v[e], v[e], xx);
          } else {
            xh = __builtin_bit_cast(bf16x8, raw[q].r[0]);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              const bf16x2 pr = {xh[2 * e], xh[2 * e + 1]};
              xx = __builtin_amdgcn_fdot2_f32_bf16(pr, pr, xx, false);
            }
          }
#pragma unroll
          for (int m = 0; m < MB; ++m) {
            const bf16x8 ch = __builtin_bit_cast(bf16x8, lds.part[0][ks][m][lane]);
            const bf16x8 cl = __builtin_bit_cast(bf16x8, lds.part[1][ks][m][lane]);
            a[m] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ch, xh, a[m], 0, 0, 0);
            a[m] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(cl, xh, a[m], 0, 0, 0);
            if constexpr (XSPLIT) a[m] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ch, xl, a[m], 0, 0, 0);
          }
        }
        if constexpr (AHEAD) {
          // operand reads kAheadLds MFMAs ahead of their use: read as late as the
          // register allocator likes, every MFMA waited for its LDS latency
          constexpr int kAheadLds = 3;
          __builtin_amdgcn_sched_group_barrier(0x100, 4 * MB + kAheadLds, 0);
#pragma unroll
          for (int q = 0; q < 2 * MB * GK; ++q) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
          }
        }
      }
      const int p_next = p0 + 32 * kAsgWaves;
      const int i_next = token_of(p_next);  // past the end: the last token again, unused
      if constexpr (AHEAD) load_raw(i_next, 0);
      xx += from_pair(xx, g);
      // X C and C^2 from above: 2^-110 covers squares lost to underflow, 1.001 the roundings of the norms
      const float xc = __builtin_amdgcn_sqrtf((xx + 0x1p-110f) * (c2max + 0x1p-110f));
      const float gap = 1.001f * (kGapXC * xc + kGapCC * c2max) + 0x1p-120f;
      const bool finite = gap < INFINITY;  // then every a_j is
      // the two largest, each with its centroid's row in the last six bits
      float top = -INFINITY, second = -INFINITY;
#pragma unroll
      for (int m = 0; m < MB; ++m)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const float v = __uint_as_float((__float_as_uint(a[m][r]) & ~63u) | (32 * m + 8 * (r >> 2) + (r & 3)));
          second = __builtin_amdgcn_fmed3f(top, second, v);
          top = vmax(top, v);
        }
      top = __uint_as_float(__float_as_uint(top) | 4 * g);
      const float top_o = from_pair(top, g), second_o = from_pair(second, g);
      second = vmax(fminf(top, top_o), vmax(second, second_o));
      top = vmax(top, top_o);
      const bool settled = finite && top - second > gap;
      int bj = __float_as_uint(top) & 63;
      int cnt = 1, j0 = 0, j1 = 0;  // near centroids, the first and the last of them
      if (__any(!settled)) {
        const float thr = top - gap;
        uint32_t near_m = 0u;  // bit 16 m + r: centroid 32 m + 8 (r / 4) + 4 g + r % 4 is near
#pragma unroll
        for (int m = 0; m < MB; ++m)
#pragma unroll
          for (int r = 0; r < 16; ++r) near_m |= !(a[m][r] < thr) ? 1u << (16 * m + r) : 0u;
        auto row_of = [&](int bit) -> int { return 2 * (bit & ~3) + (bit & 3) + 4 * g; };
        const int lo = near_m ? row_of(__builtin_ctz(near_m)) : 64, hi = near_m ? row_of(31 - __builtin_clz(near_m)) : 0;
        j0 = min(lo, static_cast<int>(from_pair(static_cast<uint32_t>(lo), g)));
        j1 = max(hi, static_cast<int>(from_pair(static_cast<uint32_t>(hi), g)));
        const uint32_t n = __popc(near_m);
        cnt = settled ? 1 : static_cast<int>(n + from_pair(n, g));
        // one near (the numbers in the last bits can hide that), or all are suspect: the full settle
        if (!settled && (cnt < 2 || !finite)) cnt = 64;
      }
      uint32_t open = static_cast<uint32_t>(__ballot(cnt > 2 && valid));
      while (open) {  // two tokens at a time with up to 32 centroids
        const int t0 = __builtin_ctz(open);
        open &= open - 1;
        int t1 = t0;
        if (MB == 1 && open) {
          t1 = __builtin_ctz(open);
          open &= open - 1;
        }
        const int ti = __shfl(i, MB == 1 && lane >= 32 ? t1 : t0, 64);
        const int le = assign_exact<D, DT, MB>(lds, x, xseg + static_cast<int64_t>(ti) * H * D, lane);
        const int l0 = __builtin_amdgcn_readlane(le, 0), l1 = __builtin_amdgcn_readlane(le, 32);
        if (li == t0) bj = l0;
        else if (li == t1) bj = l1;
      }
      const bool pair = cnt == 2 && valid && lane < 32;
      const uint64_t pm = __ballot(pair);
      if (pm) {
        int at = 0;
        if (lane == 0) at = atomicAdd(&npend_s, __popcll(pm));
        at = __builtin_amdgcn_readfirstlane(at);
        if (pair) pend_s[at + __popcll(pm & lt_mask)] = static_cast<uint32_t>(i | j0 << 16 | j1 << 24);
      }
      if (lane < 32 && valid && cnt != 2) {
        const int32_t old = prev_changed ? lab[i] : -1;
        lab[i] = bj;
        moved |= old != bj;
      }
      if (tr.ul && lane < 32 && valid) {
        // |x - c_j|^2 = |x|^2 - 2 a_j, with twice the error of a_j (and that of
        // the stored norms) below the gap and that of |x|^2 below 2^-15 of it
        const float e = gap + 0x1p-15f * xx;
        float2 st = make_float2(INFINITY, 0.0f);  // never holds
        if (settled && !(twins >> bj & 1)) {  // a repeat of the label's centroid is as near as that, and may part from it
          st.x = __builtin_amdgcn_sqrtf(fmaxf(xx - 2.0f * top, 0.0f) + e) * (1.0f + kOut) - cum_s[bj];
          st.y = __builtin_amdgcn_sqrtf(fmaxf(xx - 2.0f * second - e, 0.0f)) * (1.0f - kOut) + cmax;
        }
        tr.ul[bh * S + base + i] = st;
      }
      p0 = p_next;
      i = i_next;
    }
    __syncthreads();
    const int np = npend_s;
    for (int q0 = wave * 32; q0 < np; q0 += 32 * kAsgWaves) {
      const bool valid = q0 + li < np;
      const uint32_t e = pend_s[valid ? q0 + li : np - 1];
      const int t = e & 0xffff;
      const int bj = assign_pair<D, DT, MB>(lds, x, xseg + static_cast<int64_t>(t) * H * D, e >> (16 + 8 * g) & 0xff);
      if (valid && g == 0) {
        const int32_t old = prev_changed ? lab[t] : -1;
        lab[t] = bj;
        moved |= old != bj;
      }
    }
    // one store per wave and segment: all slices' flags share a few cache lines
    if (__any(moved) && lane == 0) changed[bh] = 1;
  }
}

// ---- update -------------------------------------------------------------------------
// fp64 per-cluster column sums of one kChunk-token chunk.  The chunk's tokens
// are first sorted by label in LDS, stably (ballot ranks within a wave, waves
// and rounds in token order), so a cluster's tokens keep their order.  Then
// wave g -- D / 64 columns a lane -- adds the runs of clusters j = g, g + 8, ...
// in that order: the token-order fp64 sums of the specification, with kPf rows
// in flight.  A whole wave to a row, because clusters are uneven: the pad
// tokens of a short sequence are one cluster.  With 8 columns a lane and 16 lanes
// to a cluster, 512 tokens with 240 of them padding waited for one chain of 30
// batches of 8 rows, 45 us a round against 19 (first round 70 against 31).
//
// The first round also finds out whether the chunk's sums are exact: values
// are multiples of the smallest nonzero one's last bit, and a sum of up to
// 2^12 of them stays below 2^12 times the bound of the largest, so if that
// span fits fp64's 53 bits no addition rounds and the order does not matter
// (bf16 normal data spans ~25 of the 33 exponents this leaves).  In an exact
// chunk a later round adds and subtracts only the tokens whose label differs
// from the one the partial sums stand for -- the same bits as summing anew --
// unless more than a quarter of the chunk moved.
//
// Bound by the row reads and the LDS sort ahead of them: at 40 x 32768 x 128
// bf16 with 32 clusters the first round (the ranges included) takes 90 us, the
// later ones 58, 24, 17, then 16 to 14 as fewer tokens move; with 64 clusters 113,
// 83, 54, then 47 to 39 (16 lanes to a cluster: 125, 67, 31, 18, 14, and every
// round 132 us with one column and a 2-byte load per lane and no moves).
//
// Where one chunk is the slice, `cent` is not null and the centroids follow at
// once: with a pass of its own ten rounds over 2 x 512 x 128 (272 tokens and
// padding) take 387 us, 303 so.
constexpr int kUpdThreads = 512;
constexpr int kMaxMoved = kChunk / 4;

// the length of a centroid's step, from above; s: the sum of its squares
__device__ __forceinline__ float step_length(float s) { return 1.001f * sqrtf(s + 0x1p-120f); }

// a lane's share of a row: D / 64 consecutive columns of dtype DT
template <int D, int DT>
struct Cols {
  static constexpr int C = D / 64;
  using Mag = typename Raw8<DT>::Mag;
  using Word = std::conditional_t<DT == kF32, std::conditional_t<C == 2, uint2, uint32_t>,
                                  std::conditional_t<C == 2, uint32_t, uint16_t>>;
  Word w;
  __device__ __forceinline__ void load(const uint8_t* row, int lane) { w = reinterpret_cast<const Word*>(row)[lane]; }
  __device__ __forceinline__ void to_f32(float (&v)[C]) const {
    if constexpr (DT == kF32) {
      if constexpr (C == 2) { v[0] = __uint_as_float(w.x); v[1] = __uint_as_float(w.y); }
      else v[0] = __uint_as_float(w);
    } else {
#pragma unroll
      for (int k = 0; k < C; ++k) {
        const uint16_t e = static_cast<uint16_t>(w >> (16 * k));
        v[k] = DT == kBF16 ? bf16_bits_to_f32(e) : f16_bits_to_f32(e);
      }
    }
  }
  __device__ __forceinline__ void range(Mag& big, Mag& small) const {
    if constexpr (DT == kF32 && C == 2) {
      Raw8<DT>::range_word(w.x, big, small);
      Raw8<DT>::range_word(w.y, big, small);
    } else {
      Raw8<DT>::range_word(w, big, small);  // a 16-bit word's upper half, zero, counts as none
    }
  }
};

template <int D, int DT>
__global__ void __launch_bounds__(kUpdThreads, 8) km_update_partial_kernel(const void* x, int64_t S, int64_t H, int K,
                                                                        const int32_t* labels, double* partial,
                                                                        int32_t* counts, const int32_t* changed,
                                                                        const Track tr, int first, float* cent,
                                                                        int32_t* clear_next) {
  using Share = Cols<D, DT>;
  constexpr int C = Share::C;
  constexpr int NW = kUpdThreads / 64;
  constexpr int kPf = DT == kF32 ? 16 : 32;  // rows in flight per wave
  constexpr int kGone = 1 << 16;             // move entry: the row left the cluster
  __shared__ int lab_s[kChunk];  // label; moved tokens: + (previous label + 1) << 8
  __shared__ int ord_s[kChunk];  // rows in cluster order, or the moves in cluster order
  __shared__ int start_s[kMaxKAssign + 1];
  __shared__ int running[kMaxKAssign];
  __shared__ int net_s[kMaxKAssign];
  __shared__ int wcnt[NW][kMaxKAssign];
  __shared__ uint32_t range_s[2];  // largest magnitude; smallest nonzero one, minus 1 (bits)
  const int64_t nchunk = (S + kChunk - 1) / kChunk;
  const int64_t bh = blockIdx.x / nchunk, c = blockIdx.x % nchunk;
  if (clear_next && threadIdx.x == 0) clear_next[bh] = 0;
  if (changed[bh] == 0) return;  // converged slice (uniform per workgroup)
  const int64_t b = bh / H, h = bh % H;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int64_t t0 = c * kChunk;
  const int n = static_cast<int>(t0 + kChunk < S ? kChunk : S - t0);
  double* const out = partial + (bh * nchunk + c) * K * D + C * lane;
  int32_t* const cnt_out = counts + (bh * nchunk + c) * K;
  const int64_t pitch = H * D * (DT == kF32 ? 4 : 2);
  const uint8_t* const row0 = static_cast<const uint8_t*>(x) + (b * S + t0) * pitch + h * D * (DT == kF32 ? 4 : 2);
  typename Share::Mag big = 0, small = ~big;
  // acc += the rows of entries p0 .. p1 - 1 in order (MOVES: minus those that
  // left; RANGES: their magnitudes as well).  Past p1 a group of 8 repeats the
  // last row as +0, which changes no sum (one that starts at +0 is never -0).
  auto add_run = [&](int p0, int p1, double (&acc)[C], auto MOVES, auto RANGES) {
    for (; p0 < p1; p0 += kPf) {
      const int mine = ord_s[p0 + lane < p1 ? p0 + lane : p1 - 1];
      Share raw[kPf];
#pragma unroll
      for (int i = 0; i < kPf; i += 8) {
        if (p0 + i < p1) {
#pragma unroll
          for (int k = i; k < i + 8; ++k) {
            const int r = __builtin_amdgcn_readlane(mine, k);
            raw[k].load(row0 + (MOVES ? r & (kGone - 1) : r) * pitch, lane);
          }
        }
      }
      asm volatile("" ::: "memory");  // all of them issued before the first is waited for
#pragma unroll
      for (int i = 0; i < kPf; i += 8) {
        if (p0 + i < p1) {
#pragma unroll
          for (int k = i; k < i + 8; ++k) {
            float v[C];
            raw[k].to_f32(v);
            const uint32_t keep = p0 + k < p1 ? ~0u : 0u;
            const uint32_t neg = MOVES ? static_cast<uint32_t>(__builtin_amdgcn_readlane(mine, k) & kGone) << 15 & keep : 0u;
#pragma unroll
            for (int e = 0; e < C; ++e)
              acc[e] += static_cast<double>(__uint_as_float((__float_as_uint(v[e]) & keep) ^ neg));
            if (RANGES) raw[k].range(big, small);
          }
        }
      }
    }
  };
  using std::false_type;
  using std::true_type;
  const bool by_moves = tr.ul && !first && tr.exact[bh * nchunk + c] != 0;  // if few enough moved
  for (int i = tid; i < K; i += kUpdThreads) { start_s[i + 1] = 0; running[i] = 0; net_s[i] = 0; }
  for (int i = tid; i < NW * K; i += kUpdThreads) wcnt[i / K][i % K] = 0;
  if (tid < 2) range_s[tid] = tid ? 0xffffffffu : 0u;
  int moved = 0;
  for (int r0 = 0; r0 < kChunk; r0 += kUpdThreads) {
    const int i = r0 + tid;
    bool mv = false;
    if (i < n) {
      const int L = labels[bh * S + t0 + i];
      int old = 0;
      if (tr.ul) {
        uint8_t* pl = tr.part_label + bh * S + t0 + i;
        if (by_moves) {
          old = *pl;
          mv = old != L;
        }
        if (!by_moves || mv) *pl = static_cast<uint8_t>(L);
      }
      lab_s[i] = mv ? L | (old + 1) << 8 : L;
    }
    if (by_moves) moved += __syncthreads_count(mv);
  }
  // a slice of one chunk: the sums are the slice's, so this is its centroid pass too
  auto centroid = [&](int j, const double (&acc)[C], int cnt) {
    float* cp = cent + (bh * K + j) * D + C * lane;
    float now[C], s = 0.0f;
#pragma unroll
    for (int e = 0; e < C; ++e) {
      const float old = cp[e];
      now[e] = cnt > 0 ? static_cast<float>(acc[e] / static_cast<double>(cnt)) : old;
      s += (now[e] - old) * (now[e] - old);
    }
#pragma unroll
    for (int e = 0; e < C; ++e) cp[e] = now[e];
    if (tr.ul) {
#pragma unroll
      for (int m = 1; m < 64; m <<= 1) s += __shfl_xor(s, m, 64);
      if (lane == 0) {
        const float step = step_length(s);
        tr.delta[bh * K + j] = step;
        tr.cum[bh * K + j] = add_up(tr.cum[bh * K + j], step);
      }
    }
  };
  if (by_moves && moved == 0) {
    if (cent && tid < K) tr.delta[bh * K + tid] = 0.0f;
    return;
  }
  const bool moves = by_moves && moved <= kMaxMoved;
  __syncthreads();
  // histogram and starts of the clusters' runs
  for (int i = tid; i < n; i += kUpdThreads) {
    const int v = lab_s[i], L = v & 0xff, old = (v >> 8) - 1;
    if (!moves) {
      atomicAdd(&start_s[L + 1], 1);
    } else if (old >= 0) {
      atomicAdd(&start_s[L + 1], 1);
      atomicAdd(&start_s[old + 1], 1);
      atomicAdd(&net_s[L], 1);
      atomicAdd(&net_s[old], -1);
    }
  }
  __syncthreads();
  if (wave == 0) {  // inclusive scan; K <= 64
    int v = lane < K ? start_s[lane + 1] : 0;
#pragma unroll
    for (int m = 1; m < 64; m <<= 1) {
      const int o = __shfl_up(v, m, 64);
      v += lane >= m ? o : 0;
    }
    if (lane < K) start_s[lane + 1] = v;
    if (lane == 0) start_s[0] = 0;
  }
  __syncthreads();
  if (moves) {  // entries of a cluster in any order: their sums are exact
    for (int i = tid; i < n; i += kUpdThreads) {
      const int v = lab_s[i], L = v & 0xff, old = (v >> 8) - 1;
      if (old >= 0) {
        ord_s[start_s[L] + atomicAdd(&running[L], 1)] = i;
        ord_s[start_s[old] + atomicAdd(&running[old], 1)] = i | kGone;
      }
    }
    if (tid < K) {
      const int cnt = cnt_out[tid] + net_s[tid];
      net_s[tid] = cnt;
      if (start_s[tid + 1] > start_s[tid]) {
        cnt_out[tid] = cnt;
        tr.touched[bh * K + tid] = 1;
      }
    }
    __syncthreads();
    for (int j = wave; j < K; j += NW) {
      const int p0 = start_s[j], p1 = start_s[j + 1];
      if (p0 == p1) {
        if (cent && lane == 0) tr.delta[bh * K + j] = 0.0f;
        continue;
      }
      double acc[C];
#pragma unroll
      for (int k = 0; k < C; ++k) acc[k] = out[j * D + k];
      add_run(p0, p1, acc, true_type{}, false_type{});
#pragma unroll
      for (int k = 0; k < C; ++k) out[j * D + k] = acc[k];
      if (cent) centroid(j, acc, net_s[j]);
    }
    return;
  }
  int nbits = 1;
  while ((1 << nbits) < K) ++nbits;
  const uint64_t lt_mask = lane == 0 ? 0ull : (~0ull >> (64 - lane));
  for (int r0 = 0; r0 < n; r0 += kUpdThreads) {
    const int r = r0 + tid;
    const bool valid = r < n;
    const int L = valid ? lab_s[r] & 0xff : -1;
    uint64_t match = __ballot(valid);
    for (int bit = 0; bit < nbits; ++bit) {
      const uint64_t bal = __ballot(valid && ((L >> bit) & 1));
      match &= (valid && ((L >> bit) & 1)) ? bal : ~bal;
    }
    const int rank = __popcll(match & lt_mask);
    if (valid && (match >> lane) == 1ull) wcnt[wave][L] = __popcll(match);  // the highest lane of its label
    __syncthreads();
    if (valid) {
      int pos = start_s[L] + running[L] + rank;
      for (int w = 0; w < wave; ++w) pos += wcnt[w][L];
      ord_s[pos] = r;
    }
    __syncthreads();
    for (int j = tid; j < K; j += kUpdThreads) {
      int sum = 0;
      for (int w = 0; w < NW; ++w) { sum += wcnt[w][j]; wcnt[w][j] = 0; }
      running[j] += sum;
    }
    __syncthreads();
  }
  if (tid < K) {
    cnt_out[tid] = start_s[tid + 1] - start_s[tid];
    if (tr.ul) tr.touched[bh * K + tid] = 1;
  }
  // column sums over the sorted runs of this wave's clusters
  for (int j = wave; j < K; j += NW) {
    double acc[C] = {};
    if (first) add_run(start_s[j], start_s[j + 1], acc, false_type{}, true_type{});
    else add_run(start_s[j], start_s[j + 1], acc, false_type{}, false_type{});
#pragma unroll
    for (int k = 0; k < C; ++k) out[j * D + k] = acc[k];
    if (cent) centroid(j, acc, start_s[j + 1] - start_s[j]);
  }
  if (tr.ul && first) {
    atomicMax(&range_s[0], Raw8<DT>::widest(big, true));
    atomicMin(&range_s[1], Raw8<DT>::widest(small, false));
    __syncthreads();
    if (tid == 0) {
      constexpr int kMant = DT == kF32 ? 23 : DT == kF16 ? 10 : 7;  // mantissa bits below the leading one
      constexpr int kExpTop = DT == kF16 ? 31 : 255;                // of infinities and NaNs
      const int eb = static_cast<int>(range_s[0] >> kMant);         // biased exponents
      int es = static_cast<int>((range_s[1] + 1u) >> kMant);
      es = es < 1 ? 1 : es;
      // 2^(eb + 1) * 2^12 terms over a last bit of 2^(es - kMant): 53 bits hold them
      tr.exact[bh * nchunk + c] = eb < kExpTop && (range_s[0] == 0u || eb + 1 + 12 - (es - kMant) <= 53) ? 1 : 0;
    }
  }
}

// changed: this round's flags; clear_next: the next round's, cleared here
// (the previous round's assignment, their last reader, has finished).  One
// workgroup per cluster: the chunk sums in chunk order, 8 chunks' loads in
// flight; a cluster that no chunk touched keeps its centroid.
template <int D>
__global__ void __launch_bounds__(D) km_finalize_kernel(const double* partial, const int32_t* counts, int64_t nchunk,
                                                        int K, float* cent, const int32_t* changed,
                                                        int32_t* clear_next, const Track tr) {
  __shared__ float red[2];
  const int64_t bh = blockIdx.x / K;
  const int j = blockIdx.x % K;
  const int d = threadIdx.x;
  if (j == 0 && d == 0) clear_next[bh] = 0;
  if (changed[bh] == 0) return;
  if (tr.ul && tr.touched[bh * K + j] == 0) {
    if (d == 0) tr.delta[bh * K + j] = 0.0f;
    return;
  }
  double tot = 0.0;
  int64_t cnt = 0;
  const double* p = partial + (bh * nchunk * K + j) * D + d;
  const int32_t* pc = counts + bh * nchunk * K + j;
  for (int64_t c0 = 0; c0 < nchunk; c0 += 8) {
    double v[8];
    int32_t n[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int64_t c = c0 + i < nchunk ? c0 + i : nchunk - 1;
      v[i] = p[c * K * D];
      n[i] = pc[c * K];
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      if (c0 + i < nchunk) { tot += v[i]; cnt += n[i]; }
    }
  }
  float* cp = cent + (bh * K + j) * D + d;
  const float old = *cp;
  const float now = cnt > 0 ? static_cast<float>(tot / static_cast<double>(cnt)) : old;
  *cp = now;
  if (tr.ul) {  // the length of the centroid's step, from above
    float s = (now - old) * (now - old);
#pragma unroll
    for (int m = 1; m < 64; m <<= 1) s += __shfl_xor(s, m, 64);
    if ((d & 63) == 0) red[d >> 6] = s;
    __syncthreads();  // also: every thread has read touched
    if (d == 0) {
      if (D == 128) s += red[1];
      const float step = step_length(s);
      tr.delta[bh * K + j] = step;
      tr.cum[bh * K + j] = add_up(tr.cum[bh * K + j], step);
      tr.touched[bh * K + j] = 0;
    }
  }
}

// ---- order ---------------------------------------------------------------------------
// Stable counting sort of the labels, a workgroup per kChunk tokens:
// order[pos] = t, inverse[t] = pos.  The chunks' histograms come first (not
// needed for a slice of one chunk); a chunk's tokens of cluster j then start
// after the smaller clusters and the earlier chunks' tokens of j.  One
// workgroup per slice took 53 us at 40 x 32768 (40 of 256 CUs, 32 rounds of
// three barriers).
constexpr int kSortThreads = 512;

__global__ void __launch_bounds__(kSortThreads) km_hist_kernel(const int32_t* labels, int64_t S, int64_t nchunk, int K,
                                                               int32_t* hist) {
  __shared__ int cnt[kMaxKAssign];
  const int64_t bh = blockIdx.x / nchunk, c = blockIdx.x % nchunk;
  const int tid = threadIdx.x;
  const int64_t t0 = c * kChunk;
  if (tid < K) cnt[tid] = 0;
  __syncthreads();
  for (int64_t t = t0 + tid; t < t0 + kChunk && t < S; t += kSortThreads) atomicAdd(&cnt[labels[bh * S + t]], 1);
  __syncthreads();
  if (tid < K) hist[blockIdx.x * K + tid] = cnt[tid];
}

__global__ void __launch_bounds__(kSortThreads) km_sort_kernel(const int32_t* labels, int64_t S, int64_t nchunk, int K,
                                                               const int32_t* hist, int32_t* order,
                                                               int32_t* inverse) {
  constexpr int NW = kSortThreads / 64;
  __shared__ int lab_s[kChunk];
  __shared__ int total[kMaxKAssign];    // the slice's tokens of each cluster
  __shared__ int running[kMaxKAssign];  // where the next token of each cluster goes
  __shared__ int wcnt[NW][kMaxKAssign];
  const int64_t bh = blockIdx.x / nchunk, c = blockIdx.x % nchunk;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int64_t t0 = c * kChunk;
  const int n = static_cast<int>(t0 + kChunk < S ? kChunk : S - t0);
  if (tid < K) { total[tid] = 0; running[tid] = 0; }
  for (int i = tid; i < NW * K; i += kSortThreads) wcnt[i / K][i % K] = 0;
  for (int i = tid; i < n; i += kSortThreads) lab_s[i] = labels[bh * S + t0 + i];
  __syncthreads();
  if (nchunk == 1) {
    for (int i = tid; i < n; i += kSortThreads) atomicAdd(&total[lab_s[i]], 1);
  } else if (lane < K) {  // lane: cluster; waves share the chunks
    int all = 0, before = 0;
    const int32_t* hp = hist + bh * nchunk * K + lane;
    for (int64_t i = wave; i < nchunk; i += NW) {
      const int v = hp[i * K];
      all += v;
      before += i < c ? v : 0;
    }
    atomicAdd(&total[lane], all);
    atomicAdd(&running[lane], before);
  }
  __syncthreads();
  if (wave == 0) {  // exclusive scan of the totals; K <= 64
    const int own = lane < K ? total[lane] : 0;
    int v = own;
#pragma unroll
    for (int m = 1; m < 64; m <<= 1) {
      const int o = __shfl_up(v, m, 64);
      v += lane >= m ? o : 0;
    }
    if (lane < K) running[lane] += v - own;
  }
  __syncthreads();
  int nbits = 1;
  while ((1 << nbits) < K) ++nbits;
  const uint64_t lt_mask = lane == 0 ? 0ull : (~0ull >> (64 - lane));
  for (int r0 = 0; r0 < n; r0 += kSortThreads) {
    const int r = r0 + tid;
    const bool valid = r < n;
    const int L = valid ? lab_s[r] : -1;
    uint64_t match = __ballot(valid);
    for (int bit = 0; bit < nbits; ++bit) {
      const uint64_t bal = __ballot(valid && ((L >> bit) & 1));
      match &= (valid && ((L >> bit) & 1)) ? bal : ~bal;
    }
    const int rank = __popcll(match & lt_mask);
    if (valid && (match >> lane) == 1ull) wcnt[wave][L] = __popcll(match);  // the highest lane of its label
    __syncthreads();
    if (valid) {
      int pos = running[L] + rank;
      for (int w = 0; w < wave; ++w) pos += wcnt[w][L];
      order[bh * S + pos] = static_cast<int32_t>(t0 + r);
      inverse[bh * S + t0 + r] = pos;
    }
    __syncthreads();
    for (int j = tid; j < K; j += kSortThreads) {
      int sum = 0;
      for (int w = 0; w < NW; ++w) { sum += wcnt[w][j]; wcnt[w][j] = 0; }
      running[j] += sum;
    }
    __syncthreads();
  }
}

struct KmWs {
  float* cent;
  double* partial;
  int32_t* counts;
  int32_t* changed;  // [2][BH]: the convergence flags of two consecutive rounds
  Track track;
};

// The workspace's pieces in order and its size; with `tracked` the state of
// struct Track follows the rest (its pointers stay null otherwise).
int64_t carve(void* ws, int64_t BH, int64_t S, int64_t D, int K, bool tracked, KmWs* w) {
  const int64_t nchunk = (S + kChunk - 1) / kChunk;
  int64_t at = 0;
  auto take = [&](auto*& ptr, int64_t count) {
    if (w) ptr = reinterpret_cast<std::remove_reference_t<decltype(ptr)>>(static_cast<uint8_t*>(ws) + at);
    at += count * static_cast<int64_t>(sizeof(*ptr));
  };
  KmWs none{};
  KmWs& k = w ? *w : none;
  take(k.partial, BH * nchunk * K * D);
  take(k.cent, BH * K * D);
  take(k.counts, BH * nchunk * K);
  take(k.changed, 2 * BH);
  if (tracked) {
    at = (at + 7) / 8 * 8;
    take(k.track.ul, BH * S);
    take(k.track.cum, BH * K);
    take(k.track.delta, BH * K);
    take(k.track.cum_max, 2 * BH);
    take(k.track.touched, BH * K);
    take(k.track.exact, BH * nchunk);
    take(k.track.part_label, BH * S);
  }
  return at;
}

int kmeans_run(const void* x, int dtype, int64_t B, int64_t S, int64_t H, int64_t D, int K, int iters, uint64_t seed,
               void* workspace, bool tracked, int32_t* labels, int32_t* order, int32_t* inverse, hipStream_t st);

}  // namespace

extern "C" int64_t lbfq_kmeans_workspace_bytes(int64_t B, int64_t S, int64_t H, int64_t D, int K) {
  return carve(nullptr, B * H, S, D, K, true, nullptr);
}

extern "C" int lbfq_kmeans(const void* x, int dtype, int64_t B, int64_t S, int64_t H, int64_t D, int K, int iters,
                           uint64_t seed, void* workspace, int32_t* labels, int32_t* order, int32_t* inverse,
                           lbfq_stream_t stream) {
  return kmeans_run(x, dtype, B, S, H, D, K, iters, seed, workspace, true, labels, order, inverse,
                    static_cast<hipStream_t>(stream));
}

namespace {
int kmeans_run(const void* x, int dtype, int64_t B, int64_t S, int64_t H, int64_t D, int K, int iters, uint64_t seed,
               void* workspace, bool tracked, int32_t* labels, int32_t* order, int32_t* inverse, hipStream_t st) {
  LBFQ_CHECK_ARG(x && workspace && labels && order && inverse, "lbfq_kmeans: null pointer");
  LBFQ_CHECK_ARG(D == 64 || D == 128, "lbfq_kmeans: D must be 64 or 128; got %lld", (long long)D);
  LBFQ_CHECK_ARG(dtype >= 0 && dtype <= 2, "lbfq_kmeans: bad dtype %d", dtype);
  LBFQ_CHECK_ARG(K >= 1 && K <= S, "n_clusters must be in [1, S]; got %d for S=%lld", K, (long long)S);
  LBFQ_CHECK_ARG(K <= kMaxKAssign, "lbfq_kmeans: at most %d clusters are supported; got %d", kMaxKAssign, K);
  LBFQ_CHECK_ARG(B * H < (1ll << 31) / 1024, "lbfq_kmeans: too many slices");
  const int64_t BH = B * H;
  const int64_t nchunk = (S + kChunk - 1) / kChunk;
  const int rounds = iters > 0 ? iters : 1;
  KmWs w{};
  carve(workspace, BH, S, D, K, tracked && rounds > 1, &w);  // one round has nothing to carry over
  hipLaunchKernelGGL(km_init_kernel, dim3(static_cast<unsigned>(BH * K)), dim3(static_cast<unsigned>(D)), 0, st, x,
                     dtype, S, H, D, K, seed, w.cent, w.track.cum);
  LBFQ_LAUNCH_CHECK("km_init");
  // assignment: two workgroups per CU, fewer where there are fewer slabs
  const int64_t nslabs = BH * ((S + kSlab - 1) / kSlab);
  const unsigned nasg = static_cast<unsigned>(nslabs < 512 ? nslabs : 512);
  for (int it = 0; it < rounds; ++it) {
    const dim3 ga(nasg), gu(static_cast<unsigned>(BH * nchunk));
    // round it writes flag slot it % 2, read by its update and finalize and by
    // round it + 1's assignment; the centroid pass clears slot (it + 1) % 2 first
    int32_t* cur = w.changed + (it & 1) * BH;
    int32_t* clear = w.changed + ((it + 1) & 1) * BH;
    const int32_t* prev = it == 0 ? nullptr : w.changed + ((it - 1) & 1) * BH;
#define LBFQ_KM(DD, DT)                                                                                             \
  if (K <= 32)                                                                                                      \
    hipLaunchKernelGGL((km_assign_kernel<DD, DT, 1>), ga, dim3(kAsgThreads), 0, st, x, BH, S, H, K, w.cent, labels, \
                       prev, cur, w.track, it);                                                                     \
  else                                                                                                              \
    hipLaunchKernelGGL((km_assign_kernel<DD, DT, 2>), ga, dim3(kAsgThreads), 0, st, x, BH, S, H, K, w.cent, labels, \
                       prev, cur, w.track, it);                                                                     \
  if (it + 1 < rounds)                                                                                              \
    hipLaunchKernelGGL((km_update_partial_kernel<DD, DT>), gu, dim3(kUpdThreads), 0, st, x, S, H, K, labels,        \
                       w.partial, w.counts, cur, w.track, it == 0, nchunk == 1 ? w.cent : nullptr,                \
                       nchunk == 1 ? clear : nullptr);
    if (D == 128) {
      if (dtype == kBF16) { LBFQ_KM(128, kBF16) } else if (dtype == kF16) { LBFQ_KM(128, kF16) } else { LBFQ_KM(128, kF32) }
    } else {
      if (dtype == kBF16) { LBFQ_KM(64, kBF16) } else if (dtype == kF16) { LBFQ_KM(64, kF16) } else { LBFQ_KM(64, kF32) }
    }
#undef LBFQ_KM
    LBFQ_LAUNCH_CHECK("km_assign / km_update_partial");
    if (it + 1 == rounds) break;  // the last update does not change the labels
    if (nchunk == 1) continue;  // done by the update
    const dim3 gf(static_cast<unsigned>(BH * K));
    if (D == 128)
      hipLaunchKernelGGL(km_finalize_kernel<128>, gf, dim3(128), 0, st, w.partial, w.counts, nchunk, K, w.cent, cur,
                         clear, w.track);
    else
      hipLaunchKernelGGL(km_finalize_kernel<64>, gf, dim3(64), 0, st, w.partial, w.counts, nchunk, K, w.cent, cur,
                         clear, w.track);
    LBFQ_LAUNCH_CHECK("km_finalize");
  }
  const dim3 gs(static_cast<unsigned>(BH * nchunk));
  if (nchunk > 1)  // the counts of the sums are done with: their place holds the histograms
    hipLaunchKernelGGL(km_hist_kernel, gs, dim3(kSortThreads), 0, st, labels, S, nchunk, K, w.counts);
  hipLaunchKernelGGL(km_sort_kernel, gs, dim3(kSortThreads), 0, st, labels, S, nchunk, K, w.counts, order, inverse);
  LBFQ_LAUNCH_CHECK("km_sort");
  return 0;
}
}  // namespace

// ---- allocation-free variant -------------------------------------------------
// For callers that cannot allocate device memory (code under HIP graph capture,
// serving loops, harnesses that forbid hipMalloc): the workspace is a
// file-scope device array, one copy per GPU, held until the process ends.
// Its device address is looked up once per device (hipGetSymbolAddress, with
// that device current) and kept; host code never uses the array's name as an
// address.  Calls that overlap on one GPU share the array and race.  The
// kernels write every workspace word they read, so nothing is cleared.  A
// problem whose centroids and sums fit the array but not the state carried
// between rounds as well runs without that state.
constexpr int64_t kKmScratchBytes = int64_t{64} << 20;  // 64 MiB: the 14B Q k-means (40 x 32768, K=32) needs 43 MB
static __device__ __align__(256) uint8_t scratch[kKmScratchBytes];
namespace {
constexpr int kMaxDevices = 64;
void* g_km_scratch[kMaxDevices] = {};
std::mutex g_km_scratch_mu;

int km_scratch_ptr(void** out) {
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  LBFQ_CHECK_ARG(e == hipSuccess, "lbfq_kmeans_noalloc: hipGetDevice failed: %s", hipGetErrorString(e));
  LBFQ_CHECK_ARG(dev >= 0 && dev < kMaxDevices, "lbfq_kmeans_noalloc: device %d out of range", dev);
  std::lock_guard<std::mutex> lock(g_km_scratch_mu);
  if (!g_km_scratch[dev]) {
    void* p = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p) {
      lbfq_set_error("lbfq_kmeans_noalloc: hipGetSymbolAddress failed: %s", hipGetErrorString(e));
      return -2;
    }
    g_km_scratch[dev] = p;
  }
  *out = g_km_scratch[dev];
  return 0;
}
}  // namespace

extern "C" int64_t lbfq_kmeans_noalloc_max_workspace_bytes(void) { return kKmScratchBytes; }

extern "C" int lbfq_kmeans_noalloc(const void* x, int dtype, int64_t B, int64_t S, int64_t H, int64_t D, int K,
                                   int iters, uint64_t seed, int32_t* labels, int32_t* order, int32_t* inverse,
                                   lbfq_stream_t stream) {
  LBFQ_CHECK_ARG(B > 0 && S > 0 && H > 0 && D > 0 && K > 0, "lbfq_kmeans_noalloc: empty shape");
  const int64_t need = carve(nullptr, B * H, S, D, K, false, nullptr);
  LBFQ_CHECK_ARG(need <= kKmScratchBytes,
                 "lbfq_kmeans_noalloc: the problem needs %lld bytes of workspace, above the %lld-byte built-in "
                 "scratch; use lbfq_kmeans with a caller workspace",
                 (long long)need, (long long)kKmScratchBytes);
  void* ws = nullptr;
  const int rc = km_scratch_ptr(&ws);
  if (rc) return rc;
  const bool tracked = lbfq_kmeans_workspace_bytes(B, S, H, D, K) <= kKmScratchBytes;
  return kmeans_run(x, dtype, B, S, H, D, K, iters, seed, ws, tracked, labels, order, inverse,
                    static_cast<hipStream_t>(stream));
}
