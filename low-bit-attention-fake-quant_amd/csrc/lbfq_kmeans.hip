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
// The order is a stable counting sort of the labels (argsort stable=True).
#include <mutex>
#include "lbfq_common.h"
#include "../../include/lbfq.h"

using namespace lbfq;

namespace {

constexpr int kChunk = 1024;
constexpr int kMaxD = 128;
constexpr int kMaxKAssign = 64;   // centroids held in LDS by the assign kernel
constexpr int kSortThreads = 1024;
constexpr int kMaxKSort = kMaxKAssign;

__device__ __forceinline__ uint64_t kmix(uint64_t seed, uint64_t bh, uint64_t K, uint64_t j) {
  uint64_t z = seed + 0x9E3779B97F4A7C15ull * (bh * K + j + 1ull);
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  return z ^ (z >> 31);
}

__global__ void km_init_kernel(const void* x, int dt, int64_t S, int64_t H, int64_t D, int K, uint64_t seed,
                               float* cent) {
  const int64_t bh = blockIdx.x / K;
  const int j = blockIdx.x % K;
  const int64_t b = bh / H, h = bh % H;
  const int64_t stride = S / K;
  const int64_t idx = j * stride + static_cast<int64_t>(kmix(seed, bh, K, j) % static_cast<uint64_t>(stride));
  const int d = threadIdx.x;
  if (d < D) cent[(bh * K + j) * D + d] = load_as_f32(x, ((b * S + idx) * H + h) * D + d, dt);
}

typedef float v16f __attribute__((ext_vector_type(16)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

// 8 consecutive elements of dtype DT: as loaded, and as fp32
template <int DT>
struct Raw8 {
  uint4 r[DT == kF32 ? 2 : 1];
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
// the last at twice the largest error of an MFMA measured on a gfx950 relative
// to the magnitudes it adds (2^-21.4 over operands of mixed magnitude, 2^-23
// over operands of one).  Twice their sum is below 2^-14 X C + 2^-15 C^2
// (2^-13 and 2^-14 with x split): two centroids whose a_j are further apart
// than that gap are in the specification's order.  A token with another
// centroid within the gap of its best -- or with a non-finite value anywhere,
// since the test counts the centroids that are NOT below the gap -- is settled
// by the specification itself: one lane per centroid runs the FMA chain, and
// the wave takes the first minimum.
//
// Bound by the token reads: 40 x 32768 x 128 bf16 (335 MB a round) with 32
// clusters took 196 us as one token per lane against LDS broadcasts (1.7 TB/s;
// 278 us with 64 clusters: the FMA issue bound it).
constexpr int kAsgWaves = 8;
constexpr int kAsgThreads = 64 * kAsgWaves;
constexpr int kSlab = 32 * kAsgWaves;  // tokens per step of a workgroup

template <int D, int MB>
struct AssignLds {
  static constexpr int P = D + 4;  // row pitch of the fp32 centroids: float4 reads of 16 rows hit distinct banks
  uint4 part[2][D / 16][MB][64];   // hi / lo operands, as the lanes read them
  float cent[32 * MB * P];
  float cn[32 * MB];
};

// The centroids of slice bh into LDS: fp32 rows, hi / lo MFMA operands and the
// norms (the specification's chain).  Rows K .. 32 MB - 1 are zero with norm
// +inf, so they never win.
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
  if (threadIdx.x < 32 * MB) {
    const float4* c = reinterpret_cast<const float4*>(lds.cent + threadIdx.x * L::P);
    float acc = 0.0f;
#pragma unroll 8
    for (int i = 0; i < D / 4; ++i) {
      const float4 v = c[i];
      acc = fmaf(v.x, v.x, acc);
      acc = fmaf(v.y, v.y, acc);
      acc = fmaf(v.z, v.z, acc);
      acc = fmaf(v.w, v.w, acc);
    }
    lds.cn[threadIdx.x] = static_cast<int>(threadIdx.x) < K ? acc : INFINITY;
  }
  __syncthreads();
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

// Grid: any number of workgroups; each takes a contiguous share of the
// BH * ceil(S / kSlab) slabs (two workgroups per CU and equal shares: no
// partial last wave of workgroups), refilling LDS when the slice changes.
// prev_changed: the flags of the previous round (NULL in the first round);
// changed: this round's flags, set to 1 for a slice in which some label
// changed.  They are zero on entry from the second round on; in the first
// round every label counts as changed, so every slice's flag is written.
template <int D, int DT, int MB>
__global__ void __launch_bounds__(kAsgThreads, 4)
    km_assign_kernel(const void* x, int64_t BH, int64_t S, int64_t H, int K, const float* cent, int32_t* labels,
                     const int32_t* prev_changed, int32_t* changed) {
  constexpr int NKS = D / 16;
  constexpr bool XSPLIT = DT != kBF16;
  constexpr float kGapXC = XSPLIT ? 0x1p-13f : 0x1p-14f, kGapCC = XSPLIT ? 0x1p-14f : 0x1p-15f;
  __shared__ AssignLds<D, MB> lds;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int li = lane & 31, g = lane >> 5;
  const int64_t nslab = (S + kSlab - 1) / kSlab, total = BH * nslab;
  const int64_t w0 = total * blockIdx.x / gridDim.x, w1 = total * (blockIdx.x + 1) / gridDim.x;
  int64_t cur = -1;
  float c2max = 0.0f;  // >= max_j |c_j|^2
  for (int64_t w = w0; w < w1; ++w) {
    const int64_t bh = w / nslab;
    if (prev_changed && prev_changed[bh] == 0) continue;  // converged slice (uniform per workgroup)
    if (bh != cur) {
      if (cur >= 0) __syncthreads();  // every wave is done with the previous slice's centroids
      assign_fill<D, MB>(lds, cent + bh * K * D, K);
      cur = bh;
      c2max = 0.0f;
      for (int j = 0; j < K; ++j) c2max = fmaxf(c2max, lds.cn[j]);
      for (int j = 0; j < K; ++j) c2max = lds.cn[j] < INFINITY ? c2max : INFINITY;
    }
    const int64_t t0 = (w - bh * nslab) * kSlab + wave * 32;
    if (t0 >= S) continue;  // no barrier below
    const int64_t b = bh / H, h = bh - b * H;
    const int64_t t = t0 + li < S ? t0 + li : S - 1;  // lanes past the end repeat the last token
    const int64_t x0 = ((b * S + t) * H + h) * D;
    float xx = 0.0f;
    v16f a[MB];
#pragma unroll
    for (int m = 0; m < MB; ++m)
#pragma unroll
      for (int r = 0; r < 16; ++r) a[m][r] = -0.5f * lds.cn[32 * m + 8 * (r >> 2) + 4 * g + (r & 3)];
    // token operands: lane (li, g) holds dimensions 16 ks + 8 g + [0, 8) of its
    // token, GK k-steps' loads in flight (all; half with fp32 tokens and 64
    // centroids, to stay under 128 registers)
    constexpr int GK = DT == kF32 && MB == 2 && NKS == 8 ? 4 : NKS;
#pragma unroll 1
    for (int k0 = 0; k0 < NKS; k0 += GK) {
      Raw8<DT> raw[GK];
#pragma unroll
      for (int i = 0; i < GK; ++i) raw[i].load(x, x0 + 16 * (k0 + i) + 8 * g);
#pragma unroll
      for (int i = 0; i < GK; ++i) {
        const int ks = k0 + i;
        float v[8];
        raw[i].to_f32(v);
        bf16x8 xh, xl;
        split8(v, xh, xl);  // of bf16 tokens xl is zero, and unused
#pragma unroll
        for (int e = 0; e < 8; ++e) xx = fmaf(v[e], v[e], xx);
#pragma unroll
        for (int m = 0; m < MB; ++m) {
          const bf16x8 ch = __builtin_bit_cast(bf16x8, lds.part[0][ks][m][lane]);
          const bf16x8 cl = __builtin_bit_cast(bf16x8, lds.part[1][ks][m][lane]);
          a[m] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ch, xh, a[m], 0, 0, 0);
          a[m] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(cl, xh, a[m], 0, 0, 0);
          if constexpr (XSPLIT) a[m] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ch, xl, a[m], 0, 0, 0);
        }
      }
    }
    xx += __shfl_xor(xx, 32, 64);
    // X C and C^2 from above: 2^-110 covers squares lost to underflow, 1.001 the roundings of the norms
    const float xc = sqrtf((xx + 0x1p-110f) * (c2max + 0x1p-110f));
    const float gap = 1.001f * (kGapXC * xc + kGapCC * c2max) + 0x1p-120f;
    float top = -INFINITY;
#pragma unroll
    for (int m = 0; m < MB; ++m)
#pragma unroll
      for (int r = 0; r < 16; ++r) top = fmaxf(top, a[m][r]);
    top = fmaxf(top, __shfl_xor(top, 32, 64));
    const float thr = top - gap;
    int cnt = 0, bj = 0;
#pragma unroll
    for (int m = 0; m < MB; ++m)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const bool near = !(a[m][r] < thr);  // NaN on either side counts as near
        cnt += near ? 1 : 0;
        bj = near ? 32 * m + 8 * (r >> 2) + (r & 3) : bj;
      }
    bj = cnt ? bj + 4 * g : 0;
    const int cnt2 = cnt + __shfl_xor(cnt, 32, 64);
    bj = max(bj, __shfl_xor(bj, 32, 64));  // the one near centroid, if there is one
    // unsettled tokens, two at a time with up to 32 centroids
    uint32_t open = static_cast<uint32_t>(__ballot(cnt2 != 1 && t0 + li < S));
    while (open) {
      const int i0 = __builtin_ctz(open);
      open &= open - 1;
      int i1 = i0;
      if (MB == 1 && open) {
        i1 = __builtin_ctz(open);
        open &= open - 1;
      }
      const int ti = MB == 1 && lane >= 32 ? i1 : i0;
      const int lab = assign_exact<D, DT, MB>(lds, x, ((b * S + t0 + ti) * H + h) * D, lane);
      const int l0 = __builtin_amdgcn_readlane(lab, 0), l1 = __builtin_amdgcn_readlane(lab, 32);
      if (li == i0) bj = l0;
      else if (li == i1) bj = l1;
    }
    if (lane < 32 && t0 + li < S) {
      int32_t* lp = labels + bh * S + t0 + li;
      const int32_t old = prev_changed ? *lp : -1;
      *lp = bj;
      if (__any(old != bj) && lane == 0) changed[bh] = 1;
    }
  }
}

// fp64 per-cluster column sums of one kChunk-token chunk.  The chunk's tokens
// are first sorted by label in LDS, stably (ballot ranks within a wave, waves
// and rounds in token order), so a cluster's tokens keep their order.  Then
// the D / 8 lanes of group g -- 8 columns each, one 16-byte load per bf16 row --
// add the runs of clusters j = g, g + NG, ... in that order: the token-order
// fp64 sums of the specification, with 8 rows in flight per lane.
// Bound by the row reads (and the LDS sort ahead of them); with one column and
// a 2-byte load per lane it took 132 us a round at 40 x 32768 x 128 bf16, 32
// clusters (2.5 TB/s).
constexpr int kUpdThreads = 512;

template <int D, int DT>
__global__ void __launch_bounds__(kUpdThreads) km_update_partial_kernel(const void* x, int64_t S, int64_t H, int K,
                                                                        const int32_t* labels, double* partial,
                                                                        int32_t* counts, const int32_t* changed) {
  constexpr int LPG = D / 8;              // lanes per cluster group
  constexpr int NG = kUpdThreads / LPG;  // cluster groups
  constexpr int NW = kUpdThreads / 64;
  __shared__ int lab_s[kChunk];
  __shared__ int ord_s[kChunk];
  __shared__ int start_s[kMaxKAssign + 1];
  __shared__ int running[kMaxKAssign];
  __shared__ int wcnt[NW][kMaxKAssign];
  const int64_t nchunk = (S + kChunk - 1) / kChunk;
  const int64_t bh = blockIdx.x / nchunk, c = blockIdx.x % nchunk;
  if (changed[bh] == 0) return;  // converged slice (uniform per workgroup)
  const int64_t b = bh / H, h = bh % H;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int64_t t0 = c * kChunk;
  const int n = static_cast<int>(t0 + kChunk < S ? kChunk : S - t0);
  for (int i = tid; i < K; i += kUpdThreads) { start_s[i + 1] = 0; running[i] = 0; }
  for (int i = tid; i < NW * K; i += kUpdThreads) wcnt[i / K][i % K] = 0;
  for (int i = tid; i < n; i += kUpdThreads) lab_s[i] = labels[bh * S + t0 + i];
  __syncthreads();
  for (int i = tid; i < n; i += kUpdThreads) atomicAdd(&start_s[lab_s[i] + 1], 1);
  __syncthreads();
  if (tid == 0) {
    start_s[0] = 0;
    for (int j = 0; j < K; ++j) start_s[j + 1] += start_s[j];
  }
  __syncthreads();
  int nbits = 1;
  while ((1 << nbits) < K) ++nbits;
  const uint64_t lt_mask = lane == 0 ? 0ull : (~0ull >> (64 - lane));
  for (int r0 = 0; r0 < n; r0 += kUpdThreads) {
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
  if (tid < K) counts[(bh * nchunk + c) * K + tid] = start_s[tid + 1] - start_s[tid];
  // column sums over the sorted runs of this group's clusters
  const int g = tid / LPG, col = 8 * (tid % LPG);
  double* out = partial + (bh * nchunk + c) * K * D + col;
  const int64_t xrow0 = (b * S + t0) * H + h;
  for (int j = g; j < K; j += NG) {
    const int p1 = start_s[j + 1];
    double acc[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) acc[k] = 0.0;
    constexpr int kPf = DT == kF32 ? 4 : 8;
    for (int p0 = start_s[j]; p0 < p1; p0 += kPf) {
      Raw8<DT> raw[kPf];
#pragma unroll
      for (int i = 0; i < kPf; ++i) {
        const int pos = p0 + i < p1 ? p0 + i : p1 - 1;
        raw[i].load(x, (xrow0 + static_cast<int64_t>(ord_s[pos]) * H) * D + col);
      }
#pragma unroll
      for (int i = 0; i < kPf; ++i) {
        if (p0 + i < p1) {
          float v[8];
          raw[i].to_f32(v);
#pragma unroll
          for (int k = 0; k < 8; ++k) acc[k] += static_cast<double>(v[k]);
        }
      }
    }
    double2* o = reinterpret_cast<double2*>(out + j * D);
#pragma unroll
    for (int k = 0; k < 4; ++k) o[k] = make_double2(acc[2 * k], acc[2 * k + 1]);
  }
}

// changed: this round's flags; clear_next: the next round's, cleared here
// (the previous round's assignment, their last reader, has finished).
__global__ void km_finalize_kernel(const double* partial, const int32_t* counts, int64_t nchunk, int K, int64_t D,
                                   float* cent, const int32_t* changed, int32_t* clear_next) {
  const int64_t bh = blockIdx.x / K;
  const int j = blockIdx.x % K;
  const int d = threadIdx.x;
  if (j == 0 && d == 0) clear_next[bh] = 0;
  if (d >= D || changed[bh] == 0) return;
  double tot = 0.0;
  int64_t cnt = 0;
  // 8 chunks' loads in flight, added in chunk order
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
  if (cnt > 0) cent[(bh * K + j) * D + d] = static_cast<float>(tot / static_cast<double>(cnt));
}

// Stable counting sort of one slice's labels: order[pos] = t, inverse[t] = pos.
__global__ void __launch_bounds__(kSortThreads) km_sort_kernel(const int32_t* labels, int64_t S, int K,
                                                               int32_t* order, int32_t* inverse) {
  __shared__ int start[kMaxKSort];
  __shared__ int running[kMaxKSort];
  __shared__ int wcnt[kSortThreads / 64][kMaxKSort];
  const int64_t bh = blockIdx.x;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  constexpr int NW = kSortThreads / 64;
  for (int i = tid; i < K; i += kSortThreads) { start[i] = 0; running[i] = 0; }
  for (int i = tid; i < NW * K; i += kSortThreads) wcnt[i / K][i % K] = 0;
  __syncthreads();
  const int32_t* lab = labels + bh * S;
  for (int64_t t = tid; t < S; t += kSortThreads) atomicAdd(&start[lab[t]], 1);
  __syncthreads();
  if (tid == 0) {
    int acc = 0;
    for (int j = 0; j < K; ++j) { int c = start[j]; start[j] = acc; acc += c; }
  }
  __syncthreads();
  int nbits = 1;
  while ((1 << nbits) < K) ++nbits;
  const uint64_t lt_mask = lane == 0 ? 0ull : (~0ull >> (64 - lane));
  for (int64_t r0 = 0; r0 < S; r0 += kSortThreads) {
    const int64_t t = r0 + tid;
    const bool valid = t < S;
    const int L = valid ? lab[t] : -1;
    uint64_t match = __ballot(valid);
    for (int bit = 0; bit < nbits; ++bit) {
      uint64_t bal = __ballot(valid && ((L >> bit) & 1));
      match &= (valid && ((L >> bit) & 1)) ? bal : ~bal;
    }
    const int rank = __popcll(match & lt_mask);
    const bool leader = valid && ((match >> lane) == 1ull);
    if (leader) wcnt[wave][L] = __popcll(match);
    __syncthreads();
    if (valid) {
      int pos = start[L] + running[L] + rank;
      for (int w = 0; w < wave; ++w) pos += wcnt[w][L];
      order[bh * S + pos] = static_cast<int32_t>(t);
      inverse[bh * S + t] = pos;
    }
    __syncthreads();
    for (int j = tid; j < K; j += kSortThreads) {
      int s = 0;
      for (int w = 0; w < NW; ++w) { s += wcnt[w][j]; wcnt[w][j] = 0; }
      running[j] += s;
    }
    __syncthreads();
  }
}

struct KmWs {
  float* cent;
  double* partial;
  int32_t* counts;
  int32_t* changed;  // [2][BH]: the convergence flags of two consecutive rounds
};

KmWs carve(void* ws, int64_t BH, int64_t S, int64_t D, int K) {
  const int64_t nchunk = (S + kChunk - 1) / kChunk;
  uint8_t* p = static_cast<uint8_t*>(ws);
  KmWs w;
  w.partial = reinterpret_cast<double*>(p);
  p += sizeof(double) * BH * nchunk * K * D;
  w.cent = reinterpret_cast<float*>(p);
  p += sizeof(float) * BH * K * D;
  w.counts = reinterpret_cast<int32_t*>(p);
  p += sizeof(int32_t) * BH * nchunk * K;
  w.changed = reinterpret_cast<int32_t*>(p);
  return w;
}

}  // namespace

extern "C" int64_t lbfq_kmeans_workspace_bytes(int64_t B, int64_t S, int64_t H, int64_t D, int K) {
  const int64_t nchunk = (S + kChunk - 1) / kChunk;
  const int64_t BH = B * H;
  return sizeof(double) * BH * nchunk * K * D + sizeof(float) * BH * K * D + sizeof(int32_t) * BH * nchunk * K +
         sizeof(int32_t) * 2 * BH;
}

extern "C" int lbfq_kmeans(const void* x, int dtype, int64_t B, int64_t S, int64_t H, int64_t D, int K, int iters,
                           uint64_t seed, void* workspace, int32_t* labels, int32_t* order, int32_t* inverse,
                           lbfq_stream_t stream) {
  LBFQ_CHECK_ARG(x && workspace && labels && order && inverse, "lbfq_kmeans: null pointer");
  LBFQ_CHECK_ARG(D == 64 || D == 128, "lbfq_kmeans: D must be 64 or 128; got %lld", (long long)D);
  LBFQ_CHECK_ARG(dtype >= 0 && dtype <= 2, "lbfq_kmeans: bad dtype %d", dtype);
  LBFQ_CHECK_ARG(K >= 1 && K <= S, "n_clusters must be in [1, S]; got %d for S=%lld", K, (long long)S);
  LBFQ_CHECK_ARG(K <= kMaxKAssign, "lbfq_kmeans: at most %d clusters are supported; got %d", kMaxKAssign, K);
  LBFQ_CHECK_ARG(B * H < (1ll << 31) / 1024, "lbfq_kmeans: too many slices");
  hipStream_t st = static_cast<hipStream_t>(stream);
  const int64_t BH = B * H;
  const int64_t nchunk = (S + kChunk - 1) / kChunk;
  KmWs w = carve(workspace, BH, S, D, K);
  hipLaunchKernelGGL(km_init_kernel, dim3(static_cast<unsigned>(BH * K)), dim3(static_cast<unsigned>(D)), 0, st, x,
                     dtype, S, H, D, K, seed, w.cent);
  LBFQ_LAUNCH_CHECK("km_init");
  // assignment: two workgroups per CU, fewer where there are fewer slabs
  const int64_t nslabs = BH * ((S + kSlab - 1) / kSlab);
  const unsigned nasg = static_cast<unsigned>(nslabs < 512 ? nslabs : 512);
  const int rounds = iters > 0 ? iters : 1;
  for (int it = 0; it < rounds; ++it) {
    const dim3 ga(nasg), gu(static_cast<unsigned>(BH * nchunk));
    // round it writes flag slot it % 2, read by its update and finalize and by
    // round it + 1's assignment; finalize clears slot (it + 1) % 2 first
    int32_t* cur = w.changed + (it & 1) * BH;
    const int32_t* prev = it == 0 ? nullptr : w.changed + ((it - 1) & 1) * BH;
#define LBFQ_KM(DD, DT)                                                                                             \
  if (K <= 32)                                                                                                      \
    hipLaunchKernelGGL((km_assign_kernel<DD, DT, 1>), ga, dim3(kAsgThreads), 0, st, x, BH, S, H, K, w.cent, labels, \
                       prev, cur);                                                                                  \
  else                                                                                                              \
    hipLaunchKernelGGL((km_assign_kernel<DD, DT, 2>), ga, dim3(kAsgThreads), 0, st, x, BH, S, H, K, w.cent, labels, \
                       prev, cur);                                                                                  \
  if (it + 1 < rounds)                                                                                              \
    hipLaunchKernelGGL((km_update_partial_kernel<DD, DT>), gu, dim3(kUpdThreads), 0, st, x, S, H, K, labels,        \
                       w.partial, w.counts, cur);
    if (D == 128) {
      if (dtype == kBF16) { LBFQ_KM(128, kBF16) } else if (dtype == kF16) { LBFQ_KM(128, kF16) } else { LBFQ_KM(128, kF32) }
    } else {
      if (dtype == kBF16) { LBFQ_KM(64, kBF16) } else if (dtype == kF16) { LBFQ_KM(64, kF16) } else { LBFQ_KM(64, kF32) }
    }
#undef LBFQ_KM
    LBFQ_LAUNCH_CHECK("km_assign / km_update_partial");
    if (it + 1 == rounds) break;  // the last update does not change the labels
    hipLaunchKernelGGL(km_finalize_kernel, dim3(static_cast<unsigned>(BH * K)), dim3(static_cast<unsigned>(D)), 0, st,
                       w.partial, w.counts, nchunk, K, D, w.cent, cur, w.changed + ((it + 1) & 1) * BH);
    LBFQ_LAUNCH_CHECK("km_finalize");
  }
  hipLaunchKernelGGL(km_sort_kernel, dim3(static_cast<unsigned>(BH)), dim3(kSortThreads), 0, st, labels, S, K, order,
                     inverse);
  LBFQ_LAUNCH_CHECK("km_sort");
  return 0;
}

// ---- allocation-free variant -------------------------------------------------
// For callers that cannot allocate device memory (code under HIP graph capture,
// serving loops, harnesses that forbid hipMalloc): the workspace is a
// file-scope device array, one copy per GPU, held until the process ends.
// Its device address is looked up once per device (hipGetSymbolAddress, with
// that device current) and kept; host code never uses the array's name as an
// address.  Calls that overlap on one GPU share the array and race.  The
// kernels write every workspace word they read, so nothing is cleared.
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
  const int64_t need = lbfq_kmeans_workspace_bytes(B, S, H, D, K);
  LBFQ_CHECK_ARG(need <= kKmScratchBytes,
                 "lbfq_kmeans_noalloc: the problem needs %lld bytes of workspace, above the %lld-byte built-in "
                 "scratch; use lbfq_kmeans with a caller workspace",
                 (long long)need, (long long)kKmScratchBytes);
  void* ws = nullptr;
  const int rc = km_scratch_ptr(&ws);
  if (rc) return rc;
  return lbfq_kmeans(x, dtype, B, S, H, D, K, iters, seed, ws, labels, order, inverse, stream);
}
