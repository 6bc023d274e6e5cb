// GQA attention-tail kernels for gfx950: decode tail (reference gqa::tail), T-token
// verify tail over a bf16 KV cache, and the KV append that precedes it.
//
// Math per query row, from contrib/qwen3.6-27b/kernels/gqa_tail_ref.py:31-70 (kernel
// doc contrib/qwen3.6-27b/kernels/gqa_tail.py:1-23):
//   q' = (1 + w) * q * rsqrt(mean(q^2) + 1e-6); partial RoPE on q'[:64] (rotate_half
//   inside the 64); s_j = q'.k_j / 16 (+ mask); p = softmax(s); out = (p V) * sigmoid(gate).
//
// Verify tail (T tokens x grp q-heads per kv head = R query rows per (b, kv head)):
//  1. qprep: q' per row, scaled by log2(e)/16 and split into bf16 hi + lo parts
//     (hi = bf16(q'), lo = bf16(q' - hi)), so the bf16 MFMA sees q' to ~16 mantissa bits.
//     Block 0 of the same launch writes the split-KV plan; with the fused append
//     (npn_gqa_tail_verify_append) further blocks append the T new K/V rows to the cache,
//     and the RoPE rows come straight from the position table.
//  2. attn: split-KV over a balanced partition. The (b, kv head) pairs' 32-key steps
//     are laid end to end (prefix sums from a one-block plan kernel) and cut into
//     W equal ranges (S steps in all; W from the plan, attn_wgs), one per workgroup of the
//     kAttnWG launched (the rest exit at once), so every workgroup streams the same
//     number of K/V bytes whatever the kv_len spread; a range may cover the end of one
//     pair and the start of the next. One wave per 16-row tile of the R rows; each
//     pair segment streams through LDS in 32-key K/V tiles:
//       S^T[32 keys x 16] = K Q'^T  (K rows from LDS as MFMA A operands, q' hi/lo held in
//                                   VGPRs as B operands)              v_mfma_f32_16x16x32_bf16
//       online softmax per row in fp32 (exp2), causal limit kv_len + t per row
//       O^T[256 x 16] += V^T P^T    (V tile read back transposed with ds_read_b64_tr_b16;
//                                   P hi/lo in bf16, taken directly from the S^T
//                                   accumulator registers)
//     Each wave writes its rows' (m, l, O) partial per pair segment, into slot w + p
//     (workgroup w, pair p: unique, as a workgroup's pairs are consecutive).
//  3. merge: log-sum-exp merge of a pair's segment partials, * sigmoid(gate) -> bf16.
//
// HBM layout: cache [B][Hkv][s_max][256] bf16, each (b, kv head) a contiguous block of
// rows; query/gate/out [B][T][Hq][256]; query row r of (b, g) is token r / grp,
// q-head g*grp + r % grp.
#include "npn_common.h"

namespace {

constexpr int DH = 256;
constexpr int ROPE = 64;
constexpr float kEps = 1e-6f;
constexpr float kLog2e = 1.4426950408889634f;
constexpr float kNegBig = -1.0e30f;   // finite "no key yet" running max (avoids inf - inf)

constexpr int kAttnWG = 512;          // attention workgroups (2 per CU on a 256-CU part)
constexpr float kRescaleLog2 = 8.0f;  // exponent base moves only when a row max grows > 2^8
constexpr int KS = 32;                // keys per step

typedef __bf16 bf16x8 __attribute__((__vector_size__(8 * sizeof(__bf16))));
typedef float f32x4 __attribute__((__vector_size__(4 * sizeof(float))));
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ bf16x8 as_bf16x8(u32x4 v) { return __builtin_bit_cast(bf16x8, v); }

__device__ __forceinline__ bf16x8 pack8(s16x4 a, s16x4 b) {
  typedef short s16x8 __attribute__((ext_vector_type(8)));
  s16x8 v = {a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]};
  return __builtin_bit_cast(bf16x8, v);
}

__device__ __forceinline__ s16x4 lds_tr16(const uint8_t* p) {
  return __builtin_amdgcn_ds_read_tr16_b64_v4i16(
      (__attribute__((address_space(3))) s16x4*)(p));
}

// ---------------------------------------------------------------------------------------
// RoPE rows of verify position (b, t): the caller's [B, T, 64] rows, or with a table [P, 64]
// (the reference's _init_rope table, contrib/qwen3.6-27b/static_decode.py:489-502) its row
// kv_len[b] + t clamped to [0, P), the rows gqa::rope_rows would gather.
struct RopeSrc {
  const float* cos;   // [B, T, 64], or the table [P, 64] when P > 0
  const float* sin;
  int P;
};

__device__ __forceinline__ size_t rope_row(const RopeSrc& r, const int32_t* kv_len, int b, int t,
                                           int T) {
  if (r.P <= 0) return ((size_t)b * T + t) * ROPE;
  long pos = (long)kv_len[b] + t;
  pos = pos < 0 ? 0 : (pos >= r.P ? r.P - 1 : pos);
  return (size_t)pos * ROPE;
}

// ---------------------------------------------------------------------------------------
// KV append: cache row kv_len[b]+t of head g <- bf16(rope(bf16(rmsnorm_1p(key)))), value copy.
// One wave per (b, t, g); lane l owns dims 4l..4l+3.
struct AppendArgs {
  const uint16_t* key;
  const uint16_t* value;
  const float* k_norm;
  RopeSrc rope;
  uint16_t* cache_k;
  uint16_t* cache_v;
  const int32_t* kv_len;
  int B, T, Hkv, s_max;
};

__device__ __forceinline__ void kv_append_wave(const AppendArgs& a, int wave, int lane) {
  if (wave >= a.B * a.T * a.Hkv) return;
  const int g = wave % a.Hkv;
  const int bt = wave / a.Hkv;
  const int b = bt / a.T, t = bt - b * a.T;
  const int pos = a.kv_len[b] + t;
  if (pos < 0 || pos >= a.s_max) return;
  const uint16_t* src = a.key + (size_t)wave * DH + 4 * lane;
  float x[4];
  float ss = 0.f;
  for (int j = 0; j < 4; ++j) {
    x[j] = npn::bf16_to_f32(src[j]);
    ss += x[j] * x[j];
  }
  ss = npn::wave_sum(ss);
  const float rn = rsqrtf(ss * (1.0f / DH) + kEps);
  for (int j = 0; j < 4; ++j)
    x[j] = npn::bf16_to_f32(npn::f32_to_bf16((1.0f + a.k_norm[4 * lane + j]) * (x[j] * rn)));
  float y[4];
  for (int j = 0; j < 4; ++j) y[j] = __shfl_xor(x[j], 8, 64);
  if (lane < ROPE / 4) {
    const size_t ro = rope_row(a.rope, a.kv_len, b, t, a.T) + 4 * lane;
    const float* cs = a.rope.cos + ro;
    const float* sn = a.rope.sin + ro;
    const float sign = lane < ROPE / 8 ? -1.0f : 1.0f;
    for (int j = 0; j < 4; ++j) x[j] = x[j] * cs[j] + sign * y[j] * sn[j];
  }
  const size_t row = (((size_t)b * a.Hkv + g) * a.s_max + pos) * DH + 4 * lane;
  for (int j = 0; j < 4; ++j) a.cache_k[row + j] = npn::f32_to_bf16(x[j]);
  const uint16_t* vs = a.value + (size_t)wave * DH + 4 * lane;
  for (int j = 0; j < 4; ++j) a.cache_v[row + j] = vs[j];
}

__global__ __launch_bounds__(256) void gqa_kv_append_kernel(AppendArgs a) {
  kv_append_wave(a, blockIdx.x * 4 + (threadIdx.x >> 6), threadIdx.x & 63);
}

// ---------------------------------------------------------------------------------------
// 1. q' = rope((1+w) * rmsnorm(q)) * log2(e)/16, split into bf16 hi/lo.
//    One wave per padded query row (b, g, r); lane l owns dims 4l..4l+3. Block 0 of the same
//    launch writes the split-KV plan instead (pstart, below), which the attention reads.
struct QPrepArgs {
  const uint16_t* query;
  const float* q_norm;
  RopeSrc rope;
  uint16_t* qhi;   // [B][Hkv][R][DH]
  uint16_t* qlo;
  const int32_t* kv_len;
  int32_t* pstart;  // [P + 2]
  int B, T, Hq, Hkv, R, P, s_max;
  int qblocks;      // blocks 1..qblocks prepare q'; any blocks after them append the new
  AppendArgs app;   // K/V rows to the cache (app.key != nullptr), one wave per row
};

__device__ __forceinline__ int pair_kend(const int32_t* kv_len, int b, int T, int s_max);

// Workgroups that take part for S steps of P pairs of `nrt` 16-row tiles (one wave each), `equal`
// when all pairs have as many steps. Two chains set a small batch's time, a workgroup's S / W
// steps (about 1.4 us each) and the merge's W / P segments of a pair (about 0.3 us each); their
// sum is least at W = sqrt(4.7 S P). Below kAttnWG that is cut to one workgroup per CU (a few CUs
// with two: 54.0 against 47.9 us for one sequence of 32768 keys), except that lone waves keep 16
// steps each (nrt = 1, one sequence of 49152 keys: 256 workgroups 74 us, 384 69). From kAttnWG on
// the chip is full, and the partial rows that every workgroup writes (R x 1 KB), which the model
// leaves out, count: three waves a workgroup do better with one per CU, and ragged batches from
// 14 steps per CU on with 16 steps each (two waves: where a pair has 128 steps to cut). With
// equal lengths, whole workgroups per pair save every pair a second partial; more than 128
// pairs don't divide one per CU. At least two steps each, since a workgroup has its q' rows to
// read and its ring to fill.
// Measured (24 q / 4 kv heads, calls in a graph, us) with 16 steps a workgroup always, with
// min(sqrt(4.7 S P), kAttnWG) whatever nrt and the lengths, and with this rule:
//   T = 8, 17 sequences of 1500 keys 44.9, 54.2, 44.6; 33 of 600 47.6, 51.5, 42.7; 8 of 4096
//   55.7, 49.2, 46.4; two of 32000 79.9, 76.2, 69.8; one of 64 38, 17, 17;
//   T = 7, 4 of 2892 to 12954 50.0, 56.2, 49.8; 6 of 1969 to 6688 47.0, 51.4, 44.6;
//   T = 4, 17 of 1500 47.4, 49.0, 42.3; T = 3, 3 of 6158 to 21369 58.2, 60.1, 57.5;
//   T = 1, 17 of 1500 52.1, 44.4, 38.5.
// Over 232 batches it is 1.32 and 1.03 times as fast as the other two. The first is nowhere faster
// by more than two runs differ (4 %), the second by up to 7 % on two ragged batches.
constexpr int kMinSteps = 2;
constexpr int kAttnCU = 256;
__device__ __forceinline__ int attn_wgs(int S, int P, int nrt, bool equal) {
  const int by16 = min(max(S / 16, 1), kAttnWG);
  int w = (int)fminf(sqrtf(4.7f * (float)S * (float)P), (float)kAttnWG);
  if (w < kAttnWG) {
    w = min(w, kAttnCU);
    if (nrt == 1) w = max(w, by16);
  } else if (by16 == kAttnWG ||
             (!equal && S >= 14 * kAttnCU && (nrt > 2 || (nrt == 2 && S >= 128 * P)))) {
    return by16;
  } else if (nrt > 2 && (!equal || P <= kAttnCU / 2)) {
    w = kAttnCU;
  }
  w = min(w, S / kMinSteps);
  if (equal && w > P) w -= w % P;
  return w < 1 ? 1 : w;
}

// The plan: pstart[p] = sum of the steps of pairs before p (exclusive scan over one block of
// 256 threads), pstart[P] = all steps, pstart[P + 1] = the workgroups that take part.
__device__ void plan_block(const int32_t* kv_len, int32_t* pstart, int P, int Hkv, int T,
                           int s_max, int nrt) {
  __shared__ int part[256];
  const int t = threadIdx.x;
  const int per = (P + 255) / 256;
  const int p0 = min(P, t * per), p1 = min(P, p0 + per);
  int sum = 0;
  for (int p = p0; p < p1; ++p) sum += (pair_kend(kv_len, p / Hkv, T, s_max) + KS - 1) / KS;
  part[t] = sum;
  __syncthreads();
  for (int off = 1; off < 256; off <<= 1) {  // inclusive Hillis-Steele scan
    const int v = t >= off ? part[t - off] : 0;
    __syncthreads();
    part[t] += v;
    __syncthreads();
  }
  const int S = part[255];
  int run = part[t] - sum, odd = 0;
  for (int p = p0; p < p1; ++p) {
    const int n = (pair_kend(kv_len, p / Hkv, T, s_max) + KS - 1) / KS;
    pstart[p] = run;
    run += n;
    odd |= (int64_t)n * P != S;
  }
  odd = __syncthreads_or(odd);
  if (t == 0) {
    pstart[P] = S;
    pstart[P + 1] = attn_wgs(S, P, nrt, odd == 0);
  }
}

__global__ __launch_bounds__(256) void gqa_qprep_kernel(QPrepArgs a) {
  if (blockIdx.x == 0) {
    plan_block(a.kv_len, a.pstart, a.P, a.Hkv, a.T, a.s_max, a.R / 16);
    return;
  }
  if ((int)blockIdx.x > a.qblocks) {
    kv_append_wave(a.app, (blockIdx.x - 1 - a.qblocks) * 4 + (threadIdx.x >> 6), threadIdx.x & 63);
    return;
  }
  const int wave = (blockIdx.x - 1) * 4 + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int grp = a.Hq / a.Hkv;
  if (wave >= a.B * a.Hkv * a.R) return;
  const int r = wave % a.R;
  const int bg = wave / a.R;
  const int b = bg / a.Hkv, g = bg - b * a.Hkv;
  uint16_t* dhi = a.qhi + (size_t)wave * DH + 4 * lane;
  uint16_t* dlo = a.qlo + (size_t)wave * DH + 4 * lane;
  if (r >= a.T * grp) {  // padding rows of the MFMA tile
    for (int j = 0; j < 4; ++j) { dhi[j] = 0; dlo[j] = 0; }
    return;
  }
  const int t = r / grp, qh = g * grp + (r - (r / grp) * grp);
  const uint16_t* src = a.query + (((size_t)b * a.T + t) * a.Hq + qh) * DH + 4 * lane;
  float x[4];
  float ss = 0.f;
  for (int j = 0; j < 4; ++j) {
    x[j] = npn::bf16_to_f32(src[j]);
    ss += x[j] * x[j];
  }
  ss = npn::wave_sum(ss);
  const float rn = rsqrtf(ss * (1.0f / DH) + kEps);
  for (int j = 0; j < 4; ++j) x[j] = (1.0f + a.q_norm[4 * lane + j]) * (x[j] * rn);
  // partial RoPE: dims 0..63 live in lanes 0..15; partner of dim d is d ^ 32 (lane ^ 8)
  float y[4];
  for (int j = 0; j < 4; ++j) y[j] = __shfl_xor(x[j], 8, 64);
  if (lane < ROPE / 4) {
    const size_t ro = rope_row(a.rope, a.kv_len, b, t, a.T) + 4 * lane;
    const float* cs = a.rope.cos + ro;
    const float* sn = a.rope.sin + ro;
    const float sign = lane < ROPE / 8 ? -1.0f : 1.0f;  // rotate_half = cat(-x[32:], x[:32])
    for (int j = 0; j < 4; ++j) x[j] = x[j] * cs[j] + sign * y[j] * sn[j];
  }
  const float scale = kLog2e / 16.0f;  // softmax scale 1/sqrt(256), in base 2
  for (int j = 0; j < 4; ++j) {
    const float v = x[j] * scale;
    const uint16_t hi = npn::f32_to_bf16(v);
    dhi[j] = hi;
    dlo[j] = npn::f32_to_bf16(v - npn::bf16_to_f32(hi));
  }
}

// ---------------------------------------------------------------------------------------
// 2. split-KV attention over one 512-key chunk of one (b, kv head).
//    Workgroup = NRT waves; wave w owns query rows 16w..16w+15 (its q' hi/lo lives in
//    VGPRs as MFMA B operands) and all waves share each 32-key K/V tile, which is DMA'd
//    from HBM straight into LDS (global_load_lds_dwordx4) through an NST-stage ring.
//
//    LDS tile layout: one DMA instruction (64 lanes x 16 B) moves cache rows 2k and 2k+1
//    into "block" k, interleaved by 16-byte chunk: lane l carries row 2k + (l & 1), chunk
//    l >> 1, so chunk c of row r sits at block(r >> 1) + (2c + (r & 1)) * 16. Blocks are
//    1024 B plus a pad (K: 32 B, V: 64 B). With that layout
//      - every DMA source is the wave-uniform address of row 2k plus a per-lane constant
//        ((l & 1) * 512 + (l >> 1) * 16), and
//      - every MFMA operand read is one per-lane base plus an immediate offset,
//    and the reads spread over the LDS banks: 16 K rows at one column land on 16 distinct
//    16-byte bank groups (pad 32), and the transposed V reads of 4 rows x 64 B per 16-lane
//    group on 4 distinct 64-byte groups (pad 64).
struct AttnArgs {
  const uint16_t* qhi;
  const uint16_t* qlo;
  const uint16_t* cache_k;
  const uint16_t* cache_v;
  const int32_t* kv_len;
  const int32_t* pstart;  // [P + 2] first step of each pair, total steps, workgroups
  float* part_o;          // [kAttnWG + P][R][DH]
  float* part_ml;         // [kAttnWG + P][R][2]
  int Hkv, s_max, T, grp, npairs;
};

// Steps of pair p = (b, kv head): ceil(kend_b / KS), kend_b = min(kv_len[b] + T, s_max).
__device__ __forceinline__ int pair_kend(const int32_t* kv_len, int b, int T, int s_max) {
  const int L = kv_len[b] > 0 ? kv_len[b] : 0;
  return L + T < s_max ? L + T : s_max;
}

// Workgroup w's step range of W workgroups is [w * S / W, (w + 1) * S / W).
__device__ __forceinline__ int wg_first_step(int w, int S, int W) {
  return (int)((int64_t)w * S / W);
}

// Largest p in [0, P) with pstart[p] <= x (pstart is strictly increasing, pstart[0] = 0):
// 64-way search, one sample per lane per round. Wave-uniform result.
__device__ __forceinline__ int find_pair(const int32_t* pstart, int P, int x, int lane) {
  int lo = 0, n = P;
  while (n > 1) {
    const int stride = (n + 63) / 64;
    const int idx = lo + lane * stride;
    const bool le = idx < lo + n && pstart[idx] <= x;
    const int t = __popcll(__builtin_amdgcn_ballot_w64(le)) - 1;  // last lane with le
    const int nlo = lo + t * stride;
    n = min(stride, lo + n - nlo);
    lo = nlo;
  }
  return __builtin_amdgcn_readfirstlane(lo);
}

constexpr int KBLK = 1024 + 32;            // bytes per 2-row block of the K tile
constexpr int VBLK = 1024 + 64;            // ... of the V tile
constexpr int KTILE = (KS / 2) * KBLK;     // 16896
constexpr int VTILE = (KS / 2) * VBLK;     // 17408
constexpr int STAGE = KTILE + VTILE + 1024;  // + one block of slack for padded DMA slots

// Reductions over the 4 lane groups (lanes i, i+16, i+32, i+48) that hold one query row,
// with gfx950's cross-row swaps instead of LDS permutes: after permlane32_swap(x, x) the
// pair holds (x[l & 31], x[(l & 31) + 32]); after permlane16_swap(y, y) it holds the two
// 16-lane rows of y's 32-lane half.
__device__ __forceinline__ float max_over_groups(float x) {
  const auto a = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  x = fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
  const auto b = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
}
__device__ __forceinline__ float sum_over_groups(float x) {
  const auto a = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  x = __uint_as_float(a[0]) + __uint_as_float(a[1]);
  const auto b = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(b[0]) + __uint_as_float(b[1]);
}

template <int NRT, int NST>  // NST: K/V ring stages
__global__ __launch_bounds__(NRT * 64, NST <= 2 ? 2 : 1) void gqa_attn_kernel(AttnArgs a) {
  constexpr int R = NRT * 16;
  constexpr int DPW = (KS + NRT - 1) / NRT;  // DMA instructions per wave per step
  const int wg = blockIdx.x;
  const int S = a.pstart[a.npairs];
  const int W = a.pstart[a.npairs + 1];
  if (wg >= W) return;
  int x = wg_first_step(wg, S, W);
  const int x_end = wg_first_step(wg + 1, S, W);
  if (x >= x_end) return;

  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int i = lane & 15, G = lane >> 4;
  const int row = w * 16 + i;  // this lane's query row (B-operand column / C column)

  __shared__ __attribute__((aligned(16))) uint8_t smem[NST * STAGE];
  const unsigned smem_lds = __builtin_amdgcn_readfirstlane(npn::lds_addr(smem));

  // Per-lane constants. DMA source offset within a 2-row block; LDS bases of the operand
  // reads: K row i (+16 for the second key tile), chunk 4*ks + G; V (transposed reads)
  // key rows 4G + (i>>2) (+16) of dims 16*dt + 4*(i&3) .. +3, i.e. chunk
  // 2*dt + ((i&3)>>1), half (i&1).
  const unsigned lane_src = (unsigned)((lane & 1) * DH * 2 + (lane >> 1) * 16);
  const int tr_row = 4 * G + (i >> 2);
  const int k_base0 = (i >> 1) * KBLK + (2 * G + (i & 1)) * 16;
  const int v_base0 = KTILE + (tr_row >> 1) * VBLK + (2 * ((i & 3) >> 1) + (tr_row & 1)) * 16 +
                      (i & 1) * 8;

  int p = find_pair(a.pstart, a.npairs, x, lane);
  while (x < x_end) {
    const int pbeg = a.pstart[p];
    const int s_lo = x - pbeg;
    const int steps = min(x_end, (int)a.pstart[p + 1]) - x;
    const int bg = p;
    const int b = bg / a.Hkv;
    const int L = a.kv_len[b] > 0 ? a.kv_len[b] : 0;
    const int kend = pair_kend(a.kv_len, b, a.T, a.s_max);  // rows [0, kend) are read
    const int c0 = s_lo * KS;
    const uint8_t* kb = reinterpret_cast<const uint8_t*>(a.cache_k + (size_t)bg * a.s_max * DH);
    const uint8_t* vb = reinterpret_cast<const uint8_t*>(a.cache_v + (size_t)bg * a.s_max * DH);

    // Every wave has finished reading the previous segment's stages.
    __builtin_amdgcn_s_barrier();

    // DMA of step s's tiles into stage s % NST: slot j < 16 is K block j, 16 <= j < 32 is
    // V block j - 16, DPW slots per wave; slots past 32 (NRT * DPW > 32) fill the slack.
    // A step that reaches past kend (a pair's last) clamps its rows to kend - 1, so V rows
    // the mask removes still hold finite cache data.
    // Each slot's LDS offset within a stage and its source at step 0 are fixed for the
    // segment (wave-uniform, kept in SGPRs), so a step's DMAs are one 64-bit add each; the
    // test for a step past kend is made once per step rather than once per slot.
    unsigned sdst[DPW];
    const uint8_t* ssrc[DPW];
#pragma unroll
    for (int q = 0; q < DPW; ++q) {
      const int j = w + NRT * q;  // wave-uniform slot
      const bool isv = j >= KS / 2;
      const int blk = (isv ? j - KS / 2 : j) & (KS / 2 - 1);
      sdst[q] = j < KS ? (isv ? KTILE + blk * VBLK : blk * KBLK) : KTILE + VTILE;
      ssrc[q] = (isv ? vb : kb) + (size_t)(c0 + 2 * blk) * DH * 2;
    }
    auto dma = [&](int s) {
      const int k0 = c0 + s * KS;
      uint8_t* st = smem + (s % NST) * STAGE;
      if (k0 + KS <= kend) {
        const size_t step = (size_t)s * KS * DH * 2;
        const unsigned st_lds = smem_lds + (unsigned)((s % NST) * STAGE);
#pragma unroll
        for (int q = 0; q < DPW; ++q) npn::lds_dma16_soff(ssrc[q] + step, lane_src, st_lds + sdst[q]);
      } else {
#pragma unroll
        for (int q = 0; q < DPW; ++q) {
          const int j = w + NRT * q;
          const bool isv = j >= KS / 2;
          const int blk = (isv ? j - KS / 2 : j) & (KS / 2 - 1);
          const int key = min(k0 + 2 * blk + (lane & 1), kend - 1);
          npn::lds_dma16_soff(isv ? vb : kb, (unsigned)key * DH * 2 + (unsigned)(lane >> 1) * 16,
                              st + sdst[q]);
        }
      }
    };
    // q' hi/lo of this lane's row as B operands: dims 32*ks + 8*G .. +7. Loaded by inline
    // asm ahead of the K/V DMAs, so the loop's own vmcnt wait for step 0 covers them (a
    // compiler-tracked load would make the compiler wait for every DMA issued after it).
    u32x4 qh[8], ql[8];
    {
      const size_t qo = ((size_t)bg * R + row) * DH + 8 * G;
#pragma unroll
      for (int ks = 0; ks < 8; ++ks) {
        asm volatile("global_load_dwordx4 %0, %1, off" : "=v"(qh[ks]) : "v"(a.qhi + qo + 32 * ks)
                     : "memory");
        asm volatile("global_load_dwordx4 %0, %1, off" : "=v"(ql[ks]) : "v"(a.qlo + qo + 32 * ks)
                     : "memory");
      }
    }
    for (int s = 0; s < NST - 1 && s < steps; ++s) dma(s);

    const int lim = row < a.T * a.grp ? L + row / a.grp : kend - 1;  // last key this row sees

    float m_run = kNegBig, l_run = 0.f;
    f32x4 acc[16];
#pragma unroll
    for (int dt = 0; dt < 16; ++dt) acc[dt] = f32x4{0.f, 0.f, 0.f, 0.f};

    for (int s = 0; s < steps; ++s) {
      const int k0 = c0 + s * KS;
      // This wave's DMA of step s has landed once at most the DMAs of the steps after it
      // stay in flight: steps up to s + NST - 2 are issued here (vmcnt holds 6 bits; a
      // smaller count only waits longer).
      if (NST >= 4 && s + 2 < steps)
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * DPW < 63 ? 2 * DPW : 63) : "memory");
      else if (NST >= 3 && s + 1 < steps)
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(DPW < 63 ? DPW : 63) : "memory");
      else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __builtin_amdgcn_s_barrier();  // ... and every other wave's; stage of step s-1 is free
      asm volatile("" ::: "memory");
#pragma unroll
      for (int ks = 0; ks < 8; ++ks) {  // q' registers are read only after that wait
        asm volatile("" : "+v"(qh[ks]));
        asm volatile("" : "+v"(ql[ks]));
      }
      if (s + NST - 1 < steps) dma(s + NST - 1);
      const uint8_t* stage = smem + (s % NST) * STAGE;
      const uint8_t* kp = stage + k_base0;
      const uint8_t* vp = stage + v_base0;

      // S^T[32 keys x 16 rows] = K Q'^T. All 16 K fragments are read first so their LDS
      // latencies overlap; the two key tiles' accumulation chains alternate.
      u32x4 kf[2][8];
#pragma unroll
      for (int kt = 0; kt < 2; ++kt)
#pragma unroll
        for (int ks = 0; ks < 8; ++ks)
          kf[kt][ks] = *reinterpret_cast<const u32x4*>(kp + kt * (KS / 4) * KBLK + ks * 128);
      f32x4 st[2] = {f32x4{0.f, 0.f, 0.f, 0.f}, f32x4{0.f, 0.f, 0.f, 0.f}};
#pragma unroll
      for (int ks = 0; ks < 8; ++ks) {
#pragma unroll
        for (int kt = 0; kt < 2; ++kt)
          st[kt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(kf[kt][ks]),
                                                           as_bf16x8(qh[ks]), st[kt], 0, 0, 0);
#pragma unroll
        for (int kt = 0; kt < 2; ++kt)
          st[kt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(kf[kt][ks]),
                                                           as_bf16x8(ql[ks]), st[kt], 0, 0, 0);
      }
      // Keep the 16 K reads ahead of the 32 MFMAs (the scheduler would otherwise pair each
      // read with its MFMAs and expose the LDS latency 8 times); V fragments then reuse
      // the K fragments' registers.
      __builtin_amdgcn_sched_group_barrier(0x100, 16, 0);
      __builtin_amdgcn_sched_group_barrier(0x008, 32, 0);
      __builtin_amdgcn_sched_barrier(0);

      // V^T fragments of all 16 dim tiles, read before the softmax so their latency
      // overlaps it.
      bf16x8 vf[16];
#pragma unroll
      for (int dt = 0; dt < 16; ++dt)
        vf[dt] = pack8(lds_tr16(vp + dt * 64), lds_tr16(vp + dt * 64 + (KS / 4) * VBLK));

      // causal mask (only a step that reaches past the first query row's limit L needs
      // one) + online softmax (base 2); P hi/lo become the B operands of P.V.
      if (k0 + KS - 1 > L) {
#pragma unroll
        for (int kt = 0; kt < 2; ++kt)
#pragma unroll
          for (int r = 0; r < 4; ++r)
            if (k0 + 16 * kt + 4 * G + r > lim) st[kt][r] = -INFINITY;
      }
      float mx = fmaxf(fmaxf(fmaxf(st[0][0], st[0][1]), fmaxf(st[0][2], st[0][3])),
                       fmaxf(fmaxf(st[1][0], st[1][1]), fmaxf(st[1][2], st[1][3])));
      mx = max_over_groups(mx);
      // The exponent base m_run moves only when a row's max exceeds it by more than 2^8,
      // so p = 2^(s - m_run) <= 256 and most steps skip rescaling O; O / l does not depend
      // on the base. The branch is wave-uniform.
      const bool grow = mx > m_run + kRescaleLog2;
      if (__builtin_amdgcn_ballot_w64(grow) != 0) {
        const float mnew = grow ? mx : m_run;
        const float corr = exp2f(m_run - mnew);
        m_run = mnew;
        l_run *= corr;
#pragma unroll
        for (int dt = 0; dt < 16; ++dt) acc[dt] *= corr;
      }
      bf16x8 ph, pl;
      float psum = 0.f;
#pragma unroll
      for (int kt = 0; kt < 2; ++kt)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float pv = exp2f(st[kt][r] - m_run);
          psum += pv;
          const __bf16 h = (__bf16)pv;
          ph[kt * 4 + r] = h;
          pl[kt * 4 + r] = (__bf16)(pv - (float)h);
        }
      l_run += psum;

      // O^T[256 x 16 rows] += V^T P^T
#pragma unroll
      for (int dt = 0; dt < 16; ++dt)
        acc[dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf[dt], ph, acc[dt], 0, 0, 0);
#pragma unroll
      for (int dt = 0; dt < 16; ++dt)
        acc[dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf[dt], pl, acc[dt], 0, 0, 0);
    }

    // Row sum over the 4 lane groups, then this wave's 16 rows of the segment partial.
    l_run = sum_over_groups(l_run);
    const size_t slot = (size_t)wg + p;
    float* po = a.part_o + (slot * R + row) * DH;
#pragma unroll
    for (int dt = 0; dt < 16; ++dt) *reinterpret_cast<f32x4*>(po + 16 * dt + 4 * G) = acc[dt];
    if (G == 0) {
      float* pml = a.part_ml + (slot * R + row) * 2;
      pml[0] = m_run;
      pml[1] = l_run;
    }
    x += steps;
    ++p;
  }
}

// ---------------------------------------------------------------------------------------
// 3. merge a pair's segment partials, apply sigmoid(gate), write bf16. One 256-thread block
//    per (query row, pair); lane l of every wave owns output dims 4l..4l+3 (float4 partial
//    reads). The workgroups that covered pair p are w(first step) .. w(last step), with
//    w(x) = ((x + 1) * W - 1) / S, W from the plan. Wave q merges segments q, q + 4, ... of
//    the pair (loads issued four segments at a time), and wave 0 then merges the four
//    waves' (m, l, O) in wave order: a small batch's pairs have tens of segments each, which
//    one wave walking them in turn paid for in memory latency.
struct MergeArgs {
  const float* part_o;
  const float* part_ml;
  const int32_t* pstart;
  const uint16_t* gate;
  uint16_t* out;
  int T, Hq, Hkv, R, npairs;
};

constexpr int kMergeRowsMinPairs = 64;  // pairs from which gqa_merge_rows_kernel merges

__global__ __launch_bounds__(256) void gqa_merge_kernel(MergeArgs a) {
  const int r = blockIdx.x;
  const int pr = blockIdx.y;
  const int b = pr / a.Hkv, g = pr - b * a.Hkv;
  const int grp = a.Hq / a.Hkv;
  const int q = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int S = a.pstart[a.npairs];
  const int64_t W = a.pstart[a.npairs + 1];
  const int x0 = a.pstart[pr], x1 = a.pstart[pr + 1] - 1;
  const int w0 = (int)(((int64_t)(x0 + 1) * W - 1) / S);
  const int w1 = (int)(((int64_t)(x1 + 1) * W - 1) / S);
  const size_t stride_ml = (size_t)a.R * 2, stride_o = (size_t)a.R * DH;
  const float* pml = a.part_ml + ((size_t)(w0 + pr) * a.R + r) * 2;
  const float* po = a.part_o + ((size_t)(w0 + pr) * a.R + r) * DH + 4 * lane;
  auto live = [&](int w) { return w <= w1 && wg_first_step(w, S, (int)W) < wg_first_step(w + 1, S, (int)W); };
  const int t = r / grp, qh = g * grp + (r - t * grp);
  const size_t oi = (((size_t)b * a.T + t) * a.Hq + qh) * DH + 4 * lane;
  // The gate is needed only by wave 0's output, after the merge: its load is issued first.
  uint2 gate_bits = make_uint2(0u, 0u);
  if (q == 0) gate_bits = *reinterpret_cast<const uint2*>(a.gate + oi);
  // This wave's segments w0 + q + 4 j: their maximum, then their rescaled sums. The first
  // batch of four (all of a pair's segments whenever it has at most 16) is loaded once and
  // kept in registers for both passes: one round trip to memory instead of two, with the
  // same arithmetic.
  float mv0[4], lv0[4];
  f32x4 ov0[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int w = w0 + q + 4 * j;
    const bool ok = live(w);
    mv0[j] = ok ? pml[(w - w0) * stride_ml] : kNegBig;
    lv0[j] = ok ? pml[(w - w0) * stride_ml + 1] : 0.f;
    ov0[j] = ok ? *reinterpret_cast<const f32x4*>(po + (w - w0) * stride_o)
                : f32x4{0.f, 0.f, 0.f, 0.f};
  }
  float M = kNegBig;
#pragma unroll
  for (int j = 0; j < 4; ++j) M = fmaxf(M, mv0[j]);
  for (int base = w0 + q + 16; base <= w1; base += 16) {
    float mv[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int w = base + 4 * j;
      mv[j] = live(w) ? pml[(w - w0) * stride_ml] : kNegBig;
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) M = fmaxf(M, mv[j]);
  }
  float l = 0.f;
  f32x4 o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const float f = exp2f(mv0[j] - M);
    l += f * lv0[j];
    o += f * ov0[j];
  }
  for (int base = w0 + q + 16; base <= w1; base += 16) {
    float mv[4], lv[4];
    f32x4 ov[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int w = base + 4 * j;
      const bool ok = live(w);
      mv[j] = ok ? pml[(w - w0) * stride_ml] : kNegBig;
      lv[j] = ok ? pml[(w - w0) * stride_ml + 1] : 0.f;
      ov[j] = ok ? *reinterpret_cast<const f32x4*>(po + (w - w0) * stride_o)
                 : f32x4{0.f, 0.f, 0.f, 0.f};
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float f = exp2f(mv[j] - M);
      l += f * lv[j];
      o += f * ov[j];
    }
  }
  __shared__ float s_ml[4][2];
  __shared__ f32x4 s_o[4][64];
  if (lane == 0) {
    s_ml[q][0] = M;
    s_ml[q][1] = l;
  }
  s_o[q][lane] = o;
  __syncthreads();
  if (q != 0) return;
  float Mt = s_ml[0][0];
#pragma unroll
  for (int k = 1; k < 4; ++k) Mt = fmaxf(Mt, s_ml[k][0]);
  float lt = 0.f;
  f32x4 ot = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const float f = exp2f(s_ml[k][0] - Mt);
    lt += f * s_ml[k][1];
    ot += f * s_o[k][lane];
  }
  const float inv = 1.0f / lt;
  const uint32_t gw[2] = {gate_bits.x, gate_bits.y};
  uint32_t w[2];
  for (int j = 0; j < 2; ++j) {
    const float g0 = npn::sigmoid(npn::bf16_to_f32((uint16_t)(gw[j] & 0xFFFFu)));
    const float g1 = npn::sigmoid(npn::bf16_to_f32((uint16_t)(gw[j] >> 16)));
    w[j] = npn::f32_to_bf16(ot[2 * j] * inv * g0) |
           ((uint32_t)npn::f32_to_bf16(ot[2 * j + 1] * inv * g1) << 16);
  }
  *reinterpret_cast<uint2*>(a.out + oi) = make_uint2(w[0], w[1]);
}

// The same merge with one wave per query row (four rows per block) walking all of the pair's
// segments itself: for batches whose pairs have a few segments each (the host picks it when
// there are at least 64 pairs, about 8 segments per pair or fewer), a quarter as many blocks
// and no LDS exchange. Segments are loaded four at a time; the first four stay in registers
// for both the max pass and the sum pass.
__global__ __launch_bounds__(256) void gqa_merge_rows_kernel(MergeArgs a) {
  const int q = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int grp = a.Hq / a.Hkv;
  const int r = blockIdx.x * 4 + q;  // query row of the pair, t * grp + head; a.R >= T * grp
  if (r >= a.T * grp) return;        // wave-uniform; the kernel has no block barrier
  const int pr = blockIdx.y;
  const int b = pr / a.Hkv, g = pr - b * a.Hkv;
  const int S = a.pstart[a.npairs];
  const int64_t W = a.pstart[a.npairs + 1];
  const int x0 = a.pstart[pr], x1 = a.pstart[pr + 1] - 1;
  const int w0 = (int)(((int64_t)(x0 + 1) * W - 1) / S);
  const int w1 = (int)(((int64_t)(x1 + 1) * W - 1) / S);
  const size_t stride_ml = (size_t)a.R * 2, stride_o = (size_t)a.R * DH;
  const float* pml = a.part_ml + ((size_t)(w0 + pr) * a.R + r) * 2;
  const float* po = a.part_o + ((size_t)(w0 + pr) * a.R + r) * DH + 4 * lane;
  auto live = [&](int w) { return w <= w1 && wg_first_step(w, S, (int)W) < wg_first_step(w + 1, S, (int)W); };
  const int t = r / grp, qh = g * grp + (r - t * grp);
  const size_t oi = (((size_t)b * a.T + t) * a.Hq + qh) * DH + 4 * lane;
  const uint2 gate_bits = *reinterpret_cast<const uint2*>(a.gate + oi);
  float mv0[4], lv0[4];
  f32x4 ov0[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int w = w0 + j;
    const bool ok = live(w);
    mv0[j] = ok ? pml[(w - w0) * stride_ml] : kNegBig;
    lv0[j] = ok ? pml[(w - w0) * stride_ml + 1] : 0.f;
    ov0[j] = ok ? *reinterpret_cast<const f32x4*>(po + (w - w0) * stride_o)
                : f32x4{0.f, 0.f, 0.f, 0.f};
  }
  float M = kNegBig;
#pragma unroll
  for (int j = 0; j < 4; ++j) M = fmaxf(M, mv0[j]);
  for (int base = w0 + 4; base <= w1; base += 4) {
    float mv[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int w = base + j;
      mv[j] = live(w) ? pml[(w - w0) * stride_ml] : kNegBig;
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) M = fmaxf(M, mv[j]);
  }
  float l = 0.f;
  f32x4 o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const float f = exp2f(mv0[j] - M);
    l += f * lv0[j];
    o += f * ov0[j];
  }
  for (int base = w0 + 4; base <= w1; base += 4) {
    float mv[4], lv[4];
    f32x4 ov[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int w = base + j;
      const bool ok = live(w);
      mv[j] = ok ? pml[(w - w0) * stride_ml] : kNegBig;
      lv[j] = ok ? pml[(w - w0) * stride_ml + 1] : 0.f;
      ov[j] = ok ? *reinterpret_cast<const f32x4*>(po + (w - w0) * stride_o)
                 : f32x4{0.f, 0.f, 0.f, 0.f};
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float f = exp2f(mv[j] - M);
      l += f * lv[j];
      o += f * ov[j];
    }
  }
  const float inv = 1.0f / l;
  const uint32_t gw[2] = {gate_bits.x, gate_bits.y};
  uint32_t w[2];
  for (int j = 0; j < 2; ++j) {
    const float g0 = npn::sigmoid(npn::bf16_to_f32((uint16_t)(gw[j] & 0xFFFFu)));
    const float g1 = npn::sigmoid(npn::bf16_to_f32((uint16_t)(gw[j] >> 16)));
    w[j] = npn::f32_to_bf16(o[2 * j] * inv * g0) |
           ((uint32_t)npn::f32_to_bf16(o[2 * j + 1] * inv * g1) << 16);
  }
  *reinterpret_cast<uint2*>(a.out + oi) = make_uint2(w[0], w[1]);
}

// ---------------------------------------------------------------------------------------
// Decode tail of the reference op (fp32 cache, one kv head, mask shared over the batch).
// HBM-bound: every fp32 K and V row is read once for Hq query rows. One workgroup per sequence
// (the first form of this kernel) left all but B CUs idle and took 3.9 ms at B = 8, Hq = 6,
// S = 4096 (67 MB, 17 GB/s), so each sequence's keys are split over workgroups, whose
// (m, l, O) partials a second launch merges.
// Products run on the fp32 matrix instruction (16x16x4, fp32 operands and sums), heads padded
// to its 16 columns, which needs no LDS and no cross-lane sums in the loop: the contraction
// index of each product may be permuted freely as long as both operands agree, so
//   S^T[16 keys x 16 heads] = K Q'^T: lane (i, g) (i = lane & 15, g = lane >> 4) takes key i,
//     dims 16 s + 4 g + j at step 4 s + j: a 16-byte load of K feeds four steps;
//   O[16 heads x 256] += P V: step r takes keys 4 g + r, so lane (i, g)'s S^T register r is its
//     A operand as it stands, and column i of output tile (n, j) is dim 64 n + 4 i + j, so a
//     16-byte load of V (256-byte runs of four rows) feeds four tiles.
// 128 instructions of 32 cycles per 16 keys and wave, a third of the time HBM needs to bring
// those keys to a CU. Two waves per SIMD, each with one tile's K and V in registers (the next
// tile's K is loaded under the softmax and P V, its V under the next Q K), hide each other's
// loads; holding two tiles per wave instead leaves one wave per SIMD and measured 30 us.
// B = 8, Hq = 6, S = 4096 as graph replays: 3923 us with one workgroup per sequence, 26.8 now
// (this kernel 18-20 us, 3.4-3.7 TB/s; the merge 4); B = 16, S = 16384: 99.6 us, 5.4 TB/s.
constexpr int TAIL_MAXQ = 16;
constexpr int TAIL_KT = 16;                    // keys per tile
constexpr int TAIL_NW = 8;                     // waves per workgroup
constexpr int TAIL_QLD = DH + 4;               // q' rows in LDS, padded off each other's banks
constexpr float kNegMax = -3.402823466e38f;    // running max before any key: exp(x - m) is 0 or finite

struct TailArgs {
  const float* query;
  const float* gate;
  const float* q_norm;
  const float* cos;
  const float* sin;
  const float* ck;
  const float* cv;
  const float* mask;
  float* out;
  float* po;    // [B][nsplit][Hq][256] unnormalised partial outputs (nsplit > 1)
  float* pml;   // [B][nsplit][Hq][2] running max and sum
  int Hq, S, nsplit, per;  // per: 16-key tiles of one split
};

__global__ __launch_bounds__(64 * TAIL_NW, 2) void gqa_tail_kernel(TailArgs a) {
  const int b = blockIdx.x / a.nsplit;
  const int sp = blockIdx.x - b * a.nsplit;
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int i = lane & 15, g = lane >> 4;
  const int Hq = a.Hq, S = a.S;
  __shared__ __attribute__((aligned(16))) float s_o[TAIL_NW][TAIL_MAXQ][DH];
  __shared__ float s_ml[TAIL_NW][TAIL_MAXQ][2];
  float (*s_q)[TAIL_QLD] = reinterpret_cast<float (*)[TAIL_QLD]>(&s_o[0][0][0]);

  // The split's tiles of 16 keys, wave w taking every TAIL_NW-th one.
  const int nt = (S + TAIL_KT - 1) / TAIL_KT;
  const int t_hi = min(nt, (sp + 1) * a.per);
  const float* kb = a.ck + (size_t)b * S * DH;
  const float* vb = a.cv + (size_t)b * S * DH;
  // Loads of tile t through buffer descriptors over its rows only: rows past S, and every row
  // when t is past the split, read as 0 without touching memory, so the loads carry no branch
  // (one would make the compiler wait for a tile's V before its K is used).
  auto rows_of = [&](const float* base, int t, int row_bytes) {
    const int rows = t < t_hi ? min(TAIL_KT, S - t * TAIL_KT) : 0;
    return __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float*>(base + (size_t)t * TAIL_KT * (row_bytes / 4)), (short)0,
        rows * row_bytes, 0x00020000);
  };
  auto load_k = [&](int t, f32x4 (&k)[16]) {
    const auto r = rows_of(kb, t, DH * 4);
#pragma unroll
    for (int s = 0; s < 16; ++s)
      k[s] = __builtin_bit_cast(
          f32x4, __builtin_amdgcn_raw_buffer_load_b128(r, i * DH * 4 + g * 16 + 64 * s, 0, 0));
  };
  auto load_v = [&](int t, f32x4 (&v)[4][4], float (&mk)[4]) {
    const auto rv = rows_of(vb, t, DH * 4), rm = rows_of(a.mask, t, 4);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      mk[r] = __builtin_bit_cast(
          float, __builtin_amdgcn_raw_buffer_load_b32(rm, 16 * g + 4 * r, 0, 0));
#pragma unroll
      for (int n = 0; n < 4; ++n)
        v[r][n] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(
                                                rv, (4 * g + r) * DH * 4 + 16 * i + 256 * n, 0, 0));
    }
  };

  // q' rows: wave w prepares rows w and w + 8; rows past Hq are zero. Their loads go out
  // first, then the first tile's, which land while q' is formed.
  f32x4 x[TAIL_MAXQ / TAIL_NW];
#pragma unroll
  for (int u = 0; u < TAIL_MAXQ / TAIL_NW; ++u) {
    const int h = w + TAIL_NW * u;
    x[u] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (h < Hq) {
      const float* src = a.query + ((size_t)b * Hq + h) * DH + 4 * lane;
#pragma unroll
      for (int j = 0; j < 4; ++j) x[u][j] = src[j];
    }
  }
  float nw[4], cs[4] = {1.f, 1.f, 1.f, 1.f}, sn[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int j = 0; j < 4; ++j) nw[j] = 1.0f + a.q_norm[4 * lane + j];
  if (lane < ROPE / 4) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      cs[j] = a.cos[4 * lane + j];
      sn[j] = (lane < ROPE / 8 ? -1.0f : 1.0f) * a.sin[4 * lane + j];
    }
  }
  int t = sp * a.per + w;
  f32x4 kc[16], v[4][4];
  float mk[4];
  load_k(t, kc);
  asm volatile("" ::: "memory");  // K before V, so that K alone is waited for below
  load_v(t, v, mk);
#pragma unroll
  for (int u = 0; u < TAIL_MAXQ / TAIL_NW; ++u) {
    const f32x4 xx = x[u] * x[u];
    const float ss = npn::wave_sum((xx[0] + xx[1]) + (xx[2] + xx[3]));
    const float rn = rsqrtf(ss * (1.0f / DH) + kEps);
    f32x4 y;
#pragma unroll
    for (int j = 0; j < 4; ++j) x[u][j] = nw[j] * (x[u][j] * rn);
#pragma unroll
    for (int j = 0; j < 4; ++j) y[j] = __shfl_xor(x[u][j], 8, 64);
    if (lane < ROPE / 4) {
#pragma unroll
      for (int j = 0; j < 4; ++j) x[u][j] = x[u][j] * cs[j] + y[j] * sn[j];
    }
    *reinterpret_cast<f32x4*>(&s_q[w + TAIL_NW * u][4 * lane]) = x[u];
  }
  __syncthreads();
  f32x4 o[4][4];  // [n][j]: rows 4 g + r = heads, column i = dim 64 n + 4 i + j
#pragma unroll
  for (int n = 0; n < 4; ++n)
#pragma unroll
    for (int j = 0; j < 4; ++j) o[n][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m = kNegMax, l = 0.f;  // of head i, l this lane's keys only
  while (t < t_hi) {
    const int key0 = t * TAIL_KT + 4 * g;  // this lane's keys key0 + r
    const int tn = t + TAIL_NW;
    f32x4 acc[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) acc[c] = f32x4{0.f, 0.f, 0.f, 0.f};
    asm volatile("" ::: "memory");  // q' is read again for each tile: 64 registers less to hold
#pragma unroll
    for (int s = 0; s < 16; ++s) {
      const f32x4 q = *reinterpret_cast<const f32x4*>(&s_q[i][16 * s + 4 * g]);
#pragma unroll
      for (int j = 0; j < 4; ++j)
        acc[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(kc[s][j], q[j], acc[j], 0, 0, 0);
    }
    load_k(tn, kc);  // kc is free again: the next tile's K under the softmax and P V
    const f32x4 dot = (acc[0] + acc[1]) + (acc[2] + acc[3]);
    float sc[4], mt = kNegMax;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      sc[r] = key0 + r < S ? dot[r] * (1.0f / 16.0f) + (1.0f - mk[r]) * -1e9f : -INFINITY;
      mt = fmaxf(mt, sc[r]);
    }
    mt = fmaxf(mt, __shfl_xor(mt, 16, 64));
    mt = fmaxf(mt, __shfl_xor(mt, 32, 64));
    if (__any(mt > m)) {
      const float mn = fmaxf(m, mt);
      const float corr = __expf(m - mn);
      m = mn;
      l *= corr;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float cr = __shfl(corr, 4 * g + r, 64);
#pragma unroll
        for (int n = 0; n < 4; ++n)
#pragma unroll
          for (int j = 0; j < 4; ++j) o[n][j][r] *= cr;
      }
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const float p = __expf(sc[r] - m);
      l += p;
#pragma unroll
      for (int n = 0; n < 4; ++n)
#pragma unroll
        for (int j = 0; j < 4; ++j)
          o[n][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(p, v[r][n][j], o[n][j], 0, 0, 0);
    }
    asm volatile("" ::: "memory");
    load_v(tn, v, mk);
    t = tn;
  }
  l += __shfl_xor(l, 16, 64);
  l += __shfl_xor(l, 32, 64);

  // The waves' (m, l, O), added in wave order.
  __syncthreads();  // every wave is done with q'
  if (g == 0) {
    s_ml[w][i][0] = m;
    s_ml[w][i][1] = l;
  }
#pragma unroll
  for (int r = 0; r < 4; ++r)
    if (4 * g + r < Hq)
#pragma unroll
      for (int n = 0; n < 4; ++n)
        *reinterpret_cast<f32x4*>(&s_o[w][4 * g + r][64 * n + 4 * i]) =
            f32x4{o[n][0][r], o[n][1][r], o[n][2][r], o[n][3][r]};
  __syncthreads();
#pragma unroll 2
  for (int h = tid >> 8; h < Hq; h += TAIL_NW / 4) {
    const int d = tid & (DH - 1);
    float M = kNegMax, L = 0.f, O = 0.f;
#pragma unroll
    for (int u = 0; u < TAIL_NW; ++u) M = fmaxf(M, s_ml[u][h][0]);
#pragma unroll
    for (int u = 0; u < TAIL_NW; ++u) {
      const float f = __expf(s_ml[u][h][0] - M);
      L += f * s_ml[u][h][1];
      O += f * s_o[u][h][d];
    }
    if (a.nsplit == 1) {
      const size_t oi = ((size_t)b * Hq + h) * DH + d;
      a.out[oi] = O / L * npn::sigmoid(a.gate[oi]);
    } else {
      const size_t row = (size_t)blockIdx.x * Hq + h;
      a.po[row * DH + d] = O;
      if (d == 0) {
        a.pml[2 * row] = M;
        a.pml[2 * row + 1] = L;
      }
    }
  }
}

// Log-sum-exp merge of one query row's split partials, in split order within each of four
// interleaved groups; one 256-thread workgroup per (b, h), wave w taking splits w, w + 4, ...
// (loads four splits at a time), lane 4 dims.
__global__ __launch_bounds__(256) void gqa_tail_merge_kernel(TailArgs a) {
  const int b = blockIdx.x / a.Hq;
  const int h = blockIdx.x - b * a.Hq;
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int n = a.nsplit;
  __shared__ __attribute__((aligned(16))) f32x4 s_o[4][64];
  __shared__ float s_ml[4][2];
  const size_t row0 = (size_t)b * n * a.Hq + h;
  const float gate = a.gate[((size_t)b * a.Hq + h) * DH + threadIdx.x];
  float M = kNegMax, L = 0.f;
  f32x4 O = {0.f, 0.f, 0.f, 0.f};
  for (int base = w; base < n; base += 16) {
    float mv[4], lv[4];
    f32x4 ov[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int sp = base + 4 * j;
      const size_t row = row0 + (size_t)(sp < n ? sp : base) * a.Hq;
      mv[j] = a.pml[2 * row];
      lv[j] = sp < n ? a.pml[2 * row + 1] : 0.f;
      ov[j] = *reinterpret_cast<const f32x4*>(a.po + row * DH + 4 * lane);
    }
    float mn = M;
#pragma unroll
    for (int j = 0; j < 4; ++j) mn = fmaxf(mn, mv[j]);
    const float c = __expf(M - mn);
    M = mn;
    L *= c;
    O *= c;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      if (base + 4 * j >= n) break;
      const float f = __expf(mv[j] - M);
      L += f * lv[j];
      O += f * ov[j];
    }
  }
  s_o[w][lane] = O;
  if (lane == 0) {
    s_ml[w][0] = M;
    s_ml[w][1] = L;
  }
  __syncthreads();
  float Mx = kNegMax, Ls = 0.f, Os = 0.f;
#pragma unroll
  for (int u = 0; u < 4; ++u) Mx = fmaxf(Mx, s_ml[u][0]);
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const float f = __expf(s_ml[u][0] - Mx);
    Ls += f * s_ml[u][1];
    Os += f * reinterpret_cast<const float*>(s_o[u])[threadIdx.x];
  }
  a.out[((size_t)b * a.Hq + h) * DH + threadIdx.x] = Os / Ls * npn::sigmoid(gate);
}

// 16-key tiles per workgroup: about one workgroup per CU (512 in all measured 35 against 28 us at
// B = 8, S = 4096: every workgroup pays its own start and merge), each with at least four tiles.
// The floor of four rather than one tile for each of the eight waves puts small problems on
// twice the CUs: B = 1, S = 1024 20.3 -> 17.6 us, B = 1, S = 4096 22.1 -> 20.8; two tiles gave
// 17.4 and 23.
constexpr int kTailWG = 256, kTailMinTiles = 4;
int tail_tiles(int B, int S) {
  const int nt = (S + TAIL_KT - 1) / TAIL_KT;
  const int n = (kTailWG + B / 2) / B;
  const int per = n > 1 ? (nt + n - 1) / n : nt;
  return per > kTailMinTiles ? per : kTailMinTiles;
}
int tail_splits(int B, int S) {
  const int nt = (S + TAIL_KT - 1) / TAIL_KT, per = tail_tiles(B, S);
  return (nt + per - 1) / per;
}

bool tail_shape_ok(int B, int Hq, int S) {
  return B >= 1 && Hq >= 1 && Hq <= TAIL_MAXQ && S >= 1;
}

struct VerifyPlan {
  int grp, R, nrt, P;
  size_t q_bytes, po_bytes, pml_bytes, ps_bytes, total;
};

VerifyPlan plan(int B, int T, int Hq, int Hkv) {
  VerifyPlan p{};
  p.grp = Hq / Hkv;
  p.nrt = (T * p.grp + 15) / 16;
  p.R = p.nrt * 16;
  p.P = B * Hkv;
  const size_t slots = (size_t)kAttnWG + p.P;
  auto up = [](size_t x) { return (x + 255) & ~size_t(255); };
  p.q_bytes = up((size_t)p.P * p.R * DH * 2);
  p.po_bytes = up(slots * p.R * DH * 4);
  p.pml_bytes = up(slots * p.R * 2 * 4);
  p.ps_bytes = up((size_t)(p.P + 2) * 4);
  p.total = 2 * p.q_bytes + p.po_bytes + p.pml_bytes + p.ps_bytes;
  return p;
}

bool verify_shape_ok(int B, int T, int Hq, int Hkv, int s_max) {
  // s_max <= 2^23 keeps cache row offsets in 32 bits; the total step count in int32.
  // B * Hkv is the merge grid's y extent (<= 65535).
  return B >= 1 && (int64_t)B * Hkv <= 65535 && T >= 1 && Hkv >= 1 && Hq >= Hkv && Hq % Hkv == 0 &&
         T * (Hq / Hkv) <= 48 && s_max >= T && s_max <= (1 << 23) &&
         (int64_t)B * Hkv * ((s_max + KS - 1) / KS) < ((int64_t)1 << 31);
}

}  // namespace

extern "C" size_t npn_gqa_tail_verify_workspace_size(int B, int T, int q_heads, int kv_heads,
                                                     int s_max) {
  if (!verify_shape_ok(B, T, q_heads, kv_heads, s_max)) return 0;
  return plan(B, T, q_heads, kv_heads).total;
}

// The verify tail's launches; with app.key set the query-prep launch also appends the new
// K/V rows (the attention launch that follows reads them).
static int tail_verify_launch(const uint16_t* query, const uint16_t* gate, const float* q_norm,
                              RopeSrc rope, const AppendArgs& app, const uint16_t* cache_k,
                              const uint16_t* cache_v, const int32_t* kv_len, uint16_t* out,
                              int B, int T, int q_heads, int kv_heads, int s_max, void* workspace,
                              size_t workspace_bytes, void* stream) {
  NPN_REQUIRE(query && gate && q_norm && rope.cos && rope.sin && cache_k && cache_v && kv_len &&
                  out,
              NPN_ERR_NULL);
  NPN_REQUIRE(verify_shape_ok(B, T, q_heads, kv_heads, s_max), NPN_ERR_SHAPE);
  NPN_REQUIRE(NPN_ALIGNED16(cache_k) && NPN_ALIGNED16(cache_v) && NPN_ALIGNED16(workspace) &&
                  NPN_ALIGNED16(gate) && NPN_ALIGNED16(out),
              NPN_ERR_ALIGN);
  const VerifyPlan p = plan(B, T, q_heads, kv_heads);
  NPN_REQUIRE(workspace != nullptr && workspace_bytes >= p.total, NPN_ERR_WORKSPACE);
  hipStream_t s = static_cast<hipStream_t>(stream);
  uint8_t* ws = static_cast<uint8_t*>(workspace);
  uint16_t* qhi = reinterpret_cast<uint16_t*>(ws);
  uint16_t* qlo = reinterpret_cast<uint16_t*>(ws + p.q_bytes);
  float* po = reinterpret_cast<float*>(ws + 2 * p.q_bytes);
  float* pml = reinterpret_cast<float*>(ws + 2 * p.q_bytes + p.po_bytes);
  int32_t* pstart = reinterpret_cast<int32_t*>(ws + 2 * p.q_bytes + p.po_bytes + p.pml_bytes);

  const int rows = B * kv_heads * p.R;
  const int qblocks = (rows + 3) / 4;
  QPrepArgs qa{query, q_norm, rope, qhi, qlo, kv_len, pstart, B, T, q_heads, kv_heads, p.R,
               p.P, s_max, qblocks, app};
  const int ablocks = app.key != nullptr ? (B * T * kv_heads + 3) / 4 : 0;
  hipLaunchKernelGGL(gqa_qprep_kernel, dim3(1 + qblocks + ablocks), dim3(256), 0, s, qa);

  AttnArgs aa{qhi, qlo, cache_k, cache_v, kv_len, pstart, po, pml, kv_heads, s_max, T, p.grp, p.P};
  const dim3 grid(kAttnWG);
  if (p.nrt == 1) hipLaunchKernelGGL((gqa_attn_kernel<1, 2>), grid, dim3(64), 0, s, aa);
  else if (p.nrt == 2) hipLaunchKernelGGL((gqa_attn_kernel<2, 2>), grid, dim3(128), 0, s, aa);
  else hipLaunchKernelGGL((gqa_attn_kernel<3, 2>), grid, dim3(192), 0, s, aa);

  MergeArgs ma{po, pml, pstart, gate, out, T, q_heads, kv_heads, p.R, p.P};
  if (p.P >= kMergeRowsMinPairs)
    hipLaunchKernelGGL(gqa_merge_rows_kernel, dim3((T * p.grp + 3) / 4, p.P), dim3(256), 0, s,
                       ma);
  else
    hipLaunchKernelGGL(gqa_merge_kernel, dim3(T * p.grp, p.P), dim3(256), 0, s, ma);
  return npn_launch_status();
}

extern "C" int npn_gqa_tail_verify(const uint16_t* query, const uint16_t* gate,
                                   const float* q_norm, const float* cos, const float* sin,
                                   const uint16_t* cache_k, const uint16_t* cache_v,
                                   const int32_t* kv_len, uint16_t* out, int B, int T,
                                   int q_heads, int kv_heads, int s_max, void* workspace,
                                   size_t workspace_bytes, void* stream) {
  AppendArgs none{};
  return tail_verify_launch(query, gate, q_norm, RopeSrc{cos, sin, 0}, none, cache_k, cache_v,
                            kv_len, out, B, T, q_heads, kv_heads, s_max, workspace,
                            workspace_bytes, stream);
}

extern "C" int npn_gqa_tail_verify_append(const uint16_t* query, const uint16_t* gate,
                                          const uint16_t* key, const uint16_t* value,
                                          const float* q_norm, const float* k_norm,
                                          const float* cos_table, const float* sin_table,
                                          int positions, uint16_t* cache_k, uint16_t* cache_v,
                                          const int32_t* kv_len, uint16_t* out, int B, int T,
                                          int q_heads, int kv_heads, int s_max, void* workspace,
                                          size_t workspace_bytes, void* stream) {
  NPN_REQUIRE(key && value && k_norm, NPN_ERR_NULL);
  NPN_REQUIRE(positions >= 1, NPN_ERR_SHAPE);
  NPN_REQUIRE(NPN_ALIGNED16(cos_table) && NPN_ALIGNED16(sin_table), NPN_ERR_ALIGN);
  const RopeSrc rope{cos_table, sin_table, positions};
  const AppendArgs app{key, value, k_norm, rope, cache_k, cache_v, kv_len, B, T, kv_heads, s_max};
  return tail_verify_launch(query, gate, q_norm, rope, app, cache_k, cache_v, kv_len, out, B, T,
                            q_heads, kv_heads, s_max, workspace, workspace_bytes, stream);
}

extern "C" int npn_gqa_kv_append(const uint16_t* key, const uint16_t* value, const float* k_norm,
                                 const float* cos, const float* sin, uint16_t* cache_k,
                                 uint16_t* cache_v, const int32_t* kv_len, int B, int T,
                                 int kv_heads, int s_max, void* stream) {
  NPN_REQUIRE(key && value && k_norm && cos && sin && cache_k && cache_v && kv_len, NPN_ERR_NULL);
  NPN_REQUIRE(B >= 1 && T >= 1 && kv_heads >= 1 && s_max >= T, NPN_ERR_SHAPE);
  AppendArgs aa{key, value, k_norm, RopeSrc{cos, sin, 0}, cache_k, cache_v, kv_len, B, T,
                kv_heads, s_max};
  const int waves = B * T * kv_heads;
  hipLaunchKernelGGL(gqa_kv_append_kernel, dim3((waves + 3) / 4), dim3(256), 0,
                     static_cast<hipStream_t>(stream), aa);
  return npn_launch_status();
}

extern "C" size_t npn_gqa_tail_workspace_size(int B, int q_heads, int S) {
  if (!tail_shape_ok(B, q_heads, S)) return 0;
  const size_t n = tail_splits(B, S);
  // at least 16 bytes, so that 0 means an unsupported shape
  return n == 1 ? 16 : (size_t)B * n * q_heads * (DH + 2) * sizeof(float);
}

static int tail_launch(const float* query, const float* gate, const float* q_norm,
                       const float* cos, const float* sin, const float* cached_k,
                       const float* cached_v, const float* mask, float* out, int B, int q_heads,
                       int S, int per, float* ws, void* stream) {
  NPN_REQUIRE(query && gate && q_norm && cos && sin && cached_k && cached_v && mask && out,
              NPN_ERR_NULL);
  NPN_REQUIRE(tail_shape_ok(B, q_heads, S), NPN_ERR_SHAPE);
  NPN_REQUIRE(NPN_ALIGNED16(cached_k) && NPN_ALIGNED16(cached_v), NPN_ERR_ALIGN);
  hipStream_t s = static_cast<hipStream_t>(stream);
  const int nt = (S + TAIL_KT - 1) / TAIL_KT, nsplit = (nt + per - 1) / per;
  float* pml = nsplit > 1 ? ws + (size_t)B * nsplit * q_heads * DH : nullptr;
  const TailArgs a{query, gate, q_norm, cos, sin, cached_k, cached_v, mask, out, ws, pml,
                   q_heads, S, nsplit, per};
  hipLaunchKernelGGL(gqa_tail_kernel, dim3(B * nsplit), dim3(64 * TAIL_NW), 0, s, a);
  if (nsplit > 1)
    hipLaunchKernelGGL(gqa_tail_merge_kernel, dim3(B * q_heads), dim3(256), 0, s, a);
  return npn_launch_status();
}

extern "C" int npn_gqa_tail(const float* query, const float* gate, const float* q_norm,
                            const float* cos, const float* sin, const float* cached_k,
                            const float* cached_v, const float* mask, float* out, int B,
                            int q_heads, int S, void* stream) {
  return tail_launch(query, gate, q_norm, cos, sin, cached_k, cached_v, mask, out, B, q_heads, S,
                     S, nullptr, stream);  // S tiles: at least every tile of the sequence
}

extern "C" int npn_gqa_tail_split(const float* query, const float* gate, const float* q_norm,
                                  const float* cos, const float* sin, const float* cached_k,
                                  const float* cached_v, const float* mask, float* out, int B,
                                  int q_heads, int S, void* workspace, size_t workspace_bytes,
                                  void* stream) {
  NPN_REQUIRE(tail_shape_ok(B, q_heads, S), NPN_ERR_SHAPE);
  NPN_REQUIRE(NPN_ALIGNED16(workspace), NPN_ERR_ALIGN);
  NPN_REQUIRE(workspace != nullptr &&
                  workspace_bytes >= npn_gqa_tail_workspace_size(B, q_heads, S),
              NPN_ERR_WORKSPACE);
  return tail_launch(query, gate, q_norm, cos, sin, cached_k, cached_v, mask, out, B, q_heads, S,
                     tail_tiles(B, S), static_cast<float*>(workspace), stream);
}
