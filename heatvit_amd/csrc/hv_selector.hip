// hv_selector.hip -- token selector (selector.token_selector,
// selector.py:503-563) over a ragged batch.
//
// k_selector_image, one 1024-thread workgroup per image (XCD-major): the
//   three heads' local MLP + head statistic (:253, :358), candidate mean
//   (:273), concat + 64->32->16->2 score MLP + 2-way selector softmax
//   (:292, :307, :338) as int8 MFMAs over tiles of 16 candidates, every
//   weight and intermediate in LDS; then, per candidate, the head-weight
//   MLP with PLAN (:370) and the head fuse (:392); the stable keep list
//   (fused >= 32768) and the per-image state of finalize_tokens (:456-500);
//   and the package token (score-weighted mean of the pruned normals plus
//   the incoming package, or their plain mean when the scores sum to
//   zero), written to a per-image scratch row.  Each candidate row is read
//   from memory by this workgroup only.
// k_selector_keep (finalize_tokens from given fused scores): the keep list
//   and state of one image per workgroup.
// k_selector_compact (the same): the image's output offset (the token counts
//   of the images before it), then CLS, the kept rows in input order and the
//   package row there (stream compaction).  k_selector_image's outputs take
//   k_selector_rows, which can also write the rows' LayerNorm.
//
// GELU layers use the int32 requant/GELU path when the host finds every
// shift in [-30, 30] and each layer's biases satisfy |b| <= 2^30 - 1 -
// K*2^14 (checked per head, uniform); otherwise the exact 64-bit form.
#include <type_traits>

#include "hv_device.h"
#include "hv_internal.h"
#include "gelu_lut.inc"  // generated at build time by gen_gelu_lut.py

namespace hv {

// A GELU layer's step table (gen_gelu_lut.py) when its output shift has one:
// words [off, off + words) of kGeluLut, clamp [qlo, qhi], cb as gelu_table
// takes it; off < 0: the layer evaluates ShiftGELU.
struct SelLut {
  int off, words, qlo, qhi, cb;
};

// Copies a step table into LDS with 16-byte loads, four rounds in flight
// (tables start on 16-byte boundaries and hold a multiple of four words).
// All NT threads call it; the caller puts a barrier after it.
template <int NT>
__device__ __forceinline__ void sel_stage_lut(const SelLut &t, unsigned *lut, int tid) {
  const v4i *src = reinterpret_cast<const v4i *>(kGeluLut + t.off);
  v4i *dst = reinterpret_cast<v4i *>(lut);
  const int n4 = t.words >> 2;
  for (int base = tid; base < n4; base += 4 * NT) {
    v4i v[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) v[r] = src[min(base + r * NT, n4 - 1)];
#pragma unroll
    for (int r = 0; r < 4; ++r) dst[min(base + r * NT, n4 - 1)] = v[r];
  }
}

// A step table held in registers between its loads and its LDS stores, so
// a layer's table loads can be in flight while the previous layer runs
// (NT threads, at most kLutRegs 16-byte words each).
constexpr int kLutRegs = 4;
template <int NT>
__device__ __forceinline__ void lut_load(const SelLut &t, v4i (&v)[kLutRegs], int tid) {
  static_assert(kGeluLutMaxWords / 4 <= kLutRegs * NT, "one round of table loads");
  const v4i *src = reinterpret_cast<const v4i *>(kGeluLut + t.off);
  const int n4 = t.words >> 2;
#pragma unroll
  for (int r = 0; r < kLutRegs; ++r) v[r] = src[min(tid + r * NT, n4 - 1)];
}
template <int NT>
__device__ __forceinline__ void lut_store(const SelLut &t, const v4i (&v)[kLutRegs],
                                          unsigned *lut, int tid) {
  const int n4 = t.words >> 2;
#pragma unroll
  for (int r = 0; r < kLutRegs; ++r) reinterpret_cast<v4i *>(lut)[min(tid + r * NT, n4 - 1)] = v[r];
}

static constexpr int kMaxCand = 196;

__device__ __forceinline__ int dot4(int a, int b, int c) {
  return __builtin_amdgcn_sdot4(a, b, c, false);
}

__device__ __noinline__ int gelu_exact(int acc, int bias, int sh_in, int sh_out) {
  return gelu_post((i64)acc + bias, sh_in, sh_out);
}

// requant(gelu(requant(acc + bias, src, -16, 24)), -16, dst, 8).
__device__ __forceinline__ int sel_gelu(int acc, int bias, bool fast, const Rq &ra, const Rq &rb,
                                        int sh_in, int sh_out) {
  if (fast) return rq(gelu_q16(rq(acc + bias, ra)), rb);
  return gelu_exact(acc, bias, sh_in, sh_out);
}

// The same with a 64-bit bias (score layer 1 after its global half is
// folded into the bias, below).
__device__ __noinline__ int gelu_exact64(int acc, i64 bias, int sh_in, int sh_out) {
  return gelu_post((i64)acc + bias, sh_in, sh_out);
}

constexpr int kCandTiles = (kMaxCand + 15) / 16;  // 13 tiles of 16 candidates
constexpr int kCandPad = kCandTiles * 16;

// Image of logical index L = XCD-major order of workgroup blockIdx.x over a
// grid that is a multiple of 8: workgroups go round-robin over the 8 XCDs,
// so XCD x runs images [x * B8, (x + 1) * B8).  -1 past the batch.
__device__ __forceinline__ int xcd_image(int batch) {
  const int B8 = (batch + 7) >> 3;
  const int L = (blockIdx.x & 7) * B8 + (blockIdx.x >> 3);
  return L < batch ? L : -1;
}

// An image the selector takes: CLS plus at least one candidate
// (selector.py:513-514), at most 196 candidates, and with an incoming
// package a normal candidate beside it (:448-449).
__device__ __forceinline__ bool image_ok(int row0, int C, int pkg) {
  return C >= 1 && C <= kMaxCand && C - pkg >= 1 && row0 >= 0;
}

__device__ __forceinline__ void state_invalid(int32_t *st) {
  st[0] = -1; st[1] = 0; st[2] = 0; st[3] = 0; st[4] = 0;
}

// Head fuse (selector.py:370-418), in three steps over one thread per
// candidate and head-weight unit: the head-weight MLP's GELU layer on the
// head statistics (3 -> 3), its PLAN layer (3 -> 3), and the weighted mean
// of the head scores (plain mean, and the warning, when the weights sum to
// zero).  The biases are any int32 and the reference adds them in int64
// (gemm.py:118-119): the three products (|sum| < 2^16; weights and bias from
// LDS) are summed in 32 bits and the bias added in 64; the empty asm keeps the
// compiler from folding bias and products into one 32-bit dot-product
// accumulation, which wraps for biases near the int32 limits.
__device__ __forceinline__ int fuse_hidden(const hv_selector_dev &p, const int8_t *stats,
                                           const int *wt, int bias) {
  const int a_in = -16 - (p.stats_out_exp + p.hw_w1_exp), a_out = p.hw_hidden_out_exp + 16;
  int dot = 0;
#pragma unroll
  for (int k = 0; k < 3; ++k) dot += (int)stats[k] * wt[k];
  asm volatile("" : "+v"(dot));
  return gelu_post((i64)bias + dot, a_in, a_out);
}

__device__ __forceinline__ int fuse_weight(const hv_selector_dev &p, const int *hid, const int *wt,
                                           int bias) {
  const int b_sh = -16 - (p.hw_hidden_out_exp + p.hw_w2_exp);
  int dot = 0;
#pragma unroll
  for (int k = 0; k < 3; ++k) dot += hid[k] * wt[k];
  asm volatile("" : "+v"(dot));
  return sat_q016(plan_sigmoid((int)requant_shift((i64)bias + dot, b_sh, 24)));
}

// hs[0], hs[kMaxCand], hs[2 * kMaxCand]: the candidate's head scores; w[0..2]
// its head weights.
__device__ __forceinline__ int fuse_mean(const int32_t *hs, const int *w, bool *warn) {
  i64 num = 0, den = 0;
#pragma unroll
  for (int j = 0; j < 3; ++j) {
    num += (i64)hs[j * kMaxCand] * w[j];
    den += w[j];
  }
  *warn = den == 0;
  if (den == 0) {
    num = (i64)hs[0] + hs[kMaxCand] + hs[2 * kMaxCand];
    den = 3;
  }
  return sat_q016(round_div_pos_d(num, den));  // num < 2^35, den < 2^18
}

// The stable keep list and state of one image (selector.py:456-500) from
// the fused scores: thread c (c < 256) holds candidate c's score fc (0 past
// C) and its head-fuse warning; every thread of the NT-thread workgroup
// calls it.  Writes kept_index ki[0 .. kept) = the kept normals (fused >=
// 32768) in input order, ki[kept .. 196) = -1, and the state {token_count,
// package_present, kept, pruned, warnings}; bad (any thread) marks the
// image invalid (state token count -1).  Returns the kept count, or -1 when
// the image is invalid; *den_out receives the sum of the partitioned
// candidates' scores (the package's divisor), thread 0's *warn_out the
// image's warning bits.
template <int NT>
__device__ __forceinline__ int keep_list(int C, int pkg, int fc, bool warn, bool bad, int32_t *ki,
                                         int32_t *st, i64 *den_out = nullptr,
                                         int *warn_out = nullptr) {
  constexpr int NWAVE = NT / 64;
  __shared__ int w_kept[NWAVE], w_flags[NWAVE], w_den[NWAVE];
  const int c = threadIdx.x, lane = c & 63, wave = c >> 6;
  const int n_norm = C - pkg;
  const bool is_norm = c < n_norm;
  const bool keep = is_norm && fc >= 32768;
  const bool part = (is_norm && !keep) || (pkg && c == C - 1);
  const u64 mask = __ballot(keep);
  // valid scores are at most 65536, so a wavefront's sum fits 32 bits (an
  // invalid image is rejected below before the sum is used)
  int d = part ? fc : 0;
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) d += __shfl_xor(d, off);
  const int flags = (__ballot(warn) != 0 ? 1 : 0) | (__ballot(bad) != 0 ? 2 : 0);
  if (lane == 0) {
    w_kept[wave] = __popcll(mask);
    w_den[wave] = d;
    w_flags[wave] = flags;
  }
  __syncthreads();
  int before = __popcll(mask & ((1ull << lane) - 1ull)), kept = 0, any = 0;
  i64 den = 0;
#pragma unroll
  for (int w = 0; w < NWAVE; ++w) {
    before += w < wave ? w_kept[w] : 0;
    kept += w_kept[w];
    den += w_den[w];
    any |= w_flags[w];
  }
  if (any & 2) {
    if (c == 0) state_invalid(st);
    return -1;
  }
  if (den_out) *den_out = den;
  if (keep) ki[before] = c;
  if (c >= kept && c < kMaxCand) ki[c] = -1;
  if (c == 0) {
    const int n_part = C - kept;  // pruned normals + the incoming package
    const int exists = n_part > 0;
    st[0] = 1 + kept + exists;
    st[1] = exists;
    st[2] = kept;
    st[3] = n_part - pkg;
    const int warn_bits = ((any & 1) ? HV_WARN_HEAD_DEN_ZERO : 0) |
                          ((exists && den == 0) ? HV_WARN_PACKAGE_DEN_ZERO : 0);
    st[4] = warn_bits;
    if (warn_out) *warn_out = warn_bits;
  }
  return kept;
}

// Package token of one image (selector.py:470-500): dst[ch] = sat8(
// round_div(sum_c w_c x_c[ch], sum_c w_c)) over the pruned normals and the
// incoming package with w_c = fused score, or their plain mean (w_c = 1,
// divisor n_part) when those scores sum to zero (den: the scores' sum, from
// keep_list).  |num| <= 196 * 65536 *
// 128 < 2^31.  Thread c holds candidate c's fused score fv; thread (channel
// group of 16, candidate group g < G) accumulates candidates g, g + G, ...
// (its candidate rows loaded at once, weight 0 for kept ones) and part_sum
// ([G][192] ints) sums the groups.  Every thread of the NT-thread workgroup
// calls it; cand points at candidate 0's row (16-byte aligned rows, RS
// bytes apart, in memory or LDS).
template <int NT, int RS, int G, int Q>
__device__ __forceinline__ void package_row(const int8_t *cand, int C, int pkg, int kept, int fv,
                                            i64 den, int8_t *dst, int *wgt, int *part_sum) {
  constexpr int kSteps = (kMaxCand + G - 1) / G;
  static_assert(12 * G <= NT && G % Q == 0 && 192 * Q <= NT, "one thread per sum");
  // 208-word rows put a quad's four reads G / 4 rows apart (G = 36) on
  // disjoint runs of 16 banks
  constexpr int kPS = Q == 1 ? 192 : 208;
  const int tid = threadIdx.x;
  const int cg = tid / 12, chg = tid - cg * 12;
  v4i xv[kSteps];
  if (tid < 12 * G) {
    const int8_t *cp = cand + chg * 16;
#pragma unroll
    for (int j = 0; j < kSteps; ++j)
      xv[j] = *reinterpret_cast<const v4i *>(cp + (size_t)min(cg + G * j, C - 1) * RS);
  }
  const int n_norm = C - pkg;
  const bool part = tid < C && ((tid < n_norm && fv < 32768) || (pkg && tid == C - 1));
  if (tid < C) wgt[tid] = part ? (den == 0 ? 1 : fv) : 0;
  __syncthreads();
  if (tid < 12 * G) {
    int acc[16];
#pragma unroll
    for (int j = 0; j < 16; ++j) acc[j] = 0;
#pragma unroll
    for (int j = 0; j < kSteps; ++j) {
      const int c = cg + G * j;
      const int w = c < C ? wgt[c] : 0;
#pragma unroll
      for (int k = 0; k < 16; ++k)
        acc[k] += __mul24(w, (int)(int8_t)(xv[j][k >> 2] >> (8 * (k & 3))));
    }
#pragma unroll
    for (int j = 0; j < 16; ++j) part_sum[cg * kPS + chg * 16 + j] = acc[j];
  }
  __syncthreads();
  const int n_part = C - kept;
  if (tid < 192 * Q) {
    const int ch = tid / Q, g0 = tid % Q * (G / Q);
    int num = 0;
#pragma unroll
    for (int g = 0; g < G / Q; ++g) num += part_sum[(g0 + g) * kPS + ch];
    if constexpr (Q == 4) {  // over the quad
      num += __builtin_amdgcn_update_dpp(0, num, 0xB1, 0xf, 0xf, false);  // lane ^ 1
      num += __builtin_amdgcn_update_dpp(0, num, 0x4E, 0xf, 0xf, false);  // lane ^ 2
    }
    dst[ch] = (int8_t)sat_bits(round_div_pos_d(num, den == 0 ? n_part : den), 8);
  }
}

// N GELU post-ops of a layer from its step table in LDS, packed four
// to a word: q = rsa(v, s) (or v << -s after the pre-clamp) with the
// direction of the launch-uniform shift chosen once; the table's clamp
// [qlo, qhi] lies inside the 24-bit range, so q needs no clamp of its own.
template <int N>
__device__ __forceinline__ void sel_gelu_pack(const int (&v)[N], const Rq &ra, const unsigned *lut,
                                              const SelLut &t, unsigned (&ow)[N / 4]) {
  int q[N];
  if (ra.s > 0) {
#pragma unroll
    for (int i = 0; i < N; ++i) q[i] = (v[i] + ra.rnd + (v[i] >> 31)) >> ra.s;
  } else {
#pragma unroll
    for (int i = 0; i < N; ++i) q[i] = min(max(v[i], ra.vlo), ra.vhi) << -ra.s;
  }
  gelu_table_pack_n<N>(q, ow, lut, t.cb, t.qlo, t.qhi);
}

// Orders this wavefront's LDS accesses before and after it as written (one
// wavefront's LDS operations complete in order: no wait is needed).
__device__ __forceinline__ void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

constexpr int kImgThreads = 1024, kXsRow = 208;

// One workgroup per image (XCD-major).  The three heads' (head, candidate
// tile of 16) units run over the sixteen wavefronts, every unit's two column
// tiles in one wavefront:
//   local = GELU(x_h [C][64] . Wl [64][32] + bl)     16x16x64, 2 column tiles
//   h1    = GELU(local . W1[0:32] + b1')             16x16x32, 2 column tiles
//   h2    = GELU(h1 . W2 + b2)                       16x16x32, 1 column tile
// where b1' = b1 + global . W1[32:64] (the global feature is the same for
// every candidate, so the concat's second half is a per-head bias, exact in
// 64 bits).  With the weights as the MFMA's first operand, result lane l of
// a tile holds output channels 16 ct + 4 (l / 16) + i of candidate l % 16,
// stored as one word.  h1 and h2 of a unit depend only on its own local
// rows, so both score layers run in one pass that rewrites the unit's rows
// in place.  Logits (16 -> 2) and the 2-way softmax are per candidate; the
// head fuse, the keep list and the package token follow in the same
// workgroup.  The package row goes to pkg_rows[b] for k_selector_rows.
//
// Bound by the latency of its dependent phases (one workgroup per CU) and,
// in the three GELU layers, by the CU's VALU issue.  So the unit index is
// scalar, the biases start the accumulators, the head statistic is one MFMA
// by ones, two step tables sit in LDS side by side, the head-weight layers
// run in wavefronts that the global mean and fold leave idle, and constants
// come from LDS, not memory, in the serial phases.  Over 64 sets of 197 tokens
// 23.6 -> 19.2 us, 256 images 26.5 -> 20.3; of the earlier form's 22 us the
// local layer took 5.8, score layer 1 4.3 and score layer 2 1.9 (units split
// by column tile left every third round half empty), the head fuse 2.7 and the
// package 1.8.
__global__ __launch_bounds__(kImgThreads) void k_selector_image(
    hv_selector_dev p, const int8_t *tokens, const int32_t *offsets, int batch,
    const uint8_t *pkg_in, int fast_shifts, hv_selector_ckpt ck, SelLut tl, SelLut t1, SelLut t2,
    int32_t *fused_out, int32_t *kept_index, int32_t *state, int8_t *pkg_rows,
    int32_t *img_warn) {
  constexpr int NT = kImgThreads, NW = NT / 64;
  // step tables: [0, kGeluLutMaxWords) the local layer's, then score layer
  // 2's; the second half score layer 1's; last the package sums
  __shared__ __attribute__((aligned(16))) unsigned lut[2 * kGeluLutMaxWords];
  unsigned *const lut_b = lut + kGeluLutMaxWords;
  __shared__ __attribute__((aligned(16))) int8_t wl[3][32 * 64];   // local_wt[h] [32][64]
  __shared__ __attribute__((aligned(16))) int8_t w1[3][32 * 64];   // w1t[h] [32][64]
  __shared__ __attribute__((aligned(16))) int8_t w2[3][16 * 32];   // w2t[h] [16][32]
  __shared__ int w3[3][8];                                         // w3t[h] [2][16] as words
  __shared__ __attribute__((aligned(16))) int bl[3][32], bb2[3][16];
  __shared__ int b1_s[3][32], b3_s[6];
  __shared__ int hwc[24];  // hw_w1t [3][3], hw_w2t [3][3], hw_b1 [3], hw_b2 [3]
  // b1 + global . W1[32:64]: its low 32 bits (exact where the int32 form runs) and in full
  __shared__ __attribute__((aligned(16))) int bb1[3][32];
  __shared__ i64 bbx[3][32];
  // a unit's rows [candidate][32]: local, then h1, then h2 in the first 16 bytes
  __shared__ __attribute__((aligned(16))) int8_t act[3 * kCandPad * 32];
  __shared__ int hs_s[3 * kMaxCand];                               // head scores [h][c]
  __shared__ int8_t st_s[kMaxCand * 3];                            // head statistics [c][h]
  __shared__ int hid_s[3 * kMaxCand], hw_s[3 * kMaxCand];          // head-weight MLP [c][j]
  __shared__ unsigned part[5][24][2];
  __shared__ __attribute__((aligned(16))) int8_t glob_s[3][32];
  __shared__ int fast_s[3][3];
  __shared__ int wgt[kMaxCand];
  // the image's candidate rows, 208-byte stride (conflict-free 16-byte
  // fragment reads of 16 consecutive rows)
  __shared__ __attribute__((aligned(16))) int8_t xs[kMaxCand * kXsRow];

  const int b = xcd_image(batch);
  if (b < 0) return;  // uniform: before any barrier
  const int tid = threadIdx.x, lane = tid & 63, col = lane & 15, grp = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int row0 = offsets[b], N = offsets[b + 1] - row0, C = N - 1;
  const int pkg = pkg_in ? (pkg_in[b] ? 1 : 0) : 0;
  int32_t *st = state + (size_t)b * 5;
  if (!image_ok(row0, C, pkg)) {
    if (tid == 0) state_invalid(st);
    return;
  }
  const int ntiles = (C + 15) >> 4, nu = 3 * ntiles;
  const int8_t *cand = tokens + (size_t)(row0 + 1) * 192;
  // Candidate rows into LDS: every 16-byte load of the image in flight at
  // once (items past the end repeat the last one), stored after the weight
  // and table loads below are issued.
  constexpr int kRowItems = (kMaxCand * 12 + NT - 1) / NT;
  v4i rv[kRowItems];
  const int n_items = C * 12;
#pragma unroll
  for (int j = 0; j < kRowItems; ++j)
    rv[j] = reinterpret_cast<const v4i *>(cand)[min(tid + j * NT, n_items - 1)];

  for (int i = tid; i < 3 * 128; i += NT) {  // 16-byte words of the three heads' weights
    const int h = i >> 7, k = i & 127;
    reinterpret_cast<v4i *>(wl[h])[k] = reinterpret_cast<const v4i *>(p.local_wt + h * 2048)[k];
    reinterpret_cast<v4i *>(w1[h])[k] = reinterpret_cast<const v4i *>(p.w1t + h * 2048)[k];
    if (k < 32)
      reinterpret_cast<v4i *>(w2[h])[k] = reinterpret_cast<const v4i *>(p.w2t + h * 512)[k];
  }
  // int32 GELU preconditions per head: |acc| <= K*2^14 for the layer's K
  // (head h's biases sit in one run of lanes of one wavefront: a ballot).
  const int lim64 = (1 << 30) - 1 - 64 * 16384, lim32 = (1 << 30) - 1 - 32 * 16384;
  if (tid < 24) w3[tid >> 3][tid & 7] = reinterpret_cast<const int *>(p.w3t)[tid];
  if (tid >= 64 && tid < 160) {  // local biases: head h in lanes 32 (h % 2) .. +31
    const int v = p.local_b[tid - 64], h = (tid - 64) >> 5;
    bl[h][(tid - 64) & 31] = v;
    const u64 m = __ballot(fast_shifts && v <= lim64 && v >= -lim64);
    if ((tid & 31) == 0) fast_s[h][0] = (unsigned)(m >> (tid & 32)) == 0xFFFFFFFFu;
  }
  if (tid >= 192 && tid < 240) {  // score layer 2 biases: head h in lanes 16 h .. +15
    const int v = p.b2[tid - 192], h = (tid - 192) >> 4;
    bb2[h][(tid - 192) & 15] = v;
    const u64 m = __ballot(fast_shifts && v <= lim32 && v >= -lim32);
    if ((tid & 15) == 0) fast_s[h][2] = ((unsigned)(m >> (16 * h)) & 0xFFFFu) == 0xFFFFu;
  }
  if (tid >= 256 && tid < 352) b1_s[(tid - 256) >> 5][tid & 31] = p.b1[tid - 256];
  if (tid >= 384 && tid < 390) b3_s[tid - 384] = p.b3[tid - 384];
  if (tid >= 448 && tid < 472) {
    const int i = tid - 448;
    hwc[i] = i < 9 ? p.hw_w1t[i] : i < 18 ? p.hw_w2t[i - 9] : i < 21 ? p.hw_b1[i - 18]
                                                                     : p.hw_b2[i - 21];
  }
  if (tl.off >= 0) sel_stage_lut<NT>(tl, lut, tid);
#pragma unroll
  for (int j = 0; j < kRowItems; ++j) {
    const int i = min(tid + j * NT, n_items - 1), c = i / 12;
    *reinterpret_cast<v4i *>(&xs[c * kXsRow + (i - c * 12) * 16]) = rv[j];
  }
  // the score layers' table loads in flight during the local layer
  v4i lv1[kLutRegs], lv2[kLutRegs];
  if (t1.off >= 0) lut_load<NT>(t1, lv1, tid);
  if (t2.off >= 0) lut_load<NT>(t2, lv2, tid);
  __syncthreads();

  // Local MLP and head statistics.
  {
    const int sh_in = -16 - (p.in_exp + p.local_w_exp), sh_out = p.local_out_exp + 16;
    const Rq ra = rq_setup(sh_in, -(1 << 23), (1 << 23) - 1), rb = rq_setup(sh_out, -128, 127);
    const v4i ones = v4i{0x01010101, 0x01010101, 0x01010101, 0x01010101};
    for (int u = wave; u < nu; u += NW) {
      const int h = (u >= ntiles ? 1 : 0) + (u >= 2 * ntiles ? 1 : 0);  // u / ntiles (< 3)
      const int rt = u - h * ntiles, cc = rt * 16 + col;
      const bool small = __builtin_amdgcn_readfirstlane(fast_s[h][0]) != 0;
      const bool table = small && tl.off >= 0;
      const v4i a =
          *reinterpret_cast<const v4i *>(&xs[min(cc, C - 1) * kXsRow + h * 64 + grp * 16]);
      v4i bias[2], acc[2];
#pragma unroll
      for (int ct = 0; ct < 2; ++ct) {
        bias[ct] = *reinterpret_cast<const v4i *>(&bl[h][ct * 16 + 4 * grp]);
        const v4i wb = *reinterpret_cast<const v4i *>(&wl[h][(ct * 16 + col) * 64 + grp * 16]);
        acc[ct] =
            __builtin_amdgcn_mfma_i32_16x16x64_i8(wb, a, table ? bias[ct] : v4i{0}, 0, 0, 0);
      }
      // lane mean of the candidate's 64 head lanes (selector.py:358-367):
      // |sum| / 64 <= 128 needs no clamp below, and 127 * 64 none above
      const int sum = __builtin_amdgcn_mfma_i32_16x16x64_i8(ones, a, v4i{0}, 0, 0, 0)[0];
      if (grp == 0 && cc < C) {
        const int8_t stat = (int8_t)((sum + 32 + (sum >> 31)) >> 6);
        st_s[cc * 3 + h] = stat;
        if (ck.head_stats) ck.head_stats[((size_t)b * kMaxCand + cc) * 3 + h] = stat;
      }
      unsigned ow[2];
      if (table) {
        const int vv[8] = {acc[0][0], acc[0][1], acc[0][2], acc[0][3],
                           acc[1][0], acc[1][1], acc[1][2], acc[1][3]};
        sel_gelu_pack<8>(vv, ra, lut, tl, ow);
      } else {
#pragma unroll
        for (int ct = 0; ct < 2; ++ct) {
          unsigned o[4];
#pragma unroll
          for (int i = 0; i < 4; ++i)
            o[i] = (unsigned)sel_gelu(acc[ct][i], bias[ct][i], small, ra, rb, sh_in, sh_out);
          ow[ct] = pack_lo4(o[0], o[1], o[2], o[3]);
        }
      }
      unsigned *dst = reinterpret_cast<unsigned *>(&act[(h * kCandPad + cc) * 32 + 4 * grp]);
      dst[0] = ow[0];
      dst[4] = ow[1];
    }
  }
  if (t1.off >= 0) lut_store<NT>(t1, lv1, lut_b, tid);
  __syncthreads();
  // score layer 2's table replaces the local layer's (barriers follow)
  if (t2.off >= 0) lut_store<NT>(t2, lv2, lut, tid);
  // Global features = sat8(round_div(sum_c local, C)) per head and channel:
  // five wavefronts per head, one word of four channels per lane, summed as
  // unsigned bytes (x + 128) in two 16-bit halves (196 * 255 < 2^16).
  if (wave < 15) {
    const int h = wave / 5, q = wave - 5 * h;
    const unsigned *ap = reinterpret_cast<const unsigned *>(act + h * kCandPad * 32);
    unsigned s0 = 0, s1 = 0;  // channels 4 w, 4 w + 2 and 4 w + 1, 4 w + 3
#pragma unroll
    for (int k = 0; k < 5; ++k) {
      const int c = 40 * k + 8 * q + (lane >> 3);  // < kCandPad
      const unsigned x = c < C ? ap[c * 8 + (lane & 7)] ^ 0x80808080u : 0u;
      s0 += x & 0x00FF00FFu;
      s1 += (x >> 8) & 0x00FF00FFu;
    }
#pragma unroll
    for (int off = 8; off <= 32; off <<= 1) {
      s0 += __shfl_xor(s0, off);
      s1 += __shfl_xor(s1, off);
    }
    if (lane < 8) {
      part[q][h * 8 + lane][0] = s0;
      part[q][h * 8 + lane][1] = s1;
    }
  }
  if (ck.local)
    for (int i = tid; i < 3 * C * 2; i += NT) {
      const int h = i / (C * 2), k = i - h * C * 2;
      reinterpret_cast<v4i *>(ck.local + ((size_t)b * 3 + h) * kMaxCand * 32)[k] =
          reinterpret_cast<const v4i *>(act + h * kCandPad * 32)[k];
    }
  __syncthreads();
  if (wave < 3) {
    // Wavefront h: head h's mean, then its fold into the bias.
    const int h = wave;
    if (lane < 32) {
      unsigned s = 0;
#pragma unroll
      for (int q = 0; q < 5; ++q) s += part[q][h * 8 + (lane >> 2)][lane & 1];
      const int sacc = (int)((s >> (8 * (lane & 2))) & 0xFFFFu) - 128 * C;
      const int gv = (int)sat_bits(round_div_pos_d(sacc, C), 8);
      glob_s[h][lane] = (int8_t)gv;
      if (ck.global) ck.global[((size_t)b * 3 + h) * 32 + lane] = (int8_t)gv;
    }
    wave_lds_fence();
    if (lane < 32) {
      // global . W1[32:64] in 32 bits (|sum| <= 32 * 128 * 127), the bias in 64
      const int *wr = reinterpret_cast<const int *>(&w1[h][lane * 64 + 32]);
      const int *gw = reinterpret_cast<const int *>(glob_s[h]);
      int dot = 0;
#pragma unroll
      for (int q = 0; q < 8; ++q) dot = dot4(gw[q], wr[q], dot);
      const i64 v = (i64)b1_s[h][lane] + dot;
      bbx[h][lane] = v;
      bb1[h][lane] = (int)v;
      const u64 m = __ballot(fast_shifts && v <= lim32 && v >= -lim32);
      if (lane == 0) fast_s[h][1] = (unsigned)m == 0xFFFFFFFFu;
    }
  } else {
    // Head fuse, hidden layer: thread j * C + c of the other wavefronts takes
    // head-weight unit j of candidate c.
    const int i = tid - 192, j = (i >= C ? 1 : 0) + (i >= 2 * C ? 1 : 0), c = i - j * C;
    static_assert(3 * kMaxCand <= NT - 192, "one thread per candidate and unit");
    if (i < 3 * C) hid_s[c * 3 + j] = fuse_hidden(p, &st_s[c * 3], &hwc[3 * j], hwc[18 + j]);
  }
  __syncthreads();
  // Head fuse, weight layer, over the last wavefronts (the first ones have a
  // unit more below).
  {
    const int i = NT - 1 - tid, j = (i >= C ? 1 : 0) + (i >= 2 * C ? 1 : 0), c = i - j * C;
    if (i < 3 * C) {
      const int w = fuse_weight(p, &hid_s[c * 3], &hwc[9 + 3 * j], hwc[21 + j]);
      hw_s[c * 3 + j] = w;
      if (ck.head_weights) ck.head_weights[((size_t)b * kMaxCand + c) * 3 + j] = w;
    }
  }
  // Score layers 1 (local half) and 2 of each unit, in place.
  {
    const int sh1 = -16 - (p.concat_out_exp + p.score_w1_exp), so1 = p.h1_out_exp + 16;
    const int sh2 = -16 - (p.h1_out_exp + p.score_w2_exp), so2 = p.h2_out_exp + 16;
    const Rq ra1 = rq_setup(sh1, -(1 << 23), (1 << 23) - 1), rb1 = rq_setup(so1, -128, 127);
    const Rq ra2 = rq_setup(sh2, -(1 << 23), (1 << 23) - 1), rb2 = rq_setup(so2, -128, 127);
    for (int u = wave; u < nu; u += NW) {
      const int h = (u >= ntiles ? 1 : 0) + (u >= 2 * ntiles ? 1 : 0);  // u / ntiles (< 3)
      const int rt = u - h * ntiles;
      int8_t *row = &act[(h * kCandPad + rt * 16 + col) * 32];
      const bool small1 = __builtin_amdgcn_readfirstlane(fast_s[h][1]) != 0;
      const bool small2 = __builtin_amdgcn_readfirstlane(fast_s[h][2]) != 0;
      const bool table1 = small1 && t1.off >= 0, table2 = small2 && t2.off >= 0;
      const long a = *reinterpret_cast<const long *>(row + grp * 8);
      v4i acc[2];
#pragma unroll
      for (int ct = 0; ct < 2; ++ct) {
        const long wb =
            *reinterpret_cast<const long *>(&w1[h][(ct * 16 + col) * 64 + grp * 8]);
        const v4i bias = *reinterpret_cast<const v4i *>(&bb1[h][ct * 16 + 4 * grp]);
        acc[ct] = __builtin_amdgcn_mfma_i32_16x16x32_i8(wb, a, table1 ? bias : v4i{0}, 0, 0, 0);
      }
      unsigned ow[2];
      if (table1) {
        const int vv[8] = {acc[0][0], acc[0][1], acc[0][2], acc[0][3],
                           acc[1][0], acc[1][1], acc[1][2], acc[1][3]};
        sel_gelu_pack<8>(vv, ra1, lut_b, t1, ow);
      } else {
#pragma unroll
        for (int ct = 0; ct < 2; ++ct) {
          unsigned o[4];
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const i64 bias = bbx[h][ct * 16 + 4 * grp + i];
            o[i] = (unsigned)(small1 ? rq(gelu_q16(rq(acc[ct][i] + (int)bias, ra1)), rb1)
                                     : gelu_exact64(acc[ct][i], bias, sh1, so1));
          }
          ow[ct] = pack_lo4(o[0], o[1], o[2], o[3]);
        }
      }
      wave_lds_fence();
      unsigned *dst = reinterpret_cast<unsigned *>(row + 4 * grp);
      dst[0] = ow[0];
      dst[4] = ow[1];
      wave_lds_fence();
      const long a2 = *reinterpret_cast<const long *>(row + grp * 8);
      const long wb2 = *reinterpret_cast<const long *>(&w2[h][col * 32 + grp * 8]);
      const v4i bias2 = *reinterpret_cast<const v4i *>(&bb2[h][4 * grp]);
      const v4i acc2 =
          __builtin_amdgcn_mfma_i32_16x16x32_i8(wb2, a2, table2 ? bias2 : v4i{0}, 0, 0, 0);
      unsigned o2[1];
      if (table2) {
        const int vv[4] = {acc2[0], acc2[1], acc2[2], acc2[3]};
        sel_gelu_pack<4>(vv, ra2, lut, t2, o2);
      } else {
        unsigned o[4];
#pragma unroll
        for (int i = 0; i < 4; ++i)
          o[i] = (unsigned)sel_gelu(acc2[i], bias2[i], small2, ra2, rb2, sh2, so2);
        o2[0] = pack_lo4(o[0], o[1], o[2], o[3]);
      }
      wave_lds_fence();
      dst[0] = o2[0];
    }
  }
  __syncthreads();
  // Logits, the 2-way selector softmax (keep = element 1) and checkpoints.
  {
    const int s3 = p.logits_out_exp - (p.h2_out_exp + p.score_w3_exp);
    const int sq = -16 - p.logits_out_exp;
    for (int i = tid; i < 3 * C; i += NT) {
      const int h = (i >= C ? 1 : 0) + (i >= 2 * C ? 1 : 0), c = i - h * C;
      const v4i hv = *reinterpret_cast<const v4i *>(&act[(h * kCandPad + c) * 32]);
      int qv[2];
#pragma unroll
      for (int lj = 0; lj < 2; ++lj) {
        const int b3 = b3_s[h * 2 + lj];
        int acc = 0;
#pragma unroll
        for (int k = 0; k < 4; ++k) acc = dot4(hv[k], w3[h][lj * 4 + k], acc);
        // |acc| <= 16 * 2^14: the sum fits the int32 requant for |b3| <= 2^29
        const int logit = b3 <= (1 << 29) && b3 >= -(1 << 29)
                              ? requant_i32(acc + b3, s3, -128, 127)
                              : (int)requant_shift((i64)acc + b3, s3, 8);
        qv[lj] = requant_i32(logit, sq, -(1 << 23), (1 << 23) - 1);
      }
      const int mx = qv[0] > qv[1] ? qv[0] : qv[1];
      const unsigned e0 = softmax_exp(qv[0] - mx), e1 = softmax_exp(qv[1] - mx);
      const unsigned ratio = softmax_ratio(e1, softmax_recip24(e0 + e1));
      const int hsv = (int)(ratio > 65536u ? 65536u : ratio);
      hs_s[h * kMaxCand + c] = hsv;
      if (ck.head_scores) ck.head_scores[((size_t)b * 3 + h) * kMaxCand + c] = hsv;
      if (ck.h2)
        *reinterpret_cast<v4i *>(ck.h2 + (((size_t)b * 3 + h) * kMaxCand + c) * 16) = hv;
    }
  }
  __syncthreads();
  // Head fuse, mean: thread c < C; keep list and state.
  int fc = 0;
  bool warn = false;
  if (tid < C) {
    fc = fuse_mean(&hs_s[tid], &hw_s[tid * 3], &warn);
    fused_out[(size_t)b * kMaxCand + tid] = fc;
  }
  i64 den = 0;
  int warn_bits = 0;
  const int kept = keep_list<NT>(C, pkg, fc, warn, false, kept_index + (size_t)b * kMaxCand, st,
                                 &den, &warn_bits);
  if (tid == 0 && img_warn && warn_bits) img_warn[b] |= warn_bits;
  if (kept < 0 || C - kept == 0) return;  // uniform; no package row
  // (the step tables' LDS is free: their last reader was score layer 2)
  static_assert(36 * 208 <= 2 * kGeluLutMaxWords, "package sums fit the tables' LDS");
  package_row<NT, kXsRow, 36, 4>(xs, C, pkg, kept, fc, den, pkg_rows + (size_t)b * 192, wgt,
                                 reinterpret_cast<int *>(lut));
}

// finalize_tokens from given fused scores (hv_selector_finalize): the keep
// list and state of one image per workgroup, one thread per candidate.
// Given scores must be Q0.16 values in [0, 65536] (selector._q016): an
// image holding any other value is rejected like a bad token count.
__global__ __launch_bounds__(256) void k_selector_keep(const int32_t *offsets,
                                                       const uint8_t *pkg_in, int batch,
                                                       const int32_t *fused, int32_t *kept_index,
                                                       int32_t *state) {
  const int b = xcd_image(batch);
  if (b < 0) return;
  const int c = threadIdx.x;
  const int row0 = offsets[b], C = offsets[b + 1] - row0 - 1;
  const int pkg = pkg_in ? (pkg_in[b] ? 1 : 0) : 0;
  int32_t *st = state + (size_t)b * 5;
  if (!image_ok(row0, C, pkg)) {
    if (c == 0) state_invalid(st);
    return;
  }
  const int fc = c < C ? fused[(size_t)b * kMaxCand + c] : 0;
  const bool bad = c < C && (unsigned)fc > 65536u;
  keep_list<256>(C, pkg, fc, false, bad, kept_index + (size_t)b * kMaxCand, st);
}

// finalize_tokens' stream compaction of one image (XCD-major): the image's
// output offset (the token counts of the images before it; an image with a
// bad count contributes 0), then CLS, the kept rows and there the package row,
// computed from the given fused scores.
__global__ __launch_bounds__(256) void k_selector_compact(
    const int8_t *tokens, const int32_t *offsets, const uint8_t *pkg_in, int batch,
    const int32_t *fused, const int32_t *kept_index, const int32_t *state,
    int8_t *out, int32_t *out_offsets, uint8_t *pkg_out) {
  __shared__ int wgt[kMaxCand];
  __shared__ int part_sum[21 * 192];
  __shared__ int src_k[kMaxCand + 1];
  __shared__ int red[4];
  const int b = xcd_image(batch);
  if (b < 0) return;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int32_t *st = state + (size_t)b * 5;
  const int count = st[0], exists = st[1], kept = st[2];
  int sum = 0;
  for (int i = tid; i < b; i += 256) sum += max(state[(size_t)i * 5], 0);
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) sum += __shfl_xor(sum, off);
  if (lane == 0) red[wave] = sum;
  __syncthreads();
  const int out0 = red[0] + red[1] + red[2] + red[3];
  if (tid == 0) {
    out_offsets[b] = out0;
    if (b == batch - 1) out_offsets[batch] = out0 + max(count, 0);
    pkg_out[b] = (uint8_t)(count > 0 ? exists : 0);
  }
  if (count <= 0) return;  // uniform
  const int row0 = offsets[b], C = offsets[b + 1] - row0 - 1;
  const int pkg = pkg_in ? (pkg_in[b] ? 1 : 0) : 0;
  // Source row of output row r is row0 + 1 + src_k[r]: -1 for the CLS row,
  // then the kept candidates.
  const int *ki = kept_index + (size_t)b * kMaxCand;
  if (tid <= kMaxCand) src_k[tid] = tid == 0 ? -1 : ki[tid - 1];
  __syncthreads();
  // CLS and kept rows, 16 bytes per item; four items per thread in flight
  // (items past the end repeat the last one, so no copy is predicated).
  const int n_items = (1 + kept) * 12;
  for (int base = tid; base < n_items; base += 1024) {
    v4i v[4];
    int dst[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int i = min(base + j * 256, n_items - 1), r = i / 12, chunk = i - r * 12;
      v[j] = reinterpret_cast<const v4i *>(tokens + (size_t)(row0 + 1 + src_k[r]) * 192)[chunk];
      dst[j] = (out0 + r) * 12 + chunk;
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) reinterpret_cast<v4i *>(out)[dst[j]] = v[j];
  }
  if (!exists) return;
  int8_t *prow = out + (size_t)(out0 + 1 + kept) * 192;
  // the partitioned candidates' score sum (finalize's scores are checked
  // to lie in [0, 65536], so a wavefront's sum fits 32 bits)
  const int fv = tid < C ? fused[(size_t)b * kMaxCand + tid] : 0;
  const bool part = tid < C && ((tid < C - pkg && fv < 32768) || (pkg && tid == C - 1));
  int d = part ? fv : 0;
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) d += __shfl_xor(d, off);
  if (lane == 0) red[wave] = d;
  __syncthreads();
  const i64 den = (i64)red[0] + red[1] + red[2] + red[3];
  package_row<256, 192, 21, 1>(tokens + (size_t)(row0 + 1) * 192, C, pkg, kept, fv, den, prow, wgt,
                            part_sum);
}

int launch_selector(const SelectorArgs &a, hipStream_t s) {
  if (a.batch <= 0) return HV_OK;
  int rc = HV_OK;
  const dim3 grid((a.batch + 7) / 8 * 8);
  if (a.p) {
    if (!a.pkg_rows)
      return fail(HV_EVALUE, HV_ERR_ADDRESS, "selector: missing workspace");
    const hv_selector_dev p = *a.p;
    auto in = [](int v) { return v >= -30 && v <= 30; };
    const int fast = in(-16 - (p.in_exp + p.local_w_exp)) && in(p.local_out_exp + 16) &&
                     in(-16 - (p.concat_out_exp + p.score_w1_exp)) && in(p.h1_out_exp + 16) &&
                     in(-16 - (p.h1_out_exp + p.score_w2_exp)) && in(p.h2_out_exp + 16);
    auto table = [](int so) {
      if (so < kGeluLutSoMin || so > kGeluLutSoMax) return SelLut{-1, 0, 0, 0, 0};
      const GeluLutInfo &t = kGeluLutInfo[so - kGeluLutSoMin];
      return SelLut{t.off, t.words, t.qlo, t.qhi, -4 * (t.qlo >> kGeluCoarseShift)};
    };
    hv_launch(k_selector_image, grid, dim3(kImgThreads), 0, s, p, a.tokens, a.offsets, a.batch,
              a.pkg_in, fast, a.ck, table(p.local_out_exp + 16), table(p.h1_out_exp + 16),
              table(p.h2_out_exp + 16), a.fused, a.kept_index, a.state, a.pkg_rows, a.img_warn);
    if ((rc = check_hip(hipGetLastError(), "k_selector_image launch"))) return rc;
    const SelectorRows rows{a.tokens, a.offsets, a.kept_index, a.state, a.pkg_rows,
                            a.out_tokens, a.out_offsets, a.pkg_out, a.token_counts,
                            a.batch, a.stage};
    if (!a.ln) return launch_selector_rows(rows, nullptr, s);
    const ProfScope ps(HV_PROF_LAYERNORM, s);  // the launch it stands in for
    return launch_selector_rows(rows, a.ln, s);
  }
  hv_launch(k_selector_keep, grid, dim3(256), 0, s, a.offsets, a.pkg_in, a.batch, a.fused,
            a.kept_index, a.state);
  if ((rc = check_hip(hipGetLastError(), "k_selector_keep launch"))) return rc;
  hv_launch(k_selector_compact, grid, dim3(256), 0, s, a.tokens, a.offsets, a.pkg_in, a.batch,
            a.fused, a.kept_index, a.state, a.out_tokens, a.out_offsets, a.pkg_out);
  return check_hip(hipGetLastError(), "k_selector_compact launch");
}

}  // namespace hv
