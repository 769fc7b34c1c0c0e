// Dense projections for several token rows on the bf16 matrix cores: the fused QKV
// nn.Linear with its bias, YaRN RoPE and the KV-cache append (2 to 64 tokens); the
// attention output nn.Linear with its bias and the residual add (2 to 48); the
// unembedding (2 to 8; model/attention.py:204,254-256; model/transformer.py:
// 95-100).
//
// y[m][n] = sum_k t[m][k] W[n][k], bf16 operands, fp32 accumulation, one bf16
// rounding, then the epilogue's own bf16 ops, as dense_gemv.hip (one token)
// does.  Bound by the bytes of W: a vector dot product per (row, token) is
// issue-bound from two tokens on, while the matrix cores multiply 16 W rows by
// 16 tokens for the price of the loads: the 201088 x 2880 unembedding at 2, 5
// and 8 tokens 399, 750 and 1122 us on the vector ALUs, 198-206 here (5.6 to 5.8
// TB/s); QKV with its norm at 2 and 8 tokens 19.1 and 54.1 us, 12.4-12.8 here; the
// output projection 10.6 and 34.1, 7.1 here (rows_wide_kernel).  (One token stays on
// the vector ALUs: unembedding 188 us against 205 here, QKV 9.1, output 6.5.)
//
// A workgroup takes 16 or 32 rows of W at a time; its sixteen waves split K
// into contiguous runs of 32-wide steps (5 or 6 each at K = 2880), so that
// every byte of the rows is in flight at once, and add their partial tiles
// through LDS in fp64 (deterministic, one rounding).  v_mfma_f32_16x16x32_bf16:
// lane (r, g) = (l % 16, l / 16) gives A row r (a W row) and B column r (a token),
// k = 8 g .. 8 g + 7 of the step for both; D element i of the lane is W row
// 4 g + i, token r.  Neither operand goes through LDS: a wave's K run of W and of
// the tokens is used by that wave alone.
// The tokens stay in registers (kSteps x 16 bytes a lane); for the unembedding a
// workgroup walks a contiguous range of row groups with two groups' W in
// flight.  The RMSNorm is the standalone kernel's arithmetic: the sum of squares
// in fp64 from the lanes' own chunks.
#include <stdint.h>

#include "moe_common.h"

namespace rows {

using moe::as_bf16x8;
using moe::bf2f;
using moe::f2bf;
using moe::f32x4;
using moe::kWave;
using moe::u32x4;

constexpr int kWaves = 16;
constexpr int kThreads = kWaves * kWave;
constexpr int kMaxGroups = 64;  // row groups of one workgroup's range (its outputs wait in LDS)

// gpt-oss attention shapes (the QKV epilogue)
constexpr int kD = 64, kHq = 64, kHkv = 8, kPage = 16;
constexpr int kHeadBlock = kPage * kD * 2;
constexpr int kPageBytes = 2 * kHkv * kHeadBlock;

enum Epi { kPlain = 0, kBiasResidual = 1, kQkv = 2 };

struct Args {
  const uint16_t* x;
  int M, K;
  const uint16_t* W;
  int N;
  uint16_t* out;
  const uint16_t* norm_w;
  float eps;
  const uint16_t* bias;
  const uint16_t* res;
  // QKV epilogue
  const int* positions;
  const int* slots;
  const float* inv_freq;
  float conc;
  uint8_t* cache;
  int num_pages;
  uint16_t* q_out;
};

// Row groups of N rows of W.  In 64 bits: N may be as large as an int.
__host__ __device__ constexpr int64_t row_groups(int N) { return ((int64_t)N + 15) / 16; }
static_assert(row_groups(INT32_MAX) == (int64_t)1 << 27 && row_groups(16) == 1 && row_groups(17) == 2);

// The W row of A row `r` of row group `group`.  QKV: eight rope pairs, a
// pair's two dimensions in one lane's result: A rows 4 g + i hold dimensions
// d0 + 2 g + i % 2 + 32 (i / 2) of a head.
template <int EPI>
__device__ __forceinline__ int w_row(int group, int r) {
  if constexpr (EPI == kQkv)
    return (group >> 2) * kD + (group & 3) * 8 + 2 * (r >> 2) + (r & 1) + 32 * ((r >> 1) & 1);
  else
    return group * 16 + r;
}

// The unembedding and QKV.  kSteps: 32-wide steps of K a wave holds (at most);
// kNorm: RMSNorm the tokens first.  Row groups of a workgroup: a range walked two
// at a time (kPlain) or two (kQkv: 160 workgroups, all resident at once; with one
// group each the 320 ran in two rounds).
template <int kSteps, int EPI, bool kNorm>
__global__ __launch_bounds__(kThreads) void rows_kernel(Args a) {
#pragma clang fp contract(off)
  constexpr int kRg = EPI == kQkv ? 2 : 1;  // row groups of a workgroup (kPlain: a range)
  // partial tiles: of the two groups, or (kPlain) of the current and the last
  __shared__ __align__(16) double part[kWaves][2][4][kWave];
  __shared__ double ssq[kWaves][16];
  static_assert(kSteps <= 8, "four chunks of the norm weight a step, in 32 lanes");
  extern __shared__ __align__(16) uint16_t outs[];  // kPlain: [M][16 row groups of the range]
  const int t = threadIdx.x, lane = t & 63;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int r = lane & 15, g = lane >> 4;
  const int M = a.M, K = a.K, N = a.N;
  const int steps = (K + 31) / 32;
  const int s0 = steps * wave / kWaves;
  const int cnt = steps * (wave + 1) / kWaves - s0;
  // Lane's k of the wave's step s; steps past the wave's run and chunks past K
  // read clamped addresses and count as zeros (in both operands).
  auto k_of = [&](int s) { return (s0 + s) * 32 + 8 * g; };
  auto valid = [&](int s) { return s < cnt && k_of(s) < K; };
  auto load = [&](const uint16_t* row, int s) {
    return *(const u32x4*)(row + min(k_of(s), K - 8));
  };
  const u32x4 zero = u32x4{0u, 0u, 0u, 0u};
  // this workgroup's row groups
  int grp0 = blockIdx.x * kRg, grp1 = grp0 + kRg;
  if constexpr (EPI == kPlain) {
    const int64_t groups = row_groups(N);
    grp0 = (int)(groups * blockIdx.x / gridDim.x);
    grp1 = (int)(groups * (blockIdx.x + 1) / gridDim.x);
  }

  // Issue order: the tokens, the epilogue's operands, then W (loads complete
  // in issue order, and the norm and RoPE factors are taken while W streams).
  u32x4 xf[kSteps];
  {
    const uint16_t* row = a.x + (size_t)min(r, M - 1) * K;
#pragma unroll
    for (int s = 0; s < kSteps; ++s) xf[s] = load(row, s);
  }
  // The epilogue task of waves 0..3, token r: element `wave` of a lane's four
  // (W row 4 g + wave), or for QKV of row group wave / 2 the rope pair wave % 2 of
  // the lane's two (elements j and j + 2).
  const bool task = wave < 4 && r < M;
  const int tm = min(r, M - 1);
  const int tgrp = grp0 + (EPI == kQkv ? (wave >> 1) & 1 : 0);
  const int ei = EPI == kQkv ? wave & 1 : wave & 3;
  uint16_t eb0 = 0, eb1 = 0;
  float ifq = 0.f, cs = 0.f, sn = 0.f;
  int eslot = -1, epos = 0, erow = 0;
  if constexpr (EPI == kQkv) {
    erow = min(w_row<EPI>(tgrp, 4 * g + ei), N - 1);
    eb0 = a.bias[erow];
    eb1 = a.bias[erow + 32];
    eslot = a.slots[tm];
    epos = a.positions[tm];
    ifq = a.inv_freq[erow % kD];
  }
  // The norm weight of the wave's K run: four chunks a step, which lane 4 s + g
  // loads for all (16 lanes need each) and passes on through the wave's part of
  // the partial tiles.  Held in every lane they spilled at eight steps (QKV at 2
  // and 16 tokens, K = 4096: 23.0 and 24.9 us, 16.2 and 18.5 so; K = 3080 21.8 and
  // 24.0, 14.4 and 16.2).
  u32x4* const nws = (u32x4*)part[wave][0][0];
  u32x4 nwl = u32x4{0u, 0u, 0u, 0u};
  if constexpr (kNorm)  // (a caller's slice at any element)
    nwl = *(const moe::u32x4_any*)(a.norm_w + min(s0 * 32 + 8 * (lane & 31), K - 8));
  __builtin_amdgcn_sched_barrier(0);
  u32x4 wa[kSteps], wb[kSteps];
  auto load_w = [&](auto& dst, int group) {
    const uint16_t* row = a.W + (size_t)min(w_row<EPI>(group, r), N - 1) * K;
#pragma unroll
    for (int s = 0; s < kSteps; ++s) dst[s] = load(row, s);
  };
  load_w(wa, min(grp0, grp1 - 1));
  // (behind the norm, whose weights hold registers until then)
  if constexpr (!kNorm) load_w(wb, min(grp0 + 1, grp1 - 1));
  __builtin_amdgcn_sched_barrier(0);

  if constexpr (EPI == kQkv) {  // the RoPE factors while W streams
    if (task && erow / kD < kHq + kHkv) {
      double sd, cd;
      moe::sincos_f64((double)((float)epos * ifq), sd, cd);
      cs = bf2f(moe::f64_to_bf16_via_f32(cd)) * a.conc;
      sn = bf2f(moe::f64_to_bf16_via_f32(sd)) * a.conc;
    }
  }
  if constexpr (kNorm) {
    // r = fp32(1 / sqrt(sum of squares / K + eps)), t = bf16(fp32(x r) w)
    double ss = 0.0;
#pragma unroll
    for (int s = 0; s < kSteps; ++s) {
      const u32x4 v = valid(s) ? xf[s] : zero;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const double lo = (double)__uint_as_float(v[j] << 16);
        const double hi = (double)__uint_as_float(v[j] & 0xFFFF0000u);
        ss += lo * lo + hi * hi;
      }
    }
    ss += __shfl_xor(ss, 16, kWave);
    ss += __shfl_xor(ss, 32, kWave);
    if (g == 0) ssq[wave][r] = ss;
    if (lane < 32) nws[lane] = nwl;
    moe::lds_barrier();
    double tot = 0.0;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) tot += ssq[w][r];
    const float rn = (float)(1.0 / sqrt(tot / (double)K + (double)a.eps));
#pragma unroll
    for (int s = 0; s < kSteps; ++s) {
      const u32x4 nw = nws[4 * s + g];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const uint32_t v = xf[s][j], w = nw[j];
        const uint32_t lo = f2bf(__fmul_rn(__fmul_rn(__uint_as_float(v << 16), rn),
                                           __uint_as_float(w << 16)));
        const uint32_t hi = f2bf(__fmul_rn(__fmul_rn(__uint_as_float(v & 0xFFFF0000u), rn),
                                           __uint_as_float(w & 0xFFFF0000u)));
        xf[s][j] = lo | (hi << 16);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
    load_w(wb, min(grp0 + 1, grp1 - 1));
    __builtin_amdgcn_sched_barrier(0);
  }
  auto zero_tail = [&](u32x4 (&v)[kSteps]) {
#pragma unroll
    for (int s = 0; s < kSteps; ++s) v[s] = valid(s) ? v[s] : zero;
  };
  // One wave's partial tile of the loaded W rows, into LDS.  It is summed in
  // fp64 after every two MFMAs (64 products): chained in fp32 over the wave's
  // steps, 110 to 145 of a million results at K = 4096 rounded to the other bf16
  // neighbour of a near tie, against 90 to 97 for the vector ALUs' short chains
  // and 55 to 94 this way.
  auto products = [&](const u32x4 (&w)[kSteps], int tile) {
    double sum[4] = {};
#pragma unroll
    for (int s = 0; s < kSteps; s += 2) {
      f32x4 acc = f32x4{0.f, 0.f, 0.f, 0.f};
      acc = moe::mfma16x16x32(as_bf16x8(w[s]), as_bf16x8(xf[s]), acc);
      acc = moe::mfma16x16x32(as_bf16x8(w[s + 1]), as_bf16x8(xf[s + 1]), acc);
#pragma unroll
      for (int i = 0; i < 4; ++i) sum[i] += (double)acc[i];
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) part[wave][tile][i][lane] = sum[i];
  };
  // element i of this lane's four of a tile: the waves' partials added in fp64
  // and rounded once
  auto total = [&](int tile, int i) {
    double v = part[0][tile][i][lane];
#pragma unroll
    for (int w = 1; w < kWaves; ++w) v += part[w][tile][i][lane];
    return (float)v;
  };

  if constexpr (EPI == kPlain) {
    zero_tail(xf);
    const int width = 16 * (grp1 - grp0);
    // a row group: products, then the group after next takes the W registers'
    // place in flight, and waves 0..3 sum one element of a lane's four each
    // into the LDS outputs (buf alternates: a buffer is written again only
    // after the next round's barrier, which follows its reads)
    auto round = [&](u32x4 (&w)[kSteps], int group, int buf) {
      zero_tail(w);
      products(w, buf);
      __builtin_amdgcn_sched_barrier(0);
      load_w(w, min(group + 2, grp1 - 1));
      __builtin_amdgcn_sched_barrier(0);
      moe::lds_barrier();
      if (task) outs[r * width + 16 * (group - grp0) + 4 * g + ei] = f2bf(total(buf, ei));
    };
    int group = grp0;
    for (; group + 1 < grp1; group += 2) {
      round(wa, group, 0);
      round(wb, group + 1, 1);
    }
    if (group < grp1) round(wa, group, 0);
    moe::lds_barrier();
    // the range's outputs: 16 (grp1 - grp0) columns of each token
    const int n0 = 16 * grp0, nc = min(width, N - n0);
    for (int i = t; i < M * width; i += kThreads) {
      const int m = i / width, c = i - m * width;
      if (c < nc) a.out[(size_t)m * N + n0 + c] = outs[i];
    }
  } else {
    zero_tail(xf);
    zero_tail(wa);
    products(wa, 0);
    zero_tail(wb);
    products(wb, 1);
    moe::lds_barrier();
    if (!task) return;
    // bias (its own bf16 rounding), then YaRN RoPE of q / k heads exactly as
    // the standalone append kernel does, then q out or the cache slot
    const int head = erow / kD, d = erow % kD;  // dimensions d and d + 32
    float lo = bf2f(f2bf(bf2f(f2bf(total(tgrp - grp0, ei))) + bf2f(eb0)));
    float hi = bf2f(f2bf(bf2f(f2bf(total(tgrp - grp0, ei + 2))) + bf2f(eb1)));
    if (head < kHq + kHkv) {
      const float nl = lo * cs - hi * sn;
      const float nh = lo * sn + hi * cs;
      lo = nl;
      hi = nh;
    }
    uint16_t* dst = nullptr;
    if (head < kHq) {
      dst = a.q_out + ((size_t)tm * kHq + head) * kD;
    } else if (eslot >= 0 && eslot < a.num_pages * kPage) {  // other slots are not written
      const int kv = head < kHq + kHkv ? 0 : 1;
      const int hk = head - kHq - kv * kHkv;
      dst = (uint16_t*)(a.cache + (size_t)(eslot / kPage) * kPageBytes +
                        (size_t)(kv * kHkv + hk) * kHeadBlock + (eslot % kPage) * (kD * 2));
    }
    if (dst) {
      dst[d] = f2bf(lo);
      dst[d + 32] = f2bf(hi);
    }
  }
}

// ---------------------------------------------------------------------------
// The two layer projections for 17 to 64 tokens (output: 2 to 48), NT tiles of 16.
// Bound by the tokens' way from L2: every workgroup reads all of them (48 x 4096
// bf16 = 393 KB against 131 KB of W for the output projection), so they stream
// through registers beside W instead of waiting in them.  Eight waves split K; a
// wave has its whole run of W (16 rows, QKV 32) in flight at once, the tokens two
// chunks of kChunk steps ahead.  Loads take 64 bytes of a row with four
// neighbouring lanes and reach the operands' order through LDS: loaded in operand
// order, where neighbouring lanes hold different rows, a load moved about 16
// bytes a clock (QKV with its norm 15.1, 17.0, 21.3 and 24.2 us at 17, 32, 48 and
// 64 tokens, output 10.9, 13.5, 17.5 and 21.4; so 13.2, 13.9, 16.1 and 17.8, output
// 8.8, 9.5, 12.0 and 15.1; at 8 and 16 tokens 7.1 and 7.3, 8.9 and 10.3 in
// rows_kernel's form).  Whole 128-byte lines per eight lanes were no better (13.6,
// 13.8, 15.6 and 20.5; output 9.3, 9.7, 11.9 and 14.7).  The partial tiles, fp32
// chains of at most 16 steps, are added over the waves in fp64 through LDS.  One
// workgroup per CU: 180 (output) and 160 (QKV), one round.  The RMSNorm is its own
// launch here (fused it would read the tokens twice).
constexpr int kWideWaves = 8;
constexpr int kWideThreads = kWideWaves * kWave;

template <int NT, int EPI>
__global__ __launch_bounds__(kWideThreads) void rows_wide_kernel(Args a) {
#pragma clang fp contract(off)
  constexpr int kRg = EPI == kQkv ? 2 : 1;         // row groups of the workgroup
  constexpr int kSteps = EPI == kQkv ? 12 : 16;    // 32-wide steps of K a wave holds
  constexpr int kChunk = EPI == kQkv ? 2 : 4;      // steps of the tokens loaded at a time
  constexpr int kFrags = kRg + NT;                 // operand tiles of a step
  // a wave's own: the operand tiles of two steps, then its partial result tiles
  __shared__ __align__(16) u32x4 lds[kWideWaves][2 * kFrags][kWave];
  static_assert(2 * kFrags >= kRg * NT, "the partial tiles take the operands' place");
  const int t = threadIdx.x, lane = t & 63;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int r = lane & 15, g = lane >> 4;    // in the matrix operands and results
  const int lr = lane >> 2, lc = lane & 3;   // in the loads: row, 16-byte chunk
  const int M = a.M, K = a.K, N = a.N;
  const int steps = (K + 31) / 32;
  const int s0 = steps * wave / kWideWaves;
  const int cnt = steps * (wave + 1) / kWideWaves - s0;
  auto k_of = [&](int s) { return (s0 + s) * 32 + 8 * lc; };
  auto valid = [&](int s) { return s < cnt && k_of(s) < K; };
  auto load = [&](const uint16_t* row, int s) {
    return *(const u32x4*)(row + min(k_of(s), K - 8));
  };
  const u32x4 zero = u32x4{0u, 0u, 0u, 0u};
  // one tile: sums in fp64 after every two products, as rows_kernel's
  constexpr bool kF64 = NT == 1;
  static_assert(!kF64 || kRg == 1, "one result tile");
  const int grp0 = blockIdx.x * kRg;

  // The epilogue task of a wave: QKV: tile (wave % 2, wave / 2), both rope pairs
  // of each lane; output: elements 2 (wave / 4) and + 1 of tile wave % 4.
  const int trg = EPI == kQkv ? wave & 1 : 0;
  const int tnt = EPI == kQkv ? wave >> 1 : wave & 3;
  const int e0 = EPI == kQkv ? 0 : 2 * (wave >> 2);
  const int tok = 16 * tnt + r;
  const bool task = tnt < NT && tok < M;
  const int tm = min(tok, M - 1);
  const int erow = w_row<EPI>(grp0 + trg, 4 * g + e0);  // element 0; 1 is the next row
  // the epilogue's operands first: the RoPE factors are taken while W streams
  uint16_t eb[4], er[2];
  int eslot = -1, epos = 0;
  float ifq[2] = {0.f, 0.f};
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int row = min(erow + j, N - 1);
    eb[j] = a.bias[row];
    if constexpr (EPI == kQkv) {
      eb[2 + j] = a.bias[row + 32];
      ifq[j] = a.inv_freq[row % kD];
    } else {
      er[j] = a.res[(size_t)tm * N + row];
    }
  }
  if constexpr (EPI == kQkv) {
    eslot = a.slots[tm];
    epos = a.positions[tm];
  }
  __builtin_amdgcn_sched_barrier(0);

  const uint16_t* xrow[NT];
#pragma unroll
  for (int i = 0; i < NT; ++i) xrow[i] = a.x + (size_t)min(16 * i + lr, M - 1) * K;
  u32x4 xa[kChunk][NT], xb[kChunk][NT], w[kSteps][kRg];
  auto load_x = [&](auto& dst, int s) {
#pragma unroll
    for (int c = 0; c < kChunk; ++c)
#pragma unroll
      for (int i = 0; i < NT; ++i) dst[c][i] = load(xrow[i], s + c);
  };
  load_x(xa, 0);
  {
    const uint16_t* row[kRg];
#pragma unroll
    for (int q = 0; q < kRg; ++q)
      row[q] = a.W + (size_t)min(w_row<EPI>(grp0 + q, lr), N - 1) * K;
#pragma unroll
    for (int s = 0; s < kSteps; ++s) {
      if (s == kChunk) load_x(xb, kChunk);
#pragma unroll
      for (int q = 0; q < kRg; ++q) w[s][q] = load(row[q], s);
    }
  }
  __builtin_amdgcn_sched_barrier(0);

  float cs[2] = {0.f, 0.f}, sn[2] = {0.f, 0.f};
  if constexpr (EPI == kQkv) {
    if (task && erow / kD < kHq + kHkv) {
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        double sd, cd;
        moe::sincos_f64((double)((float)epos * ifq[j]), sd, cd);
        cs[j] = bf2f(moe::f64_to_bf16_via_f32(cd)) * a.conc;
        sn[j] = bf2f(moe::f64_to_bf16_via_f32(sd)) * a.conc;
      }
    }
  }

  f32x4 acc[kRg][NT];
#pragma unroll
  for (int q = 0; q < kRg; ++q)
#pragma unroll
    for (int i = 0; i < NT; ++i) acc[q][i] = f32x4{0.f, 0.f, 0.f, 0.f};
  // A step's tiles go through LDS from load order (lane = row, chunk) to operand
  // order (lane = chunk, row), the chunks of a row swizzled so that the reads of
  // 16 rows spread over the banks.  Wave-private: no barrier, program order only.
  auto put = [&](const u32x4 (&x)[NT], int s) {
    const bool in = valid(s);  // else zeros, in both operands
    u32x4(*buf)[kWave] = lds[wave] + (s & 1) * kFrags;
    const int at = lr * 4 + (lc ^ (lr >> 2));
#pragma unroll
    for (int q = 0; q < kRg; ++q) buf[q][at] = in ? w[s][q] : zero;
#pragma unroll
    for (int i = 0; i < NT; ++i) buf[kRg + i][at] = in ? x[i] : zero;
  };
  u32x4 op[kFrags];
  auto get = [&](int s) {
    u32x4(*buf)[kWave] = lds[wave] + (s & 1) * kFrags;
    const int at = r * 4 + (g ^ (r >> 2));
#pragma unroll
    for (int f = 0; f < kFrags; ++f) op[f] = buf[f][at];
  };
  auto products = [&]() {
#pragma unroll
    for (int i = 0; i < NT; ++i)
#pragma unroll
      for (int q = 0; q < kRg; ++q)
        acc[q][i] = moe::mfma16x16x32(as_bf16x8(op[q]), as_bf16x8(op[kRg + i]), acc[q][i]);
  };
  auto order = [] {  // this wave's LDS accesses stay in program order
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
  };
  static_assert(kSteps % kChunk == 0 && kSteps > kChunk && kChunk > 1,
                "two token buffers, filled in turn (the first refill follows a put)");
  double sum64[4] = {};
  put(xa[0], 0);
  order();
#pragma unroll
  for (int s = 0; s < kSteps; ++s) {
    get(s);
    order();
    const int n = s + 1, c = n / kChunk;  // the next step and its chunk
    if (n < kSteps) {
      put(c & 1 ? xb[n % kChunk] : xa[n % kChunk], n);
      if (n % kChunk == kChunk - 1 && (c + 2) * kChunk < kSteps)  // its last tiles are taken
        load_x(c & 1 ? xb : xa, (c + 2) * kChunk);
      order();
    }
    products();
    if constexpr (kF64)
      if (s & 1) {
#pragma unroll
        for (int i = 0; i < 4; ++i) sum64[i] += (double)acc[0][0][i];
        acc[0][0] = f32x4{0.f, 0.f, 0.f, 0.f};
      }
  }
  f32x4(*part)[kWave] = (f32x4(*)[kWave])lds[wave];
  if constexpr (kF64) {  // [element][lane]
#pragma unroll
    for (int i = 0; i < 4; ++i) ((double*)part)[i * kWave + lane] = sum64[i];
  } else {
#pragma unroll
    for (int q = 0; q < kRg; ++q)
#pragma unroll
      for (int i = 0; i < NT; ++i) part[q * NT + i][lane] = acc[q][i];
  }
  moe::lds_barrier();
  if (!task) return;
  // the waves' partials added in fp64 and rounded once
  constexpr int kEl = EPI == kQkv ? 4 : 2;
  double sum[kEl] = {};
#pragma unroll
  for (int v = 0; v < kWideWaves; ++v) {
    const float* p = (const float*)&lds[v][trg * NT + tnt][lane] + e0;
#pragma unroll
    for (int i = 0; i < kEl; ++i) {
      if constexpr (kF64) sum[i] += ((const double*)lds[v])[(e0 + i) * kWave + lane];
      else sum[i] += (double)p[i];
    }
  }
  if constexpr (EPI == kBiasResidual) {
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const float tb = bf2f(f2bf(bf2f(f2bf((float)sum[j])) + bf2f(eb[j])));
      if (erow + j < N) a.out[(size_t)tok * N + erow + j] = f2bf(bf2f(er[j]) + tb);
    }
  } else {
    // as rows_kernel's QKV epilogue, for the lane's two rope pairs
    const int head = erow / kD, d = erow % kD;
    uint16_t* dst = nullptr;
    if (head < kHq) {
      dst = a.q_out + ((size_t)tok * kHq + head) * kD;
    } else if (eslot >= 0 && eslot < a.num_pages * kPage) {  // other slots are not written
      const int kv = head < kHq + kHkv ? 0 : 1;
      const int hk = head - kHq - kv * kHkv;
      dst = (uint16_t*)(a.cache + (size_t)(eslot / kPage) * kPageBytes +
                        (size_t)(kv * kHkv + hk) * kHeadBlock + (eslot % kPage) * (kD * 2));
    }
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      float lo = bf2f(f2bf(bf2f(f2bf((float)sum[j])) + bf2f(eb[j])));
      float hi = bf2f(f2bf(bf2f(f2bf((float)sum[2 + j])) + bf2f(eb[2 + j])));
      if (head < kHq + kHkv) {
        const float nl = lo * cs[j] - hi * sn[j];
        const float nh = lo * sn[j] + hi * cs[j];
        lo = nl;
        hi = nh;
      }
      if (dst) {
        dst[d + j] = f2bf(lo);
        dst[d + j + 32] = f2bf(hi);
      }
    }
  }
}

template <int EPI>
int launch_wide(const Args& a, unsigned grid, hipStream_t s) {
  auto go = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3(grid), dim3(kWideThreads), 0, s, a);
    return hipGetLastError() == hipSuccess ? 0 : -6;
  };
  if constexpr (EPI == kBiasResidual)
    if (a.M <= 16) return go(rows_wide_kernel<1, EPI>);
  if (a.M <= 32) return go(rows_wide_kernel<2, EPI>);
  if (a.M <= 48) return go(rows_wide_kernel<3, EPI>);
  if constexpr (EPI == kQkv)
    if (a.M <= 64) return go(rows_wide_kernel<4, EPI>);
  return -6;
}

template <int EPI, bool kNorm>
int launch(const Args& a, dim3 grid, size_t lds, hipStream_t s) {
  const bool small = a.K <= 32 * 6 * kWaves;  // 6 steps a wave; 8 cover K <= 4096
  auto go = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, grid, dim3(kThreads), lds, s, a);
    return hipGetLastError() == hipSuccess ? 0 : -6;
  };
  return small ? go(rows_kernel<6, EPI, kNorm>) : go(rows_kernel<8, EPI, kNorm>);
}

}  // namespace rows

extern "C" {

// out = bf16(t W^T) for M <= 16 rows, t = x or RMSNorm(x)
int attn_launch_rows_plain(const void* x, int M, int K, const void* W, int N, const void* norm_w,
                           float eps, void* out, hipStream_t s) {
  using namespace rows;
  Args a{};
  a.x = (const uint16_t*)x;
  a.M = M;
  a.K = K;
  a.W = (const uint16_t*)W;
  a.N = N;
  a.norm_w = (const uint16_t*)norm_w;
  a.eps = eps;
  a.out = (uint16_t*)out;
  const int64_t groups = row_groups(N);
  // one workgroup per CU, more where a range would be longer than kMaxGroups
  const int64_t fill = groups < 256 ? groups : 256;
  const int64_t need = (groups + kMaxGroups - 1) / kMaxGroups;
  const dim3 grid((unsigned)(need > fill ? need : fill));
  const int64_t range = (groups + grid.x - 1) / grid.x;
  const size_t lds = (size_t)M * range * 16 * 2;
  return norm_w ? launch<kPlain, true>(a, grid, lds, s) : launch<kPlain, false>(a, grid, lds, s);
}

// out = bf16(res + bf16(bf16(x W^T) + bias)), M <= 48
int attn_launch_rows_bias_residual(const void* x, int M, int K, const void* W, int N,
                                   const void* bias, const void* res, void* out, hipStream_t s) {
  using namespace rows;
  Args a{};
  a.x = (const uint16_t*)x;
  a.M = M;
  a.K = K;
  a.W = (const uint16_t*)W;
  a.N = N;
  a.out = (uint16_t*)out;
  a.bias = (const uint16_t*)bias;
  a.res = (const uint16_t*)res;
  const unsigned groups = (unsigned)row_groups(N);
  return launch_wide<kBiasResidual>(a, groups, s);
}

// the QKV projection with bias, RoPE and the cache append, M <= 64 (above 16
// without the norm, and K <= 3072)
int attn_launch_rows_qkv(const void* x, int M, int K, const void* W, const void* norm_w, float eps,
                         const void* bias, const int* positions, const int* slots,
                         const float* inv_freq, float conc, void* cache, int num_pages,
                         void* q_out, hipStream_t s) {
  using namespace rows;
  Args a{};
  a.x = (const uint16_t*)x;
  a.M = M;
  a.K = K;
  a.W = (const uint16_t*)W;
  a.N = (kHq + 2 * kHkv) * kD;
  a.norm_w = (const uint16_t*)norm_w;
  a.eps = eps;
  a.bias = (const uint16_t*)bias;
  a.positions = positions;
  a.slots = slots;
  a.inv_freq = inv_freq;
  a.conc = conc;
  a.cache = (uint8_t*)cache;
  a.num_pages = num_pages;
  a.q_out = (uint16_t*)q_out;
  const dim3 grid(a.N / 32);
  if (M > 16) return norm_w ? -6 : launch_wide<kQkv>(a, grid.x, s);
  return norm_w ? launch<kQkv, true>(a, grid, 0, s) : launch<kQkv, false>(a, grid, 0, s);
}

}  // extern "C"
