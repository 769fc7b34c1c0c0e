// Dense projections of the gpt-oss layer for one token (dense_rows.hip takes
// two and more): the fused QKV nn.Linear with its bias, YaRN RoPE and the
// KV-cache append; the attention output nn.Linear with its bias and the residual
// add; the unembedding (model/attention.py:204,254-256; model/transformer.py:
// 95-100).
// The QKV projection and the unembedding can also apply the RMSNorm before
// them (attention.py:80, transformer.py:63) to the rows they stage.
//
// y[n] = sum_k x[k] W[n][k], bf16 operands, fp32 accumulation, one bf16
// rounding (the matmul's output dtype), then the epilogue's own bf16 ops.
// HBM-bound on W.  A workgroup takes RW rows of W; its 4 waves split K (wave
// w takes the 16-byte chunks w * 64 + lane + 256 i of each row), so a row's
// bytes stream from four waves at once; the four partial sums are added in
// wave order through LDS (deterministic).  The token x is staged in LDS.
// Loads complete in issue order, so everything small that the workgroup
// needs (its x chunks, the epilogue's bias, residual, positions, slots and
// RoPE frequencies) is loaded before the W rows, and the epilogue's cos and
// sin are taken while W streams: the RMSNorm and the epilogue then wait for
// nothing behind the W loads.
#include "moe_common.h"

namespace gemv {

using moe::bf2f;
using moe::f2bf;
using moe::u32x4;

constexpr int kThreads = 256;  // 4 waves
constexpr int kWaves = 4;
constexpr int kIters = 2;  // 16-byte chunk rounds per lane: K <= 4096 = 2 x 256 x 8

// gpt-oss attention shapes (the QKV epilogue)
constexpr int kD = 64, kHq = 64, kHkv = 8, kPage = 16;
constexpr int kHeadBlock = kPage * kD * 2;
constexpr int kPageBytes = 2 * kHkv * kHeadBlock;

__device__ __forceinline__ float dot8(u32x4 w, u32x4 x, float acc) {
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    acc = fmaf(__uint_as_float(w[j] << 16), __uint_as_float(x[j] << 16), acc);
    acc = fmaf(__uint_as_float(w[j] & 0xFFFF0000u), __uint_as_float(x[j] & 0xFFFF0000u), acc);
  }
  return acc;
}

enum Epi { kPlain = 0, kBiasResidual = 1, kQkv = 2 };

struct Args {
  const uint16_t* x;
  int K;
  const uint16_t* W;
  int N;
  uint16_t* out;
  const uint16_t* norm_w;  // non-null: RMSNorm the staged rows first
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

template <int RW, int EPI>
__global__ __launch_bounds__(kThreads) void gemv_kernel(Args a) {
#pragma clang fp contract(off)
  extern __shared__ __align__(16) uint16_t xs[];  // the token's row, K bf16
  __shared__ float part[kWaves][RW];
  __shared__ double ssq[kWaves];
  const int t = threadIdx.x, wave = t >> 6, lane = t & 63;
  const int K = a.K, N = a.N;
  const int chunks = K / 8;
  // this workgroup's rows
  int rows[RW];
  if constexpr (EPI == kQkv) {
    // rope pairs (j, j + 32) of head h: workgroup g takes pairs
    // j = (RW / 2) * (g % (32 / (RW / 2))) .. + RW / 2 - 1
    constexpr int kPairs = RW / 2, kBlocks = 32 / kPairs;
    const int h = blockIdx.x / kBlocks, jb = blockIdx.x % kBlocks;
#pragma unroll
    for (int i = 0; i < kPairs; ++i) {
      rows[2 * i] = h * kD + jb * kPairs + i;
      rows[2 * i + 1] = h * kD + jb * kPairs + i + 32;
    }
  } else {
#pragma unroll
    for (int i = 0; i < RW; ++i) rows[i] = blockIdx.x * RW + i;
  }
  // x's chunks of this thread and the epilogue's operands first (they are needed first),
  // then every W load of this lane (K <= 4096: at most two rounds of 256
  // 16-byte chunks) with the norm weight's chunks when the rows are
  // normalised.  Every load is unconditional (indices clamped into range,
  // values past the row never used, raw bits converted where they are
  // used): a load under a branch made the compiler wait for it inside the
  // branch, which split the weight loads into three rounds with a full wait
  // between them.
  const bool norm = a.norm_w != nullptr;
  const uint16_t* const nw = norm ? a.norm_w : a.W;  // (loaded, unused, without a norm)
  u32x4 xr[kIters];
#pragma unroll
  for (int it = 0; it < kIters; ++it)
    xr[it] = *(const u32x4*)(a.x + min(it * kThreads + t, chunks - 1) * 8);
  // the epilogue task of this thread (one per row or rope pair)
  constexpr int kTasks = EPI == kQkv ? RW / 2 : RW;
  const bool task = t < kTasks;
  const int ti = task ? t : 0;
  uint16_t eb0r = 0, eb1r = 0, err = 0;
  float cs = 0.f, sn = 0.f, ifq = 0.f;
  int eslot = -1, epos = 0;
  if constexpr (EPI == kBiasResidual) {
    const int n = min(rows[ti], N - 1);
    eb0r = a.bias[n];
    err = a.res[n];
  } else if constexpr (EPI == kQkv) {
    const int nlo = rows[2 * ti], nhi = rows[2 * ti + 1];
    eb0r = a.bias[nlo];
    eb1r = a.bias[nhi];
    eslot = a.slots[0];
    epos = a.positions[0];
    ifq = a.inv_freq[nlo % kD];
  }
  __builtin_amdgcn_sched_barrier(0);
  u32x4 wv[kIters][RW];
  u32x4 nwv[kIters];
#pragma unroll
  for (int it = 0; it < kIters; ++it) {
    const int cc = min(it * kThreads + wave * 64 + lane, chunks - 1);
#pragma unroll
    for (int i = 0; i < RW; ++i)
      wv[it][i] = *(const u32x4*)(a.W + (size_t)min(rows[i], N - 1) * K + cc * 8);
    nwv[it] = *(const moe::u32x4_any*)(nw + cc * 8);  // (a caller's slice at any element)
  }
  __builtin_amdgcn_sched_barrier(0);
  // the RoPE factors while W streams
  if constexpr (EPI == kQkv) {
    if (task && rows[2 * ti] / kD < kHq + kHkv) {
      const float freq = (float)epos * ifq;
      double sd, cd;
      moe::sincos_f64((double)freq, sd, cd);
      cs = bf2f(moe::f64_to_bf16_via_f32(cd)) * a.conc;
      sn = bf2f(moe::f64_to_bf16_via_f32(sd)) * a.conc;
    }
  }
  // Stage x; for the RMSNorm, the sum of squares of the bf16 values in fp64
  // (exact for a row spanning less than 2^37) on the way, as the standalone
  // kernel: r = fp32(1 / sqrt(ss / K + eps)), t = bf16(fp32(x r) w)
  double ss = 0.0;
#pragma unroll
  for (int it = 0; it < kIters; ++it) {
    const int c = it * kThreads + t;
    if (c >= chunks) continue;
    const u32x4 v = xr[it];
    *(u32x4*)(xs + c * 8) = v;
    if (norm) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const double lo = (double)__uint_as_float(v[j] << 16);
        const double hi = (double)__uint_as_float(v[j] & 0xFFFF0000u);
        ss += lo * lo + hi * hi;
      }
    }
  }
  if (norm) {
    ss = moe::wave_sum(ss);
    if (lane == 0) ssq[wave] = ss;
  }
  __syncthreads();
  float rn = 1.0f;
  if (norm) {
    const double tot = (ssq[0] + ssq[1]) + (ssq[2] + ssq[3]);
    rn = (float)(1.0 / sqrt(tot / (double)K + (double)a.eps));
  }
  float acc[RW];
#pragma unroll
  for (int i = 0; i < RW; ++i) acc[i] = 0.f;
#pragma unroll
  for (int it = 0; it < kIters; ++it) {
    const int c = it * kThreads + wave * 64 + lane;
    if (c < chunks) {
      u32x4 xv = *(const u32x4*)(xs + c * 8);
      if (norm) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const uint32_t lo = f2bf(__fmul_rn(__fmul_rn(__uint_as_float(xv[j] << 16), rn),
                                             __uint_as_float(nwv[it][j] << 16)));
          const uint32_t hi = f2bf(__fmul_rn(__fmul_rn(__uint_as_float(xv[j] & 0xFFFF0000u), rn),
                                             __uint_as_float(nwv[it][j] & 0xFFFF0000u)));
          xv[j] = lo | (hi << 16);
        }
      }
#pragma unroll
      for (int i = 0; i < RW; ++i) acc[i] = dot8(wv[it][i], xv, acc[i]);
    }
  }
#pragma unroll
  for (int i = 0; i < RW; ++i) {
    const float v = moe::wave_sum(acc[i]);
    if (lane == 0) part[wave][i] = v;
  }
  __syncthreads();
  // epilogue: one thread per row or rope pair; partials in wave order
  auto total = [&](int i) { return ((part[0][i] + part[1][i]) + part[2][i]) + part[3][i]; };
  if constexpr (EPI == kPlain || EPI == kBiasResidual) {
    if (task) {
      const int n = rows[ti];
      if (n < N) {
        const uint16_t y = f2bf(total(ti));
        if constexpr (EPI == kPlain) {
          a.out[n] = y;
        } else {
          const float tb = bf2f(f2bf(bf2f(y) + bf2f(eb0r)));
          a.out[n] = f2bf(bf2f(err) + tb);
        }
      }
    }
  } else {
    // bias (its own bf16 rounding), then YaRN RoPE of q / k heads exactly as
    // the standalone append kernel does, then q out or the cache slot
    if (task) {
      const int nlo = rows[2 * ti];
      const int head = nlo / kD, d = nlo % kD;
      float lo = bf2f(f2bf(bf2f(f2bf(total(2 * ti))) + bf2f(eb0r)));
      float hi = bf2f(f2bf(bf2f(f2bf(total(2 * ti + 1))) + bf2f(eb1r)));
      if (head < kHq + kHkv) {
        const float nl = lo * cs - hi * sn;
        const float nh = lo * sn + hi * cs;
        lo = nl;
        hi = nh;
      }
      const uint16_t blo = f2bf(lo), bhi = f2bf(hi);
      const int slot = eslot;
      if (head < kHq) {
        uint16_t* qo = a.q_out + (size_t)head * kD;
        qo[d] = blo;
        qo[d + 32] = bhi;
      } else if (slot >= 0 && slot < a.num_pages * kPage) {
        const int kv = head < kHq + kHkv ? 0 : 1;
        const int hk = head - kHq - kv * kHkv;
        uint16_t* row = (uint16_t*)(a.cache + (size_t)(slot / kPage) * kPageBytes +
                                    (size_t)(kv * kHkv + hk) * kHeadBlock +
                                    (slot % kPage) * (kD * 2));
        row[d] = blo;
        row[d + 32] = bhi;
      }
    }
  }
}

}  // namespace gemv

extern "C" {

int attn_launch_gemv(const void* x, int K, const void* W, int N, void* out, const void* norm_w,
                     float eps, const void* bias, const void* res, hipStream_t s) {
  using namespace gemv;
  Args a{};
  a.x = (const uint16_t*)x;
  a.K = K;
  a.W = (const uint16_t*)W;
  a.N = N;
  a.out = (uint16_t*)out;
  a.norm_w = (const uint16_t*)norm_w;
  a.eps = eps;
  a.bias = (const uint16_t*)bias;
  a.res = (const uint16_t*)res;
  auto go = [&](auto kernel, unsigned rw) {
    hipLaunchKernelGGL(kernel, dim3(((unsigned)N + rw - 1) / rw), dim3(kThreads), (size_t)K * 2, s,
                       a);
    return hipGetLastError() == hipSuccess ? 0 : -6;
  };
  // Four rows a workgroup (58 VGPRs, eight waves per SIMD; us with
  // 4, 8, 12 and 16 rows, 161 VGPRs and three waves: the 201088 x 2880 unembedding
  // with its norm and the sampler behind it 201, 206, 204 and 210, alone 176, 181,
  // 180 and 187; 131072 x 4096 177, 192, 185 and 182; 4096 x 2880 7.9, 8.8, 10.7 and
  // 10.9).  A launch holds less than 2^32 threads: for more rows 16.
  if (bias) return go(gemv_kernel<4, kBiasResidual>, 4);
  constexpr int kMostGroups = (1 << 24) - 1;
  return N <= 4 * kMostGroups ? go(gemv_kernel<4, kPlain>, 4) : go(gemv_kernel<16, kPlain>, 16);
}

int attn_launch_qkv_gemv(const void* x, int K, const void* W, const void* norm_w, float eps,
                         const void* bias, const int* positions, const int* slots,
                         const float* inv_freq, float conc, void* cache, int num_pages,
                         void* q_out, hipStream_t s) {
  using namespace gemv;
  constexpr int heads = kHq + 2 * kHkv;
  constexpr int RW = 4;  // two rope pairs per workgroup
  Args a{};
  a.x = (const uint16_t*)x;
  a.K = K;
  a.W = (const uint16_t*)W;
  a.N = heads * kD;
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
  hipLaunchKernelGGL((gemv_kernel<RW, kQkv>), dim3(heads * (32 / (RW / 2))), dim3(kThreads),
                     (size_t)K * 2, s, a);
  return hipGetLastError() == hipSuccess ? 0 : -6;
}

}  // extern "C"
