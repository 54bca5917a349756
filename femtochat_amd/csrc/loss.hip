// Loss-side kernels (gfx950): cross-entropy over a vocabulary column and its
// gradient, the embedding gather and its scatter-add gradient.
//
// Semantics (reference):
//   cross_entropy            src/gpt.jl:175-195, ext/FemtoChatCUDAExt.jl:21-54
//     loss[t] = max + log(sum(exp(x - max))) - x[target[t]], 0 if ignored;
//   cross_entropy_gradient!  src/kernels.jl:16-28, CUDAExt:56-61
//     delta[:, t] += scale[t] (softmax(x) - onehot(target[t])), skipped if ignored;
//   embedding                src/gpt.jl:34, CUDAExt:63-76   y[:, t] = W[:, tokens[t]];
//   embedding_gradient!      src/kernels.jl:8-14, CUDAExt:78-94
//     dW[:, tokens[t]] += dy[:, t], zero values skipped (no atomics for padding).
// Layout: column-major as the reference (a token's vocabulary column, or an
// embedding column, is contiguous).
//
// All four are HBM-bound.  Cross-entropy: one 256-thread workgroup per token;
// a single pass keeps a running (max, sum of exp) per thread, eight 16-byte
// loads in flight per round, combined across the workgroup at the end.  The
// gradient reuses the forward's log-sum-exp when the caller passes it (one
// read of the logits instead of two) and is then elementwise over the whole
// array.
#include "attn_launch.hpp"
#include "attn_device.hpp"

#include <cmath>

namespace fc {

namespace {

constexpr float kLog2e = 1.4426950408889634f;
constexpr int kFwdBatch = 8;  // 16-byte loads in flight per thread in a forward round (4, 8, 16 within 1%)
constexpr int kWaveV = 2048;  // longest column that a wave reads in one round
constexpr int kWaveN = 1024;  // columns from which on waves take up to three rounds (four waves per CU)
constexpr int kBwdBatch = 8;  // chunks per backward round (4, 8 measured within 3%)

template <typename I>
__device__ inline int64_t read_index(const void* p, int64_t i) {
  return (int64_t) static_cast<const I*>(p)[i];
}

__device__ inline int64_t index_at(const void* p, int64_t i, int type) {
  return type == 1 ? read_index<int64_t>(p, i) : read_index<int32_t>(p, i);
}

// (m, s) with s = sum exp(x - m) over what a thread or group has seen; s = 0
// means nothing seen (m is then -inf and must not enter an exponent).
struct Lse {
  float m, s;
};

__device__ inline Lse combine(Lse a, Lse b) {
  const float m = fmaxf(a.m, b.m);
  const float sa = a.s == 0.0f ? 0.0f : a.s * exp2f((a.m - m) * kLog2e);
  const float sb = b.s == 0.0f ? 0.0f : b.s * exp2f((b.m - m) * kLog2e);
  return Lse{m, sa + sb};
}

// Workgroup-wide combine of every thread's (m, s); all threads get the result.
__device__ inline Lse block_combine(Lse v) {
  __shared__ float sm[4], ss[4];
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) v = combine(v, Lse{__shfl_xor(v.m, o), __shfl_xor(v.s, o)});
  const int wave = threadIdx.x / 64;
  if ((threadIdx.x & 63) == 0) {
    sm[wave] = v.m;
    ss[wave] = v.s;
  }
  __syncthreads();
  Lse r{sm[0], ss[0]};
#pragma unroll
  for (int w = 1; w < 4; ++w) r = combine(r, Lse{sm[w], ss[w]});
  __syncthreads();  // the shared slots are free again when this returns
  return r;
}

// One thread's pass over its part of a column: up to three values in front of
// the first 16-byte boundary and after the last one go to the first threads,
// the aligned chunks between them to thread tid, tid + 256, ...  Each round
// loads up to eight chunks, then folds their maximum into m with one rescale
// of s.  A column whose vocabulary is not a multiple of 4 starts off a
// boundary in three rows of four (1024 x 50257 took 113 us value by value, 38
// this way; 1024 x 50304, aligned, 37).
// kStream: the column is read only once (the forward), so the loads are
// nontemporal (25% faster at 8192 x 32768); the gradient, which reads the
// column again, keeps it in the caches.
// kThreads threads (tid) share the column, kBatch chunks each per round.
template <bool kStream, int kThreads = 256, int kBatch = kFwdBatch>
__device__ inline Lse column_pass(const float* col, int V, int tid) {
  const int head = min((int)((16 - (reinterpret_cast<uintptr_t>(col) & 15)) & 15) / 4, V);
  const int chunks = (V - head) / 4, tail = V - head - 4 * chunks;
  const float* body = col + head;
  Lse acc{-INFINITY, 0.0f};
  // x = -inf adds nothing (and must not set a reference of -inf).
  auto one = [](float x) { return Lse{x, x == -INFINITY ? 0.0f : 1.0f}; };
  if (tid < head) acc = combine(acc, one(col[tid]));
  if (tid < tail) acc = combine(acc, one(body[4 * chunks + tid]));
  for (int base = tid; base < chunks; base += kThreads * kBatch) {
    f32x4 v[kBatch];
    float bm = -INFINITY;
#pragma unroll
    for (int k = 0; k < kBatch; ++k) {
      const int c = base + kThreads * k;
      const f32x4* p = reinterpret_cast<const f32x4*>(body + 4 * c);
      v[k] = c < chunks ? (kStream ? __builtin_nontemporal_load(p) : *p) : f32x4{-INFINITY, -INFINITY, -INFINITY, -INFINITY};
    }
#pragma unroll
    for (int k = 0; k < kBatch; ++k) bm = fmaxf(bm, fmaxf(fmaxf(v[k][0], v[k][1]), fmaxf(v[k][2], v[k][3])));
    const float m = fmaxf(acc.m, bm);
    const float ref = m == -INFINITY ? 0.0f : m;  // every value so far is -inf: all exponentials are 0
    float s = acc.s == 0.0f ? 0.0f : acc.s * exp2f((acc.m - ref) * kLog2e);
#pragma unroll
    for (int k = 0; k < kBatch; ++k)
#pragma unroll
      for (int i = 0; i < 4; ++i) s += exp2f((v[k][i] - ref) * kLog2e);  // exp2(-inf) = 0 for padding
    acc = Lse{m, s};
  }
  return acc;
}

__device__ inline void store_loss(const XentArgs& a, int64_t token, const float* col, Lse r) {
  const float lse = r.m + logf(r.s);
  const int64_t raw = index_at(a.targets, token, a.index_type);
  const int64_t t = raw - a.index_base;
  float loss = 0.0f;
  if (raw != a.ignore_index) loss = (t >= 0 && t < a.V) ? lse - col[t] : __builtin_nanf("");
  a.losses[token] = loss;
  if (a.lse != nullptr) a.lse[token] = lse;
}

__global__ __launch_bounds__(256) void xent_fwd_kernel(XentArgs a) {
  const int64_t token = blockIdx.x;
  const float* col = a.logits + token * (int64_t)a.V;
  const Lse r = block_combine(column_pass<true>(col, a.V, threadIdx.x));
  if (threadIdx.x == 0) store_loss(a, token, col, r);
}

// Short columns: a wave each, four to a workgroup, no barrier, with as many loads
// in flight as the column has for a lane.  us, a workgroup / a wave each:
// 8192 x 50 19 / 6.0, x 1000 28 / 8.6, x 2048 27.7 / 13.5, x 4096 30.3 / 23.5, x 6001
// 36.6 / 32.8, x 8192 43.6 / 45.6; 1024 x 2048 6.7 / 4.7, x 4096 6.9 / 6.3, x 6001
// 7.6 / 7.4, x 8192 7.4 / 8.6; 512 x 3000 5.3 / 6.0; 256 x 2048 4.5 / 4.6 (with four
// loads in flight 5.3), x 3000 4.6 / 6.0; 8 x 1500 4.4 / 4.3.
template <int kBatch>
__global__ __launch_bounds__(256) void xent_fwd_wave_kernel(XentArgs a) {
  const int64_t token = (int64_t)blockIdx.x * 4 + threadIdx.x / 64;
  if (token >= a.N) return;
  const int lane = threadIdx.x & 63;
  const float* col = a.logits + token * (int64_t)a.V;
  Lse r;
  if constexpr (kBatch == 0) {  // up to 256 values: four per lane, one by one, whatever the column's alignment
    float x[4], m = -INFINITY, sum = 0.0f;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      x[k] = lane + 64 * k < a.V ? __builtin_nontemporal_load(col + lane + 64 * k) : -INFINITY;
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) m = fmaxf(m, x[k]);
    const float ref = m == -INFINITY ? 0.0f : m;
#pragma unroll
    for (int k = 0; k < 4; ++k) sum += exp2f((x[k] - ref) * kLog2e);
    r = Lse{m, sum};
  } else {
    r = column_pass<true, 64, kBatch>(col, a.V, lane);
  }
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) r = combine(r, Lse{__shfl_xor(r.m, o), __shfl_xor(r.s, o)});
  if (lane == 0) store_loss(a, token, col, r);
}

// reduced[0] = sum of losses (or their mean over valid targets), reduced[1] =
// number of valid targets; one workgroup, float64 accumulation.
__global__ __launch_bounds__(1024) void xent_reduce_kernel(XentArgs a) {
  __shared__ double part[16];
  __shared__ double cnt[16];
  double s = 0.0, c = 0.0;
  constexpr int kRun = 8;  // loads in flight per thread
  for (int64_t base = threadIdx.x; base < a.N; base += 1024 * kRun) {
    float loss[kRun];
    int64_t t[kRun];
#pragma unroll
    for (int k = 0; k < kRun; ++k) {
      const int64_t i = min(base + 1024 * k, a.N - 1);
      loss[k] = a.losses != nullptr ? a.losses[i] : 0.0f;
      t[k] = index_at(a.targets, i, a.index_type);
    }
#pragma unroll
    for (int k = 0; k < kRun; ++k) {
      if (base + 1024 * k >= a.N) continue;
      s += (double)loss[k];
      c += t[k] != a.ignore_index ? 1.0 : 0.0;
    }
  }
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) {
    s += __shfl_xor(s, o);
    c += __shfl_xor(c, o);
  }
  if ((threadIdx.x & 63) == 0) {
    part[threadIdx.x / 64] = s;
    cnt[threadIdx.x / 64] = c;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    double S = 0.0, C = 0.0;
    for (int w = 0; w < 16; ++w) {
      S += part[w];
      C += cnt[w];
    }
    if (a.reduced != nullptr) a.reduced[0] = (float)(a.reduction == 2 ? S / C : S);
    if (a.count != nullptr) *a.count = (float)C;
  }
}

// The gradient's factor: dy / count(valid) ("mean"), dy ("sum"), dy[token]
// ("none"); the division is the reference's fp32 `dy ./ sum(valid)`.
__device__ inline float grad_factor(const XentArgs& a, int64_t token) {
  const float w = a.dy[a.reduction == 0 ? token : 0];
  return a.reduction == 2 ? w / *a.count : w;
}

// Gradient with a given log-sum-exp: nothing is summed over a column, so the
// (token, vocabulary) array is taken as one run of 16-byte chunks, one per
// thread in address order, whatever V is; a chunk that crosses into the next
// token's column (V not a multiple of 4) goes value by value.  All accesses are
// nontemporal.  HBM-bound: the chip sweeps one window of 4 KB blocks instead
// of 2048 columns at a time, which took 8192 x 32768 (read and written once)
// from 472 us (one workgroup per column) to 326, 6.6 TB/s, and from 616 us to
// 497 added into the gradient.  More chunks per thread
// were slower: 342, 348 and 360 us with 2, 4 and 8, against 331 with one (the
// same pass with the targets left out), and so was a contiguous eighth of the
// array per XCD (341).
// n = N V < 2^31 values; by_V divides a value's index by V.
// One 16-byte chunk inside one token's column, values j .. j + 3 of it.
template <bool kOverwrite>
__device__ inline void grad_chunk(const XentArgs& a, uint32_t token, uint32_t e, uint32_t j) {
  const f32x4* in = reinterpret_cast<const f32x4*>(a.logits + e);
  f32x4* out = reinterpret_cast<f32x4*>(a.dlogits + e);
  const int64_t raw = index_at(a.targets, token, a.index_type);
  const float lse = a.lse_in[token];
  if (raw == a.ignore_index) {  // the reference adds zero
    if (kOverwrite && a.zero_ignored) __builtin_nontemporal_store(f32x4{0.0f, 0.0f, 0.0f, 0.0f}, out);
    return;
  }
  const f32x4 x = __builtin_nontemporal_load(in);
  f32x4 o;
  if (!kOverwrite) o = __builtin_nontemporal_load(out);
  const float w = grad_factor(a, token);
  const int64_t at = raw - a.index_base;  // outside [0, V): no one-hot term, as the reference's comparison
  const int t = at >= 0 && at < a.V ? (int)at - (int)j : -1;
  f32x4 g;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float p = exp2f((x[i] - lse) * kLog2e);
    g[i] = w * (p - (i == t ? 1.0f : 0.0f));
  }
  __builtin_nontemporal_store(kOverwrite ? g : o + g, out);
}

template <bool kOverwrite>
__global__ __launch_bounds__(256) void xent_grad_kernel(XentArgs a, FastDiv by_V, uint32_t n) {
  const uint32_t V = (uint32_t)a.V;
  // A block inside one column has its token, target and log-sum-exp in scalar
  // registers (the same pass with them per thread took 373 us).
  const uint32_t e0 = 1024 * blockIdx.x, token0 = divide(e0, by_V), j0 = e0 - token0 * V;
  if (j0 + 1024 <= V) {
    grad_chunk<kOverwrite>(a, token0, e0 + 4 * threadIdx.x, j0 + 4 * threadIdx.x);
    return;
  }
  const uint32_t e = e0 + 4 * threadIdx.x;
  const uint32_t token = divide(min(e, n - 1), by_V), j = e - token * V;
  if (__builtin_amdgcn_ballot_w64(e < n && j + 4 > V) == 0) {
    if (e < n) grad_chunk<kOverwrite>(a, token, e, j);
    return;
  }
  if (e >= n) return;
  // A wave with a chunk that crosses into the next column: all its chunks with a
  // token for each value, every load issued before its use.  (The crossing chunks
  // alone, value by value after the others, cost their wave a trip to memory for
  // each value: 1024 x 50 4.9 us, 3.5 now; 8192 x 2049 28.1, 25.4 now.)
  uint32_t tok[4], at[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const bool next = i > 0 && at[i - 1] + 1 == V;
    tok[i] = i == 0 ? token : next ? tok[i - 1] + 1 : tok[i - 1];
    at[i] = i == 0 ? j : next ? 0 : at[i - 1] + 1;
  }
  const bool whole = e + 4 <= n;
  f32x4 x, o;
  if (whole) {
    x = __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(a.logits + e));
    if (!kOverwrite) o = __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(a.dlogits + e));
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      x[i] = a.logits[min(e + i, n - 1)];
      if (!kOverwrite) o[i] = a.dlogits[min(e + i, n - 1)];
    }
  }
  bool written[4];
  f32x4 g;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const uint32_t t = e + i < n ? tok[i] : token;
    const int64_t raw = index_at(a.targets, t, a.index_type);
    const float p = exp2f((x[i] - a.lse_in[t]) * kLog2e);
    const bool ignored = raw == a.ignore_index;
    g[i] = grad_factor(a, t) * (p - ((int64_t)at[i] == raw - a.index_base ? 1.0f : 0.0f));
    g[i] = ignored ? 0.0f : kOverwrite ? g[i] : o[i] + g[i];
    written[i] = e + i < n && !(ignored && !(kOverwrite && a.zero_ignored));
  }
  if (whole && written[0] && written[1] && written[2] && written[3]) {
    __builtin_nontemporal_store(g, reinterpret_cast<f32x4*>(a.dlogits + e));
    return;
  }
#pragma unroll
  for (int i = 0; i < 4; ++i)
    if (written[i]) a.dlogits[e + i] = g[i];
}

// Gradient of one column per workgroup: the log-sum-exp is formed here when
// the caller has none, and buffers off a 16-byte boundary (kVec false) go
// value by value.
template <bool kVec>
__global__ __launch_bounds__(256) void xent_bwd_kernel(XentArgs a) {
  const int64_t token = blockIdx.x;
  const int64_t raw = index_at(a.targets, token, a.index_type);
  const float* col = a.logits + token * (int64_t)a.V;
  float* out = a.dlogits + token * (int64_t)a.V;
  if (raw == a.ignore_index) {  // the reference adds zero (uniform per workgroup)
    if (a.zero_ignored)
      for (int j = threadIdx.x; j < a.V; j += 256) out[j] = 0.0f;
    return;
  }
  float lse;
  if (a.lse_in != nullptr) {
    lse = a.lse_in[token];
  } else {
    const Lse r = block_combine(column_pass<false>(col, a.V, threadIdx.x));
    lse = r.m + logf(r.s);
  }
  const float w = grad_factor(a, token);
  const int64_t t = raw - a.index_base;  // outside [0, V): no one-hot term, as the reference's comparison
  if (kVec) {
    // rounds of kBwdBatch 16-byte chunks: every load of a round (logits and,
    // when accumulating, the gradient) is issued before its arithmetic
    const int chunks = a.V / 4;
    for (int base = threadIdx.x; base < chunks; base += 256 * kBwdBatch) {
      f32x4 x[kBwdBatch], o[kBwdBatch];
#pragma unroll
      for (int k = 0; k < kBwdBatch; ++k) {
        const int c = base + 256 * k;
        if (c < chunks) {
          x[k] = *reinterpret_cast<const f32x4*>(col + 4 * c);
          o[k] = a.overwrite ? f32x4{0.0f, 0.0f, 0.0f, 0.0f} : *reinterpret_cast<const f32x4*>(out + 4 * c);
        }
      }
#pragma unroll
      for (int k = 0; k < kBwdBatch; ++k) {
        const int c = base + 256 * k;
        if (c >= chunks) continue;
        f32x4 g;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float p = exp2f((x[k][i] - lse) * kLog2e);
          g[i] = w * (p - (4 * c + i == t ? 1.0f : 0.0f));
        }
        // nontemporal store (1.6% faster here; not in the fused kernel, where it was slower)
        __builtin_nontemporal_store(a.overwrite ? g : o[k] + g, reinterpret_cast<f32x4*>(out + 4 * c));
      }
    }
  } else {
    for (int j = threadIdx.x; j < a.V; j += 256) {
      const float p = exp2f((col[j] - lse) * kLog2e);
      const float g = w * (p - (j == t ? 1.0f : 0.0f));
      out[j] = a.overwrite ? g : out[j] + g;
    }
  }
}

// ---- fused forward and gradient ------------------------------------------------
// One 1024-thread workgroup per token holds the whole column in registers
// (up to kFusedChunks 16-byte chunks per thread: V <= 4096 kFusedChunks),
// so the logits are read once: maximum, sum of exponentials, the loss, and
// the gradient scale (p - onehot) written (or added) in the same pass.
constexpr int kFusedChunks = 8;
constexpr int kFusedThreads = 1024;

__device__ inline float block_reduce_1024(float v, bool is_max, float* slots) {
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) {
    const float u = __shfl_xor(v, o);
    v = is_max ? fmaxf(v, u) : v + u;
  }
  if ((threadIdx.x & 63) == 0) slots[threadIdx.x / 64] = v;
  __syncthreads();
  float r = slots[0];
#pragma unroll
  for (int w = 1; w < 16; ++w) r = is_max ? fmaxf(r, slots[w]) : r + slots[w];
  __syncthreads();
  return r;
}

__global__ __launch_bounds__(kFusedThreads) void xent_fused_kernel(XentArgs a) {
  __shared__ float slots[16];
  const int64_t token = blockIdx.x;
  const float* col = a.logits + token * (int64_t)a.V;
  float* out = a.dlogits + token * (int64_t)a.V;
  const int chunks = a.V / 4;
  f32x4 x[kFusedChunks];
  float mx = -INFINITY;
#pragma unroll
  for (int k = 0; k < kFusedChunks; ++k) {
    const int c = threadIdx.x + kFusedThreads * k;
    x[k] = c < chunks ? *reinterpret_cast<const f32x4*>(col + 4 * c) : f32x4{-INFINITY, -INFINITY, -INFINITY, -INFINITY};
    mx = fmaxf(mx, fmaxf(fmaxf(x[k][0], x[k][1]), fmaxf(x[k][2], x[k][3])));
  }
  const float M = block_reduce_1024(mx, true, slots);
  float sum = 0.0f;
#pragma unroll
  for (int k = 0; k < kFusedChunks; ++k)
#pragma unroll
    for (int i = 0; i < 4; ++i) sum += exp2f((x[k][i] - M) * kLog2e);
  const float lse = M + logf(block_reduce_1024(sum, false, slots));
  const int64_t raw = index_at(a.targets, token, a.index_type);
  const int64_t t = raw - a.index_base;
  const bool valid = raw != a.ignore_index;
  if (threadIdx.x == 0) {
    a.losses[token] = valid ? ((t >= 0 && t < a.V) ? lse - col[t] : __builtin_nanf("")) : 0.0f;
    if (a.lse != nullptr) a.lse[token] = lse;
  }
  if (!valid) return;  // uniform: the gradient column is left untouched, as the separate gradient does
  float w = a.dy[a.reduction == 0 ? token : 0];
  if (a.reduction == 2) w = w / *a.count;
#pragma unroll
  for (int k = 0; k < kFusedChunks; ++k) {
    const int c = threadIdx.x + kFusedThreads * k;
    if (c >= chunks) continue;
    f32x4 g;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float p = exp2f((x[k][i] - lse) * kLog2e);
      g[i] = w * (p - (4 * c + i == t ? 1.0f : 0.0f));
    }
    f32x4* o = reinterpret_cast<f32x4*>(out + 4 * c);
    *o = a.overwrite ? g : *o + g;
  }
}

// ---- embedding ----------------------------------------------------------------
// One wave per token, 16-byte chunks of its column (D % 4 == 0) or scalars.
template <bool kVec, typename Y>
__global__ __launch_bounds__(256) void embed_fwd_kernel(EmbedArgs a) {
  const int64_t token = (int64_t)blockIdx.x * 4 + threadIdx.x / 64;
  if (token >= a.N) return;
  const int lane = threadIdx.x & 63;
  const int64_t id = index_at(a.tokens, token, a.index_type) - a.index_base;
  const bool ok = id >= 0 && id < a.vocab;  // an out-of-range id poisons its column (an index error in the reference)
  const float* w = a.weights + (ok ? id : 0) * (int64_t)a.D;
  Y* y = static_cast<Y*>(a.y) + token * (int64_t)a.D;
  const float poison = ok ? 1.0f : __builtin_nanf("");
  if (kVec) {
    for (int c = lane; c < a.D / 4; c += 64) {
      f32x4 v = *reinterpret_cast<const f32x4*>(w + 4 * c);
      if (!ok) v = f32x4{poison, poison, poison, poison};
      if constexpr (sizeof(Y) == 4) {
        *reinterpret_cast<f32x4*>(y + 4 * c) = v;
      } else {
        typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
        *reinterpret_cast<bf16x4*>(y + 4 * c) = __builtin_convertvector(v, bf16x4);
      }
    }
  } else {
    for (int j = lane; j < a.D; j += 64) y[j] = static_cast<Y>(ok ? w[j] : poison);
  }
}

template <bool kVec, typename Y>
__global__ __launch_bounds__(256) void embed_bwd_kernel(EmbedArgs a) {
  const int64_t token = (int64_t)blockIdx.x * 4 + threadIdx.x / 64;
  if (token >= a.N) return;
  const int lane = threadIdx.x & 63;
  const int64_t id = index_at(a.tokens, token, a.index_type) - a.index_base;
  if (id < 0 || id >= a.vocab) return;  // nothing to add for an id outside the table
  float* dw = a.dweights + id * (int64_t)a.D;
  const Y* dy = static_cast<const Y*>(a.dy) + token * (int64_t)a.D;
  auto add = [&](int j, float v) {
    if (v != 0.0f) unsafeAtomicAdd(dw + j, v);  // hardware fp32 atomic add in L2
  };
  if (kVec) {
    for (int c = lane; c < a.D / 4; c += 64) {
      f32x4 v;
      if constexpr (sizeof(Y) == 4) {
        v = *reinterpret_cast<const f32x4*>(dy + 4 * c);
      } else {
        typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
        v = __builtin_convertvector(*reinterpret_cast<const bf16x4*>(dy + 4 * c), f32x4);
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) add(4 * c + i, v[i]);
    }
  } else {
    for (int j = lane; j < a.D; j += 64) add(j, static_cast<float>(dy[j]));
  }
}

}  // namespace

hipError_t launch_xent_fwd(const XentArgs& a, hipStream_t s) {
  const ProfileMark mk = profile_begin(s);
  const dim3 waves((unsigned)((a.N + 3) / 4)), block(256);
  if (a.V <= kWaveV / 8) hipLaunchKernelGGL(xent_fwd_wave_kernel<0>, waves, block, 0, s, a);
  else if (a.V <= kWaveV / 2) hipLaunchKernelGGL(xent_fwd_wave_kernel<4>, waves, block, 0, s, a);
  else if (a.V <= kWaveV || (a.N >= kWaveN && a.V <= 3 * kWaveV)) hipLaunchKernelGGL(xent_fwd_wave_kernel<8>, waves, block, 0, s, a);
  else hipLaunchKernelGGL(xent_fwd_kernel, dim3((unsigned)a.N), block, 0, s, a);
  hipError_t e = hipGetLastError();
  profile_end(mk, "xent_fwd", s);
  if (e != hipSuccess || (a.reduced == nullptr && a.count == nullptr)) return e;
  hipLaunchKernelGGL(xent_reduce_kernel, dim3(1), dim3(1024), 0, s, a);
  return hipGetLastError();
}

hipError_t launch_xent_count(const XentArgs& a, hipStream_t s) {
  hipLaunchKernelGGL(xent_reduce_kernel, dim3(1), dim3(1024), 0, s, a);
  return hipGetLastError();
}

bool xent_fused_supported(const XentArgs& a) {
  return a.V % 4 == 0 && a.V <= 4 * kFusedThreads * kFusedChunks &&
         ((reinterpret_cast<uintptr_t>(a.logits) | reinterpret_cast<uintptr_t>(a.dlogits)) & 15) == 0;
}

hipError_t launch_xent_fused(const XentArgs& a, hipStream_t s) {
  const ProfileMark mk = profile_begin(s);
  hipLaunchKernelGGL(xent_fused_kernel, dim3((unsigned)a.N), dim3(kFusedThreads), 0, s, a);
  hipError_t e = hipGetLastError();
  profile_end(mk, "xent_fused", s);
  if (e != hipSuccess || (a.reduced == nullptr)) return e;
  // count is the caller's input here (it scaled the gradient): the reduction
  // writes only the loss sum or mean.
  XentArgs r = a;
  r.count = nullptr;
  hipLaunchKernelGGL(xent_reduce_kernel, dim3(1), dim3(1024), 0, s, r);
  return hipGetLastError();
}

// The one-run gradient, in parts of fewer than 2^31 values whose token counts
// are multiples of 4 (every part then starts on a 16-byte boundary).
static hipError_t launch_xent_grad(const XentArgs& a, hipStream_t s) {
  const int64_t part = ((((int64_t)1 << 31) - 1) / a.V) & ~(int64_t)3;
  const size_t index_size = a.index_type == 1 ? 8 : 4;
  for (int64_t at = 0; at < a.N; at += part) {
    XentArgs p = a;
    p.N = a.N - at < part ? a.N - at : part;
    p.logits += at * a.V;
    p.dlogits += at * a.V;
    p.lse_in += at;
    p.targets = static_cast<const char*>(a.targets) + at * index_size;
    if (a.reduction == 0) p.dy += at;
    const uint32_t n = (uint32_t)(p.N * p.V);
    const dim3 grid((n + 1023) / 1024);
    if (a.overwrite) hipLaunchKernelGGL(xent_grad_kernel<true>, grid, dim3(256), 0, s, p, fast_div((uint32_t)p.V), n);
    else hipLaunchKernelGGL(xent_grad_kernel<false>, grid, dim3(256), 0, s, p, fast_div((uint32_t)p.V), n);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

hipError_t launch_xent_bwd(const XentArgs& a, hipStream_t s) {
  const bool aligned = ((reinterpret_cast<uintptr_t>(a.logits) | reinterpret_cast<uintptr_t>(a.dlogits)) & 15) == 0;
  const ProfileMark mk = profile_begin(s);
  hipError_t e;
  // One run of chunks needs the log-sum-exp beforehand, 16-byte alignment of
  // both arrays and parts of at least four columns below 2^31 values.
  if (a.lse_in != nullptr && aligned && a.V < (1 << 29)) {
    e = launch_xent_grad(a, s);
  } else {
    if (aligned && a.V % 4 == 0) hipLaunchKernelGGL(xent_bwd_kernel<true>, dim3((unsigned)a.N), dim3(256), 0, s, a);
    else hipLaunchKernelGGL(xent_bwd_kernel<false>, dim3((unsigned)a.N), dim3(256), 0, s, a);
    e = hipGetLastError();
  }
  profile_end(mk, "xent_bwd", s);
  return e;
}

hipError_t launch_embed(const EmbedArgs& a, bool backward, bool bf16_y, hipStream_t s) {
  const bool vec = a.D % 4 == 0 &&
                   ((reinterpret_cast<uintptr_t>(backward ? (const void*)a.dweights : (const void*)a.weights) |
                     reinterpret_cast<uintptr_t>(backward ? a.dy : (const void*)a.y)) &
                    15) == 0;
  const dim3 grid((unsigned)((a.N + 3) / 4)), block(256);
  const ProfileMark mk = profile_begin(s);
  if (backward) {
    if (bf16_y) {
      if (vec) hipLaunchKernelGGL((embed_bwd_kernel<true, bf16>), grid, block, 0, s, a);
      else hipLaunchKernelGGL((embed_bwd_kernel<false, bf16>), grid, block, 0, s, a);
    } else {
      if (vec) hipLaunchKernelGGL((embed_bwd_kernel<true, float>), grid, block, 0, s, a);
      else hipLaunchKernelGGL((embed_bwd_kernel<false, float>), grid, block, 0, s, a);
    }
  } else {
    if (bf16_y) {
      if (vec) hipLaunchKernelGGL((embed_fwd_kernel<true, bf16>), grid, block, 0, s, a);
      else hipLaunchKernelGGL((embed_fwd_kernel<false, bf16>), grid, block, 0, s, a);
    } else {
      if (vec) hipLaunchKernelGGL((embed_fwd_kernel<true, float>), grid, block, 0, s, a);
      else hipLaunchKernelGGL((embed_fwd_kernel<false, float>), grid, block, 0, s, a);
    }
  }
  const hipError_t e = hipGetLastError();
  profile_end(mk, backward ? "embed_bwd" : "embed_fwd", s);
  return e;
}

}  // namespace fc
