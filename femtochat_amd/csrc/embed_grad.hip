// Embedding gradient into a fresh table (gfx950): every column of dweights
// written once, the sum of its tokens' dy rows or zeros, without atomics,
// workspace or a clearing pass (reference: src/kernels.jl:8-14 into a zeroed
// δ; ext/FemtoChatCUDAExt.jl:78-94 adds with one atomic per element).
//
// A workgroup owns the table columns id = group + slot * groups (strided, so
// that the frequent ids of a text, which are neighbours, fall to different
// workgroups) and kCols of their D values.  It scans all tokens (they come
// from L2) and keeps its own in token order, orders them by column in LDS,
// and its waves take equal parts of that list: each sums the rows of a run of
// equal ids in token order, and a run cut by a part's edge is put together
// from the parts through LDS.  The sum's order follows from the tokens alone,
// so the result is the same on every call.
//
// HBM-bound: the table is written once and dy read once.  8192 tokens, table
// 32768 x 512, bf16 dy: 31 us with a text's id frequencies (the fill and the
// atomics it replaces: 91), 22 with uniform ids (67; the table alone is 10 us
// at 6.5 TB/s), 264 with one id for all tokens (952).  Small: 1000 tokens,
// 8192 x 256: 9.4 us (11.3).
#include "attn_launch.hpp"
#include "attn_device.hpp"
#include "embed_rule.hpp"

#include <hip/hip_runtime.h>

#include <cstdint>

namespace fc {
namespace {

constexpr int kEgThreads = 512, kEgWaves = kEgThreads / 64;
constexpr int kEgPer = 8;                        // tokens a thread looks at per scan step
constexpr int kEgStep = kEgThreads * kEgPer;     // tokens per scan step
constexpr int kEgCap = kEgStep + 2048;           // list entries: a full step beyond 2048 kept ones
constexpr int kEgSegs = kEgThreads / kEgSlots;   // list segments counted side by side
constexpr int kEgRows = 8;                       // rows in flight per wave

// A lane's four values of a row as loaded (lanes past the row's end read its
// last values again, without a branch; eg_store leaves them out).
template <bool kVec, typename Y>
struct EgRow {
  typedef Y Y4 __attribute__((ext_vector_type(4)));
  Y4 raw;
  __device__ inline void load(const Y* row, int d, int D, int lane) {
    if constexpr (kVec) {
      raw = *reinterpret_cast<const Y4*>(row + min(d + 4 * lane, D - 4));
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) raw[e] = row[min(d + lane + 64 * e, D - 1)];
    }
  }
  __device__ inline f32x4 value() const { return __builtin_convertvector(raw, f32x4); }
};

// add: the column already holds the sum of earlier tokens.
template <bool kVec>
__device__ inline void eg_store(float* col, int d, int D, int lane, f32x4 v, bool add) {
  if constexpr (kVec) {
    if (d + 4 * lane < D) {
      f32x4* p = reinterpret_cast<f32x4*>(col + d + 4 * lane);
      if (add) *p = *p + v;
      else __builtin_nontemporal_store(v, p);
    }
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int i = d + lane + 64 * e;
      if (i < D) col[i] = add ? col[i] + v[e] : v[e];
    }
  }
}

template <bool kVec, typename Y>
__global__ __launch_bounds__(kEgThreads) void embed_grad_kernel(EmbedArgs a, int groups, FastDiv by_groups) {
  __shared__ uint32_t s_tok[kEgCap];     // the group's tokens, in token order
  __shared__ __attribute__((aligned(16))) uint8_t s_slot[kEgCap + 16];  // and 16 past the last that name no slot
  __shared__ uint16_t s_sorted[kEgCap];  // list positions ordered by (slot, token)
  __shared__ uint32_t s_count[kEgSlots * kEgSegs];  // [slot][segment], then exclusive sums
  __shared__ uint32_t s_wave[kEgPer * kEgWaves + 1];
  __shared__ uint32_t s_done[kEgSlots / 32];  // slots whose column has been written
  __shared__ uint32_t s_seen[kEgSlots / 32];  // those and the slots in the list
  __shared__ __attribute__((aligned(16))) f32x4 s_part[kEgWaves][2][64];
  __shared__ int s_edge[kEgWaves][2];  // slot of the partial sum at each end of a wave's part, or -1

  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int group = blockIdx.x % groups, d0 = (int)(blockIdx.x / groups) * kEgCols;
  const int D = a.D;
  const int slots = (a.vocab - group + groups - 1) / groups;  // ids group, group + groups, ... below vocab
  const Y* dy = static_cast<const Y*>(a.dy);
  auto column = [&](int slot) { return a.dweights + (int64_t)(group + (int64_t)slot * groups) * D; };

  if (tid < kEgSlots / 32) s_done[tid] = s_seen[tid] = 0;
  int count = 0;  // list entries, the same on every thread
  auto mark = [&](uint32_t* bits) {
    for (int i = tid; i < count; i += kEgThreads) atomicOr(&bits[s_slot[i] >> 5], 1u << (s_slot[i] & 31));
  };

  // Sums the listed rows into their columns and empties the list.
  auto flush = [&]() {
    // Stable counting sort by slot: thread (slot, segment) counts and then
    // places its slot's entries of one quarter of the list.  The lanes of a
    // wave read the same entries (LDS broadcasts).
    const int seg = tid / kEgSlots, slot = tid % kEgSlots;
    const int per = ((count + kEgSegs - 1) / kEgSegs + 15) & ~15, from = min(seg * per, count), to = min(from + per, count);
    if (tid < 16) s_slot[count + tid] = 255;
    __syncthreads();
    // f(i) for the entries of this thread's slot, sixteen per LDS read.
    auto entries = [&](auto f) {
      for (int i0 = from; i0 < to; i0 += 16) {
        const uint4 w = *reinterpret_cast<const uint4*>(s_slot + i0);
        const uint32_t word[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
        for (int e = 0; e < 16; ++e)
          if ((int)((word[e >> 2] >> (8 * (e & 3))) & 255u) == slot) f(i0 + e);
      }
    };
    uint32_t n = 0;
    entries([&](int) { ++n; });
    s_count[slot * kEgSegs + seg] = n;
    __syncthreads();
    if (wave == 0) {  // exclusive sums of the 512 counts, eight per lane
      uint32_t c[8], sum = 0;
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        c[k] = sum;
        sum += s_count[8 * lane + k];
      }
      uint32_t incl = sum;
#pragma unroll
      for (int o = 1; o < 64; o <<= 1) {
        const uint32_t u = __shfl_up(incl, o);
        if (lane >= o) incl += u;
      }
#pragma unroll
      for (int k = 0; k < 8; ++k) s_count[8 * lane + k] = c[k] + incl - sum;
    }
    __syncthreads();
    uint32_t at = s_count[slot * kEgSegs + seg];
    entries([&](int i) { s_sorted[at++] = (uint16_t)i; });
    __syncthreads();

    const int lo = (int)((int64_t)count * wave / kEgWaves), hi = (int)((int64_t)count * (wave + 1) / kEgWaves);
    auto slot_of = [&](int i) { return __builtin_amdgcn_readfirstlane((int)s_slot[s_sorted[i]]); };
    const bool head_cut = lo > 0 && lo < hi && slot_of(lo - 1) == slot_of(lo);
    const bool tail_cut = hi < count && lo < hi && slot_of(hi) == slot_of(hi - 1);
    if (lane < 2) s_edge[wave][lane] = -1;
    f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
    int cur = lo < hi ? slot_of(lo) : -1;
    bool first = true;  // cur is the part's first run
    auto done = [&](int s) { return (s_done[s >> 5] >> (s & 31)) & 1; };
    auto finish = [&](bool last) {
      const bool cut_front = first && head_cut, cut_back = last && tail_cut;
      if (cut_front || cut_back) {  // a run cut at both ends counts as the part's front one
        const int end = cut_front ? 0 : 1;
        s_part[wave][end][lane] = acc;
        if (lane == 0) s_edge[wave][end] = cur;
      } else {
        eg_store<kVec>(column(cur), d0, D, lane, acc, done(cur));
      }
    };
    for (int b0 = lo; b0 < hi; b0 += 64) {  // 64 entries at a time, one per lane
      const int mine = s_sorted[min(b0 + lane, hi - 1)];
      const uint32_t my_tok = s_tok[mine];
      const int my_slot = s_slot[mine];
      const int b1 = min(b0 + 64, hi);
      for (int i0 = b0; i0 < b1; i0 += kEgRows) {
        EgRow<kVec, Y> row[kEgRows];
#pragma unroll
        for (int k = 0; k < kEgRows; ++k) {
          const uint32_t t = (uint32_t)__builtin_amdgcn_readlane((int)my_tok, min(i0 + k, b1 - 1) - b0);
          row[k].load(dy + (int64_t)t * D, d0, D, lane);
        }
#pragma unroll
        for (int k = 0; k < kEgRows; ++k) {
          if (i0 + k >= b1) break;
          const int s = __builtin_amdgcn_readlane(my_slot, i0 + k - b0);
          if (s != cur) {
            finish(false);
            cur = s;
            first = false;
            acc = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
          }
          acc += row[k].value();
        }
      }
    }
    if (lo < hi) finish(true);
    __syncthreads();
    // A run cut by parts: the wave that holds its beginning adds the fronts of
    // the parts after it, up to the one in which it ends.
    if (tail_cut && !(first && head_cut)) {
      f32x4 sum = s_part[wave][1][lane];
      for (int w = wave + 1; w < kEgWaves; ++w) {
        if (s_edge[w][0] != cur) {
          if ((int)((int64_t)count * w / kEgWaves) == (int)((int64_t)count * (w + 1) / kEgWaves)) continue;  // empty part
          break;
        }
        sum += s_part[w][0][lane];
      }
      eg_store<kVec>(column(cur), d0, D, lane, sum, done(cur));
    }
    __syncthreads();
    mark(s_done);
    __syncthreads();
    count = 0;
  };

  for (int64_t base = 0; base < a.N; base += kEgStep) {
    int slot[kEgPer];
#pragma unroll
    for (int k = 0; k < kEgPer; ++k) {
      const int64_t t = base + k * kEgThreads + tid;
      const int64_t at = t < a.N ? t : a.N - 1;
      const int64_t id = (a.index_type == 1 ? static_cast<const int64_t*>(a.tokens)[at]
                                            : (int64_t) static_cast<const int32_t*>(a.tokens)[at]) - a.index_base;
      const bool in = t < a.N && id >= 0 && id < a.vocab;  // an id outside the table adds nothing
      const uint32_t q = in ? divide((uint32_t)id, by_groups) : 0u;
      slot[k] = in && (uint32_t)id - q * (uint32_t)groups == (uint32_t)group ? (int)q : -1;
    }
    uint64_t mine[kEgPer];
#pragma unroll
    for (int k = 0; k < kEgPer; ++k) {
      mine[k] = __ballot(slot[k] >= 0);
      if (lane == 0) s_wave[k * kEgWaves + wave] = (uint32_t)__popcll(mine[k]);
    }
    __syncthreads();
    if (wave == 0) {  // exclusive sums of the kEgPer * kEgWaves = 64 counts
      static_assert(kEgPer * kEgWaves == 64, "one count per lane");
      const uint32_t c = s_wave[lane];
      uint32_t incl = c;
#pragma unroll
      for (int o = 1; o < 64; o <<= 1) {
        const uint32_t u = __shfl_up(incl, o);
        if (lane >= o) incl += u;
      }
      s_wave[lane] = incl - c;
      if (lane == 63) s_wave[64] = incl;
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kEgPer; ++k) {
      if (slot[k] >= 0) {
        const int at = count + (int)s_wave[k * kEgWaves + wave] + __popcll(mine[k] & (((uint64_t)1 << lane) - 1));
        s_tok[at] = (uint32_t)(base + k * kEgThreads + tid);
        s_slot[at] = (uint8_t)slot[k];
      }
    }
    count += (int)s_wave[64];
    __syncthreads();
    if (count > kEgCap - kEgStep) flush();
  }
  // Zeros into the columns no token names, ahead of the last sums (whose loads
  // they overlap).
  if (tid < kEgSlots / 32) s_seen[tid] = s_done[tid];
  __syncthreads();
  mark(s_seen);
  __syncthreads();
  for (int s = wave; s < slots; s += kEgWaves)
    if (!((s_seen[s >> 5] >> (s & 31)) & 1)) eg_store<kVec>(column(s), d0, D, lane, f32x4{0.0f, 0.0f, 0.0f, 0.0f}, false);
  if (count > 0) flush();
}

}  // namespace

// Token indices are 32-bit list entries.
bool embed_grad_full_pays(const EmbedArgs& a) {
  return embed_one_kernel_pays(a.N, a.vocab, a.D) && a.N <= UINT32_MAX &&
         (int64_t)embed_groups(a.vocab) * ((a.D + kEgCols - 1) / kEgCols) <= INT32_MAX / kEgThreads;
}

hipError_t launch_embed_grad_full(const EmbedArgs& a, bool bf16_dy, hipStream_t s) {
  if (!embed_grad_full_pays(a)) return hipErrorInvalidValue;
  const int groups = embed_groups(a.vocab);
  const int64_t blocks = (int64_t)groups * ((a.D + kEgCols - 1) / kEgCols);
  const uintptr_t dy = reinterpret_cast<uintptr_t>(a.dy);
  const bool vec = a.D % 4 == 0 && (reinterpret_cast<uintptr_t>(a.dweights) & 15) == 0 && (dy & (bf16_dy ? 7 : 15)) == 0;
  const dim3 grid((unsigned)blocks), block(kEgThreads);
  const FastDiv by = fast_div((uint32_t)groups);
  const ProfileMark mk = profile_begin(s);
  if (bf16_dy) {
    if (vec) hipLaunchKernelGGL((embed_grad_kernel<true, bf16>), grid, block, 0, s, a, groups, by);
    else hipLaunchKernelGGL((embed_grad_kernel<false, bf16>), grid, block, 0, s, a, groups, by);
  } else {
    if (vec) hipLaunchKernelGGL((embed_grad_kernel<true, float>), grid, block, 0, s, a, groups, by);
    else hipLaunchKernelGGL((embed_grad_kernel<false, float>), grid, block, 0, s, a, groups, by);
  }
  const hipError_t e = hipGetLastError();
  profile_end(mk, "embed_grad_full", s);
  return e;
}

}  // namespace fc
