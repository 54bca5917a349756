// Flash-attention forward, exact mode (fp32 in and out), gfx950.
//
// Behaviour follows the reference forward (src/kernels.jl:131-219 for the
// semantics of O, l and m).  The design is this file's own:
//
//  * one workgroup = 4 waves x 32 queries of one (batch, head), two workgroups
//    per CU; the grid takes the longest query tiles first;
//  * every product runs as six bf16 products of the operands' three parts
//    (attn_exact.hpp); Q stays in registers in parts, K and V tiles of 32 keys
//    are split once per workgroup as they are staged in swizzled LDS;
//  * each wave computes S^T = K Q^T (keys x queries), so a lane owns one query
//    column: the softmax needs one exchange between half-waves per key tile and
//    the probabilities are already the B operand of O^T += V^T P^T;
//  * K and V are single-buffered: while the S products read K, the V tile is
//    split and stored; while the P V products read V, the next K tile is, each
//    loaded a phase ahead (16 registers per thread in flight);
//  * the exponent reference of a row is the maximum of the first tile in which
//    it sees a key; a row whose scores outgrow it by 2^8 moves it and rescales
//    its O and l, in a branch that few tiles take (with a reference that never
//    moved, rows that outgrew it by 2^64 were computed again: queries times 30, 8 x
//    2048 tokens, took 1197 us at H6 D128, now 302);
//  * key tiles outside [min lb, max ub] of the workgroup are never visited,
//    fully visible tiles skip the mask, and waves with no visible key in a
//    tile skip its products.
//
// Bound by the matrix cores and, next to them, by LDS (48 KB of parts read per
// wave and tile for 96 products): 8 x 2048 tokens, causal, H6 D128 in 315 us
// (0.98 PFLOP/s of bf16 products; 474 us with fp32 MFMA), H12 D64 in 304 (525).
// At D = 112 and 128 the kernel spills 79 and 28 registers (five to seven scratch
// accesses per tile; D = 112 240 us for 4 x 2048, H6, 227 with 13 spilled).
#include "attn_exact.hpp"
#include "attn_launch.hpp"

#include <type_traits>

namespace fc {

constexpr int kExactBM = 128;  // queries per workgroup
constexpr int kExactBN = 32;   // keys per tile
constexpr float kExactGrowth = 8.0f;  // log2 units that a score may lie above its row's reference

// S^T of 32 keys from k0 in fp32 MFMA, K straight from global memory, masked.
template <int D>
__device__ inline f32x16 exact_scores(const float* Kb, int64_t kpitch, const f32x8 (&qf)[D / 16], int k0, int T, int l32,
                                      int g, int lb, int ub) {
  using M = Mma<float>;
  f32x16 s = zero16();
  const float* row = Kb + (int64_t)min(k0 + l32, T - 1) * kpitch;
  for (int c = 0; c < D / 16; ++c) s = M::mma(M::load8(row + 16 * c + 8 * g), qf[c], s);
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const int key = k0 + acc_row(r, g);
    if (key < lb || key > ub) s[r] = -INFINITY;
  }
  return s;
}

template <int D>
__global__ __launch_bounds__(kThreads, 2) void attn_fwd_exact_kernel(FwdArgs a) {
  constexpr int BN = kExactBN, KC = D / 16, DB = (D + 31) / 32;
  __shared__ __attribute__((aligned(1024))) char Ks[SplitTile<D>::kBytes];
  __shared__ __attribute__((aligned(1024))) char Vs[SplitTile<D>::kBytes];
  __shared__ int s_bounds[2][kWaves];

  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int g = lane >> 5, l32 = lane & 31;
  const int T = a.T;
  const int n_qt = (T + kExactBM - 1) / kExactBM;
  const GridItem it0 = heavy_first(paired_position(blockIdx.x, (int)gridDim.x, a.cus), a.H * a.B);
  const int qt = n_qt - 1 - it0.rank;  // longest query tiles first, over the whole grid
  int b, h;
  query_row(it0.row, a.B, a.Hkv, a.group, b, h);
  const int kvh = h / a.group;

  const int64_t qpitch = (int64_t)a.H * D, kpitch = (int64_t)a.Hkv * D;
  const float* Qb = static_cast<const float*>(a.Q) + ((int64_t)b * T * a.H + h) * D;
  const float* Kb = static_cast<const float*>(a.K) + ((int64_t)b * T * a.Hkv + kvh) * D;
  const float* Vb = static_cast<const float*>(a.V) + ((int64_t)b * T * a.Hkv + kvh) * D;
  const int32_t* pos = a.pos ? a.pos + (int64_t)b * T : nullptr;

  const int q = qt * kExactBM + wave * 32 + l32;
  const int lb = key_lb(q, T, a.left, pos), ub = key_ub(q, T, a.right);
  const int wlb_min = __builtin_amdgcn_readfirstlane(wave_min32(lb)), wlb_max = __builtin_amdgcn_readfirstlane(wave_max32(lb));
  const int wub_min = __builtin_amdgcn_readfirstlane(wave_min32(ub)), wub_max = __builtin_amdgcn_readfirstlane(wave_max32(ub));
  if (lane == 0) {
    s_bounds[0][wave] = wlb_min;
    s_bounds[1][wave] = wub_max;
  }

  Split8 qf[KC];
  split_rows<D>(Qb + (int64_t)min(q, T - 1) * qpitch, q < T, g, qf);
  FragOffsets<tile_width(D)> fo;
  fo.init(lane);

  f32x16 o[DB];
#pragma unroll
  for (int i = 0; i < DB; ++i) o[i] = zero16();
  float m_ref = -INFINITY, m_true = -INFINITY, l_run = 0.0f;  // of scores times kSplitScale2, probabilities times kSplitScale
  float c2 = a.scale_log2 * kSplitInv2, unscale = kSplitInv;  // of the scores' exponent; of O / l

  __syncthreads();
  int kmin = s_bounds[0][0], kmax = s_bounds[1][0];
#pragma unroll
  for (int w = 1; w < kWaves; ++w) {
    kmin = min(kmin, s_bounds[0][w]);
    kmax = max(kmax, s_bounds[1][w]);
  }
  const int kt0 = __builtin_amdgcn_readfirstlane((kmin / BN) * BN);
  const int ntiles = __builtin_amdgcn_readfirstlane(kmax >= kmin ? (kmax - (kmin / BN) * BN) / BN + 1 : 0);

  SplitStage<D> kst, vst;
  if (ntiles > 0) {
    kst.load(Kb, kpitch, kt0, T, tid);
    vst.load(Vb, kpitch, kt0, T, tid);
    kst.store(Ks, tid);
  }
  __syncthreads();

  for (int it = 0; it < ntiles; ++it) {
    const int kt = kt0 + it * BN;
    const bool more = it + 1 < ntiles;
    const bool active = !(wlb_min > kt + BN - 1 || wub_max < kt);
    f32x16 s = zero16();
    if (active) {
#pragma unroll
      for (int c = 0; c < KC; ++c) s = mma_split(split_nat<D>(Ks, fo, c), qf[c], s);
      vst.store(Vs, tid);
    } else {
      vst.store(Vs, tid);
    }
    if (more) kst.load(Kb, kpitch, kt + BN, T, tid);
    __syncthreads();

    if (active) {
      const bool need_mask = !(wlb_max <= kt && kt + BN - 1 <= wub_min);
      if (need_mask) {
        const int x = kt + 4 * g - lb, y = ub - (kt + 4 * g);
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int c = 8 * (r >> 2) + (r & 3);
          s[r] = (x >= -c) & (y >= c) ? s[r] : -INFINITY;
        }
      }
      float mx = s[0];
#pragma unroll
      for (int r = 1; r < 16; ++r) mx = fmaxf(mx, s[r]);
      mx = fmaxf(mx, __shfl_xor(mx, 32));
      m_true = fmaxf(m_true, mx);
      // A row's first visible key sets the reference (O and l are zero then); one
      // that outgrows it moves it.
      const bool grown = (mx - m_ref) * c2 > kExactGrowth;
      if (__builtin_amdgcn_ballot_w64(grown) != 0) {
        const float f = grown ? __builtin_amdgcn_exp2f((m_ref - mx) * c2) : 1.0f;
        m_ref = grown ? mx : m_ref;
        l_run *= f;
#pragma unroll
        for (int db = 0; db < DB; ++db) o[db] *= f;
      }
      const float ref = m_ref == -INFINITY ? 0.0f : m_ref;
      float psum = 0.0f;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        // The difference first: the largest probability is exactly 1.
        s[r] = __builtin_amdgcn_exp2f((s[r] - ref) * c2) * kSplitScale;
        psum += s[r];
      }
      l_run += psum;
#pragma unroll
      for (int kc = 0; kc < 2; ++kc) {
        const Split8 pf = kc ? split_acc<1>(s) : split_acc<0>(s);
#pragma unroll
        for (int db = 0; db < DB; ++db) o[db] = mma_split(split_tr<D>(Vs, fo, kc, db), pf, o[db]);
      }
    }
    if (more) {
      kst.store(Ks, tid);
      vst.load(Vb, kpitch, kt + BN, T, tid);
    }
    __syncthreads();
  }

  // Values or sums outside the parts' range (attn_exact.hpp).
  const bool outside = !all_finite<D>(o) | (m_true == -INFINITY && lb <= ub);
  if (__builtin_amdgcn_ballot_w64(outside) != 0) {
    // fp32 MFMA from global memory, with the exact maximum first.
    using M = Mma<float>;
    c2 = a.scale_log2;
    unscale = 1.0f;
    f32x8 q32[KC];
#pragma unroll
    for (int c = 0; c < KC; ++c) q32[c] = q < T ? M::load8(Qb + (int64_t)q * qpitch + 16 * c + 8 * g) : M::zero();
    const int klo = (wlb_min / 32) * 32;
    m_true = -INFINITY;
    for (int k0 = klo; k0 <= wub_max; k0 += 32) {
      const f32x16 s = exact_scores<D>(Kb, kpitch, q32, k0, T, l32, g, lb, ub);
#pragma unroll
      for (int r = 0; r < 16; ++r) m_true = fmaxf(m_true, s[r]);
    }
    m_true = fmaxf(m_true, __shfl_xor(m_true, 32));
    m_ref = m_true;
    l_run = 0.0f;
#pragma unroll
    for (int db = 0; db < DB; ++db) o[db] = zero16();
    for (int k0 = klo; k0 <= wub_max; k0 += 32) {
      f32x16 s = exact_scores<D>(Kb, kpitch, q32, k0, T, l32, g, lb, ub);
      const float safe = m_ref == -INFINITY ? 0.0f : m_ref;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        s[r] = __builtin_amdgcn_exp2f((s[r] - safe) * c2);
        l_run += s[r];
      }
#pragma unroll
      for (int kc = 0; kc < 2; ++kc) {
        const f32x8 pf = kc ? M::from_acc<1>(s) : M::from_acc<0>(s);
#pragma unroll
        for (int db = 0; db < DB; ++db) {
          f32x8 vf;
          load_rows_f32<D>(Vb, kpitch, k0 + 16 * kc, T, 32 * db + l32, g, vf);
          o[db] = M::mma(vf, pf, o[db]);
        }
      }
    }
  }

  const float lt = l_run + __shfl_xor(l_run, 32);
  const float inv = lt > 0.0f ? unscale / lt : 0.0f;
  if (q < T) {
    const int64_t orow = ((int64_t)b * T + q) * a.H + h;
#pragma unroll
    for (int db = 0; db < DB; ++db) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int d0 = 32 * db + 8 * j + 4 * g;
        if (d0 < D) {
          f32x4 v;
#pragma unroll
          for (int t = 0; t < 4; ++t) v[t] = o[db][4 * j + t] * inv;
          store4(static_cast<float*>(a.O) + orow * D + d0, v, false);
        }
      }
    }
    if (g == 0) {
      const int64_t si = ((int64_t)b * a.H + h) * T + q;
      const bool any = m_true != -INFINITY;
      a.l[si] = any ? lt * unscale * __builtin_amdgcn_exp2f((m_ref - m_true) * c2) : lt * unscale;
      a.m[si] = any ? m_true * c2 * kLn2 : -kFltMax;
    }
  }
}

template <int D>
static hipError_t launch_fwd_exact(const Problem& p, const FwdArgs& a, hipStream_t s) {
  const int n_qt = (p.T + kExactBM - 1) / kExactBM;
  const dim3 grid(n_qt * p.H * p.B), block(kThreads);
  const ProfileMark mk = profile_begin(s);
  hipLaunchKernelGGL((attn_fwd_exact_kernel<D>), grid, block, 0, s, a);
  const hipError_t e = hipGetLastError();
  profile_end(mk, "attn_fwd_f32", s);
  return e;
}

hipError_t launch_fwd(const Problem& p, const FwdArgs& a, hipStream_t s) {
  if (p.bf16) return launch_fwd_fast(p, a, s);
  switch (p.D) {
    case 16: return launch_fwd_exact<16>(p, a, s);
    case 32: return launch_fwd_exact<32>(p, a, s);
    case 48: return launch_fwd_exact<48>(p, a, s);
    case 64: return launch_fwd_exact<64>(p, a, s);
    case 80: return launch_fwd_exact<80>(p, a, s);
    case 96: return launch_fwd_exact<96>(p, a, s);
    case 112: return launch_fwd_exact<112>(p, a, s);
    case 128: return launch_fwd_exact<128>(p, a, s);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace fc
