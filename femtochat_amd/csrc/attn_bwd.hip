// Flash-attention backward for gfx950.
//
// Semantics follow the reference backward (src/kernels.jl:287-379:
// P = exp(S/sqrt(D) - m) / max(l, eps), Delta = rowsum(dO.O),
// dS = P (dP - Delta), dQ += K dS / sqrt(D), dK += Q dS^T / sqrt(D),
// dV += dO P^T) and, for the fast mode, ext/FemtoChatCUDAExt.jl:1829-2068
// (P and dS rounded to the input format before their second product, a query
// with a single visible key gets dS = 0, fp32 accumulation, optional add into
// the caller's gradients before the one final rounding).
//
// Three kernels, all deterministic (no atomics); the last two here are the
// exact-mode ones:
//  * attn_bwd_pre  : Delta and the base-2 log-sum-exp per query, and a bf16
//                    copy of dO when the caller hands fp32 dO in fast mode;
//  * attn_bwd_dkdv : one workgroup per (key tile of 128, KV head, batch); the
//                    4 waves own 32 keys each and loop over every query head of
//                    the GQA group and every query tile that can see the keys,
//                    so the group's contributions to dK/dV are summed in
//                    registers;
//  * attn_bwd_dq   : one workgroup per (query tile of 128, head, batch); it
//                    recomputes S^T and dP^T with the query as the lane index
//                    so dS^T is directly the B operand of dQ^T += K^T dS^T.
#include "attn_exact.hpp"
#include "attn_launch.hpp"

#include <type_traits>

namespace fc {

// ---------------------------------------------------------------------------
// Preprocess: Delta = sum_d dO*O (fp32), lse2 = m*log2(e) + log2(max(l, eps)).
template <int D, typename TO, typename TD>
__global__ __launch_bounds__(kThreads) void attn_bwd_pre_kernel(PreArgs a) {
  constexpr int LPQ = tile_width(D) / 8;  // lanes per query, 8 elements each (idle past D)
  constexpr int QPB = kThreads / LPQ;   // queries per block
  const int tid = threadIdx.x;
  const int sub = tid % LPQ;
  const int64_t idx = (int64_t)blockIdx.x * QPB + tid / LPQ;  // (b, t, h) order
  const int64_t n = (int64_t)a.B * a.T * a.H;
  if (a.queue != nullptr && blockIdx.x == 0 && tid < kXcds) a.queue[tid] = 0;
  float acc = 0.0f;
  if (idx < n && 8 * sub < D) {
    const TD* dO = static_cast<const TD*>(a.dO) + idx * D + 8 * sub;
    const TO* O = static_cast<const TO*>(a.O) + idx * D + 8 * sub;
    float x[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      x[e] = to_f32(dO[e]);
      acc += x[e] * to_f32(O[e]);
    }
    if (a.dO16 != nullptr) {
      bf16* out = static_cast<bf16*>(a.dO16) + idx * D + 8 * sub;
#pragma unroll
      for (int e = 0; e < 8; ++e) out[e] = static_cast<bf16>(x[e]);
    }
  }
#pragma unroll
  for (int o = LPQ / 2; o > 0; o >>= 1) acc += __shfl_xor(acc, o);
  if (idx < n && sub == 0) {
    const int h = (int)(idx % a.H);
    const int64_t bt = idx / a.H;
    const int t = (int)(bt % a.T), b = (int)(bt / a.T);
    const int64_t si = ((int64_t)b * a.H + h) * a.T + t;
    a.delta[si] = acc;
    a.lse2[si] = a.m[si] * kLog2e + __builtin_amdgcn_logf(fmaxf(a.l[si], kFltEps));
  }
}

// Per 32-query chunk (min, max) of the document-aware key lower bound (a
// query at or beyond T counts as T).  One lane per query, so a half-wave
// reads one chunk's 32 positions in one coalesced access and reduces them.
__global__ __launch_bounds__(kThreads) void attn_bounds_kernel(BoundsArgs a) {
  const int nc = (a.T + 31) / 32;
  const int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x;
  const int64_t chunk = i >> 5;
  const bool live = chunk < (int64_t)nc * a.B;  // uniform over each half-wave
  const int b = live ? (int)(chunk / nc) : 0;
  const int q = live ? 32 * (int)(chunk - (int64_t)b * nc) + (int)(i & 31) : a.T;
  const int lb = key_lb(q, a.T, a.left, a.pos + (int64_t)b * a.T);
  const int lo = wave_min32(lb), hi = wave_max32(lb);
  if (live && (i & 31) == 0) {
    a.chunk_lb[2 * chunk] = lo;
    a.chunk_lb[2 * chunk + 1] = hi;
  }
}

// Work order of the fast kernels' tiles with positions, in one workgroup.
// The smallest key lower bound of every 128-query tile (from the chunk
// bounds) goes to LDS; then the work of each item of 128 rows, in steps:
//  * query tile [q0, q1] (forward and dQ): the 64-key tiles from the one
//    holding its smallest lower bound up to the one holding key_ub(q1);
//  * key tile [k0, k1] (dK/dV): the 128-query tiles between k0 - right and
//    k1 + left whose smallest lower bound is at most k1, which are the
//    tiles the dK/dV kernel visits;
// and finally each item's rank: the items of more work, plus the items of
// equal work and lower index.  order[rank] = item.  The inner loops read
// LDS in runs of 8 with no exit inside a run, so the reads of a run are in
// flight together.
constexpr int kOrderThreads = 1024;
constexpr int kOrderRun = 8;

__global__ __launch_bounds__(kOrderThreads) void attn_order_kernel(OrderArgs a) {
  static_assert(kOrderKStep == kOrderRows, "a dK/dV step is one tabulated query tile");
  __shared__ int s_lb[kOrderMaxItems + kOrderRun];
  __shared__ __attribute__((aligned(16))) int s_work[kOrderMaxItems + kOrderRun];
  const int tid = threadIdx.x, T = a.T;
  const int nc = (T + 31) / 32, n128 = (T + kOrderRows - 1) / kOrderRows;
  const int items = a.B * n128;
  constexpr int kChunks = kOrderRows / 32;
  for (int i = tid; i < items; i += kOrderThreads) {
    const int b = i / n128, t = i - b * n128;
    const int32_t* cb = a.chunk_lb + (int64_t)b * nc * 2;
    int lo = T;
#pragma unroll
    for (int c = 0; c < kChunks; ++c) lo = min(lo, cb[2 * min(kChunks * t + c, nc - 1)]);  // loads without a branch
    s_lb[i] = lo;
  }
  // Padding after the last item: never counted (ranks) or masked (key steps).
  if (tid < kOrderRun) s_work[items + tid] = INT_MIN;

  // sub lanes (a power of two up to a wave) count one item's rank together,
  // each over every sub-th run of kOrderRun items, and add their counts
  // with shuffles.
  int sub = 1;
  while (sub < kWave && sub * 2 * items <= kOrderThreads) sub *= 2;
  const int per = kOrderThreads / sub, part = tid & (sub - 1);
  auto rank_into = [&](int32_t* order) {
    for (int i0 = 0; i0 < items; i0 += per) {  // the same trip count on every lane
      const int i = i0 + tid / sub;
      const bool live = i < items;
      const int w = s_work[live ? i : 0];
      int r = 0;
      for (int j0 = kOrderRun * part; j0 < items; j0 += kOrderRun * sub) {
        int v[kOrderRun];
#pragma unroll
        for (int e = 0; e < kOrderRun; ++e) v[e] = s_work[j0 + e];
#pragma unroll
        for (int e = 0; e < kOrderRun; ++e) r += (v[e] > w || (v[e] == w && j0 + e < i)) ? 1 : 0;
      }
      for (int o = 1; o < sub; o <<= 1) r += __shfl_xor(r, o);
      if (live && part == 0) order[r] = i;
    }
  };
  __syncthreads();
  if (a.qorder != nullptr) {
    for (int i = tid; i < items; i += kOrderThreads) {
      const int t = i % n128;
      const int kmin = s_lb[i];
      const int kmax = key_ub(min(t * kOrderRows + kOrderRows - 1, T - 1), T, a.right);
      s_work[i] = kmax >= kmin ? (kmax - (kmin / kOrderTile) * kOrderTile) / kOrderTile + 1 : 0;
    }
    __syncthreads();
    rank_into(a.qorder);
    __syncthreads();
  }
  if (a.korder != nullptr) {
    for (int i = tid; i < items; i += kOrderThreads) {
      const int b = i / n128, t = i - b * n128;
      const int k0 = t * kOrderRows, k1 = min(k0 + kOrderRows, T) - 1;
      const int qlo = max(0, k0 - a.right), qhi = min(T - 1, k1 + a.left);
      int n = 0;
      if (qhi >= qlo) {
        const int* row = s_lb + b * n128;
        const int ulast = qhi / kOrderKStep;
        for (int u0 = qlo / kOrderKStep; u0 <= ulast; u0 += kOrderRun) {
          int v[kOrderRun];
#pragma unroll
          for (int e = 0; e < kOrderRun; ++e) v[e] = row[u0 + e];  // within the padded table
#pragma unroll
          for (int e = 0; e < kOrderRun; ++e) n += (u0 + e <= ulast && v[e] <= k1) ? 1 : 0;
        }
      }
      s_work[i] = n;
    }
    __syncthreads();
    rank_into(a.korder);
  }
}

// ---------------------------------------------------------------------------
// dK and dV, exact mode (products in bf16 parts, attn_exact.hpp): 128 keys of
// one (batch, KV head) per workgroup, 32 per wave with K and V resident as B
// operands, their first two parts in registers and the third in LDS (all three
// in registers spilled 69-218 of them and took 0.90-2.1 ms at D = 128); the
// loop runs over the group's query heads and the 32-query tiles that can see
// the keys, whose Q and dO are split once per workgroup into swizzled LDS.
// At one wave per SIMD (D = 128) the LDS reads bound it next to the products:
// a wave reads 112 KB of parts per tile for 192 products.  8 x 2048 tokens,
// causal, H6 D128: 677 us (fp32 MFMA 1103), H12 D64: 558 (1190).
constexpr int kExactBK = 128;  // keys per workgroup
constexpr int kExactBT = 32;   // rows per staged tile (queries here, keys in dQ)

template <int D>
__global__ __launch_bounds__(kThreads, D <= 64 ? 2 : 1) void attn_bwd_dkdv_exact_kernel(BwdArgs a) {
  constexpr int BQ = kExactBT, KC = D / 16, DB = (D + 31) / 32;
  constexpr int kTile = SplitTile<D>::kBytes;
  __shared__ __attribute__((aligned(1024))) char Qbuf[2][kTile];
  __shared__ __attribute__((aligned(1024))) char Os[kTile];  // dO
  __shared__ __attribute__((aligned(1024))) bf16x8 s_low[kWaves][2][KC][kWave];  // third parts of K and V, per lane
  __shared__ __attribute__((aligned(16))) float s_lse[2][BQ];
  __shared__ __attribute__((aligned(16))) float s_delta[2][BQ];
  __shared__ __attribute__((aligned(16))) int s_lb[2][BQ];
  __shared__ int s_outside;

  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int g = lane >> 5, l32 = lane & 31;
  const int T = a.T;
  // Key tiles that the most query tiles can see come first, over the whole grid.
  const GridItem it0 = heavy_first(blockIdx.x, a.Hkv * a.B);
  const int b = it0.row / a.Hkv, kvh = it0.row - b * a.Hkv;
  const int k0 = it0.rank * kExactBK;
  const int k1 = min(k0 + kExactBK, T) - 1;
  const int kw0 = k0 + 32 * __builtin_amdgcn_readfirstlane(wave), kw1 = kw0 + 31;
  const int key = kw0 + l32;

  const int64_t qpitch = (int64_t)a.H * D, kpitch = (int64_t)a.Hkv * D;
  const float* Kb = static_cast<const float*>(a.K) + ((int64_t)b * T * a.Hkv + kvh) * D;
  const float* Vb = static_cast<const float*>(a.V) + ((int64_t)b * T * a.Hkv + kvh) * D;
  const int32_t* pos = a.pos ? a.pos + (int64_t)b * T : nullptr;
  const int nchunks = (T + 31) / 32;
  const int32_t* clb = a.chunk_lb ? a.chunk_lb + (int64_t)b * nchunks * 2 : nullptr;
  if (tid == 0) s_outside = 0;

  bf16x8 kf[KC][2], vf[KC][2];
  const int64_t krow = (int64_t)min(key, T - 1) * kpitch;
  bool outside = false;  // a row's log-sum-exp is below kSplitLse
  {
    Split8 f[KC];
    split_rows<D>(Kb + krow, key < T, g, f);
#pragma unroll
    for (int c = 0; c < KC; ++c) {
      kf[c][0] = f[c].part[0];
      kf[c][1] = f[c].part[1];
      s_low[wave][0][c][lane] = f[c].part[2];
    }
    split_rows<D>(Vb + krow, key < T, g, f);
#pragma unroll
    for (int c = 0; c < KC; ++c) {
      vf[c][0] = f[c].part[0];
      vf[c][1] = f[c].part[1];
      s_low[wave][1][c][lane] = f[c].part[2];
    }
  }
  FragOffsets<tile_width(D)> fo;
  fo.init(lane);
  f32x16 dk[DB], dv[DB];
#pragma unroll
  for (int i = 0; i < DB; ++i) {
    dk[i] = zero16();
    dv[i] = zero16();
  }

  // Query tiles that can see [k0, k1]: q in [k0 - right, k1 + left].
  const int qlo = max(0, k0 - a.right);
  const int qhi = min(T - 1, k1 + a.left);
  const int qt_begin = qlo / BQ;
  const int qt_end = qhi >= qlo ? qhi / BQ : qt_begin - 1;  // inclusive
  const int n_qt_tiles = qt_end - qt_begin + 1;             // per head
  const int total_steps = n_qt_tiles > 0 ? n_qt_tiles * a.group : 0;

  // A step is (head in group, query tile); tiles no document can see are
  // skipped when positions are given (a tile is one chunk of the bounds).
  auto next_step = [&](int st) -> int {
    while (clb != nullptr && st < total_steps && clb[2 * (qt_begin + st % n_qt_tiles)] > k1) ++st;
    return st;
  };

  SplitStage<D> qst, ost;
  float r_lse, r_delta;
  int r_lb;
  auto head_of = [&](int st) { return ((int64_t)b * T * a.H + kvh * a.group + st / n_qt_tiles) * D; };
  auto q0_of = [&](int st) { return (qt_begin + st % n_qt_tiles) * BQ; };
  auto load_q = [&](int st) {
    qst.load(static_cast<const float*>(a.Q) + head_of(st), qpitch, q0_of(st), T, tid);
    const int q = q0_of(st) + (tid & (BQ - 1));
    const int64_t si = ((int64_t)b * a.H + kvh * a.group + st / n_qt_tiles) * T + min(q, T - 1);
    r_lse = q < T ? a.lse2[si] : INFINITY;
    r_delta = q < T ? a.delta[si] : 0.0f;
    r_lb = key_lb(q, T, a.left, pos);
  };
  auto load_o = [&](int st) { ost.load(static_cast<const float*>(a.dO) + head_of(st), qpitch, q0_of(st), T, tid); };
  auto store_rows = [&](int buf) {
    if (tid < BQ) {
      s_lse[buf][tid] = r_lse;
      s_delta[buf][tid] = r_delta * kSplitScale2;
      s_lb[buf][tid] = r_lb;
      outside |= r_lse < kSplitLse && r_lse != -INFINITY;  // (-inf: a row that sees no key)
    }
  };

  // P of a tile (times pscale) in place of the scores, dS in place of dP.
  auto softmax = [&](auto need_mask, f32x16& s, f32x16& dp, int q0, int buf, float c2, float pscale)
      __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int i0 = 8 * j + 4 * g;
      const f32x4 L = *reinterpret_cast<const f32x4*>(&s_lse[buf][i0]);
      const f32x4 Dl = *reinterpret_cast<const f32x4*>(&s_delta[buf][i0]);
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const int r = 4 * j + t;
        float p = __builtin_amdgcn_exp2f(__builtin_fmaf(s[r], c2, -L[t]));
        float ds = p * (dp[r] - Dl[t]);
        p *= pscale;
        if constexpr (decltype(need_mask)::value) {
          const int lbq = s_lb[buf][i0 + t], ubq = key_ub(q0 + i0 + t, T, a.right);
          const bool vis = (key >= lbq) & (key <= ubq);
          p = vis ? p : 0.0f;
          ds = vis & (ubq > lbq) ? ds : 0.0f;
        }
        s[r] = p;
        dp[r] = ds;
      }
    }
  };

  // The tile's rows (staged) times this wave's keys (kf or vf), even and odd
  // chunks summed apart.
  auto product = [&](const char* tile, const bf16x8 (&f)[KC][2], int which) __attribute__((always_inline)) {
    auto keys = [&](int c) { return Split8{{f[c][0], f[c][1], s_low[wave][which][c][lane]}}; };
    f32x16 even = zero16(), odd = zero16();
#pragma unroll
    for (int c = 0; c + 1 < KC; c += 2)
      mma_split_pair(split_nat<D>(tile, fo, c), keys(c), even, split_nat<D>(tile, fo, c + 1), keys(c + 1), odd);
    if constexpr (KC % 2 == 1) even = mma_split(split_nat<D>(tile, fo, KC - 1), keys(KC - 1), even);
    if constexpr (KC == 1) return even;
    return even + odd;
  };

  const float c2 = a.scale_log2 * kSplitInv2;
  int st = next_step(0), st_next = total_steps;
  if (st < total_steps) {
    load_q(st);
    load_o(st);
    qst.store(Qbuf[0], tid);
    store_rows(0);
    st_next = next_step(st + 1);
  }
  __syncthreads();
  int buf = 0;
  // A step: S while this tile's dO is split and stored (all waves are done with
  // the previous one), a barrier, then dP, P and dS, dV and dK while the next
  // tile's Q is.  With no next tile, rows of the slice go to the idle buffer.
  while (st < total_steps) {
    const bool more = st_next < total_steps;
    const int q0 = q0_of(st);
    const char* Qs = Qbuf[buf];
    // The tile's bounds on its queries' key ranges (queries >= T have lb = T,
    // ub = -1); without positions both are monotone in the query.
    int lbmin, lbmax;
    if (clb != nullptr) {
      lbmin = clb[2 * (q0 / BQ)];
      lbmax = clb[2 * (q0 / BQ) + 1];
    } else {
      lbmin = key_lb(q0, T, a.left, nullptr);
      lbmax = key_lb(q0 + BQ - 1, T, a.left, nullptr);
    }
    const int ubmin = q0 + BQ - 1 >= T ? -1 : key_ub(q0, T, a.right);
    const int ubmax = key_ub(min(q0 + BQ - 1, T - 1), T, a.right);
    const bool active = !(lbmin > kw1 || ubmax < kw0);
    f32x16 s = zero16();
    if (active) {
      s = product(Qs, kf, 0);
      ost.store(Os, tid);
    } else {
      ost.store(Os, tid);
    }
    load_q(more ? st_next : st);
    load_o(more ? st_next : st);
    __syncthreads();
    if (active) {
      f32x16 dp = product(Os, vf, 1);
      if (!(lbmax <= kw0 && kw1 <= ubmin)) softmax(std::true_type{}, s, dp, q0, buf, c2, kSplitScale);
      else softmax(std::false_type{}, s, dp, q0, buf, c2, kSplitScale);
      // dV += P^T dO, dK += dS^T Q  (k = query, accumulator order)
#pragma unroll
      for (int kc = 0; kc < 2; ++kc) {
        const Split8 pf = kc ? split_acc<1>(s) : split_acc<0>(s);
        const Split8 sf = kc ? split_acc<1>(dp) : split_acc<0>(dp);
#pragma unroll
        for (int db = 0; db < DB; ++db)
          mma_split_pair(pf, split_tr<D>(Os, fo, kc, db), dv[db], sf, split_tr<D>(Qs, fo, kc, db), dk[db]);
      }
      qst.store(Qbuf[buf ^ 1], tid);
    } else {
      qst.store(Qbuf[buf ^ 1], tid);
    }
    store_rows(buf ^ 1);
    st = st_next;
    if (more) st_next = next_step(st + 1);
    buf ^= 1;
    __syncthreads();
  }

  // (columns past the head dim, d >= D, come from LDS that nothing wrote)
#pragma unroll
  for (int db = 0; db < DB; ++db) outside |= (32 * db + l32 < D) & !(all_finite(dk[db]) & all_finite(dv[db]));
  float kscale = a.scale * kSplitInv3, vscale = kSplitInv2;  // dK holds dS (2^32) times Q, dV holds P (2^16) times dO
  if (__builtin_amdgcn_ballot_w64(outside) != 0 && lane == 0) s_outside = 1;
  __syncthreads();
  if (s_outside != 0) {
    // fp32 MFMA from global memory.
    using M = Mma<float>;
    kscale = a.scale;
    vscale = 1.0f;
#pragma unroll
    for (int i = 0; i < DB; ++i) {
      dk[i] = zero16();
      dv[i] = zero16();
    }
    for (int step = next_step(0); step < total_steps; step = next_step(step + 1)) {
      const int h = kvh * a.group + step / n_qt_tiles;
      const int q0 = (qt_begin + step % n_qt_tiles) * BQ;
      const float* Qb = static_cast<const float*>(a.Q) + ((int64_t)b * T * a.H + h) * D;
      const float* Ob = static_cast<const float*>(a.dO) + ((int64_t)b * T * a.H + h) * D;
      __syncthreads();
      if (tid < BQ) {
        const int q = q0 + tid;
        const int64_t si = ((int64_t)b * a.H + h) * T + min(q, T - 1);
        s_lse[0][tid] = q < T ? a.lse2[si] : INFINITY;
        s_delta[0][tid] = q < T ? a.delta[si] : 0.0f;
        s_lb[0][tid] = key_lb(q, T, a.left, pos);
      }
      __syncthreads();
      f32x16 s = zero16(), dp = zero16();
      const int64_t qrow = (int64_t)min(q0 + l32, T - 1) * qpitch;
      for (int c = 0; c < KC; ++c) {
        const int at = 16 * c + 8 * g;
        s = M::mma(M::load8(Qb + qrow + at), key < T ? M::load8(Kb + krow + at) : M::zero(), s);
        dp = M::mma(M::load8(Ob + qrow + at), key < T ? M::load8(Vb + krow + at) : M::zero(), dp);
      }
      softmax(std::true_type{}, s, dp, q0, 0, a.scale_log2, 1.0f);
#pragma unroll
      for (int kc = 0; kc < 2; ++kc) {
        const f32x8 pf = kc ? M::from_acc<1>(s) : M::from_acc<0>(s);
        const f32x8 sf = kc ? M::from_acc<1>(dp) : M::from_acc<0>(dp);
#pragma unroll
        for (int db = 0; db < DB; ++db) {
          f32x8 of, qf;
          load_rows_f32<D>(Ob, qpitch, q0 + 16 * kc, T, 32 * db + l32, g, of);
          load_rows_f32<D>(Qb, qpitch, q0 + 16 * kc, T, 32 * db + l32, g, qf);
          dv[db] = M::mma(pf, of, dv[db]);
          dk[db] = M::mma(sf, qf, dk[db]);
        }
      }
    }
  }

  // Store: accumulator row = key, column = head-dim index.
#pragma unroll
  for (int db = 0; db < DB; ++db) {
    const int d = 32 * db + l32;
    if (d < D) {
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int kk = kw0 + acc_row(r, g);
        if (kk < T) {
          const int64_t off = ((int64_t)b * T + kk) * kpitch + (int64_t)kvh * D + d;
          float vk = dk[db][r] * kscale, vv = dv[db][r] * vscale;
          float* pk = static_cast<float*>(a.dK) + off;
          float* pv = static_cast<float*>(a.dV) + off;
          if (a.accumulate) {
            vk += *pk;
            vv += *pv;
          }
          *pk = vk;
          *pv = vv;
        }
      }
    }
  }
}

// ---------------------------------------------------------------------------
// dQ, exact mode: 128 queries of one (batch, head) per workgroup, 32 per wave
// with Q and dO resident in parts; S^T and dP^T are recomputed with the query
// as the lane index, so dS^T is directly the B operand of dQ^T += K^T dS^T.
// K and V tiles of 32 keys are split once per workgroup into double-buffered
// LDS, a tile ahead.  8 x 2048 tokens, causal, H6 D128: 497 us (fp32 MFMA
// 782), H12 D64: 398 (756).  Loading a further tile ahead, alternating
// products of two sums and fixed orders of reads and products measured within
// 3% (slower at D = 64, where they spill).
template <int D>
__global__ __launch_bounds__(kThreads, D <= 64 ? 2 : 1) void attn_bwd_dq_exact_kernel(BwdArgs a) {
  constexpr int BN = kExactBT, KC = D / 16, DB = (D + 31) / 32;
  constexpr int kTile = SplitTile<D>::kBytes, kBM = 128;
  __shared__ __attribute__((aligned(1024))) char bufs[2][2 * kTile];  // K, V
  __shared__ int s_bounds[2][kWaves];

  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int g = lane >> 5, l32 = lane & 31;
  const int T = a.T;
  const int n_qt = (T + kBM - 1) / kBM;
  const GridItem it0 = heavy_first(blockIdx.x, a.H * a.B);
  const int qt = n_qt - 1 - it0.rank;  // longest query tiles first, over the whole grid
  int b, h;
  query_row(it0.row, a.B, a.Hkv, a.group, b, h);
  const int kvh = h / a.group;

  const int64_t qpitch = (int64_t)a.H * D, kpitch = (int64_t)a.Hkv * D;
  const float* Qb = static_cast<const float*>(a.Q) + ((int64_t)b * T * a.H + h) * D;
  const float* Ob = static_cast<const float*>(a.dO) + ((int64_t)b * T * a.H + h) * D;
  const float* Kb = static_cast<const float*>(a.K) + ((int64_t)b * T * a.Hkv + kvh) * D;
  const float* Vb = static_cast<const float*>(a.V) + ((int64_t)b * T * a.Hkv + kvh) * D;
  const int32_t* pos = a.pos ? a.pos + (int64_t)b * T : nullptr;

  const int q = qt * kBM + wave * 32 + l32;
  const int lb = key_lb(q, T, a.left, pos), ub = key_ub(q, T, a.right);
  const bool multiple = ub > lb;
  const int wlb_min = __builtin_amdgcn_readfirstlane(wave_min32(lb)), wlb_max = __builtin_amdgcn_readfirstlane(wave_max32(lb));
  const int wub_min = __builtin_amdgcn_readfirstlane(wave_min32(ub)), wub_max = __builtin_amdgcn_readfirstlane(wave_max32(ub));
  if (lane == 0) {
    s_bounds[0][wave] = wlb_min;
    s_bounds[1][wave] = wub_max;
  }
  const int64_t si = ((int64_t)b * a.H + h) * T + min(q, T - 1);
  const float lse = q < T ? a.lse2[si] : INFINITY;
  float dlt = q < T ? a.delta[si] * kSplitScale2 : 0.0f;
  bool outside = lse < kSplitLse && lse != -INFINITY;  // (-inf: a row that sees no key)

  Split8 qf[KC], of[KC];
  const int64_t qrow = (int64_t)min(q, T - 1) * qpitch;
  split_rows<D>(Qb + qrow, q < T, g, qf);
  split_rows<D>(Ob + qrow, q < T, g, of);
  FragOffsets<tile_width(D)> fo;
  fo.init(lane);
  f32x16 dq[DB];
#pragma unroll
  for (int i = 0; i < DB; ++i) dq[i] = zero16();

  __syncthreads();
  int kmin = s_bounds[0][0], kmax = s_bounds[1][0];
#pragma unroll
  for (int w = 1; w < kWaves; ++w) {
    kmin = min(kmin, s_bounds[0][w]);
    kmax = max(kmax, s_bounds[1][w]);
  }
  const int kt0 = __builtin_amdgcn_readfirstlane((kmin / BN) * BN);
  const int ntiles = __builtin_amdgcn_readfirstlane(kmax >= kmin ? (kmax - (kmin / BN) * BN) / BN + 1 : 0);

  float c2 = a.scale_log2 * kSplitInv2, qscale = a.scale * kSplitInv3;  // dQ holds dS (2^32) times K

  // dS of a tile into dp.
  auto softmax = [&](auto need_mask, const f32x16& s, f32x16& dp, int kt) __attribute__((always_inline)) {
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const float p = __builtin_amdgcn_exp2f(__builtin_fmaf(s[r], c2, -lse));
      const float ds = p * (dp[r] - dlt);
      if constexpr (decltype(need_mask)::value) {
        const int kk = kt + acc_row(r, g);
        dp[r] = ((kk >= lb) & (kk <= ub) & multiple) ? ds : 0.0f;
      } else {
        dp[r] = ds;
      }
    }
  };

  SplitStage<D> kst, vst;
  // One tile: the next tile's K is split and stored between S and dP, its V
  // between dP and dQ (past the last tile, rows of the slice go to the idle
  // buffer); a mask is a uniform branch of its own, so that one copy of the
  // products serves all tiles.
  auto body = [&](int kt, int buf, bool need_mask) __attribute__((always_inline)) {
    const char* Ks = bufs[buf];
    const char* Vs = Ks + kTile;
    char* next = bufs[buf ^ 1];
    f32x16 s = zero16(), dp = zero16();
    vst.load(Vb, kpitch, kt + BN, T, tid);
#pragma unroll
    for (int c = 0; c < KC; ++c) s = mma_split(split_nat<D>(Ks, fo, c), qf[c], s);
    kst.store(next, tid);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int c = 0; c < KC; ++c) dp = mma_split(split_nat<D>(Vs, fo, c), of[c], dp);
    vst.store(next + kTile, tid);
    __builtin_amdgcn_sched_barrier(0);
    if (need_mask) softmax(std::true_type{}, s, dp, kt);
    else softmax(std::false_type{}, s, dp, kt);
#pragma unroll
    for (int kc = 0; kc < 2; ++kc) {
      const Split8 sf = kc ? split_acc<1>(dp) : split_acc<0>(dp);
#pragma unroll
      for (int db = 0; db < DB; ++db) dq[db] = mma_split(split_tr<D>(Ks, fo, kc, db), sf, dq[db]);
    }
  };
  if (ntiles > 0) {
    kst.load(Kb, kpitch, kt0, T, tid);
    vst.load(Vb, kpitch, kt0, T, tid);
    kst.store(bufs[0], tid);
    vst.store(bufs[0] + kTile, tid);
    kst.load(Kb, kpitch, kt0 + BN, T, tid);
  }
  __syncthreads();
  for (int it = 0; it < ntiles; ++it) {
    const int kt = kt0 + it * BN;
    if (wlb_min > kt + BN - 1 || wub_max < kt) {
      vst.load(Vb, kpitch, kt + BN, T, tid);
      char* next = bufs[(it + 1) & 1];
      kst.store(next, tid);
      vst.store(next + kTile, tid);
    } else {
      body(kt, it & 1, !(wlb_max <= kt && kt + BN - 1 <= wub_min));
    }
    kst.load(Kb, kpitch, kt + 2 * BN, T, tid);
    __syncthreads();
  }

  outside |= !all_finite<D>(dq);
  if (__builtin_amdgcn_ballot_w64(outside) != 0) {
    // fp32 MFMA from global memory.
    using M = Mma<float>;
    c2 = a.scale_log2;
    qscale = a.scale;
    dlt = q < T ? a.delta[si] : 0.0f;
#pragma unroll
    for (int i = 0; i < DB; ++i) dq[i] = zero16();
#pragma unroll 1
    for (int kt = (wlb_min / BN) * BN; kt <= wub_max; kt += BN) {
      f32x16 s = zero16(), dp = zero16();
      const int64_t krow = (int64_t)min(kt + l32, T - 1) * kpitch;
      for (int c = 0; c < KC; ++c) {
        const int at = 16 * c + 8 * g;
        s = M::mma(M::load8(Kb + krow + at), q < T ? M::load8(Qb + qrow + at) : M::zero(), s);
        dp = M::mma(M::load8(Vb + krow + at), q < T ? M::load8(Ob + qrow + at) : M::zero(), dp);
      }
      softmax(std::true_type{}, s, dp, kt);
#pragma unroll
      for (int kc = 0; kc < 2; ++kc) {
        const f32x8 sf = kc ? M::from_acc<1>(dp) : M::from_acc<0>(dp);
#pragma unroll
        for (int db = 0; db < DB; ++db) {
          f32x8 kfr;
          load_rows_f32<D>(Kb, kpitch, kt + 16 * kc, T, 32 * db + l32, g, kfr);
          dq[db] = M::mma(kfr, sf, dq[db]);
        }
      }
    }
  }

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
          for (int t = 0; t < 4; ++t) v[t] = dq[db][4 * j + t] * qscale;
          store4(static_cast<float*>(a.dQ) + orow * D + d0, v, a.accumulate);
        }
      }
    }
  }
}

// ---------------------------------------------------------------------------

template <int D, typename TO, typename TD>
static hipError_t launch_pre_t(const Problem& p, const PreArgs& a, hipStream_t s) {
  constexpr int QPB = kThreads / (tile_width(D) / 8);
  const int64_t n = (int64_t)p.B * p.T * p.H;
  const dim3 grid((unsigned)((n + QPB - 1) / QPB)), block(kThreads);
  const ProfileMark mk = profile_begin(s);
  hipLaunchKernelGGL((attn_bwd_pre_kernel<D, TO, TD>), grid, block, 0, s, a);
  const hipError_t e = hipGetLastError();
  profile_end(mk, "attn_bwd_pre", s);
  return e;
}

template <int D>
static hipError_t launch_pre_d(const Problem& p, const PreArgs& a, hipStream_t s) {
  if (a.O_bf16) {
    return a.dO_bf16 ? launch_pre_t<D, bf16, bf16>(p, a, s) : launch_pre_t<D, bf16, float>(p, a, s);
  }
  return a.dO_bf16 ? launch_pre_t<D, float, bf16>(p, a, s) : launch_pre_t<D, float, float>(p, a, s);
}

hipError_t launch_bounds(const Problem& p, const BoundsArgs& a, hipStream_t s) {
  const int64_t n = (int64_t)((p.T + 31) / 32) * p.B * 32;  // one lane per query slot
  const dim3 grid((unsigned)((n + kThreads - 1) / kThreads)), block(kThreads);
  const ProfileMark mk = profile_begin(s);
  hipLaunchKernelGGL(attn_bounds_kernel, grid, block, 0, s, a);
  const hipError_t e = hipGetLastError();
  profile_end(mk, "attn_bounds", s);
  return e;
}

hipError_t launch_order(const Problem& p, const OrderArgs& a, hipStream_t s) {
  if (!order_fits(p.T, p.B)) return hipErrorInvalidValue;
  const ProfileMark mk = profile_begin(s);
  hipLaunchKernelGGL(attn_order_kernel, dim3(1), dim3(kOrderThreads), 0, s, a);
  const hipError_t e = hipGetLastError();
  profile_end(mk, "attn_order", s);
  return e;
}

template <int D>
static hipError_t launch_dkdv_exact(const Problem& p, const BwdArgs& a, hipStream_t s) {
  const int n_kt = (p.T + kExactBK - 1) / kExactBK;
  const dim3 grid(n_kt * p.Hkv * p.B), block(kThreads);
  const ProfileMark mk = profile_begin(s);
  hipLaunchKernelGGL((attn_bwd_dkdv_exact_kernel<D>), grid, block, 0, s, a);
  const hipError_t e = hipGetLastError();
  profile_end(mk, "attn_bwd_dkdv_f32", s);
  return e;
}

template <int D>
static hipError_t launch_dq_exact(const Problem& p, const BwdArgs& a, hipStream_t s) {
  const int n_qt = (p.T + 127) / 128;
  const dim3 grid(n_qt * p.H * p.B), block(kThreads);
  const ProfileMark mk = profile_begin(s);
  hipLaunchKernelGGL((attn_bwd_dq_exact_kernel<D>), grid, block, 0, s, a);
  const hipError_t e = hipGetLastError();
  profile_end(mk, "attn_bwd_dq_f32", s);
  return e;
}

#define FC_DISPATCH_D(FN)                          \
  switch (p.D) {                                   \
    case 16: return FN<16>(p, a, s);               \
    case 32: return FN<32>(p, a, s);               \
    case 48: return FN<48>(p, a, s);               \
    case 64: return FN<64>(p, a, s);               \
    case 80: return FN<80>(p, a, s);               \
    case 96: return FN<96>(p, a, s);               \
    case 112: return FN<112>(p, a, s);             \
    case 128: return FN<128>(p, a, s);             \
    default: return hipErrorInvalidValue;          \
  }

hipError_t launch_bwd_pre(const Problem& p, const PreArgs& a, hipStream_t s) { FC_DISPATCH_D(launch_pre_d) }

hipError_t launch_bwd_dkdv(const Problem& p, const BwdArgs& a, hipStream_t s) {
  if (p.bf16) return launch_bwd_dkdv_fast(p, a, s);
  FC_DISPATCH_D(launch_dkdv_exact)
}

hipError_t launch_bwd_dq(const Problem& p, const BwdArgs& a, hipStream_t s) {
  if (p.bf16) return launch_bwd_dq_fast(p, a, s);
  FC_DISPATCH_D(launch_dq_exact)
}

}  // namespace fc
