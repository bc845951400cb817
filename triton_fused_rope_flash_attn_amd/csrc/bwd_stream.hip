// Split backward with streamed tiles: 16-bit tensors computed in their own type
// at head_dim 32 or 64, or in fp16 at 128; vector access to every tensor, planes
// longer than the one-pass kernel takes.
//
// Reference behaviour followed ("fa_rope_full .py"): delta = rowsum(dO * O)
// (FA:325-357); dV += P^T dO, dS = P * (dP - delta), dK-hat += dS^T Q-hat
// (FA:374-691); dQ-hat += dS K-hat (FA:708-1009); gradients are rotated back,
// the CLS row bypasses the rotation.
//
// Three launches:
//   stream_khat_kernel   K-hat * c (c = scale * log2 e) rows to the workspace
//   stream_dq_kernel     query tiles: dQ; also delta, -LSE2 and the Q-hat rows
//   stream_dkdv_kernel   key tiles: dK, dV
// The rows that a tile streams (K-hat and V, or Q-hat and dO) are then ready
// to use, so they go from memory straight to LDS (16 bytes per lane, no
// staging registers, no VALU) in stages of 64 rows, double-buffered with one
// barrier per stage.  Workgroups are 4 waves of 32 rows each (16 in 64-row tiles,
// which dK/dV always takes at head_dim 128), two on a CU, or three (dQ at
// head_dim 32 and 64): their barriers are independent, so one workgroup's
// MFMAs run under another's softmax and stage waits.
//
// Bound by instruction issue (MFMA and the softmax VALU; every operand crosses
// HBM about once).  Measured against bwd_dq_kernel + bwd_dkdv_kernel (us): D 64,
// N 577, 384 planes 264 -> 159; N 4096, 48 planes 795 -> 597; D 32, N 257, 512
// planes 71 -> 43; D 128, fp16, N 577, 384 planes 497 -> 368.
#include <type_traits>

#include "common.h"
#include "params.h"
#include "stream.h"

namespace farope {

// ---------------------------------------------------------------------------
// dQ of 128-query tiles (64 with QT = 1).  Wave w owns QT 16-query subtiles.
// S^T = K-hat Q-hat^T and dP^T = V dO^T per 32-key block, keys in natural
// order: output row 4lg + i of half h is key 16h + 4lg + i, which is
// k-slot 4h + i of the transposed reads of dQ-hat^T += K-hat^T dS^T.  Keys
// >= N have zero K-hat and V rows: in the last stage P is clamped to [0, 1] and
// their dS meets zero rows.  The last stage stands apart, so that the others
// hold neither the clamp nor a test of the plane's end (us, backward, this
// kernel and the next one so: N 4096, 48 planes 625 -> 597; N 577, 384 planes
// 163 -> 158; N 1025, 12 planes 32.0 -> 29.9).
// ---------------------------------------------------------------------------
template <typename S, int CT, int D, int QT>
__global__ void __launch_bounds__(kStreamNW * 64, D == 128 && QT == 2 ? 2 : 3) stream_dq_kernel(const BwdParams p) {
  using C = Comp<CT>;
  using Frag = typename C::Frag;
  constexpr int KS = D / 32, DT = D / 16, SR = kStageRows;
  __shared__ __attribute__((aligned(16))) S sK0[SR * D], sK1[SR * D], sV0[SR * D], sV1[SR * D];

  const int N = p.N;
  const int tile = xcd_remap(block_id(), p.n_wg);
  const int plane = tile / p.n_blk, qblk = tile - plane * p.n_blk;
  const int bb = plane / p.H, hh = plane - bb * p.H;
  const int64_t prow = (int64_t)plane * N;
  const int tid = thread_id();
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int lr = lane & 15, lg = lane >> 4;
  const int shift = 1 - p.has_cls;
  auto base = [&](const void* b, const int64_t* st) { return static_cast<const S*>(b) + bb * st[0] + hh * st[1]; };
  auto rsrc = [&](const void* b, const int64_t* st) {
    return make_rsrc(base(b, st), (unsigned)(((int64_t)(N - 1) * st[2] + D) * 2));
  };

  StreamSrc<D> srcK, srcV;
  srcK.init(static_cast<const S*>(p.khat) + prow * D, D, N, wave, lane);
  srcV.init(base(p.v, p.sv), p.sv[2], N, wave, lane);
  srcK.load(sK0, wave, 0);
  srcV.load(sV0, wave, 0);

  const int row0 = (qblk * kStreamNW + wave) * 16 * QT + lr;   // subtile t: + 16 t
  Frag qf[QT][KS], gf[QT][KS];
  f32x4 nl4[QT], nd4[QT];
  {
    const auto rQ = rsrc(p.q, p.sq), rG = rsrc(p.dout, p.sdo), rO = rsrc(p.o, p.so);
    const auto rT = make_rsrc(p.rope, (unsigned)((N + shift) * D * 4));
    const auto rL = make_rsrc(p.lse + prow, (unsigned)N * 4u);
    Raw8<S> q[QT][KS], g[QT][KS], o[QT][KS];
    u32x4 ta[QT][KS][2];
    float ls[QT];
#pragma unroll
    for (int t = 0; t < QT; ++t) {
      const int row = row0 + 16 * t;
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        const int c0 = 32 * s + 8 * lg;
        q[t][s] = buf_load8<S>(rQ, (unsigned)((row * (int)p.sq[2] + c0) * 2), 0u);
        g[t][s] = buf_load8<S>(rG, (unsigned)((row * (int)p.sdo[2] + c0) * 2), 0u);
        o[t][s] = buf_load8<S>(rO, (unsigned)((row * (int)p.so[2] + c0) * 2), 0u);
        const unsigned to = (unsigned)(((row + shift) * D + c0) * 4);
        ta[t][s][0] = __builtin_amdgcn_raw_buffer_load_b128(rT, to, 0u, 0);
        ta[t][s][1] = __builtin_amdgcn_raw_buffer_load_b128(rT, to + 16u, 0u, 0);
      }
      ls[t] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rL, (unsigned)row * 4u, 0u, 0));
    }
    const auto rH = make_rsrc(static_cast<const S*>(p.qhat_f) + prow * D, (unsigned)(N * D * 2));
    const auto rNl = make_rsrc(p.row_stat + prow, (unsigned)N * 4u);
    const auto rNd = make_rsrc(p.delta + prow, (unsigned)N * 4u);
#pragma unroll
    for (int t = 0; t < QT; ++t) {
      const int row = row0 + 16 * t;
      float ds = 0.f;
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        float x[8], cs[8];
        unpack8(q[t][s], x);
        __builtin_memcpy(cs, &ta[t][s][0], 32);
        rope_rotate8(x, cs);
        qf[t][s] = C::make(x);
        gf[t][s].v = g[t][s].v;
        ds = dot8(g[t][s], o[t][s], ds);
        buf_store16(__builtin_bit_cast(u32x4, qf[t][s].v), rH, (unsigned)((row * D + 32 * s + 8 * lg) * 2), 0u);
      }
      const float nd = -group4_sum(ds), nl = -ls[t] * kLog2e;
      // (lanes lg != 0 write past the range)
      __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(nl), rNl, (unsigned)(lg == 0 ? row : N) * 4u, 0u, 0);
      __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(nd), rNd, (unsigned)(lg == 0 ? row : N) * 4u, 0u, 0);
      nl4[t] = f32x4{nl, nl, nl, nl};
      nd4[t] = f32x4{nd, nd, nd, nd};
    }
  }
  const bool active = row0 - lr < N;   // wave-uniform
  f32x4 acc[QT][DT];
#pragma unroll
  for (int t = 0; t < QT; ++t)
#pragma unroll
    for (int d = 0; d < DT; ++d) acc[t][d] = f32x4{0.f, 0.f, 0.f, 0.f};

  const int ns = (N + SR - 1) / SR;
  // lane offsets of the operand reads (rows lr and lr/4 + 4lg; the swizzle has period 16)
  int ao[KS], to[DT];
#pragma unroll
  for (int s = 0; s < KS; ++s) ao[s] = swz<D>(lr, 32 * s + 8 * lg);
#pragma unroll
  for (int d = 0; d < DT; ++d) to[d] = swz<D>(4 * lg + (lr >> 2), 16 * d + 4 * (lr & 3));

  using Acc = f32x4[QT][2];
  auto sp = [&](const S* __restrict__ k, const S* __restrict__ v, Acc& sacc, Acc& pacc) __attribute__((always_inline)) {
#pragma unroll
    for (int s = 0; s < KS; ++s)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const Frag a = C::lds(k + ao[s] + 16 * h * D), b = C::lds(v + ao[s] + 16 * h * D);
#pragma unroll
        for (int t = 0; t < QT; ++t) {
          sacc[t][h] = C::mma(a, qf[t][s], s == 0 ? nl4[t] : sacc[t][h]);
          pacc[t][h] = C::mma(b, gf[t][s], s == 0 ? nd4[t] : pacc[t][h]);
        }
      }
  };
  // clamp: the block may hold keys >= N, whose P may overflow
  auto out = [&](auto clamp, const S* __restrict__ k, const Acc& sacc, const Acc& pacc) __attribute__((always_inline)) {
    Frag dsf[QT];
#pragma unroll
    for (int t = 0; t < QT; ++t) {
      float ds[8];
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float e = fast_exp2(sacc[t][h][i]);
          ds[4 * h + i] = (clamp.value ? __builtin_amdgcn_fmed3f(e, 0.f, 1.f) : e) * pacc[t][h][i];
        }
      dsf[t] = C::make(ds);
    }
#pragma unroll
    for (int d = 0; d < DT; ++d) {
      const Frag a = C::tr(k + to[d], k + to[d] + 16 * D);
#pragma unroll
      for (int t = 0; t < QT; ++t) acc[t][d] = C::mma(a, dsf[t], acc[t][d]);
    }
  };
  auto stage = [&](auto last, int st, const S* __restrict__ k, const S* __restrict__ v, S* __restrict__ kn, S* __restrict__ vn)
      __attribute__((always_inline)) {
    // every load into (k, v) has landed in every wave, and every wave is past
    // its reads of (kn, vn)
    stage_barrier();
    if (!last.value) {
      srcK.load(kn, wave, (st + 1) * SR);
      srcV.load(vn, wave, (st + 1) * SR);
    }
    if (active) {
      Acc sA, pA, sB, pB;
      if (!last.value || st * SR + 32 < N) {
        sp(k, v, sA, pA);
        sp(k + 32 * D, v + 32 * D, sB, pB);
        out(last, k, sA, pA);
        out(last, k + 32 * D, sB, pB);
      } else {
        sp(k, v, sA, pA);
        out(last, k, sA, pA);
      }
    }
  };
  int st = 0;
  for (; st + 2 < ns; st += 2) {
    stage(std::false_type{}, st, sK0, sV0, sK1, sV1);
    stage(std::false_type{}, st + 1, sK1, sV1, sK0, sV0);
  }
  if (st + 1 < ns) {
    stage(std::false_type{}, st, sK0, sV0, sK1, sV1);
    stage(std::true_type{}, st + 1, sK1, sV1, sK0, sV0);
  } else {
    stage(std::true_type{}, st, sK0, sV0, sK1, sV1);
  }

  // dQ = R^T dQ-hat * scale (K-hat carries c2); lane groups lg and lg^1 trade
  // halves so that each lane stores 8 consecutive channels; rows >= N drop
  const float dq_scale = p.scale / p.scale_log2;
  const auto rD = rsrc(p.dq, p.sdq);
  const auto rT = make_rsrc(p.rope, (unsigned)((N + shift) * D * 4));
#pragma unroll
  for (int t = 0; t < QT; ++t) {
    const int row = row0 + 16 * t;
#pragma unroll
    for (int d0 = 0; d0 < DT; d0 += 2) {
      u32x2 w[2];
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const int d = d0 + j;
        const u32x4 tb = __builtin_amdgcn_raw_buffer_load_b128(rT, (unsigned)(((row + shift) * D + 16 * d + 4 * lg) * 4), 0u, 0);
        typedef S s4 __attribute__((ext_vector_type(4)));
        s4 a;
#pragma unroll
        for (int r = 0; r < 2; ++r) {
          const float e = acc[t][d][2 * r] * dq_scale, o = acc[t][d][2 * r + 1] * dq_scale;
          const float c = __uint_as_float(tb[2 * r]), sn = __uint_as_float(tb[2 * r + 1]);
          a[2 * r] = (S)(e * c + o * sn);
          a[2 * r + 1] = (S)(o * c - e * sn);
        }
        __builtin_memcpy(&w[j], &a, 8);
      }
      u32x4 x;
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        const auto r = __builtin_amdgcn_permlane16_swap(w[0][k], w[1][k], false, false);
        x[k] = r[0];
        x[2 + k] = r[1];
      }
      buf_store16(x, rD, (unsigned)((row * (int)p.sdq[2] + 16 * (d0 + (lg & 1)) + 4 * (lg & 2)) * 2), 0u);
    }
  }
}

// ---------------------------------------------------------------------------
// dK / dV of 128-key tiles (64 with KT = 1).  Wave w owns KT 16-key subtiles:
// K-hat and V rows are B operands in registers, dK-hat and dV accumulate in
// registers.  In the last stage queries >= N take -LSE2 = -inf, so that P = 0.
// (Their Q-hat, -LSE2 and -delta read 0 past the range; their dO does so only
// where dO's rows do not overlap: with a row stride of 0, as the backward of a
// sum over the tokens gives it, every row reads the one real row.)
// ---------------------------------------------------------------------------
template <typename S, int CT, int D, int KT>
__global__ void __launch_bounds__(kStreamNW * 64, 2) stream_dkdv_kernel(const BwdParams p) {
  using C = Comp<CT>;
  using Frag = typename C::Frag;
  constexpr int KS = D / 32, DT = D / 16, SR = kStageRows;
  __shared__ __attribute__((aligned(16))) S sQ0[SR * D], sQ1[SR * D], sG0[SR * D], sG1[SR * D];
  __shared__ __attribute__((aligned(16))) float sL0[SR], sL1[SR], sD0[SR], sD1[SR];

  const int N = p.N;
  const int tile = xcd_remap(block_id(), p.n_wg);
  const int plane = tile / p.n_blk, kblk = tile - plane * p.n_blk;
  const int bb = plane / p.H, hh = plane - bb * p.H;
  const int64_t prow = (int64_t)plane * N;
  const int tid = thread_id();
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int lr = lane & 15, lg = lane >> 4;
  const int shift = 1 - p.has_cls;
  auto base = [&](const void* b, const int64_t* st) { return static_cast<const S*>(b) + bb * st[0] + hh * st[1]; };
  auto rsrc = [&](const void* b, const int64_t* st) {
    return make_rsrc(base(b, st), (unsigned)(((int64_t)(N - 1) * st[2] + D) * 2));
  };

  StreamSrc<D> srcQ, srcG;
  srcQ.init(static_cast<const S*>(p.qhat_f) + prow * D, D, N, wave, lane);
  srcG.init(base(p.dout, p.sdo), p.sdo[2], N, wave, lane);
  // waves 0 and 1 also fetch the stage's -LSE2 and -delta
  const auto rStat = make_rsrc((wave & 1 ? p.delta : p.row_stat) + prow, (unsigned)N * 4u);
  auto load = [&](int st, S* q, S* g, float* l, float* d) __attribute__((always_inline)) {
    srcQ.load(q, wave, st * SR);
    srcG.load(g, wave, st * SR);
    if (wave < 2) lds_dma4(rStat, wave ? d : l, (unsigned)lane * 4u, (unsigned)(st * SR) * 4u);
  };
  load(0, sQ0, sG0, sL0, sD0);

  const int row0 = (kblk * kStreamNW + wave) * 16 * KT + lr;   // subtile u: + 16 u
  Frag kf[KT][KS], vf[KT][KS];
  {
    const auto rK = make_rsrc(static_cast<const S*>(p.khat) + prow * D, (unsigned)(N * D * 2));
    const auto rV = rsrc(p.v, p.sv);
#pragma unroll
    for (int u = 0; u < KT; ++u)
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        const int row = row0 + 16 * u, c0 = 32 * s + 8 * lg;
        kf[u][s].v = __builtin_bit_cast(decltype(kf[u][s].v), buf_load8<S>(rK, (unsigned)((row * D + c0) * 2), 0u).v);
        vf[u][s].v = __builtin_bit_cast(decltype(vf[u][s].v), buf_load8<S>(rV, (unsigned)((row * (int)p.sv[2] + c0) * 2), 0u).v);
      }
  }
  const bool active = row0 - lr < N;   // wave-uniform
  f32x4 dv[KT][DT], dk[KT][DT];
#pragma unroll
  for (int u = 0; u < KT; ++u)
#pragma unroll
    for (int d = 0; d < DT; ++d) dv[u][d] = dk[u][d] = f32x4{0.f, 0.f, 0.f, 0.f};

  const int ns = (N + SR - 1) / SR;
  int ao[KS], to[DT];
#pragma unroll
  for (int s = 0; s < KS; ++s) ao[s] = swz<D>(lr, 32 * s + 8 * lg);
#pragma unroll
  for (int d = 0; d < DT; ++d) to[d] = swz<D>(4 * lg + (lr >> 2), 16 * d + 4 * (lr & 3));

  using Acc = f32x4[KT][2];
  // last: queries at left or beyond (counted from the block's first) do not exist
  auto sp = [&](auto last, int left, const S* __restrict__ q, const S* __restrict__ g, const float* __restrict__ l,
                const float* __restrict__ dl, Acc& sacc, Acc& pacc) __attribute__((always_inline)) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      f32x4 nl = *reinterpret_cast<const f32x4*>(l + 16 * h + 4 * lg);
      if constexpr (last.value) {
#pragma unroll
        for (int i = 0; i < 4; ++i) nl[i] = 16 * h + 4 * lg + i < left ? nl[i] : -INFINITY;
      }
      const f32x4 nd = *reinterpret_cast<const f32x4*>(dl + 16 * h + 4 * lg);
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        const Frag a = C::lds(q + ao[s] + 16 * h * D), b = C::lds(g + ao[s] + 16 * h * D);
#pragma unroll
        for (int u = 0; u < KT; ++u) {
          sacc[u][h] = C::mma(a, kf[u][s], s == 0 ? nl : sacc[u][h]);
          pacc[u][h] = C::mma(b, vf[u][s], s == 0 ? nd : pacc[u][h]);
        }
      }
    }
  };
  auto out = [&](const S* __restrict__ q, const S* __restrict__ g, const Acc& sacc, const Acc& pacc) __attribute__((always_inline)) {
    Frag pf[KT], dsf[KT];
#pragma unroll
    for (int u = 0; u < KT; ++u) {
      float pv[8], ds[8];
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          pv[4 * h + i] = fast_exp2(sacc[u][h][i]);
          ds[4 * h + i] = pv[4 * h + i] * pacc[u][h][i];
        }
      pf[u] = C::make(pv);
      dsf[u] = C::make(ds);
    }
#pragma unroll
    for (int d = 0; d < DT; ++d) {
      const Frag ag = C::tr(g + to[d], g + to[d] + 16 * D);
      const Frag aq = C::tr(q + to[d], q + to[d] + 16 * D);
#pragma unroll
      for (int u = 0; u < KT; ++u) {
        dv[u][d] = C::mma(ag, pf[u], dv[u][d]);
        dk[u][d] = C::mma(aq, dsf[u], dk[u][d]);
      }
    }
  };
  auto stage = [&](auto last, int st, const S* __restrict__ q, const S* __restrict__ g, const float* __restrict__ l, const float* __restrict__ dl,
                   S* __restrict__ qn, S* __restrict__ gn, float* __restrict__ ln, float* __restrict__ dn) __attribute__((always_inline)) {
    stage_barrier();
    if (!last.value) load(st + 1, qn, gn, ln, dn);
    if (active) {
      const int left = N - st * SR;
      Acc sA, pA;
      if (!last.value || left > 32) {
        Acc sB, pB;
        sp(last, left, q, g, l, dl, sA, pA);
        sp(last, left - 32, q + 32 * D, g + 32 * D, l + 32, dl + 32, sB, pB);
        out(q, g, sA, pA);
        out(q + 32 * D, g + 32 * D, sB, pB);
      } else {
        sp(last, left, q, g, l, dl, sA, pA);
        out(q, g, sA, pA);
      }
    }
  };
  int st = 0;
  for (; st + 2 < ns; st += 2) {
    stage(std::false_type{}, st, sQ0, sG0, sL0, sD0, sQ1, sG1, sL1, sD1);
    stage(std::false_type{}, st + 1, sQ1, sG1, sL1, sD1, sQ0, sG0, sL0, sD0);
  }
  if (st + 1 < ns) {
    stage(std::false_type{}, st, sQ0, sG0, sL0, sD0, sQ1, sG1, sL1, sD1);
    stage(std::true_type{}, st + 1, sQ1, sG1, sL1, sD1, sQ0, sG0, sL0, sD0);
  } else {
    stage(std::true_type{}, st, sQ0, sG0, sL0, sD0, sQ1, sG1, sL1, sD1);
  }

  const auto rdK = rsrc(p.dk, p.sdk), rdV = rsrc(p.dv, p.sdv);
  const auto rT = make_rsrc(p.rope, (unsigned)((N + shift) * D * 4));
#pragma unroll
  for (int u = 0; u < KT; ++u) {
    const int row = row0 + 16 * u;
#pragma unroll
    for (int d0 = 0; d0 < DT; d0 += 2) {
      u32x2 wk[2], wv[2];
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const int d = d0 + j;
        const u32x4 tb = __builtin_amdgcn_raw_buffer_load_b128(rT, (unsigned)(((row + shift) * D + 16 * d + 4 * lg) * 4), 0u, 0);
        typedef S s4 __attribute__((ext_vector_type(4)));
        s4 a, b;
#pragma unroll
        for (int r = 0; r < 2; ++r) {
          const float e = dk[u][d][2 * r] * p.scale, o = dk[u][d][2 * r + 1] * p.scale;
          const float c = __uint_as_float(tb[2 * r]), sn = __uint_as_float(tb[2 * r + 1]);
          a[2 * r] = (S)(e * c + o * sn);
          a[2 * r + 1] = (S)(o * c - e * sn);
          b[2 * r] = (S)dv[u][d][2 * r];
          b[2 * r + 1] = (S)dv[u][d][2 * r + 1];
        }
        __builtin_memcpy(&wk[j], &a, 8);
        __builtin_memcpy(&wv[j], &b, 8);
      }
      u32x4 xk, xv;
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        const auto r1 = __builtin_amdgcn_permlane16_swap(wk[0][k], wk[1][k], false, false);
        const auto r2 = __builtin_amdgcn_permlane16_swap(wv[0][k], wv[1][k], false, false);
        xk[k] = r1[0];
        xk[2 + k] = r1[1];
        xv[k] = r2[0];
        xv[2 + k] = r2[1];
      }
      const int ch = 16 * (d0 + (lg & 1)) + 4 * (lg & 2);
      buf_store16(xk, rdK, (unsigned)((row * (int)p.sdk[2] + ch) * 2), 0u);
      buf_store16(xv, rdV, (unsigned)((row * (int)p.sdv[2] + ch) * 2), 0u);
    }
  }
}

template <typename S, int CT, int D>
static hipError_t stream_launch(const BwdParams& p0, hipStream_t st) {
  BwdParams p = p0;
  const int planes = p.B * p.H;
  hipError_t e = launch_stream_khat(KhatParams{p.k, p.khat, {p.sk[0], p.sk[1], p.sk[2]}, p.rope, planes, p.H, p.N,
                                               p.has_cls, p.scale_log2}, CT, D, st);
  if (e != hipSuccess) return e;
  const int rows = stream_rows(planes, p.N, D, true);
  const bool half = rows < kStreamTileRows;
  p.n_blk = (p.N + rows - 1) / rows;
  p.n_wg = planes * p.n_blk;
  auto dq = half ? stream_dq_kernel<S, CT, D, 1> : stream_dq_kernel<S, CT, D, 2>;
  hipLaunchKernelGGL(dq, dim3(p.n_wg), dim3(kStreamNW * 64), 0, st, p);
  e = hipGetLastError();
  if (e != hipSuccess) return e;
  // (D 128: the dK / dV accumulators of two subtiles alone would take 128 registers)
  constexpr int KTM = D == 128 ? 1 : 2;
  const int krows = half ? kStreamTileRows / 2 : kStreamTileRows / 2 * KTM;
  p.n_blk = (p.N + krows - 1) / krows;
  p.n_wg = planes * p.n_blk;
  auto dkdv = half ? stream_dkdv_kernel<S, CT, D, 1> : stream_dkdv_kernel<S, CT, D, KTM>;
  hipLaunchKernelGGL(dkdv, dim3(p.n_wg), dim3(kStreamNW * 64), 0, st, p);
  return hipGetLastError();
}

hipError_t launch_bwd_stream(const BwdParams& p, int io, int D, hipStream_t st) {
  if (io == DT_BF16) return D == 64 ? stream_launch<bf16, DT_BF16, 64>(p, st) : stream_launch<bf16, DT_BF16, 32>(p, st);
  return D == 128 ? stream_launch<f16, DT_F16, 128>(p, st)
         : D == 64 ? stream_launch<f16, DT_F16, 64>(p, st) : stream_launch<f16, DT_F16, 32>(p, st);
}

}  // namespace farope
