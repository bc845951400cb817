// Forward with streamed tiles: 16-bit tensors computed in their own type at
// head_dim 32 or 64, or in fp16 at 128; vector access to every tensor.
//
// Reference behaviour followed: _attn_fwd in "fa_rope_full .py" (FA:91-315):
// rotation with the CLS row bypassing it (FA:176-202, FA:248-272), scaled
// logits, online softmax (FA:280-305), per-row log-sum-exp (FA:308-309).
//
// stream_khat_kernel writes the rotated, scaled K rows once; the tiles then
// stream K-hat and V from memory straight to LDS (16 bytes per lane, no
// staging registers or VALU), in double-buffered stages of 64 keys with one
// barrier each.  Three 4-wave workgroups run on a CU (two at head_dim 128, whose
// stages take 64 KB), so one's MFMAs fill the time of another's softmax.
//
// Bound by the softmax VALU (16 exponentials, maxima and row-sum adds per lane
// and 32 x 32 block against 16 MFMAs).  Measured against fwd_kernel (one 8-wave
// workgroup per CU, 256-row tiles; us): D 64, N 577, 384 planes 89 -> 58 (K-hat
// pass 11); N 4096, 48 planes 285 -> 207; N 1025, 64 planes 46 -> 37; D 32, N
// 3970, 10 planes 81 -> 43; D 128, fp16, N 577, 384 planes 137 -> 117.  Two or
// four workgroups per CU (D 32 and 64): within 1%.
#include <type_traits>

#include "common.h"
#include "params.h"
#include "stream.h"

namespace farope {

// ---------------------------------------------------------------------------
// K-hat * c2 rows, [planes][N][D] in the compute type.  A workgroup takes a
// block of rows (one 8-channel chunk per thread) in kKhatPlanes planes: their
// loads are in flight together and share one read of the table, and no thread
// divides.  Bound by memory.  Measured against one chunk per thread over a flat
// index (us, forward with this pass): 64 planes of N 1025, D 64, strided views
// 38.2 -> 37.1; 512 of N 257, D 32 24.3 -> 22.6; 384 of N 577, D 128 120.4 ->
// 117.7.  One plane: 37.0, 22.8, 120.1; four: 37.9, 22.8, 118.0.
// ---------------------------------------------------------------------------
template <typename S, int CT, int D>
__global__ void __launch_bounds__(256) stream_khat_kernel(const KhatParams p, int n_blk) {
  constexpr int CPR = D / 8, ROWS = 256 / CPR;
  const int group = block_id() / n_blk, blk = block_id() - group * n_blk;
  const int plane0 = group * kKhatPlanes;
  const int tid = thread_id();
  const int n = blk * ROWS + tid / CPR, c = 8 * (tid % CPR);
  if (n >= p.N) return;

  Raw8<S> raw[kKhatPlanes];
#pragma unroll
  for (int i = 0; i < kKhatPlanes; ++i) {
    const int plane = plane0 + i < p.planes ? plane0 + i : plane0;
    const int bb = plane / p.H, hh = plane - bb * p.H;
    raw[i] = load_raw8(static_cast<const S*>(p.k) + bb * p.sk[0] + hh * p.sk[1] + n * p.sk[2] + c, 1, true);
  }
  float cs[8];
  rope_load4(p.rope, n + 1 - p.has_cls, D / 2, c / 2, cs);
#pragma unroll
  for (int i = 0; i < kKhatPlanes; ++i) {
    if (plane0 + i >= p.planes) break;
    float x[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) x[e] = (float)raw[i].v[e];
    rope_rotate8(x, cs);
#pragma unroll
    for (int e = 0; e < 8; ++e) x[e] *= p.c2;
    Comp<CT>::put8(static_cast<S*>(p.khat) + ((int64_t)(plane0 + i) * p.N + n) * D + c, x);
  }
}

// ---------------------------------------------------------------------------
// O and LSE of 128-query tiles (64 with QT = 1).  Wave w owns QT 16-query
// subtiles; logits are computed transposed, S^T = K-hat Q-hat^T, per
// 32-key block with keys in natural order: output row 4lg + i of half h is key
// 16h + 4lg + i, which is k-slot 4h + i of the transposed V reads of
// O^T += V^T P^T, so P never leaves registers.  The accumulators start at
// minus the running max, so P = exp2 of the product's output; O and the row
// sum are rescaled only when some logit exceeds the running max by 2^8.
// ---------------------------------------------------------------------------
constexpr float kStreamSlack = 8.0f;   // log2 units: P <= 2^8 between rescales

template <typename S, int CT, int D, int QT>
__global__ void __launch_bounds__(kStreamNW * 64, D == 128 && QT == 2 ? 2 : 3) fwd_stream_kernel(const FwdParams p, const S* __restrict__ khat) {
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
  srcK.init(khat + prow * D, D, N, wave, lane);
  srcV.init(base(p.v, p.sv), p.sv[2], N, wave, lane);
  srcK.load(sK0, wave, 0);
  srcV.load(sV0, wave, 0);

  const int row0 = (qblk * kStreamNW + wave) * 16 * QT + lr;   // subtile t: + 16 t
  Frag qf[QT][KS];
  {
    const auto rQ = rsrc(p.q, p.sq);
    const auto rT = make_rsrc(p.rope, (unsigned)((N + shift) * D * 4));
    Raw8<S> q[QT][KS];
    u32x4 ta[QT][KS][2];
#pragma unroll
    for (int t = 0; t < QT; ++t)
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        const int row = row0 + 16 * t, c0 = 32 * s + 8 * lg;
        q[t][s] = buf_load8<S>(rQ, (unsigned)((row * (int)p.sq[2] + c0) * 2), 0u);
        const unsigned to = (unsigned)(((row + shift) * D + c0) * 4);
        ta[t][s][0] = __builtin_amdgcn_raw_buffer_load_b128(rT, to, 0u, 0);
        ta[t][s][1] = __builtin_amdgcn_raw_buffer_load_b128(rT, to + 16u, 0u, 0);
      }
#pragma unroll
    for (int t = 0; t < QT; ++t)
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        float x[8], cs[8];
        unpack8(q[t][s], x);
        __builtin_memcpy(cs, &ta[t][s][0], 32);
        rope_rotate8(x, cs);
        qf[t][s] = C::make(x);
      }
  }
  const bool active = row0 - lr < N;   // wave-uniform
  f32x4 acc[QT][DT];
  float m_run[QT], l_run[QT];
  f32x4 nm4[QT];       // minus the running max (0 before the first block)
  float thr = -INFINITY;   // a value above it makes the block rescale
#pragma unroll
  for (int t = 0; t < QT; ++t) {
    m_run[t] = -INFINITY;
    l_run[t] = 0.f;
    nm4[t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int d = 0; d < DT; ++d) acc[t][d] = f32x4{0.f, 0.f, 0.f, 0.f};
  }

  const int ns = (N + SR - 1) / SR;
  int ao[KS], to[DT];
#pragma unroll
  for (int s = 0; s < KS; ++s) ao[s] = swz<D>(lr, 32 * s + 8 * lg);
#pragma unroll
  for (int d = 0; d < DT; ++d) to[d] = swz<D>(4 * lg + (lr >> 2), 16 * d + 4 * (lr & 3));

  // The stage's two 32-key blocks: both logit products, one test of the running
  // max, then each block's probabilities and O product.  Keys at lim or beyond
  // (counted from this lane's first; tail: there are some) get probability 0.
  using Acc = f32x4[2][QT][2];
  auto blocks = [&](const S* __restrict__ k, const S* __restrict__ v, bool tail, int lim) __attribute__((always_inline)) {
    Acc sacc;
#pragma unroll
    for (int s = 0; s < KS; ++s)
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const Frag a = C::lds(k + ao[s] + (32 * j + 16 * h) * D);
#pragma unroll
          for (int t = 0; t < QT; ++t) sacc[j][t][h] = C::mma(a, qf[t][s], s == 0 ? nm4[t] : sacc[j][t][h]);
        }
    if (tail) {   // uniform; the plane's last stage
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int t = 0; t < QT; ++t)
#pragma unroll
          for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int i = 0; i < 4; ++i) sacc[j][t][h][i] = 32 * j + 16 * h + i < lim ? sacc[j][t][h][i] : -INFINITY;
    }
    float mx[QT], mxx = -INFINITY;
#pragma unroll
    for (int t = 0; t < QT; ++t) {
      float y[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const f32x4 x = sacc[j >> 1][t][j & 1];
        y[j] = fmaxf(fmaxf(x[0], x[1]), fmaxf(x[2], x[3]));
      }
      mx[t] = fmaxf(fmaxf(y[0], y[1]), fmaxf(y[2], y[3]));
      mxx = fmaxf(mxx, mx[t]);
    }
    if (__any(mxx > thr)) {
      thr = kStreamSlack;
#pragma unroll
      for (int t = 0; t < QT; ++t) {
        const float old = m_run[t] == -INFINITY ? 0.f : m_run[t];
        const float mnew = fmaxf(m_run[t], group4_max(mx[t]) + old);
        const float alpha = fast_exp2(m_run[t] - mnew), sh = old - mnew;
        m_run[t] = mnew;
        l_run[t] *= alpha;
#pragma unroll
        for (int d = 0; d < DT; ++d) acc[t][d] *= alpha;
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
          for (int h = 0; h < 2; ++h) sacc[j][t][h] += sh;
        nm4[t] = f32x4{-mnew, -mnew, -mnew, -mnew};
      }
    }
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      Frag pf[QT];
#pragma unroll
      for (int t = 0; t < QT; ++t) {
        float x[8];
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
          for (int i = 0; i < 4; ++i) x[4 * h + i] = fast_exp2(sacc[j][t][h][i]);
        l_run[t] += ((x[0] + x[1]) + (x[2] + x[3])) + ((x[4] + x[5]) + (x[6] + x[7]));
        pf[t] = C::make(x);
      }
#pragma unroll
      for (int d = 0; d < DT; ++d) {
        const Frag a = C::tr(v + to[d] + 32 * j * D, v + to[d] + (32 * j + 16) * D);
#pragma unroll
        for (int t = 0; t < QT; ++t) acc[t][d] = C::mma(a, pf[t], acc[t][d]);
      }
    }
  };
  // last (a type, or a run-time value): no stage follows, keys may end in this one
  auto stage = [&](auto last, int st, const S* __restrict__ k, const S* __restrict__ v, S* __restrict__ kn, S* __restrict__ vn)
      __attribute__((always_inline)) {
    stage_barrier();
    if (!last) {
      srcK.load(kn, wave, (st + 1) * SR);
      srcV.load(vn, wave, (st + 1) * SR);
    }
    if (active) {
      const int left = N - st * SR;   // keys of this stage (uniform)
      const bool tail = !std::is_same_v<decltype(last), std::false_type> && left < SR;
      const int lim = left - 4 * lg;
      blocks(k, v, tail, lim);
    }
  };
  // The last stage apart, so that the others hold no test of the plane's end.
  // Measured (us, tests in every stage / apart): 12 planes of N 1025, QT 1 13.9
  // / 13.4; D 32, N 3970, 10 planes 44.1 / 42.9; D 128, N 4096 212 / 209; but D
  // 64, QT 2, N 577, 384 planes 58.7 / 59.4, which keeps the tests.
  int st = 0;
  if constexpr (D == 64 && QT == 2) {
    for (; st + 1 < ns; st += 2) {
      stage(st + 1 >= ns, st, sK0, sV0, sK1, sV1);
      stage(st + 2 >= ns, st + 1, sK1, sV1, sK0, sV0);
    }
    if (st < ns) stage(st + 1 >= ns, st, sK0, sV0, sK1, sV1);
  } else {
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
  }

  // lane holds O[row][16d + 4lg + (0..3)]; lane groups lg and lg^1 trade
  // halves so that each lane stores 8 consecutive channels; rows >= N drop
  const auto rO = rsrc(p.o, p.so);
  const auto rL = make_rsrc(p.lse + prow, (unsigned)N * 4u);
#pragma unroll
  for (int t = 0; t < QT; ++t) {
    const int row = row0 + 16 * t;
    const float l = group4_sum(l_run[t]);
    const float inv = __builtin_amdgcn_rcpf(l);
#pragma unroll
    for (int d0 = 0; d0 < DT; d0 += 2) {
      u32x2 w[2];
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        typedef S s4 __attribute__((ext_vector_type(4)));
        s4 a;
#pragma unroll
        for (int r = 0; r < 4; ++r) a[r] = (S)(acc[t][d0 + j][r] * inv);
        __builtin_memcpy(&w[j], &a, 8);
      }
      u32x4 x;
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        const auto r = __builtin_amdgcn_permlane16_swap(w[0][k], w[1][k], false, false);
        x[k] = r[0];
        x[2 + k] = r[1];
      }
      buf_store16(x, rO, (unsigned)((row * (int)p.so[2] + 16 * (d0 + (lg & 1)) + 4 * (lg & 2)) * 2), 0u);
    }
    // (lanes lg != 0 write past the range)
    __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint((m_run[t] + fast_log2(l)) * kLn2), rL,
                                          (unsigned)(lg == 0 ? row : N) * 4u, 0u, 0);
  }
}

template <typename S, int CT>
static hipError_t khat_launch(const KhatParams& p, int D, hipStream_t st) {
  const int rows = 256 / (D / 8), n_blk = (p.N + rows - 1) / rows;
  const int n_wg = (int)khat_blocks(p.planes, p.N, D);
  auto kern = D == 128 ? stream_khat_kernel<S, CT, 128> : D == 64 ? stream_khat_kernel<S, CT, 64> : stream_khat_kernel<S, CT, 32>;
  hipLaunchKernelGGL(kern, dim3(n_wg), dim3(256), 0, st, p, n_blk);
  return hipGetLastError();
}
hipError_t launch_stream_khat(const KhatParams& p, int ct, int D, hipStream_t st) {
  return ct == DT_BF16 ? khat_launch<bf16, DT_BF16>(p, D, st) : khat_launch<f16, DT_F16>(p, D, st);
}

template <typename S, int CT, int D>
static hipError_t fwd_stream_launch(const FwdParams& p0, const void* khat, hipStream_t st) {
  FwdParams p = p0;
  const int planes = p.B * p.H;
  const int rows = stream_rows(planes, p.N, D, false);
  p.n_blk = (p.N + rows - 1) / rows;
  p.n_wg = planes * p.n_blk;
  auto kern = rows < kStreamTileRows ? fwd_stream_kernel<S, CT, D, 1> : fwd_stream_kernel<S, CT, D, 2>;
  hipLaunchKernelGGL(kern, dim3(p.n_wg), dim3(kStreamNW * 64), 0, st, p, static_cast<const S*>(khat));
  return hipGetLastError();
}
hipError_t launch_fwd_stream(const FwdParams& p, const void* khat, int io, int D, hipStream_t st) {
  if (io == DT_BF16) return D == 64 ? fwd_stream_launch<bf16, DT_BF16, 64>(p, khat, st) : fwd_stream_launch<bf16, DT_BF16, 32>(p, khat, st);
  return D == 128 ? fwd_stream_launch<f16, DT_F16, 128>(p, khat, st)
         : D == 64 ? fwd_stream_launch<f16, DT_F16, 64>(p, khat, st) : fwd_stream_launch<f16, DT_F16, 32>(p, khat, st);
}

}  // namespace farope
