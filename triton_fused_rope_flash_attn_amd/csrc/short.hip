// Short planes: forward and backward with the whole other side of a plane in
// LDS (head_dim 32 or 64, N <= 256, vector access).
//
// Reference behaviour followed ("fa_rope_full .py"): _attn_fwd (FA:91-315),
// delta (FA:325-357), _attn_bwd_dk_dv_rope (FA:374-691), _attn_bwd_dq_rope
// (FA:708-1009); the CLS row bypasses the rotation.
//
// A workgroup is 4 waves of 16 rows each: 64 query rows (forward, dQ) or 64 key
// rows (dK/dV) of one plane.  It loads every row of the other side with all
// loads in flight at once, rotates them into LDS, and after one barrier
// computes without another.  The backward's dQ and dK/dV workgroups form their
// own delta and rotations and depend on nothing but the inputs, so they share
// one launch.
//
// For calls that the persistent kernels leave the chip idle with: few planes
// (those give a plane to one wave or one workgroup), or planes far shorter
// than their 256-row tiles.  A small call is bound by one round of memory
// latency and the LDS latencies after it (12 planes of 197 rows, D 64, bf16:
// forward 22.6 -> 7.2 us, backward 16.9 -> 9.2), a large one by memory
// (4096 planes of 64 rows, D 32: forward 42 -> 13.8 us for 67 MB, backward 75 ->
// 34 us for 134 MB).  fp32 compute stages the bf16 hi / lo parts of its operands
// once, where the general kernels split every fragment again after each LDS
// read (16 planes of 197 rows: forward 26 -> 9.9 us, backward 54.7 -> 15.6).
#include <type_traits>

#include "common.h"
#include "params.h"
#include "stream.h"

namespace farope {

namespace {
constexpr int kShortNW = 4;
constexpr int kShortRows = 16 * kShortNW;   // rows of a workgroup
static_assert(kShortRows == kShortTileRows && 64 * kShortNW == kShortThreads, "");
}  // namespace

// Staged operands: 16-bit compute keeps one tile of its type; fp32 compute
// (every operand split into bf16 hi + lo, see Comp<DT_F32>) keeps the two
// parts as two bf16 tiles, split once where they are staged, so that their
// fragments and transposed fragments are plain LDS reads.
template <int CT, int ROWS, int D> struct Staged {
  using C = Comp<CT>;
  using Frag = typename C::Frag;
  static constexpr bool kSplit = CT == DT_F32;
  using S = std::conditional_t<kSplit, bf16, typename C::S>;
  static constexpr int kLo = ROWS * D;                    // offset of the lo tile
  static constexpr int kElems = (kSplit ? 2 : 1) * ROWS * D;
  static __device__ __forceinline__ void put8(S* p, const float (&x)[8]) {
    if constexpr (kSplit) {
      const Frag f = C::make(x);
      *reinterpret_cast<bf16x8*>(p) = f.h;
      *reinterpret_cast<bf16x8*>(p + kLo) = f.l;
    } else {
      C::put8(p, x);
    }
  }
  static __device__ __forceinline__ Frag lds(const S* p) {
    if constexpr (kSplit) {
      Frag f;
      f.h = *reinterpret_cast<const bf16x8*>(p);
      f.l = *reinterpret_cast<const bf16x8*>(p + kLo);
      return f;
    } else {
      return C::lds(p);
    }
  }
  static __device__ __forceinline__ Frag tr(const S* p0, const S* p1) {
    if constexpr (kSplit) {
      Frag f;
      f.h = Comp<DT_BF16>::tr(p0, p1).v;
      f.l = Comp<DT_BF16>::tr(p0 + kLo, p1 + kLo).v;
      return f;
    } else {
      return C::tr(p0, p1);
    }
  }
};

// Lane sum over the D/8 consecutive lanes that hold one row.
template <int D> __device__ __forceinline__ float row_sum(float x) {
  x += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0xB1, 0xF, 0xF, false));
  x += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x4E, 0xF, 0xF, false));
  if constexpr (D == 64) x += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x141, 0xF, 0xF, false));
  return x;
}

// One plane of a tensor: descriptor over rows 0 .. N-1 (rows >= N read 0,
// stores to them are dropped) and its row stride in bytes.
template <typename IO, int D> struct PlaneIo {
  __amdgpu_buffer_rsrc_t rs;
  unsigned row_b;
  __device__ __forceinline__ PlaneIo(const void* b, const int64_t* st, int bb, int hh, int N)
      : rs(make_rsrc(static_cast<const IO*>(b) + bb * st[0] + hh * st[1], (unsigned)(((int64_t)(N - 1) * st[2] + D) * sizeof(IO)))),
        row_b((unsigned)((int)st[2] * (int)sizeof(IO))) {}
  __device__ __forceinline__ Raw8<IO> load(int row, int c0) const {
    return buf_load8<IO>(rs, (unsigned)row * row_b + (unsigned)(c0 * (int)sizeof(IO)), 0u);
  }
};
// cos / sin of the 4 pairs from channel c0 on of table row `row` (past the table: 0).
struct TabIo {
  __amdgpu_buffer_rsrc_t rs;
  int shift;
  template <int D> __device__ __forceinline__ void load(int row, int c0, float (&cs)[8]) const {
    const unsigned to = (unsigned)(((row + shift) * D + c0) * 4);
    const u32x4 a = __builtin_amdgcn_raw_buffer_load_b128(rs, to, 0u, 0);
    const u32x4 b = __builtin_amdgcn_raw_buffer_load_b128(rs, to + 16u, 0u, 0);
    __builtin_memcpy(cs, &a, 16);
    __builtin_memcpy(cs + 4, &b, 16);
  }
};
__device__ __forceinline__ TabIo tab_io(const float* rope, int N, int has_cls, int D) {
  return TabIo{make_rsrc(rope, (unsigned)((N + 1 - has_cls) * D * 4)), 1 - has_cls};
}

// Stage rows 0 .. of two tensors of the plane: A rotated (times ascale), B as
// it is.  nd: with O, minus the row sums of B * O too (delta).
template <typename IO, int CT, int D, int NB, typename S>
__device__ __forceinline__ void stage_plane(const PlaneIo<IO, D>& A, const PlaneIo<IO, D>& B, const PlaneIo<IO, D>* O, const TabIo& T,
                                            float ascale, int N, int tid, S* sA, S* sB, float* nd) {
  using L = Staged<CT, 32 * NB, D>;
  constexpr int CPR = D / 8, NT = 64 * kShortNW, UNITS = 32 * NB * CPR;
  static_assert(UNITS % NT == 0, "every thread stages whole units");
  constexpr int U = UNITS / NT < 4 ? UNITS / NT : 4;   // units of a thread in flight
#pragma unroll
  for (int u0 = 0; u0 < UNITS; u0 += U * NT) {
    if (u0 / CPR >= N) break;   // uniform
    Raw8<IO> a[U], b[U], o[U];
    float cs[U][8];
#pragma unroll
    for (int i = 0; i < U; ++i) {
      const int u = u0 + i * NT + tid, row = u / CPR, c0 = 8 * (u % CPR);
      a[i] = A.load(row, c0);
      T.load<D>(row, c0, cs[i]);
      b[i] = B.load(row, c0);
      if (O) o[i] = O->load(row, c0);
    }
#pragma unroll
    for (int i = 0; i < U; ++i) {
      const int u = u0 + i * NT + tid, row = u / CPR, c0 = 8 * (u % CPR);
      float x[8];
      unpack8(a[i], x);
      rope_rotate8(x, cs[i]);
#pragma unroll
      for (int e = 0; e < 8; ++e) x[e] *= ascale;
      L::put8(sA + swz<D>(row, c0), x);
      if constexpr (std::is_same<IO, S>::value) {
        *reinterpret_cast<typename Raw8<IO>::vec*>(sB + swz<D>(row, c0)) = b[i].v;
      } else {
        float y[8];
        unpack8(b[i], y);
        L::put8(sB + swz<D>(row, c0), y);
      }
      if (O) {
        const float d = row_sum<D>(dot8(b[i], o[i], 0.f));
        if (c0 == 0) nd[row] = -d;
      }
    }
  }
}

// This lane's operand fragments of row `row` (channels 32s + 8lg ..), rotated and scaled, or as stored.
template <typename IO, int CT, int D>
__device__ __forceinline__ void own_rows(const PlaneIo<IO, D>& A, const PlaneIo<IO, D>& B, const TabIo& T, float ascale, int row,
                                         int lg, typename Comp<CT>::Frag (&fa)[D / 32], typename Comp<CT>::Frag (&fb)[D / 32],
                                         Raw8<IO> (&rb)[D / 32]) {
  constexpr int KS = D / 32;
  Raw8<IO> a[KS];
  float cs[KS][8];
#pragma unroll
  for (int s = 0; s < KS; ++s) {
    a[s] = A.load(row, 32 * s + 8 * lg);
    rb[s] = B.load(row, 32 * s + 8 * lg);
    T.load<D>(row, 32 * s + 8 * lg, cs[s]);
  }
#pragma unroll
  for (int s = 0; s < KS; ++s) {
    float x[8], y[8];
    unpack8(a[s], x);
    rope_rotate8(x, cs[s]);
#pragma unroll
    for (int e = 0; e < 8; ++e) x[e] *= ascale;
    fa[s] = Comp<CT>::make(x);
    unpack8(rb[s], y);
    fb[s] = Comp<CT>::make(y);
  }
}

// Rows of a 16-row subtile to memory: lane holds channels 16d + 4lg + (0..3)
// of its row.  rot: rotated back by the table first, times scale.
template <typename IO, int D, bool ROT>
__device__ __forceinline__ void put_rows(const PlaneIo<IO, D>& out, const TabIo& T, const f32x4 (&acc)[D / 16], float scale, int row,
                                         int lg) {
  constexpr int DT = D / 16;
#pragma unroll
  for (int d0 = 0; d0 < DT; d0 += 2) {
    float g[2][4];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int d = d0 + j;
      if constexpr (ROT) {
        const u32x4 t = __builtin_amdgcn_raw_buffer_load_b128(T.rs, (unsigned)(((row + T.shift) * D + 16 * d + 4 * lg) * 4), 0u, 0);
#pragma unroll
        for (int r = 0; r < 2; ++r) {
          const float e = acc[d][2 * r] * scale, o = acc[d][2 * r + 1] * scale;
          const float c = __uint_as_float(t[2 * r]), sn = __uint_as_float(t[2 * r + 1]);
          g[j][2 * r] = e * c + o * sn;
          g[j][2 * r + 1] = o * c - e * sn;
        }
      } else {
#pragma unroll
        for (int r = 0; r < 4; ++r) g[j][r] = acc[d][r] * scale;
      }
    }
    if constexpr (sizeof(IO) == 2) {
      typedef IO io4 __attribute__((ext_vector_type(4)));
      u32x2 w[2];
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        io4 a;
#pragma unroll
        for (int r = 0; r < 4; ++r) a[r] = (IO)g[j][r];
        __builtin_memcpy(&w[j], &a, 8);
      }
      u32x4 x;
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        const auto r = __builtin_amdgcn_permlane16_swap(w[0][k], w[1][k], false, false);
        x[k] = r[0];
        x[2 + k] = r[1];
      }
      buf_store16(x, out.rs, (unsigned)row * out.row_b + (unsigned)((16 * (d0 + (lg & 1)) + 4 * (lg & 2)) * 2), 0u);
    } else {
#pragma unroll
      for (int j = 0; j < 2; ++j)
        buf_store4<IO>(out.rs, (unsigned)row * out.row_b + (unsigned)((16 * (d0 + j) + 4 * lg) * 4), 0u, g[j]);
    }
  }
}

// ---------------------------------------------------------------------------
// Forward: NB 32-key blocks (N <= 32 NB).  A row's logits are all in registers
// at once (transposed products as in the other forwards: the lane holds keys
// 32j + 16h + 4lg + i of its query), so the softmax is single-pass.
// ---------------------------------------------------------------------------
template <typename IO, int CT, int D, int NB>
__global__ void __launch_bounds__(64 * kShortNW) fwd_short_kernel(const FwdParams p) {
  using C = Comp<CT>;
  using L = Staged<CT, 32 * NB, D>;
  using S = typename L::S;
  using Frag = typename C::Frag;
  constexpr int KS = D / 32, DT = D / 16;
  __shared__ __attribute__((aligned(16))) S sK[L::kElems], sV[L::kElems];
  const int N = p.N;
  const int tile = xcd_remap(block_id(), p.n_wg);
  const int plane = tile / p.n_blk, qblk = tile - plane * p.n_blk;
  const int bb = plane / p.H, hh = plane - bb * p.H;
  const int tid = thread_id();
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int lr = lane & 15, lg = lane >> 4;
  const TabIo T = tab_io(p.rope, N, p.has_cls, D);
  const PlaneIo<IO, D> Q(p.q, p.sq, bb, hh, N), K(p.k, p.sk, bb, hh, N), V(p.v, p.sv, bb, hh, N), O(p.o, p.so, bb, hh, N);
  const int row = qblk * kShortRows + wave * 16 + lr;

  Raw8<IO> q[KS];
  float qcs[KS][8];
#pragma unroll
  for (int s = 0; s < KS; ++s) {
    q[s] = Q.load(row, 32 * s + 8 * lg);
    T.load<D>(row, 32 * s + 8 * lg, qcs[s]);
  }
  stage_plane<IO, CT, D, NB>(K, V, nullptr, T, p.scale_log2, N, tid, sK, sV, nullptr);
  Frag qf[KS];
#pragma unroll
  for (int s = 0; s < KS; ++s) {
    float x[8];
    unpack8(q[s], x);
    rope_rotate8(x, qcs[s]);
    qf[s] = C::make(x);
  }
  lds_barrier();
  if (row - lr >= N) return;   // wave-uniform; no barrier follows

  f32x4 sacc[NB][2];
  float mx = -INFINITY;
#pragma unroll
  for (int j = 0; j < NB; ++j) {
#pragma unroll
    for (int h = 0; h < 2; ++h) sacc[j][h] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (32 * j < N) {   // uniform
#pragma unroll
      for (int s = 0; s < KS; ++s)
#pragma unroll
        for (int h = 0; h < 2; ++h)
          sacc[j][h] = C::mma(L::lds(sK + swz<D>(lr, 32 * s + 8 * lg) + (32 * j + 16 * h) * D), qf[s], sacc[j][h]);
    }
    if (32 * j + 32 > N) {   // uniform: keys >= N
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int i = 0; i < 4; ++i) sacc[j][h][i] = 32 * j + 16 * h + 4 * lg + i < N ? sacc[j][h][i] : -INFINITY;
    }
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int i = 0; i < 4; ++i) mx = fmaxf(mx, sacc[j][h][i]);
  }
  mx = group4_max(mx);
  float l = 0.f;
  f32x4 acc[DT];
#pragma unroll
  for (int d = 0; d < DT; ++d) acc[d] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int j = 0; j < NB; ++j) {
    if (32 * j >= N) break;   // uniform
    float pv[8];
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        pv[4 * h + i] = fast_exp2(sacc[j][h][i] - mx);
        l += pv[4 * h + i];
      }
    const Frag pf = C::make(pv);
#pragma unroll
    for (int d = 0; d < DT; ++d) {
      const S* v = sV + swz<D>(4 * lg + (lr >> 2), 16 * d + 4 * (lr & 3)) + 32 * j * D;
      acc[d] = C::mma(L::tr(v, v + 16 * D), pf, acc[d]);
    }
  }
  l = group4_sum(l);
  put_rows<IO, D, false>(O, T, acc, __builtin_amdgcn_rcpf(l), row, lg);
  const auto rL = make_rsrc(p.lse + (int64_t)plane * N, (unsigned)N * 4u);
  // (lanes lg != 0 write past the range)
  __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint((mx + fast_log2(l)) * kLn2), rL, (unsigned)(lg == 0 ? row : N) * 4u, 0u, 0);
}

// ---------------------------------------------------------------------------
// Backward: n_blk dQ workgroups, then n_blk dK/dV workgroups, of each plane.
// ---------------------------------------------------------------------------
template <typename IO, int CT, int D, int NB>
__global__ void __launch_bounds__(64 * kShortNW) bwd_short_kernel(const BwdParams p) {
  using C = Comp<CT>;
  using L = Staged<CT, 32 * NB, D>;
  using S = typename L::S;
  using Frag = typename C::Frag;
  constexpr int KS = D / 32, DT = D / 16;
  __shared__ __attribute__((aligned(16))) S sA[L::kElems], sB[L::kElems];   // K-hat, V or Q-hat, dO
  __shared__ __attribute__((aligned(16))) float sNl[32 * NB], sNd[32 * NB];     // dK/dV: -LSE2, -delta
  const int N = p.N;
  const int tile = xcd_remap(block_id(), p.n_wg);
  const int plane = tile / (2 * p.n_blk), r = tile - plane * 2 * p.n_blk;
  const bool keys = r >= p.n_blk;   // uniform
  const int bb = plane / p.H, hh = plane - bb * p.H;
  const int tid = thread_id();
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int lr = lane & 15, lg = lane >> 4;
  const TabIo T = tab_io(p.rope, N, p.has_cls, D);
  const PlaneIo<IO, D> Q(p.q, p.sq, bb, hh, N), K(p.k, p.sk, bb, hh, N), V(p.v, p.sv, bb, hh, N), O(p.o, p.so, bb, hh, N),
      G(p.dout, p.sdo, bb, hh, N);
  const auto rL = make_rsrc(p.lse + (int64_t)plane * N, (unsigned)N * 4u);
  const int row = (r - (keys ? p.n_blk : 0)) * kShortRows + wave * 16 + lr;
  // lane offsets of the operand reads in 32-row block 0 (the swizzle has period 16)
  int ao[KS], to[DT];
#pragma unroll
  for (int s = 0; s < KS; ++s) ao[s] = swz<D>(lr, 32 * s + 8 * lg);
#pragma unroll
  for (int d = 0; d < DT; ++d) to[d] = swz<D>(4 * lg + (lr >> 2), 16 * d + 4 * (lr & 3));

  Frag fa[KS], fb[KS];   // Q-hat, dO or K-hat, V of the lane's row
  Raw8<IO> rb[KS];
  if (!keys) {
    Raw8<IO> o[KS];
#pragma unroll
    for (int s = 0; s < KS; ++s) o[s] = O.load(row, 32 * s + 8 * lg);
    const float ls = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rL, (unsigned)row * 4u, 0u, 0));
    own_rows<IO, CT, D>(Q, G, T, 1.f, row, lg, fa, fb, rb);
    float ds = 0.f;
#pragma unroll
    for (int s = 0; s < KS; ++s) ds = dot8(rb[s], o[s], ds);
    const float nd = -group4_sum(ds), nl = -ls * kLog2e;
    stage_plane<IO, CT, D, NB>(K, V, nullptr, T, p.scale_log2, N, tid, sA, sB, nullptr);
    lds_barrier();
    if (row - lr >= N) return;   // wave-uniform; no barrier follows
    f32x4 acc[DT];
#pragma unroll
    for (int d = 0; d < DT; ++d) acc[d] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 2
    for (int j = 0; j < NB; ++j) {
      if (32 * j >= N) break;   // uniform
      const S *k = sA + 32 * j * D, *v = sB + 32 * j * D;
      f32x4 sacc[2], pacc[2];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        sacc[h] = f32x4{nl, nl, nl, nl};
        pacc[h] = f32x4{nd, nd, nd, nd};
#pragma unroll
        for (int s = 0; s < KS; ++s) {
          sacc[h] = C::mma(L::lds(k + ao[s] + 16 * h * D), fa[s], sacc[h]);
          pacc[h] = C::mma(L::lds(v + ao[s] + 16 * h * D), fb[s], pacc[h]);
        }
      }
      // keys >= N: zero K-hat and V rows; P is clamped to [0, 1] and their dS
      // meets zero rows
      float dsv[8];
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int i = 0; i < 4; ++i)
          dsv[4 * h + i] = __builtin_amdgcn_fmed3f(fast_exp2(sacc[h][i]), 0.f, 1.f) * pacc[h][i];
      const Frag df = C::make(dsv);
#pragma unroll
      for (int d = 0; d < DT; ++d) acc[d] = C::mma(L::tr(k + to[d], k + to[d] + 16 * D), df, acc[d]);
    }
    put_rows<IO, D, true>(PlaneIo<IO, D>(p.dq, p.sdq, bb, hh, N), T, acc, p.scale / p.scale_log2, row, lg);
    return;
  }

  own_rows<IO, CT, D>(K, V, T, p.scale_log2, row, lg, fa, fb, rb);
  // P needs no clamp here (which would turn a NaN into 0): keys >= N of a lane
  // only reach rows that are never stored.
  // -LSE2 of the staged rows; -inf for rows >= N, whose P is then 0.  (Their dO
  // rows read 0 only where dO's rows do not overlap: with a row stride of 0, as
  // the backward of a sum over the tokens gives it, they read the one real row.)
  if (tid < 32 * NB) {
    const float ls = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rL, (unsigned)tid * 4u, 0u, 0));
    sNl[tid] = tid < N ? -kLog2e * ls : -INFINITY;
  }
  stage_plane<IO, CT, D, NB>(Q, G, &O, T, 1.f, N, tid, sA, sB, sNd);
  lds_barrier();
  if (row - lr >= N) return;   // wave-uniform; no barrier follows
  f32x4 dk[DT], dv[DT];
#pragma unroll
  for (int d = 0; d < DT; ++d) dk[d] = dv[d] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 2
  for (int j = 0; j < NB; ++j) {
    if (32 * j >= N) break;   // uniform
    const S *q = sA + 32 * j * D, *g = sB + 32 * j * D;
    float pv[8], dsv[8];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      f32x4 sacc = *reinterpret_cast<const f32x4*>(sNl + 32 * j + 16 * h + 4 * lg);
      f32x4 pacc = *reinterpret_cast<const f32x4*>(sNd + 32 * j + 16 * h + 4 * lg);
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        sacc = C::mma(L::lds(q + ao[s] + 16 * h * D), fa[s], sacc);
        pacc = C::mma(L::lds(g + ao[s] + 16 * h * D), fb[s], pacc);
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        pv[4 * h + i] = fast_exp2(sacc[i]);
        dsv[4 * h + i] = pv[4 * h + i] * pacc[i];
      }
    }
    const Frag pf = C::make(pv), df = C::make(dsv);
#pragma unroll
    for (int d = 0; d < DT; ++d) {
      dv[d] = C::mma(L::tr(g + to[d], g + to[d] + 16 * D), pf, dv[d]);
      dk[d] = C::mma(L::tr(q + to[d], q + to[d] + 16 * D), df, dk[d]);
    }
  }
  put_rows<IO, D, false>(PlaneIo<IO, D>(p.dv, p.sdv, bb, hh, N), T, dv, 1.f, row, lg);
  put_rows<IO, D, true>(PlaneIo<IO, D>(p.dk, p.sdk, bb, hh, N), T, dk, p.scale, row, lg);
}

// ---------------------------------------------------------------------------
// Launch.
// ---------------------------------------------------------------------------
template <typename P, typename F1, typename F2, typename F3>
static hipError_t short_pick(P p, int per_plane, F1 k2, F2 k4, F3 k8, hipStream_t st) {
  p.n_blk = (p.N + kShortRows - 1) / kShortRows;
  p.n_wg = p.B * p.H * p.n_blk * per_plane;
  auto kern = p.N <= 64 ? k2 : p.N <= 128 ? k4 : k8;
  hipLaunchKernelGGL(kern, dim3(p.n_wg), dim3(64 * kShortNW), 0, st, p);
  return hipGetLastError();
}
template <typename IO, int CT, int D> static hipError_t fwd_short_d(const FwdParams& p, hipStream_t st) {
  return short_pick(p, 1, fwd_short_kernel<IO, CT, D, 2>, fwd_short_kernel<IO, CT, D, 4>, fwd_short_kernel<IO, CT, D, 8>, st);
}
template <typename IO, int CT, int D> static hipError_t bwd_short_d(const BwdParams& p, hipStream_t st) {
  return short_pick(p, 2, bwd_short_kernel<IO, CT, D, 2>, bwd_short_kernel<IO, CT, D, 4>, bwd_short_kernel<IO, CT, D, 8>, st);
}
#define FAROPE_SHORT(fn)                                                                           \
  if (ct == DT_F32) return D == 64 ? fn<float, DT_F32, 64>(p, st) : fn<float, DT_F32, 32>(p, st);  \
  if (ct == DT_BF16) {                                                                             \
    if (io == DT_BF16) return D == 64 ? fn<bf16, DT_BF16, 64>(p, st) : fn<bf16, DT_BF16, 32>(p, st); \
    return D == 64 ? fn<float, DT_BF16, 64>(p, st) : fn<float, DT_BF16, 32>(p, st);                \
  }                                                                                                \
  if (io == DT_F16) return D == 64 ? fn<f16, DT_F16, 64>(p, st) : fn<f16, DT_F16, 32>(p, st);      \
  return D == 64 ? fn<float, DT_F16, 64>(p, st) : fn<float, DT_F16, 32>(p, st);
hipError_t launch_fwd_short(const FwdParams& p, int io, int ct, int D, hipStream_t st) { FAROPE_SHORT(fwd_short_d) }
hipError_t launch_bwd_short(const BwdParams& p, int io, int ct, int D, hipStream_t st) { FAROPE_SHORT(bwd_short_d) }

}  // namespace farope
