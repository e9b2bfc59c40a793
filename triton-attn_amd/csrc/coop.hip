// 16-bit attention for launches with few rows on gfx950 (the reference's src/tattn/kernels.py:57-321):
// the waves of a workgroup split the dimension that is summed over, not only the rows.
//
// The block kernels give every 32-row tile to one wave, which walks all steps of the other
// dimension. With few tiles (ZH * N / 32 below the chip's wave slots) most SIMDs idle while each
// wave runs N / 32 dependent steps. Here a workgroup of NW = RW * CS waves owns RW row tiles; in one
// step it stages CS tiles of the other dimension, wave (rw, cs) works on tile cs of that step for row
// tile rw, and the CS partial results of a row tile are added through LDS at the end (the forward's
// with their own running max: O = sum_c 2^(m_c - m) O_c, l likewise). No workspace, no second launch.
//
// Measured against the block kernels (warm, us, forward / dQ / dK,dV; one MI355X, fp16 unless said):
//   1 x 16 x 2,048 x 64 causal (bf16)  49 -> 18 / 32 -> 23 / 57 -> 31     4 x 4,096 x 64: 110 -> 26 / 79 -> 31 / 106 -> 45
//   1 x 1 x 13,184 x 64 causal  212 -> 65 / 203 -> 67 / 318 -> 105      4 x 4,096 x 128: 66 -> 50 / 86 -> 60 / -
//   1 x 1 x 16,196 x 32 causal (bf16)  208 -> 60 / 194 -> 60 / 248 -> 95
// On a full chip the block kernels stay ahead at head dim 64 (16 x 8,192: 263 against 329 us): they
// pipeline a wave's matrix and vector work and stage every tile once for more rows.
//
// A step: LDS DMA (buffer_load ... lds, swizzled rows in perm32 order as in bwd_pipe.h) of the next
// step's tiles into the other of two stages, the step's MFMAs and elementwise work, one barrier.
// Waves of one SIMD overlap each other's matrix and vector work; nothing is pipelined inside a wave,
// which keeps the forward within 128 registers (four waves per SIMD).
#include <algorithm>
#include <type_traits>

#include "bwd_pipe.h"
#include "common.h"
#include "launch.h"

namespace tattn {

namespace {

template <int D, int NW, int CS>
struct Ring {
  static constexpr int RB = Swz<D>::RB, TILE = 32 * RB, PIECES = TILE / 1024;
  static constexpr int HALF = CS * TILE;       // bytes of one tensor's tiles
  static constexpr int STAGE = 2 * HALF;
  static constexpr int PW = STAGE / 1024 / NW;  // 1 KB DMA pieces per wave and step
  static_assert(PW >= 1 && PW * NW * 1024 == STAGE && NW % 2 == 0, "whole pieces, one tensor per wave");
};

// One wave's share of a step: pieces wave * PW + i of [tensor][tile][piece]; the first half of the
// waves loads the first tensor, the other half the second.
template <int D, int NW, int CS>
struct Loader {
  using R = Ring<D, NW, CS>;
  uint32_t go[R::PW];
  __amdgpu_buffer_rsrc_t rs;
  uint32_t step_bytes;
  int base;
  __device__ __forceinline__ void init(__amdgpu_buffer_rsrc_t a, int64_t sa, __amdgpu_buffer_rsrc_t b, int64_t sb,
                                       int wu, int lane) {
    const bool second = wu >= NW / 2;
    rs = second ? b : a;
    const int64_t st = second ? sb : sa;
    step_bytes = uniform32((uint32_t)(st * (64 * CS)));
    base = wu * R::PW * 1024;
#pragma unroll
    for (int i = 0; i < R::PW; ++i) {
      const int g = (wu * R::PW + i) % (CS * R::PIECES);
      const int j = 64 * (g % R::PIECES) + lane;
      constexpr int CPR = R::RB / 16;
      const int row = j / CPR, cc = ((j % CPR) ^ Swz<D>::f(row)) & (D / 8 - 1);
      go[i] = (uint32_t)((32 * (g / R::PIECES) + perm32(row)) * st * 2 + cc * 16);
    }
  }
  // Rows past the end of the slice read as zero.
  __device__ __forceinline__ void issue(char* stage, int step) const {
    const uint32_t so = (uint32_t)step * step_bytes;
#pragma unroll
    for (int i = 0; i < R::PW; ++i)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (TATTN_LDS void*)(stage + base + 1024 * i), 16, (int)(go[i] + so), 0, 0, 0);
  }
};

// Operand addresses within one tile at byte `base`: natural rows, and the transposed reads of 16-row
// slice 0 (the swizzle depends on a row's index mod 16, so slice 1 is a constant further).
template <int D>
struct OpAddr {
  static constexpr int NSD = D / 16, DT = (D + 31) / 32;
  int nat[NSD], lo[DT], hi[DT];
  __device__ __forceinline__ void init(int base, int lane) {
    const int l32 = lane & 31, h2 = lane >> 5;
#pragma unroll
    for (int s = 0; s < NSD; ++s) nat[s] = base + Swz<D>::addr(l32, (16 * s + 8 * h2) * 2);
#pragma unroll
    for (int u = 0; u < DT; ++u) {
      tr_addrs<D>(0, u, lane, lo[u], hi[u]);
      lo[u] += base;
      hi[u] += base;
    }
  }
  template <typename T>
  __device__ __forceinline__ typename H16<T>::V8 tr(const char* st, int sl, int u) const {
    return tr_pair<T>(st + 16 * sl * Swz<D>::RB, lo[u], hi[u]);
  }
};

// The raw score of a hidden key: its scaled value is -inf, so its probability is 0 (the launchers take
// scale 0, where no such score exists, elsewhere).
__device__ __forceinline__ float hidden_score(float c) { return c < 0.0f ? __builtin_inff() : -__builtin_inff(); }

// Everything this wave has in flight has landed, its LDS reads are done, then the barrier.
__device__ __forceinline__ void landed_barrier() {
  __builtin_amdgcn_s_waitcnt(0x0070);  // vmcnt(0), lgkmcnt(0)
  __atomic_signal_fence(__ATOMIC_SEQ_CST);
  __builtin_amdgcn_s_barrier();
  __atomic_signal_fence(__ATOMIC_SEQ_CST);
}

// Workgroup -> (slice, block), longest causal blocks first (grouped per XCD without a mask).
__device__ __forceinline__ BlockCoord coop_coord(int zhs, int nblk, bool causal) { return block_coord(zhs, nblk, !causal); }

// ---- forward ---------------------------------------------------------------------------------
template <typename T, int D, int RW, int CS, int OCC, bool CAUSAL>
__global__ __launch_bounds__(RW * CS * 64, OCC) void fwd_coop_kernel(const FwdParams p) {
  using H = H16<T>;
  using V8 = typename H::V8;
  using V4 = typename H::V4;
  using V2 = typename H::V2;
  constexpr int NW = RW * CS, NSD = D / 16, DT = (D + 31) / 32;
  using R = Ring<D, NW, CS>;
  // Two arrays: a DMA into one stage does not alias reads of the other.
  __shared__ __attribute__((aligned(1024))) char s0[R::STAGE];
  __shared__ __attribute__((aligned(1024))) char s1[R::STAGE];
  __shared__ float red[2][NW][32];

  const int tid = threadIdx.x;
  const int lane = tid & 63, h2 = lane >> 5, l32 = lane & 31;
  const int wu = (int)uniform32((uint32_t)(tid >> 6));
  const int rw = wu / CS, cs = wu % CS;
  const int N = p.N;
  const float c = p.c;
  const BlockCoord bc = coop_coord(p.Z * p.H, p.n_qblocks, CAUSAL);
  const int zh = bc.zh, qb = CAUSAL ? p.n_qblocks - 1 - bc.blk : bc.blk;
  const int ntile = (N + 31) / 32;
  const int qt = qb * RW + rw;  // the wave's row tile
  const int q = 32 * qt + l32;
  const int btiles = CAUSAL ? min(ntile, (qb + 1) * RW) : ntile;   // key tiles the block sees
  const int wtiles = qt >= ntile ? 0 : CAUSAL ? qt + 1 : ntile;     // ... and the wave
  const int nsteps = (btiles + CS - 1) / CS;

  Loader<D, NW, CS> ld;
  ld.init(slice_rsrc((const T*)p.k + slice_off(p.sk, zh, p.H), slice_bytes(N, p.sk[2], D)), p.sk[2],
          slice_rsrc((const T*)p.v + slice_off(p.sv, zh, p.H), slice_bytes(N, p.sv[2], D)), p.sv[2], wu, lane);
  ld.issue(s0, 0);
  V8 qop[NSD];
  {
    const T* src = (const T*)p.q + slice_off(p.sq, zh, p.H) + (int64_t)(q < N ? q : 0) * p.sq[2] + 8 * h2;
#pragma unroll
    for (int s = 0; s < NSD; ++s) {
      const V8 x = *reinterpret_cast<const V8*>(src + 16 * s);
      qop[s] = q < N ? x : V8{};
    }
  }
  OpAddr<D> at;
  at.init(cs * R::TILE, lane);

  const int lim = CAUSAL ? min(q, N - 1) : N - 1;  // last key the lane's row sees
  const float hidden = hidden_score(c);
  float mrow = -__builtin_inff(), lrow = 0.0f;
  f32x16 acc[DT];
#pragma unroll
  for (int u = 0; u < DT; ++u) acc[u] = f32x16{};

  // Raw scores of tile t (staged at `st`, lane addresses `off` bytes away), hidden keys at -inf scaled.
  auto scores = [&](const char* st, int off, int t) __attribute__((always_inline)) {
    f32x16 s = f32x16{};
#pragma unroll
    for (int sd = 0; sd < NSD; ++sd) s = Elt<T>::mfma(lds8<T>(st + (at.nat[sd] + off)), qop[sd], s);
    if (32 * t + 32 > N || (CAUSAL && t == qt)) {
      const int past = lim - 32 * t - 8 * h2;
#pragma unroll
      for (int r = 0; r < 16; ++r) s[r] = 16 * (r >> 3) + (r & 7) > past ? hidden : s[r];
    }
    return s;
  };
  auto row_max = [&](const f32x16& s) __attribute__((always_inline)) {
    float mx = -__builtin_inff();
#pragma unroll
    for (int r = 0; r < 16; ++r) mx = __builtin_fmaxf(mx, s[r] * c);
    return max_halves(mx);
  };
  // Tile t of the wave's row tile, staged in `st`. Probabilities against the running max as it
  // stands (seeded for all waves by tile 0's row max); a lane whose 16 probabilities sum above 2^12 sends
  // the wave through the row max and a rescale, as in fwd_pipe_kernel. Branches are one-sided
  // (state updated first, undone inside): two-sided ones make the allocator hold two copies of it.
  auto tile = [&](const char* st, int t) __attribute__((always_inline)) {
    const f32x16 s = scores(st, 0, t);
    V8 x[2];
    auto probs = [&]() {
      float ps = 0.0f;
#pragma unroll
      for (int sg = 0; sg < 2; ++sg)
#pragma unroll
        for (int i = 0; i < 8; i += 2) {
          const V2 pr = H::pack(fast_exp2(__builtin_fmaf(s[8 * sg + i], c, -mrow)),
                                fast_exp2(__builtin_fmaf(s[8 * sg + i + 1], c, -mrow)));
          ps = H::sum2(pr, ps);
          x[sg][i] = pr[0];
          x[sg][i + 1] = pr[1];
        }
      return ps;
    };
    const float lprev = lrow;
    const float ps = probs();
    lrow += ps;
    if (__builtin_amdgcn_ballot_w64(!(ps <= 4096.0f))) {
      const float cand = row_max(s);
      const float mnew = cand > mrow + kRescaleLog2 ? cand : mrow;
      const float alpha = fast_exp2(mrow - mnew);
      mrow = mnew;
      const float again = probs();
      lrow = lprev * alpha + again;
#pragma unroll
      for (int u = 0; u < DT; ++u) acc[u] *= alpha;
    }
#pragma unroll
    for (int sg = 0; sg < 2; ++sg)
#pragma unroll
      for (int u = 0; u < DT; ++u) {
        V8 va = at.template tr<T>(st + R::HALF, sg, u);
        if (D < 32 && 16 * ((lane >> 4) & 1) >= D) va = V8{};
        acc[u] = Elt<T>::mfma(va, x[sg], acc[u]);
      }
  };
  auto step = [&](int i, char* cur, char* nxt) __attribute__((always_inline)) {
    if (i + 1 < nsteps) ld.issue(nxt, i + 1);
    const int t = i * CS + cs;
    if (t < wtiles) {
      tile(cur, t);
    }
    landed_barrier();
  };
  landed_barrier();
  if (wtiles > 0) mrow = row_max(scores(s0, -cs * R::TILE, 0));
  int i = 0;
  for (; i + 1 < nsteps; i += 2) {
    step(i, s0, s1);
    step(i + 1, s1, s0);
  }
  if (i < nsteps) step(i, s0, s1);

  // Merge the CS partial rows of each row tile (the stages are free: every wave passed the last
  // barrier and no DMA is in flight).
  const float lt = sum_halves(lrow);
  if (h2 == 0) {
    red[0][wu][l32] = mrow;
    red[1][wu][l32] = lt;
  }
  __syncthreads();
  float mall = -__builtin_inff();
#pragma unroll
  for (int k = 0; k < CS; ++k) mall = __builtin_fmaxf(mall, red[0][rw * CS + k][l32]);
  float lall = 0.0f;
#pragma unroll
  for (int k = 0; k < CS; ++k) {
    lall += fast_exp2(red[0][rw * CS + k][l32] - mall) * red[1][rw * CS + k][l32];
  }
  const float wgt = fast_exp2(mrow - mall) / lall;
  constexpr int PART = DT * 16 * 64 * 4;  // bytes of one wave's partial O^T
  constexpr int PER = R::STAGE / PART;    // partials per stage array
  static_assert(2 * PER >= NW, "partials fit the stages");
  auto part = [&](int k) { return (TATTN_LDS float*)(k < PER ? s0 + k * PART : s1 + (k - PER) * PART); };
  {
    TATTN_LDS float* dst = part(wu) + lane;
#pragma unroll
    for (int u = 0; u < DT; ++u)
#pragma unroll
      for (int r = 0; r < 16; ++r) dst[(16 * u + r) * 64] = acc[u][r] * wgt;
  }
  __syncthreads();
  if (q < N) {
    T* orow = (T*)p.o + slice_off(p.so, zh, p.H) + (int64_t)q * p.so[2];
    for (int gr = cs; gr < DT * 4; gr += CS) {  // four consecutive columns per register group
      const int d0 = 8 * gr + 4 * h2;
      if (d0 < D) {
        f32x4 x = f32x4{};
#pragma unroll
        for (int k = 0; k < CS; ++k) {
          const TATTN_LDS float* src = part(rw * CS + k) + lane + 4 * gr * 64;
#pragma unroll
          for (int e = 0; e < 4; ++e) x[e] += src[64 * e];
        }
        V4 y;
#pragma unroll
        for (int e = 0; e < 4; ++e) y[e] = (T)x[e];
        *reinterpret_cast<V4*>(orow + d0) = y;
      }
    }
    if (cs == 0 && h2 == 0 && p.m) p.m[(int64_t)zh * N + q] = mall + __log2f(lall);
  }
}

// ---- dQ --------------------------------------------------------------------------------------
template <typename T, int D, int RW, int CS, int OCC, bool CAUSAL>
__global__ __launch_bounds__(RW * CS * 64, OCC) void dq_coop_kernel(const BwdParams p) {
  using H = H16<T>;
  using V8 = typename H::V8;
  using V4 = typename H::V4;
  using V2 = typename H::V2;
  constexpr int NW = RW * CS, NSD = D / 16, DT = (D + 31) / 32;
  using R = Ring<D, NW, CS>;
  __shared__ __attribute__((aligned(1024))) char s0[R::STAGE];
  __shared__ __attribute__((aligned(1024))) char s1[R::STAGE];

  const int tid = threadIdx.x;
  const int lane = tid & 63, h2 = lane >> 5, l32 = lane & 31;
  const int wu = (int)uniform32((uint32_t)(tid >> 6));
  const int rw = wu / CS, cs = wu % CS;
  const int N = p.N;
  const float c = p.c;
  const BlockCoord bc = coop_coord(p.Z * p.H, p.n_blocks, CAUSAL);
  const int zh = bc.zh, qb = CAUSAL ? p.n_blocks - 1 - bc.blk : bc.blk;
  const int ntile = (N + 31) / 32;
  const int qt = qb * RW + rw;
  const int q = 32 * qt + l32;
  const int btiles = CAUSAL ? min(ntile, (qb + 1) * RW) : ntile;
  const int wtiles = qt >= ntile ? 0 : CAUSAL ? qt + 1 : ntile;
  const int nsteps = (btiles + CS - 1) / CS;
  const int64_t hoff = slice_off(p.s, zh, p.H);
  const int64_t rs = p.s[2];

  Loader<D, NW, CS> ld;
  ld.init(slice_rsrc((const T*)p.k + hoff, slice_bytes(N, rs, D)), rs, slice_rsrc((const T*)p.v + hoff, slice_bytes(N, rs, D)),
          rs, wu, lane);
  ld.issue(s0, 0);
  V8 qop[NSD], dop[NSD];
  const int64_t off = hoff + (int64_t)(q < N ? q : 0) * rs + 8 * h2;
#pragma unroll
  for (int s = 0; s < NSD; ++s) {
    const V8 a = *reinterpret_cast<const V8*>((const T*)p.q + off + 16 * s);
    const V8 b = *reinterpret_cast<const V8*>((const T*)p.dout + off + 16 * s);
    qop[s] = q < N ? a : V8{};
    dop[s] = q < N ? b : V8{};
  }
  const float nm = -(q < N ? p.m[(int64_t)zh * N + q] : 0.0f);
  float dl;
  if (p.fuse_delta) {  // delta = rowsum(dO * O), stored for the dK/dV kernel that follows
    float sd[NSD];
#pragma unroll
    for (int s = 0; s < NSD; ++s) sd[s] = chunk_dot(*reinterpret_cast<const V8*>((const T*)p.o + off + 16 * s), dop[s]);
    dl = row_delta(sd);
    if (q >= N) dl = 0.0f;
    else if (h2 == 0 && cs == 0) p.delta[(int64_t)zh * N + q] = dl;
  } else {
    dl = q < N ? p.delta[(int64_t)zh * N + q] : 0.0f;
  }
  OpAddr<D> at;
  at.init(cs * R::TILE, lane);
  const int lim = CAUSAL ? min(q, N - 1) : N - 1;  // last key the lane's row sees
  f32x16 dq[DT];
#pragma unroll
  for (int u = 0; u < DT; ++u) dq[u] = f32x16{};

  auto tile = [&](const char* st, int t) __attribute__((always_inline)) {
    f32x16 s = f32x16{}, dp;
#pragma unroll
    for (int r = 0; r < 16; ++r) dp[r] = -dl;  // seeds dP - delta
#pragma unroll
    for (int sd = 0; sd < NSD; ++sd) {
      s = Elt<T>::mfma(lds8<T>(st + at.nat[sd]), qop[sd], s);
      dp = Elt<T>::mfma(lds8<T>(st + R::HALF + at.nat[sd]), dop[sd], dp);
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) s[r] = fast_exp2(__builtin_fmaf(s[r], c, nm));
    if (32 * t + 32 > N || (CAUSAL && t == qt)) {  // hidden keys: probability 0
      const int past = lim - 32 * t - 8 * h2;
#pragma unroll
      for (int r = 0; r < 16; ++r) s[r] = 16 * (r >> 3) + (r & 7) > past ? 0.0f : s[r];
    }
    V8 ds[2];
#pragma unroll
    for (int sl = 0; sl < 2; ++sl)
#pragma unroll
      for (int i = 0; i < 8; i += 2) {
        const int r = 8 * sl + i;
        const V2 dh = H::pack(s[r] * dp[r], s[r + 1] * dp[r + 1]);
        ds[sl][i] = dh[0];
        ds[sl][i + 1] = dh[1];
      }
#pragma unroll
    for (int sl = 0; sl < 2; ++sl)
#pragma unroll
      for (int u = 0; u < DT; ++u) {
        V8 a = at.template tr<T>(st, sl, u);
        if (D < 32 && 16 * ((lane >> 4) & 1) >= D) a = V8{};
        dq[u] = Elt<T>::mfma(a, ds[sl], dq[u]);
      }
  };
  auto step = [&](int i, char* cur, char* nxt) __attribute__((always_inline)) {
    if (i + 1 < nsteps) ld.issue(nxt, i + 1);
    const int t = i * CS + cs;
    if (t < wtiles) {
      tile(cur, t);
    }
    landed_barrier();
  };
  landed_barrier();
  int i = 0;
  for (; i + 1 < nsteps; i += 2) {
    step(i, s0, s1);
    step(i + 1, s1, s0);
  }
  if (i < nsteps) step(i, s0, s1);

  constexpr int PART = DT * 16 * 64 * 4;
  constexpr int PER = R::STAGE / PART;
  static_assert(2 * PER >= NW, "partials fit the stages");
  auto part = [&](int k) { return (TATTN_LDS float*)(k < PER ? s0 + k * PART : s1 + (k - PER) * PART); };
  {
    TATTN_LDS float* dst = part(wu) + lane;
#pragma unroll
    for (int u = 0; u < DT; ++u)
#pragma unroll
      for (int r = 0; r < 16; ++r) dst[(16 * u + r) * 64] = dq[u][r];
  }
  __syncthreads();
  if (q < N) {
    T* row = (T*)p.dq + slice_off(p.so, zh, p.H) + (int64_t)q * p.so[2];
    for (int gr = cs; gr < DT * 4; gr += CS) {
      const int d0 = 8 * gr + 4 * h2;
      if (d0 < D) {
        f32x4 x = f32x4{};
#pragma unroll
        for (int k = 0; k < CS; ++k) {
          const TATTN_LDS float* src = part(rw * CS + k) + lane + 4 * gr * 64;
#pragma unroll
          for (int e = 0; e < 4; ++e) x[e] += src[64 * e];
        }
        V4 y;
#pragma unroll
        for (int e = 0; e < 4; ++e) y[e] = (T)(x[e] * p.scale);
        *reinterpret_cast<V4*>(row + d0) = y;
      }
    }
  }
}

// ---- dK / dV ---------------------------------------------------------------------------------
template <typename T, int D, int RW, int CS, int OCC, bool CAUSAL>
__global__ __launch_bounds__(RW * CS * 64, OCC) void dkdv_coop_kernel(const BwdParams p) {
  using H = H16<T>;
  using V8 = typename H::V8;
  using V2 = typename H::V2;
  constexpr int NW = RW * CS, NSD = D / 16, DT = (D + 31) / 32;
  using R = Ring<D, NW, CS>;
  __shared__ __attribute__((aligned(1024))) char s0[R::STAGE];
  __shared__ __attribute__((aligned(1024))) char s1[R::STAGE];
  __shared__ __attribute__((aligned(16))) float md[NW][2][64];  // per wave and parity: M[32], -delta[32]

  const int tid = threadIdx.x;
  const int lane = tid & 63, h2 = lane >> 5, l32 = lane & 31;
  const int wu = (int)uniform32((uint32_t)(tid >> 6));
  const int rw = wu / CS, cs = wu % CS;
  const int N = p.N;
  const float c = p.c;
  const BlockCoord bc = coop_coord(p.Z * p.H, p.n_blocks, CAUSAL);
  const int zh = bc.zh, kb = bc.blk;  // causal: small key blocks (most work) first
  const int ntile = (N + 31) / 32;
  const int kt = kb * RW + rw;  // the wave's key tile
  const int key = 32 * kt + l32;
  const int lo = CAUSAL ? kb * RW : 0;  // first query tile the block sees
  const int nsteps = (ntile - lo + CS - 1) / CS;
  const int64_t hoff = slice_off(p.s, zh, p.H);
  const int64_t rs = p.s[2];

  Loader<D, NW, CS> ld;
  {
    const int64_t o = hoff + (int64_t)(32 * lo) * rs;
    const uint64_t bytes = slice_bytes(N - 32 * lo, rs, D);
    ld.init(slice_rsrc((const T*)p.q + o, bytes), rs, slice_rsrc((const T*)p.dout + o, bytes), rs, wu, lane);
  }
  ld.issue(s0, 0);
  // Lanes 0-31 fetch M and lanes 32-63 delta of the wave's tile; zero past the end.
  const float* mdsrc = (h2 ? p.delta : p.m) + (int64_t)zh * N;
  auto md_load = [&](int i) {
    const int q = 32 * (lo + i * CS + cs) + l32;
    const float x = q < N ? mdsrc[q] : 0.0f;
    return h2 ? -x : x;
  };
  md[wu][0][lane] = md_load(0);
  V8 kop[NSD], vop[NSD];
  {
    const int64_t off = hoff + (int64_t)(key < N ? key : 0) * rs + 8 * h2;
#pragma unroll
    for (int s = 0; s < NSD; ++s) {
      const V8 a = *reinterpret_cast<const V8*>((const T*)p.k + off + 16 * s);
      const V8 b = *reinterpret_cast<const V8*>((const T*)p.v + off + 16 * s);
      kop[s] = key < N ? a : V8{};
      vop[s] = key < N ? b : V8{};
    }
  }
  OpAddr<D> at;
  at.init(cs * R::TILE, lane);
  f32x16 dk[DT], dv[DT];
#pragma unroll
  for (int u = 0; u < DT; ++u) dk[u] = dv[u] = f32x16{};

  auto tile = [&](const char* st, const float* mdw, int t) __attribute__((always_inline)) {
    f32x16 s = f32x16{}, dp;
    float mv[16];
#pragma unroll
    for (int a = 0; a < 4; ++a) {
      const int at = 16 * (a >> 1) + 8 * h2 + 4 * (a & 1);
      const f32x4 x = *reinterpret_cast<const TATTN_LDS f32x4*>((const TATTN_LDS float*)mdw + at);
      const f32x4 y = *reinterpret_cast<const TATTN_LDS f32x4*>((const TATTN_LDS float*)mdw + 32 + at);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        mv[4 * a + i] = x[i];
        dp[4 * a + i] = y[i];
      }
    }
#pragma unroll
    for (int sd = 0; sd < NSD; ++sd) {
      s = Elt<T>::mfma(lds8<T>(st + at.nat[sd]), kop[sd], s);
      dp = Elt<T>::mfma(lds8<T>(st + R::HALF + at.nat[sd]), vop[sd], dp);
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) s[r] = fast_exp2(__builtin_fmaf(s[r], c, -mv[r]));
    if (CAUSAL && t == kt) {  // queries of the tile before the lane's key: probability 0
      const int before = key - 32 * t - 8 * h2;
#pragma unroll
      for (int r = 0; r < 16; ++r) s[r] = 16 * (r >> 3) + (r & 7) < before ? 0.0f : s[r];
    }
    V8 pp[2], ds[2];
#pragma unroll
    for (int sl = 0; sl < 2; ++sl)
#pragma unroll
      for (int i = 0; i < 8; i += 2) {
        const int r = 8 * sl + i;
        const V2 ph = H::pack(s[r], s[r + 1]), dh = H::pack(s[r] * dp[r], s[r + 1] * dp[r + 1]);
        pp[sl][i] = ph[0];
        pp[sl][i + 1] = ph[1];
        ds[sl][i] = dh[0];
        ds[sl][i + 1] = dh[1];
      }
#pragma unroll
    for (int sl = 0; sl < 2; ++sl)
#pragma unroll
      for (int u = 0; u < DT; ++u) {
        V8 dob = at.template tr<T>(st + R::HALF, sl, u);
        V8 qb = at.template tr<T>(st, sl, u);
        if (D < 32 && 16 * ((lane >> 4) & 1) >= D) dob = qb = V8{};
        dv[u] = Elt<T>::mfma(pp[sl], dob, dv[u]);
        dk[u] = Elt<T>::mfma(ds[sl], qb, dk[u]);
      }
  };
  auto step = [&](int i, char* cur, char* nxt, int par) __attribute__((always_inline)) {
    float mdn = 0.0f;
    if (i + 1 < nsteps) {
      ld.issue(nxt, i + 1);
      mdn = md_load(i + 1);
    }
    const int t = lo + i * CS + cs;
    if (t < ntile && kt < ntile && (!CAUSAL || t >= kt)) {
      tile(cur, md[wu][par], t);
    }
    md[wu][par ^ 1][lane] = mdn;  // the wave's own rows: no barrier needed
    landed_barrier();
  };
  landed_barrier();
  int i = 0;
  for (; i + 1 < nsteps; i += 2) {
    step(i, s0, s1, 0);
    step(i + 1, s1, s0, 1);
  }
  if (i < nsteps) step(i, s0, s1, 0);

  // Sum the CS partials of each key tile, dK then dV. C register r of a lane: key
  // 8 (r/4) + 4 h2 + r%4 of the tile, column 32 u + l32.
  constexpr int PART = DT * 16 * 64 * 4;
  constexpr int PER = R::STAGE / PART;
  static_assert(2 * PER >= NW, "partials fit the stages");
  auto part = [&](int k) { return (TATTN_LDS float*)(k < PER ? s0 + k * PART : s1 + (k - PER) * PART); };
  auto reduce = [&](const f32x16 (&a)[DT], float mul, T* dst) __attribute__((always_inline)) {
    TATTN_LDS float* mine = part(wu) + lane;
#pragma unroll
    for (int u = 0; u < DT; ++u)
#pragma unroll
      for (int r = 0; r < 16; ++r) mine[(16 * u + r) * 64] = a[u][r];
    __syncthreads();
    for (int g = cs; g < DT * 16; g += CS) {
      const int u = g >> 4, r = g & 15;
      const int row = 32 * kt + 8 * (r >> 2) + 4 * h2 + (r & 3), d = 32 * u + l32;
      float x = 0.0f;
#pragma unroll
      for (int k = 0; k < CS; ++k) x += (part(rw * CS + k) + lane)[g * 64];
      if (row < N && d < D) dst[(int64_t)row * p.so[2] + d] = (T)(x * mul);
    }
  };
  const int64_t goff = slice_off(p.so, zh, p.H);
  reduce(dk, p.scale, (T*)p.dk + goff);
  __syncthreads();
  reduce(dv, 1.0f, (T*)p.dv + goff);
}

// Row tiles per workgroup and tiles of the other dimension per step: two stages of CS tile pairs
// stay within 64 KB, the reach of an LDS instruction's immediate offset.
template <int D> struct Shape { static constexpr int RW = 2, CS = D == 128 ? 2 : 4, NW = RW * CS; };

template <typename T, int D>
int fwd_d(FwdParams p, bool causal, hipStream_t st) {
  using S = Shape<D>;
  p.n_qblocks = (p.N + 32 * S::RW - 1) / (32 * S::RW);
  const dim3 grid((unsigned)((int64_t)p.n_qblocks * p.Z * p.H)), block(S::NW * 64);
  constexpr int OCC = D == 128 ? 2 : 4;
  if (causal) fwd_coop_kernel<T, D, S::RW, S::CS, OCC, true><<<grid, block, 0, st>>>(p);
  else fwd_coop_kernel<T, D, S::RW, S::CS, OCC, false><<<grid, block, 0, st>>>(p);
  return check_launch("tattn_fwd");
}

template <typename T, int D>
int dq_d(BwdParams p, bool causal, hipStream_t st) {
  using S = Shape<D>;
  p.n_blocks = (p.N + 32 * S::RW - 1) / (32 * S::RW);
  const dim3 grid((unsigned)((int64_t)p.n_blocks * p.Z * p.H)), block(S::NW * 64);
  constexpr int OCC = D >= 64 ? 2 : 4;  // 128 registers would spill at head dim 64 (35 -> 44 us at 1 x 16 x 2048)
  if (causal) dq_coop_kernel<T, D, S::RW, S::CS, OCC, true><<<grid, block, 0, st>>>(p);
  else dq_coop_kernel<T, D, S::RW, S::CS, OCC, false><<<grid, block, 0, st>>>(p);
  return check_launch("tattn_bwd_dq");
}

template <typename T, int D>
int dkdv_d(BwdParams p, bool causal, hipStream_t st) {
  using S = Shape<D>;
  p.n_blocks = (p.N + 32 * S::RW - 1) / (32 * S::RW);
  const dim3 grid((unsigned)((int64_t)p.n_blocks * p.Z * p.H)), block(S::NW * 64);
  constexpr int OCC = D >= 64 ? 2 : D == 32 ? 3 : 4;
  if (causal) dkdv_coop_kernel<T, D, S::RW, S::CS, OCC, true><<<grid, block, 0, st>>>(p);
  else dkdv_coop_kernel<T, D, S::RW, S::CS, OCC, false><<<grid, block, 0, st>>>(p);
  return check_launch("tattn_bwd_dkdv");
}

#define TATTN_COOP_CASE(FN, D_) \
  case D_: return dtype == 0 ? FN<f16, D_>(p, causal, st) : FN<bf16, D_>(p, causal, st);
#define TATTN_COOP_SWITCH(FN, CASE_128)                                                   \
  switch (D) {                                                                          \
    TATTN_COOP_CASE(FN, 16) TATTN_COOP_CASE(FN, 32) TATTN_COOP_CASE(FN, 64) CASE_128      \
  }                                                                                     \
  return set_error(TATTN_E_ARG, "%s: no kernel with split sums at head dim %d", #FN, D);

}  // namespace

int launch_fwd_coop(const FwdParams& p, int D, int dtype, bool causal, hipStream_t st) {
  TATTN_COOP_SWITCH(fwd_d, TATTN_COOP_CASE(fwd_d, 128))
}
int launch_dq_coop(const BwdParams& p, int D, int dtype, bool causal, hipStream_t st) {
  TATTN_COOP_SWITCH(dq_d, TATTN_COOP_CASE(dq_d, 128))
}
// Head dim 128: dK, dV, K and V of a tile do not fit a wave's 256 registers (never picked).
int launch_dkdv_coop(const BwdParams& p, int D, int dtype, bool causal, hipStream_t st) { TATTN_COOP_SWITCH(dkdv_d, ) }

}  // namespace tattn
