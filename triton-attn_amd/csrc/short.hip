// 16-bit attention for short rows (N <= 128) on gfx950: forward, and the whole backward in one
// launch (the reference's src/tattn/kernels.py:57-337 for such rows).
//
// A (z, h) slice of at most 32 TT rows is owned by TT waves, one 32-row tile each, and a
// workgroup of four waves holds 4 / TT slices. The block kernels give each slice a workgroup of
// its own, whose waves past the slice's rows idle, and run its one to four steps through a ring
// with a barrier per step. Such launches are bound by bytes and latency, not by the matrix cores:
// here a slice's rows are read once, land in LDS (rows in perm32 order, chunks swizzled, as in
// bwd_pipe.h) and everything is computed from there with one barrier.
//
//   forward   S^T of every key tile at once, softmax, O^T += V^T P^T. The max in the exponent is
//             the row max of tile 0, which the block kernels start from and keep at least while no score
//             rises more than 2^kRescaleLog2 above it, and tile sums are added tile by tile: O and M
//             are then theirs bit for bit. Rows that do rise take the max over all their keys at
//             once, where the block kernels rescale on the way.
//   backward  delta of the wave's queries; then, as owner of a key tile, dV and dK over the
//             slice's query tiles; then, as owner of a query tile, dQ over its key tiles. Same
//             operands, MFMA chains and orders as dkdv_pipe_kernel and dq_pipe_kernel, so the
//             gradients and delta are theirs bit for bit; Q, K, V, dO are read once instead of
//             twice, and delta and M stay in LDS.
//
// Measured against the block kernels (warm, us, forward / backward; one MI355X):
//   65,536 slices x 24 rows x 16, fp16: 140 -> 39 / 517 -> 89 (HBM floor 38 / 75 at a copy's rate)
//   8,192 x 24 x 64: 40 -> 17 / 200 -> 38        4,096 x 64 x 64 causal: 37 -> 22 / 98 -> 52
//   2,048 x 128 x 64: 30 -> 25 / 116 -> 64       2,048 x 128 x 16: 12.1 -> 11.7 / 34 -> 25
//   1,024 x 128 x 128: 36 -> 27 / 96 -> 88       96 x 128 x 64 causal: 8.4 -> 5.8 / 16 -> 9
// Past 128 rows a slice's tiles no longer fit the LDS and registers of four waves.
#include <type_traits>

#include "bwd_pipe.h"
#include "common.h"
#include "launch.h"

namespace tattn {

namespace {

// Rows of slice tiles into LDS: TT * 32 rows of D elements, 16-byte chunks, by the slice's TT * 64
// threads (st = thread within the slice). Rows at or past N read as zero (range-checked loads).
template <int D, int TT>
struct ShortTile {
  static constexpr int RB = Swz<D>::RB;
  static constexpr int TILE = 32 * RB;
  static constexpr int CPR = D / 8;
  static constexpr int CPT = CPR / 2;  // chunks per thread: TT * 32 * CPR over TT * 64 threads
  static __device__ __forceinline__ void load(u32x4 (&x)[CPT], __amdgpu_buffer_rsrc_t r, uint32_t row_bytes, int st) {
#pragma unroll
    for (int i = 0; i < CPT; ++i) {
      const int ch = st + i * TT * 64;
      x[i] = rsrc_load(r, (uint32_t)(ch / CPR) * row_bytes + (uint32_t)(ch % CPR) * 16);
    }
  }
  static __device__ __forceinline__ void store(char* tile, const u32x4 (&x)[CPT], int st) {
#pragma unroll
    for (int i = 0; i < CPT; ++i) {
      const int ch = st + i * TT * 64;
      const int row = ch / CPR;
      st16(tile + (row >> 5) * TILE + Swz<D>::addr(perm32(row & 31), (ch % CPR) * 16), x[i]);
    }
  }
};

// With one wave per slice its LDS rows are its own: program order is enough. Otherwise the
// workgroup's barrier publishes them (every wave runs the same number of barriers).
template <int TT>
__device__ __forceinline__ void slice_sync() {
  if constexpr (TT > 1) __syncthreads();
}

// Natural 8-element MFMA operand of tile row `row` (sequence order) at columns 16 s + 8 h2.
template <typename T, int D>
__device__ __forceinline__ typename H16<T>::V8 row_operand(const char* tile, int row, int s, int h2) {
  return lds8<T>(tile + Swz<D>::addr(perm32(row), (16 * s + 8 * h2) * 2));
}

// A C-layout tile whose lanes own columns and registers own rows (dK, dV), or whose lanes own
// rows (O, dQ), leaves through the wave's LDS rows as 16-byte chunks of the rows below N.
template <typename T, int D>
__device__ __forceinline__ void rows_out(const TATTN_LDS char* wl, T* dst, int64_t row_stride, int rows, int lane) {
  constexpr int CPR = D / 8;
#pragma unroll
  for (int it = 0; it < 32 * CPR / 64; ++it) {
    const int j = lane + 64 * it;
    const int row = j / CPR, cc = j % CPR;
    if (row < rows)
      st16(dst + (int64_t)row * row_stride + 8 * cc, *reinterpret_cast<const TATTN_LDS u32x4*>(wl + Swz<D>::addr(row, 16 * cc)));
  }
}

template <int D, int TT> constexpr int fwd_short_occ() { return D == 128 ? 2 : D == 64 ? 3 : 4; }

template <typename T, int D, int TT, bool CAUSAL>
__global__ __launch_bounds__(256, (fwd_short_occ<D, TT>())) void fwd_short_kernel(const FwdParams p) {
  using H = H16<T>;
  using V8 = typename H::V8;
  using V4 = typename H::V4;
  using V2 = typename H::V2;
  using L = ShortTile<D, TT>;
  constexpr int SPW = 4 / TT, NSD = D / 16, DT = (D + 31) / 32;
  __shared__ __attribute__((aligned(16))) char smem[SPW][2][TT * L::TILE];

  const int tid = threadIdx.x;
  const int lane = tid & 63, w = tid >> 6, h2 = lane >> 5, l32 = lane & 31;
  const int sub = (int)uniform32((uint32_t)(w / TT)), wt = (int)uniform32((uint32_t)(w % TT));
  const int st = wt * 64 + lane;
  const int N = p.N;
  const float c = p.c;
  const int zhs = p.Z * p.H;
  const int zh_raw = blockIdx.x * SPW + sub;
  const bool live = zh_raw < zhs;  // a last workgroup's spare waves run a copy of the last slice
  const int zh = live ? zh_raw : zhs - 1;
  const int64_t qo = slice_off(p.sq, zh, p.H), ko = slice_off(p.sk, zh, p.H), vo = slice_off(p.sv, zh, p.H);
  char* const ks = smem[sub][0];
  char* const vs = smem[sub][1];
  const int q = 32 * wt + l32;

  u32x4 ck[L::CPT], cv[L::CPT];
  L::load(ck, slice_rsrc((const T*)p.k + ko, slice_bytes(N, p.sk[2], D)), (uint32_t)p.sk[2] * 2, st);
  L::load(cv, slice_rsrc((const T*)p.v + vo, slice_bytes(N, p.sv[2], D)), (uint32_t)p.sv[2] * 2, st);
  V8 qop[NSD];
  {
    const T* src = (const T*)p.q + qo + (int64_t)(q < N ? q : 0) * p.sq[2] + 8 * h2;
#pragma unroll
    for (int s = 0; s < NSD; ++s) {
      const V8 x = *reinterpret_cast<const V8*>(src + 16 * s);
      qop[s] = q < N ? x : V8{};
    }
  }
  L::store(ks, ck, st);
  L::store(vs, cv, st);
  slice_sync<TT>();

  // S^T of the key tiles the wave's rows see; C register r of a lane: key kappa(r, h2) of the tile.
  const int nt = CAUSAL ? min(wt + 1, (N + 31) / 32) : (N + 31) / 32;
  f32x16 s[TT];
#pragma unroll
  for (int t = 0; t < TT; ++t)
    if (t < nt) {
      s[t] = f32x16{};
#pragma unroll
      for (int sd = 0; sd < NSD; ++sd)
        s[t] = Elt<T>::mfma(lds8<T>(ks + t * L::TILE + Swz<D>::addr(l32, (16 * sd + 8 * h2) * 2)), qop[sd], s[t]);
    }
  // Only the tile on the diagonal or across the sequence end hides keys (wave-uniform).
  auto partial = [&](int t) { return TT == 1 || 32 * t + 32 > N || (CAUSAL && t == wt); };
  auto hidden = [&](int t, int r) {
    const int key = 32 * t + kappa(r, h2);
    return key >= N || (CAUSAL && key > q);
  };
  float mx = -__builtin_inff(), mx0 = mx;
#pragma unroll
  for (int t = 0; t < TT; ++t)
    if (t < nt) {
      if (partial(t)) {
#pragma unroll
        for (int r = 0; r < 16; ++r) mx = hidden(t, r) ? mx : __builtin_fmaxf(mx, s[t][r] * c);
      } else {
#pragma unroll
        for (int r = 0; r < 16; ++r) mx = __builtin_fmaxf(mx, s[t][r] * c);
      }
      if (t == 0) mx0 = mx;
    }
  mx = max_halves(mx);
  if constexpr (TT > 1) {
    mx0 = max_halves(mx0);
    mx = mx > mx0 + kRescaleLog2 ? mx : mx0;
  }
  float sum = 0.0f;
  f32x16 acc[DT];
#pragma unroll
  for (int u = 0; u < DT; ++u) acc[u] = f32x16{};
  auto probs = [&](int t, V8 (&x)[2], auto mask_tag) {
    constexpr bool MASK = decltype(mask_tag)::value;
    float ps = 0.0f;
#pragma unroll
    for (int sg = 0; sg < 2; ++sg)
#pragma unroll
      for (int i = 0; i < 8; i += 2) {
        float e[2];
#pragma unroll
        for (int b = 0; b < 2; ++b) {
          const int r = 8 * sg + i + b;
          e[b] = fast_exp2(__builtin_fmaf(s[t][r], c, -mx));
          if constexpr (MASK) e[b] = hidden(t, r) ? 0.0f : e[b];
        }
        const V2 pr = H::pack(e[0], e[1]);
        ps = H::sum2(pr, ps);
        x[sg][i] = pr[0];
        x[sg][i + 1] = pr[1];
      }
    sum += ps;
  };
#pragma unroll
  for (int t = 0; t < TT; ++t)
    if (t < nt) {
      V8 x[2];
      if (partial(t)) probs(t, x, std::true_type{});
      else probs(t, x, std::false_type{});
#pragma unroll
      for (int sg = 0; sg < 2; ++sg)
#pragma unroll
        for (int u = 0; u < DT; ++u) {
          int a0, a1;
          tr_addrs<D>(sg, u, lane, a0, a1);
          V8 vop = tr_pair<T>(vs + t * L::TILE, a0, a1);
          if (D < 32 && 16 * ((lane >> 4) & 1) >= D) vop = V8{};
          acc[u] = Elt<T>::mfma(vop, x[sg], acc[u]);
        }
    }
  const float lt = sum_halves(sum);
  const float inv = 1.0f / lt;
  if (live && p.m && h2 == 0 && q < N) p.m[(int64_t)zh * N + q] = mx + __log2f(lt);

  // O rows through the wave's own tile of the K stage, once every wave is done with it.
  slice_sync<TT>();
  TATTN_LDS char* wl = (TATTN_LDS char*)ks + wt * L::TILE;
#pragma unroll
  for (int u = 0; u < DT; ++u)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int d0 = 32 * u + 8 * g + 4 * h2;
      if (d0 < D) {
        V4 x;
#pragma unroll
        for (int i = 0; i < 4; ++i) x[i] = (T)(acc[u][4 * g + i] * inv);
        *reinterpret_cast<TATTN_LDS V4*>(wl + Swz<D>::addr(l32, 2 * d0)) = x;
      }
    }
  if (live)
    rows_out<T, D>(wl, (T*)p.o + slice_off(p.so, zh, p.H) + (int64_t)(32 * wt) * p.so[2], p.so[2], N - 32 * wt, lane);
}

template <int D, int TT> constexpr int bwd_short_occ() { return D == 128 ? 1 : D == 64 ? 2 : TT > 1 ? 3 : 4; }

template <typename T, int D, int TT, bool CAUSAL>
__global__ __launch_bounds__(256, (bwd_short_occ<D, TT>())) void bwd_short_kernel(const BwdParams p) {
  using H = H16<T>;
  using V8 = typename H::V8;
  using V4 = typename H::V4;
  using V2 = typename H::V2;
  using L = ShortTile<D, TT>;
  constexpr int SPW = 4 / TT, NSD = D / 16, DT = (D + 31) / 32;
  constexpr int BYTES = TT * L::TILE;
  __shared__ __attribute__((aligned(16))) char smem[SPW][4][BYTES];
  __shared__ __attribute__((aligned(16))) float md[SPW][2][TT * 32];

  const int tid = threadIdx.x;
  const int lane = tid & 63, w = tid >> 6, h2 = lane >> 5, l32 = lane & 31;
  const int sub = (int)uniform32((uint32_t)(w / TT)), wt = (int)uniform32((uint32_t)(w % TT));
  const int st = wt * 64 + lane;
  const int N = p.N;
  const float c = p.c;
  const int zhs = p.Z * p.H;
  const int zh_raw = blockIdx.x * SPW + sub;
  const bool live = zh_raw < zhs;  // a last workgroup's spare waves run a copy of the last slice
  const int zh = live ? zh_raw : zhs - 1;
  const int64_t off = slice_off(p.s, zh, p.H);
  const uint64_t bytes = slice_bytes(N, p.s[2], D);
  const uint32_t row_bytes = (uint32_t)p.s[2] * 2;
  char* const qs = smem[sub][0];
  char* const ks = smem[sub][1];
  char* const vs = smem[sub][2];
  char* const os = smem[sub][3];  // dO
  const int row = 32 * wt + l32;  // the wave's query (delta, dQ) and key (dK, dV) of this lane

  {
    u32x4 a[L::CPT], b[L::CPT], d[L::CPT], e[L::CPT];
    L::load(a, slice_rsrc((const T*)p.q + off, bytes), row_bytes, st);
    L::load(b, slice_rsrc((const T*)p.k + off, bytes), row_bytes, st);
    L::load(d, slice_rsrc((const T*)p.v + off, bytes), row_bytes, st);
    L::load(e, slice_rsrc((const T*)p.dout + off, bytes), row_bytes, st);
    // delta of the lane's query: the preprocess's chunk sums and order.
    float sd[NSD];
    const __amdgpu_buffer_rsrc_t ors = slice_rsrc((const T*)p.o + off, bytes), dors = slice_rsrc((const T*)p.dout + off, bytes);
#pragma unroll
    for (int s = 0; s < NSD; ++s) {
      const uint32_t at = (uint32_t)row * row_bytes + (uint32_t)(32 * s + 16 * h2);
      sd[s] = chunk_dot(__builtin_bit_cast(V8, rsrc_load(ors, at)), __builtin_bit_cast(V8, rsrc_load(dors, at)));
    }
    const float dl = row_delta(sd);
    if (h2 == 0) {
      const bool in = row < N;
      md[sub][0][row] = in ? p.m[(int64_t)zh * N + row] : 0.0f;
      md[sub][1][row] = in ? -dl : 0.0f;  // negated: seeds the dP accumulators
      if (in && live) p.delta[(int64_t)zh * N + row] = dl;
    }
    L::store(qs, a, st);
    L::store(ks, b, st);
    L::store(vs, d, st);
    L::store(os, e, st);
  }
  slice_sync<TT>();

  int nat[NSD], tra[2][DT][2];
#pragma unroll
  for (int s = 0; s < NSD; ++s) nat[s] = Swz<D>::addr(l32, (16 * s + 8 * h2) * 2);
#pragma unroll
  for (int sl = 0; sl < 2; ++sl)
#pragma unroll
    for (int u = 0; u < DT; ++u) tr_addrs<D>(sl, u, lane, tra[sl][u][0], tra[sl][u][1]);
  const int nt = (N + 31) / 32;

  // ---- dV and dK of key tile wt over the query tiles ------------------------------------------
  f32x16 dk[DT], dv[DT];
#pragma unroll
  for (int u = 0; u < DT; ++u) dk[u] = dv[u] = f32x16{};
  {
    V8 kop[NSD], vop[NSD];
#pragma unroll
    for (int s = 0; s < NSD; ++s) {
      kop[s] = row_operand<T, D>(ks + wt * L::TILE, l32, s, h2);
      vop[s] = row_operand<T, D>(vs + wt * L::TILE, l32, s, h2);
    }
#pragma unroll
    for (int j = 0; j < TT; ++j)
      if (j < nt && (!CAUSAL || j >= wt)) {
        const char* qt = qs + j * L::TILE;
        const char* ot = os + j * L::TILE;
        f32x16 s = f32x16{}, dp;
        float mv[16];
#pragma unroll
        for (int a = 0; a < 4; ++a) {
          const int at = 32 * j + 16 * (a >> 1) + 8 * h2 + 4 * (a & 1);
          const f32x4 x = *reinterpret_cast<const TATTN_LDS f32x4*>((const TATTN_LDS float*)md[sub][0] + at);
          const f32x4 y = *reinterpret_cast<const TATTN_LDS f32x4*>((const TATTN_LDS float*)md[sub][1] + at);
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            mv[4 * a + i] = x[i];
            dp[4 * a + i] = y[i];
          }
        }
#pragma unroll
        for (int sd = 0; sd < NSD; ++sd) {
          s = Elt<T>::mfma(lds8<T>(qt + nat[sd]), kop[sd], s);
          dp = Elt<T>::mfma(lds8<T>(ot + nat[sd]), vop[sd], dp);
        }
#pragma unroll
        for (int sl = 0; sl < 2; ++sl) {
          V8 pp, ds;
#pragma unroll
          for (int i = 0; i < 8; i += 2) {
            float pr[2], dr[2];
#pragma unroll
            for (int b = 0; b < 2; ++b) {
              const int r = 8 * sl + i + b;
              float pv = fast_exp2(__builtin_fmaf(s[r], c, -mv[r]));
              if (CAUSAL && j == wt) pv = row > 32 * j + kappa(r, h2) ? 0.0f : pv;
              pr[b] = pv;
              dr[b] = pv * dp[r];
            }
            const V2 ph = H::pack(pr[0], pr[1]), dh = H::pack(dr[0], dr[1]);
            pp[i] = ph[0];
            pp[i + 1] = ph[1];
            ds[i] = dh[0];
            ds[i + 1] = dh[1];
          }
#pragma unroll
          for (int u = 0; u < DT; ++u) {
            V8 dob = tr_pair<T>(ot, tra[sl][u][0], tra[sl][u][1]);
            V8 qb = tr_pair<T>(qt, tra[sl][u][0], tra[sl][u][1]);
            if (D < 32 && 16 * ((lane >> 4) & 1) >= D) dob = qb = V8{};
            dv[u] = Elt<T>::mfma(pp, dob, dv[u]);
            dk[u] = Elt<T>::mfma(ds, qb, dk[u]);
          }
        }
      }
  }

  // ---- dQ of query tile wt over the key tiles -------------------------------------------------
  f32x16 dq[DT];
#pragma unroll
  for (int u = 0; u < DT; ++u) dq[u] = f32x16{};
  {
    V8 qop[NSD], dop[NSD];
#pragma unroll
    for (int s = 0; s < NSD; ++s) {
      qop[s] = row_operand<T, D>(qs + wt * L::TILE, l32, s, h2);
      dop[s] = row_operand<T, D>(os + wt * L::TILE, l32, s, h2);
    }
    const float nm = -((const TATTN_LDS float*)md[sub][0])[row], ndl = ((const TATTN_LDS float*)md[sub][1])[row];
#pragma unroll
    for (int t = 0; t < TT; ++t)
      if (t < nt && (!CAUSAL || t <= wt)) {
        const char* kt = ks + t * L::TILE;
        const char* vt = vs + t * L::TILE;
        f32x16 s = f32x16{}, dp;
#pragma unroll
        for (int r = 0; r < 16; ++r) dp[r] = ndl;
#pragma unroll
        for (int sd = 0; sd < NSD; ++sd) {
          s = Elt<T>::mfma(lds8<T>(kt + nat[sd]), qop[sd], s);
          dp = Elt<T>::mfma(lds8<T>(vt + nat[sd]), dop[sd], dp);
        }
        V8 ds[2];
        auto dsv = [&](auto mask_tag) {
          constexpr bool MASK = decltype(mask_tag)::value;
#pragma unroll
          for (int sl = 0; sl < 2; ++sl)
#pragma unroll
            for (int i = 0; i < 8; i += 2) {
              float dr[2];
#pragma unroll
              for (int b = 0; b < 2; ++b) {
                const int r = 8 * sl + i + b;
                const int key = 32 * t + kappa(r, h2);
                float pv = fast_exp2(__builtin_fmaf(s[r], c, nm));
                if constexpr (MASK) pv = (key >= N || (CAUSAL && key > row)) ? 0.0f : pv;
                dr[b] = pv * dp[r];
              }
              const V2 dh = H::pack(dr[0], dr[1]);
              ds[sl][i] = dh[0];
              ds[sl][i + 1] = dh[1];
            }
        };
        // Only the tile on the diagonal or across the sequence end hides keys (wave-uniform).
        if (TT == 1 || 32 * t + 32 > N || (CAUSAL && t == wt)) dsv(std::true_type{});
        else dsv(std::false_type{});
#pragma unroll
        for (int sl = 0; sl < 2; ++sl)
#pragma unroll
          for (int u = 0; u < DT; ++u) {
            V8 a = tr_pair<T>(kt, tra[sl][u][0], tra[sl][u][1]);
            if (D < 32 && 16 * ((lane >> 4) & 1) >= D) a = V8{};
            dq[u] = Elt<T>::mfma(a, ds[sl], dq[u]);
          }
      }
  }

  // ---- the three gradients through the wave's own tiles, once every wave has read its operands --
  slice_sync<TT>();
  const int rows = N - 32 * wt;
  const int64_t goff = slice_off(p.so, zh, p.H) + (int64_t)(32 * wt) * p.so[2];
  // dK (scaled), dV: C register r of a lane holds key 8 (r/4) + 4 h2 + r%4, column 32 u + l32.
  auto stage_cols = [&](TATTN_LDS char* wl, const f32x16 (&a)[DT], float mul) {
#pragma unroll
    for (int u = 0; u < DT; ++u)
      if (32 * u + l32 < D) {
#pragma unroll
        for (int r = 0; r < 16; ++r)
          *reinterpret_cast<TATTN_LDS T*>(wl + Swz<D>::addr(8 * (r >> 2) + 4 * h2 + (r & 3), 2 * (32 * u + l32))) =
              (T)(a[u][r] * mul);
      }
  };
  TATTN_LDS char* wk = (TATTN_LDS char*)ks + wt * L::TILE;
  TATTN_LDS char* wv = (TATTN_LDS char*)vs + wt * L::TILE;
  TATTN_LDS char* wq = (TATTN_LDS char*)qs + wt * L::TILE;
  stage_cols(wk, dk, p.scale);
  stage_cols(wv, dv, 1.0f);
#pragma unroll
  for (int u = 0; u < DT; ++u)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int d0 = 32 * u + 8 * g + 4 * h2;
      if (d0 < D) {
        V4 x;
#pragma unroll
        for (int i = 0; i < 4; ++i) x[i] = (T)(dq[u][4 * g + i] * p.scale);
        *reinterpret_cast<TATTN_LDS V4*>(wq + Swz<D>::addr(l32, 2 * d0)) = x;
      }
    }
  if (live) {
    rows_out<T, D>(wk, (T*)p.dk + goff, p.so[2], rows, lane);
    rows_out<T, D>(wv, (T*)p.dv + goff, p.so[2], rows, lane);
    rows_out<T, D>(wq, (T*)p.dq + goff, p.so[2], rows, lane);
  }
}

template <typename T, int D, int TT>
int fwd_tt(const FwdParams& p, bool causal, hipStream_t st) {
  const int64_t blocks = ((int64_t)p.Z * p.H + 4 / TT - 1) / (4 / TT);
  if (causal)
    fwd_short_kernel<T, D, TT, true><<<dim3((unsigned)blocks), dim3(256), 0, st>>>(p);
  else
    fwd_short_kernel<T, D, TT, false><<<dim3((unsigned)blocks), dim3(256), 0, st>>>(p);
  return check_launch("tattn_fwd");
}

template <typename T, int D, int TT>
int bwd_tt(const BwdParams& p, bool causal, hipStream_t st) {
  const int64_t blocks = ((int64_t)p.Z * p.H + 4 / TT - 1) / (4 / TT);
  if (causal)
    bwd_short_kernel<T, D, TT, true><<<dim3((unsigned)blocks), dim3(256), 0, st>>>(p);
  else
    bwd_short_kernel<T, D, TT, false><<<dim3((unsigned)blocks), dim3(256), 0, st>>>(p);
  return check_launch("tattn_bwd");
}

template <typename T, int D>
int fwd_d(const FwdParams& p, bool causal, hipStream_t st) {
  return p.N <= 32 ? fwd_tt<T, D, 1>(p, causal, st) : p.N <= 64 ? fwd_tt<T, D, 2>(p, causal, st) : fwd_tt<T, D, 4>(p, causal, st);
}

template <typename T, int D>
int bwd_d(const BwdParams& p, bool causal, hipStream_t st) {
  return p.N <= 32 ? bwd_tt<T, D, 1>(p, causal, st) : p.N <= 64 ? bwd_tt<T, D, 2>(p, causal, st) : bwd_tt<T, D, 4>(p, causal, st);
}

template <typename T>
int fwd_t(const FwdParams& p, int D, bool causal, hipStream_t st) {
  switch (D) {
    case 16: return fwd_d<T, 16>(p, causal, st);
    case 32: return fwd_d<T, 32>(p, causal, st);
    case 64: return fwd_d<T, 64>(p, causal, st);
    case 128: return fwd_d<T, 128>(p, causal, st);
  }
  return set_error(TATTN_E_ARG, "head dim must be 16, 32, 64 or 128, got %d", D);
}

template <typename T>
int bwd_t(const BwdParams& p, int D, bool causal, hipStream_t st) {
  switch (D) {
    case 16: return bwd_d<T, 16>(p, causal, st);
    case 32: return bwd_d<T, 32>(p, causal, st);
    case 64: return bwd_d<T, 64>(p, causal, st);
    case 128: return bwd_d<T, 128>(p, causal, st);
  }
  return set_error(TATTN_E_ARG, "head dim must be 16, 32, 64 or 128, got %d", D);
}

}  // namespace

int launch_fwd_short(const FwdParams& p, int D, int dtype, bool causal, hipStream_t st) {
  return dtype == 0 ? fwd_t<f16>(p, D, causal, st) : fwd_t<bf16>(p, D, causal, st);
}

int launch_bwd_short(const BwdParams& p, int D, int dtype, bool causal, hipStream_t st) {
  return dtype == 0 ? bwd_t<f16>(p, D, causal, st) : bwd_t<bf16>(p, D, causal, st);
}

}  // namespace tattn
