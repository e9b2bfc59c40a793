// float32 attention on the 16-bit matrix cores of gfx950 (the reference's src/tattn/kernels.py:57-321
// with float32 inputs): every float32 operand as an exact sum of three bf16 planes.
//
// The float32 MFMA runs at 1/16 of the bf16 rate and bounds the kernels built on it. Here x = hi + mid +
// lo (all 24 bits are held), and a product of two operands is the six bf16 products of plane pairs down to
// 2^-16 of it, smallest first, into a float32 accumulator. What is dropped (mid lo, lo mid, lo lo) is at
// most 2^-24.1 of a product of two inputs, 2^-27.4 in the root mean square, and 2^-23.3 and 2^-26.4 for P and dS
// times an input (4 million pairs each; a float32 product's rounding is 2^-24.0 and 2^-25.2). P and dS are split
// the same way, so nothing is held in 16 bits. A bf16 MFMA adds 16 products per rounding of the accumulator
// where the float32 one adds 2: the error against float64 is below the float32 MFMA kernels' at every size
// from N = 4 to 4,096 and every head dim (relative, O / dK: 1,024 slices x 16 x 16
// 8.2e-8 / 1.7e-7 against 1.3e-7 / 2.1e-7; 8 x 1,024 x 64 3.3e-7 / 4.7e-7 against 6.5e-7 / 7.5e-7; 4 x 4,096 x 64 causal
// 2.7e-7 / 6.9e-7 against 5.0e-7 / 1.5e-6).
//
// A bf16 plane cannot carry what an infinite float32 operand means (inf - inf has no middle plane), nor
// bits below 2^-133, which numbers from 2^-110 up do not have. Where a wave's operands hold an infinity, or are all
// below 2^-100 without being zero, the step is staged again as the halves of the float32 bits and runs on the
// float32 MFMA: what the block kernels give there, in 1.1 to 1.5 times their time. A number below 2^-110 beside one
// of 2^-100 or more in the same wave is held to 2^-134.
//
// Split of the work: a workgroup of NW = RW * CS waves owns RW 32-row tiles; a step stages CS tile
// pairs of the other dimension (read from HBM once per workgroup, split into planes once, by the thread
// that loaded them), and wave (rw, cs) works on pair cs for row tile rw; partial results of a row tile
// are added through LDS at the end. Which RW and CS: pick_shape, below.
//
// What bounds it: matrix and vector work of the two waves of a SIMD barely overlap (forward of 4 x 16 x
// 1,024 x 64, counters per SIMD: 98 thousand MFMA cycles and 93 thousand of vector issue, of 214 thousand
// busy; no bank conflicts). Per tile and wave: about 90 vector instructions for splitting P (twice that for P and
// dS), 130 for staging, 60 for the exponentials. Eight row tiles per workgroup halve the staging and took the
// same time within 7%; wave priorities changed nothing. dK/dV at head dim 64 keeps K in LDS and still spills.
//
// Measured (us, block kernels on the float32 MFMA -> here, forward / backward; one MI355X):
//   4 x 16 x 1,024 x 64   172 / 531 -> 110 / 341       causal  127 / 402 -> 65 / 227
//   2 x 4 x 128 x 64      18.3 / 57 -> 10.1 / 39        1 x 4 x 4,096 x 64 causal  371 / 1,144 -> 119 / 403
//   2 x 16 x 2,048 x 128  792 / 2,177 -> 515 / 2,089    2 x 8 x 1,000 x 128 causal  184 / 575 -> 92 / 342
//   8 x 16 x 512 x 32     51 / 157 -> 37 / 98           3 x 5 x 777 x 16  46 / 123 -> 16 / 41
#include <type_traits>

#include "bwd_pipe.h"
#include "common.h"
#include "launch.h"

namespace tattn {

namespace {

using H = H16<bf16>;
using V8 = bf16x8;

// Eight consecutive k values of an MFMA operand in three planes.
struct Planes {
  V8 hi, mid, lo;
};

__device__ __forceinline__ uint32_t bits(float x) { return __builtin_bit_cast(uint32_t, x); }
__device__ __forceinline__ float top(float x) { return __builtin_bit_cast(float, bits(x) & 0xffff0000u); }
__device__ __forceinline__ bf16x2 tops(float a, float b) {  // upper halves of a, b: exact for values that are bf16
  return __builtin_bit_cast(bf16x2, __builtin_amdgcn_perm(bits(b), bits(a), 0x07060302u));
}

// mid and lo rounded to nearest (lo exactly representable). hi: the nearest bf16 (ties away from zero) for
// operands that are LOADED, own rows and staged rows alike, so that S has the same bits in every kernel;
// truncated for those made in registers, which need no rounded copy then (with it the backward spills 16
// registers more: 4 x 16 x 1,024 x 64 345 -> 387 us). The rounding is an integer add (with v_cvt_pk dK/dV at head
// dim 64 takes 4 us more per launch: 256 x 128 rows 30.2 -> 34.4, against 30.3 with the add).
template <bool LOADED>
__device__ __forceinline__ void split2(float a, float b, bf16x2& hi, bf16x2& mid, bf16x2& lo) {
  const float ha = LOADED ? __builtin_bit_cast(float, bits(a) + 0x8000u) : a;
  const float hb = LOADED ? __builtin_bit_cast(float, bits(b) + 0x8000u) : b;
  hi = tops(ha, hb);
  const float ra = a - top(ha), rb = b - top(hb);
  mid = H::pack(ra, rb);
  const uint32_t m = __builtin_bit_cast(uint32_t, mid);
  lo = H::pack(ra - __builtin_bit_cast(float, m << 16), rb - __builtin_bit_cast(float, m & 0xffff0000u));
}
template <bool LOADED = false, typename F>
__device__ __forceinline__ Planes split8(F at) {
  Planes p;
#pragma unroll
  for (int i = 0; i < 8; i += 2) {
    bf16x2 h, m, l;
    split2<LOADED>(at(i), at(i + 1), h, m, l);
    p.hi[i] = h[0], p.hi[i + 1] = h[1];
    p.mid[i] = m[0], p.mid[i + 1] = m[1];
    p.lo[i] = l[0], p.lo[i + 1] = l[1];
  }
  return p;
}
// The float32 value again, for the float32 MFMA: raw planes hold the two halves of its bits (lo is not
// used), split ones its parts (exact from 2^-110 up).
__device__ __forceinline__ float whole(const Planes& p, int i, bool raw) {
  typedef uint16_t U8 __attribute__((ext_vector_type(8)));
  const U8 h = __builtin_bit_cast(U8, p.hi), m = __builtin_bit_cast(U8, p.mid);
  const uint32_t b = ((uint32_t)h[i] << 16) | m[i];
  return raw ? __builtin_bit_cast(float, b) : (float)p.hi[i] + ((float)p.mid[i] + (float)p.lo[i]);
}
__device__ __forceinline__ bf16x2 bottoms(float a, float b) {  // lower halves of the bits
  return __builtin_bit_cast(bf16x2, __builtin_amdgcn_perm(bits(b), bits(a), 0x05040100u));
}

// c += a b over 16 k values, smallest plane products first.
__device__ __forceinline__ f32x16 mm(const Planes& a, const Planes& b, f32x16 c) {
  using E = Elt<bf16>;
  c = E::mfma(a.lo, b.hi, c);
  c = E::mfma(a.hi, b.lo, c);
  c = E::mfma(a.mid, b.mid, c);
  c = E::mfma(a.mid, b.hi, c);
  c = E::mfma(a.hi, b.mid, c);
  return E::mfma(a.hi, b.hi, c);
}
// Two of them in turn, so that an MFMA need not wait for the one before it (a wave alone on its SIMD, head
// dim 128: backward of 2 x 16 x 2,048 2,241 -> 2,071 us; with two waves per SIMD no difference). swap exchanges the
// roles in the MFMA, not the order of the plane products: the backward's S, of queries by keys or of keys
// by queries, has the bits of the forward's, which M goes with.
__device__ __forceinline__ void mm2(const Planes& a, const Planes& b, f32x16& c, const Planes& x, const Planes& y, f32x16& z,
                                    bool swap = false) {
  auto one = [&](const V8& p, const V8& q, f32x16& r) __attribute__((always_inline)) {
    r = swap ? Elt<bf16>::mfma(q, p, r) : Elt<bf16>::mfma(p, q, r);
  };
  one(a.lo, b.hi, c);
  one(x.lo, y.hi, z);
  one(a.hi, b.lo, c);
  one(x.hi, y.lo, z);
  one(a.mid, b.mid, c);
  one(x.mid, y.mid, z);
  one(a.mid, b.hi, c);
  one(x.mid, y.hi, z);
  one(a.hi, b.mid, c);
  one(x.hi, y.mid, z);
  one(a.hi, b.hi, c);
  one(x.hi, y.hi, z);
}
// The same on the float32 MFMA: lane-half h holds k values 8 h + i of both operands. raw: how a is held.
template <typename F>
__device__ __forceinline__ f32x16 mm32(const Planes& a, bool raw, F b, f32x16 c) {
#pragma unroll
  for (int i = 0; i < 8; ++i) c = Elt<float>::mfma(whole(a, i, raw), b(i), c);
  return c;
}

// Whether a wave's operand values (the lane's largest magnitude, not-a-numbers aside) need the float32
// MFMA: an infinity or a number that bf16 rounds to one, or nothing but numbers so small that their planes
// may lose bits. (Gradients of a mean over many elements are ordinary down to 2^-60 or so: with the line at
// 2^-40 the backward of 4 x 16 x 1,024 x 64 took 675 us on them, the block kernels 531, the planes 341.)
constexpr float kLarge = 0x1.ffp127f, kSmall = 0x1p-100f;
__device__ __forceinline__ bool needs32(float amax) {
  return __builtin_amdgcn_ballot_w64(amax >= kLarge) != 0 ||
         (__builtin_amdgcn_ballot_w64(amax >= kSmall) == 0 && __builtin_amdgcn_ballot_w64(amax > 0.0f) != 0);
}

// A stage: CS pairs of [tensor][plane][32 rows]; rows in perm32 order, swizzled chunks (bwd_pipe.h).
template <int D, int RW, int CS>
struct Shape {
  static constexpr int NW = RW * CS, NSD = D / 16, DT = (D + 31) / 32;
  static constexpr int TILE = 32 * Swz<D>::RB, PAIR = 6 * TILE, STAGE = CS * PAIR;
  static constexpr int NBUF = (NW <= 4 && D <= 64) || 2 * STAGE > 110 * 1024 ? 1 : 2;
  static constexpr int GT = CS * 32 * (D / 4) / 64;      // 64-lane groups of 16-byte loads per tensor
  static constexpr int PW = (2 * GT + NW - 1) / NW;      // ... per wave and step, both tensors
  static_assert(GT * 64 == CS * 32 * (D / 4), "whole groups");
  static constexpr int PART = DT * 16 * 64 * 4;          // bytes of one wave's accumulator
  static_assert(CS == 1 || NW * PART <= NBUF * STAGE, "partials fit the stages");
};

// HBM -> registers -> planes in LDS. Rows past the end of the slice read as zero.
template <int D, int RW, int CS>
struct Stager {
  using S = Shape<D, RW, CS>;
  __amdgpu_buffer_rsrc_t ra, rb;
  uint32_t go[S::PW], step_a, step_b;
  int dst[S::PW], wu;
  f32x4 x[S::PW];
  __device__ __forceinline__ void init(__amdgpu_buffer_rsrc_t a, int64_t sa, __amdgpu_buffer_rsrc_t b, int64_t sb,
                                       int w, int lane) {
    ra = a;
    rb = b;
    wu = w;
    step_a = uniform32((uint32_t)(sa * (128 * CS)));
    step_b = uniform32((uint32_t)(sb * (128 * CS)));
#pragma unroll
    for (int i = 0; i < S::PW; ++i) {
      const int g = wu + i * S::NW;
      const bool second = g >= S::GT;
      const int j = (second ? g - S::GT : g) * 64 + lane;
      constexpr int CPR = D / 4;
      const int row = j / CPR, ch = j % CPR;
      go[i] = (uint32_t)(row * (second ? sb : sa) * 4 + ch * 16);
      dst[i] = (row >> 5) * S::PAIR + (second ? 3 * S::TILE : 0) + Swz<D>::addr(perm32(row & 31), ch * 8);
    }
  }
  __device__ __forceinline__ bool live(int i) const {
    return (2 * S::GT) % S::NW == 0 || wu + i * S::NW < 2 * S::GT;
  }
  __device__ __forceinline__ void load(int step) {
#pragma unroll
    for (int i = 0; i < S::PW; ++i) {
      if (!live(i)) continue;
      const bool second = wu + i * S::NW >= S::GT;
      x[i] = __builtin_bit_cast(f32x4, rsrc_load(second ? rb : ra, go[i] + (uint32_t)step * (second ? step_b : step_a)));
    }
  }
  // Writes the planes; returns whether this wave's values need the float32 MFMA.
  __device__ __forceinline__ bool store(char* stage) const {
    bool odd = false;
#pragma unroll
    for (int i = 0; i < S::PW; ++i) {
      if (!live(i)) continue;
      bf16x2 h[2], m[2], l[2];
      split2<true>(x[i][0], x[i][1], h[0], m[0], l[0]);
      split2<true>(x[i][2], x[i][3], h[1], m[1], l[1]);
      TATTN_LDS char* d = (TATTN_LDS char*)stage + dst[i];
      *reinterpret_cast<TATTN_LDS bf16x4*>(d) = bf16x4{h[0][0], h[0][1], h[1][0], h[1][1]};
      *reinterpret_cast<TATTN_LDS bf16x4*>(d + S::TILE) = bf16x4{m[0][0], m[0][1], m[1][0], m[1][1]};
      *reinterpret_cast<TATTN_LDS bf16x4*>(d + 2 * S::TILE) = bf16x4{l[0][0], l[0][1], l[1][0], l[1][1]};
      const float a = __builtin_fmaxf(__builtin_fabsf(x[i][0]), __builtin_fabsf(x[i][1]));
      odd |= needs32(__builtin_fmaxf(a, __builtin_fmaxf(__builtin_fabsf(x[i][2]), __builtin_fabsf(x[i][3]))));
    }
    return odd;
  }
};

// The rows last loaded, as raw planes.
template <int D, int RW, int CS>
__device__ __forceinline__ void store_raw(const Stager<D, RW, CS>& ld, char* stage) {
  using S = Shape<D, RW, CS>;
#pragma unroll
  for (int i = 0; i < S::PW; ++i) {
    if (!ld.live(i)) continue;
    TATTN_LDS char* d = (TATTN_LDS char*)stage + ld.dst[i];
    const f32x4 x = ld.x[i];
    const bf16x2 h0 = tops(x[0], x[1]), h1 = tops(x[2], x[3]), m0 = bottoms(x[0], x[1]), m1 = bottoms(x[2], x[3]);
    *reinterpret_cast<TATTN_LDS bf16x4*>(d) = bf16x4{h0[0], h0[1], h1[0], h1[1]};
    *reinterpret_cast<TATTN_LDS bf16x4*>(d + S::TILE) = bf16x4{m0[0], m0[1], m1[0], m1[1]};
  }
}

// Operand addresses in one stage (the wave's pair): natural rows, transposed reads of 16-row slice 0.
template <int D, int PAIRB>
struct Operands {
  static constexpr int NSD = D / 16, DT = (D + 31) / 32, TILE = 32 * Swz<D>::RB;
  int nat[NSD], lo[DT], hi[DT];
  bool upper;  // D = 16: the lane's column of a transposed read does not exist
  __device__ __forceinline__ void init(int cs, int lane) {
    const int l32 = lane & 31, h2 = lane >> 5, base = cs * PAIRB;
#pragma unroll
    for (int s = 0; s < NSD; ++s) nat[s] = base + Swz<D>::addr(l32, (16 * s + 8 * h2) * 2);
#pragma unroll
    for (int u = 0; u < DT; ++u) {
      tr_addrs<D>(0, u, lane, lo[u], hi[u]);
      lo[u] += base;
      hi[u] += base;
    }
    upper = D < 32 && 16 * ((lane >> 4) & 1) >= D;
  }
  __device__ __forceinline__ Planes natural(const char* st, int tensor, int sd) const {
    const char* p = st + tensor * 3 * TILE + nat[sd];
    return {lds8<bf16>(p), lds8<bf16>(p + TILE), lds8<bf16>(p + 2 * TILE)};
  }
  __device__ __forceinline__ Planes transposed(const char* st, int tensor, int sl, int u) const {
    const char* p = st + tensor * 3 * TILE + 16 * sl * Swz<D>::RB;
    Planes x{tr_pair<bf16>(p, lo[u], hi[u]), tr_pair<bf16>(p + TILE, lo[u], hi[u]),
             tr_pair<bf16>(p + 2 * TILE, lo[u], hi[u])};
    if (D < 32 && upper) x = Planes{};
    return x;
  }
};

// A wave's own 32 rows as MFMA operands (zero past the end): in registers, or in LDS where OL says so
// ([s][plane][lane]; the CS waves of a row tile write the same values to the same place).
template <int NSD, bool OL>
struct OwnRows {
  Planes reg[OL ? 1 : NSD];
  char* lds;
  const float* src;
  bool valid;
  __device__ __forceinline__ void set(int s, const Planes& p) {
    if constexpr (OL) {
      TATTN_LDS char* d = (TATTN_LDS char*)lds + 3072 * s;
      *reinterpret_cast<TATTN_LDS V8*>(d) = p.hi;
      *reinterpret_cast<TATTN_LDS V8*>(d + 1024) = p.mid;
      *reinterpret_cast<TATTN_LDS V8*>(d + 2048) = p.lo;
    } else {
      reg[s] = p;
    }
  }
  template <typename F>
  __device__ __forceinline__ void each(F f) {
#pragma unroll
    for (int s = 0; s < NSD; ++s) {
      f32x4 a = *reinterpret_cast<const f32x4*>(src + 16 * s), b = *reinterpret_cast<const f32x4*>(src + 16 * s + 4);
      if (!valid) a = b = f32x4{};
      f(s, a, b);
    }
  }
  // Returns whether the rows need the float32 MFMA.
  __device__ __forceinline__ bool init(char* base, int lane, const float* rows, bool ok) {
    lds = base + 16 * lane;
    src = rows;
    valid = ok;
    float amax = 0.0f;
    each([&](int s, f32x4 a, f32x4 b) __attribute__((always_inline)) {
#pragma unroll
      for (int i = 0; i < 4; ++i) amax = __builtin_fmaxf(amax, __builtin_fmaxf(__builtin_fabsf(a[i]), __builtin_fabsf(b[i])));
      set(s, split8<true>([&](int i) { return i < 4 ? a[i & 3] : b[i & 3]; }));
    });
    return needs32(amax);
  }
  __device__ __forceinline__ void raw() {
    each([&](int s, f32x4 a, f32x4 b) __attribute__((always_inline)) {
      Planes p{};
#pragma unroll
      for (int i = 0; i < 8; i += 2) {
        const float x = i < 4 ? a[i & 3] : b[i & 3], y = i < 4 ? a[(i + 1) & 3] : b[(i + 1) & 3];
        const bf16x2 h = tops(x, y), m = bottoms(x, y);
        p.hi[i] = h[0], p.hi[i + 1] = h[1];
        p.mid[i] = m[0], p.mid[i + 1] = m[1];
      }
      set(s, p);
    });
  }
  __device__ __forceinline__ Planes operator[](int s) const {
    if constexpr (OL) return {lds8<bf16>(lds + 3072 * s), lds8<bf16>(lds + 3072 * s + 1024), lds8<bf16>(lds + 3072 * s + 2048)};
    else return reg[s];
  }
};
__device__ __forceinline__ uint64_t slice_bytes4(int64_t N, int64_t rs, int64_t D) { return (uint64_t)((N - 1) * rs + D) * 4; }

// The steps of a workgroup: next step's rows are fetched while this one's are worked on. odd: per
// buffer and wave, whether what it staged, or its own rows, need the float32 MFMA; any such wave takes the
// whole workgroup there for the step, so that the barrier in it is met by all.
template <int D, int RW, int CS, typename Work>
__device__ __forceinline__ void run_steps(Stager<D, RW, CS>& ld, char* smem, int (*odd)[RW * CS], bool own32, int nsteps, int wu,
                                          int lane, Work work) {
  using S = Shape<D, RW, CS>;
  ld.load(0);
  auto put = [&](int b) {
    const bool o = ld.store(smem + b * S::STAGE) || own32;
    if (lane == 0) odd[b][wu] = o;
  };
  put(0);
  __syncthreads();
  for (int i = 0; i < nsteps; ++i) {
    const int b = S::NBUF == 2 ? i & 1 : 0;
    const bool more = i + 1 < nsteps;
    const bool slow = __builtin_amdgcn_ballot_w64(odd[b][lane % S::NW] != 0) != 0;
    if (slow) {
      store_raw(ld, smem + b * S::STAGE);
      __syncthreads();
    }
    if (more) ld.load(i + 1);
    work(smem + b * S::STAGE, i, slow);
    if (S::NBUF == 1 && more) __syncthreads();
    if (more) put(S::NBUF == 2 ? b ^ 1 : 0);
    __syncthreads();
  }
}

// ---- forward ---------------------------------------------------------------------------------
template <int D, int RW, int CS, int OCC, bool CAUSAL>
__global__ __launch_bounds__(RW * CS * 64, OCC) void fwd_f32_kernel(const FwdParams p) {
  using S = Shape<D, RW, CS>;
  constexpr int NW = S::NW, NSD = S::NSD, DT = S::DT;
  __shared__ __attribute__((aligned(1024))) char smem[S::NBUF * S::STAGE];
  __shared__ int odd[2][NW];
  __shared__ float red[2][NW][32];

  const int tid = threadIdx.x;
  const int lane = tid & 63, h2 = lane >> 5, l32 = lane & 31;
  const int wu = (int)uniform32((uint32_t)(tid >> 6));
  const int rw = wu / CS, cs = wu % CS;
  const int N = p.N;
  const float c = p.c;
  const BlockCoord bc = block_coord(p.Z * p.H, p.n_qblocks, !CAUSAL);
  const int zh = bc.zh, qb = CAUSAL ? p.n_qblocks - 1 - bc.blk : bc.blk;  // longest rows first
  const int ntile = (N + 31) / 32;
  const int qt = qb * RW + rw;
  const int q = 32 * qt + l32;
  const int btiles = CAUSAL ? min(ntile, (qb + 1) * RW) : ntile;
  const int wtiles = qt >= ntile ? 0 : CAUSAL ? qt + 1 : ntile;
  const int nsteps = (btiles + CS - 1) / CS;

  Stager<D, RW, CS> ld;
  ld.init(slice_rsrc((const float*)p.k + slice_off(p.sk, zh, p.H), slice_bytes4(N, p.sk[2], D)), p.sk[2],
          slice_rsrc((const float*)p.v + slice_off(p.sv, zh, p.H), slice_bytes4(N, p.sv[2], D)), p.sv[2], wu, lane);
  OwnRows<NSD, false> qop;
  const bool own32 = qop.init(nullptr, lane, (const float*)p.q + slice_off(p.sq, zh, p.H) + (int64_t)(q < N ? q : 0) * p.sq[2] + 8 * h2,
                              q < N);
  if (own32) qop.raw();
  Operands<D, S::PAIR> at;
  at.init(cs, lane);

  const int lim = CAUSAL ? min(q, N - 1) : N - 1;  // last key the lane's row sees
  float mrow = -__builtin_inff(), lrow = 0.0f;
  f32x16 acc[DT];
#pragma unroll
  for (int u = 0; u < DT; ++u) acc[u] = f32x16{};

  run_steps<D, RW, CS>(ld, smem, odd, own32, nsteps, wu, lane, [&](const char* st, int i, bool slow) __attribute__((always_inline)) {
    const int t = i * CS + cs;
    if (t >= wtiles) return;
    f32x16 s = f32x16{};
    if (!slow) {
#pragma unroll
      for (int sd = 0; sd < NSD; ++sd) s = mm(at.natural(st, 0, sd), qop[sd], s);
    } else {
#pragma unroll
      for (int sd = 0; sd < NSD; ++sd) s = mm32(at.natural(st, 0, sd), true, [&, o = qop[sd]](int e) { return whole(o, e, own32); }, s);
    }
    // Scaled scores; hidden keys leave the max and get probability 0.
    const bool mask = 32 * t + 32 > N || (CAUSAL && t == qt);
    const int past = lim - 32 * t - 8 * h2;
    float mx = -__builtin_inff();
    if (mask) {
#pragma unroll
      for (int r = 0; r < 16; ++r) mx = kappa(r, 0) > past ? mx : __builtin_fmaxf(mx, s[r] * c);
    } else {
#pragma unroll
      for (int r = 0; r < 16; ++r) mx = __builtin_fmaxf(mx, s[r] * c);
    }
    const float cand = max_halves(mx);
    const bool up = cand > mrow + kRescaleLog2;
    if (__builtin_amdgcn_ballot_w64(up)) {
      const float alpha = up ? fast_exp2(mrow - cand) : 1.0f;  // a row that stays at -inf stays as it is
      mrow = up ? cand : mrow;
      lrow *= alpha;
#pragma unroll
      for (int u = 0; u < DT; ++u) acc[u] *= alpha;
    }
    // No key with a score above -inf so far: exponents against 0 (probability 0), not against -inf.
    const float base = mrow == -__builtin_inff() ? 0.0f : mrow;
#pragma unroll
    for (int r = 0; r < 16; ++r) s[r] = __builtin_fmaf(s[r], c, -base);
    // The max is a rounded product, which the FMA does not round: an exponent is at most kRescaleLog2 plus
    // half an ulp of the max. That is below 2 up to 2^24; beyond it (keys hidden by a huge negative score,
    // all that this wave has seen so far) it is cut, or P would be infinite and 0 times it, where a later
    // tile or another wave raises the max, not 0.
    if (__builtin_amdgcn_ballot_w64(__builtin_fabsf(base) > 0x1p24f)) {
#pragma unroll
      for (int r = 0; r < 16; ++r) s[r] = s[r] > kRescaleLog2 + 2.0f ? kRescaleLog2 + 2.0f : s[r];
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) s[r] = fast_exp2(s[r]);
    if (mask) {
#pragma unroll
      for (int r = 0; r < 16; ++r) s[r] = kappa(r, 0) > past ? 0.0f : s[r];
    }
    float ps[4];
#pragma unroll
    for (int r = 0; r < 16; ++r) ps[r & 3] = r < 4 ? s[r] : ps[r & 3] + s[r];
    lrow += (ps[0] + ps[1]) + (ps[2] + ps[3]);
    if (!slow) {
#pragma unroll
      for (int sl = 0; sl < 2; ++sl) {
        const Planes x = split8([&](int e) { return s[8 * sl + e]; });
#pragma unroll
        for (int u = 0; u + 1 < DT; u += 2)
          mm2(at.transposed(st, 1, sl, u), x, acc[u], at.transposed(st, 1, sl, u + 1), x, acc[u + 1]);
        if constexpr (DT == 1) acc[0] = mm(at.transposed(st, 1, sl, 0), x, acc[0]);
      }
    } else {
#pragma unroll
      for (int sl = 0; sl < 2; ++sl)
#pragma unroll
        for (int u = 0; u < DT; ++u)
          acc[u] = mm32(at.transposed(st, 1, sl, u), slow, [&](int e) { return s[8 * sl + e]; }, acc[u]);
    }
  });

  const float lt = sum_halves(lrow);
  float* orow = (float*)p.o + slice_off(p.so, zh, p.H) + (int64_t)q * p.so[2];
  if constexpr (CS == 1) {
    const float inv = 1.0f / lt;
    if (q < N) {
#pragma unroll
      for (int gr = 0; gr < DT * 4; ++gr) {
        const int d0 = 8 * gr + 4 * h2;
        if (d0 < D) {
          f32x4 y;
#pragma unroll
          for (int e = 0; e < 4; ++e) y[e] = acc[gr >> 2][4 * (gr & 3) + e] * inv;
          *reinterpret_cast<f32x4*>(orow + d0) = y;
        }
      }
      if (h2 == 0 && p.m) p.m[(int64_t)zh * N + q] = mrow + __log2f(lt);
    }
  } else {
    // Merge the CS partial rows: O = sum_c 2^(m_c - m) O_c / l, l likewise. A wave that saw no tile has
    // m_c = -inf and adds nothing. (The stages are free: all waves passed the last barrier.)
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
    for (int k = 0; k < CS; ++k) lall += fast_exp2(red[0][rw * CS + k][l32] - mall) * red[1][rw * CS + k][l32];
    const float wgt = fast_exp2(mrow - mall) / lall;
    TATTN_LDS float* dst = (TATTN_LDS float*)(smem + wu * S::PART) + lane;
#pragma unroll
    for (int u = 0; u < DT; ++u)
#pragma unroll
      for (int r = 0; r < 16; ++r) dst[(16 * u + r) * 64] = acc[u][r] * wgt;
    __syncthreads();
    if (q < N) {
      for (int gr = cs; gr < DT * 4; gr += CS) {
        const int d0 = 8 * gr + 4 * h2;
        if (d0 < D) {
          f32x4 y = f32x4{};
#pragma unroll
          for (int k = 0; k < CS; ++k) {
            const TATTN_LDS float* src = (const TATTN_LDS float*)(smem + (rw * CS + k) * S::PART) + lane + 4 * gr * 64;
#pragma unroll
            for (int e = 0; e < 4; ++e) y[e] += src[64 * e];
          }
          *reinterpret_cast<f32x4*>(orow + d0) = y;
        }
      }
      if (cs == 0 && h2 == 0 && p.m) p.m[(int64_t)zh * N + q] = mall + __log2f(lall);
    }
  }
}

// Whether the planes hold a tile's probabilities or dS (the MFMA operands made in registers).
__device__ __forceinline__ bool planes_hold(const f32x16& a) {
  float m = 0.0f;
#pragma unroll
  for (int r = 0; r < 16; ++r) m = __builtin_fmaxf(m, __builtin_fabsf(a[r]));
  return !needs32(m);
}

// ---- dQ --------------------------------------------------------------------------------------
template <int D, int RW, int CS, int OCC, bool CAUSAL>
__global__ __launch_bounds__(RW * CS * 64, OCC) void dq_f32_kernel(const BwdParams p) {
  using S = Shape<D, RW, CS>;
  constexpr int NW = S::NW, NSD = S::NSD, DT = S::DT;
  __shared__ __attribute__((aligned(1024))) char smem[S::NBUF * S::STAGE];
  __shared__ int odd[2][NW];
  constexpr bool OL = OCC == 2 && D == 64;
  __shared__ __attribute__((aligned(16))) char own[OL ? RW * NSD * 3072 : 16];

  const int tid = threadIdx.x;
  const int lane = tid & 63, h2 = lane >> 5, l32 = lane & 31;
  const int wu = (int)uniform32((uint32_t)(tid >> 6));
  const int rw = wu / CS, cs = wu % CS;
  const int N = p.N;
  const float c = p.c;
  const BlockCoord bc = block_coord(p.Z * p.H, p.n_blocks, !CAUSAL);
  const int zh = bc.zh, qb = CAUSAL ? p.n_blocks - 1 - bc.blk : bc.blk;
  const int ntile = (N + 31) / 32;
  const int qt = qb * RW + rw;
  const int q = 32 * qt + l32;
  const int btiles = CAUSAL ? min(ntile, (qb + 1) * RW) : ntile;
  const int wtiles = qt >= ntile ? 0 : CAUSAL ? qt + 1 : ntile;
  const int nsteps = (btiles + CS - 1) / CS;
  const int64_t hoff = slice_off(p.s, zh, p.H), rs = p.s[2];

  Stager<D, RW, CS> ld;
  ld.init(slice_rsrc((const float*)p.k + hoff, slice_bytes4(N, rs, D)), rs,
          slice_rsrc((const float*)p.v + hoff, slice_bytes4(N, rs, D)), rs, wu, lane);
  const int64_t off = hoff + (int64_t)(q < N ? q : 0) * rs + 8 * h2;
  OwnRows<NSD, OL> qop;
  OwnRows<NSD, false> dop;
  const bool q32 = qop.init(own + (OL ? rw * NSD * 3072 : 0), lane, (const float*)p.q + off, q < N);
  const bool own32 = dop.init(nullptr, lane, (const float*)p.dout + off, q < N) || q32;
  if (own32) {
    qop.raw();
    dop.raw();
  }
  const float nm = -(q < N ? p.m[(int64_t)zh * N + q] : 0.0f);
  float dl;
  if (p.fuse_delta) {  // delta = rowsum(dO * O) in the preprocess's order, stored for the dK/dV kernel
    float part[2][NSD];
#pragma unroll
    for (int s = 0; s < NSD; ++s)
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const f32x4 x = *reinterpret_cast<const f32x4*>((const float*)p.o + off + 16 * s + 4 * j);
        const f32x4 y = *reinterpret_cast<const f32x4*>((const float*)p.dout + off + 16 * s + 4 * j);
        float a = 0.0f;
#pragma unroll
        for (int e = 0; e < 4; ++e) a += x[e] * y[e];
        part[j][s] = a;
      }
    dl = row_delta(part[0]) + row_delta(part[1]);
    if (q >= N) dl = 0.0f;
    else if (h2 == 0 && cs == 0) p.delta[(int64_t)zh * N + q] = dl;
  } else {
    dl = q < N ? p.delta[(int64_t)zh * N + q] : 0.0f;
  }
  Operands<D, S::PAIR> at;
  at.init(cs, lane);
  const int lim = CAUSAL ? min(q, N - 1) : N - 1;
  f32x16 dq[DT];
#pragma unroll
  for (int u = 0; u < DT; ++u) dq[u] = f32x16{};

  run_steps<D, RW, CS>(ld, smem, odd, own32, nsteps, wu, lane, [&](const char* st, int i, bool slow) __attribute__((always_inline)) {
    const int t = i * CS + cs;
    if (t >= wtiles) return;
    f32x16 s = f32x16{}, dp = f32x16{};
    if (!slow) {
#pragma unroll
      for (int sd = 0; sd < NSD; ++sd) {
        mm2(at.natural(st, 0, sd), qop[sd], s, at.natural(st, 1, sd), dop[sd], dp);
      }
    } else {
#pragma unroll
      for (int sd = 0; sd < NSD; ++sd) {
        s = mm32(at.natural(st, 0, sd), true, [&, o = qop[sd]](int e) { return whole(o, e, own32); }, s);
        dp = mm32(at.natural(st, 1, sd), true, [&, o = dop[sd]](int e) { return whole(o, e, own32); }, dp);
      }
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) s[r] = fast_exp2(__builtin_fmaf(s[r], c, nm));
    if (32 * t + 32 > N || (CAUSAL && t == qt)) {  // hidden keys: probability 0
      const int past = lim - 32 * t - 8 * h2;
#pragma unroll
      for (int r = 0; r < 16; ++r) s[r] = kappa(r, 0) > past ? 0.0f : s[r];
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) s[r] *= dp[r] - dl;
    if (!slow && planes_hold(s)) {
#pragma unroll
      for (int sl = 0; sl < 2; ++sl) {
        const Planes x = split8([&](int e) { return s[8 * sl + e]; });
#pragma unroll
        for (int u = 0; u + 1 < DT; u += 2)
          mm2(at.transposed(st, 0, sl, u), x, dq[u], at.transposed(st, 0, sl, u + 1), x, dq[u + 1]);
        if constexpr (DT == 1) dq[0] = mm(at.transposed(st, 0, sl, 0), x, dq[0]);
      }
    } else {
#pragma unroll
      for (int sl = 0; sl < 2; ++sl)
#pragma unroll
        for (int u = 0; u < DT; ++u)
          dq[u] = mm32(at.transposed(st, 0, sl, u), slow, [&](int e) { return s[8 * sl + e]; }, dq[u]);
    }
  });

  float* row = (float*)p.dq + slice_off(p.so, zh, p.H) + (int64_t)q * p.so[2];
  if constexpr (CS == 1) {
    if (q < N) {
#pragma unroll
      for (int gr = 0; gr < DT * 4; ++gr) {
        const int d0 = 8 * gr + 4 * h2;
        if (d0 < D) {
          f32x4 y;
#pragma unroll
          for (int e = 0; e < 4; ++e) y[e] = dq[gr >> 2][4 * (gr & 3) + e] * p.scale;
          *reinterpret_cast<f32x4*>(row + d0) = y;
        }
      }
    }
  } else {
    TATTN_LDS float* dst = (TATTN_LDS float*)(smem + wu * S::PART) + lane;
#pragma unroll
    for (int u = 0; u < DT; ++u)
#pragma unroll
      for (int r = 0; r < 16; ++r) dst[(16 * u + r) * 64] = dq[u][r];
    __syncthreads();
    if (q < N) {
      for (int gr = cs; gr < DT * 4; gr += CS) {
        const int d0 = 8 * gr + 4 * h2;
        if (d0 < D) {
          f32x4 y = f32x4{};
#pragma unroll
          for (int k = 0; k < CS; ++k) {
            const TATTN_LDS float* src = (const TATTN_LDS float*)(smem + (rw * CS + k) * S::PART) + lane + 4 * gr * 64;
#pragma unroll
            for (int e = 0; e < 4; ++e) y[e] += src[64 * e];
          }
#pragma unroll
          for (int e = 0; e < 4; ++e) y[e] *= p.scale;
          *reinterpret_cast<f32x4*>(row + d0) = y;
        }
      }
    }
  }
}

// ---- dK / dV ---------------------------------------------------------------------------------
template <int D, int RW, int CS, int OCC, bool CAUSAL>
__global__ __launch_bounds__(RW * CS * 64, OCC) void dkdv_f32_kernel(const BwdParams p) {
  using S = Shape<D, RW, CS>;
  constexpr int NW = S::NW, NSD = S::NSD, DT = S::DT;
  __shared__ __attribute__((aligned(1024))) char smem[S::NBUF * S::STAGE];
  __shared__ int odd[2][NW];
  constexpr bool OL = OCC == 2 && D == 64;
  __shared__ __attribute__((aligned(16))) char own[OL ? RW * NSD * 3072 : 16];
  __shared__ __attribute__((aligned(16))) float md[NW][2][64];  // per wave and parity: M[32], delta[32]

  const int tid = threadIdx.x;
  const int lane = tid & 63, h2 = lane >> 5, l32 = lane & 31;
  const int wu = (int)uniform32((uint32_t)(tid >> 6));
  const int rw = wu / CS, cs = wu % CS;
  const int N = p.N;
  const float c = p.c;
  const BlockCoord bc = block_coord(p.Z * p.H, p.n_blocks, !CAUSAL);
  const int zh = bc.zh, kb = bc.blk;  // causal: small key blocks (most work) first
  const int ntile = (N + 31) / 32;
  const int kt = kb * RW + rw;
  const int key = 32 * kt + l32;
  const int lo = CAUSAL ? kb * RW : 0;  // first query tile the block sees
  const int nsteps = (ntile - lo + CS - 1) / CS;
  const int64_t hoff = slice_off(p.s, zh, p.H), rs = p.s[2];

  Stager<D, RW, CS> ld;
  {
    const int64_t o = hoff + (int64_t)(32 * lo) * rs;
    const uint64_t bytes = slice_bytes4(N - 32 * lo, rs, D);
    ld.init(slice_rsrc((const float*)p.q + o, bytes), rs, slice_rsrc((const float*)p.dout + o, bytes), rs, wu, lane);
  }
  // Lanes 0-31 fetch M and lanes 32-63 delta of the wave's tile of a step; zero past the end.
  const float* mdsrc = (h2 ? p.delta : p.m) + (int64_t)zh * N;
  auto md_load = [&](int i) {
    const int q = 32 * (lo + i * CS + cs) + l32;
    return q < N ? mdsrc[q] : 0.0f;
  };
  md[wu][0][lane] = md_load(0);
  OwnRows<NSD, OL> kop;
  OwnRows<NSD, false> vop;
  const int64_t off = hoff + (int64_t)(key < N ? key : 0) * rs + 8 * h2;
  const bool k32 = kop.init(own + (OL ? rw * NSD * 3072 : 0), lane, (const float*)p.k + off, key < N);
  const bool own32 = vop.init(nullptr, lane, (const float*)p.v + off, key < N) || k32;
  if (own32) {
    kop.raw();
    vop.raw();
  }
  Operands<D, S::PAIR> at;
  at.init(cs, lane);
  f32x16 dk[DT], dv[DT];
#pragma unroll
  for (int u = 0; u < DT; ++u) dk[u] = dv[u] = f32x16{};

  auto tile = [&](const char* st, const float* mdw, int t, bool slow) __attribute__((always_inline)) {
    if (t >= ntile || kt >= ntile || (CAUSAL && t < kt)) return;
    f32x16 s = f32x16{}, dp = f32x16{};
    if (!slow) {
#pragma unroll
      for (int sd = 0; sd < NSD; ++sd) {
        mm2(kop[sd], at.natural(st, 0, sd), s, vop[sd], at.natural(st, 1, sd), dp, true);
      }
    } else {
#pragma unroll
      for (int sd = 0; sd < NSD; ++sd) {
        s = mm32(at.natural(st, 0, sd), true, [&, o = kop[sd]](int e) { return whole(o, e, own32); }, s);
        dp = mm32(at.natural(st, 1, sd), true, [&, o = vop[sd]](int e) { return whole(o, e, own32); }, dp);
      }
    }
#pragma unroll
    for (int a = 0; a < 4; ++a) {
      const int at4 = 16 * (a >> 1) + 8 * h2 + 4 * (a & 1);
      const f32x4 m4 = *reinterpret_cast<const TATTN_LDS f32x4*>((const TATTN_LDS float*)mdw + at4);
      const f32x4 d4 = *reinterpret_cast<const TATTN_LDS f32x4*>((const TATTN_LDS float*)mdw + 32 + at4);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        s[4 * a + e] = fast_exp2(__builtin_fmaf(s[4 * a + e], c, -m4[e]));
        dp[4 * a + e] -= d4[e];
      }
    }
    if (CAUSAL && t == kt) {  // queries of the tile before the lane's key: probability 0
      const int before = key - 32 * t - 8 * h2;
#pragma unroll
      for (int r = 0; r < 16; ++r) s[r] = kappa(r, 0) < before ? 0.0f : s[r];
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) dp[r] *= s[r];
    if (!slow && planes_hold(s) && planes_hold(dp)) {
#pragma unroll
      for (int sl = 0; sl < 2; ++sl) {
        const Planes x = split8([&](int e) { return s[8 * sl + e]; });
        const Planes y = split8([&](int e) { return dp[8 * sl + e]; });
#pragma unroll
        for (int u = 0; u < DT; ++u) mm2(x, at.transposed(st, 1, sl, u), dv[u], y, at.transposed(st, 0, sl, u), dk[u]);
      }
    } else {
#pragma unroll
      for (int sl = 0; sl < 2; ++sl)
#pragma unroll
        for (int u = 0; u < DT; ++u) {
          const Planes o = at.transposed(st, 1, sl, u), q = at.transposed(st, 0, sl, u);
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            dv[u] = Elt<float>::mfma(s[8 * sl + e], whole(o, e, slow), dv[u]);
            dk[u] = Elt<float>::mfma(dp[8 * sl + e], whole(q, e, slow), dk[u]);
          }
        }
    }
  };
  run_steps<D, RW, CS>(ld, smem, odd, own32, nsteps, wu, lane, [&](const char* st, int i, bool slow) __attribute__((always_inline)) {
    const float next = i + 1 < nsteps ? md_load(i + 1) : 0.0f;
    tile(st, md[wu][i & 1], lo + i * CS + cs, slow);
    md[wu][(i & 1) ^ 1][lane] = next;  // the wave's own rows: no barrier needed
  });

  // C register r of a lane: key 8 (r/4) + 4 h2 + r%4 of the tile, column 32 u + l32.
  const int64_t goff = slice_off(p.so, zh, p.H);
  auto put = [&](const f32x16 (&a)[DT], float mul, float* dst) __attribute__((always_inline)) {
    if constexpr (CS == 1) {
#pragma unroll
      for (int g = 0; g < DT * 16; ++g) {
        const int u = g >> 4, r = g & 15;
        const int row = 32 * kt + 8 * (r >> 2) + 4 * h2 + (r & 3), d = 32 * u + l32;
        if (row < N && d < D) dst[(int64_t)row * p.so[2] + d] = a[u][r] * mul;
      }
    } else {
      TATTN_LDS float* mine = (TATTN_LDS float*)(smem + wu * S::PART) + lane;
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
        for (int k = 0; k < CS; ++k) x += ((const TATTN_LDS float*)(smem + (rw * CS + k) * S::PART) + lane)[g * 64];
        if (row < N && d < D) dst[(int64_t)row * p.so[2] + d] = x * mul;
      }
      __syncthreads();
    }
  };
  put(dk, p.scale, (float*)p.dk + goff);
  put(dv, 1.0f, (float*)p.dv + goff);
}

// Launch shapes {row tiles, tile pairs per step}.
enum Pick { ROWS, HALF, FEW, SHORT };
template <int D, Pick W> struct Launch {
  static constexpr int RW = W == FEW ? 2 : W == SHORT ? 1 : 4;
  static constexpr int CS = W == HALF || (W == FEW && D == 128) ? 2 : W == FEW ? 4 : 1;
  static constexpr int OCC = D == 128 ? 1 : 2;
};

// The shape with the least time on the busiest CU, from what a step of a workgroup takes (us, forward,
// head dim 64): {4, 1} 2.0 alone on a CU and 3.2 for two side by side, {4, 2} 3.2 (2.8 where the longest
// causal chain sets the time), {2, 4} 4.2 (3.6); head dim 128 {4, 1} 4.0, {2, 2} 5.9. Merging partial
// results takes about 1.6. Causal: total work over the CUs, or the longest workgroup. Measured (forward
// / backward, us, {4, 1}, {4, 2}, {2, 4}): 4 x 16 x 1,024 x 64: 103 / 343, 106 / 378, 135 / 480; causal: 73 / 266,
// 63 / 232, 86 / 308; 1 x 16 x 2,048: 129 / 410, 102 / 357, 123 / 435; 1 x 4 x 4,096 causal: 247 / 828, 166 / 566,
// 113 / 383; 32 x 8 x 128: 15 / 48, 15 / 51, 21 / 77. At most 32 rows (64 backward): one wave per row tile
// (256 x 8 x 16 x 64: 24 / 81 -> 22 / 48; 64 x 8 x 64 x 64: 13 / 47, 16 / 37).
Pick pick_shape(int D, int64_t zh, int64_t n, bool causal, bool backward) {
  if (D < 128 && n <= (backward ? 64 : 32)) return SHORT;
  auto cost = [&](int rw, int cs, double one, double two, double chain, double merge) {
    const double wgs = (double)(zh * ((n + 32 * rw - 1) / (32 * rw))), steps = (double)((n + 32 * cs - 1) / (32 * cs));
    if (causal) {
      const double mean = __builtin_fmin(steps, (steps + __builtin_fmax(1.0, (double)rw / cs)) / 2);
      return __builtin_fmax(wgs * mean / 256 * two / 2, steps * chain) + merge;
    }
    const int64_t k = ((int64_t)wgs + 255) / 256;
    return steps * ((double)(k / 2) * two + (double)(k % 2) * one) + merge;
  };
  if (D == 128) {
    // Causal, {2, 2}: one workgroup fills a CU, and with more workgroups than CUs some CU gets two long ones unless
    // the chain is long (against {4, 1}, us, forward / backward: 100 x 146 35 / 166, 27 / 117; 3,000 x 146 706 / 3,533,
    // 597 / 2,455; 64 x 400 58 / 263, 57 / 240; 32 x 800 82 / 350, 102 / 411; 16 x 2,048 203 / 854, 256 / 1,006).
    const int64_t wgs = zh * ((n + 63) / 64);
    if (causal && wgs > 256 && (n <= 256 || wgs > (backward && n < 768 ? 384 : 512))) return ROWS;
    return cost(2, 2, 5.9, 11.8, 5.9, 1.6) < cost(4, 1, 4.0, 8.0, 4.0, 0.0) ? FEW : ROWS;
  }
  const double rows = cost(4, 1, 2.0, 3.2, 2.0, 0.0), half = cost(4, 2, 3.2, 6.4, 2.8, 1.6), few = cost(2, 4, 4.2, 8.4, 3.6, 1.6);
  return few < rows && few < half ? FEW : half < rows ? HALF : ROWS;
}

#define TATTN_F32_LAUNCH(NAME, KERNEL, PARAMS, BLOCKS, WHAT)                                        \
  template <int D, Pick W>                                                                         \
  int NAME(PARAMS p, bool causal, hipStream_t st) {                                                \
    using L = Launch<D, W>;                                                                        \
    p.BLOCKS = (p.N + 32 * L::RW - 1) / (32 * L::RW);                                              \
    const dim3 grid((unsigned)((int64_t)p.BLOCKS * p.Z * p.H)), block(L::RW * L::CS * 64);          \
    if (causal) KERNEL<D, L::RW, L::CS, L::OCC, true><<<grid, block, 0, st>>>(p);                   \
    else KERNEL<D, L::RW, L::CS, L::OCC, false><<<grid, block, 0, st>>>(p);                         \
    return check_launch(WHAT);                                                                     \
  }
TATTN_F32_LAUNCH(fwd_launch, fwd_f32_kernel, FwdParams, n_qblocks, "tattn_fwd")
TATTN_F32_LAUNCH(dq_launch, dq_f32_kernel, BwdParams, n_blocks, "tattn_bwd_dq")
TATTN_F32_LAUNCH(dkdv_launch, dkdv_f32_kernel, BwdParams, n_blocks, "tattn_bwd_dkdv")

#define TATTN_F32_CASE(FN, D_, BWD)                                                   \
  case D_:                                                                            \
    switch (pick_shape(D_, (int64_t)p.Z * p.H, p.N, causal, BWD)) {                   \
      case SHORT: return FN<D_, D_ == 128 ? ROWS : SHORT>(p, causal, st);             \
      case HALF: return FN<D_, D_ == 128 ? ROWS : HALF>(p, causal, st);               \
      case FEW: return FN<D_, FEW>(p, causal, st);                                    \
      default: return FN<D_, ROWS>(p, causal, st);                                    \
    }
#define TATTN_F32_SWITCH(FN, BWD)                                                       \
  switch (D) {                                                                         \
    TATTN_F32_CASE(FN, 16, BWD) TATTN_F32_CASE(FN, 32, BWD) TATTN_F32_CASE(FN, 64, BWD) \
    TATTN_F32_CASE(FN, 128, BWD)                                                       \
  }                                                                                    \
  return set_error(TATTN_E_ARG, "head dim must be 16, 32, 64 or 128, got %d", D);

}  // namespace

int launch_fwd_f32(const FwdParams& p, int D, bool causal, hipStream_t st) { TATTN_F32_SWITCH(fwd_launch, false) }
int launch_dq_f32(const BwdParams& p, int D, bool causal, hipStream_t st) { TATTN_F32_SWITCH(dq_launch, true) }
int launch_dkdv_f32(const BwdParams& p, int D, bool causal, hipStream_t st) { TATTN_F32_SWITCH(dkdv_launch, true) }

}  // namespace tattn
