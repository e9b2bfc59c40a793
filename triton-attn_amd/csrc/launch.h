// Host-side helpers shared by the kernel translation units: error reporting and launchers.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <utility>

#include "common.h"
#include "tiles.h"

#define TATTN_OK 0
#define TATTN_E_ARG 1
#define TATTN_E_CONFIG 2
#define TATTN_E_LAUNCH 3
#define TATTN_E_DEVICE 4

namespace tattn {

// Records a printf-style message as this thread's last error and returns `code`.
int set_error(int code, const char* fmt, ...) __attribute__((format(printf, 2, 3)));
// Returns TATTN_OK, or TATTN_E_LAUNCH with the HIP error text if the last launch failed.
int check_launch(const char* what);

int launch_fwd(const FwdParams& p, int D, int dtype, bool causal, int config_id, hipStream_t st);
int launch_bwd_preprocess(const BwdParams& p, int D, int dtype, hipStream_t st);
int launch_bwd_dkdv(const BwdParams& p, int D, int dtype, bool causal, int config_id, hipStream_t st);
int launch_bwd_dq(const BwdParams& p, int D, int dtype, bool causal, int config_id, hipStream_t st);

int fwd_lds_bytes(int D, int dtype, const TileEntry& e);

// Kernels that get their own translation unit, compiled with the instruction scheduler that
// measured fastest for them (tattn/_build.py: SOURCE_FLAGS); dtype 0 = fp16, 2 = bf16.
// Persistent causal forward with two query tiles per wave (fwd_persist_causal.hip): runs entry
// `config_id` of the forward table; returns 1 (nothing launched) when the problem does not fit
// the kernel, else 0 with *rc the launch status.
int launch_fwd_persist_causal2(const FwdParams& p, int D, int dtype, int config_id, hipStream_t st, int* rc);
// Persistent dQ (bwd_dq_persist.hip): runs entry `config_id` of the dQ table; the caller has
// checked bwd_persist_fits and bwd_fits32.
int launch_dq_persist(const BwdParams& p, int D, int dtype, int config_id, bool causal, hipStream_t st);
// Persistent dK/dV (bwd_dkdv_persist.hip): runs entry `config_id` of the dK/dV table; the caller
// has checked bwd_persist_fits and bwd_fits32.
int launch_dkdv_persist(const BwdParams& p, int D, int dtype, int config_id, bool causal, hipStream_t st);
// Paired-wave backward (bwd_split.hip): dK/dV (dkdv = true) or dQ with 128 rows per workgroup,
// p.n_blocks set by the caller; the caller has checked bwd_fits32.
int launch_split(const BwdParams& p, int D, int dtype, bool dkdv, bool causal, hipStream_t st);

// Whether the backward's (z, h) slices fit 32-bit buffer offsets (plus two steps of look-ahead) and
// rows past the sequence end lie past the slice's last byte, so that range-checked loads give zeros for
// them (rows that overlap, such as a broadcast row of stride 0, do not: queries past the end would add
// to dK and dV). Every backward kernel but the generic ones needs both; those check row indices and take
// 64-bit addresses.
inline bool bwd_fits32(const BwdParams& p, int D) {
  return p.s[2] >= D && slice_bytes(p.N, p.s[2], D) + (uint64_t)p.s[2] * 128 < (1ull << 31);
}

// Short rows (short.hip): up to 128 rows of a slice in one workgroup's waves, the whole backward in
// one launch. The rules check that a problem is one (16-bit, N within the limit) and that its row
// offsets fit 32 bits.
constexpr int kShortRows = 128;
int launch_fwd_short(const FwdParams& p, int D, int dtype, bool causal, hipStream_t st);
int launch_bwd_short(const BwdParams& p, int D, int dtype, bool causal, hipStream_t st);
inline bool fwd_short_fits(const FwdParams& p, int dtype) {
  return dtype != 1 && p.N <= kShortRows && (p.sk[2] | p.sv[2]) * 256 < (1ll << 30);
}
inline bool bwd_short_fits(const BwdParams& p, int D, int dtype) {
  return dtype != 1 && p.N <= kShortRows && p.s[2] >= D && p.s[2] * 256 < (1ll << 30);
}

// Waves of a workgroup split the summed dimension (coop.hip); 16-bit, slices that fit 32-bit
// offsets, fewer than the 2^32 threads that a launch may have (eight per row, where the block kernels take two),
// and for the forward a scale other than 0 (it hides keys at a score whose scaled value is -inf).
int launch_fwd_coop(const FwdParams& p, int D, int dtype, bool causal, hipStream_t st);
int launch_dq_coop(const BwdParams& p, int D, int dtype, bool causal, hipStream_t st);
int launch_dkdv_coop(const BwdParams& p, int D, int dtype, bool causal, hipStream_t st);
inline bool coop_launches(int64_t Z, int64_t H, int64_t N) { return Z * H * ((N + 63) / 64) * 512 < (1ll << 32); }
inline bool fwd_coop_fits(const FwdParams& p, int D, int dtype) {
  return dtype != 1 && p.c != 0.0f && coop_launches(p.Z, p.H, p.N) &&
         slice_bytes(p.N, p.sk[2], D) + (uint64_t)p.sk[2] * 128 < (1ull << 31) &&
         slice_bytes(p.N, p.sv[2], D) + (uint64_t)p.sv[2] * 128 < (1ull << 31) && (p.sk[2] | p.sv[2]) < (1ll << 22);
}
inline bool bwd_coop_fits(const BwdParams& p, int D, int dtype) {
  return dtype != 1 && coop_launches(p.Z, p.H, p.N) && bwd_fits32(p, D) && p.s[2] < (1ll << 22);
}

// float32 on split operands (f32_split.hip): row offsets of a slice, with a step's look-ahead, fit 32
// bits, and rows past the end of a slice lie past its last element (rows that overlap do not). One to three
// keys stay with the block kernels: sums of so few products are no closer to float64 here (dV of 2 keys,
// causal, head dim 16: 5.4e-8 against 5.1e-8). So do, where they are the faster ones (us, forward / backward, split
// against block kernels):
//   head dim 128 up to 96 rows, where one wave per SIMD is all that fits (64 x 16 x 24: 41 / 159, 37 / 113; 64 x 8 x 64:
//   35 / 131, 37 / 119; 16 x 16 x 128 causal: 31 / 108, 40 / 122);
//   32 and 64 up to 32 rows with at most two slices per CU and up to 40 with one, where one wave stages and splits
//   what four share there (64: 47 x 26 8.5 / 22.3, 6.0 / 19.2; 520 x 32 10.0 / 25.7, 11.4 / 39.1; 256 x 40 9.3 / 33.8,
//   9.8 / 30.8; 260 x 40 10.6 / 33.8, 14.3 / 47.8; 32: 256 x 16 5.9 / 14.2, 4.8 / 12.7).
// Both
// directions have to go the same way, since M belongs to the bits of the forward's S: they do where K and V
// of the forward and the inputs of the backward pass or fail alike, and a caller that copies in between (api.py) asks
// for the block kernels by index where the forward ran them.
int launch_fwd_f32(const FwdParams& p, int D, bool causal, hipStream_t st);
int launch_dq_f32(const BwdParams& p, int D, bool causal, hipStream_t st);
int launch_dkdv_f32(const BwdParams& p, int D, bool causal, hipStream_t st);
inline bool f32_rows_fit(int64_t ZH, int64_t N, int64_t row_stride, int D) {
  const int64_t most = D == 128 ? 96 : D < 32 || ZH > 512 ? 3 : ZH > 256 ? 32 : 40;  // rows of the block kernels
  return N > most && row_stride >= D && row_stride < (1ll << 22) && (N + 256) * row_stride * 4 < (1ll << 31);
}
inline bool fwd_f32_fits(const FwdParams& p, int D) {
  const int64_t zh = (int64_t)p.Z * p.H;
  return f32_rows_fit(zh, p.N, p.sk[2], D) && f32_rows_fit(zh, p.N, p.sv[2], D);
}
inline bool bwd_f32_fits(const BwdParams& p, int D) { return f32_rows_fit((int64_t)p.Z * p.H, p.N, p.s[2], D); }

// Compute units of the current device (cached per device).
inline int device_cus() {
  static int cus[64] = {};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
  if (cus[dev] <= 0) {
    int n = 0;
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) n = 256;
    cus[dev] = n;
  }
  return cus[dev];
}

// Whether a persistent backward entry (kind 2) runs a problem itself; otherwise the launcher
// runs the pipelined kernel of the same waves. Z*H a multiple of 8, N a multiple of the block
// and of 128 (whole groups of four steps), causal: an even number of blocks per slice (pairs).
inline bool bwd_persist_fits(const TileEntry& e, int64_t ZH, int64_t N, bool causal) {
  const int64_t blk = (int64_t)e.nw * 32;
  if (e.pipe != 2 || ZH % 8 != 0 || N % blk != 0 || N % 128 != 0) return false;
  return !causal || (N / blk) % 2 == 0;
}

// Whether a persistent forward entry (kind 2) runs a problem itself; otherwise the launcher runs
// the pipelined kernel of the same tiles. Z*H a multiple of 8 (whole slices per XCD), N a
// multiple of the block and of the ring period (whole unrolled groups), causal: an even number
// of blocks per slice (pairs), a diagonal region of one or two ring periods, and one 32-row tile
// per wave or a ring of 4 (the causal kernel with two tiles per wave and a ring of 8 does not fit
// the 256 registers a wave has at two waves per SIMD; those entries run their pipelined twin for
// causal problems).
constexpr bool fwd_persist_causal_ok(const TileEntry& e) {
  return (e.tiles == 1 || e.ring == 4) && (e.nw * e.tiles) % e.ring == 0 && e.nw * e.tiles / e.ring <= 2;
}
inline bool fwd_persist_fits(const TileEntry& e, int64_t ZH, int64_t N, bool causal) {
  const int64_t bm = (int64_t)e.nw * e.tiles * 32;
  if (e.pipe != 2 || ZH % 8 != 0 || N % bm != 0 || N % (32 * e.ring) != 0) return false;
  return !causal || ((N / bm) % 2 == 0 && fwd_persist_causal_ok(e));
}
int dkdv_lds_bytes(int D, int dtype, const TileEntry& e);
int dq_lds_bytes(int D, int dtype, const TileEntry& e);

}  // namespace tattn
