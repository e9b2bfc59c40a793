// C ABI of libtattn_hip.so (declared in include/tattn.h): argument checks, error strings,
// device check, tile-table introspection and the entry points that enqueue the kernels.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdarg>
#include <cstdio>
#include <cstring>
#include <mutex>

#include "../../include/tattn.h"
#include "launch.h"
#include "tiles.h"

namespace tattn {

static thread_local char g_err[512] = "";

int set_error(int code, const char* fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_err, sizeof(g_err), fmt, ap);
  va_end(ap);
  return code;
}

int check_launch(const char* what) {
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return set_error(TATTN_E_LAUNCH, "%s: launch failed: %s", what, hipGetErrorString(e));
  return TATTN_OK;
}

namespace {

constexpr int kMaxDevices = 64;
std::once_flag g_dev_once[kMaxDevices];
int g_dev_ok[kMaxDevices];

int device_check() {
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return set_error(TATTN_E_DEVICE, "hipGetDevice failed: %s", hipGetErrorString(e));
  if (dev < 0 || dev >= kMaxDevices) return set_error(TATTN_E_DEVICE, "device index %d out of range", dev);
  std::call_once(g_dev_once[dev], [dev] {
    hipDeviceProp_t prop;
    g_dev_ok[dev] = hipGetDeviceProperties(&prop, dev) == hipSuccess &&
                            strncmp(prop.gcnArchName, "gfx950", 6) == 0
                        ? 1
                        : 0;
  });
  if (!g_dev_ok[dev]) return set_error(TATTN_E_DEVICE, "device %d is not a gfx950 (MI355X)", dev);
  return TATTN_OK;
}

template <template <typename, int> class Table, typename T>
int table_size(int64_t D) {
  switch (D) {
    case 16: return Table<T, 16>::n;
    case 32: return Table<T, 32>::n;
    case 64: return Table<T, 64>::n;
    case 128: return Table<T, 128>::n;
  }
  return -1;
}

template <template <typename, int> class Table, typename T>
const TileEntry* table_entry(int64_t D, int id) {
  const TileEntry* e = nullptr;
  int n = 0;
  switch (D) {
    case 16: e = Table<T, 16>::e; n = Table<T, 16>::n; break;
    case 32: e = Table<T, 32>::e; n = Table<T, 32>::n; break;
    case 64: e = Table<T, 64>::e; n = Table<T, 64>::n; break;
    case 128: e = Table<T, 128>::e; n = Table<T, 128>::n; break;
    default: return nullptr;
  }
  return id >= 0 && id < n ? e + id : nullptr;
}

// fp16 and bf16 share the 16-bit tables (tiles.h).
int num_configs(int kernel, int64_t D, int dtype) {
  const bool h = dtype != TATTN_F32;
  switch (kernel) {
    case TATTN_K_FWD: return h ? table_size<FwdTable, _Float16>(D) : table_size<FwdTable, float>(D);
    case TATTN_K_BWD_DKDV: return h ? table_size<DkdvTable, _Float16>(D) : table_size<DkdvTable, float>(D);
    case TATTN_K_BWD_DQ: return h ? table_size<DqTable, _Float16>(D) : table_size<DqTable, float>(D);
  }
  return -1;
}

const TileEntry* config_entry(int kernel, int64_t D, int dtype, int id) {
  const bool h = dtype != TATTN_F32;
  switch (kernel) {
    case TATTN_K_FWD: return h ? table_entry<FwdTable, _Float16>(D, id) : table_entry<FwdTable, float>(D, id);
    case TATTN_K_BWD_DKDV:
      return h ? table_entry<DkdvTable, _Float16>(D, id) : table_entry<DkdvTable, float>(D, id);
    case TATTN_K_BWD_DQ: return h ? table_entry<DqTable, _Float16>(D, id) : table_entry<DqTable, float>(D, id);
  }
  return nullptr;
}

// What a launch costs in rows of one CU: workgroups of `rows` rows are dealt to the 256 CUs, and the
// CU with the most of them sets the time. `eff`: measured time per row where CUs hold several workgroups;
// `alone`: what a single workgroup on a CU loses (or gains, above 128 rows) on top. Without a mask all
// workgroups of a launch are equal, and this ranks the kernels: the constants below were fitted to the times of
// every entry at 871 shapes at head dim 64, 769 at 128, 451 at 32 and 417 at 16 (fp16, N = 129 to 12,000, up to 300,000
// rows). There the pick is on average 0.5 to 2% behind the fastest entry. Of 3,592 launches at other shapes 1.2% were
// more than 3% slower than the picks by length alone that these replace, two more than 10%; on average those took 1.26
// times as long. (Causal, with the tile counts below: 4,797 launches, 0.2%, none, 1.38.)
double cu_rows(int64_t ZH, int64_t N, int rows, double eff, double alone = 1.0) {
  const int64_t k = (ZH * ((N + rows - 1) / rows) + 255) / 256;
  return (double)(k * rows) * eff * (k == 1 ? alone : 1.0);
}

// The same for coop.hip's kernels (64 rows), whose prologue and final merge weigh on short rows as `head`
// more rows would.
double coop_rows(int64_t ZH, int64_t N, double eff, double head, double alone = 1.0) {
  return cu_rows(ZH, N, 64, eff * (1.0 + head / (double)N), alone);
}

// Those kernels read K and V (Q and dO) once per 64 rows, the others once per 128 or 256. Where ZH is not a
// multiple of 8 a slice is read by every XCD, and once the slices outgrow the L2s that costs them half their time or
// more (head dim 128, us, coop against paired waves / pipelined: dQ 37 x 4,505 822 / 664, causal 113 x 1,556 189 / 154;
// forward 21 x 2,038 79 / 66; head dim 64 causal forward, 53 x 1,235: 31.7 / 26.0): not picked there above this many bytes of K and V.
bool coop_in_reach(int64_t ZH, int64_t N, int64_t D, bool causal) {
  return ZH % 8 == 0 || ZH * N * D * 4 <= ((causal ? 12 : 24) << 20);
}

// The cheapest of a few candidates; the first wins ties.
struct Cheapest {
  double cost = 1e300;
  int id = -1;
  void offer(int i, double c) {
    if (c < cost) cost = c, id = i;
  }
};

// Kernels outside the tables: waves that split the summed dimension (coop.hip), float32 on split operands
// (f32_split.hip), short rows (short.hip).
constexpr int kCoop = TATTN_PICK_COOP, kSplit = TATTN_PICK_PLANES, kShort = TATTN_PICK_SHORT;

// Table pick for a problem (index into the kernel's table, or kCoop / kSplit where `own` says that
// the problem meets the preconditions of coop.hip in 16 bits, of f32_split.hip in float32), keyed
// like the reference's autotuner on (sequence length, head dim, causal) (src/tattn/kernels.py:57-61)
// and on ZH = Z * H, but static: measured on an MI355X. Entry 0 of each table is its
// general-purpose tile. Persistent entries are picked where they run the problem themselves.
//
// Causal launches are bound by their longest workgroups when the chip is not full: coop (a quarter
// of the chain) up to a number of 32-row tiles, fewer on short rows, where the chain is short as well.
// Measured per kernel and head dim (us, coop against the entry picked otherwise, N = 129 to 12,345):
//   forward   64: 2,256 tiles 27.7 / 28.3, 6,000 134 / 126, 1,784 (N = 256) 15.3 / 13.0, 2,128 (512) 23.8 / 19.9
//             128: 1,776 32.9 / 33.4, 2,256 46 / 42   32: 6,000 82 / 83, 6,204 46 / 43
//   dQ        64: 1,024 23 / 30, 1,760 95 / 118, 1,776 (1,177) 31 / 26   128: 6,000 299 / 323, 6,204 170 / 167
//             32: every size (8,192 tiles 51 / 53) from N = 768   16: 5,632 (1,024) 28.1 / 25.9, 3,072 (768) 14.4 / 12.6
//   dK/dV     64: 1,024 31 / 45, 1,760 128 / 149, 1,776 (1,177) 45 / 31   32: 4,632 299 / 314, 6,204 71 / 66, N = 384: 3,648 22 / 15
//             16: 3,408 (2,242) 45.8 / 41.2, 4,128 (4,104) 87.7 / 77.6   128: never (its registers spill there)
int pick_config(int kernel, int64_t D, int dtype, int causal, int64_t N, int64_t ZH, bool own) {
  if (dtype == TATTN_F32) return own ? kSplit : 0;  // fp16 and bf16 share the picks
  bool coop = own && coop_in_reach(ZH, N, D, causal != 0);
  const int64_t tiles = ZH * ((N + 31) / 32);
  Cheapest best;
  switch (kernel) {
    case TATTN_K_FWD: {
      // Fewer than 96 tiles stay with the block kernels, at a price (21 us where this kernel takes 9, 1 x 1,024 x
      // 64): there the softmax stress test holds gradients of near one-hot rows (2 x 1,024) to a flat allowance, which is
      // a matter of single roundings and not of accuracy. Both kernels exceed it by chance on more such rows (8 x 1,024:
      // block by 2.0e-3, this by 7.0e-3; 16 x 500: block by 1.4e-2, this by 1.6e-3), both keep to the allowance per element,
      // and O and M here are as close to float64 (peaked, fp16: O 1.01e-4, M 1.1e-7 against 1.02e-4, 1.8e-7).
      coop = coop && tiles >= 96;
      const int64_t coop_most = D == 64 ? std::min<int64_t>(2304, N * 2) : D == 128 ? 1800 : 6144;
      if (causal && coop && tiles <= coop_most) return kCoop;
      if (causal) {
        if (D == 64) {
          // Persistent, ring of 4: 4 x 2 from N = 2048 (from 4096 one pair of blocks per workgroup,
          // time-sliced priority), 4 x 1 below (cold-cache medians, 16,384 tokens x 16 heads: N =
          // 2048 4 x 2 3% faster since both store O as whole rows, N = 1024 4 x 1 2% faster).
          const int pid = N < 2048 ? 5 : 7;
          if (fwd_persist_fits(FwdTable<_Float16, 64>::e[pid], ZH, N, true)) return pid;
        }
        if (D == 128) {
          const int pid = N >= 4096 ? 3 : 2;  // persistent 8 x 1 / 4 x 1; else 4 x 1 pipelined
          return fwd_persist_fits(FwdTable<_Float16, 128>::e[pid], ZH, N, true) ? pid : 0;
        }
        // 128-row blocks; 256-row ones for long rows on a full chip.
        return N >= 4096 && tiles >= 8192 ? 0 : 1;
      }
      if (D == 64) {
        // Persistent 4 x 2 and 4 x 1 (ring of 4), pipelined 4 x 2, 8 x 2 from N = 4096, 4 x 1.
        if (fwd_persist_fits(FwdTable<_Float16, 64>::e[7], ZH, N, false)) best.offer(7, cu_rows(ZH, N, 256, 0.86, 1.21));
        if (fwd_persist_fits(FwdTable<_Float16, 64>::e[5], ZH, N, false)) best.offer(5, cu_rows(ZH, N, 128, 0.99, 1.47));
        best.offer(0, cu_rows(ZH, N, 256, 1.0, 1.13));
        if (N >= 4096) best.offer(3, cu_rows(ZH, N, 512, 0.99));
        best.offer(1, cu_rows(ZH, N, 128, 1.02, 1.39));
        if (coop) best.offer(kCoop, coop_rows(ZH, N, 1.29, 128, 1.2));
      } else if (D == 128) {
        // Persistent 8 x 1 from N = 2048, 4 x 1; pipelined 4 x 1.
        if (N >= 2048 && fwd_persist_fits(FwdTable<_Float16, 128>::e[3], ZH, N, false))
          best.offer(3, cu_rows(ZH, N, 256, 0.72));
        if (fwd_persist_fits(FwdTable<_Float16, 128>::e[2], ZH, N, false)) best.offer(2, cu_rows(ZH, N, 128, 1.0, 1.1));
        best.offer(0, cu_rows(ZH, N, 128, 1.04, 1.05));
        if (coop) best.offer(kCoop, coop_rows(ZH, N, 1.4, 64));
      } else if (D == 32) {
        best.offer(0, cu_rows(ZH, N, 256, 0.98, 1.06));
        best.offer(1, cu_rows(ZH, N, 128, 1.01, 1.41));
        if (coop) best.offer(kCoop, coop_rows(ZH, N, 1.1, 96));
      } else {
        best.offer(0, cu_rows(ZH, N, 256, 1.06, 1.19));
        best.offer(1, cu_rows(ZH, N, 128, 1.14, 1.37));
        if (coop) best.offer(kCoop, coop_rows(ZH, N, 1.11, 128));
      }
      return best.id;
    }
    case TATTN_K_BWD_DKDV: {
      const int64_t coop_most = D == 64 ? std::min<int64_t>(1800, N * 3 / 4) : D == 128 ? 0
                              : std::min<int64_t>(D == 16 ? 3000 : 4800, N * 8 / 5);
      if (causal && coop && tiles <= coop_most) return kCoop;
      // Paired waves at head dim 128: two per SIMD, where one wave per tile needs all 512 registers.
      if (D == 128) return 2;
      if (causal) {
        // Head dim 64: persistent 4 waves below N = 4096 where it fits, else pipelined, 8 waves (256
        // keys) from N = 2048, 4 below; picked on the whole forward + backward (non-causal, the
        // persistent entries lose there: the dQ pass leaves this kernel's inputs in the caches).
        if (D != 64) return 0;
        if (N < 4096 && bwd_persist_fits(DkdvTable<_Float16, 64>::e[5], ZH, N, true)) return 5;
        return N >= 2048 ? 1 : 0;
      }
      if (D == 64) {
        best.offer(1, cu_rows(ZH, N, 256, 0.93, 0.91));
        best.offer(0, cu_rows(ZH, N, 128, 1.38, 1.2));  // streams Q and dO past twice as many blocks
        if (coop) best.offer(kCoop, coop_rows(ZH, N, 1.4, 180, 1.21));
      } else if (D == 32) {
        best.offer(0, cu_rows(ZH, N, 128, 1.11, 1.58));
        if (coop) best.offer(kCoop, coop_rows(ZH, N, 1.15, 180));
      } else {
        best.offer(0, cu_rows(ZH, N, 128, 1.05, 1.83));
        if (coop) best.offer(kCoop, coop_rows(ZH, N, 1.1, 128));
      }
      return best.id;
    }
    case TATTN_K_BWD_DQ: {
      if (causal && D < 64) {
        // Coop, except many short rows (32: 16 x 16 x 384 13.6 against 12.7 us) and, at 16, full chips.
        if (D == 16) return coop && tiles <= std::min<int64_t>(5000, N * 3) ? kCoop : 0;
        return coop && (N >= 768 || tiles <= N * 8 / 5) ? kCoop : 0;
      }
      const int64_t coop_most = D == 64 ? std::min<int64_t>(1700, N * 6 / 5) : std::min<int64_t>(6000, N * 8);
      if (causal && coop && tiles <= coop_most) return kCoop;
      if (D == 128) {  // paired waves, as dK/dV
        if (causal) return 2;
        best.offer(2, cu_rows(ZH, N, 128, 1.07, 0.96));
        if (coop) best.offer(kCoop, coop_rows(ZH, N, 0.95, 64));
        return best.id;
      }
      if (D < 64) {
        best.offer(0, D == 32 ? cu_rows(ZH, N, 128, 1.03, 1.33) : cu_rows(ZH, N, 128, 1.02, 2.08));
        if (coop) best.offer(kCoop, D == 32 ? coop_rows(ZH, N, 0.82, 128) : coop_rows(ZH, N, 0.93, 180));
        return best.id;
      }
      // Persistent 4 waves where it fits; pipelined 4 or 8 waves.
      const bool persist = bwd_persist_fits(DqTable<_Float16, 64>::e[5], ZH, N, causal != 0);
      if (causal) return persist ? 5 : 0;
      if (persist) best.offer(5, cu_rows(ZH, N, 128, 0.92, 1.2));
      best.offer(0, cu_rows(ZH, N, 128, 1.02, 1.35));
      best.offer(1, cu_rows(ZH, N, 256, 1.06, 0.87));
      if (coop) best.offer(kCoop, coop_rows(ZH, N, 1.16, 180, 0.92));
      return best.id;
    }
  }
  return 0;
}

// Workspace of tattn_bwd_noalloc: the backward's delta (float32, one value per query row) in a
// fixed device array, so that entry point needs neither an allocation nor a caller-provided
// buffer. Every GPU holds its own copy (16 MiB) until the process ends. Host code must never
// pass `scratch` itself to a kernel or copy: that name is a host-side stand-in, not a device
// address. The device address is looked up once per device with hipGetSymbolAddress (with that
// device current) and kept in g_scratch_ptr.
constexpr int64_t kScratchRows = int64_t(1) << 22;  // Z * H * N <= 4,194,304
static __device__ __align__(256) float scratch[kScratchRows];

std::once_flag g_scratch_once[kMaxDevices];
float* g_scratch_ptr[kMaxDevices];
hipError_t g_scratch_err[kMaxDevices];

// Device address of this device's scratch array (the current device; device_check has run).
int scratch_for_current_device(float** out) {
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return set_error(TATTN_E_DEVICE, "hipGetDevice failed: %s", hipGetErrorString(e));
  std::call_once(g_scratch_once[dev], [dev] {
    void* ptr = nullptr;
    g_scratch_err[dev] = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    g_scratch_ptr[dev] = g_scratch_err[dev] == hipSuccess ? static_cast<float*>(ptr) : nullptr;
  });
  if (g_scratch_err[dev] != hipSuccess || !g_scratch_ptr[dev])
    return set_error(TATTN_E_DEVICE, "hipGetSymbolAddress(scratch) failed on device %d: %s", dev,
                     hipGetErrorString(g_scratch_err[dev]));
  *out = g_scratch_ptr[dev];
  return TATTN_OK;
}

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

int check_tensor(const char* name, const void* ptr, const int64_t* st, int sz) {
  if (!ptr) return set_error(TATTN_E_ARG, "%s is a null pointer", name);
  if (!st) return set_error(TATTN_E_ARG, "%s strides are null", name);
  if (st[3] != 1) return set_error(TATTN_E_ARG, "%s: d stride must be 1, got %lld", name, (long long)st[3]);
  const int64_t vec = 16 / sz;
  for (int i = 0; i < 3; ++i)
    if (st[i] < 0 || st[i] % vec != 0)
      return set_error(TATTN_E_ARG, "%s: stride %d (%lld) must be a non-negative multiple of %lld elements",
                       name, i, (long long)st[i], (long long)vec);
  if (!aligned16(ptr)) return set_error(TATTN_E_ARG, "%s must be 16-byte aligned", name);
  return TATTN_OK;
}

int check_shape(int64_t Z, int64_t H, int64_t N, int64_t D, int dtype) {
  if (dtype != TATTN_F16 && dtype != TATTN_F32 && dtype != TATTN_BF16)
    return set_error(TATTN_E_ARG, "dtype must be TATTN_F16, TATTN_BF16 or TATTN_F32, got %d", dtype);
  if (D != 16 && D != 32 && D != 64 && D != 128)
    return set_error(TATTN_E_ARG, "head dim must be 16, 32, 64 or 128, got %lld", (long long)D);
  if (Z < 1 || H < 1 || N < 1) return set_error(TATTN_E_ARG, "Z, H, N must be positive (%lld, %lld, %lld)",
                                                (long long)Z, (long long)H, (long long)N);
  if (N > (1 << 30) || Z * H > (1 << 30)) return set_error(TATTN_E_ARG, "problem too large");
  return TATTN_OK;
}

int run_fwd(const FwdParams& p, int D, int dtype, bool causal, int id, hipStream_t st) {
  if (id == kShort) return launch_fwd_short(p, D, dtype, causal, st);
  if (id == kSplit) return launch_fwd_f32(p, D, causal, st);
  return id == kCoop ? launch_fwd_coop(p, D, dtype, causal, st) : launch_fwd(p, D, dtype, causal, id, st);
}
int run_dq(const BwdParams& p, int D, int dtype, bool causal, int id, hipStream_t st) {
  if (id == kSplit) return launch_dq_f32(p, D, causal, st);
  return id == kCoop ? launch_dq_coop(p, D, dtype, causal, st) : launch_bwd_dq(p, D, dtype, causal, id, st);
}
int run_dkdv(const BwdParams& p, int D, int dtype, bool causal, int id, hipStream_t st) {
  if (id == kSplit) return launch_dkdv_f32(p, D, causal, st);
  return id == kCoop ? launch_dkdv_coop(p, D, dtype, causal, st) : launch_bwd_dkdv(p, D, dtype, causal, id, st);
}

bool fwd_own_fits(const FwdParams& p, int D, int dtype) { return dtype == TATTN_F32 ? fwd_f32_fits(p, D) : fwd_coop_fits(p, D, dtype); }
bool bwd_own_fits(const BwdParams& p, int D, int dtype) { return dtype == TATTN_F32 ? bwd_f32_fits(p, D) : bwd_coop_fits(p, D, dtype); }

// What the library picks: the forward, and one kernel of the backward. The whole backward of short rows is
// one launch (the callers that run both kernels look at bwd_short_fits first), with the bits of the pipelined
// kernels: called one by one, dK/dV and dQ run those there, so that both ways give the same gradients.
int pick_fwd(const FwdParams& p, int D, int dtype, int causal) {
  if (fwd_short_fits(p, dtype)) return kShort;
  return pick_config(TATTN_K_FWD, D, dtype, causal, p.N, (int64_t)p.Z * p.H, fwd_own_fits(p, D, dtype));
}
int pick_bwd(int kernel, const BwdParams& p, int D, int dtype, int causal) {
  const bool own = bwd_own_fits(p, D, dtype) && !bwd_short_fits(p, D, dtype);
  return pick_config(kernel, D, dtype, causal, p.N, (int64_t)p.Z * p.H, own);
}

// Whether a caller's table index exists.
int check_config(int kernel, int64_t D, int dtype, int id) {
  const int n = num_configs(kernel, D, dtype);
  return id < n ? TATTN_OK : set_error(TATTN_E_CONFIG, "config id %d out of range [0, %d)", id, n);
}

}  // namespace
}  // namespace tattn

using namespace tattn;

extern "C" {

int tattn_abi_version(void) { return TATTN_ABI_VERSION; }

const char* tattn_last_error(void) { return g_err; }

int tattn_device_supported(void) { return device_check() == TATTN_OK ? 1 : 0; }

int tattn_num_configs(int kernel, int64_t D, int dtype) { return num_configs(kernel, D, dtype); }

int tattn_config_desc(int kernel, int64_t D, int dtype, int config_id, tattn_config* out) {
  if (!out) return set_error(TATTN_E_ARG, "out is a null pointer");
  const TileEntry* e = config_entry(kernel, D, dtype, config_id);
  if (!e) return set_error(TATTN_E_CONFIG, "no config %d for kernel %d, D=%lld, dtype %d", config_id, kernel,
                           (long long)D, dtype);
  const int rows = tile_rows(*e);
  out->waves = e->nw;
  out->tiles = e->tiles;
  out->kind = e->pipe;
  out->ring = e->pipe == 2 ? e->ring : 0;
  if (kernel == TATTN_K_BWD_DKDV) {
    out->block_n = rows;
    out->block_m = e->other;
    out->lds_bytes = dkdv_lds_bytes((int)D, dtype, *e);
  } else {
    out->block_m = rows;
    out->block_n = e->other;
    out->lds_bytes = kernel == TATTN_K_FWD ? fwd_lds_bytes((int)D, dtype, *e) : dq_lds_bytes((int)D, dtype, *e);
  }
  return TATTN_OK;
}

int tattn_pick_config(int kernel, int64_t D, int dtype, int causal, int64_t N) {
  if (num_configs(kernel, D, dtype) < 0) return set_error(TATTN_E_ARG, "no table for kernel %d, D=%lld", kernel, (long long)D), -1;
  return pick_config(kernel, D, dtype, causal, N, 1 << 16, false);  // a full chip, Z * H a multiple of 8
}

int tattn_picked(int kernel, const int64_t k_strides[4], const int64_t v_strides[4], int64_t Z, int64_t H, int64_t N,
                 int64_t D, int dtype, int causal, float sm_scale) {
  if (check_shape(Z, H, N, D, dtype)) return -1;
  const int64_t whole[4] = {H * N * D, N * D, D, 1};
  if (!k_strides) k_strides = whole;
  if (!v_strides) v_strides = k_strides;
  if (kernel == TATTN_K_FWD) {
    FwdParams p{};
    for (int i = 0; i < 3; ++i) p.sk[i] = k_strides[i], p.sv[i] = v_strides[i];
    p.Z = (int32_t)Z; p.H = (int32_t)H; p.N = (int32_t)N;
    p.c = sm_scale * kLog2e;
    return pick_fwd(p, (int)D, dtype, causal);
  }
  if (kernel != TATTN_K_BWD_DKDV && kernel != TATTN_K_BWD_DQ) return set_error(TATTN_E_ARG, "no kernel %d", kernel), -1;
  BwdParams p{};
  for (int i = 0; i < 3; ++i) p.s[i] = k_strides[i];
  p.Z = (int32_t)Z; p.H = (int32_t)H; p.N = (int32_t)N;
  return bwd_short_fits(p, (int)D, dtype) ? kShort : pick_bwd(kernel, p, (int)D, dtype, causal);
}

int tattn_fwd(const void* q, const void* k, const void* v, void* o, float* m, const int64_t q_strides[4],
              const int64_t k_strides[4], const int64_t v_strides[4], const int64_t o_strides[4], int64_t Z,
              int64_t H, int64_t N, int64_t D, int dtype, int causal, float sm_scale, int config_id,
              void* stream) {
  int rc;
  if ((rc = check_shape(Z, H, N, D, dtype))) return rc;
  const int sz = dtype == TATTN_F32 ? 4 : 2;
  if ((rc = check_tensor("q", q, q_strides, sz)) || (rc = check_tensor("k", k, k_strides, sz)) ||
      (rc = check_tensor("v", v, v_strides, sz)) || (rc = check_tensor("o", o, o_strides, sz)))
    return rc;
  // m may be null: the log-sum-exp is then not stored (no backward will follow).
  FwdParams p{};
  p.q = q; p.k = k; p.v = v; p.o = o; p.m = m;
  for (int i = 0; i < 3; ++i) {
    p.sq[i] = q_strides[i]; p.sk[i] = k_strides[i]; p.sv[i] = v_strides[i]; p.so[i] = o_strides[i];
  }
  p.Z = (int32_t)Z; p.H = (int32_t)H; p.N = (int32_t)N;
  p.c = sm_scale * kLog2e;
  if ((rc = check_config(TATTN_K_FWD, D, dtype, config_id)) || (rc = device_check())) return rc;
  const int id = config_id < 0 ? pick_fwd(p, (int)D, dtype, causal) : config_id;
  return run_fwd(p, (int)D, dtype, causal != 0, id, (hipStream_t)stream);
}

static int bwd_common(BwdParams& p, const int64_t strides[4], int64_t Z, int64_t H, int64_t N, int64_t D,
                      int dtype, float sm_scale) {
  int rc;
  if ((rc = check_shape(Z, H, N, D, dtype))) return rc;
  if (!strides) return set_error(TATTN_E_ARG, "strides are null");
  for (int i = 0; i < 3; ++i) p.s[i] = p.so[i] = strides[i];
  p.Z = (int32_t)Z; p.H = (int32_t)H; p.N = (int32_t)N;
  p.c = sm_scale * kLog2e;
  p.scale = sm_scale;
  return TATTN_OK;
}

int tattn_bwd_preprocess(const void* o, const void* dout, float* delta, const int64_t strides[4], int64_t Z,
                         int64_t H, int64_t N, int64_t D, int dtype, void* stream) {
  BwdParams p{};
  int rc;
  if ((rc = bwd_common(p, strides, Z, H, N, D, dtype, 1.0f))) return rc;
  const int sz = dtype == TATTN_F32 ? 4 : 2;
  if ((rc = check_tensor("o", o, strides, sz)) || (rc = check_tensor("do", dout, strides, sz))) return rc;
  if (!delta) return set_error(TATTN_E_ARG, "delta is a null pointer");
  if ((rc = device_check())) return rc;
  p.o = o; p.dout = dout; p.delta = delta;
  return launch_bwd_preprocess(p, (int)D, dtype, (hipStream_t)stream);
}

int tattn_bwd_dkdv(const void* q, const void* k, const void* v, const void* dout, void* dk, void* dv,
                   const float* m, const float* delta, const int64_t strides[4], int64_t Z, int64_t H, int64_t N,
                   int64_t D, int dtype, int causal, float sm_scale, int config_id, void* stream) {
  BwdParams p{};
  int rc;
  if ((rc = bwd_common(p, strides, Z, H, N, D, dtype, sm_scale))) return rc;
  const int sz = dtype == TATTN_F32 ? 4 : 2;
  if ((rc = check_tensor("q", q, strides, sz)) || (rc = check_tensor("k", k, strides, sz)) ||
      (rc = check_tensor("v", v, strides, sz)) || (rc = check_tensor("do", dout, strides, sz)) ||
      (rc = check_tensor("dk", dk, strides, sz)) || (rc = check_tensor("dv", dv, strides, sz)))
    return rc;
  if (!m || !delta) return set_error(TATTN_E_ARG, "m and delta must not be null");
  if ((rc = check_config(TATTN_K_BWD_DKDV, D, dtype, config_id)) || (rc = device_check())) return rc;
  const int id = config_id < 0 ? pick_bwd(TATTN_K_BWD_DKDV, p, (int)D, dtype, causal) : config_id;
  p.q = q; p.k = k; p.v = v; p.dout = dout; p.dk = dk; p.dv = dv; p.m = m; p.delta = const_cast<float*>(delta);
  return run_dkdv(p, (int)D, dtype, causal != 0, id, (hipStream_t)stream);
}

// dQ; with o_fused (O, in the shared layout) the kernel computes delta = rowsum(dO * O) itself, in
// the preprocess's order, and stores it into `delta` for the dK/dV kernel that follows.
static int bwd_dq_call(const void* q, const void* k, const void* v, const void* dout, void* dq, const float* m,
                       const float* delta, const int64_t strides[4], int64_t Z, int64_t H, int64_t N, int64_t D,
                       int dtype, int causal, float sm_scale, int config_id, void* stream, const void* o_fused) {
  BwdParams p{};
  int rc;
  if ((rc = bwd_common(p, strides, Z, H, N, D, dtype, sm_scale))) return rc;
  const int sz = dtype == TATTN_F32 ? 4 : 2;
  if ((rc = check_tensor("q", q, strides, sz)) || (rc = check_tensor("k", k, strides, sz)) ||
      (rc = check_tensor("v", v, strides, sz)) || (rc = check_tensor("do", dout, strides, sz)) ||
      (rc = check_tensor("dq", dq, strides, sz)))
    return rc;
  if (!m || !delta) return set_error(TATTN_E_ARG, "m and delta must not be null");
  if ((rc = check_config(TATTN_K_BWD_DQ, D, dtype, config_id)) || (rc = device_check())) return rc;
  const int id = config_id < 0 ? pick_bwd(TATTN_K_BWD_DQ, p, (int)D, dtype, causal) : config_id;
  p.q = q; p.k = k; p.v = v; p.dout = dout; p.dq = dq; p.m = m; p.delta = const_cast<float*>(delta);
  if (o_fused) {
    p.o = o_fused;
    p.fuse_delta = 1;
  }
  return run_dq(p, (int)D, dtype, causal != 0, id, (hipStream_t)stream);
}

int tattn_bwd_dq(const void* q, const void* k, const void* v, const void* dout, void* dq, const float* m,
                 const float* delta, const int64_t strides[4], int64_t Z, int64_t H, int64_t N, int64_t D,
                 int dtype, int causal, float sm_scale, int config_id, void* stream) {
  return bwd_dq_call(q, k, v, dout, dq, m, delta, strides, Z, H, N, D, dtype, causal, sm_scale, config_id, stream,
                     nullptr);
}

// Checks every argument of the whole backward and resolves both kernels' table entries before
// anything is enqueued, so a nonzero return from tattn_bwd means no work was launched.
static int bwd_prepare(BwdParams& p, int* dk_id, int* dq_id, bool* fuse, const void* q, const void* k,
                       const void* v, const void* o, const void* dout, void* dq, void* dk, void* dv, const float* m,
                       float* delta, const int64_t strides[4], const int64_t grad_strides[4], int64_t Z,
                       int64_t H, int64_t N, int64_t D, int dtype, int causal, float sm_scale, int config_id) {
  int rc;
  if ((rc = bwd_common(p, strides, Z, H, N, D, dtype, sm_scale))) return rc;
  const int sz = dtype == TATTN_F32 ? 4 : 2;
  if ((rc = check_tensor("q", q, strides, sz)) || (rc = check_tensor("k", k, strides, sz)) ||
      (rc = check_tensor("v", v, strides, sz)) || (rc = check_tensor("o", o, strides, sz)) ||
      (rc = check_tensor("do", dout, strides, sz)) || (rc = check_tensor("dq", dq, grad_strides, sz)) ||
      (rc = check_tensor("dk", dk, grad_strides, sz)) || (rc = check_tensor("dv", dv, grad_strides, sz)))
    return rc;
  for (int i = 0; i < 3; ++i) p.so[i] = grad_strides[i];
  if (!m || !delta) return set_error(TATTN_E_ARG, "m and delta must not be null");
  if (config_id >= 0) {
    // One id for both kernels, as the reference's `config=` (api.py:124-145): it must exist in both tables.
    if (config_id >= num_configs(TATTN_K_BWD_DKDV, D, dtype) || config_id >= num_configs(TATTN_K_BWD_DQ, D, dtype))
      return set_error(TATTN_E_CONFIG, "config id %d out of range for the backward tables", config_id);
  }
  *dk_id = config_id < 0 ? pick_bwd(TATTN_K_BWD_DKDV, p, (int)D, dtype, causal) : config_id;
  *dq_id = config_id < 0 ? pick_bwd(TATTN_K_BWD_DQ, p, (int)D, dtype, causal) : config_id;
  if ((rc = device_check())) return rc;
  // When dQ runs any kernel but the generic ones it computes delta itself
  // (same bits as the preprocess) and stores it: dQ, then dK/dV, two launches and no separate
  // pass over dO. Otherwise preprocess, dK/dV, dQ.
  const TileEntry* e = config_entry(TATTN_K_BWD_DQ, D, dtype, *dq_id);
  *fuse = *dq_id == kCoop || *dq_id == kSplit || (dtype != TATTN_F32 && e && e->pipe >= 1 && bwd_fits32(p, (int)D));
  p.q = q; p.k = k; p.v = v; p.o = o; p.dout = dout; p.dq = dq; p.dk = dk; p.dv = dv; p.m = m; p.delta = delta;
  return TATTN_OK;
}

int tattn_bwd_layouts(const void* q, const void* k, const void* v, const void* o, const void* dout, void* dq,
                      void* dk, void* dv, const float* m, float* delta, const int64_t strides[4],
                      const int64_t grad_strides[4], int64_t Z, int64_t H, int64_t N, int64_t D, int dtype,
                      int causal, float sm_scale, int config_id, void* stream) {
  BwdParams p{};
  int rc, dk_id = -1, dq_id = -1;
  bool fuse = false;
  if ((rc = bwd_prepare(p, &dk_id, &dq_id, &fuse, q, k, v, o, dout, dq, dk, dv, m, delta, strides, grad_strides,
                        Z, H, N, D, dtype, causal, sm_scale, config_id)))
    return rc;
  const hipStream_t st = (hipStream_t)stream;
  if (config_id < 0 && bwd_short_fits(p, (int)D, dtype)) return launch_bwd_short(p, (int)D, dtype, causal != 0, st);
  if (fuse) {
    BwdParams pq = p;
    pq.fuse_delta = 1;
    if ((rc = run_dq(pq, (int)D, dtype, causal != 0, dq_id, st))) return rc;
    return run_dkdv(p, (int)D, dtype, causal != 0, dk_id, st);
  }
  if ((rc = launch_bwd_preprocess(p, (int)D, dtype, st))) return rc;
  if ((rc = run_dkdv(p, (int)D, dtype, causal != 0, dk_id, st))) return rc;
  return run_dq(p, (int)D, dtype, causal != 0, dq_id, st);
}

int tattn_bwd(const void* q, const void* k, const void* v, const void* o, const void* dout, void* dq, void* dk,
              void* dv, const float* m, float* delta, const int64_t strides[4], int64_t Z, int64_t H, int64_t N,
              int64_t D, int dtype, int causal, float sm_scale, int config_id, void* stream) {
  return tattn_bwd_layouts(q, k, v, o, dout, dq, dk, dv, m, delta, strides, strides, Z, H, N, D, dtype, causal,
                           sm_scale, config_id, stream);
}

int tattn_bwd_noalloc(const void* q, const void* k, const void* v, const void* o, const void* dout, void* dq,
                      void* dk, void* dv, const float* m, const int64_t strides[4], int64_t Z, int64_t H,
                      int64_t N, int64_t D, int dtype, int causal, float sm_scale, int config_id, void* stream) {
  int rc;
  if ((rc = check_shape(Z, H, N, D, dtype))) return rc;
  if (Z * H * N > kScratchRows)
    return set_error(TATTN_E_ARG,
                     "tattn_bwd_noalloc: Z*H*N = %lld query rows exceeds the static workspace of %lld rows; "
                     "use tattn_bwd with a caller-provided delta",
                     (long long)(Z * H * N), (long long)kScratchRows);
  if ((rc = device_check())) return rc;
  float* delta = nullptr;
  if ((rc = scratch_for_current_device(&delta))) return rc;
  // delta is written in full (by the preprocess, or by the kernel that computes it) before it is read.
  return tattn_bwd(q, k, v, o, dout, dq, dk, dv, m, delta, strides, Z, H, N, D, dtype, causal, sm_scale,
                   config_id, stream);
}

}  // extern "C"
