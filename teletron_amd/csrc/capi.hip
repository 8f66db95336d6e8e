// C ABI of the fused normalisation kernels: argument validation, launch planning
// (variant, grid, workspace) and the kernel launches.  See include/teletron_op.h.
#include "teletron_op.h"

#include <atomic>
#include <initializer_list>
#include <mutex>
#include <unordered_map>

#include "generic_kernels.hpp"
#include "kernel_table.hpp"
#include "probe_kernels.hpp"

namespace tt {
namespace {

thread_local int g_last_hip_error = 0;

int hip_fail(hipError_t e) {
  g_last_hip_error = static_cast<int>(e);
  (void)hipGetLastError();  // clear the sticky launch error, it has been recorded
  return TT_ERR_HIP;
}

struct DeviceInfo {
  int cus = 0;
};

int current_device_cus(int* cus) {
  static std::mutex mu;
  static DeviceInfo info[64];
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return hip_fail(e);
  if (dev < 0 || dev >= 64) return TT_ERR_INVALID_ARGUMENT;
  std::lock_guard<std::mutex> lock(mu);
  if (info[dev].cus == 0) {
    int n = 0;
    e = hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev);
    if (e != hipSuccess) return hip_fail(e);
    info[dev].cus = n > 0 ? n : 1;
  }
  *cus = info[dev].cus;
  return TT_OK;
}

// Resident workgroups per CU for a kernel, from the HIP occupancy calculator (cached).
int resident_wgs_per_cu(const KernelInfo& k, int* out) {
  static std::mutex mu;
  static std::unordered_map<const void*, int> cache;
  {
    std::lock_guard<std::mutex> lock(mu);
    auto it = cache.find(k.fn);
    if (it != cache.end()) { *out = it->second; return TT_OK; }
  }
  int n = 0;
  hipError_t e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, k.fn, k.threads, 0);
  if (e != hipSuccess) return hip_fail(e);
  if (n < 1) n = 1;
  std::lock_guard<std::mutex> lock(mu);
  cache[k.fn] = n;
  *out = n;
  return TT_OK;
}

// Backward workspace of tt_adaln_backward_static: a file-scope device array, so that the entry
// point never allocates.  Every device the library runs on holds its own copy at its own address;
// the host-side name below is only a handle for hipGetSymbolAddress, never a kernel argument.
// The entry point takes what the kernels of whole-line rows (or the element-wise ones) do within
// TT_STATIC_WORKSPACE_BYTES; those of ragged rows keep up to twice the workgroups resident.
constexpr size_t kScratchBytes = 2 * (size_t)TT_STATIC_WORKSPACE_BYTES;
static __device__ __align__(256) unsigned char scratch[kScratchBytes];

// Device address of `scratch` on the current device, looked up once per device.
int static_scratch(void** out) {
  static std::mutex mu;
  static void* addr[64];
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return hip_fail(e);
  if (dev < 0 || dev >= 64) return TT_ERR_INVALID_ARGUMENT;
  std::lock_guard<std::mutex> lock(mu);
  if (!addr[dev]) {
    void* p = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess) return hip_fail(e);
    if (!p) return TT_ERR_HIP;
    addr[dev] = p;
  }
  *out = addr[dev];
  return TT_OK;
}

std::atomic<int> g_wgs_per_cu_override{0};
std::atomic<int> g_grid_override{0};

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

struct Rope {
  const float* freqs = nullptr;
  int64_t head_dim = 0, seq_len = 0;
  int64_t heads = 0;   // 0: a row holds every head of a token; > 0: one head per row, `heads` rows per token
};

// How the parameters of a norm forward lie in memory, where not as dense bf16 (see FwdArgs).
struct Params {
  int64_t stride0, stride1;
  int f32;
  void* copy;
};

struct Plan {
  KernelInfo k;
  int64_t n_batches = 0;
  int64_t n_tiles = 0;   // per batch
  int grid_x = 0;        // most workgroups per batch: what workspaces are sized for
  int max_x = 0;         // workgroups per batch that are launched at most, 0: grid_x
  int packs = 0;
  // workgroups per batch that are launched == partial sums per batch
  int grid() const { return max_x && max_x < grid_x ? max_x : grid_x; }
};

enum Dir { kFwd, kBwd, kBwdSaved, kFwdXn };   // kFwdXn: AdaLN forward that also stores x_norm
constexpr int kGateKind = 2;   // third op family next to kAdaLN / kRMS

// Upper bound on workgroups per batch used by any plan: what the workspace is sized for.
constexpr int kMaxWgsPerCu = 8;

// `force`: kOdd for rows of any length and 2-byte aligned tensors (wide norm_fwd / norm_bwd kernels only),
// kMasked for the plan that ragged rows would have on the kernels of whole-line rows.
// `res`: 0, or the residual + LayerNorm fusion: 1 plain, 2 gated (wide rows, kFwd / kBwd only).
int make_plan(int kind, Dir dir, int64_t rows, int64_t cols, int64_t rows_per_batch, Plan* plan, bool rope = false,
              int res = 0, int64_t rope_heads = 0, int force = -1) {
  const bool odd = force == kOdd;
  if (rows <= 0 || cols <= 0 || rows_per_batch <= 0 || rows % rows_per_batch != 0)
    return TT_ERR_INVALID_ARGUMENT;
  if (cols > TT_MAX_COLS) return TT_ERR_UNSUPPORTED;
  if (cols % kPack != 0 && !odd) return TT_ERR_UNSUPPORTED;
  const int packs = static_cast<int>((cols + kPack - 1) / kPack);
  const bool narrow = packs <= kNarrowMaxPacks;
  if (odd && (narrow || res || rope || dir == kBwdSaved || kind == kGateKind)) return TT_ERR_UNSUPPORTED;
  const int idx = narrow ? select_narrow(packs) : select_wide(packs);
  if (idx < 0) return TT_ERR_UNSUPPORTED;
  const int slots = narrow ? kNarrowL[idx] : 64 * kWideW[idx] * kWideP[idx];
  const bool full = (slots == packs);
  const bool cache_resident = rows * cols * 2 < (int64_t)64 << 20;
  if (res && (narrow || kind != kAdaLN || dir == kBwdSaved || dir == kFwdXn)) return TT_ERR_UNSUPPORTED;
  if (rope && (kind != kRMS || dir == kBwdSaved || dir == kFwdXn)) return TT_ERR_UNSUPPORTED;
  if (dir == kFwdXn && kind != kAdaLN) return TT_ERR_UNSUPPORTED;
  // a row of whole 128-byte lines or not: see enum Rows
  int mode = odd ? kOdd : full ? kFull : (cols * 2) % 128 == 0 || force == kMasked ? kMasked : kRagged;
  int cus = 0, per_cu = 0;
  int rc = current_device_cus(&cus);
  if (rc != TT_OK) return rc;
  // beyond the caches one CU in 32 is left without a workgroup
  const int usable_cus = !cache_resident && cus >= 32 ? cus - cus / 32 : cus;
  const int64_t groups = rows / rows_per_batch;
  const bool uneven = !cache_resident && usable_cus / groups * groups * 20 < (int64_t)usable_cus * 19;
  if (mode == kRagged)
    mode |= (cache_resident ? kCached : uneven ? kUneven : 0) | (packs * 4 < slots * 3 ? kIdle : packs * 16 >= slots * 15 ? kDense : 0);
  if (rope) {
    // Token mode saves table look-ups, but its tiles are three times those of the look-up per row: on tensors
    // that the caches hold, its forward waits for one tile a CU, and with four loads a wave it is slower
    // throughout; its backward has fewer waves resident (237 registers against 138).  Kernel us per token | per row:
    //   forward  24 heads of 128,   1 MB 4.7 | 3.8    4: 4.8 | 4.0    12: 5.5 | 6.2    32: 12.3 | 13.8    63: 23.7 | 24.6
    //            12 of 128 (R = 3), 1: 4.0 | 3.6      4: 3.9 | 4.0    12: 6.1 | 6.2    32: 13.4 | 14.1    63: 25.4 | 25.2
    //            16 of 128 (R = 4), 1: 4.1 | 3.5      4: 4.2 | 4.1    12: 5.9 | 6.0    32: 14.2 | 13.9    63: 27.9 | 24.6
    //   backward 24 heads of 128,   1: 5.4 | 4.8      4: 5.7 | 5.4    12: 7.7 | 8.3    32: 19.4 | 17.5    63: 36.5 | 35.3
    //            16 of 128,         1: 5.5 | 4.7      4: 5.6 | 5.2    12: 9.7 | 8.3    32: 19.7 | 17.5    63: 35.7 | 35.6
    // (48 heads of 128 as 24; 64 columns as 128 with half the heads.  Beyond the caches: see rope_token_R.)
    if (narrow && rope_heads > 0 && cache_resident) {
      const int r = rope_token_R(kNarrowL[idx], rope_heads);
      if (dir == kBwd || r == 4 || rows < (int64_t)cus * rope_token_NW(r) * r * (kWave / kNarrowL[idx])) rope_heads = 0;
    }
  }
  const auto pick = [&](int rows_kind) -> KernelInfo {
    if (res == 2) return resnorm_gated_kernel(dir == kBwd, idx, rows_kind);
    if (res) return resnorm_plain_kernel(dir == kBwd, idx, rows_kind);
    if (rope) return rms_rope_kernel(narrow, dir == kBwd, idx, rows_kind, rope_heads);
    if (dir == kFwdXn) return adaln_fwd_xnorm_kernel(narrow, idx, rows_kind);
    if (kind == kAdaLN)
      return dir == kFwd ? adaln_fwd_kernel(narrow, idx, rows_kind)
           : dir == kBwd ? adaln_bwd_kernel(narrow, idx, rows_kind) : adaln_bwd_saved_kernel(narrow, idx, rows_kind);
    if (kind == kRMS)
      return dir == kFwd ? rms_fwd_kernel(narrow, idx, rows_kind)
           : dir == kBwd ? rms_bwd_kernel(narrow, idx, rows_kind) : rms_bwd_saved_kernel(narrow, idx, rows_kind);
    return dir == kFwd ? gate_fwd_kernel(narrow, idx, rows_kind) : gate_bwd_kernel(narrow, idx, rows_kind);
  };
  const KernelInfo k = pick(mode);
  if (!k.fn) return TT_ERR_UNSUPPORTED;

  rc = resident_wgs_per_cu(k, &per_cu);
  if (rc != TT_OK) return rc;
  // HBM streams fastest with a modest number of requests in flight: measured on MI355X,
  // throughput peaks near kFwdLoadsPerCu / kBwdLoadsPerCu outstanding 128-bit loads per lane
  // column of a CU (waves x loads per lane) and streamed tensor, falls off by 10-20 % at full
  // occupancy, and is a few percent better with one CU in 32 left without a workgroup.
  // Tensors that fit the caches take what fits a CU, or one workgroup (max_x below).
  if (!cache_resident) {
    const int per_wg = (k.threads / kWave) * k.lane_loads;
    // two streamed inputs (backward kernels, both gate kernels) or one (normalisation forward)
    const int target = dir == kFwdXn ? kFwdXnLoadsPerCu
                     : (dir == kFwd && kind != kGateKind && !res) ? kFwdLoadsPerCu : kBwdLoadsPerCu;
    int want = (2 * target + per_wg) / (2 * per_wg);
    if (want < 1) want = 1;
    if (want < per_cu) per_cu = want;
  }
  const int ov = g_wgs_per_cu_override.load(std::memory_order_relaxed);
  const int gov = g_grid_override.load(std::memory_order_relaxed);
  if (ov > 0) per_cu = ov;
  if (per_cu > kMaxWgsPerCu) per_cu = kMaxWgsPerCu;

  // The backward kernels of wide rows leave partial sums of 4 to 12 bytes a column and workgroup, which on tensors
  // that the caches hold cost more than a second workgroup on the CU gives: one a CU.  Kernel us, two -> one, backward +
  // reduction: saved AdaLN 1692 x 3072 14.3 + 4.4 -> 10.8 + 3.2, 9000 x 3072 32.7 + 4.8 -> 30.4 + 4.7, AdaLN 1200 x 5128
  // 18.1 + 6.7 -> 15.5 + 4.3, residual + norm 1300 x 3072 14.1 + 4.4 -> 11.0 + 3.9, gate 1222 x 3536 8.9 + 3.8 -> 8.2 + 3.1,
  // RMSNorm 3000 x 3072 15.3 + 3.8 -> 13.6 + 3.8, with the rotary embedding 5000 x 3072 23.7 + 3.9 -> 21.2 + 3.9.
  // Not where over a quarter of the lanes are idle: one workgroup then has too little in flight (RMSNorm 19660 x 640
  // 17.9 -> 19.7 with the reduction), nor for narrow rows, whose partial sums are small (40 heads of 128 x 3000 17 -> 22).
  // Nor, beyond 12 MiB, where over a sixteenth of them are, with one pack a lane and two tensors to read: RMSNorm
  // 1664 columns 15 / 20 / 60 MB 12.0 / 14.4 / 34.9 -> 13.6 / 15.9 / 37.2, 1544: 48 / 60 MB 30.1 / 35.5 -> 31.5 / 38.0, with the
  // rotary embedding 896: 20 / 60 MB 17.4 / 36.7 -> 18.4 / 39.1, saved AdaLN 392: 33 / 60 MB 24.9 / 41.7 -> 26.6 / 43.8, gate 1160:
  // 20 MB 14.3 -> 15.2 (up to 8 MB, or with every lane in use, one is the faster there too: RMSNorm 1544 11.4 -> 10.5, 1536 10.4 -> 9.9).
  // Nor where the batches divide the CUs so badly that over a third of them would go without a workgroup.  Backward +
  // reduction, as many as fit | whole workgroups a batch up to one a CU | rounded up to one a CU:
  //   140 x 60 x 3072 (140 of 256 CUs): residual + norm 46.3 + 18.2 | 52.4 + 17.8 | 62.1 + 18.2, gate 24.8 + 14.4 | 31.7 + 13.3 | 26.4 + 14.1
  //   86 x 90 x 3072 (172): residual + norm 40.5 + 13.3 | 41.6 + 12.0 | 58.4 + 12.5, gate 23.2 + 9.8 | 24.0 + 9.2 | 24.9 + 9.5, AdaLN
  //     86 x 34 x 2696 16.6 + 12.0 | 15.7 + 11.0
  //   100 x 50 x 3072 (200): residual + norm 28.5 + 14.9 | 29.5 + 13.3 | 36.4 + 13.4, gate 15.9 + 10.9 | 14.8 + 10.4 | 16.5 + 10.6
  //   43 x 45 x 3072 (215): residual + norm 15.0 + 9.2 | 13.3 + 7.2, gate 7.5 + 7.5 | 7.7 + 6.3
  // (Rounded up, a few CUs have two workgroups, and all the others wait for them.)
  // Workspaces stay sized for grid_x, so that sizes asked for once hold.
  const int64_t per_group = cus / groups;
  if (ov <= 0 && gov <= 0 && cache_resident && !narrow && (dir == kBwd || dir == kBwdSaved) && packs * 4 >= slots * 3 &&
      (res || kWideP[idx] > 1 || packs * 16 >= slots * 15 || rows * cols * 2 < (int64_t)12 << 20) &&
      per_group * groups * 3 >= (int64_t)cus * 2)
    plan->max_x = (int)per_group;

  // Tensors that fit the caches are read with ordinary loads (kKeep; the plan is that of the other kernel).  As fast
  // as streaming loads on inputs that no cache holds, and the next kernel to read them finds them there (forward, then
  // backward, three sets of tensors in turn; kernel us, streaming -> kept, forward and backward): AdaLN 1500 x 5120 7.6 / 14.0
  // -> 6.6 / 11.0, 5000 x 4096 16.1 / 24.5 -> 12.9 / 21.8, RMSNorm 5000 x 1536 7.6 / 11.6 -> 6.2 / 9.4, gate 2500 x 3072 10.4 / 10.4
  // -> 8.8 / 6.2, residual + norm 2000 x 3072 11.9 / 17.0 -> 9.4 / 14.1.  With more tensors a call the limit is lower (means
  // over 28 widths, streaming / kept): residual + norm forward 16 MB 1.11, 17.5 MB 1.02, 20 MB 1.00 (down to 0.94: 2441 x 4096 15.5 -> 16.3,
  // 1627 x 6144 16.8 -> 17.9), gate forward with idle lanes 48 MB 1.05, 53 MB 1.00, 60 MB 0.95 (25862 x 1160 30.1 ->
  // 33.0; its backward goes with it: behind a streaming forward 36.2 streaming, 40.5 kept, behind a keeping one 35.0 kept), with
  // every lane in use 60 MB 0.99 and its backward 1.10 (19531 x 1536 31.2 / 32.0 -> 30.6 / 27.0); x_norm
  // forward and its backward 4972 x 3072 18.1 / 21.8 -> 17.0 / 20.9, 9000 x 3072 31.0 / 32.4 -> 30.8 / 33.4; gated, 4000 x 3072
  // 18.8 / 29.1 -> 18.6 / 29.1.  Beyond the caches streaming is the faster (75600 x 5120 374 -> 410).
  const int64_t keep_mib = res == 2 ? 0 : res ? 18 : dir == kFwdXn || dir == kBwdSaved ? 40
                         : kind == kGateKind && !full ? 52 : 64;
  plan->k = rows * cols * 2 < keep_mib << 20 ? pick(mode | kKeep) : k;
  plan->packs = packs;
  plan->n_batches = rows / rows_per_batch;
  plan->n_tiles = (rows_per_batch + k.tile_rows - 1) / k.tile_rows;
  if (plan->n_batches > 65535) return TT_ERR_UNSUPPORTED;
  int64_t gx = (int64_t)per_cu * usable_cus / plan->n_batches;
  if (gx < 1) gx = 1;
  if (gov > 0 && gov <= kMaxWgsPerCu * cus) gx = gov / plan->n_batches > 0 ? gov / plan->n_batches : 1;
  if (gx > plan->n_tiles) gx = plan->n_tiles;
  plan->grid_x = static_cast<int>(gx);
  return TT_OK;
}

size_t partial_bytes(const Plan& p, int n_acc, int64_t cols) {
  return (size_t)p.n_batches * p.grid_x * n_acc * cols * sizeof(float);
}

// Caps the grid so that the partial sums fit `bytes`; false if one workgroup a batch does not.
bool fit_grid(Plan* p, int n_acc, int64_t cols, size_t bytes) {
  const size_t fit = bytes / ((size_t)p->n_batches * n_acc * cols * sizeof(float));
  if (fit < 1) return false;
  if (fit < (size_t)p->grid_x) p->grid_x = (int)fit;
  return true;
}

// Whether tt_adaln_backward_static takes an aligned tensor.
bool static_takes(int64_t rows, int64_t cols, int64_t rows_per_batch) {
  Plan p;
  return make_plan(kAdaLN, kBwd, rows, cols, rows_per_batch, &p, false, 0, 0, kMasked) == TT_OK &&
         partial_bytes(p, 2, cols) <= TT_STATIC_WORKSPACE_BYTES;
}

// Plan of the backward of aligned rows.  tt_adaln_backward_static runs what tt_adaln_backward does, so where it
// takes the shape the partial sums have to fit its array (they do without the cap while ragged rows have no more
// than twice the workgroups of whole-line rows).
int backward_plan(int kind, int64_t rows, int64_t cols, int64_t rows_per_batch, Plan* p, bool rope = false,
                  int64_t rope_heads = 0) {
  const int rc = make_plan(kind, kBwd, rows, cols, rows_per_batch, p, rope, 0, rope_heads);
  if (rc == TT_OK && kind == kAdaLN && partial_bytes(*p, 2, cols) > kScratchBytes && static_takes(rows, cols, rows_per_batch))
    fit_grid(p, 2, cols, kScratchBytes);
  return rc;
}

size_t workspace_for(int kind, int n_acc, int64_t rows, int64_t cols, int64_t rows_per_batch);

// Backward of rows that the 128-bit kernels do not take (cols % 8 != 0, or tensors that are only 2-byte
// aligned).  Rows of more than 256 values take the kOdd kernels, which leave partial column sums like
// all others, as long as those stay small: at most the size of the scratch array or of x and dy.  Beyond
// that (a modulation vector for every few rows), and for shorter rows, the element-wise kernels run, which
// keep two floats a row (their column sums have cols / 64 workgroups).  us forward / backward, element-wise ->
// these: RMSNorm 5000 x 1001 12.6 / 117 -> 9.4 / 16, AdaLN 8000 x 1999 33 / 125 -> 17 / 29, 60000 x 1537
// 283 / 2122 -> 79 / 133 (1544 columns, 16-byte aligned rows: 67 / 109).  Rows of more than 16384 values stay
// element-wise: their wide kernel (16 waves of four packs a lane) spills its column sums and is the slower one,
// AdaLN / RMSNorm 10485 x 20001 1080 / 904 -> 2256 / 1738, 2047 x 16391 128 / 103 -> 453 / 337, against
// 12800 x 16383 1085 / 919 -> 907 / 420.
// Where cols % 8 == 0 the size query does not know of the misaligned tensor and answers for the aligned
// kernels, which may want less (two rows a tile: half the workgroups).  The grid is then what the answer
// holds, so that which kernels run, and the order of their sums, depends on the shape and not on what else
// the workspace has room for.  For the same reason AdaLN's partial sums fit the scratch array, with which
// tt_adaln_backward_static gives the same bits (300 x 10 x 16383 472 -> 343 us; element-wise where one
// workgroup a batch does not fit: 5000 x 10 x 1001 338 -> 353).
constexpr int64_t kOddBwdMaxCols = 16384;
bool odd_plan(int kind, int64_t rows, int64_t cols, int64_t rows_per_batch, Plan* p) {
  if (cols > kOddBwdMaxCols || make_plan(kind, kBwd, rows, cols, rows_per_batch, p, false, 0, 0, kOdd) != TT_OK) return false;
  const int n_acc = kind == kAdaLN ? 2 : 1;
  const size_t tensors = (size_t)rows * cols * 4;
  const size_t most = tensors > TT_STATIC_WORKSPACE_BYTES ? tensors : (size_t)TT_STATIC_WORKSPACE_BYTES;
  if (partial_bytes(*p, n_acc, cols) > most) return false;
  if (kind == kAdaLN && !fit_grid(p, n_acc, cols, kScratchBytes)) return false;
  return cols % kPack != 0 || fit_grid(p, n_acc, cols, workspace_for(kind, n_acc, rows, cols, rows_per_batch));
}

// Workspace bound that does not depend on the launch-time occupancy query.
size_t workspace_bound(int n_acc, int64_t rows, int64_t cols, int64_t rows_per_batch) {
  if (rows <= 0 || cols <= 0 || rows_per_batch <= 0 || rows % rows_per_batch != 0) return 0;
  if (cols % kPack != 0) return (size_t)rows * 2 * sizeof(float);   // element-wise path: row statistics
  int cus = 0;
  if (current_device_cus(&cus) != TT_OK) cus = 256;
  const int64_t n_batches = rows / rows_per_batch;
  int64_t gx = (int64_t)kMaxWgsPerCu * cus / n_batches;
  if (gx < 1) gx = 1;
  if (gx > rows_per_batch) gx = rows_per_batch;
  return (size_t)n_batches * gx * n_acc * cols * sizeof(float);
}

// What the backward entry points of `kind` need for this shape: the partial sums of the plan they
// will actually launch (the larger of the two backward contracts).  Falls back to the
// plan-independent bound when a plan cannot be made here or a tuning override is active.
size_t workspace_for(int kind, int n_acc, int64_t rows, int64_t cols, int64_t rows_per_batch) {
  const size_t bound = workspace_bound(n_acc, rows, cols, rows_per_batch);
  if (bound == 0) return bound;
  if (cols % kPack != 0) {
    Plan po;
    if (!odd_plan(kind, rows, cols, rows_per_batch, &po)) return bound;
    const size_t need = partial_bytes(po, n_acc, cols);
    return need > bound ? need : bound;
  }
  if (g_wgs_per_cu_override.load() > 0 || g_grid_override.load() > 0) return bound;
  Plan p;
  if (backward_plan(kind, rows, cols, rows_per_batch, &p) != TT_OK) return bound;
  size_t need = partial_bytes(p, n_acc, cols);
  if (kind != kGateKind && rows_per_batch == rows) {
    Plan ps;
    if (make_plan(kind, kBwdSaved, rows, cols, rows, &ps) != TT_OK) return bound;
    const size_t ns = partial_bytes(ps, n_acc, cols);
    if (ns > need) need = ns;
  }
  if (kind == kRMS) {   // tt_rmsnorm_rope[_heads]_backward share this size query: per-row and per-token kernels
    for (int64_t heads : {0, 12, 16, 24, 32, 48}) {   // 0: one lookup a row; each token mode of both row lengths
      if (heads && cols > 128) break;
      Plan pr;
      if (make_plan(kRMS, kBwd, rows, cols, rows, &pr, true, 0, heads) == TT_OK) {
        const size_t nr = partial_bytes(pr, n_acc, cols);
        if (nr > need) need = nr;
      }
    }
  }
  return need < 16 ? 16 : need;
}

template <typename Args>
int launch(const Plan& p, Args& args, void* stream) {
  void* kargs[] = {&args};
  hipError_t e = hipLaunchKernel(p.k.fn, dim3(p.grid(), (unsigned)p.n_batches, 1), dim3(p.k.threads, 1, 1),
                                 kargs, 0, static_cast<hipStream_t>(stream));
  if (e != hipSuccess) return hip_fail(e);
  return TT_OK;
}

// ---------------------------------------------------------------- element-wise fallback
bool aligned4(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 3u) == 0; }
bool aligned2(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 1u) == 0; }

int generic_grid(int64_t rows, int* grid) {
  int cus = 0;
  int rc = current_device_cus(&cus);
  if (rc != TT_OK) return rc;
  const int64_t cap = (int64_t)cus * 8;
  *grid = (int)(rows < cap ? rows : cap);
  return TT_OK;
}

int check_shape(int64_t rows, int64_t cols, int64_t rows_per_batch) {
  if (rows <= 0 || cols <= 0 || rows_per_batch <= 0 || rows % rows_per_batch != 0) return TT_ERR_INVALID_ARGUMENT;
  if (cols > TT_MAX_COLS || rows / rows_per_batch > 65535) return TT_ERR_UNSUPPORTED;
  return TT_OK;
}

int reduce(void* out0, void* out1, const void* workspace, int n_batches, int n_partials, int n_acc,
           int64_t cols, bool out_bf16, void* stream, void* out2 = nullptr);

int forward_generic(int kind, void* y, const void* x, const void* p0, const void* p1, float* mean, float* rstd,
                    void* x_norm, int64_t rows, int64_t cols, int64_t rows_per_batch, float eps, void* stream,
                    const Params* params) {
  int rc = check_shape(rows, cols, rows_per_batch);
  if (rc != TT_OK) return rc;
  if (!aligned2(y) || !aligned2(x) || !aligned2(p0) || !aligned2(p1) || !aligned2(x_norm)) return TT_ERR_INVALID_ARGUMENT;
  if (params && (!aligned2(params->copy) || (params->f32 && !aligned4(p0)))) return TT_ERR_INVALID_ARGUMENT;
  Plan p;
  if (make_plan(kind, x_norm ? kFwdXn : kFwd, rows, cols, rows_per_batch, &p, false, 0, 0, kOdd) == TT_OK) {
    FwdArgs f = {};
    f.p0_stride = params ? params->stride0 : cols; f.p1_stride = params ? params->stride1 : cols;
    f.p0_f32 = params ? params->f32 : 0; f.p0_copy = params ? params->copy : nullptr;
    f.y = y; f.x = x; f.p0 = p0; f.p1 = p1; f.mean = mean; f.rstd = rstd; f.x_norm = x_norm;
    f.rows_per_batch = rows_per_batch; f.n_tiles = p.n_tiles;
    f.cols = (int)cols; f.packs = p.packs; f.eps = eps; f.inv_cols = 1.0f / (float)cols;
    return launch(p, f, stream);
  }
  if (params) return TT_ERR_UNSUPPORTED;   // the element-wise kernels read dense bf16 parameters only
  int grid = 0;
  rc = generic_grid(rows, &grid);
  if (rc != TT_OK) return rc;
  GenFwdArgs a;
  a.y = static_cast<uint16_t*>(y); a.x = static_cast<const uint16_t*>(x);
  a.p0 = static_cast<const uint16_t*>(p0); a.p1 = static_cast<const uint16_t*>(p1);
  a.mean = mean; a.rstd = rstd; a.x_norm = static_cast<uint16_t*>(x_norm);
  a.rows = rows; a.rows_per_batch = rows_per_batch; a.cols = (int)cols; a.eps = eps; a.inv_cols = 1.0f / (float)cols;
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (kind == kAdaLN) hipLaunchKernelGGL(norm_fwd_generic<kAdaLN>, dim3(grid), dim3(kGenThreads), 0, s, a);
  else                hipLaunchKernelGGL(norm_fwd_generic<kRMS>, dim3(grid), dim3(kGenThreads), 0, s, a);
  hipError_t e = hipGetLastError();
  return e == hipSuccess ? TT_OK : hip_fail(e);
}

int backward_generic(int kind, void* dx, void* out0, void* out1, const void* dy, const void* x, const void* p0,
                     void* workspace, size_t workspace_bytes, int64_t rows, int64_t cols, int64_t rows_per_batch,
                     float eps, void* stream, bool out_bf16) {
  int rc = check_shape(rows, cols, rows_per_batch);
  if (rc != TT_OK) return rc;
  if (!dx || !dy || !x || !p0 || !out0 || (kind == kAdaLN && !out1)) return TT_ERR_INVALID_ARGUMENT;
  if (!aligned2(dx) || !aligned2(dy) || !aligned2(x) || !aligned2(p0)) return TT_ERR_INVALID_ARGUMENT;
  if (!workspace || (reinterpret_cast<uintptr_t>(workspace) & 3u) != 0 ||
      workspace_bytes < (size_t)rows * 2 * sizeof(float))
    return TT_ERR_WORKSPACE;
  Plan p;
  if (odd_plan(kind, rows, cols, rows_per_batch, &p)) {
    const int n_acc = kind == kAdaLN ? 2 : 1;
    if (workspace_bytes >= partial_bytes(p, n_acc, cols)) {
      BwdArgs b = {};
      b.dx = dx; b.dy = dy; b.x = x; b.p0 = p0; b.partials = static_cast<float*>(workspace);
      b.rows_per_batch = rows_per_batch; b.n_tiles = p.n_tiles;
      b.cols = (int)cols; b.packs = p.packs; b.eps = eps; b.inv_cols = 1.0f / (float)cols;
      rc = launch(p, b, stream);
      if (rc != TT_OK) return rc;
      return reduce(out0, out1, workspace, (int)p.n_batches, p.grid(), n_acc, cols, out_bf16, stream);
    }
  }
  int grid = 0;
  rc = generic_grid(rows, &grid);
  if (rc != TT_OK) return rc;
  GenBwdArgs a;
  a.dx = static_cast<uint16_t*>(dx); a.dy = static_cast<const uint16_t*>(dy); a.x = static_cast<const uint16_t*>(x);
  a.p0 = static_cast<const uint16_t*>(p0); a.stats = static_cast<float*>(workspace); a.out0 = out0; a.out1 = out1;
  a.rows = rows; a.rows_per_batch = rows_per_batch; a.cols = (int)cols; a.eps = eps; a.inv_cols = 1.0f / (float)cols;
  a.out_bf16 = out_bf16 ? 1 : 0;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const dim3 cgrid((unsigned)((cols + 63) / 64), (unsigned)(rows / rows_per_batch), 1);
  if (kind == kAdaLN) {
    hipLaunchKernelGGL(norm_bwd_generic<kAdaLN>, dim3(grid), dim3(kGenThreads), 0, s, a);
    hipLaunchKernelGGL(norm_colgrad_generic<kAdaLN>, cgrid, dim3(1024), 0, s, a);
  } else {
    hipLaunchKernelGGL(norm_bwd_generic<kRMS>, dim3(grid), dim3(kGenThreads), 0, s, a);
    hipLaunchKernelGGL(norm_colgrad_generic<kRMS>, cgrid, dim3(1024), 0, s, a);
  }
  hipError_t e = hipGetLastError();
  return e == hipSuccess ? TT_OK : hip_fail(e);
}

// The vector kernels need 128-bit packs: cols % 8 == 0 and 16-byte aligned tensors.
bool vector_path(int64_t cols, std::initializer_list<const void*> ptrs) {
  if (cols % kPack != 0) return false;
  for (const void* p : ptrs)
    if (!aligned16(p)) return false;
  return true;
}

int check_rope(const Rope& rope, int64_t rows, int64_t cols) {
  if (!rope.freqs || rope.head_dim <= 0 || rope.seq_len <= 0 || rope.heads < 0) return TT_ERR_INVALID_ARGUMENT;
  if (rope.head_dim % kPack != 0 || rope.head_dim > 256 || cols % rope.head_dim != 0 || !aligned16(rope.freqs))
    return TT_ERR_UNSUPPORTED;
  if (rope.heads > 0) {   // one head per row: the narrow kernels
    if (cols != rope.head_dim) return TT_ERR_UNSUPPORTED;
    if (rows % rope.heads != 0) return TT_ERR_INVALID_ARGUMENT;
  } else if (cols / kPack <= kNarrowMaxPacks) {
    return TT_ERR_UNSUPPORTED;   // all heads in one row: the wide kernels
  }
  return TT_OK;
}

int forward(int kind, void* y, const void* x, const void* p0, const void* p1, float* mean, float* rstd, void* x_norm,
            int64_t rows, int64_t cols, int64_t rows_per_batch, float eps, void* stream, const Rope* rope = nullptr,
            const Params* params = nullptr) {
  if (rows == 0) return TT_OK;
  if (!y || !x || !p0 || (kind == kAdaLN && !p1)) return TT_ERR_INVALID_ARGUMENT;
  const Params dense{cols, cols, 0, nullptr};
  const Params& pm = params ? *params : dense;
  const bool aligned = vector_path(cols, {y, x, p0, p1, x_norm, pm.copy}) && (pm.stride0 | pm.stride1) % kPack == 0;
  if (rope) {
    if (!aligned) return TT_ERR_UNSUPPORTED;
    const int rrc = check_rope(*rope, rows, cols);
    if (rrc != TT_OK) return rrc;
  } else if (!aligned) {
    return forward_generic(kind, y, x, p0, p1, mean, rstd, x_norm, rows, cols, rows_per_batch, eps, stream, params);
  }
  Plan p;
  if (x_norm && (kind != kAdaLN || rope)) return TT_ERR_UNSUPPORTED;
  int rc = make_plan(kind, x_norm ? kFwdXn : kFwd, rows, cols, rows_per_batch, &p, rope != nullptr, 0,
                     rope ? rope->heads : 0);
  if (rc != TT_OK) return rc;
  FwdArgs a;
  a.freqs = rope ? rope->freqs : nullptr; a.seq_len = rope ? rope->seq_len : 1; a.head_dim = rope ? (int)rope->head_dim : 8;
  a.rows_per_pos = rope && rope->heads > 0 ? rope->heads : 1;
  a.p0_stride = pm.stride0; a.p1_stride = pm.stride1; a.p0_f32 = pm.f32; a.p0_copy = pm.copy;
  a.y = y; a.x = x; a.p0 = p0; a.p1 = p1; a.mean = mean; a.rstd = rstd; a.x_norm = x_norm;
  a.rows_per_batch = rows_per_batch; a.n_tiles = p.n_tiles;
  a.cols = (int)cols; a.packs = p.packs; a.eps = eps; a.inv_cols = 1.0f / (float)cols;
  return launch(p, a, stream);
}

int backward_partials(int kind, void* dx, const void* dy, const void* x, const void* p0,
                      void* workspace, size_t workspace_bytes, int* n_partials,
                      int64_t rows, int64_t cols, int64_t rows_per_batch, float eps, void* stream,
                      const Rope* rope = nullptr) {
  if (n_partials) *n_partials = 0;
  if (rows == 0) return TT_OK;
  if (!dx || !dy || !x || !p0) return TT_ERR_INVALID_ARGUMENT;
  if (!aligned16(dx) || !aligned16(dy) || !aligned16(x) || !aligned16(p0)) return TT_ERR_UNSUPPORTED;
  if (rope) {
    const int rrc = check_rope(*rope, rows, cols);
    if (rrc != TT_OK) return rrc;
  }
  Plan p;
  int rc = backward_plan(kind, rows, cols, rows_per_batch, &p, rope != nullptr, rope ? rope->heads : 0);
  if (rc != TT_OK) return rc;
  const int n_acc = kind == kAdaLN ? 2 : 1;
  if (!rope && workspace_bytes < partial_bytes(p, n_acc, cols)) {
    // Ragged rows: a workspace smaller than asked for, but large enough for the kernels of whole-line rows
    // (which have fewer workgroups resident), gets the grid of those.
    Plan pm;
    if (make_plan(kind, kBwd, rows, cols, rows_per_batch, &pm, false, 0, 0, kMasked) == TT_OK &&
        pm.grid_x < p.grid_x && workspace_bytes >= partial_bytes(pm, n_acc, cols))
      p.grid_x = pm.grid_x;
  }
  if (!workspace || !aligned16(workspace) || workspace_bytes < partial_bytes(p, n_acc, cols)) return TT_ERR_WORKSPACE;
  BwdArgs a;
  a.freqs = rope ? rope->freqs : nullptr; a.seq_len = rope ? rope->seq_len : 1; a.head_dim = rope ? (int)rope->head_dim : 8;
  a.rows_per_pos = rope && rope->heads > 0 ? rope->heads : 1;
  a.dx = dx; a.dy = dy; a.x = x; a.p0 = p0; a.partials = static_cast<float*>(workspace);
  a.rows_per_batch = rows_per_batch; a.n_tiles = p.n_tiles;
  a.cols = (int)cols; a.packs = p.packs; a.eps = eps; a.inv_cols = 1.0f / (float)cols;
  rc = launch(p, a, stream);
  if (rc == TT_OK && n_partials) *n_partials = p.grid();
  return rc;
}

int backward_saved_partials(int kind, void* dx, const void* dy, const void* xs, const void* p0, const float* rstd,
                            void* workspace, size_t workspace_bytes, int* n_partials,
                            int64_t rows, int64_t cols, void* stream) {
  *n_partials = 0;
  if (rows == 0) return TT_OK;
  if (!dx || !dy || !xs || !p0 || !rstd) return TT_ERR_INVALID_ARGUMENT;
  if (!aligned16(dx) || !aligned16(dy) || !aligned16(xs) || !aligned16(p0)) return TT_ERR_UNSUPPORTED;
  Plan p;
  int rc = make_plan(kind, kBwdSaved, rows, cols, rows, &p);
  if (rc != TT_OK) return rc;
  const int n_acc = kind == kAdaLN ? 2 : 1;
  if (!workspace || !aligned16(workspace) || workspace_bytes < partial_bytes(p, n_acc, cols)) return TT_ERR_WORKSPACE;
  BwdSavedArgs a;
  a.dx = dx; a.dy = dy; a.xs = xs; a.p0 = p0; a.rstd = rstd; a.partials = static_cast<float*>(workspace);
  a.rows_per_batch = rows; a.n_tiles = p.n_tiles;
  a.cols = (int)cols; a.packs = p.packs; a.inv_cols = 1.0f / (float)cols;
  rc = launch(p, a, stream);
  if (rc == TT_OK) *n_partials = p.grid();
  return rc;
}

int reduce(void* out0, void* out1, const void* workspace, int n_batches, int n_partials, int n_acc,
           int64_t cols, bool out_bf16, void* stream, void* out2) {
  if (n_batches == 0) return TT_OK;
  if (!out0 || !workspace || n_batches < 0 || n_batches > 65535 || n_partials <= 0 || cols <= 0 ||
      cols > TT_MAX_COLS || n_acc < 1 || n_acc > 3 || (n_acc >= 2 && !out1) || (n_acc == 3 && !out2))
    return TT_ERR_INVALID_ARGUMENT;
  // 32 columns a workgroup where 64 would leave CUs without one (see reduce_partials); with many batches, which have
  // few partials each, it would only double the idle waves (300 batches of 5120 columns 58 -> 118 us).  Up to 128 partials
  // are one round of loads at 64 columns as well: us at 32 -> 64, three sums each, 85 partials of 3 x 5120 6.3 -> 4.8, 82 of
  // 3 x 3072 6.0 -> 4.7, 62 of 4 x 3072 6.0 -> 4.7, 50 of 2 x 5120 6.5 -> 4.3; one batch or fewer sums 0.0 to 0.2 faster.
  // So do long rows of partial sums that are no whole lines, which two workgroups of 32 columns share: 256 partials, three |
  // two sums, 32 -> 64 columns, 4616 columns 5.7 -> 5.8 | 4.8 -> 4.2, 5640: 6.4 -> 5.9 | 4.8 -> 4.2, 8184: 8.3 -> 7.1 | 5.8 -> 5.0;
  // the other way round at 4104 (5.4 -> 5.6 | 4.1 -> 4.6) and 3080 (4.7 -> 5.6 | 4.0 -> 4.1).
  int cus = 0;
  const int rc = current_device_cus(&cus);
  if (rc != TT_OK) return rc;
  const bool wide = (cols + 63) / 64 * n_batches >= cus || n_partials <= 128 || (cols % 32 != 0 && cols > 4608);
  const int lc = wide ? 64 : 32;
  const dim3 grid((unsigned)((cols + lc - 1) / lc), (unsigned)n_batches, 1);
  using Kernel = void (*)(void*, void*, void*, const float*, int, int, int);
  static constexpr Kernel kernels[3][2] = {{reduce_partials<1, 32>, reduce_partials<1, 64>},
                                           {reduce_partials<2, 32>, reduce_partials<2, 64>},
                                           {reduce_partials<3, 32>, reduce_partials<3, 64>}};
  hipLaunchKernelGGL(kernels[n_acc - 1][wide], grid, dim3(1024), 0, static_cast<hipStream_t>(stream), out0, out1, out2,
                     static_cast<const float*>(workspace), n_partials, (int)cols, out_bf16 ? 1 : 0);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return hip_fail(e);
  return TT_OK;
}

}  // namespace
}  // namespace tt

using namespace tt;

extern "C" {

int tt_version(void) { return 100; }

const char* tt_error_string(int code) {
  switch (code) {
    case TT_OK: return "ok";
    case TT_ERR_INVALID_ARGUMENT: return "invalid argument (null pointer, non-positive size, or rows not a multiple of rows_per_batch)";
    case TT_ERR_UNSUPPORTED: return "unsupported shape or alignment";
    case TT_ERR_WORKSPACE: return "workspace missing, misaligned or too small";
    case TT_ERR_HIP: return "HIP runtime error (see tt_last_hip_error)";
    case TT_ERR_STATIC_LIMIT: return "shape needs more than TT_STATIC_WORKSPACE_BYTES of scratch (partial sums, or rows * 8 bytes where cols % 8 != 0 or a tensor is misaligned): use the entry point that takes a workspace";
    default: return "unknown error code";
  }
}

int tt_last_hip_error(void) { return g_last_hip_error; }

#ifdef TT_TUNING_HOOKS
// Tuning hooks, compiled only into sweep builds (not part of the public header): force the number
// of resident workgroups per CU that launch plans assume, or the total number of workgroups of a
// launch; 0 restores the plan's own choice.
TT_API void tt_debug_set_wgs_per_cu(int n) { g_wgs_per_cu_override.store(n < 0 ? 0 : n); }
TT_API void tt_debug_set_grid(int n) { g_grid_override.store(n < 0 ? 0 : n); }
#endif

int tt_adaln_forward(void* y, const void* x, const void* scale, const void* shift, float* mean, float* rstd,
                     int64_t rows, int64_t cols, int64_t rows_per_batch, float eps, void* stream) {
  return forward(kAdaLN, y, x, scale, shift, mean, rstd, nullptr, rows, cols, rows_per_batch, eps, stream);
}

int tt_rmsnorm_forward(void* y, const void* x, const void* weight, float* rstd,
                       int64_t rows, int64_t cols, float eps, void* stream) {
  return forward(kRMS, y, x, weight, nullptr, nullptr, rstd, nullptr, rows, cols, rows, eps, stream);
}

size_t tt_adaln_backward_workspace_bytes(int64_t rows, int64_t cols, int64_t rows_per_batch) {
  return workspace_for(kAdaLN, 2, rows, cols, rows_per_batch);
}
size_t tt_rmsnorm_backward_workspace_bytes(int64_t rows, int64_t cols) {
  return workspace_for(kRMS, 1, rows, cols, rows);
}

int tt_adaln_backward_partials(void* dx, const void* dy, const void* x, const void* scale,
                               void* workspace, size_t workspace_bytes, int* n_partials,
                               int64_t rows, int64_t cols, int64_t rows_per_batch, float eps, void* stream) {
  return backward_partials(kAdaLN, dx, dy, x, scale, workspace, workspace_bytes, n_partials,
                           rows, cols, rows_per_batch, eps, stream);
}
int tt_rmsnorm_backward_partials(void* dx, const void* dy, const void* x, const void* weight,
                                 void* workspace, size_t workspace_bytes, int* n_partials,
                                 int64_t rows, int64_t cols, float eps, void* stream) {
  return backward_partials(kRMS, dx, dy, x, weight, workspace, workspace_bytes, n_partials,
                           rows, cols, rows, eps, stream);
}

int tt_reduce_partials(float* out0, float* out1, const void* workspace,
                       int n_batches, int n_partials, int n_acc, int64_t cols, void* stream) {
  return reduce(out0, out1, workspace, n_batches, n_partials, n_acc, cols, false, stream);
}

int tt_adaln_backward_typed(void* dx, void* dscale, void* dshift, int grads_bf16, const void* dy, const void* x,
                            const void* scale, void* workspace, size_t workspace_bytes,
                            int64_t rows, int64_t cols, int64_t rows_per_batch, float eps, void* stream) {
  if (rows == 0) return TT_OK;
  if (!dscale || !dshift) return TT_ERR_INVALID_ARGUMENT;
  if (!vector_path(cols, {dx, dy, x, scale, workspace}))
    return backward_generic(kAdaLN, dx, dscale, dshift, dy, x, scale, workspace, workspace_bytes,
                            rows, cols, rows_per_batch, eps, stream, grads_bf16 != 0);
  int n_partials = 0;
  int rc = backward_partials(kAdaLN, dx, dy, x, scale, workspace, workspace_bytes, &n_partials,
                             rows, cols, rows_per_batch, eps, stream);
  if (rc != TT_OK) return rc;
  return reduce(dscale, dshift, workspace, (int)(rows / rows_per_batch), n_partials, 2, cols, grads_bf16 != 0, stream);
}

int tt_adaln_backward(void* dx, float* dscale, float* dshift, const void* dy, const void* x, const void* scale,
                      void* workspace, size_t workspace_bytes,
                      int64_t rows, int64_t cols, int64_t rows_per_batch, float eps, void* stream) {
  return tt_adaln_backward_typed(dx, dscale, dshift, 0, dy, x, scale, workspace, workspace_bytes,
                                 rows, cols, rows_per_batch, eps, stream);
}

int tt_adaln_backward_static(void* dx, float* dscale, float* dshift, const void* dy, const void* x,
                             const void* scale, int64_t rows, int64_t cols, int64_t rows_per_batch, float eps,
                             void* stream) {
  void* ws = nullptr;
  int rc = static_scratch(&ws);   // per-device set-up on the first call; a rows == 0 call does only this
  if (rc != TT_OK) return rc;
  if (rows == 0) return TT_OK;
  // More is refused than the array could hold: see kScratchBytes.  (Invalid arguments are for tt_adaln_backward to name.)
  if (rows > 0 && cols > 0 && rows_per_batch > 0 && rows % rows_per_batch == 0 && cols <= TT_MAX_COLS &&
      rows / rows_per_batch <= 65535 && dx && dy && x && scale && dscale && dshift) {
    if (vector_path(cols, {dx, dy, x, scale}) ? !static_takes(rows, cols, rows_per_batch)
                                              : (size_t)rows * 2 * sizeof(float) > TT_STATIC_WORKSPACE_BYTES)
      return TT_ERR_STATIC_LIMIT;
  }
  rc = tt_adaln_backward(dx, dscale, dshift, dy, x, scale, ws, kScratchBytes, rows, cols, rows_per_batch, eps, stream);
  return rc == TT_ERR_WORKSPACE ? TT_ERR_STATIC_LIMIT : rc;
}

int tt_rmsnorm_backward_typed(void* dx, void* dweight, int grads_bf16, const void* dy, const void* x, const void* weight,
                              const float* freqs, int64_t head_dim, int64_t heads, int64_t seq_len,
                              void* workspace, size_t workspace_bytes,
                              int64_t rows, int64_t cols, float eps, void* stream) {
  if (rows == 0) return TT_OK;
  if (!dweight) return TT_ERR_INVALID_ARGUMENT;
  Rope rope;
  rope.freqs = freqs; rope.head_dim = head_dim; rope.seq_len = seq_len; rope.heads = heads;
  if (!freqs && !vector_path(cols, {dx, dy, x, weight, workspace}))
    return backward_generic(kRMS, dx, dweight, nullptr, dy, x, weight, workspace, workspace_bytes,
                            rows, cols, rows, eps, stream, grads_bf16 != 0);
  int n_partials = 0;
  int rc = backward_partials(kRMS, dx, dy, x, weight, workspace, workspace_bytes, &n_partials,
                             rows, cols, rows, eps, stream, freqs ? &rope : nullptr);
  if (rc != TT_OK) return rc;
  return reduce(dweight, nullptr, workspace, 1, n_partials, 1, cols, grads_bf16 != 0, stream);
}

int tt_rmsnorm_backward(void* dx, float* dweight, const void* dy, const void* x, const void* weight,
                        void* workspace, size_t workspace_bytes,
                        int64_t rows, int64_t cols, float eps, void* stream) {
  return tt_rmsnorm_backward_typed(dx, dweight, 0, dy, x, weight, nullptr, 0, 0, 0, workspace, workspace_bytes,
                                   rows, cols, eps, stream);
}

int tt_adaln_forward_strided(void* y, const void* x, const void* scale, int64_t scale_stride,
                             const void* shift, int64_t shift_stride, void* scale_copy,
                             int64_t rows, int64_t cols, int64_t rows_per_batch, float eps, void* stream) {
  if (scale_stride < 0 || shift_stride < 0) return TT_ERR_INVALID_ARGUMENT;
  const Params pm{scale_stride, shift_stride, 0, scale_copy};
  return forward(kAdaLN, y, x, scale, shift, nullptr, nullptr, nullptr, rows, cols, rows_per_batch, eps, stream, nullptr, &pm);
}

int tt_rmsnorm_forward_f32_weight(void* y, const void* x, const float* weight, void* weight_copy,
                                  int64_t rows, int64_t cols, float eps, void* stream) {
  const Params pm{0, 0, 1, weight_copy};
  return forward(kRMS, y, x, weight, nullptr, nullptr, nullptr, nullptr, rows, cols, rows, eps, stream, nullptr, &pm);
}

// ---------------------------------------------------------------- RMSNorm + rotary embedding
int tt_rmsnorm_rope_forward(void* y, const void* x, const void* weight, const float* freqs, float* rstd,
                            int64_t rows, int64_t cols, int64_t head_dim, int64_t seq_len, float eps, void* stream) {
  Rope rope; rope.freqs = freqs; rope.head_dim = head_dim; rope.seq_len = seq_len;
  return forward(kRMS, y, x, weight, nullptr, nullptr, rstd, nullptr, rows, cols, rows, eps, stream, &rope);
}

int tt_rmsnorm_rope_backward(void* dx, float* dweight, const void* dy, const void* x, const void* weight,
                             const float* freqs, void* workspace, size_t workspace_bytes,
                             int64_t rows, int64_t cols, int64_t head_dim, int64_t seq_len, float eps, void* stream) {
  if (rows == 0) return TT_OK;
  if (!dweight) return TT_ERR_INVALID_ARGUMENT;
  Rope rope; rope.freqs = freqs; rope.head_dim = head_dim; rope.seq_len = seq_len;
  int n_partials = 0;
  int rc = backward_partials(kRMS, dx, dy, x, weight, workspace, workspace_bytes, &n_partials,
                             rows, cols, rows, eps, stream, &rope);
  if (rc != TT_OK) return rc;
  return reduce(dweight, nullptr, workspace, 1, n_partials, 1, cols, false, stream);
}

int tt_rmsnorm_rope_heads_forward(void* y, const void* x, const void* weight, const float* freqs, float* rstd,
                                  int64_t rows, int64_t head_dim, int64_t heads, int64_t seq_len, float eps,
                                  void* stream) {
  if (heads <= 0) return TT_ERR_INVALID_ARGUMENT;
  Rope rope; rope.freqs = freqs; rope.head_dim = head_dim; rope.seq_len = seq_len; rope.heads = heads;
  return forward(kRMS, y, x, weight, nullptr, nullptr, rstd, nullptr, rows, head_dim, rows, eps, stream, &rope);
}

int tt_rmsnorm_rope_heads_backward(void* dx, float* dweight, const void* dy, const void* x, const void* weight,
                                   const float* freqs, void* workspace, size_t workspace_bytes,
                                   int64_t rows, int64_t head_dim, int64_t heads, int64_t seq_len, float eps,
                                   void* stream) {
  if (rows == 0) return TT_OK;
  if (!dweight || heads <= 0) return TT_ERR_INVALID_ARGUMENT;
  Rope rope; rope.freqs = freqs; rope.head_dim = head_dim; rope.seq_len = seq_len; rope.heads = heads;
  int n_partials = 0;
  int rc = backward_partials(kRMS, dx, dy, x, weight, workspace, workspace_bytes, &n_partials,
                             rows, head_dim, rows, eps, stream, &rope);
  if (rc != TT_OK) return rc;
  return reduce(dweight, nullptr, workspace, 1, n_partials, 1, head_dim, false, stream);
}

// ---------------------------------------------------------------- gated residual add
int tt_gate_residual_forward_strided(void* out, const void* x, const void* gate, int64_t gate_stride, void* gate_copy,
                                     const void* residual, int64_t rows, int64_t cols, int64_t rows_per_batch,
                                     void* stream) {
  if (rows == 0) return TT_OK;
  if (!out || !x || !gate || !residual || gate_stride < 0) return TT_ERR_INVALID_ARGUMENT;
  if (!vector_path(cols, {out, x, gate, residual, gate_copy}) || gate_stride % kPack != 0) return TT_ERR_UNSUPPORTED;
  Plan p;
  int rc = make_plan(kGateKind, kFwd, rows, cols, rows_per_batch, &p);
  if (rc != TT_OK) return rc;
  GateArgs a;
  a.out = out; a.a = x; a.b = residual; a.gate = gate; a.partials = nullptr;
  a.gate_stride = gate_stride; a.gate_copy = gate_copy;
  a.rows_per_batch = rows_per_batch; a.n_tiles = p.n_tiles; a.cols = (int)cols; a.packs = p.packs;
  return launch(p, a, stream);
}

int tt_gate_residual_forward(void* out, const void* x, const void* gate, const void* residual,
                             int64_t rows, int64_t cols, int64_t rows_per_batch, void* stream) {
  return tt_gate_residual_forward_strided(out, x, gate, cols, nullptr, residual, rows, cols, rows_per_batch, stream);
}

size_t tt_gate_residual_backward_workspace_bytes(int64_t rows, int64_t cols, int64_t rows_per_batch) {
  return cols % kPack == 0 ? workspace_for(kGateKind, 1, rows, cols, rows_per_batch) : 0;
}

int tt_gate_residual_backward_typed(void* dresidual, void* dgate, int grads_bf16, const void* dout, const void* gate,
                                    const void* residual, void* workspace, size_t workspace_bytes,
                                    int64_t rows, int64_t cols, int64_t rows_per_batch, void* stream) {
  if (rows == 0) return TT_OK;
  if (!dresidual || !dgate || !dout || !gate || !residual) return TT_ERR_INVALID_ARGUMENT;
  if (!vector_path(cols, {dresidual, dout, gate, residual})) return TT_ERR_UNSUPPORTED;
  Plan p;
  int rc = make_plan(kGateKind, kBwd, rows, cols, rows_per_batch, &p);
  if (rc != TT_OK) return rc;
  if (!workspace || !aligned16(workspace) || workspace_bytes < partial_bytes(p, 1, cols)) return TT_ERR_WORKSPACE;
  GateArgs a;
  a.out = dresidual; a.a = dout; a.b = residual; a.gate = gate; a.partials = static_cast<float*>(workspace);
  a.gate_stride = cols; a.gate_copy = nullptr;
  a.rows_per_batch = rows_per_batch; a.n_tiles = p.n_tiles; a.cols = (int)cols; a.packs = p.packs;
  rc = launch(p, a, stream);
  if (rc != TT_OK) return rc;
  return reduce(dgate, nullptr, workspace, (int)(rows / rows_per_batch), p.grid(), 1, cols, grads_bf16 != 0, stream);
}

int tt_gate_residual_backward(void* dresidual, float* dgate, const void* dout, const void* gate,
                              const void* residual, void* workspace, size_t workspace_bytes,
                              int64_t rows, int64_t cols, int64_t rows_per_batch, void* stream) {
  return tt_gate_residual_backward_typed(dresidual, dgate, 0, dout, gate, residual, workspace, workspace_bytes,
                                         rows, cols, rows_per_batch, stream);
}

// ---------------------------------------------------------------- residual update + LayerNorm
// scale / shift / gate hold either one vector for all batches or one per batch.
static bool stride_ok(int64_t n_vectors, int64_t n_batches) { return n_vectors == 1 || n_vectors == n_batches; }

int tt_residual_norm_forward_strided(void* s, void* y, const void* x, const void* r,
                                     const void* gate, int64_t n_gate, int64_t gate_stride, void* gate_copy,
                                     const void* scale, int64_t scale_stride, void* scale_copy,
                                     const void* shift, int64_t shift_stride, int64_t n_param, int affine,
                                     float* mean, float* rstd, int64_t rows, int64_t cols, int64_t rows_per_batch,
                                     float eps, void* stream) {
  if (rows == 0) return TT_OK;
  if (!s || !y || !x || !r || !scale || !shift) return TT_ERR_INVALID_ARGUMENT;
  if (gate_stride < 0 || scale_stride < 0 || shift_stride < 0) return TT_ERR_INVALID_ARGUMENT;
  if (!vector_path(cols, {s, y, x, r, gate, scale, shift, gate_copy, scale_copy}) ||
      (gate_stride | scale_stride | shift_stride) % kPack != 0)
    return TT_ERR_UNSUPPORTED;
  Plan p;
  int rc = make_plan(kAdaLN, kFwd, rows, cols, rows_per_batch, &p, false, gate ? 2 : 1);
  if (rc != TT_OK) return rc;
  if (!stride_ok(n_param, p.n_batches) || (gate && !stride_ok(n_gate, p.n_batches))) return TT_ERR_INVALID_ARGUMENT;
  ResFwdArgs a;
  a.s = s; a.y = y; a.x = x; a.r = r; a.gate = gate; a.scale = scale; a.shift = shift; a.mean = mean; a.rstd = rstd;
  a.rows_per_batch = rows_per_batch; a.n_tiles = p.n_tiles;
  a.gate_stride = n_gate == 1 ? 0 : gate_stride; a.gate_copy = gate_copy; a.scale_copy = scale_copy;
  a.gate_copy_stride = n_gate == 1 ? 0 : cols; a.scale_copy_stride = n_param == 1 ? 0 : cols;
  a.scale_stride = n_param == 1 ? 0 : scale_stride; a.shift_stride = n_param == 1 ? 0 : shift_stride;
  a.cols = (int)cols; a.packs = p.packs; a.eps = eps; a.inv_cols = 1.0f / (float)cols; a.one = affine ? 0.f : 1.f;
  return launch(p, a, stream);
}

int tt_residual_norm_forward(void* s, void* y, const void* x, const void* r, const void* gate, int64_t n_gate,
                             const void* scale, const void* shift, int64_t n_param, int affine,
                             float* mean, float* rstd, int64_t rows, int64_t cols, int64_t rows_per_batch,
                             float eps, void* stream) {
  return tt_residual_norm_forward_strided(s, y, x, r, gate, n_gate, cols, nullptr, scale, cols, nullptr, shift, cols,
                                          n_param, affine, mean, rstd, rows, cols, rows_per_batch, eps, stream);
}

size_t tt_residual_norm_backward_workspace_bytes(int64_t rows, int64_t cols, int64_t rows_per_batch, int gated) {
  if (rows <= 0 || cols <= 0 || cols % kPack != 0) return 0;
  Plan p;
  if (make_plan(kAdaLN, kBwd, rows, cols, rows_per_batch, &p, false, gated ? 2 : 1) != TT_OK) return 0;
  if (g_wgs_per_cu_override.load() > 0 || g_grid_override.load() > 0)
    return workspace_bound(gated ? 3 : 2, rows, cols, rows_per_batch);
  const size_t need = partial_bytes(p, gated ? 3 : 2, cols);
  return need < 16 ? 16 : need;
}

int tt_residual_norm_backward_typed(void* dx, void* dr, void* dscale, void* dshift, void* dgate, int grads_bf16,
                              const void* dy, const void* ds_in, const void* s, const void* r,
                              const void* gate, int64_t n_gate, const void* scale, int64_t n_param, int affine,
                              void* workspace, size_t workspace_bytes,
                              int64_t rows, int64_t cols, int64_t rows_per_batch, float eps, void* stream) {
  if (rows == 0) return TT_OK;
  const bool gated = gate != nullptr;
  if (!dx || !dscale || !dshift || !dy || !s || !scale) return TT_ERR_INVALID_ARGUMENT;
  if (gated && (!dr || !dgate || !r)) return TT_ERR_INVALID_ARGUMENT;
  if (!vector_path(cols, {dx, dr, dy, ds_in, s, r, gate, scale})) return TT_ERR_UNSUPPORTED;
  Plan p;
  int rc = make_plan(kAdaLN, kBwd, rows, cols, rows_per_batch, &p, false, gated ? 2 : 1);
  if (rc != TT_OK) return rc;
  if (!stride_ok(n_param, p.n_batches) || (gated && !stride_ok(n_gate, p.n_batches))) return TT_ERR_INVALID_ARGUMENT;
  const int n_acc = gated ? 3 : 2;
  if (!workspace || !aligned16(workspace) || workspace_bytes < partial_bytes(p, n_acc, cols)) return TT_ERR_WORKSPACE;
  ResBwdArgs a;
  a.dx = dx; a.dr = dr; a.dy = dy; a.ds_in = ds_in; a.s = s; a.r = r; a.gate = gate; a.scale = scale;
  a.partials = static_cast<float*>(workspace);
  a.rows_per_batch = rows_per_batch; a.n_tiles = p.n_tiles;
  a.gate_stride = n_gate == 1 ? 0 : cols; a.param_stride = n_param == 1 ? 0 : cols;
  a.cols = (int)cols; a.packs = p.packs; a.eps = eps; a.inv_cols = 1.0f / (float)cols; a.one = affine ? 0.f : 1.f;
  rc = launch(p, a, stream);
  if (rc != TT_OK) return rc;
  return reduce(dscale, dshift, workspace, (int)p.n_batches, p.grid(), n_acc, cols, grads_bf16 != 0, stream, dgate);
}

int tt_residual_norm_backward(void* dx, void* dr, float* dscale, float* dshift, float* dgate,
                              const void* dy, const void* ds_in, const void* s, const void* r,
                              const void* gate, int64_t n_gate, const void* scale, int64_t n_param, int affine,
                              void* workspace, size_t workspace_bytes,
                              int64_t rows, int64_t cols, int64_t rows_per_batch, float eps, void* stream) {
  return tt_residual_norm_backward_typed(dx, dr, dscale, dshift, dgate, 0, dy, ds_in, s, r, gate, n_gate, scale, n_param,
                                         affine, workspace, workspace_bytes, rows, cols, rows_per_batch, eps, stream);
}

// ---------------------------------------------------------------- bare streaming probe
int tt_stream_probe(void* out, const void* a, const void* b, size_t bytes, void* stream) {
  if (bytes == 0) return TT_OK;
  if ((!out && !a) || (b && (!out || !a))) return TT_ERR_INVALID_ARGUMENT;
  if (bytes % 16 != 0 || !aligned16(out) || !aligned16(a) || !aligned16(b)) return TT_ERR_UNSUPPORTED;
  int cus = 0;
  const int rc = current_device_cus(&cus);
  if (rc != TT_OK) return rc;
  const size_t n = bytes / 16;
  // One workgroup per CU; threads and packs per lane in flight are what streamed fastest for each
  // mix on MI355X (reads want many requests in flight, writes few: 4 waves with one store each).
  const int threads = !a ? 256 : kProbeMaxThreads;
  const size_t want = (n + threads - 1) / threads;
  // two reads per write stream best with one CU in 32 left without a workgroup, like the kernels
  const size_t wgs = (b && cus >= 32) ? (size_t)(cus - cus / 32) : (size_t)cus;
  const dim3 grid((unsigned)(want < wgs ? want : wgs));
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (!out)    hipLaunchKernelGGL((stream_probe<kProbeRead, 4>), grid, dim3(threads), 0, s, out, a, b, n);
  else if (!a) hipLaunchKernelGGL((stream_probe<kProbeWrite, 1>), grid, dim3(threads), 0, s, out, a, b, n);
  else if (b)  hipLaunchKernelGGL((stream_probe<kProbeXor, 1>), grid, dim3(threads), 0, s, out, a, b, n);
  else         hipLaunchKernelGGL((stream_probe<kProbeCopy, 2>), grid, dim3(threads), 0, s, out, a, b, n);
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? TT_OK : hip_fail(e);
}

int tt_stream_probe_two_outputs(void* out0, void* out1, const void* a, size_t bytes, void* stream) {
  if (bytes == 0) return TT_OK;
  if (!out0 || !out1 || !a) return TT_ERR_INVALID_ARGUMENT;
  if (bytes % 16 != 0 || !aligned16(out0) || !aligned16(out1) || !aligned16(a)) return TT_ERR_UNSUPPORTED;
  int cus = 0;
  const int rc = current_device_cus(&cus);
  if (rc != TT_OK) return rc;
  // four waves per CU with four packs per lane in flight streamed this mix fastest on MI355X
  constexpr int kThreads = 256, kU = 4;
  const size_t n = bytes / 16;
  const size_t tiles = (n + kThreads * kU - 1) / (kThreads * kU);
  const dim3 grid((unsigned)(tiles < (size_t)cus ? tiles : (size_t)cus));
  hipLaunchKernelGGL((stream_probe_two_outputs<kU>), grid, dim3(kThreads), 0, static_cast<hipStream_t>(stream),
                     out0, out1, a, n);
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? TT_OK : hip_fail(e);
}

// ---------------------------------------------------------------- reference-compatible contract
int tt_launch_adaln_forward(void* output, void* x_norm, const void* input, const void* scale, const void* shift,
                            int64_t rows, int64_t cols, double epsilon, float* inv_variance, void* stream) {
  if (rows != 0 && (!x_norm || !inv_variance)) return TT_ERR_INVALID_ARGUMENT;
  return forward(kAdaLN, output, input, scale, shift, nullptr, inv_variance, x_norm, rows, cols, rows,
                 static_cast<float>(epsilon), stream);
}

int tt_launch_adaln_backward(void* dinp, void* dscale, void* dshift, const void* dout, const void* x_norm,
                             const void* scale, const float* inv_variance, int64_t rows, int64_t cols,
                             void* workspace, size_t workspace_bytes, void* stream) {
  if (rows == 0) return TT_OK;
  if (!dscale || !dshift) return TT_ERR_INVALID_ARGUMENT;
  int n_partials = 0;
  int rc = backward_saved_partials(kAdaLN, dinp, dout, x_norm, scale, inv_variance, workspace, workspace_bytes,
                                   &n_partials, rows, cols, stream);
  if (rc != TT_OK) return rc;
  return reduce(dscale, dshift, workspace, 1, n_partials, 2, cols, true, stream);
}

int tt_launch_rms_forward(void* output, const void* input, const void* weight, int64_t rows, int64_t cols,
                          double epsilon, float* inv_variance, void* stream) {
  if (rows != 0 && !inv_variance) return TT_ERR_INVALID_ARGUMENT;
  return forward(kRMS, output, input, weight, nullptr, nullptr, inv_variance, nullptr, rows, cols, rows,
                 static_cast<float>(epsilon), stream);
}

int tt_launch_rms_backward(void* dinp, void* dweight, const void* dout, const void* x_rmsnorm, const void* weight,
                           const float* inv_variance, int64_t rows, int64_t cols,
                           void* workspace, size_t workspace_bytes, void* stream) {
  if (rows == 0) return TT_OK;
  if (!dweight) return TT_ERR_INVALID_ARGUMENT;
  int n_partials = 0;
  int rc = backward_saved_partials(kRMS, dinp, dout, x_rmsnorm, weight, inv_variance, workspace, workspace_bytes,
                                   &n_partials, rows, cols, stream);
  if (rc != TT_OK) return rc;
  return reduce(dweight, nullptr, workspace, 1, n_partials, 1, cols, true, stream);
}

}  // extern "C"
