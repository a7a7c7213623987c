// The C ABI of the kernel library (include/pml_hip.h): device set-up, memory,
// streams and the dispatch / invoke pairs that select a tiling once and launch
// it many times.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <atomic>
#include <chrono>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <mutex>
#include <string>
#include <thread>
#include <vector>

#include "device_common.h"
#include "plans.h"

namespace pml {
namespace {

thread_local std::string g_err;

int fail(const std::string& msg) {
  g_err = msg;
  return 1;
}
int check(hipError_t e, const char* what) {
  if (e == hipSuccess) return 0;
  g_err = std::string(what) + ": " + hipGetErrorString(e);
  (void)hipGetLastError();  // (reported here, and not again by the launch that comes next)
  return 1;
}

int device_cus();

// Device memory that a caller can do without: nullptr when there is none.
void* alloc_or_null(size_t bytes) {
  void* p = nullptr;
  if (hipMalloc(&p, bytes) == hipSuccess) return p;
  (void)hipGetLastError();
  return nullptr;
}

enum PlanKind { PLAN_GEMM = 1, PLAN_CONV, PLAN_DWCONV, PLAN_POOL, PLAN_ELTWISE, PLAN_CONTRACT, PLAN_PRODUCT, PLAN_CONV_GRAD };

struct DirectTiles {
  int rows = -1, given = -1;
};

struct Plan {
  int kind = 0;
  int mfma_kind = 0;
  int tile = 0;
  pml_hip_gemm_desc gemm;
  pml_hip_conv2d_desc conv;
  pml_hip_dwconv2d_desc dw;
  pml_hip_pool2d_desc pool;
  pml_hip_eltwise_desc elt;
  pml_hip_contract_desc con;
  // packed right-hand side Bt[N][K]
  void* bt = nullptr;
  int64_t bt_ld = 0;
  size_t bt_bytes = 0;
  bool packed = false;
  bool b_split = false;  // split fp32 kind: a right-hand side packed once is kept as bf16 heads + remainders
  std::atomic<bool> bt_is_split{false};  // ... and `bt` holds that form now (an invoke that turns its own right-hand side into `bt` clears it)
  // large tiles that take B[K][N] as it lies (given.hip) keep a packed right-hand side in that form, rows of n elements
  bool b_kn = false;
  std::atomic<bool> bt_is_kn{false};  // ... and `bt` holds it now (as above)
  // second product of a GEMM: its packed right-hand side Bt2[N][K2]
  void* bt2 = nullptr;
  bool packed2 = false;
  // convolution whose channels do not fill 16-byte vectors: patch matrix [M][kpad] + GEMM
  void* patches = nullptr;
  int64_t kpad = 0;
  // stride-2 convolution over few channels, run as a unit-stride one over 2x2 pixel blocks: the
  // re-blocked input [N][s2d_h][s2d_w][s2d_ch]; filter taps s2d_ka x s2d_kaw blocks
  // (allocated by the first invoke that needs it: the row-walking stem kernel builds its blocks from the image)
  bool via_s2d = false;
  void* s2d = nullptr;
  std::mutex s2d_mutex;
  int s2d_h = 0, s2d_w = 0, s2d_ch = 0, s2d_ka = 0, s2d_kaw = 0;
  // depthwise convolution: a constant filter kept by the plan ([kh][kw][c] as the caller holds it), and its paired
  // form for the 3x3 bf16 kernel when every weight is finite
  void* dw_filter = nullptr;
  void* dw_paired = nullptr;
  // K split over workgroups: workspace of partial tiles and how the slabs are shared out (splits < 2: no split)
  void* ws = nullptr;
  int sk_splits = 0, sk_per = 0, sk_pitch = 0;
  // the direct tiles a product takes instead of `tile`, and the one a convolution takes (-1: none)
  DirectTiles direct;
  int tile_direct = -1;
  int tile_given = -1;  // ... and over a filter that comes with the call, as it lies
  // a convolution that runs over its window in LDS (`bt` holds the filter as that kernel multiplies it)
  WinShape win;
  // a product that runs in panels once its right-hand sides are packed: the configuration (-1: it does not) and their fragments
  int panel = -1;
  void* panel_bt = nullptr;
  bool panel_fresh[2] = {false, false};  // they hold what `bt` holds; what `bt2` holds
  // register-filter convolution: a filter packed once, in the order the kernel holds it in registers
  void* reg_image = nullptr;
  // product over free strides, and a convolution's gradients built on it: the prepared arguments (workspace in `ws`),
  // element kind, tile; a data gradient of unit stride is a convolution of the gradient (`sub`, its channels padded to
  // whole 16-byte vectors in `padded`), one of a larger stride a product into `cols`, images `grad_chunk` at a time
  StridedArgs strided;
  bool strided_bf = false, strided_conv = false;
  int strided_mi = 1, grad_which = 0, product_rows = 0;
  Plan* sub = nullptr;
  void *padded = nullptr, *cols = nullptr;
  int64_t co_pad = 0, grad_chunk = 0;
  // resident-filter convolution: LDS bytes (0 = not used), window rows, tile count, CUs of the device
  size_t halo_lds = 0;
  int halo_rows = 0, halo_tiles = 0, halo_variant = 0, n_cus = 0;
  std::string text;
  std::atomic<size_t> held{0};  // bytes of device memory in all of the above
  void* hold(size_t bytes) {
    void* mem = alloc_or_null(bytes);
    if (mem) held += bytes;
    return mem;
  }
  void drop(void** mem, size_t bytes) {
    if (*mem) {
      (void)hipFree(*mem);
      held -= bytes;
    }
    *mem = nullptr;
  }
  ~Plan() {
    if (bt) (void)hipFree(bt);
    if (bt2) (void)hipFree(bt2);
    if (panel_bt) (void)hipFree(panel_bt);
    if (patches) (void)hipFree(patches);
    if (s2d) (void)hipFree(s2d);
    if (reg_image) (void)hipFree(reg_image);
    if (ws) (void)hipFree(ws);
    if (dw_filter) (void)hipFree(dw_filter);
    if (dw_paired) (void)hipFree(dw_paired);
    if (padded) (void)hipFree(padded);
    if (cols) (void)hipFree(cols);
    delete sub;
  }
};

int mfma_kind_of(int in_dtype, int flags = 0) {
  switch (in_dtype) {
    case PML_HIP_F32: return (flags & PML_HIP_FP32_AS_BF16X3) ? KIND_F32X3 : KIND_F32;
    case PML_HIP_BF16: return KIND_BF16;
    case PML_HIP_I8: return KIND_I8;
  }
  return -1;
}

const char* const kFilterLies = ", with the filter as it lies tile=";
const char* tile_name(int t) {
  switch (t) {
    case TILE_64x64: return "64x64";
    case TILE_128x64: return "128x64";
    case TILE_128x128: return "128x128";
    case TILE_128x64_W8: return "128x64 (8 wavefronts)";
    case TILE_128x128_W8: return "128x128 (8 wavefronts)";
    case TILE_256x128_W16: return "256x128 (16 wavefronts)";
    case TILE_64x64_W8_K2: return "64x64 (8 wavefronts, K split in two)";
    case TILE_256x256_W8: return "256x256 (8 wavefronts of 128x64)";
    case TILE_128x64_N2: return "128x64 (4 wavefronts of 32x64)";
    case TILE_128x128_W8_S2: return "128x128 (8 wavefronts, 2 stages)";
    case TILE_192x384_W8: return "192x384 (8 wavefronts of 96x96)";
    case TILE_64x64_KSPLIT: return "64x64, K split over workgroups";
    case TILE_16x16_W8: return "16x16 (8 wavefronts sharing K)";
    case TILE_32x32_W8: return "32x32 (8 wavefronts sharing K)";
  }
  return "?";
}

constexpr int kScheduleBits = 0xff << 8 | 0xf << 16;
constexpr int kMaxpoolBits = 0x1f << 20;
bool schedule_bits_ok(int flags) {
  return PML_HIP_FLAG_TILE_OF(flags) < PML_HIP_TILE_COUNT_ && PML_HIP_FLAG_CONV_OF(flags) <= PML_HIP_CONV_WINDOW;
}
const char* const kTileShort[PML_HIP_TILE_COUNT_] = {"64x64", "128x64", "128x128", "128x64w8", "128x128w8", "256x128w16", "128x128w8s2", "64x64w8k2", "256x256w8", "128x64n2", "192x384w8", "64x64ks", "16x16w8", "32x32w8"};

// Whether the K loop of 64 x 64 tiles is shared out among workgroups (TILE_64x64_KSPLIT).  Few tiles and a long K: always.
// Up to five eighths of a round of tiles it is where the chain is long enough to pay for the second launch, for bf16 and the
// split fp32 kind: bf16 40 x 20 x 20 x 96 (*) 7 x 7 x 96 stride 2, 126 tiles of 74 slabs, 29.8 -> 20.5 us; 593 x 606, K = 3808
// 28.9 -> 17.5; 900 x 512, K = 2992 24.0 -> 17.4; but 700 x 600, K = 2048 11.2, 13.9 split (the operands of the longer ones
// are past an L2's 4 MB).  fp32 as three products 1210 x 511, K = 2832 41.1 -> 35.6.  fp32 takes direct tiles there, or is
// slower split (725 x 364, K = 880: 13.1, 17.3).
bool splits_k(int64_t m, int64_t n, int64_t k_bytes, int kind) {
  const int64_t t = ((m + 63) / 64) * ((n + 63) / 64);
  if (k_bytes < 2048) return false;
  return t <= 64 || (t <= 160 && ((kind == KIND_BF16 && k_bytes >= 5632) || (kind == KIND_F32X3 && k_bytes >= 8192)));
}

// Microseconds per 128-byte slab of K of an fp32 product in tiles through LDS: 0.58 per round of 64 x 64 tiles, or as much less per
// result in 128 x 128 tiles as those fill their rounds better.  fp32 is bound by its MFMAs, and tiles of 128 gain 5 % at best
// (3881 x 3959, K = 2992 723 us, 760 in tiles of 64; 2381 x 1595, K = 2608 171, 180), while half a round of them more costs as much as
// two of 64: 3271 x 547, K = 448 36.2 -> 21.6, 2322 x 2041, K = 304 47.7 -> 35.4, 1246 x 4028, K = 208 35.6 -> 27.1, convolutions
// 38400 x 122, K = 2304 294 -> 209, 13689 x 179, K = 3200 212 -> 168.
// (One slab is tail more than MFMAs, and two tiles of 128 share a CU: there a last round more than half full is no whole one.
// 7295 x 944, K = 12 13.1, in tiles of 64 14.1, 4690 x 1308, K = 28 13.1, 13.7; with a smaller share of both grids for edges alike.)
bool f32_tiles_of_128(int64_t m, int64_t n, int64_t k_bytes) {
  const int64_t cus = device_cus(), t128 = ((m + 127) / 128) * ((n + 127) / 128), t64 = ((m + 63) / 64) * ((n + 63) / 64);
  if (k_bytes <= 128 && t128 >= cus && 2 * (t128 % cus) >= cus && 10 * t64 >= 37 * t128) return true;
  return t128 >= 128 && 4 * ((t128 + cus - 1) / cus) <= (t64 + cus - 1) / cus;
}
double f32_slab_us(int64_t m, int64_t n, int64_t k_bytes) {
  const int64_t cus = device_cus(), t128 = ((m + 127) / 128) * ((n + 127) / 128), t64 = ((m + 63) / 64) * ((n + 63) / 64);
  return f32_tiles_of_128(m, n, k_bytes) ? 2.2 * (double)((t128 + cus - 1) / cus) : 0.58 * (double)((t64 + cus - 1) / cus);
}

// One of the direct tiles (direct.hip) where it beats the LDS kernels, or -1.  Both sides are priced in microseconds, from
// measurements of 27 matrix products and 18 convolutions per element kind (one row to 3136, K of 64 to 4608; back to back
// in a recorded graph): a direct kernel takes 2.6 plus, per round of one tile on each CU (fp32 and 32 x 64: whole
// rounds), 0.8 (fp32 32 x 32: 1.9; 32 x 64, which replaces 32 x 32 beyond one round: bf16 1.6, int8 1.0, fp32 2.3) and its
// operand bytes at 40 KB a microsecond and CU (32 x 64: bf16 50, int8 60, fp32, all 64 columns of a tile, 35, of several rounds 42).  An LDS kernel takes 4.2 plus its chain
// of 128-byte slabs (0.23 each, int8 0.28, fp32 `f32_slab_us`), or -- K split over workgroups -- 5.2 plus 0.4 per KB of K
// (more than 64 tiles: 0.5 per slab of a split; fp32: 8.5 and 0.68 per slab of a split) plus writing and reading the partial tiles at 3 TB/s.  The prices meet the measurements to about 15 %; a direct tile has
// to be 5 % ahead.
//   us, before -> direct                       bf16              fp32              int8
//   1 x 1000, K = 2048                     7.4 ->  5.0       9.3 ->  7.3       6.7 ->  4.3
//   196 x 256, K = 1024                    7.5 ->  5.2       9.7 ->  6.5       6.4 ->  4.4
//   784 x 512, K = 256: 32 x 64            5.1 ( 5.4)       9.6 ->  8.5       4.8 ->  4.5
//   28 x 28 x 128 (*) 3 x 3 x 128          9.1 ->  7.7      11.1 (12.8)        7.4 ->  5.2
//   49 x 512, K = 4608: stays split        8.6 (11.2)       12.9 (18.7)        7.6 ( 7.4)
// and of fp32 where tiles through LDS are priced by their rounds and a split by its slabs, as 120 products and convolutions with 5e7
// multiply-adds and more were timed: 251 x 658, K = 848 [K][N] 18.7 -> 8.2, 836 x 2331, K = 592 46.2 -> 32.6, 214 x 271, K = 3632 17.0 -> 12.5,
// convolutions 38 x 23 x 23 x 256 (*) 3 x 3 x 39 91.6 -> 67.0, 13 x 25 x 25 x 32 (*) 3 x 3 x 139 28.1 -> 17.0.
// A right-hand side that arrives with the call as [K][N]: tiles are then 16 or 32 x 64 (60 KB a microsecond; fp32 45,
// int8 36 unless rows are whole 64-byte runs), and an LDS kernel that needs Bt pays for the transposed copy besides, 3 and
// its bytes both ways at 2.2 TB/s:
// bf16 512 x 512 x 512 9.4 -> 5.0, 1024^3 14.6 -> 10.6, 64 x 2048 x 2048 16.5 -> 8.8; fp32 128 x 4096 x 1024 23.4 -> 12.3.
// kn_ldb: that right-hand side's row pitch in bytes (0: Bt); always: the better of the two whatever the LDS kernel takes;
// can_split: the LDS kernel may split K; lds: what an LDS kernel takes; as_given: it reads a [K][N] right-hand side as it lies (256 x 49152, K = 4096 bf16:
// 409 us direct, 135 with 256 x 256 tiles; charged the copy of 800 MB, they lost)
int direct_tile_of(int64_t m, int64_t n, int64_t k_bytes, int kind, int64_t kn_ldb = 0, bool always = false, bool can_split = true, bool as_given = false, double* us = nullptr, double* lds = nullptr) {
  if (kind != KIND_F32 && kind != KIND_BF16 && kind != KIND_I8) return -1;
  auto tiles = [&](int64_t bm, int64_t bn) { return ((m + bm - 1) / bm) * ((n + bn - 1) / bn); };
  const double kb = (double)k_bytes;
  const int es = kind == KIND_BF16 ? 2 : (kind == KIND_I8 ? 1 : 4);
  const bool kn = kn_ldb > 0, f32 = kind == KIND_F32;
  const int n_cus = device_cus();
  const bool wide_tiles = !kn && tiles(32, 32) > n_cus;  // (32 x 64 in the place of 32 x 32)
  const double rate = !kn ? 40e3 : f32 ? 45e3 : (kind == KIND_I8 && kn_ldb % 64 != 0) ? 36e3 : 60e3;
  auto direct_us = [&](int64_t side) {
    const bool w = wide_tiles && side == 32;
    const int64_t wide = kn || w ? 64 : side;
    double rounds = std::max(1.0, (double)tiles(side, wide) / n_cus);
    if ((f32 && !kn) || w) rounds = std::ceil(rounds);
    // (fp32 in many rounds of 16 x 16: convolution 32368 x 11, K = 1152, eight of them, 42.4)
    const double start = w ? (f32 ? 2.3 : kind == KIND_I8 ? 1.0 : 1.6) : f32 && !kn ? (side == 32 ? 1.9 : rounds > 4 ? 1.7 : 0.8) : 0.8;
    const double r = w ? (f32 ? (rounds > 1 ? 42e3 : 35e3) : kind == KIND_I8 ? 60e3 : 50e3) : rate;
    return 2.6 + rounds * (start + (double)(std::min(m, side) + (f32 && w ? wide : std::min(n, wide))) * kb / r);
  };
  const int64_t slabs = (k_bytes + 127) / 128;
  double lds_us = 4.2 + (f32 ? f32_slab_us(m, n, k_bytes) : kind == KIND_I8 ? 0.28 : 0.23) * (double)slabs;
  bool needs_bt = !as_given && (kind == KIND_BF16 || n % (16 / es) != 0 || kn_ldb % 16 != 0);
  if (can_split && splits_k(m, n, k_bytes, kind)) {
    int splits = 1, per = 0;
    igemm_split_plan(m, n, slabs, n_cus, &splits, &per);
    if (splits >= 2) {
      lds_us = (f32 ? 8.5 + 0.68 * (double)per : 5.2 + (tiles(64, 64) <= 64 ? kb / 2500 : 0.5 * (double)per)) + 8.0 * splits * (double)m * (double)n / 3e6;
      needs_bt = true;
    }
  }
  if (kn && needs_bt) lds_us += 3.0 + 2.0 * kb * (double)n / 2.2e6;
  const double small = direct_us(16), large = direct_us(32);
  const bool direct = always || std::min(small, large) <= 0.95 * lds_us;
  if (us) *us = direct ? std::min(small, large) : lds_us;
  if (lds) *lds = lds_us;
  if (!direct) return -1;
  return small <= large ? TILE_16x16_W8 : TILE_32x32_W8;
}

// Microseconds of a 16 or 32 x 64 direct tile over a right-hand side [K][N] as it lies, from 260 timings of 130 convolutions (8 to
// 13 % rms): 2.6, and per round of one tile on each CU (a last one that is not full counts for most of one) a start and so much per
// KB of K -- not per byte of few columns: it is the requests for K-rows that take the time, more of them for int8, whose rows off a
// word take two words each.  (int8 on a word, but not in whole 16 bytes: 400 x 12, K = 3136 10.4, 864 x 24, K = 2000 7.6, 300 x 92, K = 1600 7.2; in whole ones
// 441 x 16, K = 3200 7.0, 256 x 208, K = 2400 5.9.)
double direct_lies_us(int64_t m, int64_t n, int64_t k_bytes, int kind, int side) {
  const bool small = side == 16, odd = n % 4 != 0;
  double start, per_kb;
  if (kind == KIND_BF16) start = small ? 1.35 : 1.7, per_kb = small ? 1.17 : 1.52;
  else if (kind == KIND_I8) start = small ? 1.3 : 1.6, per_kb = n % 16 == 0 ? 1.2 : !odd ? 2.3 : small ? 2.05 : 2.45;
  else start = small ? 2.2 : 1.7, per_kb = small ? 1.2 : 2.3;
  const double rounds = std::max(1.0, (double)((m + side - 1) / side) * (double)((n + 63) / 64) / device_cus());
  return 2.6 + (0.75 * std::ceil(rounds) + 0.25 * rounds) * (start + per_kb * (double)k_bytes / 1024);
}

// Whether a product that may be taken as three bf16 products is better off in a direct tile of plain fp32 MFMAs: the split kind
// has no direct tiles, and with few results it is latency that bounds both.  Its tiles take 4.2 us and 0.42 per slab, or split as
// `direct_tile_of` says.  Decided by the sizes alone, so that a product has the same bits from [K][N] as it lies, packed and from
// [N][K]: the direct tiles have to be cheaper over rows of K and over [K][N].  us, split -> direct: 1 x 1724, K = 656 packed 9.4 -> 4.9,
// 7 x 1293, K = 208 [N][K] 6.9 -> 5.3, 16 x 26, K = 416 [K][N] 12.8 -> 6.1, 382 x 253, K = 336 packed 9.7 -> 6.7; but 2 x 22, K = 3104
// [K][N] 15.1 (18.7), 672 x 491, K = 800 packed 12.0 (14.2).  Of 100 drawn products 54 are cheaper over the layout that they have.
bool fp32_beats_split(int64_t m, int64_t n, int64_t k_bytes) {
  const int64_t slabs = (k_bytes + 127) / 128;
  double us = 0, split_us = 4.2 + 0.42 * (double)slabs;
  bool needs_bt = n % 4 != 0;  // (from [K][N]: a transposed copy)
  if (splits_k(m, n, k_bytes, KIND_F32X3)) {
    int splits = 1, per = 0;
    igemm_split_plan(m, n, slabs, device_cus(), &splits, &per);
    if (splits >= 2) {
      split_us = 5.2 + (((m + 63) / 64) * ((n + 63) / 64) <= 64 ? (double)k_bytes / 2500 : 0.5 * (double)per) + 8.0 * splits * (double)m * (double)n / 3e6;
      needs_bt = true;
    }
  }
  if (direct_tile_of(m, n, k_bytes, KIND_F32) < 0) return false;
  // (two rounds of 16 x 16 tiles over few K take longer than that price: 29 x 3872, K = 96 [N][K] 5.2, direct 6.0; odd columns,
  // which the split's tail stores one by one, do not: 191 x 381, K = 64 6.0, direct 5.0)
  if (direct_tile_of(m, n, k_bytes, KIND_F32, 0, /*always=*/true, true, false, &us) == TILE_16x16_W8 && ((m + 15) / 16) * ((n + 15) / 16) > device_cus() && !needs_bt) us += 0.7;
  const double copy = needs_bt ? 3.0 + 2.0 * (double)k_bytes * (double)n / 2.2e6 : 0;
  // (16 x 64 tiles of one round take fewer steps in flight where they have few: 2.6 + 1.3 + 1.25 per KB of K, to 10 %)
  const bool one_round = ((m + 15) / 16) * ((n + 63) / 64) <= device_cus();
  const double small = one_round ? 3.9 + 1.25 * (double)k_bytes / 1024 : direct_lies_us(m, n, k_bytes, KIND_F32, 16);
  return us <= 0.95 * split_us && std::min(small, direct_lies_us(m, n, k_bytes, KIND_F32, 32)) <= 0.95 * (split_us + copy);
}

// What of a tail decides between tiles.
struct TailForm {
  bool plain;             // leaves a 256 x 256 tile in one go
  bool bare = false;      // one product, and start values, ReLU and requantisation at most
  bool residual = false;  // + a whole tensor, ReLU
  bool two = false;       // a second product, with start values of its own
  bool steps = false;     // steps on column vectors and single values: scale and shift
};

// Stated tiling choice per shape class.  Measured on MI355X, bf16 unless said otherwise (us; w8 / w16 =
// 8 / 16 wavefronts per workgroup; s2 = two ring stages and LDS cut to what the result tile needs, so that two
// workgroups share a CU; the 4-wavefront 256x128 and 256x256 tiles that were tried as well are slower than
// 256x128w16 everywhere and are no longer built):
//                                    64x64  128x64  128x128  128x128w8  128x128w8s2  256x128w16
//   4096^3 (int8)                      137       -      119        112          121          83
//   4096^3                             198       -      173        163          115         108
//   conv 128x28x28x128 (*) 3x3x128      66      76       89         71           49          52
//   conv 128x14x14x256 (*) 3x3x256      64      72       73         61           45          45
//   conv 128x7x7x512   (*) 3x3x512      72      67       64         57           65          77
//   conv 128x56x56x256 (*) 1x1x512 /2   83     101        -         99           62          74
//   gemm 401408x256x64                  82     127      177        123           76          84
//   gemm 100352x512x128                 52      71      100         70           44          51
//   gemm 25088x256x1024                 27      27       30         24           20          22
//   gemm 6272x512x2048                  25      23       25         21           30          28
//   gemm 23104x728x728                  72      67       78         65           57          58
//   gemm 128x1000x2048                  14       -        -         19           19          25
//   gemm 1024^3 (fp32)                  33      45       77         71            -         127
// A descriptor may name its tile (PML_HIP_FLAG_TILE); every tile is tested on a ragged problem that way.
// One tile per workgroup and a serial load / multiply / store life per tile: latency is hidden by the
// other wavefronts of a SIMD -- 8 or 16 per workgroup instead of 4 -- and, for the bandwidth-bound shapes
// with a short K, by a second workgroup on the CU whose loads run under the first one's tail.  So: long K
// and at least two rounds of 256x128 tiles take that tile with 16 wavefronts; otherwise 128x128 with 8
// wavefronts, two to a CU if that still gives every CU a workgroup, one to a CU (three stages) below
// that; and for small problems the smaller of 64x64 and 128x64 by (rounds of resident workgroups) x
// (tile area), the larger tile on a tie.
// forced: a tile named by the descriptor's schedule bits (PML_HIP_FLAG_TILE), -1 = none
int choose_tile(int64_t m, int64_t n, int64_t k_bytes, int kind, const TailForm& tail, int forced = -1, bool allow_split = true) {
  if (forced >= 0 && forced < PML_HIP_TILE_COUNT_ && (forced != TILE_128x64_N2 || kind == KIND_F32X3) &&
      (forced != TILE_192x384_W8 || kind == KIND_BF16 || kind == KIND_I8))
    return forced;
  auto tiles = [&](int64_t bm, int64_t bn) { return ((m + bm - 1) / bm) * ((n + bn - 1) / bn); };
  // Few tiles and a long K (a network's last stages at batch 1: 49 x 512 x 4608 is 8 tiles of 72 slabs): the K loop is
  // shared out among workgroups and a second launch adds the partial tiles up.  Measured inside ResNet-50 at batch 1.
  if (allow_split && splits_k(m, n, k_bytes, kind)) return TILE_64x64_KSPLIT;
  if (kind == KIND_F32X3) {
    // A fragment that is split in registers costs 24 vector instructions whatever it is multiplied with, so the
    // tile a wavefront holds decides how many MFMAs share that cost -- but the problems this kind meets here are
    // short of tiles first.  Measured: 128 x 56 x 56 x 64 (*) 3 x 3 x 64 137 us with 64x64, 146 with 128x64 as 32x64 per
    // wavefront, 155 with 128x64 as 64x32; 1024^3 25-27 us with 64x64 (either form), 34-47 with larger tiles.
    if (n > 64 && tiles(128, 128) >= 512) return TILE_128x128;
    if (tiles(64, 64) <= 512 && k_bytes >= 2048) return TILE_64x64_W8_K2;
    return TILE_64x64;
  }
  if (n <= 64) return kind != KIND_F32 && tail.bare && tiles(64, 64) <= 256 ? TILE_64x64_W8_K2 : TILE_64x64;  // (the 7x7 stem of ResNet-50 over 2x2 pixel blocks: 191 us against 207 us with 128x64w8)
  // Long K, at least three quarters of a round of 256x256 tiles and little of them hanging over the edges:
  // eight wavefronts of 128x64 (0.75 KB of LDS fragment reads per MFMA instead of 1.5).  Measured with N(0,1) /
  // uniform int8 data, 4096^3: bf16 121 us against 139 (256x128, 16 wavefronts), int8 73 against 84.
  // (Not under a tail that runs in steps -- requantisation chains: a wavefront stages its 128x64 part through a
  // 16 KB share of LDS in four rounds, 4096^3 int8 with that tail 132 us against 106 with 256x128.)
  if (kind != KIND_F32 && tail.plain && k_bytes >= 2048 && tiles(256, 256) >= 192 && tiles(256, 256) * 65536 * 10 <= m * n * 11)
    return TILE_256x256_W8;
  // Eight wavefronts of 96 x 96 on a 192 x 384 tile: per MFMA half the global -> LDS bytes of a 128 x 128 tile (the vector
  // memory path moves 64 bytes per clock and CU, which 128 x 128 tiles use up entirely) and 0.67 KB of fragment reads.
  // One workgroup per CU, so its tail is not hidden by a neighbour: it pays where the K loop is most of the work, the
  // columns fill whole tiles and the tiles fill a round of the chip -- 23104 x 728 x 728 (242 tiles) 39 us against 48.
  if (kind != KIND_F32 && kind != KIND_F32X3 && k_bytes >= 1024) {
    const int64_t tn = (n + 383) / 384, t = tiles(192, 384);
    if (tn * 384 * 100 <= n * 108 && ((t >= 200 && t <= 256) || t >= 640)) return TILE_192x384_W8;
  }
  if (k_bytes >= 4096 && tiles(256, 128) >= 512) return TILE_256x128_W16;
  // One round of 256x128 tiles that fills at least three quarters of the chip, K of 2 KB and more per row, bf16: the
  // 16-wavefront tile instead of 1.53 rounds of 128x128 tiles -- 25088 x 256 results, ResNet-50's 14x14x256 layers at
  // batch 128: the 3x3 convolutions 38.9 -> 37.3 us, the 1x1 layers with K = 1024 26.7 -> 25.3, the network 2.59 -> 2.57 ms
  // (measured with a schedule file before the rule was written down).
  if (kind == KIND_BF16 && k_bytes >= 2048 && tiles(256, 128) >= 192 && tiles(256, 128) <= 256) return TILE_256x128_W16;
  // fp32: up to two 64 x 64 tiles a CU share K in two wavefront grids (1024^3 32.5 -> 28.8 us), whatever the K: of 118 products and
  // convolutions with K of less than 2 KB those of up to 256 tiles took 1.05 to 1.16 x as long in plain ones (relu 1.08, residual 1.11,
  // scale and shift 1.05), those of up to 512 1.00 to 1.07 -- but for scale and shift, 0.96 to 1.03, unless rows off 16 bytes leave
  // step by step (1.3).
  if (kind == KIND_F32 && !f32_tiles_of_128(m, n, k_bytes))
    return tiles(64, 64) <= (k_bytes < 2048 && tail.steps && n % 4 == 0 ? 256 : 512) ? TILE_64x64_W8_K2 : TILE_64x64;
  if (tiles(128, 128) >= 256) return TILE_128x128_W8_S2;
  // (two slabs and less are all launch, first loads and tail: bf16 conv 8750 x 138, K = 64 9.4 -> 6.6 us, 23958 x 105, K = 128 9.6 -> 8.1.
  // But bf16 tiles of 64 that are more than three a CU take another round for that: of 60 products and convolutions with whole 16-byte
  // rows those of up to 768 took 1.06 x as long in tiles of 128 (relu 0.96 to 1.13, scale and shift 1.01 to 1.17), those of more 0.94 x
  // (0.91 to 0.98, 0.93 to 0.99; residuals 1.02), two products 0.99 x and 0.91; int8 and rows off 16 bytes 1.0 to 1.5 x.)
  const bool short_k = k_bytes <= 256 && !tail.two && (kind == KIND_I8 || n % 8 != 0 || tail.residual || tiles(64, 64) <= 3 * 256);
  if (tiles(128, 128) >= 128 && (kind == KIND_F32 || !short_k)) return TILE_128x128_W8;
  // at most two 64x64 tiles per CU and a long K: a second wavefront grid takes half of every slab
  // (bf16 128x1000x2048: 13.4 -> 11.6 us; bf16 2048^3, 1024 tiles: 26.7 -> 40.5 us)
  // (one tile a CU: whatever the K, eight wavefronts to its loads and its tail; bf16 650 x 593, K = 720 8.7 -> 7.5 us, 915 x 588,
  // K = 224 5.9 -> 5.1, int8 2085 x 435, K = 48 5.6 -> 5.1.  Not under a residual or scale and shift, whose operands it waits for with
  // half the tiles' wavefronts on a CU: 648 x 632, K = 632 with scale, shift, ReLU in its block 16.4 us, 17.1; ResNet-50 on one image, three such layers 394.0, 395.2.
  // Nor where a second product follows, with start values of its own: 40 of them 0.96 x, 784 x 512, K = 128 + 256 in ResNet-50 1.4 us a call)
  if (tiles(64, 64) <= (k_bytes >= 2048 ? 512 : tail.bare ? 256 : 0)) return TILE_64x64_W8_K2;
  const int64_t rounds_small = (tiles(64, 64) + 5 * 256 - 1) / (5 * 256);
  const int64_t rounds_wide = (tiles(128, 64) + 2 * 256 - 1) / (2 * 256);
  return rounds_small < 2 * rounds_wide ? TILE_64x64 : TILE_128x64;
}

// A tail that is only "relu?" can use the fast store path.
void classify_tail(const pml_hip_epilogue& t, int out_dtype, int c_dtype, int* mode, int* relu) {
  *mode = 0;
  *relu = 0;
  // int32 accumulators followed by stores / casts between si32, f32, si8 / f32 arithmetic on immediates,
  // scalars and per-column vectors (requantisation): checked by walking the element type through the chain
  if (out_dtype == PML_HIP_I32 && t.n_ops >= 1 && t.n_ops <= 8) {
    int cur = PML_HIP_I32;
    bool ok = true;
    for (int i = 0; i < t.n_ops && ok; ++i) {
      const pml_hip_epi_op& op = t.ops[i];
      if (op.opcode == PML_HIP_EPI_STORE) continue;
      if (op.opcode == PML_HIP_EPI_CAST) {
        if (op.dtype != PML_HIP_F32 && op.dtype != PML_HIP_I32 && op.dtype != PML_HIP_I8) ok = false;
        if (cur == PML_HIP_I8 && op.dtype != PML_HIP_I8) ok = false;  // si8 is only ever the last type
        cur = op.dtype;
        continue;
      }
      switch (op.opcode) {
        case PML_HIP_EPI_ADD: case PML_HIP_EPI_SUB: case PML_HIP_EPI_RSUB: case PML_HIP_EPI_MUL: case PML_HIP_EPI_DIV:
        case PML_HIP_EPI_RDIV: case PML_HIP_EPI_MAX: case PML_HIP_EPI_MIN: case PML_HIP_EPI_RELU: case PML_HIP_EPI_NEG:
        case PML_HIP_EPI_MAX_GT: case PML_HIP_EPI_ROUND: case PML_HIP_EPI_FLOOR: case PML_HIP_EPI_CEIL:
          break;
        default:
          ok = false;
      }
      if (cur != PML_HIP_F32 || op.dtype != PML_HIP_F32) ok = false;
      if (op.operand_kind == PML_HIP_OPND_TENSOR) {
        const int q = op.operand;
        if (t.operand_dtype[q] != PML_HIP_F32 || t.operand_row_stride[q] != 0 ||
            (t.operand_col_stride[q] != 0 && t.operand_col_stride[q] != 1))
          ok = false;
      }
    }
    bool plain = true;  // a chain of nothing but "relu" on si32 stays with mode 1 below
    for (int i = 0; i < t.n_ops; ++i)
      if (t.ops[i].opcode != PML_HIP_EPI_RELU) plain = false;
    if (ok && !plain && cur == c_dtype) {
      *mode = 4;
      return;
    }
  }
  if (c_dtype != out_dtype) return;
  if (t.n_ops == 0) {
    *mode = 1;
    return;
  }
  if (t.n_ops == 1 && t.ops[0].opcode == PML_HIP_EPI_RELU && t.ops[0].dtype == out_dtype) {
    *mode = 1;
    *relu = 1;
    return;
  }
  // + residual (a full tensor of the result type, unit column stride, rows on 4-element boundaries), relu?
  if ((t.n_ops == 1 || t.n_ops == 2) && t.ops[0].opcode == PML_HIP_EPI_ADD && t.ops[0].operand_kind == PML_HIP_OPND_TENSOR &&
      t.ops[0].operand == 0 && t.ops[0].dtype == out_dtype && t.operand_dtype[0] == out_dtype &&
      t.operand_col_stride[0] == 1 && (t.operand_row_stride[0] & 3) == 0 &&
      (t.n_ops == 1 || (t.ops[1].opcode == PML_HIP_EPI_RELU && t.ops[1].dtype == out_dtype))) {
    *mode = 2;
    *relu = t.n_ops == 2;
    return;
  }
  // up to four float steps in the result type on immediates, scalars and per-column vectors
  if ((out_dtype == PML_HIP_F32 || out_dtype == PML_HIP_BF16) && t.n_ops >= 1 && t.n_ops <= 4) {
    bool ok = true;
    for (int i = 0; i < t.n_ops && ok; ++i) {
      const pml_hip_epi_op& op = t.ops[i];
      switch (op.opcode) {
        case PML_HIP_EPI_ADD: case PML_HIP_EPI_SUB: case PML_HIP_EPI_RSUB: case PML_HIP_EPI_MUL: case PML_HIP_EPI_DIV:
        case PML_HIP_EPI_RDIV: case PML_HIP_EPI_MAX: case PML_HIP_EPI_MIN: case PML_HIP_EPI_RELU: case PML_HIP_EPI_NEG:
        case PML_HIP_EPI_MAX_GT:
          break;
        default:
          ok = false;
      }
      if (op.dtype != out_dtype) ok = false;
      if (op.operand_kind == PML_HIP_OPND_TENSOR) {
        const int q = op.operand;
        if (t.operand_dtype[q] != out_dtype || t.operand_row_stride[q] != 0 ||
            (t.operand_col_stride[q] != 0 && t.operand_col_stride[q] != 1))
          ok = false;
      }
    }
    if (ok) *mode = 3;
  }
}

// The scale / shift (/ relu) chain of a folded batch normalisation, bf16 throughout: result * v0[col] + v1[col].
// 0: the chain is something else; 1: without relu; 2: with relu.
int tail_scale_shift(const pml_hip_epilogue& t, int out_dtype, int mode) {
  if (mode != 3 || out_dtype != PML_HIP_BF16 || (t.n_ops != 2 && t.n_ops != 3)) return 0;
  const int want[3] = {PML_HIP_EPI_MUL, PML_HIP_EPI_ADD, PML_HIP_EPI_RELU};
  for (int i = 0; i < t.n_ops; ++i) {
    const pml_hip_epi_op& op = t.ops[i];
    if (op.opcode != want[i] || op.dtype != PML_HIP_BF16) return 0;
    if (i < 2 && (op.operand_kind != PML_HIP_OPND_TENSOR || t.operand_col_stride[op.operand] != 1 || t.operand_row_stride[op.operand] != 0 ||
                  t.operand_dtype[op.operand] != PML_HIP_BF16))
      return 0;
  }
  return t.n_ops - 1;
}

// The requantisation chain of an int8 contraction: store? cast f32, mul by a per-column (or single) f32 tensor operand,
// maxgt immediate, min immediate, round, cast si8.  Fills the kernel arguments that describe it; false: something else.
bool tail_requant(const pml_hip_epilogue& t, int out_dtype, int c_dtype, int mode, IgemmArgs* g) {
  if (g) g->tail_rq = 0;
  if (mode != 4 || out_dtype != PML_HIP_I32 || c_dtype != PML_HIP_I8) return false;
  const int first = (t.n_ops > 0 && t.ops[0].opcode == PML_HIP_EPI_STORE) ? 1 : 0;
  if (t.n_ops != first + 6) return false;
  const pml_hip_epi_op* o = t.ops + first;
  const bool shape = o[0].opcode == PML_HIP_EPI_CAST && o[0].dtype == PML_HIP_F32 && o[1].opcode == PML_HIP_EPI_MUL &&
                     o[1].dtype == PML_HIP_F32 && o[1].operand_kind == PML_HIP_OPND_TENSOR && o[2].opcode == PML_HIP_EPI_MAX_GT &&
                     o[2].dtype == PML_HIP_F32 && o[2].operand_kind == PML_HIP_OPND_IMM && o[3].opcode == PML_HIP_EPI_MIN &&
                     o[3].dtype == PML_HIP_F32 && o[3].operand_kind == PML_HIP_OPND_IMM && o[4].opcode == PML_HIP_EPI_ROUND &&
                     o[4].dtype == PML_HIP_F32 && o[5].opcode == PML_HIP_EPI_CAST && o[5].dtype == PML_HIP_I8;
  if (!shape) return false;
  if (g) {
    g->tail_rq = 1;
    g->rq_store = first ? t.ops[0].operand : -1;
    g->rq_scale = o[1].operand;
    g->rq_lo = (float)o[2].imm;
    g->rq_hi = (float)o[3].imm;
  }
  return true;
}

// ... and what of a tail decides between tiles.  (A convolution's never counts as leaving a 256 x 256 tile in one go.)
TailForm tail_form(const pml_hip_epilogue& t, int out_dtype, int c_dtype, bool conv, bool two) {
  int mode = 0, relu = 0;
  classify_tail(t, out_dtype, c_dtype, &mode, &relu);
  const bool requant = tail_requant(t, out_dtype, c_dtype, mode, nullptr);
  return {!conv && (mode == 1 || mode == 2 || requant), (mode == 1 || (requant && !conv)) && !two, mode == 2, two, mode == 3};
}

// allow64: the standalone elementwise kernel also runs 64-bit steps; the tails of the contraction kernels do not
bool valid_tail(const pml_hip_epilogue& t, bool allow64 = false) {
  if (t.n_ops < 0 || t.n_ops > PML_HIP_MAX_EPI_OPS) return false;
  if (t.n_operands < 0 || t.n_operands > PML_HIP_MAX_EPI_OPERANDS) return false;
  for (int i = 0; i < t.n_ops; ++i) {
    const pml_hip_epi_op& op = t.ops[i];
    if (op.opcode < PML_HIP_EPI_ADD || op.opcode > PML_HIP_EPI_LAST_) return false;
    if (op.operand_kind == PML_HIP_OPND_TENSOR && (op.operand < 0 || op.operand >= t.n_operands)) return false;
    if (op.opcode == PML_HIP_EPI_STORE && (op.operand < 0 || op.operand >= PML_HIP_MAX_EPI_OPERANDS)) return false;
    if (!allow64 && dt_size(op.dtype) == 8 && op.opcode != PML_HIP_EPI_STORE) return false;  // 64-bit steps: general path only
  }
  return true;
}

// fp32 rounded to bf16 (nearest even), as fp32; NaNs stay NaNs
float host_round_bf16(float f) {
  uint32_t u;
  std::memcpy(&u, &f, 4);
  u = (u & 0x7fffffffu) > 0x7f800000u ? ((u & 0xffff0000u) | 0x00400000u) : ((u + 0x7fffu + ((u >> 16) & 1u)) & 0xffff0000u);
  std::memcpy(&f, &u, 4);
  return f;
}

// Row kernels have up to 256 threads for a row: a launch takes 2^23 of them, the next one the rows that follow.
template <typename F>
int in_row_runs(int64_t rows, F&& launch) {
  constexpr int64_t kRun = (int64_t)1 << 23;
  static_assert(kRun * 256 <= kMaxLaunchThreads, "a run of rows is one launch");
  for (int64_t first = 0; first < rows; first += kRun)
    if (int rc = launch(first, std::min(kRun, rows - first))) return rc;
  return 0;
}

// Compute units of the current device (persistent kernels size their grids by it).
int device_cus() {
  static int cached[64] = {0};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
  if (cached[dev] == 0) {
    hipDeviceProp_t prop;
    cached[dev] = hipGetDeviceProperties(&prop, dev) == hipSuccess ? prop.multiProcessorCount : 256;
  }
  return cached[dev];
}

// Device memory of the entry point that allocates nothing (pml_hip_gemm_run_static): the transposed
// right-hand side Bt[N][K].  Every GPU the library runs on holds its own copy of the array until the process
// ends.  In host code the array's name is only a handle: the address kernels and copies use is looked up once
// per device, with that device current, and kept here.
static __device__ __align__(256) unsigned char scratch[PML_HIP_STATIC_SCRATCH_BYTES];
constexpr int kMaxDevices = 64;
void* g_scratch_ptr[kMaxDevices] = {nullptr};
std::mutex g_scratch_mutex;

// Address of `scratch` on the current device; null (and the error text set) on failure.
void* scratch_of_current_device() {
  int dev = 0;
  if (check(hipGetDevice(&dev), "hipGetDevice")) return nullptr;
  if (dev < 0 || dev >= kMaxDevices) {
    fail("device ordinal beyond the per-device table");
    return nullptr;
  }
  std::lock_guard<std::mutex> lock(g_scratch_mutex);
  if (!g_scratch_ptr[dev]) {
    void* ptr = nullptr;
    if (check(hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)), "hipGetSymbolAddress(scratch)")) return nullptr;
    g_scratch_ptr[dev] = ptr;
  }
  return g_scratch_ptr[dev];
}

// A plan whose tile is TILE_64x64_KSPLIT and is what its invokes may run: decides the split for m x n results over `slabs` slabs of K and allocates the
// workspace.  Leaves the plan unsplit (the plain 64 x 64 tile runs) when a split is not worth it or memory is short.
void prepare_split(Plan* p, int64_t m, int64_t n, int64_t slabs) {
  if (p->tile != TILE_64x64_KSPLIT) return;
  int splits = 1, per = 0;
  igemm_split_plan(m, n, slabs, device_cus(), &splits, &per);
  if (splits < 2) return;
  const int64_t pitch = (n + 3) / 4 * 4;
  if (pitch >= ((int64_t)1 << 31)) return;
  p->ws = p->hold((size_t)splits * m * pitch * 4);
  if (!p->ws) return;
  p->sk_splits = splits;
  p->sk_per = per;
  p->sk_pitch = (int)pitch;
}
void split_args(const Plan* p, IgemmArgs& g) {
  g.ws = p->ws;
  g.sk_splits = p->ws ? p->sk_splits : 0;
  g.sk_per = p->sk_per;
  g.sk_pitch = p->sk_pitch;
}

// A convolution whose pixels fill no whole 128-byte slabs takes the taps of a filter row as one: neighbouring pixels follow
// each other in memory, and a chunk of the run finds its pixel by multiply-and-shift (exact below 2^20, checked here).  Slabs
// per filter row then hold kw ci values instead of ci each: int8 ci = 32 k = 5, 25 slabs of which a quarter is values -> 10;
// bf16 ci = 16 k = 3, 9 -> 3; fp32 ci = 16 k = 7, 49 -> 28.  Measured: bf16 5 x 107 x 107 x 16 (*) 7 x 7 33.1 -> 14.1 us,
// 8 x 125 x 125 x 16 (*) 5 x 5 45.1 -> 29.2, int8 85 x 22 x 22 x 32 (*) 3 x 3 25.0 -> 18.8; 36 sizes drawn 1.13x in the mean.
bool conv_tap_runs(const pml_hip_conv2d_desc& d) {
  const int64_t pixel = d.ci * dt_size(d.in_dtype), run = d.kw * pixel;
  return d.dil_w == 1 && d.kw > 1 && pixel % 16 == 0 && (run + 127) / 128 < d.kw * ((pixel + 127) / 128) && run * pixel < (1 << 20);
}
// 128-byte slabs of K of an implicit-GEMM convolution
int64_t conv_slabs(const pml_hip_conv2d_desc& d) {
  const int64_t pixel = d.ci * dt_size(d.in_dtype);
  return d.kh * (conv_tap_runs(d) ? (d.kw * pixel + 127) / 128 : d.kw * ((pixel + 127) / 128));
}

// Everything of the kernel arguments that the descriptor fixes (no operand pointers, no right-hand side).
void gemm_args(const pml_hip_gemm_desc& d, IgemmArgs& g) {
  std::memset(&g, 0, sizeof g);
  if (d.k2 > 0) {
    g.K2 = d.k2;
    g.lda2 = d.lda2;
    g.ldbt2 = d.b_layout ? d.ldb2 : d.k2;
    g.g2_stride = d.a2_stride;
    if (d.a2_stride > 0) {
      g.g2_h = (int)d.a2_h;
      g.g2_w = (int)d.a2_w;
      g.g2_ohw = (int)(d.a2_oh * d.a2_ow);
      g.g2_ow = (int)d.a2_ow;
      fast_div_magic((unsigned)g.g2_ohw, &g.g2_ohw_magic, &g.g2_ohw_shift);
      fast_div_magic((unsigned)g.g2_ow, &g.g2_ow_magic, &g.g2_ow_shift);
    }
  }
  g.M = d.m;
  g.N = d.n;
  g.K = d.k;
  g.lda = d.lda;
  g.ldc = d.ldc;
  g.out_dtype = d.out_dtype;
  g.init_dtype = d.init_dtype;
  g.init_rs = d.init_row_stride;
  g.init_cs = d.init_col_stride;
  g.c_dtype = d.c_dtype;
  g.n_cus = device_cus();
  g.stream = PML_HIP_FLAG_TILE_OF(d.flags) < 0;
  classify_tail(d.tail, d.out_dtype, d.c_dtype, &g.tail_mode, &g.tail_relu);
  g.tail_ssr = tail_scale_shift(d.tail, d.out_dtype, g.tail_mode);
  tail_requant(d.tail, d.out_dtype, d.c_dtype, g.tail_mode, &g);
  g.tail = d.tail;
}
void conv_args(const Plan* p, IgemmArgs& g) {
  const pml_hip_conv2d_desc& d = p->conv;
  const int64_t K = d.kh * d.kw * d.ci;
  std::memset(&g, 0, sizeof g);
  g.M = d.n * d.oh * d.ow;
  g.N = d.co;
  g.K = K;
  g.A = nullptr;
  g.Bt = p->bt;
  g.ldbt = p->bt_ld;
  g.C = nullptr;
  g.ldc = d.co;
  g.H = (int)d.h;
  g.W = (int)d.w;
  g.CI = (int)d.ci;
  g.OH = (int)d.oh;
  g.OW = (int)d.ow;
  g.KH = (int)d.kh;
  g.KW = (int)d.kw;
  g.SH = (int)d.stride_h;
  g.SW = (int)d.stride_w;
  g.PH = (int)d.pad_h;
  g.PW = (int)d.pad_w;
  g.DH = (int)d.dil_h;
  g.DW = (int)d.dil_w;
  g.out_dtype = d.out_dtype;
  g.init = nullptr;
  g.init_dtype = d.init_dtype;
  g.init_rs = d.init_row_stride;
  g.init_cs = d.init_col_stride;
  g.c_dtype = d.c_dtype;
  classify_tail(d.tail, d.out_dtype, d.c_dtype, &g.tail_mode, &g.tail_relu);
  g.tail_ssr = tail_scale_shift(d.tail, d.out_dtype, g.tail_mode);
  tail_requant(d.tail, d.out_dtype, d.c_dtype, g.tail_mode, &g);
  g.tail = d.tail;
  g.NB = (int)d.n;
  g.n_cus = device_cus();
  g.stream = PML_HIP_FLAG_TILE_OF(d.flags) < 0;
  g.halo_rows = p->halo_rows;
  g.n_tiles = p->halo_tiles;
  g.halo_variant = p->halo_variant;
  fast_div_magic((unsigned)(d.oh * d.ow), &g.div_per_magic, &g.div_per_shift);
  fast_div_magic((unsigned)d.ow, &g.div_ow_magic, &g.div_ow_shift);
  if (const int mp = PML_HIP_FLAG_MAXPOOL_OF(d.flags)) {
    g.pool = 1;
    g.pool_pt = (mp >> 1) & 1;
    g.pool_pl = (mp >> 3) & 1;
    g.pool_oh = (int)((d.oh + ((mp >> 1) & 1) + ((mp >> 2) & 1) - 3) / 2 + 1);
    g.pool_ow = (int)((d.ow + ((mp >> 3) & 1) + ((mp >> 4) & 1) - 3) / 2 + 1);
  }
  if (p->via_s2d) {
    // unit-stride convolution over the re-blocked input: one "tap" per block row, whose K-run covers
    // s2d_kaw neighbouring blocks of s2d_ch channels
    const int es = dt_size(d.in_dtype);
    g.K = (int64_t)p->s2d_ka * p->s2d_kaw * p->s2d_ch;
    g.H = p->s2d_h;
    g.W = p->s2d_w;
    g.CI = p->s2d_kaw * p->s2d_ch;
    g.pix_pitch = p->s2d_ch * es;
    g.KH = p->s2d_ka;
    g.KW = 1;
    g.SH = g.SW = 1;
    g.PH = ((int)d.pad_h + ((int)d.pad_h & 1)) / 2;
    g.PW = ((int)d.pad_w + ((int)d.pad_w & 1)) / 2;
  }
}

void s2d_args(const Plan* p, S2dArgs& a) {
  const pml_hip_conv2d_desc& d = p->conv;
  std::memset(&a, 0, sizeof a);
  a.N = (int)d.n, a.H = (int)d.h, a.W = (int)d.w, a.CI = (int)d.ci;
  a.HS = p->s2d_h, a.WS = p->s2d_w, a.CH = p->s2d_ch;
  a.KH = (int)d.kh, a.KW = (int)d.kw, a.CO = (int)d.co;
  a.KA = p->s2d_ka, a.KAW = p->s2d_kaw;
  a.EH = (int)d.pad_h & 1, a.EW = (int)d.pad_w & 1;
}

// Whether and how a convolution runs over its window in LDS (winconv.hip) in the place of an implicit GEMM.
//   * an implicit GEMM fetches every pixel once per tap: bf16 and int8 always run over windows, 1.2 to 2.6 x as fast (bf16 128 x
//     28 x 28 x 128 (*) 3 x 3 x 128 44 -> 31 us, 103 x 11 x 11 x 256 (*) 7 x 7 x 29 74.8 -> 28.3).  fp32 is bound by its MFMAs: where
//     they are not mostly work done for edges, which a tile of 448 x 64 has more of than one of 64 x 64, or where the rounds of tiles
//     that an implicit GEMM takes cost more (16 x 56 x 56 x 64 (*) 3 x 3 x 64, 3.06 rounds, 44.8 -> 39.2 us, 8 x 40 x 40 x 64 (*) 7 x 7 x 45 72.6 -> 66.3).
//   * a direct tile, or a K loop split over workgroups, is left where the window is cheaper by these kernels' prices, which are
//     a microsecond below what launches back to back take (bf16 22 x 11 x 11 x 128 (*) 5 x 5 x 86 15.3 -> 10.4 from a split;
//     11 x 11 x 11 x 64 (*) 3 x 3 x 20 stays, 5.5 both ways; 3 x 30 x 30 x 256 (*) 7 x 7 x 18 stride 2 stays, 14.6, over windows 34.6).
//   * 3 x 3 filters that the kernels of conv_halo.hip keep on the chip stay there (128 x 56 x 56 x 64 (*) 3 x 3 x 64 36); their general
//     form for any other filter that fits LDS does not (40 x 30 x 30 x 64 (*) 3 x 3 x 48 23.9 -> 9.1).
WinShape window_shape(Plan* p, bool named, double* window_us) {
  const pml_hip_conv2d_desc& d = p->conv;
  const int out = p->mfma_kind == KIND_BF16 ? PML_HIP_BF16 : p->mfma_kind == KIND_I8 ? PML_HIP_I32 : PML_HIP_F32;
  if (d.init_kind && !(d.init_row_stride == 0 && d.init_col_stride == 1 && d.init_dtype == out)) return {};
  IgemmArgs g;
  conv_args(p, g);
  double us = 0;
  const WinShape shape = winconv_shape(p->mfma_kind, g, &us);
  *window_us = us;
  if (shape.config < 0 || named) return shape;
  // (a last block of channels that is mostly empty, int8 of 96 channels: 62 x 45 x 45 x 96 (*) 5 x 5 x 23 stride 2 15.4, over windows 17.0)
  const int64_t ci_bytes = d.ci * dt_size(d.in_dtype);
  if ((ci_bytes + 63) / 64 * 64 * 5 > ci_bytes * 6) return {};
  const int64_t k_bytes = g.K * dt_size(d.in_dtype);
  if (p->tile_direct >= 0 || splits_k(g.M, g.N, k_bytes, p->mfma_kind)) {
    double other = 0;
    (void)direct_tile_of(g.M, g.N, k_bytes, p->mfma_kind, 0, false, true, false, &other);
    return us < 0.95 * other + 0.6 ? shape : WinShape{};
  }
  if (p->mfma_kind == KIND_F32) {
    const double mma_us = (double)((g.M + 63) / 64 * 64) * (double)((g.N + 63) / 64 * 64) * (double)g.K * 2 / 154e6;
    const double tiles_us = 4.2 + f32_slab_us(g.M, g.N, k_bytes) * (double)conv_slabs(d);
    return us < std::max(4 + 1.45 * mma_us, 0.93 * tiles_us) ? shape : WinShape{};
  }
  return shape;
}

// The direct tile of a convolution whose filter comes with the call and is read as it lies (-1: it is packed by a launch of its
// own first): where that is cheaper than the plan's kernel and the packing.  fp32 sums are the same bits either way, so there it is for
// convolutions that take a direct tile over a packed filter, too.  us a call, packing first -> as it lies:
//   1 x 1    bf16 28 x 9 x 9 x 256 (*) 62 10.3 -> 5.9     int8 36 x 7 x 7 x 128 (*) 46 8.5 -> 4.7     fp32 3 x 9 x 9 x 96 (*) 23 stride 2 9.7 -> 6.7
//   3 x 3    bf16 5 x 25 x 25 x 32 (*) 76 8.8 -> 5.2      int8 34 x 14 x 14 x 64 (*) 59 9.5 -> 6.0    fp32 2 x 15 x 15 x 32 (*) 37 10.2 -> 6.8
//   5 x 5    bf16 11 x 21 x 21 x 64 (*) 102 stride 2 11.7 -> 8.7; but 2 x 69 x 69 x 64 (*) 19, two rounds, 12.2, as it lies 16.9
//   7 x 7    bf16 from 3 KB of K on by 15 % where whole words of columns are packed quickly, 74 x 18 x 40 (*) 16 7.5, as it lies 7.9, 968
//            pixels of 64 (*) 56 11.3, 12.3, 5 x 5 432 of 96 (*) 60 9.5, 10.4, and under tails with operands and functions (a workgroup's is of
//            four times the results): with tanh 10.6, 11.9, 2 x 61 x 13 x 32 (*) 9 with a residual 13.9, 14.3.  But odd columns 300 pixels of
//            40 (*) 37 9.0, as it lies 8.2, 5 x 5 1089 of 128 (*) 50 18.7, 12.7, and 256 channels 3 x 3 882 of 256 (*) 64 10.3, 9.05
// and of 140 drawn convolutions with the filter in the call 59 take it, 1.36 x in the mean.
int given_filter_tile(const Plan* p, double window_us) {
  const pml_hip_conv2d_desc& d = p->conv;
  const int es = dt_size(d.in_dtype);
  const int64_t M = d.n * d.oh * d.ow, k_bytes = (p->patches ? p->kpad : d.kh * d.kw * d.ci) * es;
  const bool window = p->win.config >= 0;
  if (p->mfma_kind == KIND_F32X3 || (p->mfma_kind == KIND_F32 && p->tile_direct < 0)) return -1;
  double packed_us = window_us;
  if (!window) (void)direct_tile_of(M, d.co, k_bytes, p->mfma_kind, 0, p->tile_direct >= 0, /*can_split=*/!p->patches, false, &packed_us);
  const double small = direct_lies_us(M, d.co, k_bytes, p->mfma_kind, 16), large = direct_lies_us(M, d.co, k_bytes, p->mfma_kind, 32), packing = 3.0 + 2.0 * (double)k_bytes * (double)d.co / 2.2e6;
  const bool bare = tail_form(d.tail, d.out_dtype, d.c_dtype, true, false).bare;
  const bool one_round = ((M + 15) / 16) * ((d.co + 15) / 16) <= device_cus();  // (612 pixels of 5 x 5 x 96 (*) 100, two over a packed filter: 12.9, as it lies 10.3)
  const bool close = p->tile_direct >= 0 && !(p->mfma_kind == KIND_BF16 && k_bytes >= 3072 && ((d.co % 4 == 0 && d.ci < 256 && one_round) || !bare));
  if (std::min(small, large) > (close ? 0.95 : 0.85) * (packed_us + packing)) return -1;
  return small <= large ? TILE_16x16_W8 : TILE_32x32_W8;
}

// Packs the caller's HWCK filter into the plan's Bt.
hipError_t pack_conv_filter(Plan* p, const void* filter, hipStream_t s) {
  const pml_hip_conv2d_desc& d = p->conv;
  const int es = dt_size(d.in_dtype);
  if (p->win.config >= 0) return winconv_pack_launch(es, filter, {(int)(d.kh * d.kw), (int)d.ci, (int)d.co, 0, d.ci * d.co, d.co, 1}, p->bt, s);
  if (p->via_s2d) {
    S2dArgs a;
    s2d_args(p, a);
    a.filter = filter;
    a.gt = p->bt;
    return s2d_filter_launch(es, a, s);
  }
  if (hipError_t e = transpose_pack(es, filter, p->bt, d.kh * d.kw * d.ci, d.co, d.co, p->bt_ld, s); e != hipSuccess) return e;
  if (p->b_split) return split_rows_launch(p->bt, d.co, p->bt_ld, d.kh * d.kw * d.ci, s);
  return hipSuccess;
}

}  // namespace
}  // namespace pml

using namespace pml;

extern "C" {

const char* pml_hip_last_error(void) { return g_err.c_str(); }

int pml_hip_device_count(void) {
  int n = 0;
  if (hipGetDeviceCount(&n) != hipSuccess) return 0;
  return n;
}

int pml_hip_init(int device_ordinal) {
  int n = pml_hip_device_count();
  if (n <= 0) return fail("no HIP device is visible");
  if (device_ordinal < 0 || device_ordinal >= n) return fail("device ordinal out of range");
  if (check(hipSetDevice(device_ordinal), "hipSetDevice")) return 1;
  return scratch_of_current_device() ? 0 : 1;
}

int pml_hip_device_name(char* buf, size_t buf_len) {
  if (!buf || buf_len == 0) return fail("null buffer");
  int dev = 0;
  if (check(hipGetDevice(&dev), "hipGetDevice")) return 1;
  hipDeviceProp_t prop;
  if (check(hipGetDeviceProperties(&prop, dev), "hipGetDeviceProperties")) return 1;
  std::snprintf(buf, buf_len, "%s (%s, %d CUs)", prop.name, prop.gcnArchName, prop.multiProcessorCount);
  return 0;
}

int pml_hip_malloc(void** dptr, size_t nbytes) {
  if (!dptr) return fail("null out pointer");
  *dptr = nullptr;
  if (nbytes == 0) nbytes = 16;
  return check(hipMalloc(dptr, nbytes), "hipMalloc");
}
int pml_hip_free(void* dptr) { return dptr ? check(hipFree(dptr), "hipFree") : 0; }
int pml_hip_host_alloc(void** hptr, size_t nbytes) {
  if (!hptr) return fail("null out pointer");
  return check(hipHostMalloc(hptr, nbytes ? nbytes : 16, hipHostMallocDefault), "hipHostMalloc");
}
int pml_hip_host_free(void* hptr) { return hptr ? check(hipHostFree(hptr), "hipHostFree") : 0; }

int pml_hip_memcpy_h2d(void* dst, const void* src, size_t nbytes, pml_hip_stream s) {
  if (nbytes == 0) return 0;
  if (check(hipMemcpyAsync(dst, src, nbytes, hipMemcpyHostToDevice, (hipStream_t)s), "hipMemcpyAsync(h2d)")) return 1;
  return check(hipStreamSynchronize((hipStream_t)s), "hipStreamSynchronize");
}
int pml_hip_memcpy_d2h(void* dst, const void* src, size_t nbytes, pml_hip_stream s) {
  if (nbytes == 0) return 0;
  if (check(hipMemcpyAsync(dst, src, nbytes, hipMemcpyDeviceToHost, (hipStream_t)s), "hipMemcpyAsync(d2h)")) return 1;
  return check(hipStreamSynchronize((hipStream_t)s), "hipStreamSynchronize");
}
int pml_hip_memcpy_d2d(void* dst, const void* src, size_t nbytes, pml_hip_stream s) {
  if (nbytes == 0) return 0;
  return check(hipMemcpyAsync(dst, src, nbytes, hipMemcpyDeviceToDevice, (hipStream_t)s), "hipMemcpyAsync(d2d)");
}
int pml_hip_memcpy_h2d_async(void* dst, const void* src, size_t nbytes, pml_hip_stream s) {
  return nbytes ? check(hipMemcpyAsync(dst, src, nbytes, hipMemcpyHostToDevice, (hipStream_t)s), "hipMemcpyAsync(h2d)") : 0;
}
int pml_hip_memcpy_d2h_async(void* dst, const void* src, size_t nbytes, pml_hip_stream s) {
  return nbytes ? check(hipMemcpyAsync(dst, src, nbytes, hipMemcpyDeviceToHost, (hipStream_t)s), "hipMemcpyAsync(d2h)") : 0;
}
int pml_hip_copy_spans(int n, void* const* dst, const void* const* src, const size_t* nbytes, pml_hip_stream s) {
  return pml_hip_copy_spans_stamped(n, dst, src, nbytes, nullptr, 0, s);
}
int pml_hip_copy_spans_stamped(int n, void* const* dst, const void* const* src, const size_t* nbytes, uint64_t* stamp, int after,
                               pml_hip_stream s) {
  if (n < 0 || (n > 0 && (!dst || !src || !nbytes))) return fail("copy_spans: bad argument");
  for (int i = 0; i == 0 || i < n; i += kMaxSpans) {
    SpanArgs a;
    std::memset(&a, 0, sizeof a);
    for (int j = i; j < n && j < i + kMaxSpans; ++j) {
      if (nbytes[j] == 0) continue;
      if (!dst[j] || !src[j]) return fail("copy_spans: null pointer");
      a.dst[a.n] = dst[j];
      a.src[a.n] = src[j];
      a.bytes[a.n++] = nbytes[j];
    }
    if (after ? i + kMaxSpans >= n : i == 0) a.stamp = stamp;
    a.stamp_after = after;
    if (check(copy_spans_launch(a, (hipStream_t)s), "copy_spans_launch")) return 1;
  }
  return 0;
}
int pml_hip_copy_spans_marked(int n, void* const* dst, const void* const* src, const size_t* nbytes, uint64_t* stamp, uint32_t* mark,
                              uint32_t* arrived, uint32_t value, pml_hip_stream s) {
  if (!mark || !arrived) return fail("copy_spans: bad argument");
  if (pml_hip_copy_spans_stamped(n, dst, src, nbytes, stamp, 0, s)) return 1;
  return check(mark_launch(mark, value, (hipStream_t)s), "mark");
}
int pml_hip_wait_mark(const uint32_t* mark, uint32_t value, pml_hip_stream s) {
  if (!mark) return fail("wait_mark: null pointer");
  using clock = std::chrono::steady_clock;
  const clock::time_point begin = clock::now();
  for (clock::duration waited{}; waited < std::chrono::milliseconds(1); waited = clock::now() - begin) {
    for (int i = 0; i < 64; ++i) {
      if (__atomic_load_n(mark, __ATOMIC_ACQUIRE) == value) return 0;
      __builtin_ia32_pause();
    }
    if (waited > std::chrono::microseconds(20)) std::this_thread::yield();
  }
  return pml_hip_stream_sync(s);
}
int pml_hip_clock_khz(void) {
  int dev = 0, khz = 0;
  if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&khz, hipDeviceAttributeWallClockRate, dev) != hipSuccess) return 0;
  return khz;
}
int pml_hip_fill_u32(void* dptr, uint32_t pattern, size_t n_words, pml_hip_stream s) {
  return check(fill_u32_launch(dptr, pattern, n_words, (hipStream_t)s), "fill");
}

int pml_hip_stream_create(pml_hip_stream* s) {
  hipStream_t st;
  if (check(hipStreamCreate(&st), "hipStreamCreate")) return 1;
  *s = (pml_hip_stream)st;
  return 0;
}
int pml_hip_stream_destroy(pml_hip_stream s) { return check(hipStreamDestroy((hipStream_t)s), "hipStreamDestroy"); }
int pml_hip_stream_sync(pml_hip_stream s) { return check(hipStreamSynchronize((hipStream_t)s), "hipStreamSynchronize"); }
int pml_hip_event_create(pml_hip_event* e) {
  hipEvent_t ev;
  if (check(hipEventCreate(&ev), "hipEventCreate")) return 1;
  *e = (pml_hip_event)ev;
  return 0;
}
int pml_hip_capture_begin(pml_hip_stream s) {
  if (!s) return fail("pml_hip_capture_begin: the default stream cannot be captured");
  // (thread-local mode: other threads of the process may go on allocating while this one records)
  return check(hipStreamBeginCapture((hipStream_t)s, hipStreamCaptureModeThreadLocal), "hipStreamBeginCapture");
}
int pml_hip_capture_end(pml_hip_stream s, pml_hip_graph* graph) {
  if (!s || !graph) return fail("pml_hip_capture_end: null argument");
  *graph = nullptr;
  hipGraph_t g = nullptr;
  // (always called, also after a failed recording: it is what takes the stream out of capture mode)
  const hipError_t e = hipStreamEndCapture((hipStream_t)s, &g);
  if (e != hipSuccess || !g) {
    (void)hipGetLastError();
    return fail(std::string("hipStreamEndCapture: ") + hipGetErrorString(e));
  }
  Replay* r = nullptr;
  if (check(replay_create(g, &r), "hipGraphInstantiate")) return 1;
  *graph = (pml_hip_graph)r;
  return 0;
}
int pml_hip_graph_launch(pml_hip_graph graph, pml_hip_stream s) {
  if (!graph) return fail("pml_hip_graph_launch: null graph");
  return check(replay_launch(*(const Replay*)graph, (hipStream_t)s), "hipGraphLaunch");
}
int pml_hip_graph_destroy(pml_hip_graph graph) {
  replay_destroy((Replay*)graph);
  return 0;
}
int pml_hip_event_destroy(pml_hip_event e) { return check(hipEventDestroy((hipEvent_t)e), "hipEventDestroy"); }
int pml_hip_event_record(pml_hip_event e, pml_hip_stream s) {
  return check(hipEventRecord((hipEvent_t)e, (hipStream_t)s), "hipEventRecord");
}
int pml_hip_event_sync(pml_hip_event e) { return check(hipEventSynchronize((hipEvent_t)e), "hipEventSynchronize"); }
int pml_hip_event_done(pml_hip_event e) {
  const bool done = hipEventQuery((hipEvent_t)e) == hipSuccess;
  if (!done) (void)hipGetLastError();
  return done ? 1 : 0;
}
int pml_hip_stream_wait_event(pml_hip_stream s, pml_hip_event e) {
  return check(hipStreamWaitEvent((hipStream_t)s, (hipEvent_t)e, 0), "hipStreamWaitEvent");
}

int pml_hip_event_elapsed_ms(pml_hip_event start, pml_hip_event stop, float* ms) {
  return check(hipEventElapsedTime(ms, (hipEvent_t)start, (hipEvent_t)stop), "hipEventElapsedTime");
}

// ---------------------------------------------------------------------------
// GEMM
// ---------------------------------------------------------------------------

// Checks a GEMM descriptor; the MFMA kind (>= 0) or -1 with the error text set.
static int gemm_desc_kind(const pml_hip_gemm_desc* d) {
  if (!d) {
    fail("null descriptor");
    return -1;
  }
  const int kind = mfma_kind_of(d->in_dtype, d->flags);
  if (kind < 0) {
    fail("gemm: in_dtype must be F32, BF16 or I8");
    return -1;
  }
  const bool out_ok = (kind == KIND_I8) ? d->out_dtype == PML_HIP_I32
                                        : (d->out_dtype == PML_HIP_F32 || (kind == KIND_BF16 && d->out_dtype == PML_HIP_BF16));
  if (!out_ok) {
    fail("gemm: out_dtype does not fit in_dtype");
    return -1;
  }
  if ((d->flags & ~(PML_HIP_FP32_AS_BF16X3 | kScheduleBits)) != 0 || ((d->flags & PML_HIP_FP32_AS_BF16X3) && d->in_dtype != PML_HIP_F32) ||
      !schedule_bits_ok(d->flags)) {
    fail("gemm: flags may only hold PML_HIP_FP32_AS_BF16X3 (with in_dtype F32) and schedule overrides that name an existing tile");
    return -1;
  }
  if (d->m <= 0 || d->n <= 0 || d->k <= 0 || d->lda < d->k || d->ldb < (d->b_layout ? d->k : d->n) || d->ldc < d->n ||
      (d->b_layout != 0 && d->b_layout != 1)) {
    fail("gemm: bad sizes or leading dimensions");
    return -1;
  }
  const int es = dt_size(d->in_dtype);
  if ((d->k * es) % 16 != 0 || (d->lda * es) % 16 != 0 || (d->b_layout && (d->ldb * es) % 16 != 0)) {
    fail("gemm: K and the K-contiguous leading dimensions must cover whole 16-byte vectors");
    return -1;
  }
  if (!valid_tail(d->tail)) {
    fail("gemm: malformed tail");
    return -1;
  }
  if (d->k2 != 0) {
    if (kind != KIND_BF16 || d->k2 < 0 || (d->k2 * es) % 16 != 0 || (d->lda2 * es) % 16 != 0 || d->lda2 < d->k2 ||
        d->ldb2 < (d->b_layout ? d->k2 : d->n) || (d->b_layout && (d->ldb2 * es) % 16 != 0) || d->a2_stride < 0 ||
        (d->init2_kind != 0 && d->init2_kind != 1)) {
      fail("gemm: malformed second product (bf16 only; k2 and lda2 must cover whole 16-byte vectors)");
      return -1;
    }
    if (d->a2_stride > 0) {
      // rows of a strided 1x1 convolution: the result rows are the pixels of whole images
      if (d->a2_oh <= 0 || d->a2_ow <= 0 || d->m % (d->a2_oh * d->a2_ow) != 0 || (d->a2_oh - 1) * d->a2_stride >= d->a2_h ||
          (d->a2_ow - 1) * d->a2_stride >= d->a2_w || d->a2_oh * d->a2_ow > INT32_MAX || d->a2_h > INT32_MAX || d->a2_w > INT32_MAX) {
        fail("gemm: the second product's pixel rows do not fit its image");
        return -1;
      }
    }
  } else if (d->init2_kind != 0) {
    fail("gemm: a second initial value needs a second product");
    return -1;
  }
  if (kind == KIND_F32X3 && PML_HIP_FLAG_TILE_OF(d->flags) < 0 && fp32_beats_split(d->m, d->n, d->k * es)) return KIND_F32;
  return kind;
}

int pml_hip_gemm_tail_cheaper_apart(const pml_hip_gemm_desc* d) {
  if (!d || d->tail.n_ops == 0 || d->k2 != 0) return 0;
  const int kind = gemm_desc_kind(d);
  if (kind != KIND_I8) return 0;
  int mode = 0, relu = 0;
  classify_tail(d->tail, d->out_dtype, d->c_dtype, &mode, &relu);
  if (mode == 1 || mode == 2 || tail_requant(d->tail, d->out_dtype, d->c_dtype, mode, nullptr)) return 0;
  const int64_t k_bytes = d->k * dt_size(d->in_dtype);
  if (PML_HIP_FLAG_TILE_OF(d->flags) >= 0) return 0;  // a named tile is taken whatever the tail
  return choose_tile(d->m, d->n, k_bytes, kind, {true}) == TILE_256x256_W8 && choose_tile(d->m, d->n, k_bytes, kind, {false}) != TILE_256x256_W8;
}

// Whether a product's 256 x 256 tile reads B[K][N] with rows of `ldb` elements as it lies: four neighbouring columns per lane
// and K-row, through registers (given.hip).  For bf16 it is then the better form of a packed right-hand side, too: 4096^3 from
// the [K][N] copy 107.6 us, from Bt through LDS 113.6 (int8: 72.8 and 69.0; all back to back until the clock settles).
static bool takes_b_as_given(const pml_hip_gemm_desc& d, int mfma_kind, int tile, int64_t ldb) {
  return tile == TILE_256x256_W8 && (mfma_kind == KIND_BF16 || mfma_kind == KIND_I8) && !d.b_layout && d.k2 == 0 && d.n % 4 == 0 &&
         ldb % 4 == 0 && given_span(d.k, ldb, dt_size(d.in_dtype)) < ((int64_t)1 << 31);
}

// The direct tiles of a product (-1: none): over Bt rows that are at hand (packed earlier, or [N][K] as given), and over a
// [K][N] right-hand side as it lies.  One that has to be transposed first, and a tile the descriptor names, stay with the
// plan's tile -- except that fp32 sums are the same bits in either layout: there the layout decides which direct tile, not whether.
// lds_tile: the plan's tile.
static DirectTiles direct_tiles(const pml_hip_gemm_desc& d, int kind, int lds_tile) {
  DirectTiles t;
  if (PML_HIP_FLAG_TILE_OF(d.flags) >= 0) return t;
  const int es = dt_size(d.in_dtype);
  // (Two products are priced against one chain of all slabs: of 49 x 2048, K = 512 + 1024 the split takes 9.2 us and the direct
  // tile 8.8, of 196 x 256, K = 1024 + 512 9.0 and 5.8; only a K of 4096 turns that round, 10.7 and 17.0.)
  t.rows = direct_tile_of(d.m, d.n, (d.k + d.k2) * es, kind, 0, false, /*can_split=*/d.k2 == 0);
  // (fp32 of a long K over a few columns, which gains little from rows of K and loses more over [K][N], where K is not split: 6 x 59,
  // K = 4000 12.9 -> 13.1 and 17.3 -> 21.4, 120 x 71, K = 2688 17.5 -> 18.2 from [K][N]; 1030 x 36, K = 2608 12.6 -> 9.7 and 16.0 -> 16.9 stays)
  if (kind == KIND_F32 && t.rows >= 0 && splits_k(d.m, d.n, d.k * es, kind)) {
    double rows_us = 0, lds_us = 0;
    (void)direct_tile_of(d.m, d.n, d.k * es, kind, 0, /*always=*/true, true, false, &rows_us, &lds_us);
    const double lies_us = std::min(direct_lies_us(d.m, d.n, d.k * es, kind, 16), direct_lies_us(d.m, d.n, d.k * es, kind, 32));
    const double split_us = lds_us + 3.0 + 2.0 * (double)(d.k * es * d.n) / 2.2e6;
    if ((rows_us > 0.8 * lds_us && lies_us > 1.2 * split_us) || (rows_us > 0.9 * lds_us && lies_us > split_us)) t.rows = -1;
  }
  if (d.b_layout || d.k2 > 0 || (kind == KIND_F32 && t.rows < 0)) return t;
  t.given = direct_tile_of(d.m, d.n, d.k * es, kind, d.ldb * es, /*always=*/kind == KIND_F32, /*can_split=*/true, takes_b_as_given(d, kind, lds_tile, d.ldb));
  return t;
}

// Whether a launch streams its rows past the [K][N] right-hand side `b` as it lies, with the arguments then changed to that.
static bool streams_given(int mfma_kind, int tile, bool conv, const void* b, int64_t ldb, IgemmArgs& g) {
  if (mfma_kind != KIND_BF16) return false;
  const void* const bt = g.Bt;
  const int64_t ldbt = g.ldbt;
  g.Bt = b, g.ldbt = ldb, g.b_kn = 1;
  if (stream_takes(tile, conv, g)) return true;
  g.Bt = bt, g.ldbt = ldbt, g.b_kn = 0;
  return false;
}

static const char* mfma16_name(int kind) { return kind == KIND_F32 ? "f32_16x16x4" : kind == KIND_BF16 ? "f32_16x16x32_bf16" : "i32_16x16x64_i8"; }

// The part of a plan's text that says which right-hand sides its rows stream past (stream.hip), given operands that are aligned
// to 16 bytes: rows of K (`rows_tile`: the tile taken otherwise), and a [K][N] one as it lies (kn_ldb > 0).
static std::string stream_text(int mfma_kind, bool conv, IgemmArgs g, bool init, const pml_hip_epilogue& tail, int rows_tile, bool rows_packed, int kn_tile, int64_t kn_ldb) {
  if (mfma_kind != KIND_BF16) return "";
  const void* const aligned = (const void*)256;  // (stands for an operand that is there; nothing is read)
  if (init) g.init = aligned;
  for (int i = 0; i < tail.n_operands; ++i) g.operands[i] = aligned;
  const bool rows = stream_takes(rows_tile, conv, g), kn = kn_ldb > 0 && streams_given(mfma_kind, kn_tile, conv, aligned, kn_ldb, g);
  if (!rows && !kn) return "";
  const std::string packed = rows_packed ? "B packed" : "B";
  return ", streamed rows past " + (rows && kn ? packed + " or as it lies" : rows ? packed : std::string("B as it lies")) + " mfma=" + mfma16_name(mfma_kind);
}

// Microseconds of a product in the tiles that a panel may stand in for, from the same timings as panel_us (990 products, 10 to 13 %
// rms): so many tiles run together on a CU, a tile takes a slab's time for every 128 bytes of K and its results' time; `value_bytes`
// go to and from memory per result.  Tiles of other kinds: infinity.
static double tiled_us(int kind, int tile, int64_t m, int64_t n, int64_t k_bytes, int value_bytes, int cus) {
  struct Times { double launch, tile, slab, value, ceil; int held, edge; };
  const Times bf16_w8 = {1.64, 1.79, 0.539, 0.898, 0.77, 1, 128}, bf16_s2 = {0, 2.96, 0.616, 0.845, 0.57, 2, 128}, bf16_k2 = {4.91, 2.82, 0.24, 0, 0.77, 2, 64};
  const Times i8_w8 = {3.0, 3.65, 0.554, 0.194, 0.77, 1, 128}, i8_s2 = {0.41, 4.89, 0.634, 0.471, 0.57, 2, 128};
  const bool i8 = kind == KIND_I8;
  const Times* const t = tile == TILE_128x128_W8 ? (i8 ? &i8_w8 : &bf16_w8) : tile == TILE_128x128_W8_S2 ? (i8 ? &i8_s2 : &bf16_s2) :
                         tile == TILE_64x64_W8_K2 && !i8 ? &bf16_k2 : nullptr;
  if (!t) return std::numeric_limits<double>::infinity();
  const double per_cu = (double)((m + t->edge - 1) / t->edge) * (double)((n + t->edge - 1) / t->edge) / cus, turns = per_cu / t->held;
  const double together = std::min((double)t->held, std::max(1.0, std::ceil(per_cu)));
  const double rounds = turns <= 1 ? 1 : t->ceil * std::ceil(turns) + (1 - t->ceil) * turns;
  return t->launch + rounds * (t->tile + (double)((k_bytes + 127) / 128) * t->slab * std::pow(together, 0.9) + t->value * value_bytes * together);
}

// Whether, and as what, a product whose right-hand sides are packed runs in panels (panel.hip).  bf16, where no tile is named, no
// direct tile is cheaper, K is not split over workgroups and the rows do not stream (512 bytes of K).  Of 1000 products (ranges at
// panel_us) those of 256 x 256, 256 x 128 and 192 x 384 tiles gain 1.21 to 1.25 x on average and none loses; of 128 x 128 tiles
// those priced 5 % below the tile gain 1.16 (three stages) and 1.32 (two), 1 in 200 loses more than 3 %; of 64 x 64 tiles that share
// K those priced 10 % below gain 1.12, the others 1.03.  Plain 64 x 64 tiles, several of which share a CU, lose as often as they
// gain (0.98), and 128 x 128 tiles over up to 160 columns, most of a 256 columns wide panel, lose (0.86 to 0.97).
// int8, of 650 products: requantised from wide tiles 1.18 to 1.38 x, also over few columns (1.19), from 64 x 64 tiles 0.90 to 1.02;
// with int32 results, four bytes of which leave for one of A, 1.23 x from 128 x 128 tiles of two stages with 1 KB of K and up to 1024
// columns, and about as often less as more elsewhere (0.71 to 1.29).
static int panel_of(const pml_hip_gemm_desc& d, int kind, int tile, const DirectTiles& direct, const void* ws) {
  const int64_t k_bytes = (d.k + d.k2) * dt_size(d.in_dtype);
  if ((kind != KIND_BF16 && kind != KIND_I8) || d.b_layout || PML_HIP_FLAG_TILE_OF(d.flags) >= 0 || direct.rows >= 0 || ws || k_bytes <= 512) return -1;
  const bool wide = tile == TILE_128x128_W8 || tile == TILE_128x128_W8_S2 || tile == TILE_256x128_W16 || tile == TILE_256x256_W8 || tile == TILE_192x384_W8;
  if (kind == KIND_I8) {
    if (!wide || (d.c_dtype == PML_HIP_I32 && !(tile == TILE_128x128_W8_S2 && k_bytes >= 1024 && d.n <= 1024))) return -1;
  } else if (!(wide && d.n > 160) && (tile != TILE_64x64_W8_K2 || k_bytes < 2048)) {
    return -1;
  }
  IgemmArgs g;
  gemm_args(d, g);
  g.Bt = g.A = g.C = (void*)256;  // (stand for operands that are there; nothing is read)
  for (int i = 0; i < d.tail.n_operands; ++i) g.operands[i] = g.A;
  if (d.init_kind) g.init = g.A;
  g.ldbt = d.k;
  if (stream_takes(tile, false, g)) return -1;
  double us;
  const int config = panel_config(kind, g, d.init_kind != 0, &us);
  const int value_bytes = dt_size(d.c_dtype) * (g.tail_mode == 2 ? 2 : 1);
  const double share = kind == KIND_BF16 && tile != TILE_64x64_W8_K2 ? 0.95 : 0.9;
  return us < share * tiled_us(kind, tile, d.m, d.n, k_bytes, value_bytes, g.n_cus) ? config : -1;
}

static size_t panel_bytes(const pml_hip_gemm_desc& d, int kind) {
  IgemmArgs g;
  gemm_args(d, g);
  const int es = dt_size(d.in_dtype), frags = panel_frags(kind, g);
  return winconv_pack_bytes(es, 1, d.k, d.n, frags) + winconv_pack_bytes(es, 1, d.k2, d.n, frags);
}

// The fragments of a product that runs in panels: its configuration (-1: it does not), where they lie.
struct PanelRoom {
  int config = -1;
  void* image = nullptr;
};

// Whether a product in panels has room for the fragments of a right-hand side that comes with the call: not where that is read as
// it lies (int8 by size: gemm_run).  And pml_hip_gemm_run_static gives the same bits, so floats are packed where its array holds
// the fragments, too, which whole blocks make larger than the transposed form, or where it refuses the call.
static bool packs_given(const pml_hip_gemm_desc& d, int kind, int tile) {
  if (kind == KIND_I8) return true;
  return !takes_b_as_given(d, kind, tile, d.ldb) && (panel_bytes(d, kind) <= PML_HIP_STATIC_SCRATCH_BYTES || d.n * d.k * dt_size(d.in_dtype) > PML_HIP_STATIC_SCRATCH_BYTES);
}

// Whether a right-hand side that comes with the call is packed for a panel by a launch of its own, as it would be transposed by
// one.  An int8 one that a 256 x 256 tile reads as it lies pays for that launch from 50 G products on: requantised 4096 x 4096,
// K = 4096 71 us as it lies, 67.5 packed, 6000 x 3200, K = 3072 90 and 75, 4096 x 4096, K = 2048 38.6 and 40.6.
static bool packs_in_call(const pml_hip_gemm_desc& d, int kind, bool as_given) {
  return d.k2 == 0 && (!as_given || (kind == KIND_I8 && (double)d.m * (double)d.n * (double)d.k >= 5e10));
}

static bool reads_b_as_given(const pml_hip_gemm_desc& d, int mfma_kind, const void* b, int tile);

int64_t pml_hip_gemm_dispatch(const pml_hip_gemm_desc* d) {
  const int kind = gemm_desc_kind(d);
  if (kind < 0) return 0;
  const int es = dt_size(d->in_dtype);
  Plan* p = new Plan();
  p->kind = PLAN_GEMM;
  p->mfma_kind = kind;
  p->gemm = *d;
  {
    p->tile = choose_tile(d->m, d->n, (d->k + d->k2) * dt_size(d->in_dtype), kind, tail_form(d->tail, d->out_dtype, d->c_dtype, false, d->k2 > 0), PML_HIP_FLAG_TILE_OF(d->flags));
    // (a second product's slabs follow the first one's on the slab axis the splits share out.)  With a direct tile over rows
    // that are at hand the LDS tile is only left for a [K][N] right-hand side that arrives with the call and cannot be read
    // as it lies; pml_hip_gemm_pack_b ends that.
    p->direct = direct_tiles(*d, kind, p->tile);
    if (!(p->direct.rows >= 0 && (d->b_layout || kind == KIND_F32)))
      prepare_split(p, d->m, d->n, (d->k * dt_size(d->in_dtype) + 127) / 128 + (d->k2 * dt_size(d->in_dtype) + 127) / 128);
  }
  p->bt_ld = d->k;
  p->bt_bytes = (size_t)d->n * d->k * es;
  // (the text names the LDS tile of the problem's shape beside the direct tile that takes its place)
  const int lds_tile = p->tile;
  if (p->tile == TILE_64x64_KSPLIT && !p->ws) p->tile = TILE_64x64;  // (not worth splitting, no memory for the workspace, or not run)
  p->b_split = kind == KIND_F32X3 && !d->b_layout && d->k % 32 == 0 && !p->ws;
  p->b_kn = kind == KIND_BF16 && p->direct.rows < 0 && takes_b_as_given(*d, kind, p->tile, d->n);
  if (!d->b_layout && !(p->bt = p->hold(p->bt_bytes))) {
    delete p;
    fail("gemm: cannot allocate the packed right-hand side");
    return 0;
  }
  if (d->k2 > 0 && !d->b_layout && !(p->bt2 = p->hold((size_t)d->n * d->k2 * es))) {
    delete p;
    fail("gemm: cannot allocate the second packed right-hand side");
    return 0;
  }
  p->panel = panel_of(*d, kind, p->tile, p->direct, p->ws);
  // (no memory for the fragments: the product runs in tiles)
  if (p->panel >= 0 && packs_given(*d, kind, p->tile) && !(p->panel_bt = p->hold(panel_bytes(*d, kind)))) p->panel = -1;
  char buf[256];
  std::snprintf(buf, sizeof buf, "gemm %s m=%lld n=%lld k=%lld tile=%s mfma=%s", d->in_dtype == PML_HIP_F32 ? "f32" : d->in_dtype == PML_HIP_BF16 ? "bf16" : "i8",
                (long long)d->m, (long long)d->n, (long long)d->k, tile_name(p->direct.rows >= 0 ? lds_tile : p->tile),
                kind == KIND_F32 ? "f32_32x32x2" : kind == KIND_BF16 ? "f32_32x32x16_bf16" : kind == KIND_I8 ? "i32_32x32x32_i8" : "3 x f32_32x32x16_bf16 (fp32 split into bf16 head + remainder)");
  p->text = buf;
  if (p->direct.rows >= 0) p->text += std::string(", with rows of K at hand tile=") + tile_name(p->direct.rows) + " mfma=" + mfma16_name(kind);
  if (p->direct.given >= 0)
    p->text += std::string(", with B as it lies tile=") + (p->direct.given == TILE_16x16_W8 ? "16x64" : "32x64") + " (8 wavefronts sharing K) mfma=" + mfma16_name(kind);
  // (of a right-hand side on 16 bytes)
  const bool in_call = p->panel_bt && p->direct.given < 0 && packs_in_call(*d, kind, reads_b_as_given(*d, kind, (const void*)256, p->tile));
  if (p->direct.given < 0 && takes_b_as_given(*d, kind, p->tile, d->ldb) && !in_call)
    p->text += std::string(", with B as it lies") + (p->b_kn && p->panel < 0 ? " or packed" : "") + " through registers mfma=" + mfma16_name(kind);
  else if (p->b_kn && p->panel < 0)
    p->text += std::string(", with B packed through registers mfma=") + mfma16_name(kind);
  if (p->panel >= 0) p->text += std::string(", with B packed ") + (in_call ? "ahead or in the call " : "") + panel_text(p->panel) + " mfma=" + mfma16_name(kind);
  {
    IgemmArgs g;
    gemm_args(*d, g);
    g.ldbt = d->b_layout ? d->ldb : p->bt_ld;
    g.ws = p->ws;
    p->text += stream_text(kind, false, g, d->init_kind != 0, d->tail, p->direct.rows >= 0 ? p->direct.rows : p->tile, !d->b_layout,
                           p->direct.given >= 0 ? p->direct.given : p->tile, d->b_layout || d->k2 > 0 ? 0 : d->ldb);
  }
  if (d->k2 > 0) p->text += " + second product k2=" + std::to_string(d->k2) + (d->a2_stride > 0 ? " over pixel rows of stride " + std::to_string(d->a2_stride) : "");
  return (int64_t)(intptr_t)p;
}

// One GEMM launch sequence: the per-run transposition of a [K][N] right-hand side into `bt` (device memory of
// n x bt_ld elements; skipped when b is null, i.e. packed earlier, or already [N][K]), then the MFMA kernel.
// Shared by the plan-based entry point and by the one that allocates nothing.
struct SecondProduct {
  const void* a2 = nullptr;
  const void* b2 = nullptr;
  const void* init2 = nullptr;
  void* bt2 = nullptr;
  bool packed2 = false;
};

// Whether a right-hand side that arrives with the call in its row-major [K][N] form is read as it lies: by direct tiles
// whatever it is, by 256 x 256 tiles of bf16 and int8 through registers, and by the other tiles of fp32 (K-values gathered
// from [k][n] slabs) and int8 (transposing LDS reads) where rows are whole 16-byte vectors.  Everything else is transposed
// into Bt[N][K] first, unless its rows stream (streams_given).
static bool reads_b_as_given(const pml_hip_gemm_desc& d, int mfma_kind, const void* b, int tile) {
  if ((tile == TILE_16x16_W8 || tile == TILE_32x32_W8) && mfma_kind != KIND_F32X3) {
    // (four neighbouring columns per lane and K-row, whatever the type and wherever the rows begin: direct.hip)
    const int64_t es = dt_size(d.in_dtype);
    return b && !d.b_layout && d.k2 == 0 && ((uintptr_t)b & (es - 1)) == 0 && d.k * d.ldb * es < ((int64_t)1 << 31);
  }
  if (tile == TILE_256x256_W8 && (mfma_kind == KIND_BF16 || mfma_kind == KIND_I8))
    return b && takes_b_as_given(d, mfma_kind, tile, d.ldb) && ((uintptr_t)b & (4 * dt_size(d.in_dtype) - 1)) == 0;
  if (mfma_kind != KIND_F32 && mfma_kind != KIND_F32X3 && mfma_kind != KIND_I8) return false;
  if (tile == TILE_64x64_KSPLIT) return false;  // (the split kernel reads Bt)
  if (tile == TILE_192x384_W8) return false;  // (24 chunks per row: the position swizzle of the [k][n] form needs a power of two)
  const int64_t es = mfma_kind == KIND_I8 ? 1 : 4, v = 16 / es;
  if (!(b && !d.b_layout && d.k2 == 0 && d.n % v == 0 && d.ldb % v == 0 && ((uintptr_t)b & 15) == 0 &&
        d.k * d.ldb * es < ((int64_t)1 << 31)))
    return false;
  if (mfma_kind == KIND_I8) {
    // The transposing reads make an int8 tile about 15 % slower (measured at 4096^3, which takes the path above now: 86 us
    // against 74 + 10 for the copy), so they pay while the transposed copy -- a launch of at least 5 us, 3.2 TB/s beyond
    // that -- costs more than that share of the multiplication (priced at the 1.8 POP/s the kernel reaches): always for
    // small problems.
    const double t_gemm = 2.0 * (double)d.m * (double)d.n * (double)d.k / 1.8e15;
    const double t_copy = std::max(5e-6, 2.0 * (double)d.k * (double)d.n / 3.2e12);
    return 0.15 * t_gemm < t_copy;
  }
  return true;
}

// A right-hand side (second: of the second product) in the order a panel multiplies it.
static int pack_fragments(const pml_hip_gemm_desc& d, int kind, void* image, const void* b, bool second, hipStream_t s) {
  IgemmArgs g;
  gemm_args(d, g);
  const int es = dt_size(d.in_dtype), frags = panel_frags(kind, g);
  const size_t first = winconv_pack_bytes(es, 1, d.k, d.n, frags);
  const WinFilter w = {1, (int)(second ? d.k2 : d.k), (int)d.n, 0, 0, second ? d.ldb2 : d.ldb, 1, frags};
  return check(winconv_pack_launch(es, b, w, (char*)image + (second ? first : 0), s), "winconv_pack_launch");
}
// ... kept by a plan, besides the form that tiles read.  (Where the plan has no room for it yet and the packing is recorded into a
// graph, which may not allocate, the product runs in tiles.)
static int pack_panel(Plan* p, const void* b, bool second, hipStream_t s) {
  if (p->panel < 0) return 0;
  if (!p->panel_bt) {
    hipStreamCaptureStatus recorded = hipStreamCaptureStatusActive;
    if (hipStreamIsCapturing(s, &recorded) != hipSuccess) (void)hipGetLastError();
    if (recorded != hipStreamCaptureStatusNone || !(p->panel_bt = p->hold(panel_bytes(p->gemm, p->mfma_kind)))) return 0;
  }
  if (pack_fragments(p->gemm, p->mfma_kind, p->panel_bt, b, second, s)) return 1;
  p->panel_fresh[second] = true;
  return 0;
}
static int gemm_run(const pml_hip_gemm_desc& d, int mfma_kind, int tile, const DirectTiles& direct, void* bt, int64_t bt_ld, bool packed,
                    const void* a, const void* b, void* c, const void* init, const void* const* operands,
                    void* const* outs, pml_hip_stream s, const SecondProduct* second, Plan* plan, PanelRoom panel) {
  // (a right-hand side that arrives with the call is transposed per run and split in the kernel's registers: a
  // second small launch costs more than it saves; one packed once is kept split)
  const bool b_split = plan && plan->bt_is_split && !b;
  if (!a || !c) return fail("gemm_invoke: null operand");
  if (!b && (!packed || d.b_layout)) return fail("gemm_invoke: b is null and no packed right-hand side exists");
  if (d.b_layout && ((uintptr_t)b & 15) != 0) return fail("gemm_invoke: an [N][K] right-hand side must be 16-byte aligned");
  if (((uintptr_t)a & 15) != 0) return fail("gemm_invoke: A must be 16-byte aligned");
  if (d.init_kind && !init) return fail("gemm_invoke: the plan expects an initial value");
  const int es = dt_size(d.in_dtype);
  if (!b || d.b_layout) {
    if (direct.rows >= 0) tile = direct.rows;
  } else if (direct.given >= 0 && reads_b_as_given(d, mfma_kind, b, direct.given)) {
    tile = direct.given;
  } else if (direct.rows >= 0 && mfma_kind == KIND_F32) {
    tile = direct.rows;
  }
  const bool packed_kn = plan && plan->bt_is_kn && !b;
  const bool b_as_given = packed_kn || reads_b_as_given(d, mfma_kind, b, tile);
  const bool transposed = b && !d.b_layout && !b_as_given;
  if (d.k2 > 0) {
    if (!second || !second->a2) return fail("gemm_invoke: the plan has a second product: use pml_hip_gemm_invoke2");
    if (!second->b2 && (!second->packed2 || d.b_layout)) return fail("gemm_invoke2: b2 is null and no packed right-hand side exists");
    if (((uintptr_t)second->a2 & 15) != 0 || (d.b_layout && ((uintptr_t)second->b2 & 15) != 0)) return fail("gemm_invoke2: the second product's operands must be 16-byte aligned");
    if (d.init2_kind && !second->init2) return fail("gemm_invoke2: the plan expects a second initial value");
    if (plan && second->b2) plan->panel_fresh[1] = false;
    if (second->b2 && !d.b_layout &&
        check(transpose_pack(es, second->b2, second->bt2, d.k2, d.n, d.ldb2, d.k2, (hipStream_t)s), "transpose_pack"))
      return 1;
  }
  IgemmArgs g;
  gemm_args(d, g);
  if (d.k2 > 0) {
    g.A2 = second->a2;
    g.Bt2 = d.b_layout ? second->b2 : second->bt2;
    g.init2 = d.init2_kind ? second->init2 : nullptr;
  }
  g.A = a;
  g.Bt = (d.b_layout || b_as_given) && !packed_kn ? b : bt;
  g.ldbt = packed_kn ? d.n : (d.b_layout || b_as_given) ? d.ldb : bt_ld;
  g.b_kn = b_as_given ? 1 : 0;
  g.C = c;
  g.init = d.init_kind ? init : nullptr;
  for (int i = 0; i < d.tail.n_operands; ++i) {
    if (!operands || !operands[i]) return fail("gemm_invoke: missing tail operand");
    g.operands[i] = operands[i];
  }
  for (int i = 0; i < PML_HIP_MAX_EPI_OPERANDS; ++i) g.outs[i] = outs ? outs[i] : nullptr;
  // the vector tails need 16-byte aligned operands and extra outputs; otherwise the interpreter runs
  if (g.tail_mode == 2 && ((uintptr_t)g.operands[0] & 15) != 0) g.tail_mode = 0;
  if (g.tail_mode == 3 || g.tail_mode == 4) {
    for (int i = 0; i < d.tail.n_operands; ++i)
      if (((uintptr_t)g.operands[i] & 15) != 0) g.tail_mode = 0;
    for (int i = 0; i < PML_HIP_MAX_EPI_OPERANDS; ++i)
      if (((uintptr_t)g.outs[i] & 15) != 0) g.tail_mode = 0;
  }
  for (int i = 0; i < d.tail.n_ops; ++i)
    if (d.tail.ops[i].opcode == PML_HIP_EPI_STORE && !g.outs[d.tail.ops[i].operand])
      return fail("gemm_invoke: missing extra output");
  // (the K split over workgroups is not built for a right-hand side packed split)
  if (plan && !b_split) split_args(plan, g);
  // (Not where one was packed ahead: calls without any would multiply by that from then on, and tiles read `bt`.  The entry without
  // a plan leaves its array untouched by what can be read as it lies: calls that share the array count on that.)
  if (b && !d.b_layout && (transposed || plan) && panel.image && !packed && packs_in_call(d, mfma_kind, b_as_given) && panel_runs(mfma_kind, g)) {
    if (pack_fragments(d, mfma_kind, panel.image, b, false, (hipStream_t)s)) return 1;
    return check(panel_launch(mfma_kind, panel.config, g, panel.image, (hipStream_t)s), "panel_launch");
  }
  // (rows that stream take a [K][N] right-hand side as it lies, too)
  if (transposed && !(!packed && streams_given(mfma_kind, tile, false, b, d.ldb, g))) {
    // (from here on `bt` holds the plain transposed form, whatever a packed copy was kept in before)
    if (plan) plan->bt_is_split = plan->bt_is_kn = plan->panel_fresh[0] = false;
    if (check(transpose_pack(es, b, bt, d.k, d.n, d.ldb, bt_ld, (hipStream_t)s), "transpose_pack")) return 1;
  }
  if (plan && plan->panel_fresh[0] && (d.k2 == 0 || plan->panel_fresh[1]) && !b && (!second || !second->b2) && panel_runs(mfma_kind, g))
    return check(panel_launch(mfma_kind, panel.config, g, panel.image, (hipStream_t)s), "panel_launch");
  return check(igemm_launch(b_split ? KIND_F32X3P : mfma_kind, tile, false, g, (hipStream_t)s), "igemm_launch");
}

int pml_hip_gemm_invoke(int64_t plan, const void* a, const void* b, void* c, const void* init,
                        const void* const* operands, void* const* outs, pml_hip_stream s) {
  Plan* p = (Plan*)(intptr_t)plan;
  if (!p || p->kind != PLAN_GEMM) return fail("gemm_invoke: not a gemm plan");
  return gemm_run(p->gemm, p->mfma_kind, p->tile, p->direct, p->bt, p->bt_ld, p->packed, a, b, c, init, operands, outs, s, nullptr, p, {p->panel, p->panel_bt});
}

int pml_hip_gemm_invoke2(int64_t plan, const void* a, const void* b, void* c, const void* init, const void* a2, const void* b2,
                         const void* init2, const void* const* operands, void* const* outs, pml_hip_stream s) {
  Plan* p = (Plan*)(intptr_t)plan;
  if (!p || p->kind != PLAN_GEMM) return fail("gemm_invoke2: not a gemm plan");
  if (p->gemm.k2 <= 0) return fail("gemm_invoke2: the plan has no second product");
  SecondProduct sp;
  sp.a2 = a2;
  sp.b2 = b2;
  sp.init2 = init2;
  sp.bt2 = p->bt2;
  sp.packed2 = p->packed2;
  return gemm_run(p->gemm, p->mfma_kind, p->tile, p->direct, p->bt, p->bt_ld, p->packed, a, b, c, init, operands, outs, s, &sp, p, {p->panel, p->panel_bt});
}

static bool chain_descs(const pml_hip_gemm_desc& first, const pml_hip_gemm_desc& next) {
  auto columns = [](int kind, int dtype, int64_t rs, int64_t cs) { return kind == 0 || (dtype == PML_HIP_BF16 && rs == 0 && cs == 1); };
  for (const pml_hip_gemm_desc* d : {&first, &next})
    if (d->in_dtype != PML_HIP_BF16 || d->b_layout != 0 || d->flags != 0 || d->m <= 0 || !valid_tail(d->tail) ||
        !columns(d->init_kind, d->init_dtype, d->init_row_stride, d->init_col_stride))
      return false;
  IgemmArgs g, n;
  gemm_args(first, g);
  gemm_args(next, n);
  return chain_takes(g, n);
}

int pml_hip_gemm_chain_takes(const pml_hip_gemm_desc* first, const pml_hip_gemm_desc* next) {
  return first && next && chain_descs(*first, *next) ? 1 : 0;
}

int pml_hip_gemm_chain_invoke(int64_t first, int64_t next, const void* a, void* c, const void* init, const void* a2, const void* init2,
                              const void* const* operands, void* next_c, const void* next_init, pml_hip_stream s) {
  Plan *p = (Plan*)(intptr_t)first, *q = (Plan*)(intptr_t)next;
  if (!p || p->kind != PLAN_GEMM || !q || q->kind != PLAN_GEMM) return fail("gemm_chain_invoke: not two gemm plans");
  if (!chain_descs(p->gemm, q->gemm)) return fail("gemm_chain_invoke: the second plan does not multiply the first one's result onward");
  IgemmArgs g, n;
  gemm_args(p->gemm, g);
  gemm_args(q->gemm, n);
  const bool second = p->gemm.k2 > 0, residual = g.tail_mode == 2;
  if (!a || !c || !next_c || !p->packed || !q->packed || (second && (!a2 || !p->packed2))) return fail("gemm_chain_invoke: null operand or unpacked right-hand side");
  if ((p->gemm.init_kind && !init) || (second && p->gemm.init2_kind && !init2) || (q->gemm.init_kind && !next_init)) return fail("gemm_chain_invoke: the plans expect initial values");
  if (residual && (!operands || !operands[0])) return fail("gemm_chain_invoke: missing tail operand");
  const uintptr_t places = (uintptr_t)a | (uintptr_t)c | (uintptr_t)next_c | (second ? (uintptr_t)a2 : 0) | (residual ? (uintptr_t)operands[0] : 0);
  if ((places & 15) != 0 || p->bt_is_kn || q->bt_is_kn) {  // one after the other
    void* none[PML_HIP_MAX_EPI_OPERANDS] = {};
    const int rc = second ? pml_hip_gemm_invoke2(first, a, nullptr, c, init, a2, nullptr, init2, operands, none, s)
                          : pml_hip_gemm_invoke(first, a, nullptr, c, init, operands, none, s);
    return rc ? rc : pml_hip_gemm_invoke(next, c, nullptr, next_c, next_init, nullptr, none, s);
  }
  g.A = a, g.Bt = p->bt, g.ldbt = p->bt_ld, g.C = c;
  g.init = p->gemm.init_kind ? init : nullptr;
  if (second) g.A2 = a2, g.Bt2 = p->bt2, g.init2 = p->gemm.init2_kind ? init2 : nullptr;
  if (residual) g.operands[0] = operands[0];
  n.Bt = q->bt, n.ldbt = q->bt_ld, n.C = next_c, n.init = q->gemm.init_kind ? next_init : nullptr;
  return check(chain_launch(g, n, (hipStream_t)s), "chain_launch");
}

int pml_hip_gemm_run_static(const pml_hip_gemm_desc* d, const void* a, const void* b, void* c, const void* init,
                            const void* const* operands, void* const* outs, pml_hip_stream s) {
  const int kind = gemm_desc_kind(d);
  if (kind < 0) return 1;
  if (d->k2 != 0) return fail("gemm_run_static: a second product is not supported by this entry point");
  if (!b) return fail("gemm_run_static: b is null");
  void* bt = nullptr;
  if (!d->b_layout) {
    // n and k are positive and each below 2^31 by the check below, so the product cannot overflow
    if (d->n > PML_HIP_STATIC_SCRATCH_BYTES || d->k > PML_HIP_STATIC_SCRATCH_BYTES ||
        (uint64_t)d->n * (uint64_t)d->k * (uint64_t)dt_size(d->in_dtype) > (uint64_t)PML_HIP_STATIC_SCRATCH_BYTES)
      return fail("gemm_run_static: the transposed right-hand side (n x k elements) exceeds PML_HIP_STATIC_SCRATCH_BYTES (32 MiB)");
    bt = scratch_of_current_device();
    if (!bt) return 1;
  }
  // (no workspace may be allocated here: the K loop is never split over workgroups)
  const int tile = choose_tile(d->m, d->n, d->k * dt_size(d->in_dtype), kind, tail_form(d->tail, d->out_dtype, d->c_dtype, false, false), PML_HIP_FLAG_TILE_OF(d->flags), /*allow_split=*/false);
  const DirectTiles direct = direct_tiles(*d, kind, tile);
  PanelRoom panel;
  if (bt && (panel.config = panel_of(*d, kind, tile, direct, nullptr)) >= 0 && packs_given(*d, kind, tile) && panel_bytes(*d, kind) <= PML_HIP_STATIC_SCRATCH_BYTES)
    panel.image = bt;
  return gemm_run(*d, kind, tile, direct, bt, d->k, false, a, b, c, init, operands, outs, s, nullptr, nullptr, panel);
}

// ---------------------------------------------------------------------------
// conv2d
// ---------------------------------------------------------------------------

// A plan (its descriptor, element kind and 2x2-block geometry filled in) whose convolution the row-walking kernel takes,
// with a result the fused 3x3 stride-2 max-pool can walk: a pooled row per thread group of 512 threads, eight per pixel.
static bool conv2d_takes_maxpool(const Plan* p) {
  const pml_hip_conv2d_desc& d = p->conv;
  const int path = PML_HIP_FLAG_CONV_OF(d.flags);
  if (!p->via_s2d || path == PML_HIP_CONV_IGEMM || path == PML_HIP_CONV_PATCHES) return false;
  IgemmArgs g;
  conv_args(p, g);
  // (the filter pointer's alignment is the allocator's: not part of the question)
  g.Bt = nullptr;
  if (!conv_blocks4x4_prepare(p->mfma_kind, g)) return false;
  return d.oh >= 3 && d.ow >= 3 && g.pool_oh >= 1 && g.pool_ow >= 1 && g.pool_ow <= 64 && d.tail.n_operands == 0;
}

int64_t pml_hip_conv2d_dispatch(const pml_hip_conv2d_desc* d) {
  if (!d) {
    fail("null descriptor");
    return 0;
  }
  const int kind = mfma_kind_of(d->in_dtype, d->flags);
  if (kind < 0) {
    fail("conv2d: in_dtype must be F32, BF16 or I8");
    return 0;
  }
  const bool out_ok = (kind == KIND_I8) ? d->out_dtype == PML_HIP_I32
                                        : (d->out_dtype == PML_HIP_F32 || (kind == KIND_BF16 && d->out_dtype == PML_HIP_BF16));
  if (!out_ok) {
    fail("conv2d: out_dtype does not fit in_dtype");
    return 0;
  }
  if ((d->flags & ~(PML_HIP_FP32_AS_BF16X3 | kScheduleBits | kMaxpoolBits)) != 0 || ((d->flags & PML_HIP_FP32_AS_BF16X3) && d->in_dtype != PML_HIP_F32) ||
      !schedule_bits_ok(d->flags) || (PML_HIP_FLAG_MAXPOOL_OF(d->flags) != 0 && (PML_HIP_FLAG_MAXPOOL_OF(d->flags) & 1) == 0)) {
    fail("conv2d: flags may only hold PML_HIP_FP32_AS_BF16X3 (with in_dtype F32) and schedule overrides that name an existing tile and path");
    return 0;
  }
  if (d->n <= 0 || d->h <= 0 || d->w <= 0 || d->ci <= 0 || d->co <= 0 || d->kh <= 0 || d->kw <= 0 || d->oh <= 0 ||
      d->ow <= 0 || d->stride_h <= 0 || d->stride_w <= 0 || d->dil_h <= 0 || d->dil_w <= 0) {
    fail("conv2d: bad geometry");
    return 0;
  }
  const int es = dt_size(d->in_dtype);
  // channels that do not fill 16-byte vectors: stride 2 runs over 2x2 pixel blocks, anything else over a patch matrix
  const bool odd_channels = (d->ci * es) % 16 != 0;
  const int path = PML_HIP_FLAG_CONV_OF(d->flags);
  const bool via_s2d = odd_channels && d->stride_h == 2 && d->stride_w == 2 && d->dil_h == 1 && d->dil_w == 1 &&
                       es >= 2 && d->ci <= 16 && path != PML_HIP_CONV_PATCHES;
  const bool via_patches = odd_channels && !via_s2d;
  if (d->n * d->h * d->w * d->ci >= ((int64_t)1 << 40) || d->h * d->w * d->ci * es >= ((int64_t)1 << 31) ||
      d->kh * d->kw * d->ci * es >= ((int64_t)1 << 31)) {
    fail("conv2d: tensor too large");
    return 0;
  }
  if (!valid_tail(d->tail)) {
    fail("conv2d: malformed tail");
    return 0;
  }
  Plan* p = new Plan();
  p->kind = PLAN_CONV;
  p->mfma_kind = kind;
  p->conv = *d;
  const int64_t M = d->n * d->oh * d->ow;
  const int64_t K = d->kh * d->kw * d->ci;
  const TailForm tail = tail_form(d->tail, d->out_dtype, d->c_dtype, true, false);
  p->tile = choose_tile(M, d->co, K * es, kind, tail, PML_HIP_FLAG_TILE_OF(d->flags));
  p->bt_ld = K;
  if (via_s2d) {
    const int v = 16 / es;
    p->s2d_h = (int)(d->h + 1) / 2;
    p->s2d_w = (int)(d->w + 1) / 2;
    p->s2d_ch = (int)(4 * d->ci + v - 1) / v * v;
    p->s2d_ka = (int)(d->kh + (d->pad_h & 1) + 1) / 2;
    p->s2d_kaw = (int)(d->kw + (d->pad_w & 1) + 1) / 2;
    const int64_t k2 = (int64_t)p->s2d_ka * p->s2d_kaw * p->s2d_ch;
    p->tile = choose_tile(M, d->co, k2 * es, kind, tail, PML_HIP_FLAG_TILE_OF(d->flags), /*allow_split=*/false);
    p->bt_ld = k2;
    p->via_s2d = true;
  }
  if (via_patches) {
    // rows padded with zeros to whole 16-byte vectors on both GEMM operands
    const int64_t v = 16 / es;
    p->kpad = (K + v - 1) / v * v;
    p->bt_ld = p->kpad;
    if (!(p->patches = p->hold((size_t)M * p->kpad * es))) {
      delete p;
      fail("conv2d: cannot allocate the patch matrix");
      return 0;
    }
  }
  if (!via_s2d && PML_HIP_FLAG_TILE_OF(d->flags) < 0)
    p->tile_direct = direct_tile_of(M, d->co, (via_patches ? p->kpad : K) * es, kind, 0, false, /*can_split=*/!via_patches);
  {
    // Filter small enough to stay in LDS: persistent resident-filter kernel (PML_HIP_CONV_IGEMM keeps the generic one).
    int dev = 0;
    hipDeviceProp_t prop;
    if (!odd_channels && kind != KIND_F32X3 && path != PML_HIP_CONV_IGEMM && hipGetDevice(&dev) == hipSuccess &&
        hipGetDeviceProperties(&prop, dev) == hipSuccess) {
      IgemmArgs g;
      conv_args(p, g);
      const size_t lds = conv_halo_prepare(kind, &g, path == PML_HIP_CONV_LDSFILTER);
      if (lds && lds <= prop.sharedMemPerBlock) {
        p->halo_lds = lds;
        p->halo_rows = g.halo_rows;
        p->halo_tiles = g.n_tiles;
        p->halo_variant = g.halo_variant;
        p->n_cus = prop.multiProcessorCount;
      }
    }
  }
  const bool named = path == PML_HIP_CONV_WINDOW;
  double window_us = 0;
  if (!odd_channels && PML_HIP_FLAG_TILE_OF(d->flags) < 0 && (named || (path == PML_HIP_CONV_AUTO && (!p->halo_lds || p->halo_variant == 0)))) {
    p->win = window_shape(p, named, &window_us);
    if (p->win.config >= 0) {
      p->halo_lds = 0;
      p->tile_direct = -1;
    }
  }
  if (!via_s2d && !p->halo_lds && !named && PML_HIP_FLAG_TILE_OF(d->flags) < 0) p->tile_given = given_filter_tile(p, window_us);
  p->bt_bytes = p->win.config >= 0 ? winconv_pack_bytes(es, (int)(d->kh * d->kw), d->ci, d->co) : (size_t)d->co * p->bt_ld * es;
  if (!(p->bt = p->hold(p->bt_bytes)) || hipMemset(p->bt, 0, p->bt_bytes) != hipSuccess) {
    delete p;
    fail("conv2d: cannot allocate the packed filter");
    return 0;
  }
  if (!via_s2d && !via_patches && !p->halo_lds && p->win.config < 0 && p->tile_direct < 0) prepare_split(p, M, d->co, conv_slabs(*d));
  const int lds_tile = p->tile;  // (named in the text beside the direct tile that takes its place)
  if (p->tile == TILE_64x64_KSPLIT && !p->ws) p->tile = TILE_64x64;
  // (whole 128-byte chunks per filter tap, so that no chunk of heads + remainders straddles two taps)
  p->b_split = kind == KIND_F32X3 && !via_s2d && !via_patches && d->ci % 32 == 0 && !p->ws;
  const std::string kernel = p->win.config >= 0 ? winconv_text(p->win)
                             : std::string("tile=") + (p->halo_lds ? (p->halo_variant == 3 ? "256x64 resident filter, in registers" : p->halo_variant ? "256x64 resident filter, pipelined 3x3" : "256x64 resident filter")
                                                                   : tile_name(p->tile_direct >= 0 ? lds_tile : p->tile));
  char buf[256];
  std::snprintf(buf, sizeof buf, "conv2d %s n=%lld %lldx%lldx%lld k=%lldx%lld co=%lld -> %lldx%lld (implicit gemm m=%lld n=%lld k=%lld) %s",
                d->in_dtype == PML_HIP_F32 ? "f32" : d->in_dtype == PML_HIP_BF16 ? "bf16" : "i8", (long long)d->n,
                (long long)d->h, (long long)d->w, (long long)d->ci, (long long)d->kh, (long long)d->kw, (long long)d->co,
                (long long)d->oh, (long long)d->ow, (long long)M, (long long)d->co, (long long)K, kernel.c_str());
  p->text = buf;
  if (kind == KIND_F32X3) p->text += " mfma=3 x f32_32x32x16_bf16 (fp32 split into bf16 head + remainder)";
  if (p->tile_direct >= 0 && !p->halo_lds) p->text += std::string(", direct tile=") + tile_name(p->tile_direct);
  if (p->tile_given >= 0) p->text += std::string(kFilterLies) + (p->tile_given == TILE_16x16_W8 ? "16x64" : "32x64") + " (8 wavefronts sharing K)";
  if (via_patches) p->text += " via patch matrix (k padded to " + std::to_string(p->kpad) + ")";
  if (!p->halo_lds && p->win.config < 0 && !via_s2d) {
    IgemmArgs g;
    conv_args(p, g);
    if (via_patches) g.K = g.lda = p->kpad;
    g.ws = p->ws;
    const int tile = p->tile_direct >= 0 ? p->tile_direct : p->tile;
    p->text += stream_text(kind, !via_patches, g, d->init_kind != 0, d->tail, tile, true, tile, via_patches ? 0 : d->co);
  }
  if (via_s2d) {
    p->text += " over 2x2 pixel blocks (" + std::to_string(p->s2d_ka) + "x" + std::to_string(p->s2d_kaw) + " block taps of " +
               std::to_string(p->s2d_ch) + " channels, k=" + std::to_string(p->bt_ld) + ")";
    IgemmArgs g;
    conv_args(p, g);
    if (path != PML_HIP_CONV_IGEMM && conv_blocks4x4_prepare(kind, g)) p->text += ", row by row with the filter in registers";
  }
  if (PML_HIP_FLAG_MAXPOOL_OF(d->flags)) {
    if (!conv2d_takes_maxpool(p)) {
      delete p;
      fail("conv2d: the fused max-pool needs the row-walking kernel (see pml_hip_conv2d_takes_maxpool) and a convolution result of at least 3 x 3 and at most 128 pixels a row");
      return 0;
    }
    IgemmArgs g;
    conv_args(p, g);
    p->text += " + max-pool 3x3 stride 2 -> " + std::to_string(g.pool_oh) + "x" + std::to_string(g.pool_ow);
  }
  return (int64_t)(intptr_t)p;
}

int pml_hip_conv2d_takes_maxpool(const pml_hip_conv2d_desc* d) {
  if (!d || !PML_HIP_FLAG_MAXPOOL_OF(d->flags)) return 0;
  const int kind = mfma_kind_of(d->in_dtype, d->flags);
  if (kind != KIND_BF16 || d->n <= 0 || d->h <= 0 || d->w <= 0 || d->ci <= 0 || d->co <= 0 || d->kh <= 0 || d->kw <= 0 || d->oh <= 0 ||
      d->ow <= 0 || !valid_tail(d->tail))
    return 0;
  // the plan's fields that conv_args reads, without any of its allocations
  Plan p;
  p.kind = PLAN_CONV;
  p.mfma_kind = kind;
  p.conv = *d;
  const int es = 2, v = 8;
  const bool via_s2d = (d->ci * es) % 16 != 0 && d->stride_h == 2 && d->stride_w == 2 && d->dil_h == 1 && d->dil_w == 1 && d->ci <= 16 &&
                       PML_HIP_FLAG_CONV_OF(d->flags) != PML_HIP_CONV_PATCHES;
  if (!via_s2d) return 0;
  p.s2d_h = (int)(d->h + 1) / 2;
  p.s2d_w = (int)(d->w + 1) / 2;
  p.s2d_ch = (int)(4 * d->ci + v - 1) / v * v;
  p.s2d_ka = (int)(d->kh + (d->pad_h & 1) + 1) / 2;
  p.s2d_kaw = (int)(d->kw + (d->pad_w & 1) + 1) / 2;
  p.bt_ld = (int64_t)p.s2d_ka * p.s2d_kaw * p.s2d_ch;
  p.via_s2d = true;
  return conv2d_takes_maxpool(&p) ? 1 : 0;
}

int pml_hip_conv2d_invoke(int64_t plan, const void* input, const void* filter, void* output, const void* init,
                          const void* const* operands, void* const* outs, pml_hip_stream s) {
  Plan* p = (Plan*)(intptr_t)plan;
  if (!p || p->kind != PLAN_CONV) return fail("conv2d_invoke: not a conv2d plan");
  const pml_hip_conv2d_desc& d = p->conv;
  if (!input || !output) return fail("conv2d_invoke: null operand");
  if (!filter && !p->packed) return fail("conv2d_invoke: filter is null and no packed filter exists");
  if (!p->patches && !p->via_s2d && ((uintptr_t)input & 15) != 0) return fail("conv2d_invoke: input must be 16-byte aligned");
  if (d.init_kind && !init) return fail("conv2d_invoke: the plan expects an initial value");
  const int es = dt_size(d.in_dtype);
  const int64_t K = d.kh * d.kw * d.ci;
  // the HWCK filter is a row-major [K][CO] matrix; the pipelined resident-filter kernel transposes it itself
  const bool raw_filter = filter && p->halo_lds && p->halo_variant && p->mfma_kind != KIND_I8;
  IgemmArgs g;
  conv_args(p, g);
  if (raw_filter) {
    if (((uintptr_t)filter & 15) != 0) return fail("conv2d_invoke: filter must be 16-byte aligned");
    g.Bt = filter;
    g.ldbt = d.co;
    g.b_raw = 1;
  } else if (!filter && p->reg_image && p->halo_lds && p->halo_variant == 3) {
    g.Bt = p->reg_image;
    g.b_raw = 2;
  }
  g.A = input;
  g.C = output;
  g.init = d.init_kind ? init : nullptr;
  for (int i = 0; i < d.tail.n_operands; ++i) {
    if (!operands || !operands[i]) return fail("conv2d_invoke: missing tail operand");
    g.operands[i] = operands[i];
  }
  for (int i = 0; i < PML_HIP_MAX_EPI_OPERANDS; ++i) g.outs[i] = outs ? outs[i] : nullptr;
  // the vector tails need 16-byte aligned operands and extra outputs; otherwise the interpreter runs
  if (g.tail_mode == 2 && ((uintptr_t)g.operands[0] & 15) != 0) g.tail_mode = 0;
  if (g.tail_mode == 3 || g.tail_mode == 4) {
    for (int i = 0; i < d.tail.n_operands; ++i)
      if (((uintptr_t)g.operands[i] & 15) != 0) g.tail_mode = 0;
    for (int i = 0; i < PML_HIP_MAX_EPI_OPERANDS; ++i)
      if (((uintptr_t)g.outs[i] & 15) != 0) g.tail_mode = 0;
  }
  for (int i = 0; i < d.tail.n_ops; ++i)
    if (d.tail.ops[i].opcode == PML_HIP_EPI_STORE && !g.outs[d.tail.ops[i].operand])
      return fail("conv2d_invoke: missing extra output");
  int tile = p->tile_direct >= 0 ? p->tile_direct : p->tile;
  // (a 1x1 convolution whose rows stream takes the filter as it lies; a packed one stays what later calls use)
  const bool given_filter = filter && !p->packed && !p->patches && !p->via_s2d && !p->halo_lds && p->win.config < 0 && streams_given(p->mfma_kind, tile, true, filter, d.co, g);
  // A filter that comes with the call and that no packed one is kept beside: direct tiles read it as it lies.  (Behind a patch
  // matrix whose rows are padded, the filter has to end on a whole word: what the word holds besides would meet the padding.)
  const int lies_tile = PML_HIP_FLAG_TILE_OF(d.flags) >= 0 ? p->tile : p->tile_given;
  const bool as_it_lies = filter && !given_filter && !p->packed && !p->via_s2d && !p->halo_lds && p->mfma_kind != KIND_F32X3 &&
                          (lies_tile == TILE_16x16_W8 || lies_tile == TILE_32x32_W8) && ((uintptr_t)filter & (es - 1)) == 0 &&
                          (p->patches ? p->kpad : K) * d.co * es < ((int64_t)1 << 31) && (!p->patches || (((uintptr_t)filter + (uintptr_t)(K * d.co * es)) & 3) == 0);
  if (as_it_lies) {
    tile = lies_tile;
    g.Bt = filter;
    g.ldbt = d.co;
    g.b_kn = 1;
    g.b_rows = (int)K;
  }
  if (filter && !raw_filter && !given_filter && !as_it_lies) {
    if (check(pack_conv_filter(p, filter, (hipStream_t)s), "pack_conv_filter")) return 1;
    // (a filter that arrives with the call replaces the packed one; its register-order copy follows it)
    if (p->reg_image && check(regfilter_image_launch(p->bt, p->bt_ld * es, p->reg_image, (hipStream_t)s), "regfilter_image_launch")) return 1;
  }
  if (p->patches) {
    Im2colArgs ic;
    ic.in = input;
    ic.out = p->patches;
    ic.M = g.M;
    ic.K = (int)K;
    ic.kpad = (int)p->kpad;
    ic.H = g.H, ic.W = g.W, ic.CI = g.CI, ic.OH = g.OH, ic.OW = g.OW, ic.KH = g.KH, ic.KW = g.KW;
    ic.SH = g.SH, ic.SW = g.SW, ic.PH = g.PH, ic.PW = g.PW, ic.DH = g.DH, ic.DW = g.DW;
    if (check(im2col_launch(es, ic, (hipStream_t)s), "im2col_launch")) return 1;
    g.A = p->patches;
    g.lda = p->kpad;
    g.K = p->kpad;
    return check(igemm_launch(p->mfma_kind, tile, false, g, (hipStream_t)s), "igemm_launch");
  }
  if (p->via_s2d) {
    // 4x4 block taps onto 64 channels (the 7x7x3 stride-2 head of an image network): the kernel that walks down
    // the rows with the filter in registers (PML_HIP_CONV_IGEMM keeps the implicit GEMM).  From a 3-channel bf16
    // image of even width it builds the 2x2 pixel blocks itself, row by row, and the re-blocking launch is skipped.
    const int path = PML_HIP_FLAG_CONV_OF(d.flags);
    const size_t lds = path == PML_HIP_CONV_IGEMM ? 0 : conv_blocks4x4_prepare(p->mfma_kind, g);
    const bool from_image = lds && d.ci == 3 && d.w % 2 == 0 && ((uintptr_t)input & 3) == 0 && path != PML_HIP_CONV_BLOCKS;
    if (!from_image) {
      {
        std::lock_guard<std::mutex> lock(p->s2d_mutex);
        // 256 spare bytes: a K-run that starts left of the image is addressed (never read) below the buffer's end only
        if (!p->s2d) p->s2d = p->hold((size_t)d.n * p->s2d_h * p->s2d_w * p->s2d_ch * es + 256);
        if (!p->s2d) return fail("conv2d_invoke: cannot allocate the re-blocked input");
      }
      g.A = p->s2d;
      S2dArgs sa;
      s2d_args(p, sa);
      sa.in = input;
      sa.out = p->s2d;
      if (check(s2d_input_launch(es, sa, (hipStream_t)s), "s2d_input_launch")) return 1;
    } else {
      g.raw_in = input;
      g.raw_h = (int)d.h;
      g.raw_w = (int)d.w;
    }
    if (lds) return check(conv_blocks4x4_launch(g, lds, device_cus(), (hipStream_t)s), "conv_blocks4x4_launch");
    return check(igemm_launch(p->mfma_kind, p->tile, true, g, (hipStream_t)s), "igemm_launch");
  }
  if (p->win.config >= 0 && !as_it_lies) return check(winconv_launch(p->mfma_kind, g, p->win, (hipStream_t)s), "winconv_launch");
  if (p->halo_lds)
    return check(conv_halo_launch(p->mfma_kind, g, p->halo_lds, p->n_cus, (hipStream_t)s), "conv_halo_launch");
  if (!as_it_lies) split_args(p, g);
  if (conv_tap_runs(d)) {
    g.pix_pitch = (int)(d.ci * es);
    g.CI = (int)(d.kw * d.ci);
    g.KW = 1;
  }
  return check(igemm_launch(p->b_split ? KIND_F32X3P : p->mfma_kind, tile, true, g, (hipStream_t)s), "igemm_launch");
}

int pml_hip_gemm_pack_b(int64_t plan, const void* b, pml_hip_stream s) {
  Plan* p = (Plan*)(intptr_t)plan;
  if (!p || p->kind != PLAN_GEMM || !b) return fail("gemm_pack_b: bad argument");
  const pml_hip_gemm_desc& d = p->gemm;
  if (d.b_layout) return fail("gemm_pack_b: an [N][K] right-hand side needs no packing");
  const size_t es = dt_size(d.in_dtype);
  if (p->b_kn) {
    if (check(hipMemcpy2DAsync(p->bt, d.n * es, b, d.ldb * es, d.n * es, d.k, hipMemcpyDeviceToDevice, (hipStream_t)s), "copy of the right-hand side"))
      return 1;
  } else if (check(transpose_pack((int)es, b, p->bt, d.k, d.n, d.ldb, p->bt_ld, (hipStream_t)s), "transpose_pack")) {
    return 1;
  }
  p->bt_is_kn = p->b_kn;
  if (p->b_split && check(split_rows_launch(p->bt, d.n, p->bt_ld, d.k, (hipStream_t)s), "split_rows_launch")) return 1;
  p->bt_is_split = p->b_split;
  if (pack_panel(p, b, false, (hipStream_t)s)) return 1;
  p->packed = true;
  if (p->direct.rows >= 0 && p->ws) {
    // (its invokes take the direct tile from now on; one that brings a right-hand side all the same does not split K)
    p->drop(&p->ws, (size_t)p->sk_splits * d.m * p->sk_pitch * 4);
    p->tile = TILE_64x64;
  }
  return 0;
}

int pml_hip_probe_mfma(int random_data, int iters, double* tflops, double* core_mhz) {
  if (iters <= 0 || iters > 100000) return fail("probe_mfma: iters out of range");
  const int blocks = device_cus();
  float* sink = nullptr;
  unsigned long long* clk = nullptr;
  hipEvent_t e0 = nullptr, e1 = nullptr;
  int rc = 1;
  do {
    if (check(hipMalloc((void**)&sink, 64), "hipMalloc") || check(hipMalloc((void**)&clk, 64), "hipMalloc")) break;
    if (check(hipEventCreate(&e0), "hipEventCreate") || check(hipEventCreate(&e1), "hipEventCreate")) break;
    if (check(mfma_probe_launch(blocks, 16, random_data, sink, clk, nullptr), "mfma_probe_launch")) break;  // warm-up
    if (check(hipEventRecord(e0, nullptr), "hipEventRecord")) break;
    if (check(mfma_probe_launch(blocks, iters, random_data, sink, clk, nullptr), "mfma_probe_launch")) break;
    if (check(hipEventRecord(e1, nullptr), "hipEventRecord") || check(hipEventSynchronize(e1), "hipEventSynchronize")) break;
    float ms = 0;
    if (check(hipEventElapsedTime(&ms, e0, e1), "hipEventElapsedTime")) break;
    unsigned long long host_clk[2] = {0, 0};
    if (check(hipMemcpy(host_clk, clk, sizeof host_clk, hipMemcpyDeviceToHost), "hipMemcpy")) break;
    const double mfmas = (double)iters * 4 * 8 * 8 * blocks;  // rounds x K-blocks x MFMAs per wavefront x wavefronts x workgroups
    if (tflops) *tflops = mfmas * 32768.0 / (ms * 1e-3) / 1e12;
    if (core_mhz) *core_mhz = host_clk[1] ? (double)host_clk[0] / ((double)host_clk[1] / 100.0) : 0.0;
    rc = 0;
  } while (false);
  if (e0) (void)hipEventDestroy(e0);
  if (e1) (void)hipEventDestroy(e1);
  if (sink) (void)hipFree(sink);
  if (clk) (void)hipFree(clk);
  return rc;
}

const char* pml_hip_tile_name(int tile) { return tile >= 0 && tile < PML_HIP_TILE_COUNT_ ? kTileShort[tile] : nullptr; }
int pml_hip_tile_by_name(const char* name) {
  if (!name) return -1;
  for (int t = 0; t < PML_HIP_TILE_COUNT_; ++t)
    if (std::strcmp(name, kTileShort[t]) == 0) return t;
  return -1;
}

int pml_hip_tile_of_workgroup(int tiles_m, int tiles_n, int workgroup, int* tile_m, int* tile_n) {
  if (tiles_m <= 0 || tiles_n <= 0 || (int64_t)tiles_m * tiles_n >= ((int64_t)1 << 31) || workgroup < 0 ||
      workgroup >= tiles_m * tiles_n || !tile_m || !tile_n)
    return fail("tile_of_workgroup: bad argument");
  const TileOrder o = make_tile_order(tiles_m, tiles_n);
  tile_of(o, (unsigned)workgroup, tile_m, tile_n);
  return 0;
}

int pml_hip_gemm_pack_b2(int64_t plan, const void* b2, pml_hip_stream s) {
  Plan* p = (Plan*)(intptr_t)plan;
  if (!p || p->kind != PLAN_GEMM || !b2 || p->gemm.k2 <= 0) return fail("gemm_pack_b2: bad argument");
  const pml_hip_gemm_desc& d = p->gemm;
  if (d.b_layout) return fail("gemm_pack_b2: an [N][K] right-hand side needs no packing");
  if (check(transpose_pack(dt_size(d.in_dtype), b2, p->bt2, d.k2, d.n, d.ldb2, d.k2, (hipStream_t)s), "transpose_pack")) return 1;
  if (pack_panel(p, b2, true, (hipStream_t)s)) return 1;
  p->packed2 = true;
  return 0;
}

int pml_hip_conv2d_pack_filter(int64_t plan, const void* filter, pml_hip_stream s) {
  Plan* p = (Plan*)(intptr_t)plan;
  if (!p || p->kind != PLAN_CONV || !filter) return fail("conv2d_pack_filter: bad argument");
  const pml_hip_conv2d_desc& d = p->conv;
  if (check(pack_conv_filter(p, filter, (hipStream_t)s), "pack_conv_filter")) return 1;
  if (p->halo_lds && p->halo_variant == 3 && regfilter_takes_image((int)d.ow)) {
    // the register-filter kernel takes a constant filter in its own register order: no trip through LDS per launch
    if (!p->reg_image && !(p->reg_image = p->hold(kRegfilterImageBytes))) return fail("conv2d_pack_filter: cannot allocate the filter in register order");
    if (check(regfilter_image_launch(p->bt, p->bt_ld * dt_size(d.in_dtype), p->reg_image, (hipStream_t)s), "regfilter_image_launch")) return 1;
  }
  p->packed = true;
  return 0;
}

// ---------------------------------------------------------------------------
// operations along rows
// ---------------------------------------------------------------------------

int pml_hip_rows_takes(const pml_hip_rows_desc* d) {
  if (!d || (d->dtype != PML_HIP_F32 && d->dtype != PML_HIP_BF16) || d->rows < 0 || d->cols < 0 || d->cols > (1 << 20) || d->n_steps < 0 ||
      d->n_steps > PML_HIP_ROWS_STEPS || d->n_vectors < 0 || d->n_vectors > PML_HIP_ROWS_VECTORS || d->n_in < 0 || d->n_in > PML_HIP_ROWS_IO ||
      d->n_out < 0 || d->n_out > PML_HIP_ROWS_IO)
    return 0;
  auto operand = [&](int kind, int index, bool scalar) {
    switch (kind) {
      case PML_HIP_ROWS_NONE: case PML_HIP_ROWS_IMM: return true;
      case PML_HIP_ROWS_VECTOR: return !scalar && index >= 0 && index < d->n_vectors;
      case PML_HIP_ROWS_SCALAR: return index >= 0 && index < PML_HIP_ROWS_SCALARS;
      case PML_HIP_ROWS_FULL: case PML_HIP_ROWS_COLUMNS: return !scalar && index >= 0 && index < d->n_in;
      case PML_HIP_ROWS_ROW: case PML_HIP_ROWS_ONE: return index >= 0 && index < d->n_in;
    }
    return false;
  };
  for (int i = 0; i < d->n_steps; ++i) {
    const pml_hip_rows_step& s = d->steps[i];
    bool ok = s.dst >= 0;
    switch (s.kind) {
      case PML_HIP_ROWS_MAP: ok = ok && s.dst < d->n_vectors && operand(s.a_kind, s.a, false) && operand(s.b_kind, s.b, false); break;
      case PML_HIP_ROWS_MAP_SCALAR: ok = ok && s.dst < PML_HIP_ROWS_SCALARS && operand(s.a_kind, s.a, true) && operand(s.b_kind, s.b, true); break;
      case PML_HIP_ROWS_REDUCE: ok = ok && s.dst < PML_HIP_ROWS_SCALARS && operand(s.a_kind, s.a, false) && s.opcode >= PML_HIP_AGG_ADD && s.opcode <= PML_HIP_AGG_MUL; break;
      case PML_HIP_ROWS_STORE: ok = ok && s.dst < d->n_out && operand(s.a_kind, s.a, false); break;
      case PML_HIP_ROWS_STORE_SCALAR: ok = ok && s.dst < d->n_out && s.a >= 0 && s.a < PML_HIP_ROWS_SCALARS; break;
      default: ok = false;
    }
    if (!ok) return 0;
  }
  int lanes = 0;
  if (rows_program_lds(*d, &lanes) > 158 * 1024) return 0;
  return (d->rows + 256 / lanes - 1) / (256 / lanes) <= kMaxLaunchThreads / 256 ? 1 : 0;
}

int pml_hip_rows(const pml_hip_rows_desc* d, const void* const* in, void* const* out, pml_hip_stream s) {
  if (!pml_hip_rows_takes(d)) return fail("rows: malformed program, or rows too long for it");
  RowsProgramArgs a;
  std::memset(&a, 0, sizeof a);
  a.d = *d;
  for (int i = 0; i < d->n_in; ++i) {
    if (!in || !in[i]) return fail("rows: missing input");
    a.in[i] = in[i];
  }
  for (int i = 0; i < d->n_out; ++i) {
    if (!out || !out[i]) return fail("rows: missing output");
    a.out[i] = out[i];
  }
  return check(rows_program_launch(a, (hipStream_t)s), "rows_program_launch");
}

int pml_hip_argmax_rows(int dtype, int64_t rows, int64_t cols, const void* x, int32_t* out, pml_hip_stream s) {
  if ((dtype != PML_HIP_F32 && dtype != PML_HIP_BF16) || rows < 0 || cols <= 0 || cols > 0x7fffffff) return fail("argmax_rows: bad type or sizes");
  if (rows && (!x || !out)) return fail("argmax_rows: null operand");
  return in_row_runs(rows, [&](int64_t first, int64_t n) {
    return check(argmax_rows_launch(dtype, n, cols, (const char*)x + first * cols * dt_size(dtype), out + first, (hipStream_t)s), "argmax_rows_launch");
  });
}

int pml_hip_topk_rows(int dtype, int descending, int64_t rows, int64_t cols, int k, const void* x, void* values, int32_t* positions,
                      pml_hip_stream s) {
  if (dt_size(dtype) == 0 || dt_size(dtype) == 8 || rows < 0 || k < 0 || k > cols || cols > PML_HIP_MAX_SORT_LINE) return fail("topk_rows: bad type or sizes");
  if (rows && k && (!x || (!values && !positions))) return fail("topk_rows: null operand");
  return in_row_runs(rows, [&](int64_t first, int64_t n) {
    return check(topk_rows_launch(dtype, descending != 0, n, cols, k, (const char*)x + first * cols * dt_size(dtype),
                                  values ? (char*)values + first * k * dt_size(dtype) : nullptr, positions ? positions + first * k : nullptr, (hipStream_t)s),
                 "topk_rows_launch");
  });
}

// ---------------------------------------------------------------------------
// products over free strides, gradients of a convolution
// ---------------------------------------------------------------------------

int pml_hip_product_takes_tail(const pml_hip_epilogue* t, int out_dtype) {
  if (!t || !valid_tail(*t) || t->n_ops > 4 || (out_dtype != PML_HIP_F32 && out_dtype != PML_HIP_BF16)) return 0;
  for (int i = 0; i < t->n_ops; ++i) {
    const pml_hip_epi_op& op = t->ops[i];
    switch (op.opcode) {
      case PML_HIP_EPI_ADD: case PML_HIP_EPI_SUB: case PML_HIP_EPI_RSUB: case PML_HIP_EPI_MUL: case PML_HIP_EPI_DIV:
      case PML_HIP_EPI_RDIV: case PML_HIP_EPI_MAX: case PML_HIP_EPI_MIN: case PML_HIP_EPI_MAX_GT: case PML_HIP_EPI_RELU: case PML_HIP_EPI_NEG:
        break;
      default: return 0;
    }
    if (op.dtype != out_dtype || (op.operand_kind == PML_HIP_OPND_TENSOR && t->operand_dtype[op.operand] != out_dtype)) return 0;
  }
  return 1;
}

// Grid, split and workspace of a plan whose `strided` arguments name the problem; false with the error text set.
static bool prepare_strided(Plan* p) {
  StridedArgs& a = p->strided;
  strided_plan(&a, p->strided_bf, p->strided_conv, device_cus(), &p->strided_mi);
  a.ws = nullptr;
  if (a.splits > 1) p->ws = p->hold((size_t)a.splits * a.ws_rows * a.ws_pitch * 4);
  if (a.splits > 1 && !p->ws) {  // (no memory for the partial results: the K loop is not split)
    a.splits = 1;
    a.k_per_split = (a.K + 63) / 64 * 64;
  }
  a.ws = (float*)p->ws;
  int64_t nb = (int64_t)a.tiles_m * a.tiles_n;
  for (int d = 0; d < a.n_batch; ++d) nb *= a.batch[d];
  if (nb > kMaxLaunchThreads / 256) {
    fail("product: too many result tiles for one launch");
    return false;
  }
  return true;
}

// nullptr, or what is wrong with a product's types, sizes and strides; *batches: their number
static const char* product_fault(const pml_hip_product_desc* d, int64_t* batches) {
  if (!d) return "null descriptor";
  const bool bf = d->in_dtype == PML_HIP_BF16;
  if ((d->in_dtype != PML_HIP_F32 && !bf) || (d->out_dtype != PML_HIP_F32 && (!bf || d->out_dtype != PML_HIP_BF16)))
    return "product: in_dtype must be F32 or BF16 and out_dtype F32 or in_dtype";
  bool ok = d->m > 0 && d->n > 0 && d->k > 0 && d->n_batch >= 0 && d->n_batch <= 3 && d->a_ms >= 0 && d->a_ks >= 0 && d->b_ks >= 0 &&
            d->b_ns >= 0 && d->c_ms >= 0 && d->row_len > 0 && (d->init_kind == 0 || d->init_kind == 1);
  *batches = 1;
  for (int i = 0; ok && i < d->n_batch; ++i) {
    ok = d->batch[i] > 0 && d->a_batch[i] >= 0 && d->b_batch[i] >= 0 && d->c_batch[i] >= 0 && d->batch[i] < ((int64_t)1 << 31);
    if (ok) *batches *= d->batch[i];
    ok = ok && *batches < ((int64_t)1 << 31);
  }
  return ok ? nullptr : "product: bad sizes or strides";
}

// The kernel arguments that sizes and strides fix.
static StridedArgs product_args(const pml_hip_product_desc* d) {
  StridedArgs a;
  std::memset(&a, 0, sizeof a);
  a.M = d->m, a.N = d->n, a.K = d->k;
  a.a_ms = d->a_ms, a.a_ks = d->a_ks, a.b_ks = d->b_ks, a.b_ns = d->b_ns, a.c_ms = d->c_ms;
  a.row_len = d->row_len;
  a.n_batch = d->n_batch;
  a.out_bf16 = d->out_dtype == PML_HIP_BF16;
  for (int i = 0; i < d->n_batch; ++i) {
    a.batch[i] = d->batch[i];
    a.a_batch[i] = d->a_batch[i];
    a.b_batch[i] = d->b_batch[i];
    a.c_batch[i] = d->c_batch[i];
  }
  return a;
}

int pml_hip_product_pays(const pml_hip_product_desc* d) {
  int64_t batches = 1;
  if (product_fault(d, &batches)) return 0;
  const bool bf = d->in_dtype == PML_HIP_BF16;
  StridedArgs a = product_args(d);
  int mi = 1;
  double us = 0;
  const int n_cus = 256;  // (of the whole device; asking for it would start the GPU runtime in a process that only plans)
  strided_plan(&a, bf, false, n_cus, &mi);
  (void)product_direct_rows(a, bf, mi, n_cus, &us);
  return us <= contract_product_us((double)batches * (double)d->m * (double)d->n, (double)d->k) ? 1 : 0;
}

int64_t pml_hip_product_dispatch(const pml_hip_product_desc* d) {
  int64_t batches = 1;
  if (const char* fault = product_fault(d, &batches)) {
    fail(fault);
    return 0;
  }
  const bool bf = d->in_dtype == PML_HIP_BF16;
  if (!pml_hip_product_takes_tail(&d->tail, d->out_dtype)) {
    fail("product: the tail holds steps this kernel does not run");
    return 0;
  }
  Plan* p = new Plan();
  p->kind = PLAN_PRODUCT;
  p->strided_bf = bf;
  p->strided = product_args(d);
  StridedArgs& a = p->strided;
  a.init_rs = d->init_row_stride;
  a.init_cs = d->init_col_stride;
  p->gemm.init_kind = d->init_kind;
  p->gemm.tail = d->tail;
  a.n_ops = d->tail.n_ops;
  for (int i = 0; i < d->tail.n_ops; ++i) {
    const pml_hip_epi_op& op = d->tail.ops[i];
    StridedOp& o = a.ops[i];
    o.opcode = op.opcode;
    o.imm = op.operand_kind != PML_HIP_OPND_IMM ? 0.f : a.out_bf16 ? host_round_bf16((float)op.imm) : (float)op.imm;
    if (op.operand_kind == PML_HIP_OPND_TENSOR) {
      o.rs = d->tail.operand_row_stride[op.operand];
      o.cs = d->tail.operand_col_stride[op.operand];
    }
  }
  strided_plan(&a, bf, false, device_cus(), &p->strided_mi);
  double us = 0;
  p->product_rows = product_direct_rows(a, bf, p->strided_mi, device_cus(), &us);
  if (!p->product_rows && !prepare_strided(p)) {
    delete p;
    return 0;
  }
  char buf[256];
  std::snprintf(buf, sizeof buf, "product %s batch=%lld m=%lld n=%lld k=%lld tile=%dx%d splits=%d", bf ? "bf16" : "f32", (long long)batches,
                (long long)d->m, (long long)d->n, (long long)d->k, p->product_rows ? p->product_rows : 64 * p->strided_mi,
                p->product_rows ? 64 : 64 * p->strided_mi, p->product_rows ? 1 : a.splits);
  p->text = buf;
  return (int64_t)(intptr_t)p;
}

int pml_hip_product_invoke(int64_t plan, const void* a, const void* b, void* c, const void* init, const void* const* operands,
                           pml_hip_stream s) {
  Plan* p = (Plan*)(intptr_t)plan;
  if (!p || p->kind != PLAN_PRODUCT) return fail("product_invoke: not a product plan");
  if (!a || !b || !c) return fail("product_invoke: null operand");
  if (p->gemm.init_kind && !init) return fail("product_invoke: the plan expects an initial value");
  StridedArgs g = p->strided;
  g.A = a;
  g.B = b;
  g.C = c;
  g.init = p->gemm.init_kind ? init : nullptr;
  for (int i = 0; i < g.n_ops; ++i) {
    const pml_hip_epi_op& op = p->gemm.tail.ops[i];
    if (op.operand_kind != PML_HIP_OPND_TENSOR) continue;
    if (!operands || !operands[op.operand]) return fail("product_invoke: missing tail operand");
    g.ops[i].ptr = operands[op.operand];
  }
  if (p->product_rows) return check(product_direct_launch(g, p->strided_bf, p->product_rows, (hipStream_t)s), "product_direct_launch");
  return check(strided_launch(g, p->strided_bf, false, p->strided_mi, (hipStream_t)s), "strided_launch");
}

int pml_hip_conv2d_grad_takes(const pml_hip_conv2d_desc* d, int which) {
  if (!d || (which != 0 && which != 1) || (d->in_dtype != PML_HIP_F32 && d->in_dtype != PML_HIP_BF16) || d->out_dtype != d->in_dtype || d->flags != 0 ||
      d->tail.n_ops != 0 || d->init_kind != 0)
    return 0;
  if (d->n <= 0 || d->h <= 0 || d->w <= 0 || d->ci <= 0 || d->kh <= 0 || d->kw <= 0 || d->co <= 0 || d->oh <= 0 || d->ow <= 0 ||
      d->stride_h <= 0 || d->stride_w <= 0 || d->dil_h <= 0 || d->dil_w <= 0)
    return 0;
  const int64_t lim = (int64_t)1 << 31;  // (pixel numbers and offsets inside an image are 32-bit)
  if (d->n * d->oh * d->ow >= lim || d->h * d->w * d->ci >= lim || d->kh * d->kw * d->ci >= lim || d->kh * d->kw * d->co >= lim ||
      d->n * d->h * d->w >= lim || std::llabs(d->pad_h) >= (1 << 20) || std::llabs(d->pad_w) >= (1 << 20) ||
      (d->ow * d->stride_w + std::llabs(d->pad_w) + d->kw) * d->ci >= lim)
    return 0;
  return which == 0 || d->dil_w == 1 || d->kw == 1;
}

int64_t pml_hip_conv2d_grad_dispatch(const pml_hip_conv2d_desc* d, int which) {
  if (!pml_hip_conv2d_grad_takes(d, which)) {
    fail("conv2d_grad: bad geometry, types or options");
    return 0;
  }
  const bool bf = d->in_dtype == PML_HIP_BF16;
  const int es = bf ? 2 : 4;
  Plan* p = new Plan();
  p->kind = PLAN_CONV_GRAD;
  p->conv = *d;
  p->grad_which = which;
  p->strided_bf = bf;
  StridedArgs& a = p->strided;
  std::memset(&a, 0, sizeof a);
  a.row_len = 1;
  char buf[256];
  if (which == 1) {
    p->strided_conv = true;
    a.row_cols = d->kw * d->ci;
    a.M = d->kh * a.row_cols;
    a.N = d->co;
    a.K = d->n * d->oh * d->ow;
    a.b_ks = d->co;
    a.b_ns = 1;
    a.c_ms = d->co;
    a.out_bf16 = bf;
    a.H = (int)d->h, a.W = (int)d->w, a.CI = (int)d->ci, a.OH = (int)d->oh, a.OW = (int)d->ow;
    a.SH = (int)d->stride_h, a.SW = (int)d->stride_w, a.PH = (int)d->pad_h, a.PW = (int)d->pad_w, a.DH = (int)d->dil_h;
    fast_div_magic((unsigned)(d->oh * d->ow), &a.div_per_magic, &a.div_per_shift);
    fast_div_magic((unsigned)d->ow, &a.div_ow_magic, &a.div_ow_shift);
    if (!prepare_strided(p)) {
      delete p;
      return 0;
    }
    std::snprintf(buf, sizeof buf, "conv2d filter gradient %s: %lld pixels x (%lld window values, %lld channels) tile=%dx%d splits=%d", bf ? "bf16" : "f32",
                  (long long)a.K, (long long)a.M, (long long)a.N, 64 * p->strided_mi, 64 * p->strided_mi, a.splits);
    p->text = buf;
    return (int64_t)(intptr_t)p;
  }
  // Data gradient.  Unit stride: the convolution of the gradient with the filter's taps in reverse and its channels'
  // roles exchanged, on the convolution kernels; channel counts that do not fill 16-byte vectors are padded with zeros
  // in a copy of the gradient (one pass over it, against a patch matrix of kh * kw times its size).
  const int64_t v = 16 / es;
  p->co_pad = (d->co + v - 1) / v * v;
  const int64_t back_h = d->dil_h * (d->kh - 1) - d->pad_h, back_w = d->dil_w * (d->kw - 1) - d->pad_w;
  if (d->stride_h == 1 && d->stride_w == 1 && back_h >= 0 && back_w >= 0 && d->n * d->oh * d->ow * p->co_pad * es < ((int64_t)1 << 31)) {
    pml_hip_conv2d_desc c = *d;
    c.h = d->oh, c.w = d->ow, c.ci = p->co_pad, c.co = d->ci, c.oh = d->h, c.ow = d->w;
    c.pad_h = back_h, c.pad_w = back_w;
    c.c_dtype = d->in_dtype;
    p->sub = (Plan*)(intptr_t)pml_hip_conv2d_dispatch(&c);
    if (!p->sub) {
      delete p;
      return 0;
    }
    p->sub->packed = true;  // (every invoke lays the filter out itself)
    p->sub->tile_given = -1;
    if (p->co_pad != d->co && !(p->padded = p->hold((size_t)(d->n * d->oh * d->ow * p->co_pad * es)))) {
      delete p;
      fail("conv2d_grad: cannot allocate the padded gradient");
      return 0;
    }
    if (const size_t at = p->sub->text.find(kFilterLies); at != std::string::npos) p->sub->text.erase(at, p->sub->text.find(')', at) + 1 - at);
    p->text = "conv2d data gradient as a convolution of the gradient: " + p->sub->text;
    return (int64_t)(intptr_t)p;
  }
  // Larger strides: every gradient pixel's product with the whole filter, cols[pixel][ky][kx][ci] in fp32, then a pass
  // that adds the columns up into the image.  (A convolution over the gradient spread out with zeros would multiply
  // stride^2 times as much.)  Columns are made for as many images at a time as fit 256 MiB.
  const int64_t taps_ci = d->kh * d->kw * d->ci, per_image = d->oh * d->ow * taps_ci * 4;
  p->grad_chunk = std::max<int64_t>(1, std::min<int64_t>(d->n, ((int64_t)256 << 20) / per_image));
  p->grad_chunk = std::max<int64_t>(1, std::min(p->grad_chunk, kMaxLaunchThreads / (d->h * d->w * d->ci)));  // (a thread per value at most)
  a.M = p->grad_chunk * d->oh * d->ow;
  a.N = taps_ci;
  a.K = d->co;
  a.a_ms = d->co;
  a.a_ks = 1;
  a.b_ks = 1;
  a.b_ns = d->co;
  a.c_ms = taps_ci;
  if (!(p->cols = p->hold((size_t)(p->grad_chunk * per_image)))) {
    delete p;
    fail("conv2d_grad: cannot allocate the columns");
    return 0;
  }
  if (!prepare_strided(p)) {
    delete p;
    return 0;
  }
  std::snprintf(buf, sizeof buf, "conv2d data gradient %s by columns: product m=%lld n=%lld k=%lld tile=%dx%d splits=%d, %lld images at a time", bf ? "bf16" : "f32",
                (long long)a.M, (long long)a.N, (long long)a.K, 64 * p->strided_mi, 64 * p->strided_mi, a.splits, (long long)p->grad_chunk);
  p->text = buf;
  return (int64_t)(intptr_t)p;
}

int pml_hip_conv2d_grad_invoke(int64_t plan, const void* g, const void* other, void* result, pml_hip_stream s) {
  Plan* p = (Plan*)(intptr_t)plan;
  if (!p || p->kind != PLAN_CONV_GRAD) return fail("conv2d_grad_invoke: not a gradient plan");
  if (!g || !other || !result) return fail("conv2d_grad_invoke: null operand");
  const pml_hip_conv2d_desc& d = p->conv;
  const int es = p->strided_bf ? 2 : 4;
  hipStream_t st = (hipStream_t)s;
  if (p->grad_which == 1) {
    StridedArgs a = p->strided;
    a.A = other;
    a.B = g;
    a.C = result;
    return check(strided_launch(a, p->strided_bf, true, p->strided_mi, st), "strided_launch");
  }
  if (p->sub) {
    const void* const in = p->padded ? p->padded : g;
    const bool window = p->sub->win.config >= 0;
    if (window) {  // (the taps in reverse, the channels' roles exchanged)
      const WinFilter w{(int)(d.kh * d.kw), (int)d.co, (int)d.ci, (d.kh * d.kw - 1) * d.ci * d.co, -d.ci * d.co, 1, d.co};
      if (check(winconv_pack_launch(es, other, w, p->sub->bt, st), "winconv_pack_launch")) return 1;
    }
    if (check(gradient_operands_launch(es, g, p->padded, p->padded ? d.n * d.oh * d.ow : 0, d.co, p->co_pad, other, window ? nullptr : p->sub->bt,
                                       d.kh * d.kw, d.ci, d.co, st),
              "gradient_operands_launch"))
      return 1;
    if (pml_hip_conv2d_invoke((int64_t)(intptr_t)p->sub, in, nullptr, result, nullptr, nullptr, nullptr, s)) return 1;
    ConvBorderArgs b;
    b.g = g, b.f = other, b.out = result;
    b.N = (int)d.n, b.H = (int)d.h, b.W = (int)d.w, b.CI = (int)d.ci, b.OH = (int)d.oh, b.OW = (int)d.ow, b.CO = (int)d.co;
    b.KH = (int)d.kh, b.KW = (int)d.kw, b.PH = (int)d.pad_h, b.PW = (int)d.pad_w, b.DH = (int)d.dil_h, b.DW = (int)d.dil_w;
    // an image row y meets the gradient's rows y + pad - ky * dil
    auto inside = [](int64_t size, int64_t grad, int64_t k, int64_t dil, int64_t pad, int* from, int* to) {
      *from = (int)std::min(size, std::max<int64_t>(0, dil * (k - 1) - pad));
      *to = (int)std::max<int64_t>(*from, std::min(size, grad - pad));
    };
    inside(d.h, d.oh, d.kh, d.dil_h, d.pad_h, &b.y0, &b.y1);
    inside(d.w, d.ow, d.kw, d.dil_w, d.pad_w, &b.x0, &b.x1);
    return check(conv_border_launch(b, p->strided_bf, st), "conv_border_launch");
  }
  const int64_t g_step = d.oh * d.ow * d.co * es, r_step = d.h * d.w * d.ci * es;
  for (int64_t i = 0; i < d.n; i += p->grad_chunk) {
    const int64_t cnt = std::min<int64_t>(p->grad_chunk, d.n - i);
    StridedArgs a = p->strided;
    a.A = (const char*)g + i * g_step;
    a.B = other;
    a.C = p->cols;
    if (cnt != p->grad_chunk) {  // (a last, shorter run: its rows past the end would be another image's)
      a.M = cnt * d.oh * d.ow;
      a.tiles_m = (int)((a.M + 64 * p->strided_mi - 1) / (64 * p->strided_mi));
      a.ws_rows = a.M;
    }
    if (check(strided_launch(a, p->strided_bf, false, p->strided_mi, st), "strided_launch")) return 1;
    Col2imArgs c;
    c.cols = (const float*)p->cols;
    c.out = (char*)result + i * r_step;
    c.N = (int)cnt, c.H = (int)d.h, c.W = (int)d.w, c.CI = (int)d.ci, c.OH = (int)d.oh, c.OW = (int)d.ow, c.KH = (int)d.kh, c.KW = (int)d.kw;
    c.SH = (int)d.stride_h, c.SW = (int)d.stride_w, c.PH = (int)d.pad_h, c.PW = (int)d.pad_w, c.DH = (int)d.dil_h, c.DW = (int)d.dil_w;
    if (check(col2im_launch(c, p->strided_bf, st), "col2im_launch")) return 1;
  }
  return 0;
}

// ---------------------------------------------------------------------------
// depthwise conv, pooling
// ---------------------------------------------------------------------------

int64_t pml_hip_dwconv2d_dispatch(const pml_hip_dwconv2d_desc* d) {
  if (!d) {
    fail("null descriptor");
    return 0;
  }
  if (d->dtype != PML_HIP_F32 && d->dtype != PML_HIP_BF16) {
    fail("dwconv2d: dtype must be F32 or BF16");
    return 0;
  }
  const int V = 16 / dt_size(d->dtype);
  if (d->c <= 0 || d->c % V != 0) {
    fail("dwconv2d: channels must cover whole 16-byte vectors");
    return 0;
  }
  if (d->n <= 0 || d->h <= 0 || d->w <= 0 || d->kh <= 0 || d->kw <= 0 || d->oh <= 0 || d->ow <= 0 ||
      d->stride_h <= 0 || d->stride_w <= 0 || d->dil_h <= 0 || d->dil_w <= 0 || !valid_tail(d->tail)) {
    fail("dwconv2d: bad geometry or tail");
    return 0;
  }
  if (d->out_pitch != 0 && d->out_pitch != d->c &&
      (d->out_pitch < d->c || d->out_pitch % V != 0 || d->tail.n_ops != 0 ||
       d->n * d->oh * d->ow * (int64_t)d->out_pitch >= ((int64_t)1 << 40))) {
    fail("dwconv2d: the output pitch must be at least c, a whole number of 16-byte vectors, and has no tail");
    return 0;
  }
  Plan* p = new Plan();
  p->kind = PLAN_DWCONV;
  p->dw = *d;
  char buf[200];
  std::snprintf(buf, sizeof buf, "dwconv2d %s n=%lld %lldx%lldx%lld k=%lldx%lld -> %lldx%lld (16B channel vectors)",
                d->dtype == PML_HIP_F32 ? "f32" : "bf16", (long long)d->n, (long long)d->h, (long long)d->w,
                (long long)d->c, (long long)d->kh, (long long)d->kw, (long long)d->oh, (long long)d->ow);
  p->text = buf;
  int64_t ysegs, seg_rows;
  if (dwconv2d_walks_rows(*d, device_cus(), &ysegs, &seg_rows)) {
    std::snprintf(buf, sizeof buf, ", window rows walked in registers (%lld runs of %lld rows)", (long long)ysegs, (long long)seg_rows);
    p->text += buf;
  }
  return (int64_t)(intptr_t)p;
}

int pml_hip_dwconv2d_invoke(int64_t plan, const void* input, const void* filter, void* output,
                            const void* const* operands, void* const* outs, pml_hip_stream s) {
  Plan* p = (Plan*)(intptr_t)plan;
  if (!p || p->kind != PLAN_DWCONV) return fail("dwconv2d_invoke: not a dwconv2d plan");
  if (!input || !output) return fail("dwconv2d_invoke: null operand");
  if (!filter && !p->dw_filter) return fail("dwconv2d_invoke: filter is null and no packed filter exists");
  if ((((uintptr_t)input | (uintptr_t)filter | (uintptr_t)output) & 15) != 0)
    return fail("dwconv2d_invoke: buffers must be 16-byte aligned");
  DwconvArgs a;
  std::memset(&a, 0, sizeof a);
  a.d = p->dw;
  a.in = input;
  a.filter = filter ? filter : p->dw_filter;
  a.paired_filter = filter ? nullptr : p->dw_paired;
  a.n_cus = device_cus();
  a.out = output;
  for (int i = 0; i < a.d.tail.n_operands; ++i) {
    if (!operands || !operands[i]) return fail("dwconv2d_invoke: missing tail operand");
    a.operands[i] = operands[i];
  }
  for (int i = 0; i < PML_HIP_MAX_EPI_OPERANDS; ++i) a.outs[i] = outs ? outs[i] : nullptr;
  return check(dwconv2d_launch(a, (hipStream_t)s), "dwconv2d_launch");
}

int pml_hip_dwconv2d_pack_filter(int64_t plan, const void* filter, pml_hip_stream s) {
  Plan* p = (Plan*)(intptr_t)plan;
  if (!p || p->kind != PLAN_DWCONV || !filter) return fail("dwconv2d_pack_filter: bad argument");
  const pml_hip_dwconv2d_desc& d = p->dw;
  const size_t bytes = (size_t)d.kh * d.kw * d.c * dt_size(d.dtype);
  if (!p->dw_filter && !(p->dw_filter = p->hold(bytes))) return fail("dwconv2d_pack_filter: cannot allocate the filter");
  if (check(hipMemcpyAsync(p->dw_filter, filter, bytes, hipMemcpyDeviceToDevice, (hipStream_t)s), "hipMemcpyAsync")) return 1;
  p->drop(&p->dw_paired, (size_t)12 * (d.c / 8) * 4 * 4);
  if (!dwconv2d_takes_paired_filter(d)) return 0;
  // once per filter: its weights are looked at on the host (the paired kernel is for finite weights only) and re-laid there
  std::vector<uint16_t> host(bytes / 2);
  if (check(hipMemcpyAsync(host.data(), p->dw_filter, bytes, hipMemcpyDeviceToHost, (hipStream_t)s), "hipMemcpyAsync") ||
      check(hipStreamSynchronize((hipStream_t)s), "hipStreamSynchronize"))
    return 1;
  std::vector<uint32_t> packed((size_t)12 * (d.c / 8) * 4);
  if (!dwconv2d_pair_filter(host.data(), d.c, packed.data())) return 0;  // an infinite or NaN weight: the general kernel
  if (!(p->dw_paired = p->hold(packed.size() * 4))) return fail("dwconv2d_pack_filter: cannot allocate the paired filter");
  if (check(hipMemcpy(p->dw_paired, packed.data(), packed.size() * 4, hipMemcpyHostToDevice), "hipMemcpy")) {
    p->drop(&p->dw_paired, packed.size() * 4);
    return 1;
  }
  return 0;
}

int64_t pml_hip_pool2d_dispatch(const pml_hip_pool2d_desc* d) {
  if (!d) {
    fail("null descriptor");
    return 0;
  }
  if (d->dtype != PML_HIP_F32 && d->dtype != PML_HIP_BF16) {
    fail("pool2d: dtype must be F32 or BF16");
    return 0;
  }
  if (d->agg != PML_HIP_AGG_MAX && d->agg != PML_HIP_AGG_MIN && d->agg != PML_HIP_AGG_ADD) {
    fail("pool2d: aggregation must be max, min or add");
    return 0;
  }
  const int V = 16 / dt_size(d->dtype);
  if (d->c <= 0 || d->c % V != 0 || d->n <= 0 || d->h <= 0 || d->w <= 0 || d->kh <= 0 || d->kw <= 0 || d->oh <= 0 ||
      d->ow <= 0 || d->stride_h <= 0 || d->stride_w <= 0) {
    fail("pool2d: bad geometry (channels must cover whole 16-byte vectors)");
    return 0;
  }
  if (d->divisor != 0.f) {
    // (what pool_whole_kernel takes: pool2d_launch's own test)
    const int64_t chunks = (d->c / V + 31) / 32;
    const bool whole = d->agg == PML_HIP_AGG_ADD && d->oh == 1 && d->ow == 1 && d->kh == d->h && d->kw == d->w && d->pad_h == 0 &&
                       d->pad_w == 0 && !d->with_index && d->h * d->w >= 16 && d->n * chunks <= 0x7fffffff;
    if (!whole || !(d->divisor == d->divisor)) {
      fail("pool2d: a divisor goes with the sum over a whole image of at least 16 pixels only");
      return 0;
    }
  }
  Plan* p = new Plan();
  p->kind = PLAN_POOL;
  p->pool = *d;
  char buf[200];
  std::snprintf(buf, sizeof buf, "pool2d %s agg=%d n=%lld %lldx%lldx%lld k=%lldx%lld -> %lldx%lld%s",
                d->dtype == PML_HIP_F32 ? "f32" : "bf16", d->agg, (long long)d->n, (long long)d->h, (long long)d->w,
                (long long)d->c, (long long)d->kh, (long long)d->kw, (long long)d->oh, (long long)d->ow,
                d->with_index ? " +argmax" : "");
  p->text = buf;
  return (int64_t)(intptr_t)p;
}

int pml_hip_pool2d_invoke(int64_t plan, const void* input, void* output, void* index_output, pml_hip_stream s) {
  Plan* p = (Plan*)(intptr_t)plan;
  if (!p || p->kind != PLAN_POOL) return fail("pool2d_invoke: not a pool2d plan");
  if (!input || !output) return fail("pool2d_invoke: null operand");
  if (p->pool.with_index && !index_output) return fail("pool2d_invoke: the plan expects an index output");
  if ((((uintptr_t)input | (uintptr_t)output | (uintptr_t)index_output) & 15) != 0)
    return fail("pool2d_invoke: buffers must be 16-byte aligned");
  PoolArgs a;
  a.d = p->pool;
  a.in = input;
  a.out = output;
  a.idx = index_output;
  return check(pool2d_launch(a, (hipStream_t)s), "pool2d_launch");
}

// ---------------------------------------------------------------------------
// elementwise, select, index
// ---------------------------------------------------------------------------

int64_t pml_hip_eltwise_dispatch(const pml_hip_eltwise_desc* d) {
  if (!d) {
    fail("null descriptor");
    return 0;
  }
  if (d->rank < 0 || d->rank > PML_HIP_MAX_RANK) {
    fail("eltwise: rank out of range");
    return 0;
  }
  const pml_hip_epilogue& t = d->tail;
  if (t.n_ops < 0 || t.n_ops > PML_HIP_MAX_EPI_OPS || t.n_operands < 0 || t.n_operands > PML_HIP_MAX_EPI_OPERANDS) {
    fail("eltwise: malformed tail");
    return 0;
  }
  if (!valid_tail(t, /*allow64=*/true)) {
    fail("eltwise: a step of the chain names an unknown operation or an operand outside the operand list");
    return 0;
  }
  Plan* p = new Plan();
  p->kind = PLAN_ELTWISE;
  p->elt = *d;
  p->text = "eltwise chain of " + std::to_string(t.n_ops) + " steps, rank " + std::to_string(d->rank);
  return (int64_t)(intptr_t)p;
}

int pml_hip_eltwise_invoke(int64_t plan, const void* input, void* output, const void* const* operands,
                           void* const* outs, pml_hip_stream s) {
  Plan* p = (Plan*)(intptr_t)plan;
  if (!p || p->kind != PLAN_ELTWISE) return fail("eltwise_invoke: not an eltwise plan");
  if (!input || !output) return fail("eltwise_invoke: null operand");
  EltwiseArgs a;
  std::memset(&a, 0, sizeof a);
  a.d = p->elt;
  a.in = input;
  a.out = output;
  a.total = 1;
  for (int r = 0; r < a.d.rank; ++r) a.total *= a.d.sizes[r];
  bool wide = dt_size(a.d.in_dtype) == 8 || dt_size(a.d.out_dtype) == 8;
  for (int i = 0; i < a.d.tail.n_operands; ++i) {
    if (!operands || !operands[i]) return fail("eltwise_invoke: missing operand");
    a.operands[i] = operands[i];
    wide = wide || dt_size(a.d.tail.operand_dtype[i]) == 8;
  }
  for (int i = 0; i < a.d.tail.n_ops; ++i) wide = wide || dt_size(a.d.tail.ops[i].dtype) == 8;
  for (int i = 0; i < PML_HIP_MAX_EPI_OPERANDS; ++i) a.outs[i] = outs ? outs[i] : nullptr;
  a.wide = wide ? 1 : 0;
  return check(eltwise_launch(a, (hipStream_t)s), "eltwise_launch");
}

int pml_hip_select(const pml_hip_select_desc* d, const void* cond, const void* t, const void* f, void* out,
                   pml_hip_stream s) {
  if (!d || !cond || !t || !f || !out) return fail("select: null argument");
  if (d->rank < 0 || d->rank > PML_HIP_MAX_RANK) return fail("select: rank out of range");
  return check(select_launch(*d, cond, t, f, out, (hipStream_t)s), "select_launch");
}

int pml_hip_softmax(const pml_hip_softmax_desc* d, const void* x, void* y, pml_hip_stream s) {
  if (!d || !x || !y) return fail("softmax: null argument");
  if (d->dtype != PML_HIP_F32 && d->dtype != PML_HIP_BF16) return fail("softmax: dtype must be F32 or BF16");
  if (d->rows < 0 || d->cols < 0 || d->rows > 0x7fffffff) return fail("softmax: rows or cols out of range");
  return in_row_runs(d->rows, [&](int64_t first, int64_t rows) {
    pml_hip_softmax_desc run = *d;
    run.rows = rows;
    const int64_t at = first * d->cols * dt_size(d->dtype);
    return check(softmax_launch(run, (const char*)x + at, (char*)y + at, (hipStream_t)s), "softmax_launch");
  });
}

int pml_hip_index(void* out, int32_t rank, const int64_t* sizes, int32_t axis, pml_hip_stream s) {
  if (!out || !sizes || rank <= 0 || axis < 0 || axis >= rank) return fail("index: bad argument");
  return check(index_launch(out, rank, sizes, axis, (hipStream_t)s), "index_launch");
}

// ---------------------------------------------------------------------------
// special operations
// ---------------------------------------------------------------------------

namespace {
bool sizes_ok(const int64_t* sizes, int rank) {
  for (int i = 0; i < rank; ++i)
    if (sizes[i] < 0) return false;
  return true;
}
int64_t count_of(const int64_t* sizes, int rank) {
  int64_t n = 1;
  for (int i = 0; i < rank; ++i) n *= sizes[i];
  return n;
}
}  // namespace

int pml_hip_gather(const pml_hip_gather_desc* d, const void* tensor, const void* indices, void* out, pml_hip_stream s) {
  if (!d || !tensor || !indices || !out) return fail("gather: null argument");
  if (d->rank < 1 || d->rank > PML_HIP_MAX_SPECIAL_RANK || d->idx_rank < 0 || d->idx_rank > PML_HIP_MAX_SPECIAL_RANK)
    return fail("gather: rank out of range");
  if (!sizes_ok(d->sizes, d->rank) || !sizes_ok(d->idx_sizes, d->idx_rank)) return fail("gather: negative size");
  if (dt_size(d->dtype) == 0 || dt_size(d->idx_dtype) == 0) return fail("gather: bad element type");
  if (d->mode == PML_HIP_GATHER_NORMAL) {
    if (d->axis < 0 || d->axis >= d->rank) return fail("gather: axis out of range");
    if (d->rank - 1 + d->idx_rank > PML_HIP_MAX_SPECIAL_RANK) return fail("gather: result rank out of range");
    if (dt_is_float(d->idx_dtype) && dt_is_float(d->dtype)) {
      if (d->interpolation < PML_HIP_INTERP_NEAREST || d->interpolation > PML_HIP_INTERP_CUBIC)
        return fail("gather: floating indices need an interpolation mode");
      if (d->interpolation == PML_HIP_INTERP_NEAREST && (d->nearest < 0 || d->nearest > PML_HIP_NEAREST_SIMPLE))
        return fail("gather: bad nearest mode");
      if (d->oob != PML_HIP_OOB_EDGE_PADDED_INPUT && d->oob != PML_HIP_OOB_RETURN_ZERO) return fail("gather: bad out-of-bounds mode");
    }
  } else if (d->mode == PML_HIP_GATHER_ND) {
    if (dt_is_float(d->idx_dtype)) return fail("gather: ND mode needs integer indices");
    if (d->idx_rank < 1) return fail("gather: ND mode needs indices of rank >= 1");
    const int64_t k = d->idx_sizes[d->idx_rank - 1];
    if (d->batch_dims < 0 || d->batch_dims > d->idx_rank - 1 || d->batch_dims + k > d->rank)
      return fail("gather: ND index depth out of range");
    if (d->idx_rank - 1 + d->rank - d->batch_dims - k > PML_HIP_MAX_SPECIAL_RANK) return fail("gather: result rank out of range");
    for (int i = 0; i < d->batch_dims; ++i)
      if (d->sizes[i] != d->idx_sizes[i]) return fail("gather: batch dimensions differ");
  } else {
    return fail("gather: bad mode");
  }
  return check(gather_launch(*d, tensor, indices, out, (hipStream_t)s), "gather_launch");
}

int pml_hip_scatter(const pml_hip_scatter_desc* d, const void* data, const void* indices, const void* updates, void* out,
                    pml_hip_stream s) {
  if (!d || !data || !indices || !updates || !out) return fail("scatter: null argument");
  if (out == data) return fail("scatter: the result must not alias the data");
  if (d->rank < 1 || d->rank > PML_HIP_MAX_SPECIAL_RANK || d->idx_rank < 1 || d->idx_rank > PML_HIP_MAX_SPECIAL_RANK ||
      d->upd_rank < 1 || d->upd_rank > PML_HIP_MAX_SPECIAL_RANK)
    return fail("scatter: rank out of range");
  if (!sizes_ok(d->sizes, d->rank) || !sizes_ok(d->idx_sizes, d->idx_rank) || !sizes_ok(d->upd_sizes, d->upd_rank))
    return fail("scatter: negative size");
  if (d->idx_dtype != PML_HIP_I32 && d->idx_dtype != PML_HIP_U32) return fail("scatter: indices must be si32 or ui32");
  if (dt_size(d->dtype) == 0) return fail("scatter: bad element type");
  if (d->axis < 0 || d->axis >= d->rank) return fail("scatter: axis out of range");
  // every update element must name a full coordinate of the result
  int dst_rank = 0;
  switch (d->mode) {
    case PML_HIP_SCATTER_UPDATE_ND: {
      const int64_t k = d->idx_sizes[d->idx_rank - 1];
      if (d->upd_rank < d->idx_rank - 1) return fail("scatter: updates have too few dimensions");
      dst_rank = (int)k + d->upd_rank - (d->idx_rank - 1);
      for (int i = 0; i + 1 < d->idx_rank; ++i)
        if (d->upd_sizes[i] != d->idx_sizes[i]) return fail("scatter: updates and indices disagree");
      break;
    }
    case PML_HIP_SCATTER_UPDATE_SLICE:
      if (d->upd_rank < d->axis + d->idx_rank) return fail("scatter: updates have too few dimensions");
      dst_rank = d->upd_rank - d->idx_rank + 1;
      for (int i = 0; i < d->idx_rank; ++i)
        if (d->upd_sizes[d->axis + i] != d->idx_sizes[i]) return fail("scatter: updates and indices disagree");
      break;
    case PML_HIP_SCATTER_NORMAL:
    case PML_HIP_SCATTER_UPDATE_ELT:
      if (d->upd_rank < d->idx_rank) return fail("scatter: updates have too few dimensions");
      dst_rank = d->upd_rank;
      for (int i = 0; i < d->idx_rank; ++i)
        if (d->upd_sizes[i] != d->idx_sizes[i]) return fail("scatter: updates and indices disagree");
      break;
    default: return fail("scatter: bad mode");
  }
  if (dst_rank != d->rank) return fail("scatter: updates do not address the result's rank");
  return check(scatter_launch(*d, data, indices, updates, out, (hipStream_t)s), "scatter_launch");
}

int pml_hip_prng(const void* state, int64_t count, void* values, void* new_state, pml_hip_stream s) {
  if (!state) return fail("prng: null state");
  if (count < 0) return fail("prng: negative count");
  if (!values && !new_state) return 0;
  return check(prng_launch(state, count, values, new_state, (hipStream_t)s), "prng_launch");
}

int pml_hip_argsort(const pml_hip_argsort_desc* d, const void* tensor, void* out, pml_hip_stream s) {
  if (!d || !tensor || !out) return fail("argsort: null argument");
  if (d->rank < 1 || d->rank > PML_HIP_MAX_SPECIAL_RANK) return fail("argsort: rank out of range");
  if (!sizes_ok(d->sizes, d->rank)) return fail("argsort: negative size");
  if (d->axis < 0 || d->axis >= d->rank) return fail("argsort: axis out of range");
  if (d->direction != 0 && d->direction != 1) return fail("argsort: bad direction");
  if (dt_size(d->dtype) == 0 || d->dtype == PML_HIP_BOOL) return fail("argsort: bad element type");
  if (d->sizes[d->axis] > PML_HIP_MAX_SORT_LINE)
    return fail("argsort: more than PML_HIP_MAX_SORT_LINE (16384) elements along the sorted axis");
  if (count_of(d->sizes, d->rank) == 0) return 0;
  return check(argsort_launch(*d, tensor, out, (hipStream_t)s), "argsort_launch");
}

// ---------------------------------------------------------------------------
// any contraction
// ---------------------------------------------------------------------------

int64_t pml_hip_contract_dispatch(const pml_hip_contract_desc* d) {
  if (!d) {
    fail("null descriptor");
    return 0;
  }
  if (d->n_idx < 0 || d->n_idx > PML_HIP_MAX_IDX || d->n_out_idx < 0 || d->n_out_idx > d->n_idx || d->n_forms < 0 ||
      d->n_forms > PML_HIP_MAX_FORMS || d->n_src < 1 || d->n_src > 3) {
    fail("contract: descriptor out of range");
    return 0;
  }
  int64_t outs = 1;
  for (int v = 0; v < d->n_out_idx; ++v) {
    if (d->hi[v] < d->lo[v]) {
      outs = 0;
      break;
    }
    outs *= d->hi[v] - d->lo[v] + 1;
  }
  if (outs != d->out_elems) {
    fail("contract: out_elems does not match the output index ranges");
    return 0;
  }
  for (int f = 0; f < d->n_forms; ++f) {
    if (d->forms[f].den <= 0 || d->forms[f].operand < -1 || d->forms[f].operand > d->n_src) {
      fail("contract: malformed form");
      return 0;
    }
  }
  if (d->combo == PML_HIP_COMBO_EQ && (d->dtype != PML_HIP_BOOL || d->n_src != 2)) {
    fail("contract: the eq combination takes two operands and gives a boolean result");
    return 0;
  }
  Plan* p = new Plan();
  p->kind = PLAN_CONTRACT;
  p->con = *d;
  p->text = "contract (thread per output element) agg=" + std::to_string(d->agg) + " combo=" + std::to_string(d->combo) +
            " idx=" + std::to_string(d->n_idx) + " outputs=" + std::to_string((long long)d->out_elems);
  return (int64_t)(intptr_t)p;
}

int pml_hip_contract_invoke(int64_t plan, const void* const* srcs, void* out, pml_hip_stream s) {
  Plan* p = (Plan*)(intptr_t)plan;
  if (!p || p->kind != PLAN_CONTRACT) return fail("contract_invoke: not a contract plan");
  if (!srcs || !out) return fail("contract_invoke: null operand");
  ContractArgs a;
  std::memset(&a, 0, sizeof a);
  a.d = p->con;
  for (int i = 0; i < a.d.n_src; ++i) {
    if (!srcs[i]) return fail("contract_invoke: null source");
    a.srcs[i] = srcs[i];
  }
  a.out = out;
  return check(contract_launch(a, (hipStream_t)s), "contract_launch");
}

size_t pml_hip_struct_size(int which) {
  switch (which) {
    case 0: return sizeof(pml_hip_epilogue);
    case 1: return sizeof(pml_hip_gemm_desc);
    case 2: return sizeof(pml_hip_conv2d_desc);
    case 3: return sizeof(pml_hip_dwconv2d_desc);
    case 4: return sizeof(pml_hip_pool2d_desc);
    case 5: return sizeof(pml_hip_eltwise_desc);
    case 6: return sizeof(pml_hip_select_desc);
    case 7: return sizeof(pml_hip_contract_desc);
    case 8: return sizeof(pml_hip_form);
    case 9: return sizeof(pml_hip_gather_desc);
    case 10: return sizeof(pml_hip_scatter_desc);
    case 11: return sizeof(pml_hip_argsort_desc);
    case 12: return sizeof(pml_hip_softmax_desc);
    case 13: return sizeof(pml_hip_product_desc);
    case 14: return sizeof(pml_hip_rows_desc);
  }
  return 0;
}

int pml_hip_plan_free(int64_t plan) {
  delete (Plan*)(intptr_t)plan;
  return 0;
}

size_t pml_hip_plan_bytes(int64_t plan) {
  const Plan* p = (const Plan*)(intptr_t)plan;
  return p ? p->held + (p->sub ? p->sub->held.load() : 0) : 0;
}

int pml_hip_plan_describe(int64_t plan, char* buf, size_t buf_len) {
  Plan* p = (Plan*)(intptr_t)plan;
  if (!p || !buf || buf_len == 0) return fail("plan_describe: bad argument");
  std::snprintf(buf, buf_len, "%s", p->text.c_str());
  return 0;
}

}  // extern "C"
