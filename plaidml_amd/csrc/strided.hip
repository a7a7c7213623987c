// Matrix products over free strides: batched products, products whose rows are no whole 16-byte vectors, products of
// transposed operands, and the filter gradient of a convolution, all on the matrix cores.
//
// igemm.hip streams K-contiguous, 16-byte aligned rows straight into LDS; what it cannot address comes here.  Operands
// pass through registers on their way to LDS, which costs a few vector instructions per 16 bytes but takes any
// alignment (global loads of 8 and 16 bytes need none on this target) and any of three layouts per operand:
//   ROWS_K     row m (column n) of the operand is contiguous along K
//   ROWS_M     row k is contiguous along m (n), or has a free element stride there
//   ROWS_CONV  (left-hand side of a filter gradient) row k is an output pixel; its elements are the kw * ci
//              neighbouring values of one filter row's window, which lie contiguously in an NHWC image (dilation 1)
// A workgroup of four wavefronts owns a tile of 64 MI x 64 NI results, each wavefront a quarter as MI x NI blocks of
// 32 x 32.  K goes by in slabs of 32 (fp32) or 64 (bf16) values, double-buffered in LDS: the next slab's global loads
// are in flight while the current one is multiplied, one barrier per slab.
//   fp32: LDS holds [k][m]; a lane reads one word per operand and MFMA (v_mfma_f32_32x32x2_f32), 32 neighbouring
//         words per half wavefront.
//   bf16: LDS holds [m][k], 128 bytes a row, the 16-byte chunk c of row m at slot c ^ key(m): both the transposed
//         8-byte stores of a ROWS_M operand (lanes step m by 4) and the 16-byte fragment reads (lanes step m by 1)
//         then meet all banks (v_mfma_f32_32x32x16_bf16).
// Few tiles and a long K (a filter gradient: 9 tiles of 50176 pixels at 16 x 56 x 56 x 64): the K loop is split over
// workgroups, partial tiles go to a workspace and a second launch adds them in a fixed order and runs the tail.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <limits>
#include <numeric>

#include "device_common.h"
#include "plans.h"

namespace pml {
namespace {

enum { ROWS_K = 0, ROWS_M = 1, ROWS_CONV = 2 };
constexpr int kThreads = 256;

template <int N>
struct Words {
  uint32_t w[N];
};

// N 32-bit words from an address of any alignment
template <int N>
__device__ __forceinline__ Words<N> load_words(const void* p) {
  Words<N> v;
  __builtin_memcpy(&v, p, sizeof v);
  return v;
}

// The tail on four neighbouring results of one row: the contraction's value rounded to the result type, then each step
// in that type.  `row_at`: the row's element offset in the result.
__device__ __forceinline__ void strided_tail(const StridedArgs& p, float (&v)[4], int64_t row_at, int64_t col, int live) {
  const bool bf = p.out_bf16;
  auto rnd = [&](float x) { return bf ? round_to_bf16(x) : x; };
  auto fetch = [&](const void* base, int64_t at) { return bf ? bf16_bits_to_f32(((const uint16_t*)base)[at]) : ((const float*)base)[at]; };
  const int64_t row = (p.init != nullptr || p.n_ops > 0) ? row_at / p.row_len : 0;
  if (p.init) {
#pragma unroll
    for (int q = 0; q < 4; ++q)
      if (q < live) v[q] += fetch(p.init, row * p.init_rs + (col + q) * p.init_cs);
  }
#pragma unroll
  for (int q = 0; q < 4; ++q) v[q] = rnd(v[q]);
  for (int s = 0; s < p.n_ops; ++s) {
    const StridedOp& op = p.ops[s];
    float x[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) x[q] = op.ptr ? (q < live ? fetch(op.ptr, row * op.rs + (col + q) * op.cs) : 0.f) : op.imm;
#define PML_EACH(EXPR)                                                            \
  _Pragma("unroll") for (int q = 0; q < 4; ++q) {                                 \
    const float a = v[q], b = x[q];                                               \
    v[q] = rnd(EXPR);                                                             \
  }                                                                               \
  break;
    switch (op.opcode) {
      case PML_HIP_EPI_ADD: PML_EACH(a + b)
      case PML_HIP_EPI_SUB: PML_EACH(a - b)
      case PML_HIP_EPI_RSUB: PML_EACH(b - a)
      case PML_HIP_EPI_MUL: PML_EACH(a * b)
      case PML_HIP_EPI_DIV: PML_EACH(a / b)
      case PML_HIP_EPI_RDIV: PML_EACH(b / a)
      case PML_HIP_EPI_MAX: PML_EACH((a < b) ? b : a)
      case PML_HIP_EPI_MIN: PML_EACH((a < b) ? a : b)
      case PML_HIP_EPI_RELU: PML_EACH((a < 0.f) ? 0.f : a)
      case PML_HIP_EPI_NEG: PML_EACH(-a)
      case PML_HIP_EPI_MAX_GT: PML_EACH((a > b) ? a : b)
      default: break;
    }
#undef PML_EACH
  }
}

__device__ __forceinline__ void store_results(const StridedArgs& p, void* c, int64_t at, const float (&v)[4], int live) {
  if (p.out_bf16) {
    uint16_t h[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) h[q] = f32_to_bf16_bits(v[q]);
    uint16_t* const to = (uint16_t*)c + at;
    if (live == 4) {
      __builtin_memcpy(to, h, 8);
    } else {
#pragma unroll
      for (int q = 0; q < 4; ++q)
        if (q < live) to[q] = h[q];
    }
  } else {
    float* const to = (float*)c + at;
    if (live == 4) {
      __builtin_memcpy(to, v, 16);
    } else {
#pragma unroll
      for (int q = 0; q < 4; ++q)
        if (q < live) to[q] = v[q];
    }
  }
}

// Filter gradient: a tap that leaves the image is no term of the sum, but the matrix cores multiply the zeros read in its
// place with the gradient, and a zero times an infinity or a NaN is a NaN.  Such a product can only turn a result into a NaN:
// results that are none are right as they are, and a lane's results that are (v[0 .. live - 1], row m, from column n) are
// summed again here without those taps, one after the other by the whole wavefront -- every lane has to come here, those
// without results with live = 0.  Costs nothing but the test while gradients are finite; a NaN that belongs into the sum
// ends it where it is met.
__device__ __forceinline__ void leave_outside_taps_out(const StridedArgs& p, bool bf, int m, int n, int live, float (&v)[4]) {
  const bool nan = (live > 0 && v[0] != v[0]) || (live > 1 && v[1] != v[1]) || (live > 2 && v[2] != v[2]) || (live > 3 && v[3] != v[3]);
  uint64_t lanes = __ballot(nan);
  if (lanes == 0) return;
  const int lane = threadIdx.x & 63;
  auto fetch = [&](const void* base, int64_t at) { return bf ? bf16_bits_to_f32(((const uint16_t*)base)[at]) : ((const float*)base)[at]; };
  for (; lanes != 0; lanes &= lanes - 1) {
    const int of = __builtin_ctzll(lanes);
    const int row = __builtin_amdgcn_readlane(m, of), col0 = __builtin_amdgcn_readlane(n, of), count = __builtin_amdgcn_readlane(live, of);
    const int tap = row / (int)p.row_cols, j = row - tap * (int)p.row_cols, kx = j / p.CI, ci = j - kx * p.CI;
#pragma unroll 1
    for (int q = 0; q < count; ++q) {
      const float had = q == 0 ? v[0] : q == 1 ? v[1] : q == 2 ? v[2] : v[3];
      if (__ballot(lane == of && had != had) == 0) continue;
      float sum = 0.f;
      for (int64_t k0 = 0; k0 < p.K; k0 += 256) {
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const int64_t k = k0 + 64 * u + lane;
          if (k >= p.K) continue;
          const unsigned img = fast_div((unsigned)k, p.div_per_magic, p.div_per_shift);
          const unsigned rem = (unsigned)k - img * (unsigned)(p.OH * p.OW);
          const unsigned oy = fast_div(rem, p.div_ow_magic, p.div_ow_shift);
          const int iy = (int)oy * p.SH + tap * p.DH - p.PH, ix = (int)(rem - oy * (unsigned)p.OW) * p.SW + kx - p.PW;
          if (iy < 0 || iy >= p.H || ix < 0 || ix >= p.W) continue;
          sum += fetch(p.A, (((int64_t)img * p.H + iy) * p.W + ix) * p.CI + ci) * fetch(p.B, k * p.N + col0 + q);
        }
        if (__ballot(sum != sum) != 0) break;
      }
#pragma unroll
      for (int w = 32; w > 0; w >>= 1) sum += __shfl_xor(sum, w, 64);
      if (lane == of) {
        v[0] = q == 0 ? sum : v[0];
        v[1] = q == 1 ? sum : v[1];
        v[2] = q == 2 ? sum : v[2];
        v[3] = q == 3 ? sum : v[3];
      }
    }
  }
}

// One operand's share of a workgroup: T rows (of m or n) by one slab of K.
//   fetch(k0): the slab's values of this thread, into registers;   put(lds): from there into the slab's LDS buffer
template <bool BF, int MODE, int T, bool FLAT>
struct Side {
  static constexpr int BK = BF ? 64 : 32;
  static constexpr int kPitch = BF ? 0 : (MODE == ROWS_K ? T + 1 : T + 4);  // fp32: words per K-row
  static constexpr int kBytes = BF ? T * 128 : (BK * kPitch * 4 + 15) / 16 * 16;
  static constexpr int kPasses = T / 32;  // fp32, and bf16 ROWS_K: 16-byte chunks per thread
  static constexpr int kBlocks = T / 64;  // bf16 ROWS_M: blocks of 4 x 4 values per thread
  const char* base;     // the tile's first row, K-index 0 (ROWS_CONV: the image)
  int64_t ms, ks;       // element strides
  int64_t live;         // rows of the tile that exist
  int64_t extent;       // elements from the base up to and with the operand's last one that this tile may read (contiguous rows)
  bool whole;           // every row exists and is contiguous where the layout says so
  bool cut;             // the slab in the registers has runs that clear() has to clear
  int keep[BF && MODE != ROWS_K ? kBlocks * 4 : kPasses];  // their first value that stays, and how many do
  uint32_t regs[BF ? (MODE == ROWS_K ? kPasses * 4 : kBlocks * 8) : kPasses * 4];

  __device__ __forceinline__ static int key(int m) { return (m ^ (m >> 2)) & 7; }

  // ROWS_CONV: where a thread's pixels lie, counted on from slab to slab (two divisions a row of every slab before)
  struct Pixel {
    int img, oy, ox;
  };
  Pixel px, slab_step, run_step;  // this thread's first pixel; from slab to slab; from one of its runs (bf16: of four) to the next
  __device__ __forceinline__ static Pixel pixel(const StridedArgs& p, unsigned k) {
    const unsigned img = fast_div(k, p.div_per_magic, p.div_per_shift), rem = k - img * (unsigned)(p.OH * p.OW);
    const unsigned oy = fast_div(rem, p.div_ow_magic, p.div_ow_shift);
    return {(int)img, (int)oy, (int)(rem - oy * (unsigned)p.OW)};
  }
  __device__ __forceinline__ static Pixel ahead(const StridedArgs& p, Pixel a, int img, int oy, int ox) {
    a.ox += ox;
    const bool row = a.ox >= p.OW;
    a.ox -= row ? p.OW : 0;
    a.oy += oy + (row ? 1 : 0);
    const bool image = a.oy >= p.OH;
    a.oy -= image ? p.OH : 0;
    a.img += img + (image ? 1 : 0);
    return a;
  }
  static constexpr int kPer = T / 4;                                             // runs of four columns
  static constexpr int kRowStep = BF ? 4 * kThreads / kPer : kThreads / kPer;  // between a thread's rows (bf16: of its blocks of four)
  __device__ __forceinline__ void start(const StridedArgs& p, int64_t k_begin, int tid) {
    px = pixel(p, (unsigned)k_begin + (unsigned)(tid / kPer) * (BF ? 4 : 1));
    slab_step = pixel(p, BK);
    run_step = pixel(p, BF ? kRowStep - 3 : kRowStep);  // (bf16: from the last row of a block of four)
  }

  static constexpr int kVals = BF && MODE == ROWS_K ? 8 : 4, kWords = kVals * (BF ? 2 : 4) / 4;
  static constexpr int kRuns = BF && MODE != ROWS_K ? 4 * kBlocks : kPasses;
  __device__ __forceinline__ Pixel next_pixel(const StridedArgs& p, const Pixel& pix, int r) const {
    if (BF && r % 4 != 3) return ahead(p, pix, 0, 0, 1);
    return r + 1 < kRuns ? ahead(p, pix, run_step.img, run_step.oy, run_step.ox) : pix;
  }

  // A thread's runs of neighbouring values: where run r of the slab at k0 begins, and which of its values belong to it.
  struct Run {
    int64_t at;
    int lo, hi;
  };
  __device__ __forceinline__ static int row_of(int r, int tid) {  // in the slab (ROWS_K: in the tile)
    if constexpr (MODE == ROWS_K) return tid / 8 + 32 * r;
    if constexpr (BF) return (tid / kPer) * 4 + (r / 4) * kRowStep + r % 4;
    return tid / kPer + r * kRowStep;
  }
  __device__ __forceinline__ Run run(const StridedArgs& p, int r, int64_t k0, int64_t k_end, int tid, const Pixel& pix) const {
    const int row = row_of(r, tid);
    Run at;
    at.lo = 0;
    int64_t last;
    if constexpr (MODE == ROWS_K) {
      const int kq = (tid % 8) * kVals;
      at.at = row * ms + (k0 + kq) * ks;
      last = row < live ? k_end - k0 - kq : 0;
    } else if constexpr (MODE == ROWS_M) {
      const int m4 = (tid % kPer) * 4;
      at.at = (k0 + row) * ks + m4 * ms;
      last = k0 + row < k_end ? live - m4 : 0;
    } else {
      // the values of the pixel's window row from column j0 of the tile on (ks: the tile's first column inside the window row)
      const int j0 = (tid % kPer) * 4, iy = pix.oy * p.SH + (int)ms * p.DH - p.PH, row_elems = p.W * p.CI;
      const int first = (pix.ox * p.SW - p.PW) * p.CI + (int)ks + j0;
      at.at = ((int64_t)pix.img * p.H + iy) * row_elems + first;
      at.lo = first < 0 ? -first : 0;
      const int end = row_elems - first < (int)live - j0 ? row_elems - first : (int)live - j0;
      last = k0 + row < k_end && iy >= 0 && iy < p.H ? end : 0;
    }
    at.hi = (int)(last < 0 ? 0 : last > kVals ? kVals : last);
    return at;
  }

  // a run's values `apart` elements from each other
  __device__ __forceinline__ void gather(uint32_t* to, int64_t at, int lo, int hi, int64_t apart) const {
    if constexpr (BF) {
      uint16_t h[kVals];
#pragma unroll
      for (int e = 0; e < kVals; ++e) h[e] = e >= lo && e < hi ? ((const uint16_t*)base)[at + e * apart] : (uint16_t)0;
      __builtin_memcpy(to, h, sizeof h);
    } else {
#pragma unroll
      for (int e = 0; e < kVals; ++e) {
        to[e] = e >= lo && e < hi ? ((const uint32_t*)base)[at + e * apart] : 0u;
      }
    }
  }
  __device__ __forceinline__ void straight(uint32_t* to, int64_t at) const {
    const Words<kWords> v = load_words<kWords>(base + at * (BF ? 2 : 4));
#pragma unroll
    for (int e = 0; e < kWords; ++e) to[e] = v.w[e];
  }

  // Where nothing is cut and rows are contiguous the loads go out as they are; elsewhere run by run, or value by value where a run is
  // cut.  FLAT (filter gradients, where a slab's pixels always have cut window rows among them; see `flat_fetch`): the loads go out whole
  // there, too, and put() clears what does not belong to the operand -- but for a slab with a run that sticks out of the operand's
  // `extent` elements.  (Tried: two slabs on their way instead of one, 219 registers, 46.6 us for 35.6; loads of what is not there beside
  // what is instead of from the base, 3 % slower.)
  __device__ __forceinline__ void fetch(const StridedArgs& p, int64_t k0, int64_t k_end, int tid) {
    Pixel pix{0, 0, 0};
    if constexpr (MODE == ROWS_CONV) {
      pix = px;
      px = ahead(p, px, slab_step.img, slab_step.oy, slab_step.ox);
    }
    const bool full = MODE != ROWS_CONV && whole && k0 + BK <= k_end;  // uniform: no lane checks anything
    const int64_t apart = MODE == ROWS_K ? ks : MODE == ROWS_M ? ms : 1;
    cut = false;
    if (full || !FLAT) {
#pragma unroll
      for (int r = 0; r < kRuns; ++r) {
        const Run at = run(p, r, k0, k_end, tid, pix);
        if constexpr (MODE == ROWS_CONV) pix = next_pixel(p, pix, r);
        if (full || (at.lo == 0 && at.hi == kVals && apart == 1))
          straight(&regs[kWords * r], at.at);
        else
          gather(&regs[kWords * r], at.at, at.lo, at.hi, apart);
      }
      return;
    }
    Run runs[kRuns];
    bool out = false;
#pragma unroll
    for (int r = 0; r < kRuns; ++r) {
      runs[r] = run(p, r, k0, k_end, tid, pix);
      if constexpr (MODE == ROWS_CONV) pix = next_pixel(p, pix, r);
      const bool any = runs[r].hi > runs[r].lo;
      keep[r] = any ? runs[r].lo | (runs[r].hi - runs[r].lo) << 8 : 0;
      out = out || (any && (runs[r].at < 0 || runs[r].at + kVals > extent));
    }
    cut = extent >= kVals && apart == 1 && __ballot(out) == 0;
    // (nothing but the runs' values differs between the two ways: a store that both end with goes through scratch otherwise)
    if (cut) {
#pragma unroll
      for (int r = 0; r < kRuns; ++r) straight(&regs[kWords * r], runs[r].hi > runs[r].lo ? runs[r].at : 0);
    } else {
#pragma unroll
      for (int r = 0; r < kRuns; ++r) gather(&regs[kWords * r], runs[r].at, runs[r].lo, runs[r].hi, apart);
    }
  }

  // clears the values of a slab's runs that do not belong to the operand
  __device__ __forceinline__ void clear() {
    if (!FLAT || !cut) return;
#pragma unroll
    for (int r = 0; r < kRuns; ++r) {
      const int lo = keep[r] & 255;
      const unsigned count = (unsigned)keep[r] >> 8;
#pragma unroll
      for (int w = 0; w < kWords; ++w) {
        uint32_t& v = regs[kWords * r + w];
        if constexpr (BF)
          v &= ((unsigned)(2 * w - lo) < count ? 0xffffu : 0u) | ((unsigned)(2 * w + 1 - lo) < count ? 0xffff0000u : 0u);
        else
          v = (unsigned)(w - lo) < count ? v : 0u;
      }
    }
  }

  __device__ __forceinline__ void put(char* lds, int tid) {
    clear();
    if constexpr (BF && MODE == ROWS_K) {
#pragma unroll
      for (int i = 0; i < kPasses; ++i) {
        const int row = tid / 8 + 32 * i, c = tid % 8;
        *(i32x4_t*)(lds + row * 128 + ((c ^ key(row)) * 16)) =
            i32x4_t{(int)regs[4 * i], (int)regs[4 * i + 1], (int)regs[4 * i + 2], (int)regs[4 * i + 3]};
      }
    } else if constexpr (BF) {
      constexpr int PER = T / 4;
#pragma unroll
      for (int i = 0; i < kBlocks; ++i) {
        const int c = tid + kThreads * i, k4 = c / PER, m4 = (c % PER) * 4;
        const uint32_t* r = &regs[8 * i];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          // value e of the four K-rows
          const unsigned sel = (e & 1) ? 0x07060302u : 0x05040100u;
          const int h = e >> 1;
          const uint2 w = make_uint2(__builtin_amdgcn_perm(r[2 + h], r[h], sel), __builtin_amdgcn_perm(r[6 + h], r[4 + h], sel));
          const int m = m4 + e;
          *(uint2*)(lds + m * 128 + (((k4 >> 1) ^ key(m)) * 16) + (k4 & 1) * 8) = w;
        }
      }
    } else if constexpr (MODE == ROWS_K) {
#pragma unroll
      for (int i = 0; i < kPasses; ++i) {
        const int row = tid / 8 + 32 * i, kq = (tid % 8) * 4;
#pragma unroll
        for (int e = 0; e < 4; ++e) *(uint32_t*)(lds + ((kq + e) * kPitch + row) * 4) = regs[4 * i + e];
      }
    } else {
      constexpr int PER = T / 4;
#pragma unroll
      for (int i = 0; i < kPasses; ++i) {
        const int c = tid + kThreads * i, k = c / PER, m4 = (c % PER) * 4;
        *(i32x4_t*)(lds + (k * kPitch + m4) * 4) = i32x4_t{(int)regs[4 * i], (int)regs[4 * i + 1], (int)regs[4 * i + 2], (int)regs[4 * i + 3]};
      }
    }
  }
};

template <bool BF, int AMODE, int BMODE, int MI, int NI, bool FLAT = false>
__global__ __launch_bounds__(kThreads) void strided_kernel(StridedArgs p_by_value) {
  // (read where the dispatcher put it: indexing a by-value copy would move the copy to scratch memory)
  const StridedArgs& p = *(const StridedArgs*)(const __attribute__((address_space(4))) void*)__builtin_amdgcn_kernarg_segment_ptr();
  constexpr int TM = 64 * MI, TN = 64 * NI, ES = BF ? 2 : 4;
  typedef Side<BF, AMODE, TM, FLAT> side_a;
  typedef Side<BF, BMODE, TN, FLAT> side_b;
  constexpr int BK = side_a::BK, kStage = side_a::kBytes + side_b::kBytes;
  extern __shared__ __attribute__((aligned(16))) char smem[];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), wm = wave >> 1, wn = wave & 1;

  unsigned t = blockIdx.x;
  const int tn = (int)(t % (unsigned)p.tiles_n);
  t /= (unsigned)p.tiles_n;
  const int tm = (int)(t % (unsigned)p.tiles_m);
  t /= (unsigned)p.tiles_m;
  int64_t a_at = 0, b_at = 0, c_at = 0;
  const unsigned batch = t;
  for (int d = p.n_batch - 1; d >= 0; --d) {
    const unsigned sz = (unsigned)p.batch[d], i = t % sz;
    t /= sz;
    a_at += i * p.a_batch[d];
    b_at += i * p.b_batch[d];
    c_at += i * p.c_batch[d];
  }
  int64_t m0, m_rows;  // first result row of the tile, rows it has
  side_a sa;
  side_b sb;
  if constexpr (AMODE == ROWS_CONV) {
    // tiles of one filter row's window columns after those of the row before it
    const int tap = tm / p.tiles_per_tap, j0 = (tm - tap * p.tiles_per_tap) * TM;
    m0 = (int64_t)tap * p.row_cols + j0;
    m_rows = p.row_cols - j0 < TM ? p.row_cols - j0 : TM;
    sa.base = (const char*)p.A;
    sa.ks = j0;
    sa.ms = tap;  // (the filter row)
    sa.live = m_rows;
    sa.whole = false;
    sa.extent = (int64_t)fast_div((unsigned)p.K, p.div_per_magic, p.div_per_shift) * p.H * p.W * p.CI;
  } else {
    m0 = (int64_t)tm * TM;
    m_rows = p.M - m0 < TM ? p.M - m0 : TM;
    sa.base = (const char*)p.A + (a_at + m0 * p.a_ms) * ES;
    sa.ms = p.a_ms;
    sa.ks = p.a_ks;
    sa.live = m_rows;
    sa.whole = m_rows == TM && (AMODE == ROWS_K ? p.a_ks : p.a_ms) == 1;
    sa.extent = (m_rows - 1) * p.a_ms + (p.K - 1) * p.a_ks + 1;
  }
  const int64_t n0 = (int64_t)tn * TN;
  const int64_t n_cols = p.N - n0 < TN ? p.N - n0 : TN;
  sb.base = (const char*)p.B + (b_at + n0 * p.b_ns) * ES;
  sb.ms = p.b_ns;
  sb.ks = p.b_ks;
  sb.live = n_cols;
  sb.whole = n_cols == TN && (BMODE == ROWS_K ? p.b_ks : p.b_ns) == 1;
  sb.extent = (n_cols - 1) * p.b_ns + (p.K - 1) * p.b_ks + 1;

  const int64_t k_begin = (int64_t)blockIdx.y * p.k_per_split;
  const int64_t k_end = k_begin + p.k_per_split < p.K ? k_begin + p.k_per_split : p.K;

  f32x16_t acc[MI][NI];
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < NI; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;

  if constexpr (AMODE == ROWS_CONV) sa.start(p, k_begin, tid);
  sa.fetch(p, k_begin, k_end, tid);
  sb.fetch(p, k_begin, k_end, tid);
  sa.put(smem, tid);
  sb.put(smem + side_a::kBytes, tid);
  __syncthreads();
  int stage = 0;
  const int row = lane & 31, half = lane >> 5;
  for (int64_t k = k_begin; k < k_end; k += BK) {
    const bool more = k + BK < k_end;
    if (more) {
      sa.fetch(p, k + BK, k_end, tid);
      sb.fetch(p, k + BK, k_end, tid);
    }
    const char* la = smem + stage * kStage;
    const char* lb = la + side_a::kBytes;
    if constexpr (BF) {
#pragma unroll
      for (int kk = 0; kk < 4; ++kk) {
        bf16x8_t fa[MI], fb[NI];
#pragma unroll
        for (int i = 0; i < MI; ++i) {
          const int m = (wm * MI + i) * 32 + row;
          fa[i] = *(const bf16x8_t*)(la + m * 128 + (((kk * 2 + half) ^ side_a::key(m)) * 16));
        }
#pragma unroll
        for (int j = 0; j < NI; ++j) {
          const int n = (wn * NI + j) * 32 + row;
          fb[j] = *(const bf16x8_t*)(lb + n * 128 + (((kk * 2 + half) ^ side_b::key(n)) * 16));
        }
        // (the right-hand fragment is the row operand: a lane then holds one result row m = lane % 32 and in it the
        // columns 8 (r / 4) + 4 (lane / 32) + r % 4 -- runs of four)
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
          for (int j = 0; j < NI; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fb[j], fa[i], acc[i][j], 0, 0, 0);
      }
    } else {
#pragma unroll
      for (int kk = 0; kk < BK / 2; ++kk) {
        float fa[MI], fb[NI];
#pragma unroll
        for (int i = 0; i < MI; ++i) fa[i] = *(const float*)(la + ((kk * 2 + half) * side_a::kPitch + (wm * MI + i) * 32 + row) * 4);
#pragma unroll
        for (int j = 0; j < NI; ++j) fb[j] = *(const float*)(lb + ((kk * 2 + half) * side_b::kPitch + (wn * NI + j) * 32 + row) * 4);
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
          for (int j = 0; j < NI; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(fb[j], fa[i], acc[i][j], 0, 0, 0);
      }
    }
    stage ^= 1;
    if (more) {
      sa.put(smem + stage * kStage, tid);
      sb.put(smem + stage * kStage + side_a::kBytes, tid);
    }
    __syncthreads();
  }

  // The tile goes through LDS once, so that a row's results leave in runs of 16 (8) bytes per lane and the tail is one
  // small loop over them.
  float* const ctile = (float*)smem;
  constexpr int CS = TN + 4;
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < NI; ++j)
#pragma unroll
      for (int g = 0; g < 4; ++g)
        *(f32x4_t*)&ctile[((wm * MI + i) * 32 + row) * CS + (wn * NI + j) * 32 + 8 * g + 4 * half] =
            f32x4_t{acc[i][j][4 * g], acc[i][j][4 * g + 1], acc[i][j][4 * g + 2], acc[i][j][4 * g + 3]};
  __syncthreads();
  const int lc = (tid % (TN / 4)) * 4;
  if (AMODE != ROWS_CONV && lc >= n_cols) return;
  const int live = lc >= n_cols ? 0 : n_cols - lc < 4 ? (int)(n_cols - lc) : 4;
  const int64_t n = n0 + lc;
  if (AMODE == ROWS_CONV && p.ws == nullptr) {
    // (every lane stays to the end: see leave_outside_taps_out)
    for (int l0 = 0; l0 < m_rows; l0 += kThreads / (TN / 4)) {
      const int lr = l0 + tid / (TN / 4), have = lr < m_rows ? live : 0;
      const int64_t m = m0 + lr;
      const f32x4_t w = *(const f32x4_t*)&ctile[lr * CS + lc];
      float v[4] = {w[0], w[1], w[2], w[3]};
      leave_outside_taps_out(p, BF, (int)m, (int)n, have, v);
      if (have) store_results(p, p.C, m * p.c_ms + n, v, have);
    }
    return;
  }
  if (live == 0) return;
  for (int lr = tid / (TN / 4); lr < m_rows; lr += kThreads / (TN / 4)) {
    const int64_t m = m0 + lr;
    const f32x4_t w = *(const f32x4_t*)&ctile[lr * CS + lc];
    if (p.ws != nullptr) {
      // (rows of the workspace are whole 16-byte vectors)
      *(f32x4_t*)(p.ws + (((int64_t)blockIdx.y * p.ws_rows + (int64_t)batch * p.M + m) * p.ws_pitch + n)) = w;
    } else {
      float v[4] = {w[0], w[1], w[2], w[3]};
      const int64_t at = c_at + m * p.c_ms;
      strided_tail(p, v, at, n, live);
      store_results(p, p.C, at + n, v, live);
    }
  }
}

// Adds the partial results up and runs the tail: PARTS threads per four columns of a row, each with a run of the splits in their
// order, whose sums are added up in that order.  (What bounds it is a thread's chain of loads, eight at a time: 153 x 38 results
// of 241 splits 20.2 us with one thread each, 5.4 with sixteen.)
template <int PARTS>
__global__ __launch_bounds__(256) void strided_reduce_kernel(StridedArgs p_by_value) {
  const StridedArgs& p = *(const StridedArgs*)(const __attribute__((address_space(4))) void*)__builtin_amdgcn_kernarg_segment_ptr();
  constexpr int G = 256 / PARTS;
  __shared__ f32x4_t sums[PARTS > 1 ? 256 : 1];
  const int64_t per_row = p.ws_pitch / 4;
  int64_t g = (int64_t)blockIdx.x * G + threadIdx.x % G;
  const int part = threadIdx.x / G, per = (p.splits + PARTS - 1) / PARTS, first = part * per;
  const int behind = first + per < p.splits ? first + per : p.splits;
  const bool conv = p.row_cols != 0;
  bool mine = g < p.ws_rows * per_row;
  if (!mine) {
    if (!conv && PARTS == 1) return;
    g = 0;  // (every lane stays: see leave_outside_taps_out)
  }
  const int64_t row = g / per_row, n = (g - row * per_row) * 4;
  const f32x4_t* at = (const f32x4_t*)(p.ws + row * p.ws_pitch + n);
  const int64_t step = p.ws_rows * p.ws_pitch / 4;
  f32x4_t sum = {0.f, 0.f, 0.f, 0.f};
  for (int s = first; s < behind; s += 8) {
    f32x4_t got[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) got[u] = s + u < behind ? at[(s + u) * step] : f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int u = 0; u < 8; ++u) sum += got[u];
  }
  if constexpr (PARTS > 1) {
    sums[threadIdx.x] = sum;
    __syncthreads();
    if (threadIdx.x >= (G + 63) / 64 * 64) return;  // (whole wavefronts)
    mine = mine && part == 0;
    if (!mine && !conv) return;
#pragma unroll
    for (int q = 1; q < PARTS; ++q) sum += sums[q * G + threadIdx.x % G];
  }
  float v[4] = {sum[0], sum[1], sum[2], sum[3]};
  int64_t b = row / p.M, c_at = (row - b * p.M) * p.c_ms;
  for (int d = p.n_batch - 1; d >= 0; --d) {
    c_at += (b % p.batch[d]) * p.c_batch[d];
    b /= p.batch[d];
  }
  const int live = p.N - n < 4 ? (int)(p.N - n) : 4;
  if (conv) {
    leave_outside_taps_out(p, p.out_bf16, (int)row, (int)n, mine ? live : 0, v);
    if (!mine) return;
  }
  strided_tail(p, v, c_at, n, live);
  store_results(p, p.C, c_at + n, v, live);
}

template <bool BF, int AMODE, int BMODE, int MI, int NI, bool FLAT = false>
hipError_t launch_tile(const StridedArgs& a, hipStream_t s) {
  const size_t lds = std::max<size_t>(2 * (Side<BF, AMODE, 64 * MI, FLAT>::kBytes + Side<BF, BMODE, 64 * NI, FLAT>::kBytes), 64 * MI * (64 * NI + 4) * 4);
  auto kern = strided_kernel<BF, AMODE, BMODE, MI, NI, FLAT>;
  static DynamicLdsLimit limit;
  if (hipError_t e = limit.ensure((const void*)kern, lds); e != hipSuccess) return e;
  int64_t nb = (int64_t)a.tiles_m * a.tiles_n;
  for (int d = 0; d < a.n_batch; ++d) nb *= a.batch[d];
  hipLaunchKernelGGL(kern, dim3((unsigned)nb, (unsigned)a.splits), dim3(kThreads), lds, s, a);
  return hipGetLastError();
}

// Whether a filter gradient's loads go out whole.  With a branch per run the loads of a slab wait for each other, without one every
// run's place and what it keeps are counted out ahead: 35 registers more and twice the instructions.  That pays in bf16, with half the values
// a load's wait: of 105 sizes 1.03 x as fast (10000 pixels of 3 x 177 x 242 34.9 -> 31.5 us, 30276 of 3 x 519 x 62
// 72.2 -> 55.1).  It does not in fp32 (135 sizes, run by run 1.06 x as fast, none slower; 33800 pixels of 5 x 185 x 95 130.2 -> 122.9, one pixel
// of 8 x 47 5.0 -> 4.5), nor for two slabs and less (4 pixels of 7 x 106 5.7 -> 5.0), nor for many pixels of long windows, whose tiles keep
// every CU at its instructions (5000 of 5 x 480 x 96 38.2 -> 30.2, 12150 of 5 x 775 x 68 123.7 -> 101.2, 2028 of 7 x 434 x 200 39.2 -> 31.7; but
// 17787 of 5 x 430 x 45 0.89 x, 35000 of 5 x 375 x 24 0.93, and where the tiles alone are more than the CUs 2916 of 7 x 1386 x 164 0.92).
bool flat_fetch(const StridedArgs& a) {
  return a.K > 128 && !(a.splits > 1 && a.M >= 5 * a.row_cols && a.M >= 2240 && a.K >= 2000);
}

template <bool BF, int MI>
hipError_t launch_modes(const StridedArgs& a, int amode, int bmode, hipStream_t s) {
  if (amode == ROWS_CONV) {
    if constexpr (BF)
      if (flat_fetch(a)) return launch_tile<BF, ROWS_CONV, ROWS_M, MI, MI, true>(a, s);
    return launch_tile<BF, ROWS_CONV, ROWS_M, MI, MI>(a, s);
  }
  if (amode == ROWS_K) return bmode == ROWS_K ? launch_tile<BF, ROWS_K, ROWS_K, MI, MI>(a, s) : launch_tile<BF, ROWS_K, ROWS_M, MI, MI>(a, s);
  return bmode == ROWS_K ? launch_tile<BF, ROWS_M, ROWS_K, MI, MI>(a, s) : launch_tile<BF, ROWS_M, ROWS_M, MI, MI>(a, s);
}

// Few result tiles: the direct form (direct.hip has the reasons), over rows of any alignment.  16 MB x 64 results per
// workgroup; its eight wavefronts share K and load fragments from memory into registers, the whole steps of K without a
// check per lane (rows past the last one are read as the last one and never stored), U steps in flight; what is left of K
// after the last whole step is the last wavefront's.  A lane holds the columns 4 r .. 4 r + 3 of a 16-row block: from a
// [K][N] right-hand side four neighbours of every K-row, turned with v_perm (bf16) or by naming (fp32), near the right edge
// the last four columns instead; from an [N][K] one four rows.  The partial tiles meet in LDS and are added in wavefront order.
// WORDS (bf16, matrices below 2 GiB): rows that begin at any value are fetched as the aligned words around a lane's values,
// through descriptors that end with the matrix, and shifted together (16-byte loads from 2-byte boundaries reach 17 KB a
// microsecond and CU); a broken last step of K is a step like the others with the values past K cleared on both sides.
// Columns past N are whatever follows, and never stored.  Two steps in flight: three and four are slower (registers).
// 300 x 777, K = 1001 10.1 -> 7.1 us from [K][N], 15.1 -> 9.4 from [N][K]; 33 x 131, K = 255 8.7 -> 4.6; 1000 x 1001, K = 1001
// 19.6 -> 13.2.
template <bool BF, int BMODE, int MB, bool WORDS>
__global__ __launch_bounds__(512, 4) void product_direct_kernel(StridedArgs p_by_value) {
  const StridedArgs& p = *(const StridedArgs*)(const __attribute__((address_space(4))) void*)__builtin_amdgcn_kernarg_segment_ptr();
  constexpr int kWaves = 8, TM = 16 * MB, TN = 64, CS = TN + 4, ES = BF ? 2 : 4;
  constexpr int E = 16 / ES, KS = 4 * E;  // K-values per lane and step, per step
  constexpr int U = !WORDS && MB == 1 ? 4 : 2, NA = BF ? 1 : 2;
  static_assert(!WORDS || BF, "fp32 values are words wherever they lie");
  extern __shared__ __attribute__((aligned(16))) char smem[];
  float* const parts = (float*)smem;  // [wavefront][TM][CS]
  const int tid = threadIdx.x, lane = tid & 63, r = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);

  // XCD x (workgroup ids x, x + 8, ...) takes a run of tiles, the rows of a column block one after the other
  const unsigned nb = gridDim.x, x = blockIdx.x & 7u, rem = nb & 7u;
  unsigned t = x * (nb >> 3) + (x < rem ? x : rem) + (blockIdx.x >> 3);
  const int64_t m0 = (int64_t)(t % (unsigned)p.tiles_m) * TM;
  t /= (unsigned)p.tiles_m;
  const int64_t n0 = (int64_t)(t % (unsigned)p.tiles_n) * TN;
  t /= (unsigned)p.tiles_n;
  int64_t a_at = 0, b_at = 0, c_at = 0;
  for (int d = p.n_batch - 1; d >= 0; --d) {
    const unsigned sz = (unsigned)p.batch[d], i = t % sz;
    t /= sz;
    a_at += i * p.a_batch[d];
    b_at += i * p.b_batch[d];
    c_at += i * p.c_batch[d];
  }

  const int64_t steps = WORDS ? (p.K + KS - 1) / KS : p.K / KS;  // (whole ones)
  const int64_t per = (steps + kWaves - 1) / kWaves, first = wave * per;
  const int64_t last = first + per < steps ? first + per : steps;

  constexpr unsigned kFlags = 0x00020000u;     // raw buffer, 32-bit data format
  constexpr unsigned kOutside = 0x80000000u;   // past every range, with any offset below 2 GiB added
  const int64_t n = n0 + 4 * r;
  const int64_t b_pitch = p.b_ks * ES;
  constexpr int NB = BMODE == ROWS_K ? 4 : 1;
  const char* a_ptr[WORDS ? 1 : MB];
  const char* b_ptr[WORDS ? 1 : NB];
  // WORDS: offsets of the words the lane's chunks begin in, and by how many bits the values begin behind that
  unsigned a_off[MB], a_shift[MB], b_off[NB], b_shift[NB];
  int b_rem = 0;
  __amdgpu_buffer_rsrc_t ra, rb;
  if constexpr (WORDS) {
    auto matrix = [&](const void* base, int64_t at, int64_t values, int* rem) {
      const uintptr_t first = (uintptr_t)base + (uintptr_t)(at * ES);
      *rem = (int)(first & 3);
      return __builtin_amdgcn_make_buffer_rsrc((void*)(first - *rem), 0, (*rem + (int)(values * ES) + 3) & ~3, kFlags);
    };
    int a_rem;
    ra = matrix(p.A, a_at, (p.M - 1) * p.a_ms + p.K, &a_rem);
    rb = matrix(p.B, b_at, (p.K - 1) * p.b_ks + (p.N - 1) * p.b_ns + 1, &b_rem);
#pragma unroll
    for (int i = 0; i < MB; ++i) {
      const int64_t m = m0 + 16 * i + r;
      const unsigned at = (unsigned)((m * p.a_ms + g * E) * ES) + (unsigned)a_rem;
      a_off[i] = m < p.M ? at & ~3u : kOutside;
      a_shift[i] = (at & 3) * 8;
    }
#pragma unroll
    for (int j = 0; j < NB; ++j) {
      const unsigned at = BMODE == ROWS_K ? (unsigned)(((n + j) * p.b_ns + g * E) * ES) + (unsigned)b_rem : (unsigned)((n + g * E * p.b_ks) * ES);
      b_off[j] = n + j < p.N ? (BMODE == ROWS_K ? at & ~3u : at) : kOutside;
      b_shift[j] = (at & 3) * 8;
    }
  } else {
#pragma unroll
    for (int i = 0; i < MB; ++i) {
      const int64_t m = m0 + 16 * i + r;
      a_ptr[i] = (const char*)p.A + (a_at + (m < p.M ? m : p.M - 1) * p.a_ms + g * E) * ES;
    }
    if constexpr (BMODE == ROWS_K) {
#pragma unroll
      for (int j = 0; j < 4; ++j) b_ptr[j] = (const char*)p.B + (b_at + (n + j < p.N ? n + j : p.N - 1) * p.b_ns + g * E) * ES;
    } else {
      b_ptr[0] = (const char*)p.B + (b_at + (n + 4 <= p.N ? n : p.N - 4) + g * E * p.b_ks) * ES;  // (N is at least four)
    }
  }

  f32x4_t sums[MB][4][NA];
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int c = 0; c < NA; ++c) sums[i][j][c] = f32x4_t{0.f, 0.f, 0.f, 0.f};

  auto multiply = [&](const Words<4> (&fa)[MB], const uint32_t (&raw)[16]) {
    Words<4> frag[4];
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        if constexpr (BMODE == ROWS_K)
          frag[j].w[q] = raw[4 * j + q];
        else if constexpr (BF)
          frag[j].w[q] = __builtin_amdgcn_perm(raw[4 * q + 2 + (j >> 1)], raw[4 * q + (j >> 1)], (j & 1) ? 0x07060302u : 0x05040100u);
        else
          frag[j].w[q] = raw[4 * q + j];
      }
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        if constexpr (BF) {
          bf16x8_t av, bv;
          __builtin_memcpy(&av, &fa[i], 16);
          __builtin_memcpy(&bv, &frag[j], 16);
          sums[i][j][0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bv, av, sums[i][j][0], 0, 0, 0);
        } else {
#pragma unroll
          for (int q = 0; q < 4; ++q)
            sums[i][j][q % NA] = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(frag[j].w[q]), __uint_as_float(fa[i].w[q]), sums[i][j][q % NA], 0, 0, 0);
        }
      }
  };

  if constexpr (WORDS) {
    constexpr int WB = BMODE == ROWS_K ? 20 : 24;  // words fetched of B's 16
    typedef int i32x3_t __attribute__((ext_vector_type(3)));
    auto fetch5 = [](__amdgpu_buffer_rsrc_t rs, unsigned off, uint32_t* to) {
      const i32x4_t v = __builtin_bit_cast(i32x4_t, __builtin_amdgcn_raw_buffer_load_b128(rs, (int)off, 0, 0));
#pragma unroll
      for (int q = 0; q < 4; ++q) to[q] = (uint32_t)v[q];
      to[4] = (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(rs, (int)(off + 16), 0, 0);
    };
    for (int64_t s0 = first; s0 < last; s0 += U) {
      uint32_t wa[U][MB][5], wb[U][WB];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const bool live = s0 + u < last;
        const unsigned k = (unsigned)((s0 + u) * KS);
#pragma unroll
        for (int i = 0; i < MB; ++i) fetch5(ra, live ? a_off[i] + k * ES : kOutside, wa[u][i]);
        if constexpr (BMODE == ROWS_K) {
#pragma unroll
          for (int j = 0; j < 4; ++j) fetch5(rb, live ? b_off[j] + k * ES : kOutside, &wb[u][5 * j]);
        } else {
          const unsigned at = b_off[0] + k * (unsigned)b_pitch;
#pragma unroll
          for (int e = 0; e < E; ++e) {
            const bool in = live & (b_off[0] != kOutside) & (k + g * E + e < (unsigned)p.K);
            const i32x3_t v = __builtin_bit_cast(i32x3_t, __builtin_amdgcn_raw_buffer_load_b96(rb, (int)(in ? at + (unsigned)((b_rem + e * (int)b_pitch) & ~3) : kOutside), 0, 0));
#pragma unroll
            for (int q = 0; q < 3; ++q) wb[u][3 * e + q] = (uint32_t)v[q];
          }
        }
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        if (s0 + u >= last) continue;
        Words<4> fa[MB];
        uint32_t raw[16];
#pragma unroll
        for (int i = 0; i < MB; ++i)
#pragma unroll
          for (int q = 0; q < 4; ++q) fa[i].w[q] = __builtin_amdgcn_alignbit(wa[u][i][q + 1], wa[u][i][q], a_shift[i]);
        if constexpr (BMODE == ROWS_K) {
#pragma unroll
          for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int q = 0; q < 4; ++q) raw[4 * j + q] = __builtin_amdgcn_alignbit(wb[u][5 * j + q + 1], wb[u][5 * j + q], b_shift[j]);
        } else {
#pragma unroll
          for (int e = 0; e < E; ++e) {
            const unsigned shift = (unsigned)((b_rem + e * (int)b_pitch) & 3) * 8;
#pragma unroll
            for (int q = 0; q < 2; ++q) raw[2 * e + q] = __builtin_amdgcn_alignbit(wb[u][3 * e + q + 1], wb[u][3 * e + q], shift);
          }
        }
        if ((s0 + u + 1) * KS > p.K) {
          // the values past K: cleared in A, and in B where a lane holds values of K (its rows past K arrive as zeros)
          const int have = (int)(p.K - (s0 + u) * KS) - g * E;
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            const uint32_t keep = 2 * q + 1 < have ? 0xffffffffu : 2 * q < have ? 0xffffu : 0u;
#pragma unroll
            for (int i = 0; i < MB; ++i) fa[i].w[q] &= keep;
            if constexpr (BMODE == ROWS_K) {
#pragma unroll
              for (int j = 0; j < 4; ++j) raw[4 * j + q] &= keep;
            }
          }
        }
        multiply(fa, raw);
      }
    }
  }
  for (int64_t s0 = first; !WORDS && s0 < last; s0 += U) {
    Words<4> fa[U][MB];
    uint32_t raw[U][16];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int64_t k = (s0 + u < last ? s0 + u : last - 1) * KS;  // (a step past the run is read again and not multiplied)
#pragma unroll
      for (int i = 0; i < MB; ++i) fa[u][i] = load_words<4>(a_ptr[WORDS ? 0 : i] + k * ES);
      if constexpr (BMODE == ROWS_K) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const Words<4> v = load_words<4>(b_ptr[WORDS ? 0 : j] + k * ES);
#pragma unroll
          for (int q = 0; q < 4; ++q) raw[u][4 * j + q] = v.w[q];
        }
      } else {
#pragma unroll
        for (int e = 0; e < E; ++e) {
          const Words<ES> v = load_words<ES>(b_ptr[0] + (k + e) * b_pitch);
#pragma unroll
          for (int q = 0; q < ES; ++q) raw[u][ES * e + q] = v.w[q];
        }
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (s0 + u < last) multiply(fa[u], raw[u]);
  }

  const int left = WORDS ? 0 : (int)(p.K - steps * KS);
  if (left > 0 && wave == kWaves - 1) {
    // value by value, zeros past the end on both sides
    const int64_t k = steps * KS;
    Words<4> fa[MB];
    uint32_t raw[16];
    auto value = [&](const char* at, bool ok) -> uint32_t { return !ok ? 0u : BF ? *(const uint16_t*)at : *(const uint32_t*)at; };
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const char* const at = a_ptr[WORDS ? 0 : i] + k * ES + 4 * q;
        const int kk = g * E + (BF ? 2 * q : q);
        fa[i].w[q] = value(at, kk < left) | (BF ? value(at + 2, kk + 1 < left) << 16 : 0u);
      }
    if constexpr (BMODE == ROWS_K) {
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const char* const at = b_ptr[WORDS ? 0 : j] + k * ES + 4 * q;
          const int kk = g * E + (BF ? 2 * q : q);
          raw[4 * j + q] = value(at, kk < left) | (BF ? value(at + 2, kk + 1 < left) << 16 : 0u);
        }
    } else {
#pragma unroll
      for (int e = 0; e < E; ++e)
#pragma unroll
        for (int q = 0; q < ES; ++q) {
          const char* const at = b_ptr[0] + (k + e) * b_pitch + 4 * q;
          raw[ES * e + q] = value(at, g * E + e < left) | (BF ? value(at + 2, g * E + e < left) << 16 : 0u);
        }
    }
    multiply(fa, raw);
  }

  // lane r, g holds row r and, of block j, the rows 4 g + e: column 4 (4 g + e) + j
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      f32x4_t q = {sums[i][0][0][e], sums[i][1][0][e], sums[i][2][0][e], sums[i][3][0][e]};
      if constexpr (NA == 2) q += f32x4_t{sums[i][0][1][e], sums[i][1][1][e], sums[i][2][1][e], sums[i][3][1][e]};
      *(f32x4_t*)&parts[(wave * TM + 16 * i + r) * CS + 16 * g + 4 * e] = q;
    }
  __syncthreads();
  const int lr = tid / 16, lc = (tid & 15) * 4;
  const int64_t m = m0 + lr, col = n0 + lc;
  if (lr >= TM || m >= p.M || col >= p.N) return;
  const float* const at = &parts[lr * CS + lc];
  f32x4_t sum = *(const f32x4_t*)at;
#pragma unroll
  for (int w = 1; w < kWaves; ++w) sum += *(const f32x4_t*)(at + w * (TM * CS));
  const int live = p.N - col < 4 ? (int)(p.N - col) : 4;
  float v[4] = {sum[0], sum[1], sum[2], sum[3]};
  if (!WORDS && BMODE != ROWS_K && live < 4) {  // the quad holds the last four columns: its own are the last `live` of them
    v[0] = live == 3 ? sum[1] : live == 2 ? sum[2] : sum[3];
    v[1] = live == 3 ? sum[2] : sum[3];
    v[2] = sum[3];
  }
  const int64_t c_row = c_at + m * p.c_ms;
  strided_tail(p, v, c_row, col, live);
  store_results(p, p.C, c_row + col, v, live);
}

// Whether a direct bf16 tile takes its rows as shifted words (offsets fit 31 bits): where one begins off a word or K ends
// within a step, and with 16 rows between 64 and 512 of K, where a wavefront has one or two steps and the other form fetches four
// (33 x 136, K = 256: [K][N] 5.1 -> 4.7 us, [N][K] 6.0 -> 5.4).
bool direct_by_words(const StridedArgs& a, int64_t rows) {
  int64_t odd = a.a_ms | (a.b_ks == 1 ? a.b_ns : a.b_ks);
  for (int d = 0; d < a.n_batch; ++d) odd |= a.a_batch[d] | a.b_batch[d];
  const bool off_words = (odd & 1) != 0 || (((uintptr_t)a.A | (uintptr_t)a.B) & 3) != 0;
  if (!off_words && a.K % 32 == 0 && (rows != 16 || a.K <= 64 || a.K > 512)) return false;
  const int64_t limit = ((int64_t)1 << 30) - 64;
  return (double)a.M * (double)a.a_ms + (double)a.K < (double)limit &&
         (double)(a.K + 64) * (double)a.b_ks + (double)a.N * (double)a.b_ns < (double)limit;
}

template <bool BF, int BMODE, int MB, bool WORDS = false>
hipError_t launch_direct(const StridedArgs& a, hipStream_t s) {
  if constexpr (BF && !WORDS)
    if (direct_by_words(a, 16 * MB)) return launch_direct<BF, BMODE, MB, true>(a, s);
  const size_t lds = (size_t)8 * 16 * MB * 68 * 4;
  auto kern = product_direct_kernel<BF, BMODE, MB, WORDS>;
  static DynamicLdsLimit limit;
  if (hipError_t e = limit.ensure((const void*)kern, lds); e != hipSuccess) return e;
  StridedArgs b = a;
  b.tiles_m = (int)((a.M + 16 * MB - 1) / (16 * MB));
  b.tiles_n = (int)((a.N + 63) / 64);
  int64_t nb = (int64_t)b.tiles_m * b.tiles_n;
  for (int d = 0; d < a.n_batch; ++d) nb *= a.batch[d];
  if (nb <= 0 || nb > kMaxLaunchThreads / 512) return hipErrorInvalidValue;
  hipLaunchKernelGGL(kern, dim3((unsigned)nb), dim3(512), lds, s, b);
  return hipGetLastError();
}

}  // namespace

// Which of its two kernels a product takes -- the direct tile's rows (16 or 32), or 0: the tiles through LDS that strided_plan
// has laid out -- and what it is expected to take in microseconds (an infinity: neither can be launched).  Both sides are
// priced from 25 shapes per type and layout (1 to 2000 rows, K of 32 to 2047, batches up to 96) and from 45 with many small
// tiles (batches of 100 to 100000, 1 to 128 rows and columns, K of 3 to 4096); bf16 again from 136 of both sorts, half of them
// with odd rows, and the choice checked on 70 others: it takes 0.9 % longer than the best of the three would on average.
// Direct, fp32: 2.6 plus, per round of one tile on each CU, 0.8 (1.4 from the second round on where K has a broken last step)
// and the tile's operand bytes at 38 KB a microsecond with 16 rows, 32 with 32 rows (the matrix cores).  Direct, bf16, whose
// workgroups share CUs: 3.6 plus the operand bytes at 60 KB a microsecond from [K][N] and 38 from [N][K], 48 and 28 as shifted
// words, and for every further tile per CU as much and 0.95, with 32 rows 0.5 once.  Through LDS: 3 and 1.65 a slab (bf16 4.8 and
// 1.5, [N][K] 1.1); every further round 0.6 and 0.95 a slab (bf16 0.8 and 0.5, 1.2 from odd [K][N] rows, [N][K] 0.9 and 0.35,
// 0.55 more where the rows are read element by element); tiles of 128 in the first round 4 and 6 (bf16 10 and 6 or 2.5), in the
// others 1.5 and 3.1 (bf16 1 and 6, 1.7 and 1.75); split, 1.8 more and the partial results written and read at 3 TB/s.  A direct
// fp32 tile has to be 8 % ahead.
//   us, through LDS -> direct              fp32 [K][N]       bf16 [K][N]       bf16 [N][K]
//   3 x 1001, K = 333                    14.9 ->  5.0      13.5 ->  4.2      11.0 ->  4.6
//   300 x 777, K = 1001                  20.5 -> 10.9      14.4 ->  7.2      13.3 ->  9.4
//   1000 x 1001, K = 1001                55.3 -> 32.1      28.7 -> 13.2      22.2 -> 18.7
//   20 of 100 x 77, K = 100              10.4 ->  4.6       8.6 ->  4.5       7.8 ->  4.4
//   50 x 777, K = 1777: fp32, [N][K] split  13.6 (22.1)    13.1 ->  9.1      12.0 (14.0)
//   10000 of 1 x 16, K = 64              99.4 -> 66.2        60 ->   45        46 ->   40
//   10000 of 17 x 17, K = 17                                 68 ->   54        54 ->   48
//   96 of 128 x 64, K = 128                                 6.9 ->  4.5       6.4 ->  5.2
//   1000 of 1 x 1, K = 4096               463 -> 113                          135 ->   23
int product_direct_rows(const StridedArgs& a, bool bf, int mi, int n_cus, double* us) {
  const bool nk = a.b_ks == 1;
  double batches = 1;
  for (int d = 0; d < a.n_batch; ++d) batches *= (double)a.batch[d];
  const double never = std::numeric_limits<double>::infinity();
  const double lds_tiles = batches * (double)a.tiles_m * (double)a.tiles_n;
  double lds_us = never;
  if (lds_tiles * kThreads <= (double)kMaxLaunchThreads) {
    const double slabs = (double)((std::min(a.K, a.k_per_split) + (bf ? 63 : 31)) / (bf ? 64 : 32));
    const double more = std::max(0.0, lds_tiles / n_cus - 1);
    const bool gathered = bf && a.a_ks != 1 && a.a_ms != 1;
    double first, each;
    if (mi == 2) {
      first = !bf ? 4 + 6 * slabs : 10 + (nk ? 2.5 : 6) * slabs;
      each = !bf ? 1.5 + 3.1 * slabs : nk ? 1.7 + 1.75 * slabs : 1 + 6 * slabs;
    } else {
      first = !bf ? 3 + 1.65 * slabs : nk ? 4.8 + 1.1 * slabs : 4.8 + 1.5 * slabs;
      each = !bf ? 0.6 + 0.95 * slabs : nk ? 0.9 + 0.35 * slabs : 0.8 + 0.5 * slabs;
      if (bf && !nk && (a.b_ks & 1)) each += 0.7 * slabs;
      if (gathered) each += 0.55 * slabs * (double)std::min<int64_t>(a.M, 64) / 64;
    }
    lds_us = first + more * each;
    if (a.splits > 1) lds_us += 1.8 + 8.0 * a.splits * (double)a.ws_rows * (double)a.ws_pitch / 3e6;
  }
  const double kb = (double)a.K * (bf ? 2 : 4);
  auto direct_us = [&](int64_t rows) {
    const double tiles = batches * (double)((a.M + rows - 1) / rows) * (double)((a.N + 63) / 64);
    if (tiles * 512 > (double)kMaxLaunchThreads) return never;
    const double live = (double)(rows == 16 ? std::min<int64_t>(a.M, 16) : 32) + 64;
    if (bf) {
      const double each = live * kb / (direct_by_words(a, rows) ? (nk ? 28e3 : 48e3) : nk ? 38e3 : 60e3), more = std::max(0.0, tiles / n_cus - 1);
      return 3.6 + each + more * (0.95 + each) + (rows == 32 ? 0.5 * std::min(1.0, more) : 0);
    }
    const double rate = rows == 16 ? 38e3 : 32e3;
    const double rounds = std::ceil(tiles / n_cus);
    return 2.6 + rounds * (0.8 + live * kb / rate) + (a.K % 16 != 0 ? 0.6 * (rounds - 1) : 0);
  };
  *us = lds_us;
  if (a.a_ks != 1 || (!nk && (a.b_ns != 1 || a.N < 4))) return 0;
  const double small = direct_us(16), large = direct_us(32), direct = std::min(small, large);
  if (direct > (bf ? 1 : 0.92) * lds_us || direct == never) return 0;
  *us = direct;
  return small <= large ? 16 : 32;
}

hipError_t product_direct_launch(const StridedArgs& a, bool bf, int rows, hipStream_t s) {
  const bool nk = a.b_ks == 1;
  if (bf) {
    if (rows == 16) return nk ? launch_direct<true, ROWS_K, 1>(a, s) : launch_direct<true, ROWS_M, 1>(a, s);
    return nk ? launch_direct<true, ROWS_K, 2>(a, s) : launch_direct<true, ROWS_M, 2>(a, s);
  }
  if (rows == 16) return nk ? launch_direct<false, ROWS_K, 1>(a, s) : launch_direct<false, ROWS_M, 1>(a, s);
  return nk ? launch_direct<false, ROWS_K, 2>(a, s) : launch_direct<false, ROWS_M, 2>(a, s);
}

// The tile and, for few tiles and a long K, the split: 128 x 128 where that still gives every CU a workgroup (half the
// operand traffic per result) and covers at most a third more results than 64 x 64, which otherwise is the tile (1000 of
// 64 x 64 with K = 64, fp32: 43.7 us with tiles of 128, three quarters of them empty, 18.7 with tiles of 64; 1000 of 48 x 48,
// K = 33, bf16: 44.1 and 18.4); K is split when the tiles alone leave CUs idle, into runs of at least
// four slabs, for about three workgroups per CU (their LDS fits four times into one).  A filter gradient's slab takes as long as
// its loads: runs of two slabs and more (567 pixels of 3 x 45 x 20 in bf16 12.4 -> 9.5 us, 2116 of 3 x 60 x 18 in fp32 12.4 -> 9.2),
// and in fp32, whose workgroups fit four times into a CU's registers, four per CU (50176 of 3 x 192 x 64 64.5 -> 61.1) -- but for
// partial results in fp32 of 300 KB a split, which a second launch reads again: those only up to 6 MB, or with six slabs a run left (1512
// pixels of 3 x 348 x 112 in fp32, 468 KB: 12 splits 18.2, 24 of two slabs 20.1; 2173 of 3 x 510 x 66, 404 KB: 14 24.1, 17 25.7;
// bf16, whose slabs are twice the pixels, takes them: 900 of 3 x 456 x 240 4 splits 1.07 x as long as 7, 2304 of 3 x 438 x 190 9 1.07 x 13).
void strided_plan(StridedArgs* a, bool bf, bool conv, int n_cus, int* mi) {
  int64_t batches = 1;
  for (int d = 0; d < a->n_batch; ++d) batches *= a->batch[d];
  const int64_t bk = bf ? 64 : 32, slabs = (a->K + bk - 1) / bk;
  auto tiles = [&](int64_t t) {
    const int64_t rows = conv ? (a->M / a->row_cols) * ((a->row_cols + t - 1) / t) : (a->M + t - 1) / t;
    return rows * ((a->N + t - 1) / t) * batches;
  };
  *mi = tiles(128) >= n_cus && 3 * tiles(128) <= tiles(64) ? 2 : 1;
  const int64_t t = 64 * *mi;
  a->tiles_per_tap = conv ? (int)((a->row_cols + t - 1) / t) : 1;
  a->tiles_m = conv ? (int)(a->M / a->row_cols) * a->tiles_per_tap : (int)((a->M + t - 1) / t);
  a->tiles_n = (int)((a->N + t - 1) / t);
  a->splits = 1;
  a->k_per_split = slabs * bk;
  a->ws_rows = batches * a->M;
  a->ws_pitch = (a->N + 3) / 4 * 4;
  const int64_t have = tiles(t);
  if (have < n_cus && slabs >= 8) {
    const int64_t three = (3 * n_cus + have - 1) / have, bytes = std::max<int64_t>(1, a->ws_rows * a->ws_pitch * 4);
    int64_t want = std::min(three, slabs / 4);
    if (conv) {
      const int64_t fits = bf || bytes <= 300 << 10 ? slabs : std::max(((int64_t)6 << 20) / bytes, slabs / 6);
      want = std::max(want, std::min({bf ? three : 4 * n_cus / have, slabs / 2, fits}));
    }
    // the partial results: at most 256 MiB of them
    want = std::min<int64_t>(want, ((int64_t)256 << 20) / bytes);
    if (want >= 2) {
      const int64_t per = (slabs + want - 1) / want;
      a->k_per_split = per * bk;
      a->splits = (int)((slabs + per - 1) / per);
    }
  }
}

hipError_t strided_launch(const StridedArgs& a, bool bf, bool conv, int mi, hipStream_t s) {
  int64_t nb = (int64_t)a.tiles_m * a.tiles_n;
  for (int d = 0; d < a.n_batch; ++d) nb *= a.batch[d];
  if (nb <= 0 || nb > kMaxLaunchThreads / kThreads || a.splits < 1 || a.splits > 65535 || (a.splits > 1) != (a.ws != nullptr)) return hipErrorInvalidValue;
  const int amode = conv ? ROWS_CONV : (a.a_ks == 1 ? ROWS_K : ROWS_M), bmode = a.b_ks == 1 && !conv ? ROWS_K : ROWS_M;
  hipError_t e;
  if (bf)
    e = mi == 2 ? launch_modes<true, 2>(a, amode, bmode, s) : launch_modes<true, 1>(a, amode, bmode, s);
  else
    e = mi == 2 ? launch_modes<false, 2>(a, amode, bmode, s) : launch_modes<false, 1>(a, amode, bmode, s);
  if (e != hipSuccess || a.splits == 1) return e;
  // threads per four results: so many that a thread's splits are one round of loads, while workgroups are few
  const int64_t groups = a.ws_rows * (a.ws_pitch / 4);
  int parts = 1;
  while (parts < 16 && a.splits > 8 * parts && groups * parts < 256 * 1024) parts *= 2;
  const int64_t blocks = (groups * parts + 255) / 256;
  if (blocks > kMaxLaunchThreads / 256) return hipErrorInvalidValue;
  auto* const kern = parts == 1 ? strided_reduce_kernel<1> : parts == 2 ? strided_reduce_kernel<2> : parts == 4 ? strided_reduce_kernel<4>
                     : parts == 8 ? strided_reduce_kernel<8> : strided_reduce_kernel<16>;
  hipLaunchKernelGGL(kern, dim3((unsigned)blocks), dim3(256), 0, s, a);
  return hipGetLastError();
}

namespace {

// The columns of a strided convolution's data gradient, cols[pixel of the gradient][ky][kx][ci] in fp32, added up into
// the image: an image value takes the columns of every tap and gradient pixel whose window covers it, taps in order.
// A thread per V channels of an image pixel (the last V of a pixel overlap the ones before them where CI is no multiple of V);
// columns are read once, V * 4 bytes at a time.  What bounds it is a thread's chain of loads: only the taps that meet a gradient
// pixel are visited, up to four of a filter row are on their way at once.  5 x 75 x 75 x 121 from 5 x 5 taps of stride 2, bf16:
// 60 us a value a thread and a tap at a time, now 16.  Few taps are a chain of divisions: those by W and the strides are multiplies.
// ONE: filters of one tap, where there is nothing to add up.
template <bool BF, int V, bool ONE>
__global__ __launch_bounds__(256) void col2im_kernel(Col2imArgs a) {
  const unsigned cv = (unsigned)(a.CI + V - 1) / V, per_img = (unsigned)(a.H * a.W);
  const unsigned g = blockIdx.x * 256 + threadIdx.x;
  const unsigned at_pixel = g / cv;  // (up to 2^32 of them: no multiply-and-shift)
  if (at_pixel >= (unsigned)a.N * per_img) return;
  const unsigned chunk = g - at_pixel * cv, img = at_pixel / per_img, pix = at_pixel - img * per_img;
  const int y = (int)fast_div(pix, a.w_magic, a.w_shift), x = (int)(pix - (unsigned)y * (unsigned)a.W);
  const int c = (int)chunk * V + V <= a.CI ? (int)chunk * V : a.CI - V;
  float sum[V];
#pragma unroll
  for (int e = 0; e < V; ++e) sum[e] = 0.f;
  if constexpr (ONE) {
    const int ty = y + a.PH, tx = x + a.PW;  // (a crop, which is a negative padding, leaves pixels ahead of the first window)
    const int gy = (int)fast_div((unsigned)ty, a.sh_magic, a.sh_shift), gx = (int)fast_div((unsigned)tx, a.sw_magic, a.sw_shift);
    if (ty >= 0 && tx >= 0 && gy * a.SH == ty && gx * a.SW == tx && gy < a.OH && gx < a.OW) {
      const Words<V> w = load_words<V>(a.cols + (((int64_t)img * a.OH + gy) * a.OW + gx) * a.CI + c);
#pragma unroll
      for (int e = 0; e < V; ++e) sum[e] += __uint_as_float(w.w[e]);
    }
  } else {
    // the first tap of a column or row of them whose window meets a row or column of the gradient, and which; from there every
    // period-th does, further up and left (above and left of the gradient: no further tap meets it)
    auto first = [](int at, int taps, int period, int stride, unsigned magic, int shift, int dil, int* grad) {
      for (int k = 0; k < period && k < taps && at >= 0; ++k, at -= dil) {
        *grad = (int)fast_div((unsigned)at, magic, shift);
        if (*grad * stride == at) return k;
      }
      return taps;
    };
    int gy0 = 0, gx0 = 0;
    const int ky0 = first(y + a.PH, a.KH, a.period_h, a.SH, a.sh_magic, a.sh_shift, a.DH, &gy0);
    const int kx0 = first(x + a.PW, a.KW, a.period_w, a.SW, a.sw_magic, a.sw_shift, a.DW, &gx0);
    const int dy = a.step_h, dx = a.step_w;
    const int taps = a.KH * a.KW;
    for (int ky = ky0, gy = gy0; ky < a.KH; ky += a.period_h, gy -= dy) {
      if (gy < 0 || gy >= a.OH) continue;
      const float* const row = a.cols + ((int64_t)img * a.OH + gy) * a.OW * taps * a.CI + (int64_t)ky * a.KW * a.CI + c;
      constexpr int U = 4;
      for (int kx = kx0, gx = gx0; kx < a.KW; kx += U * a.period_w, gx -= U * dx) {
        Words<V> w[U];
        bool in[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const int k = kx + u * a.period_w, g = gx - u * dx;
          in[u] = k < a.KW && g >= 0 && g < a.OW;
          if (in[u]) w[u] = load_words<V>(row + ((int64_t)g * taps + k) * a.CI);
        }
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
          for (int e = 0; e < V; ++e) sum[e] += in[u] ? __uint_as_float(w[u].w[e]) : 0.f;
      }
    }
  }
  const int64_t o = (int64_t)at_pixel * a.CI + c;
  if constexpr (BF) {
    uint16_t h[V];
#pragma unroll
    for (int e = 0; e < V; ++e) h[e] = f32_to_bf16_bits(sum[e]);
    __builtin_memcpy((uint16_t*)a.out + o, h, sizeof h);
  } else {
    __builtin_memcpy((float*)a.out + o, sum, sizeof sum);
  }
}

// What the unit-stride data gradient's convolution reads, in one launch: the gradient's rows of `cols` elements copied to rows of
// whole 16-byte vectors, the rest of a row zeros (pad_rows = 0: they are so already), and its right-hand side
//   Bt[ci][tap][pitch] = F[taps - 1 - tap][ci][co]
// -- the filter's taps in reverse and the channels' roles exchanged, contiguous along what that convolution sums over.  The first
// `flip_blocks` workgroups flip.  A thread copies 16 bytes of a padded row: 154154 rows of 38 bf16 12.8 us an element at a time and
// 4.7 for the filter in a launch of its own, now 7.5 for both.
template <typename T>
__global__ __launch_bounds__(256) void gradient_operands_kernel(const T* in, T* out, int64_t pad_rows, int cols, int pitch, const T* f, T* bt, int taps, int ci,
                                                                 int co, int64_t flip_blocks) {
  if (blockIdx.x < flip_blocks) {
    const int64_t g = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (g >= (int64_t)ci * taps * co) return;
    const int c = (int)(g % co);
    const int64_t r = g / co;
    const int tap = (int)(r % taps), n = (int)(r / taps);
    bt[((int64_t)n * taps + tap) * pitch + c] = f[((int64_t)(taps - 1 - tap) * ci + n) * co + c];
    return;
  }
  constexpr int V = 16 / sizeof(T);
  const int64_t per_row = pitch / V, total = pad_rows * per_row, stride = (int64_t)(gridDim.x - flip_blocks) * 256;
  for (int64_t g = (blockIdx.x - flip_blocks) * 256 + threadIdx.x; g < total; g += stride) {
    const int64_t row = g / per_row;
    const int c = (int)(g - row * per_row) * V;
    T v[V];
    if (c + V <= cols) {
      __builtin_memcpy(v, in + row * cols + c, 16);
    } else {
#pragma unroll
      for (int e = 0; e < V; ++e) v[e] = c + e < cols ? in[row * cols + c + e] : (T)0;
    }
    __builtin_memcpy(out + g * V, v, 16);
  }
}

// The unit-stride data gradient runs as a convolution of the gradient, and the convolution kernels read taps outside the
// gradient as zeros: an infinite or NaN filter value times such a zero is a NaN in a result that the contraction leaves that
// tap out of.  Only pixels with a tap outside can be struck, and only by becoming a NaN: those that hold one are summed again
// without the taps outside.  A thread per value of the image's border: the rows above y0 and from y1 on, of the rows between
// them the columns left of x0 and from x1 on.  The launch adds 2 to 3 us: both gradients of 16 x 56 x 56 x 64 (*) 3 x 3 x 64
// 130 -> 133 us in fp32, 66 -> 69 in bf16.
template <bool BF>
__global__ __launch_bounds__(256) void conv_border_kernel(ConvBorderArgs a) {
  const int64_t full = (int64_t)(a.y0 + a.H - a.y1) * a.W, side = a.x0 + a.W - a.x1;
  const int64_t pixels = full + (int64_t)(a.y1 - a.y0) * side, total = (int64_t)a.N * pixels * a.CI;
  const int64_t stride = (int64_t)gridDim.x * 256;
  for (int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x; t < total; t += stride) {
    const int ci = (int)(t % a.CI);
    const int64_t at = t / a.CI, img = at / pixels, px = at - img * pixels;
    int y, x;
    if (px < full) {
      y = (int)(px / a.W);
      x = (int)(px - (int64_t)y * a.W);
      if (y >= a.y0) y += a.y1 - a.y0;
    } else {
      const int64_t r = px - full;
      y = (int)(r / side);
      x = (int)(r - y * side);
      y += a.y0;
      if (x >= a.x0) x += a.x1 - a.x0;
    }
    const int64_t o = ((img * a.H + y) * a.W + x) * a.CI + ci;
    const float had = BF ? bf16_bits_to_f32(((const uint16_t*)a.out)[o]) : ((const float*)a.out)[o];
    if (had == had) continue;
    float sum = 0.f;
    for (int ky = 0; ky < a.KH; ++ky) {
      const int gy = y + a.PH - ky * a.DH;
      if (gy < 0 || gy >= a.OH) continue;
      for (int kx = 0; kx < a.KW; ++kx) {
        const int gx = x + a.PW - kx * a.DW;
        if (gx < 0 || gx >= a.OW) continue;
        const int64_t g = ((img * a.OH + gy) * a.OW + gx) * a.CO, f = (((int64_t)ky * a.KW + kx) * a.CI + ci) * a.CO;
        float part = 0.f;
        for (int c = 0; c < a.CO; ++c) {
          if constexpr (BF)
            part += bf16_bits_to_f32(((const uint16_t*)a.g)[g + c]) * bf16_bits_to_f32(((const uint16_t*)a.f)[f + c]);
          else
            part += ((const float*)a.g)[g + c] * ((const float*)a.f)[f + c];
        }
        sum += part;
      }
    }
    if constexpr (BF)
      ((uint16_t*)a.out)[o] = f32_to_bf16_bits(sum);
    else
      ((float*)a.out)[o] = sum;
  }
}

}  // namespace

hipError_t conv_border_launch(const ConvBorderArgs& a, bool bf, hipStream_t s) {
  const int64_t pixels = (int64_t)(a.y0 + a.H - a.y1) * a.W + (int64_t)(a.y1 - a.y0) * (a.x0 + a.W - a.x1);
  const int64_t total = (int64_t)a.N * pixels * a.CI;
  if (total == 0) return hipSuccess;
  const unsigned blocks = (unsigned)std::min<int64_t>((total + 255) / 256, 256 * 32);
  if (bf)
    hipLaunchKernelGGL(conv_border_kernel<true>, dim3(blocks), dim3(256), 0, s, a);
  else
    hipLaunchKernelGGL(conv_border_kernel<false>, dim3(blocks), dim3(256), 0, s, a);
  return hipGetLastError();
}

hipError_t col2im_launch(const Col2imArgs& args, bool bf, hipStream_t s) {
  Col2imArgs a = args;
  a.period_h = a.SH / std::gcd(a.SH, a.DH);
  a.period_w = a.SW / std::gcd(a.SW, a.DW);
  a.step_h = a.period_h * a.DH / a.SH;
  a.step_w = a.period_w * a.DW / a.SW;
  const int v = a.CI >= 4 ? 4 : 1;
  const int64_t blocks = ((int64_t)a.N * a.H * a.W * ((a.CI + v - 1) / v) + 255) / 256;
  if (blocks <= 0 || blocks > kMaxLaunchThreads / 256) return hipErrorInvalidValue;
  fast_div_magic((unsigned)a.W, &a.w_magic, &a.w_shift);
  fast_div_magic((unsigned)a.SH, &a.sh_magic, &a.sh_shift);
  fast_div_magic((unsigned)a.SW, &a.sw_magic, &a.sw_shift);
  const dim3 grid((unsigned)blocks), block(256);
  const bool one = a.KH * a.KW == 1;
#define PML_GO(BF, V)                                                                          \
  if (one) hipLaunchKernelGGL((col2im_kernel<BF, V, true>), grid, block, 0, s, a);            \
  else hipLaunchKernelGGL((col2im_kernel<BF, V, false>), grid, block, 0, s, a)
  if (bf && v == 4) {
    PML_GO(true, 4);
  } else if (bf) {
    PML_GO(true, 1);
  } else if (v == 4) {
    PML_GO(false, 4);
  } else {
    PML_GO(false, 1);
  }
#undef PML_GO
  return hipGetLastError();
}

hipError_t gradient_operands_launch(int es, const void* in, void* out, int64_t pad_rows, int64_t cols, int64_t pitch, const void* f, void* bt, int64_t taps,
                                    int64_t ci, int64_t co, hipStream_t s) {
  const int64_t flip = bt ? (taps * ci * co + 255) / 256 : 0;
  const int64_t pad = std::min<int64_t>((pad_rows * (pitch * es / 16) + 255) / 256, 256 * 32);
  if (flip + pad <= 0) return hipSuccess;
  if (flip + pad > kMaxLaunchThreads / 256) return hipErrorInvalidValue;
  const dim3 grid((unsigned)(flip + pad)), block(256);
  if (es == 2)
    hipLaunchKernelGGL(gradient_operands_kernel<uint16_t>, grid, block, 0, s, (const uint16_t*)in, (uint16_t*)out, pad_rows, (int)cols, (int)pitch, (const uint16_t*)f,
                       (uint16_t*)bt, (int)taps, (int)ci, (int)co, flip);
  else
    hipLaunchKernelGGL(gradient_operands_kernel<uint32_t>, grid, block, 0, s, (const uint32_t*)in, (uint32_t*)out, pad_rows, (int)cols, (int)pitch, (const uint32_t*)f,
                       (uint32_t*)bt, (int)taps, (int)ci, (int)co, flip);
  return hipGetLastError();
}

}  // namespace pml
