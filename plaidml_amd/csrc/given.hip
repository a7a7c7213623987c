// Large products of bf16 or int8 over a right-hand side B[K][N] as it lies: 256 x 256 tiles, A through LDS, B through
// registers.
//
// A 256 x 256 tile that stages both operands in LDS (igemm.hip) uses LDS up: eight wavefronts of 128 x 64 read
// 192 bytes of fragments per byte of K where the ring's refill writes another 64, together the 128 bytes per clock and
// CU that LDS moves -- and a [K][N] right-hand side has to be transposed by a launch of its own before that.  Here only
// A goes through LDS (160 bytes instead of 256 per byte of K, and room for a ring of four slabs instead of two).  B goes
// from memory into the registers of the wavefronts that multiply it, one slab of 128 bytes of K ahead: a lane fetches four
// neighbouring columns of every K-row of its chunk, 128 contiguous bytes (bf16) of four K-rows per request, and turns
// them with v_perm into the fragments of four column blocks, block j holding the columns 4 r + j -- which is why the
// MFMAs are the 16 x 16 ones, whose operand has four K-chunks per row: the K-values of a lane's chunk are then whole rows
// of B and the ones its A fragment holds.  (32 x 32 MFMAs leave two columns per lane, twice the requests of half the
// width: bf16 4096^3 115 us.)  There is no transposed copy, no wait for memory at the one barrier of a slab, and the
// requests are spread evenly between the MFMAs.
// Measured on N(0,1) / uniform int8 data, B arriving with the call, ranges over boxes:
//   bf16 4096^3  133 us (transposed copy 13, igemm 120) -> 104-114 with bias and relu (1.21-1.32 PFLOP/s).  It spends as many
//                cycles as the tile over Bt, the matrix pipe busy for 68 % of them, at a higher clock (1.71 GHz for 1.63 on
//                one box, 107.6 us for 113.6): less passes through LDS.  Parts of it compiled out: MFMAs alone 85 (with
//                launch and tail), with A's fragment reads 91, with A's requests 97.
//   int8 4096^3  73 us (9 + 64) -> 62-68 requantised (2.0-2.2 POP/s), 72 as int32 sums, where the tile over Bt takes 69: matrix
//                pipe busy 40 %, the other vector instructions (64 permutations for B per slab and wavefront; a byte matrix
//                is turned four rows at a time) another 22, and 256 tiles on 256 CUs that write their 67 MB at once 17.
#include <hip/hip_runtime.h>

#include "device_common.h"
#include "igemm_tail.h"
#include "plans.h"

namespace pml {
namespace {

constexpr int kWaves = 8, kThreads = 64 * kWaves;
constexpr int kTile = 256;                       // rows and columns of a workgroup's tile
constexpr int kSlab = 128;                       // bytes of K per slab and row
constexpr int kStage = kTile * kSlab;            // LDS bytes of one slab of A
constexpr int kStages = 4;
constexpr unsigned kRsrcFlags = 0x00020000u;     // raw buffer, 32-bit data format
constexpr unsigned kBufRange = 0x80000000u;      // every real offset is below 2 GiB (checked at launch) ...
constexpr unsigned kOutside = 0x80000000u;       // ... and this one reads as zeros, with any row's offset added (given_span)

#define PML_LDS(p) ((__attribute__((address_space(3))) void*)(p))

typedef unsigned int u32x2_t __attribute__((ext_vector_type(2)));

template <int KIND>
struct Given;
template <>
struct Given<KIND_BF16> {
  static constexpr int ES = 2, kRows = 8;  // K-rows of a lane's 16-byte chunk
  typedef u32x2_t raw_t;                   // four columns of a K-row
  typedef f32x4_t acc_t;
  static __device__ __forceinline__ raw_t load(__amdgpu_buffer_rsrc_t r, unsigned off, int row_off) {
    return __builtin_bit_cast(raw_t, __builtin_amdgcn_raw_buffer_load_b64(r, (int)off, row_off, 0));
  }
  static constexpr int kTurnRows = 2;  // rows that make one register of each fragment
  static __device__ __forceinline__ void turn(const raw_t (&raw)[kRows], int q, i32x4_t (&f)[4]) {
    const raw_t a = raw[2 * q], b = raw[2 * q + 1];
    unsigned w[4] = {__builtin_amdgcn_perm(b[0], a[0], 0x05040100u), __builtin_amdgcn_perm(b[0], a[0], 0x07060302u),
                     __builtin_amdgcn_perm(b[1], a[1], 0x05040100u), __builtin_amdgcn_perm(b[1], a[1], 0x07060302u)};
    // (opaque: the raw registers are free for the next request from here on.  Left to itself the compiler moves the
    // permutations behind that request, into other registers, and waits for the request at the end of the loop to copy it.)
    asm volatile("" : "+v"(w[0]), "+v"(w[1]), "+v"(w[2]), "+v"(w[3]));
#pragma unroll
    for (int j = 0; j < 4; ++j) f[j][q] = (int)w[j];
  }
  static __device__ __forceinline__ void mma(acc_t& c, const i32x4_t& b, const i32x4_t& a) {
    c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, b), __builtin_bit_cast(bf16x8_t, a), c, 0, 0, 0);
  }
};
template <>
struct Given<KIND_I8> {
  static constexpr int ES = 1, kRows = 16;
  typedef unsigned raw_t;
  typedef i32x4_t acc_t;
  static __device__ __forceinline__ raw_t load(__amdgpu_buffer_rsrc_t r, unsigned off, int row_off) {
    return (raw_t)__builtin_amdgcn_raw_buffer_load_b32(r, (int)off, row_off, 0);
  }
  static constexpr int kTurnRows = 4;
  static __device__ __forceinline__ void turn(const raw_t (&raw)[kRows], int q, i32x4_t (&f)[4]) {
    const unsigned r0 = raw[4 * q], r1 = raw[4 * q + 1], r2 = raw[4 * q + 2], r3 = raw[4 * q + 3];
    const unsigned t0 = __builtin_amdgcn_perm(r1, r0, 0x05010400u), t1 = __builtin_amdgcn_perm(r1, r0, 0x07030602u);
    const unsigned t2 = __builtin_amdgcn_perm(r3, r2, 0x05010400u), t3 = __builtin_amdgcn_perm(r3, r2, 0x07030602u);
    unsigned w[4] = {__builtin_amdgcn_perm(t2, t0, 0x05040100u), __builtin_amdgcn_perm(t2, t0, 0x07060302u),
                     __builtin_amdgcn_perm(t3, t1, 0x05040100u), __builtin_amdgcn_perm(t3, t1, 0x07060302u)};
    asm volatile("" : "+v"(w[0]), "+v"(w[1]), "+v"(w[2]), "+v"(w[3]));
#pragma unroll
    for (int j = 0; j < 4; ++j) f[j][q] = (int)w[j];
  }
  static __device__ __forceinline__ void mma(acc_t& c, const i32x4_t& b, const i32x4_t& a) {
    c = __builtin_amdgcn_mfma_i32_16x16x64_i8(b, a, c, 0, 0, 0);
  }
};

// The bf16 tails direct_tail_ok allows, straight from the accumulators (the steps and roundings of direct_tail_bf16).
// A lane holds, for row r = lane % 16 of a row block, the sixteen columns from 16 (lane / 16) of the wavefront's 64.  Memory
// is touched 64 bytes of a row at a time: two lane exchanges take the lane's two 8-column pieces to the arrangement in
// which access t covers the columns 32 t + 8 (lane / 16) of sixteen rows, and back (each exchange is its own inverse).
__device__ __forceinline__ void to_memory(i32x4_t& a, i32x4_t& b) {
#pragma unroll
  for (int d = 0; d < 4; ++d) {
    const auto x = __builtin_amdgcn_permlane16_swap((unsigned)a[d], (unsigned)b[d], false, false);
    const auto y = __builtin_amdgcn_permlane32_swap(x[0], x[1], false, false);
    a[d] = (int)y[0];
    b[d] = (int)y[1];
  }
}
__device__ __forceinline__ void from_memory(i32x4_t& a, i32x4_t& b) {
#pragma unroll
  for (int d = 0; d < 4; ++d) {
    const auto x = __builtin_amdgcn_permlane32_swap((unsigned)a[d], (unsigned)b[d], false, false);
    const auto y = __builtin_amdgcn_permlane16_swap(x[0], x[1], false, false);
    a[d] = (int)y[0];
    b[d] = (int)y[1];
  }
}

template <int MI>
__device__ __forceinline__ void given_tail_bf16(const IgemmArgs& p, const f32x4_t (&acc)[MI][4], int64_t mw, int64_t nw, int lane) {
  const int r = lane & 15, g = lane >> 4;
  const bool residual = p.tail_mode == 2, scale_shift = p.tail_mode == 3;
  const int64_t rs = p.tail.operand_row_stride[0];
  const uint16_t* const scale = scale_shift ? (const uint16_t*)p.operands[p.tail.ops[0].operand] : nullptr;
  const uint16_t* const shift = scale_shift ? (const uint16_t*)p.operands[p.tail.ops[1].operand] : nullptr;
  const bool relu = scale_shift ? p.tail_ssr == 2 : p.tail_relu != 0;
  const float lo = relu ? 0.f : -__builtin_inff();  // relu as a lower clamp (the IEEE maximum keeps a NaN)
  float bias[2][8], mul[2][8], add[2][8];
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    const int64_t n = nw + 16 * g + 8 * t;
    auto column_vector = [&](const uint16_t* src, float* out) {
      const i32x4_t bits = (src != nullptr && n < p.N) ? *(const i32x4_t*)(src + n) : i32x4_t{0, 0, 0, 0};
      unpack_bf16x8(bits, out);
    };
    column_vector((const uint16_t*)p.init, bias[t]);
    if (scale_shift) {
      column_vector(scale, mul[t]);
      column_vector(shift, add[t]);
    }
  }
#pragma unroll
  for (int i = 0; i < MI; ++i) {
    const int64_t m = mw + 16 * i + r;
    const bool row_ok = m < p.M;
    i32x4_t res[2] = {i32x4_t{0, 0, 0, 0}, i32x4_t{0, 0, 0, 0}};
    if (residual) {
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        const int64_t n = nw + 32 * t + 8 * g;
        if (row_ok && n < p.N) res[t] = *(const i32x4_t*)((const uint16_t*)p.operands[0] + m * rs + n);
      }
      from_memory(res[0], res[1]);
    }
    i32x4_t packed[2];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      float v[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = acc[i][e & 3][2 * t + (e >> 2)] + bias[t][e];
      if (residual) {
        // the contraction result is rounded first, then the bf16 addition rounds again
        float x[8];
        unpack_bf16x8(res[t], x);
#pragma unroll
        for (int e = 0; e < 8; e += 2) round_pair_to_bf16(v[e], v[e + 1]);
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] += x[e];
      }
      if (scale_shift) {
        // three roundings: the contraction result, the product, the sum
#pragma unroll
        for (int e = 0; e < 8; e += 2) round_pair_to_bf16(v[e], v[e + 1]);
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] *= mul[t][e];
#pragma unroll
        for (int e = 0; e < 8; e += 2) round_pair_to_bf16(v[e], v[e + 1]);
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] += add[t][e];
      }
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = __builtin_elementwise_maximum(v[e], lo);
      packed[t] = pack_bf16x8(v);
    }
    to_memory(packed[0], packed[1]);
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      const int64_t n = nw + 32 * t + 8 * g;
      if (row_ok && n < p.N) *(i32x4_t*)((uint16_t*)p.C + m * p.ldc + n) = packed[t];
    }
  }
}

// int8's requantisation chain (the straight code of tile_tail, tail_mode 4 with tail_rq, and its arithmetic) straight from the
// accumulators: a lane's sixteen neighbouring columns are one 16-byte store, where the trip through LDS makes 4-byte ones
// (4096^3: 66.2 us with it).  Not where the sums are stored as well: their rows leave in 16-byte pieces 64 bytes apart here
// (81.7 us), and whole behind the trip through LDS.
__device__ __forceinline__ bool requant_direct_ok(const IgemmArgs& p) {
  if (p.tail_mode != 4 || !p.tail_rq || p.rq_store >= 0 || (p.N & 15) != 0 || (p.ldc & 15) != 0 || ((uintptr_t)p.C & 15) != 0) return false;
  return p.init == nullptr || (p.init_rs == 0 && p.init_cs == 1 && p.init_dtype == PML_HIP_I32 && ((uintptr_t)p.init & 15) == 0);
}

template <int MI>
__device__ __forceinline__ void given_tail_requant(const IgemmArgs& p, const i32x4_t (&acc)[MI][4], int64_t mw, int64_t nw, int lane) {
  const int r = lane & 15, g = lane >> 4;
  const int64_t n = nw + 16 * g;
  if (n >= p.N) return;
  const float* const scale = (const float*)p.operands[p.rq_scale];
  const bool one_scale = p.tail.operand_col_stride[p.rq_scale] == 0;
  const float lo = p.rq_lo, hi = p.rq_hi;
  f32x4_t sc[4];
  i32x4_t start[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    sc[e] = one_scale ? f32x4_t{scale[0], scale[0], scale[0], scale[0]} : *(const f32x4_t*)(scale + n + 4 * e);
    start[e] = p.init != nullptr ? *(const i32x4_t*)((const int*)p.init + n + 4 * e) : i32x4_t{0, 0, 0, 0};
  }
#pragma unroll
  for (int i = 0; i < MI; ++i) {
    const int64_t m = mw + 16 * i + r;
    if (m >= p.M) continue;
    i32x4_t bytes;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      i32x4_t a;
#pragma unroll
      for (int q = 0; q < 4; ++q) a[q] = (int)((unsigned)acc[i][q][e] + (unsigned)start[e][q]);
      uint32_t w = 0;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        float v = (float)a[q] * sc[e][q];
        v = __builtin_fmaxf(v, lo);
        v = __builtin_fminf(v, hi);
        const int t = (int)(v + __builtin_copysignf(0.5f, v));
        w |= (uint32_t)(t & 255) << (8 * q);
      }
      bytes[e] = (int)w;
    }
    *(i32x4_t*)((int8_t*)p.C + m * p.ldc + n) = bytes;
  }
}

template <int KIND>
__global__ __launch_bounds__(kThreads, 2) void given_kernel(IgemmArgs p_by_value) {
  warm_arguments<sizeof(IgemmArgs)>();
  // (read where the dispatcher put it: indexing a by-value copy would move the copy to scratch memory)
  const IgemmArgs& p = *(const IgemmArgs*)(const __attribute__((address_space(4))) void*)__builtin_amdgcn_kernarg_segment_ptr();
  typedef Given<KIND> G;
  typedef typename G::raw_t raw_t;
  typedef typename G::acc_t acc_t;
  constexpr int ES = G::ES, kRows = G::kRows;
  constexpr int MI = 8, NI = 4;               // 16 x 16 blocks of a wavefront: 128 x 64 results
  constexpr int kParts = kStage / (kThreads * 16);  // requests of a thread per slab of A
  constexpr int kPerBlock = kRows + kParts / 2;     // requests of a thread per 64 bytes of K: B's rows and half of A's
  static_assert(64 / ES + kRows == 80 / ES, "the rows a request's offset reaches are the ones given_span counts");
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave >> 2, wn = wave & 3, r = lane & 15, g = lane >> 4;
  int tile_m, tile_n;
  tile_of(p.order, blockIdx.x, &tile_m, &tile_n);
  const int64_t m0 = (int64_t)tile_m * kTile, n0 = (int64_t)tile_n * kTile;

  const __amdgpu_buffer_rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc((void*)p.A, 0, (int)kBufRange, kRsrcFlags);
  const __amdgpu_buffer_rsrc_t rb = __builtin_amdgcn_make_buffer_rsrc((void*)p.Bt, 0, (int)kBufRange, kRsrcFlags);
  const int kbytes = (int)(p.K * ES);
  const int slabs = (kbytes + kSlab - 1) / kSlab;

  // A: slot tid % 8 of rows tid / 8 + 64 i takes the chunk of the row that the swizzle puts there (igemm.hip)
  const int lr = tid >> 3, a_chunk = ((tid & 7) ^ ((lr >> 1) & 7)) * 16;
  unsigned a_off[kParts];
#pragma unroll
  for (int i = 0; i < kParts; ++i) {
    const int64_t m = m0 + lr + 64 * i;
    a_off[i] = m < p.M ? (unsigned)(m * p.lda * ES + a_chunk) : kOutside;
  }
  // (past the last slab, and in the chunks of it that lie past the row's end: outside)
  auto request_a = [&](int slab, int part) {
    unsigned char* const to = smem + (slab & (kStages - 1)) * kStage + part * (kThreads * 16) + wave * 1024;
    const int at = slab * kSlab;
    const unsigned off = (a_chunk + at < kbytes) & (a_off[part] != kOutside) ? a_off[part] + (unsigned)at : kOutside;
    __builtin_amdgcn_raw_ptr_buffer_load_lds(ra, PML_LDS(to), 16, (int)off, 0, 0, 0);
  };

  // B: the lane's columns n .. n + 3 of the K-rows kRows g .. of a block of 64 bytes of K; a slab holds two blocks.  K is
  // whole 16-byte vectors: the rows of a lane's chunk exist together or not at all.
  const unsigned pitch = (unsigned)__builtin_amdgcn_readfirstlane((int)(p.ldbt * ES));
  const int64_t n = n0 + wn * 64 + 4 * r;
  const bool n_ok = n < p.N;  // (N is a multiple of four)
  const unsigned b_first = (unsigned)(kRows * g) * pitch + (unsigned)(n * ES);
  auto b_offset = [&](int slab, int block) {
    const int k = slab * (kSlab / ES) + block * (64 / ES) + kRows * g;  // the chunk's first K-row
    return n_ok & (k < (int)p.K) ? b_first + (unsigned)(slab * (kSlab / ES)) * pitch : kOutside;
  };
  auto request_b = [&](unsigned off, int block, int e) { return G::load(rb, off, (int)((unsigned)(block * (64 / ES) + e) * pitch)); };

  raw_t raw[2][kRows];
  acc_t acc[MI][NI];
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < NI; ++j) acc[i][j] = acc_t{0, 0, 0, 0};

  // Requests return in the order they were made.  Ahead of the loop: slab 0 of A, slab 0 of B, A up to slab kStages - 2, and
  // then what the second block of a pass through the loop requests, in its order (the compiler's waits in the loop are as
  // strict as the stricter of the two ways into it).
#pragma unroll
  for (int i = 0; i < kParts; ++i) request_a(0, i);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int b = 0; b < 2; ++b) {
    const unsigned off = b_offset(0, b);
#pragma unroll
    for (int e = 0; e < kRows; ++e) raw[b][e] = request_b(off, b, e);
  }
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int s = 1; s < kStages - 1; ++s)
#pragma unroll
    for (int i = 0; i < kParts; ++i) request_a(s, i);
  __builtin_amdgcn_sched_barrier(0);

  int fslot[2];  // the lane's chunk of each block of its fragment rows
#pragma unroll
  for (int b = 0; b < 2; ++b) fslot[b] = ((b * 4 + g) ^ ((r >> 1) & 7)) * 16;
  const unsigned char* const a_base = smem + (wm * 128 + r) * kSlab;
  i32x4_t fa[MI], fb[2][NI];
  // slab 0 of A has landed: everything younger may be outstanding
  constexpr int kAhead = 2 * kRows + (kStages - 2) * kParts;
  static_assert(kAhead <= 63, "the vmcnt field counts at most 63 requests");
  __builtin_amdgcn_s_waitcnt(0x0F70 | (kAhead & 15) | ((kAhead >> 4) << 14));
  __builtin_amdgcn_s_barrier();
#pragma unroll
  for (int i = 0; i < MI; ++i) fa[i] = *(const i32x4_t*)(a_base + i * 16 * kSlab + fslot[0]);
#pragma unroll
  for (int q = 0; q < 4; ++q) G::turn(raw[0], q, fb[0]);
  unsigned b_next = b_offset(1, 0);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int i = 0; i < MI; ++i) {
#pragma unroll
    for (int e = i * (kRows / MI); e < (i + 1) * (kRows / MI); ++e) raw[0][e] = request_b(b_next, 0, e);
    if (i % 4 == 3) request_a(kStages - 1, i / 4);
    __builtin_amdgcn_sched_barrier(0);
  }

  // A block of the loop multiplies 64 bytes of K with fragments that are in registers, turns the next block's rows of B,
  // requests those rows of the next slab in their place, and replaces A's fragments one by one as they have been used.
  // The barrier of a slab sits between its two blocks: by then everything of its stage has been read (lgkmcnt 0), so the
  // stage may be filled again, and the next slab's A has landed -- it was requested before the rows of B that the block
  // before turned: of the requests in flight only those of the last two blocks are younger than these.
#pragma clang loop unroll(disable)
  for (int s = 0; s < slabs; ++s) {
    const unsigned char* const a_cur = a_base + (s & (kStages - 1)) * kStage;
    const unsigned char* const a_nxt = a_base + ((s + 1) & (kStages - 1)) * kStage;
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      const int nb = b ^ 1;
      if (b == 1) {
        __builtin_amdgcn_s_waitcnt(0x0070 | ((2 * kPerBlock) & 15) | (((2 * kPerBlock) >> 4) << 14));
        __builtin_amdgcn_s_barrier();
      }
      b_next = b_offset(b == 1 ? s + 2 : s + 1, nb);
      const unsigned char* const a_from = (b == 1 ? a_nxt : a_cur) + fslot[nb];
#pragma unroll
      for (int i = 0; i < MI; ++i) {
#pragma unroll
        for (int j = 0; j < NI; ++j) G::mma(acc[i][j], fb[b][j], fa[i]);
        __builtin_amdgcn_sched_barrier(0);
        fa[i] = *(const i32x4_t*)(a_from + i * 16 * kSlab);
        if ((i & 1) == 0) {
          G::turn(raw[nb], i / 2, fb[nb]);
          __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int e = i * (kRows / MI); e < (i + 1) * (kRows / MI); ++e) raw[nb][e] = request_b(b_next, nb, e);
        if (i % 4 == 3) {
          const int part = i / 4;  // block 1: the first half of slab s + kStages, block 0: the second half of the one before
          if (b == 1)
            request_a(s + kStages, part);
          else
            request_a(s + kStages - 1, kParts / 2 + part);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  }
  // drain the (all-outside) requests still in flight before LDS is reused
  __builtin_amdgcn_s_waitcnt(0x0F70);
  const int64_t mw = m0 + wm * 128, nw = n0 + wn * 64;
  // (the lane number through an opaque move: the tail's addresses are then worked out here instead of being carried
  // through the loop)
  int lane_now = lane;
  asm volatile("" : "+v"(lane_now));
  if constexpr (KIND == KIND_BF16) {
    if (direct_tail_ok<KIND>(p, n0, kTile)) {
      given_tail_bf16<MI>(p, acc, mw, nw, lane_now);
      return;
    }
  } else {
    if (requant_direct_ok(p)) {
      given_tail_requant<MI>(p, acc, mw, nw, lane_now);
      return;
    }
  }
  __syncthreads();
  // the common tail, 32 rows of the wavefront at a time through a part of LDS that is its own
  typedef typename Acc<KIND>::scalar accs_t;
  constexpr int CS = 64 + 4;
  static_assert(32 * CS * 4 <= kStages * kStage / kWaves, "two row blocks of a wavefront must fit its share of LDS");
  accs_t* const wtile = (accs_t*)(smem + wave * (kStages * kStage / kWaves));
  const int row = lane_now & 15, col = 16 * (lane_now >> 4);
  static_for<0, MI, 2>([&](auto i0c) {
    constexpr int i0 = decltype(i0c)::value;
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e)
        *(acc_t*)&wtile[(16 * i + row) * CS + col + 4 * e] = acc_t{acc[i0 + i][0][e], acc[i0 + i][1][e], acc[i0 + i][2][e], acc[i0 + i][3][e]};
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    tile_tail<KIND, 32, 64, 64>(p, wtile, mw + 16 * i0, nw, lane_now);
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  });
}

template <int KIND>
hipError_t launch(const IgemmArgs& a, hipStream_t s) {
  const int64_t tiles_m = (a.M + kTile - 1) / kTile, tiles_n = (a.N + kTile - 1) / kTile, tiles = tiles_m * tiles_n;
  if (tiles <= 0 || tiles >= ((int64_t)1 << 31)) return hipErrorInvalidValue;
  constexpr size_t lds = (size_t)kStages * kStage;
  auto kern = given_kernel<KIND>;
  static DynamicLdsLimit limit;
  if (hipError_t e = limit.ensure((const void*)kern, lds); e != hipSuccess) return e;
  IgemmArgs b = a;
  b.order = make_tile_order((int)tiles_m, (int)tiles_n);
  hipLaunchKernelGGL(kern, dim3((unsigned)tiles), dim3(kThreads), lds, s, b);
  return hipGetLastError();
}

}  // namespace

hipError_t given_launch(int kind, const IgemmArgs& a, hipStream_t s) {
  // (rows of A are whole 16-byte vectors; a lane's four columns exist together and lie on a 4-element boundary)
  const int es = kind == KIND_BF16 ? 2 : 1;
  if (!a.b_kn || a.K2 > 0 || a.N % 4 != 0 || a.ldbt % 4 != 0 || a.K * es % 16 != 0 || ((uintptr_t)a.Bt & (4 * es - 1)) != 0) return hipErrorInvalidValue;
  if (a.M * a.lda * es >= ((int64_t)1 << 31) || given_span(a.K, a.ldbt, es) >= ((int64_t)1 << 31)) return hipErrorInvalidValue;
  switch (kind) {
    case KIND_BF16: return launch<KIND_BF16>(a, s);
    case KIND_I8: return launch<KIND_I8>(a, s);
  }
  return hipErrorInvalidValue;
}

}  // namespace pml
