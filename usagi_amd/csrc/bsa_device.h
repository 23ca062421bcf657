// Device-side definitions shared by the forward kernels of libusagi_bsa.so (bsa_fwd.hip,
// bsa_ksplit.hip): the kernel arguments, the work-item order, the cross-lane and packing helpers,
// the Q·K^T MFMA and the HBM -> LDS DMA.
#ifndef USAGI_BSA_DEVICE_H
#define USAGI_BSA_DEVICE_H

#include <hip/hip_runtime.h>

#include <math.h>
#include <stdint.h>

#include <type_traits>

#include "usagi_bsa.h"

namespace usagi_bsa {

constexpr int kBlk = USAGI_BSA_BLOCK;    // rows per query / key block
constexpr int kHd = USAGI_BSA_HEAD_DIM;  // head dimension
constexpr int kThreads = 256;            // 4 wave64s
constexpr float kLn2 = 0.6931471805599453f;
constexpr float kSpecSum = 4096.0f;      // acceptance bound of a speculative P row sum

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half4 __attribute__((ext_vector_type(4)));
typedef _Float16 half2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

struct Args {
  const uint16_t* q;
  const uint16_t* k;
  const uint16_t* v;
  uint16_t* o;
  float* lse;
  const int32_t* row_ptr;
  const int32_t* col_idx;
  const int32_t* seq_lens;
  int heads;
  int T;
  int nqb;
  int bh_count;
  int max_nnz;
  float qk_scale;  // log2(e) / sqrt(128)
  int head_major;  // work-item order without a plan, see item_coords
  int window;      // analytic rows (kRowsWindow): window length in blocks
  int n_global;    // analytic rows: global prefix blocks
  const int32_t* sched;  // planned order (usagi_bsa_plan): slot -> item, or NULL
  int n_slots;           // slots of the planned order, or n_items
  int n_items;           // B * H * nqb
};

// Work item (workgroup index) -> (query block, b*h) when no plan is given.
// head_major == 0: query blocks in descending order (for causal window patterns the longest
//   rows first), b*h fastest.
// head_major == 1 (B*H a multiple of 8): workgroups are dealt to the 8 XCDs round-robin by
//   index, so item i runs on XCD i % 8; each XCD walks its heads x, x+8, ... one at a time, and
//   within a head takes the query blocks in descending order. The key/value tiles of the head being
//   walked (4 MiB at T = 8192) then stay in that XCD's L2 while all its query blocks read them.
__device__ __forceinline__ void item_coords(const Args& a, int item, int& qb, int& bh) {
  if (a.head_major) {
    const int x = item & 7;
    const int j = item >> 3;
    const int hl = j / a.nqb;
    qb = a.nqb - 1 - (j - hl * a.nqb);
    bh = x + 8 * hl;
  } else {
    const int qslot = item / a.bh_count;
    qb = a.nqb - 1 - qslot;
    bh = item - qslot * a.bh_count;
  }
}

__device__ __forceinline__ float wave_pair_max(float x) {
  // {x[l], x[l ^ 32]} in some order; max is symmetric.
  auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}

__device__ __forceinline__ float wave_pair_sum(float x) {
  auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// Max / sum over lanes l, l^16, l^32, l^48 (the four lane groups that hold one query row in the
// 16x16 MFMA layouts): {x[l], x[l ^ 16]} then {y[l], y[l ^ 32]}, each in some order.
__device__ __forceinline__ float wave_quad_max(float x) {
  auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  const float y = fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
  return wave_pair_max(y);
}

__device__ __forceinline__ float wave_quad_sum(float x) {
  auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  const float y = __uint_as_float(r[0]) + __uint_as_float(r[1]);
  return wave_pair_sum(y);
}

typedef float floatx2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));

// Two bf16 (one dword) -> two fp16 (one dword), round to nearest even: each bf16 widens exactly
// to fp32 (its bits in the upper half), then one v_cvt_pk_f16_f32 packs the pair.
__device__ __forceinline__ uint32_t bf16x2_to_f16x2(uint32_t w) {
  const float lo = __uint_as_float(w << 16);
  const float hi = __uint_as_float(w & 0xffff0000u);
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(floatx2{lo, hi}, half2));
}
// Two fp32 -> one dword of two fp16 / bf16 (v_cvt_pk_*_f32, round to nearest even). O is
// rounded twice, to fp32 by the multiply with 1/l and then to the output type, as the reference's
// fp32 division and cast do.
template <bool kBf16>
__device__ __forceinline__ uint32_t pack_out(float x, float y) {
  if constexpr (kBf16) {
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(floatx2{x, y}, bf16x2));
  } else {
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(floatx2{x, y}, half2));
  }
}

template <bool kBf16>
__device__ __forceinline__ floatx4 mfma_qk16(u32x4 a, u32x4 b, floatx4 c) {
  if constexpr (kBf16) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a),
                                                   __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
  } else {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8, a),
                                                  __builtin_bit_cast(half8, b), c, 0, 0, 0);
  }
}

typedef short v4i16 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) v4i16 lds_v4i16;
typedef __attribute__((address_space(3))) void lds_void;

// One 16-byte-per-lane DMA: global (uniform base + per-lane byte offset) -> LDS at the uniform
// byte address lds_addr + 16 * lane. Issued as inline asm so that the compiler's wait-count pass
// does not treat it as aliasing every later LDS read; the kernel waits for it explicitly
// (s_waitcnt vmcnt + s_barrier) before any wave reads the tile.
template <int kImm>
__device__ __forceinline__ void dma_16b(const void* gbase, uint32_t voff, uint32_t lds_addr) {
  // M0 holds the LDS destination. It is listed as clobbered, but the compiler does not preserve
  // a reserved register across an asm statement; this is safe because nothing else in the
  // kernel uses M0 (tests/test_device_code.py checks the assembly for that).
  asm volatile(
      "s_mov_b32 m0, %0\n\t"
      "s_nop 0\n\t"
      "global_load_lds_dwordx4 %1, %2 offset:%3"
      :
      : "s"(lds_addr), "v"(voff), "s"(gbase), "i"(kImm)
      : "memory", "m0");
}

// 8 DMAs of one wave's 8 KiB share of a tile: instruction i moves row group i (1 KiB). The
// instruction's immediate offset moves both the global and the LDS address, so 1024 (i % 4) goes
// there and i >= 4 use global and LDS bases 4096 bytes further on.
__device__ __forceinline__ void dma_tile8(const char* src, const uint32_t off[4], uint32_t lds) {
  const char* src_hi = src + 4096;
  const uint32_t lds_hi = lds + 4096;
  dma_16b<0>(src, off[0], lds);
  dma_16b<1024>(src, off[1], lds);
  dma_16b<2048>(src, off[2], lds);
  dma_16b<3072>(src, off[3], lds);
  dma_16b<0>(src_hi, off[0], lds_hi);
  dma_16b<1024>(src_hi, off[1], lds_hi);
  dma_16b<2048>(src_hi, off[2], lds_hi);
  dma_16b<3072>(src_hi, off[3], lds_hi);
}

__device__ __forceinline__ uint32_t lds_addr_of(const void* p) {
  return (uint32_t)(uintptr_t)(lds_void*)p;
}

// Zeroes rows `from` and above of a wave's kSliceRows rows of V in LDS (256 bytes a row; from <= 0: all
// of them). V past seq_len may hold anything, and P = 0 does not cancel a NaN or an infinity there. Runs
// only on the key blocks that seq_len cuts. A row at a time and 4 bytes a lane, with the address made
// here: wider stores, or an address made ahead of the branch, spill in the bf16 generic kernel.
template <int kSliceRows>
__device__ __forceinline__ void zero_v_tail(char* slice, int lane, int from) {
  asm volatile("" : "+v"(lane));
  uint32_t* row = (uint32_t*)slice + lane;
#pragma unroll 1
  for (int r = max(from, 0); r < kSliceRows; ++r) row[r * (kHd / 2)] = 0;
}

#define USAGI_BARRIER() asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory")
#define USAGI_WAIT_VM(n) asm volatile("s_waitcnt vmcnt(" #n ")" ::: "memory")

// Rows of one query block (kRows):
//   kRowsCsr     the CSR walk of kernels/v7_blockptr_warpspec.py:77-136: entries before the last
//                are attended unmasked, the last entry stands for the diagonal, which is taken
//                implicitly as kb = qb and causally masked.
//   kRowsWindow  analytic rows instead of the CSR (no row_ptr / col_idx reads): query block qb
//                attends the global prefix 0 .. n_global-1 and the window max(0, qb-window+1) ..
//                qb, deduplicated and ascending, the rows of kernels/v1_baseline.py:141-322
//                (_fwd_window, _fwd_window_global).
//   kRowsGeneric the generic CSR walk of kernels/v1_baseline.py:331-406: every entry of the row,
//                in any order; an entry equal to qb takes the causal mask, keys at or past
//                seq_len are masked, and a row without the diagonal does not attend it (an empty
//                row gives O = 0, LSE = -inf). The first entry equal to qb is walked first.
// kFullSeq: no seq_lens (every sequence has length T), so no query row or key is ever masked
// by length and the masking code is compiled out.
enum : int { kRowsCsr = 0, kRowsWindow = 1, kRowsGeneric = 2 };

}  // namespace usagi_bsa

#endif  // USAGI_BSA_DEVICE_H
