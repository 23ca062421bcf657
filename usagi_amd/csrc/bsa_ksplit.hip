// Forward kernels for launches that do not fill the GPU with one four-wave workgroup per query
// block, where the time is the chain of key blocks of the longest row and not the chip's
// throughput. Same semantics as bsa_fwd_dma_kernel (bsa_fwd.hip); what differs is that the keys of
// a block, and not only its query rows, are divided over the waves, so that a block costs a wave
// fewer MFMAs:
//
//   bsa_ksplit_kernel  32 query rows per workgroup (four workgroups per query block), four waves of
//                      32 keys each: 32 MFMAs per wave and block instead of 128. A wave reads only
//                      the rows of K and V that its own DMA brought in, so there is no barrier in
//                      the key loop.
//   bsa_wide_kernel    eight waves: 8 / kKG groups of 32 query rows x kKG groups of 128 / kKG keys.
//                      kKG = 4: 64 query rows (two workgroups per query block), 32 MFMAs per wave
//                      and block; kKG = 2: the whole query block, 64 MFMAs.
//
// Each wave keeps a running max, row sum and O (fp32) of its own keys; they are merged through LDS
// at the end of the row. One workgroup per CU (128 KiB of LDS): K and V are double-buffered and
// requested a whole block (bsa_ksplit_kernel: two) ahead, so no DMA latency is exposed.
//
// What a row of 8 blocks takes (sliding window, fp16 / bf16, kernel time in us):
//   query blocks   bsa_fwd_dma_kernel   bsa_ksplit_kernel   bsa_wide_kernel<4>   <2>
//   64             18.6 / 22.6          9.5 / 10.5          13.6 / 15.5          18.1 / 19.8
//   128            18.9 / 22.9          17.9 / 20.6         13.7 / 15.4          18.4 / 19.8
//   256            19.3 / 23.2          30.7 / 35.2         26.2 / 29.5          18.6 / 20.0
// Per block that is 0.5, 0.85 and 1.3 us against 1.75-2.3 us (one workgroup of bsa_fwd_dma_kernel on
// a CU). What is left bounds is the chain of a step: Q·K^T, softmax and P·V of bsa_wide_kernel<2> take
// 3,500 cycles for 1,024 cycles of a wave's MFMAs (2,048 of its SIMD's), its DMA wait 50 of them.
#include "bsa_device.h"

#include "bsa_internal.h"

namespace {

using namespace usagi_bsa;

constexpr int kTileBytes = kBlk * kHd * 2;

// Workgroup index -> slot of the work order and part of its query block (kSub parts). The parts of
// one query block read the same K and V: they follow each other on one XCD (index % 8).
template <int kSub>
__device__ __forceinline__ bool work_of(const Args& a, int& sub, int& qb, int& bh) {
  const int j = blockIdx.x >> 3;
  sub = j % kSub;
  const int slot = (j / kSub) * 8 + (blockIdx.x & 7);
  if (slot >= a.n_slots) return false;
  if (a.sched) {
    const int item = a.sched[slot];
    if ((unsigned)item >= (unsigned)a.n_items) return false;
    bh = item / a.nqb;
    qb = item - bh * a.nqb;
  } else {
    item_coords(a, slot, qb, bh);
  }
  bh = __builtin_amdgcn_readfirstlane(bh);
  qb = __builtin_amdgcn_readfirstlane(qb);
  return true;
}

// The key blocks of one row, in the order bsa_fwd_dma_kernel walks them: the diagonal first (when
// the row has it), then the other entries; 64 column indices at a time in one VGPR.
template <int kRows>
struct Row {
  int n_blk;      // key blocks of the row
  bool has_diag;  // step 0 is the diagonal
  int qb, nqb_m1, lane;
  const int32_t* cols;
  int n_ent, diag_pos, col_chunk, colv;
  int win_lo, win_ng;

  __device__ __forceinline__ Row(const Args& a, int qb_, int bh, int lane_) {
    qb = qb_;
    lane = lane_;
    nqb_m1 = a.nqb - 1;
    has_diag = true;
    cols = nullptr;
    n_ent = diag_pos = col_chunk = colv = win_lo = win_ng = 0;
    int n_off;
    if constexpr (kRows == kRowsWindow) {
      win_lo = max(qb - a.window + 1, 0);
      win_ng = min(a.n_global, win_lo);
      n_off = win_ng + (qb - win_lo);
    } else {
      const int32_t* rp = a.row_ptr + (size_t)bh * (a.nqb + 1) + qb;
      int rs = rp[0];
      int re = rp[1];
      rs = min(max(rs, 0), a.max_nnz);
      re = min(max(re, rs), a.max_nnz);
      cols = a.col_idx + (size_t)bh * a.max_nnz + rs;
      if constexpr (kRows == kRowsGeneric) {
        n_ent = re - rs;
        colv = lane < n_ent ? cols[lane] : -1;
        int pos = -1;
        for (int c = 0; c < n_ent && pos < 0; c += 64) {
          const int e = c + lane;
          const int x = c == 0 ? colv : (e < n_ent ? cols[e] : -1);
          const uint64_t hit = __ballot(x == qb);
          if (hit) pos = c + __builtin_ctzll(hit);
        }
        has_diag = pos >= 0;
        diag_pos = has_diag ? pos : n_ent;
        n_off = has_diag ? n_ent - 1 : n_ent;
      } else {
        n_ent = max(re - rs - 1, 0);
        n_off = n_ent;
        colv = lane < n_ent ? cols[lane] : 0;
      }
    }
    n_blk = __builtin_amdgcn_readfirstlane(n_off + (has_diag ? 1 : 0));
  }

  __device__ __forceinline__ int key_block(int i) {
    int j = i - (has_diag ? 1 : 0);
    if (j < 0) return qb;
    if constexpr (kRows == kRowsWindow) {
      return j < win_ng ? j : win_lo + (j - win_ng);
    } else {
      if constexpr (kRows == kRowsGeneric) j += (j >= diag_pos) ? 1 : 0;
      const int c = j >> 6;
      if (c != col_chunk) {
        col_chunk = c;
        const int e = c * 64 + lane;
        colv = e < n_ent ? cols[e] : 0;
      }
      const int kb = __builtin_amdgcn_readlane(colv, j & 63);
      return min(max(kb, 0), nqb_m1);
    }
  }
};

// Per-lane byte offsets of a DMA of 16 rows (instruction i: rows 4i + L/16), 16-byte chunks
// XOR-swizzled inside a row as in bsa_fwd_dma_kernel (K: chunk ^ (row % 16), V: chunk ^ 2 *
// (row % 8)).
__device__ __forceinline__ void dma_offsets(int lane, uint32_t k_off[4], uint32_t v_off[4]) {
  const int r = lane >> 4;
  const int pc = lane & 15;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    k_off[i] = (uint32_t)(r * 256 + 16 * (pc ^ (4 * i + r)));
    v_off[i] = (uint32_t)(r * 256 + 16 * (pc ^ (8 * (i & 1) + 2 * r)));
  }
}

// DMA piece i (rows 4i .. 4i+3) of a slice.
__device__ __forceinline__ void dma_piece(const char* src, const uint32_t off[4], uint32_t dst, int i) {
  const char* from = src + (i >= 4 ? 4096 : 0);
  const uint32_t to = dst + (i >= 4 ? 4096 : 0);
  switch (i & 3) {
    case 0: dma_16b<0>(from, off[0], to); break;
    case 1: dma_16b<1024>(from, off[1], to); break;
    case 2: dma_16b<2048>(from, off[2], to); break;
    default: dma_16b<3072>(from, off[3], to); break;
  }
}

// Output of query rows past seq_len: O = 0, LSE = -inf.
template <int kR, int kWgThreads>
__device__ __forceinline__ void store_empty(const Args& a, size_t base, int bh, int q0) {
  const int tid = threadIdx.x;
  uint16_t* out = a.o + base + (size_t)q0 * kHd;
#pragma unroll
  for (int i = 0; i < (kR * kHd) / (8 * kWgThreads); ++i) {
    *(u32x4*)(out + (size_t)(i * kWgThreads + tid) * 8) = u32x4{0, 0, 0, 0};
  }
  if (a.lse && tid < kR) a.lse[(size_t)bh * a.T + q0 + tid] = -INFINITY;
}

// Q^T operands of a wave's 32 rows from q0 (query tile qt: rows 16qt + c16; k-step ks: d = 32ks +
// 8g4 .. +7). Rows past seq_len may hold anything: they are taken as zero, so their scores stay
// finite.
__device__ __forceinline__ void load_q(const Args& a, size_t base, int q0, int seq_len, int c16, int g4,
                                       u32x4 (&qf)[2][4]) {
#pragma unroll
  for (int qt = 0; qt < 2; ++qt) {
    const int row = q0 + 16 * qt + c16;
    const uint16_t* qp = a.q + base + (size_t)row * kHd + 8 * g4;
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      const u32x4 x = *(const u32x4*)(qp + 32 * ks);
      qf[qt][ks] = row < seq_len ? x : u32x4{0, 0, 0, 0};
    }
  }
}

// Scores of kNT 16-key tiles x two query tiles (st[qt][t]: keys key0 + 16t + 4g4 .. +3 of row row0 +
// 16qt + c16 of the query block) masked above each row's last key.
template <int kNT>
__device__ __forceinline__ void mask_above(floatx4 (&st)[2][kNT], int qt, int lim) {
#pragma unroll
  for (int t = 0; t < kNT; ++t) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      if (16 * t + r > lim) st[qt][t][r] = -INFINITY;
    }
  }
}
template <int kNT>
__device__ __forceinline__ void mask_diag(floatx4 (&st)[2][kNT], int row0, int key0, int c16, int g4) {
#pragma unroll
  for (int qt = 0; qt < 2; ++qt) mask_above<kNT>(st, qt, row0 + 16 * qt + c16 - (key0 + 4 * g4));
}
// Generic rows off the diagonal step: an entry equal to qb (a repeated diagonal) causally, one above
// it by seq_len.
template <int kNT>
__device__ __forceinline__ void mask_generic(floatx4 (&st)[2][kNT], int kb, int qb, int seq_len, int row0,
                                             int key0, int c16, int g4) {
  if (kb < qb) return;
#pragma unroll
  for (int qt = 0; qt < 2; ++qt) {
    int last = kb == qb ? row0 + 16 * qt + c16 : kBlk - 1;
    if (kb > qb) last = min(last, seq_len - 1 - kb * kBlk);
    mask_above<kNT>(st, qt, last - (key0 + 4 * g4));
  }
}

// Softmax state of a wave's 32 rows over its keys.
struct State {
  floatx4 o[2][8];  // O^T: query tile qt, d-tile u (d = 16u + 4g4 .. +3 of row 16qt + c16)
  float m[2];
  float l[2];       // this lane's share of the row sum
  __device__ __forceinline__ State() {
#pragma unroll
    for (int qt = 0; qt < 2; ++qt) {
      m[qt] = -1e30f;
      l[qt] = 0.0f;
#pragma unroll
      for (int u = 0; u < 8; ++u) o[qt][u] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
    }
  }
};

// P = exp2(S·scale - m) in fp16 (pb[qt][ks]: 32-key step ks) and its row sum. kExact: the block's
// exact row max first (the diagonal, whose O and l are still zero). Otherwise the running max as it
// stands, accepted when the lane's sum is <= 2^12 (every P is then finite in fp16, as in
// bsa_fwd_dma_kernel), else the row max moves to the exact one and O and l are rescaled. A wave whose
// keys all lie above its rows on the diagonal keeps m = -1e30 and takes the exact max of the next
// block that way. The sum is taken from the fp32 P: an fp16 dot product would wait for the matrix
// core, which the SIMD's other wave keeps busy.
template <int kNT, bool kExact>
__device__ __forceinline__ void softmax(const floatx4 (&st)[2][kNT], State& s, float scale,
                                        half8 (&pb)[2][kNT / 2]) {
  float sum[2];
  auto make_p = [&]() {
#pragma unroll
    for (int qt = 0; qt < 2; ++qt) {
      float acc = 0.0f;
#pragma unroll
      for (int ks = 0; ks < kNT / 2; ++ks) {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const float p = __builtin_amdgcn_exp2f(fmaf(st[qt][2 * ks + (e >> 2)][e & 3], scale, -s.m[qt]));
          acc += p;
          pb[qt][ks][e] = (_Float16)p;
        }
      }
      sum[qt] = acc;
    }
  };
  auto row_max = [&](int qt) {
    float mx = st[qt][0][0];
#pragma unroll
    for (int t = 0; t < kNT; ++t) {
#pragma unroll
      for (int r = 0; r < 4; ++r) mx = fmaxf(mx, st[qt][t][r]);
    }
    return wave_quad_max(mx);
  };
  if constexpr (kExact) {
#pragma unroll
    for (int qt = 0; qt < 2; ++qt) s.m[qt] = fmaxf(s.m[qt], row_max(qt) * scale);
    make_p();
  } else {
    make_p();
    if (__builtin_expect(__any(!(sum[0] <= kSpecSum) || !(sum[1] <= kSpecSum)), 0)) {
#pragma unroll
      for (int qt = 0; qt < 2; ++qt) {
        const float m_new = fmaxf(s.m[qt], row_max(qt) * scale);
        const float alpha = __builtin_amdgcn_exp2f(s.m[qt] - m_new);
        s.m[qt] = m_new;
        s.l[qt] *= alpha;
#pragma unroll
        for (int u = 0; u < 8; ++u) s.o[qt][u] *= alpha;
      }
      make_p();
    }
  }
  s.l[0] += sum[0];
  s.l[1] += sum[1];
}

// V^T fragment (16 d x 32 keys) at LDS address vb: the two transpose reads of bsa_fwd_dma_kernel.
__device__ __forceinline__ half8 v_fragment(const char* vb) {
  const v4i16 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4i16*)vb);
  const v4i16 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4i16*)(vb + 4096));
  return __builtin_shufflevector(__builtin_bit_cast(half4, lo), __builtin_bit_cast(half4, hi), 0, 1, 2, 3,
                                 4, 5, 6, 7);
}

// End of a row: each wave's O (fp32), m and l go to LDS (part: kPart bytes per wave), then wave w
// merges the key groups of its share of the kR rows, normalises and stores whole 256-byte rows. The
// rows of row group g (32 rows) were computed by waves g, g + kRG, ...
template <bool kBf16, int kRG, int kKG>
__device__ __forceinline__ void merge_store(const Args& a, State& s, char* lds, int part_stride,
                                            float2 (*ml)[32], size_t base, int bh, int q0, int seq_len,
                                            int wave, int c16, int g4) {
  constexpr int kWaves = kRG * kKG;
  constexpr int kShare = 32 * kRG / kWaves;  // rows of a wave's share
  char* part = lds + wave * part_stride;
#pragma unroll
  for (int qt = 0; qt < 2; ++qt) {
    const float l = wave_quad_sum(s.l[qt]);
    if (g4 == 0) ml[wave][16 * qt + c16] = float2{s.m[qt], l};
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      // Row 16qt + c16 (512 B), 16-byte chunk 4u + g4 stored at chunk ^ c16.
      *(floatx4*)(part + (16 * qt + c16) * 512 + 16 * ((4 * u + g4) ^ c16)) = s.o[qt][u];
    }
  }
  USAGI_BARRIER();
#pragma unroll
  for (int n = 0; n < kShare / 4; ++n) {
    const int row = kShare * wave + 4 * n + g4;
    const int g = row >> 5;
    const int r = row & 31;
    float m = -1e30f;
#pragma unroll
    for (int w = 0; w < kKG; ++w) m = fmaxf(m, ml[w * kRG + g][r].x);
    float l = 0.0f;
    floatx4 acc[2] = {floatx4{0.0f, 0.0f, 0.0f, 0.0f}, floatx4{0.0f, 0.0f, 0.0f, 0.0f}};
#pragma unroll
    for (int w = 0; w < kKG; ++w) {
      const float2 x = ml[w * kRG + g][r];
      const float f = __builtin_amdgcn_exp2f(x.x - m);
      l = fmaf(f, x.y, l);
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        const floatx4 p =
            *(const floatx4*)(lds + (w * kRG + g) * part_stride + r * 512 + 16 * ((2 * c16 + e) ^ (r & 15)));
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[e][i] = fmaf(f, p[i], acc[e][i]);
      }
    }
    const bool valid = q0 + row < seq_len;
    const float inv = l > 0.0f ? 1.0f / l : 1.0f;
    u32x4 out;
#pragma unroll
    for (int e = 0; e < 2; ++e) {
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        out[2 * e + h] = pack_out<kBf16>(acc[e][2 * h] * inv, acc[e][2 * h + 1] * inv);
      }
    }
    if (!valid) out = u32x4{0, 0, 0, 0};
    __builtin_nontemporal_store(out, (u32x4*)(a.o + base + (size_t)(q0 + row) * kHd + 8 * c16));
    if (a.lse && c16 == 0) {
      a.lse[(size_t)bh * a.T + q0 + row] = valid && l > 0.0f ? (m + log2f(l)) * kLn2 : -INFINITY;
    }
  }
}

// ---------------------------------------------------------------------------------------------
// 32 query rows per workgroup; wave w holds keys 32w .. 32w+31 of every block.
// ---------------------------------------------------------------------------------------------
template <bool kBf16, int kRows>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1)))
void bsa_ksplit_kernel(Args a) {
  constexpr bool kGeneric = kRows == kRowsGeneric;
  constexpr int kSlice = 8192;  // a wave's 32 rows of a K or V tile
  constexpr int kWaveLds = 4 * kSlice;
  // Wave w: K and V slices of two stages (K at 32 KiB w + 16 KiB stage, V 8 KiB after it); at the
  // end the wave's fp32 O.
  __shared__ __attribute__((aligned(1024))) char lds[4 * kWaveLds];
  __shared__ float2 ml[4][32];

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int c16 = lane & 15;
  const int g4 = lane >> 4;
  int sub, qb, bh;
  if (!work_of<4>(a, sub, qb, bh)) return;
  const size_t base = (size_t)bh * a.T * kHd;
  const char* k_head = (const char*)(a.k + base) + wave * kSlice;
  const char* v_head = (const char*)(a.v + base) + wave * kSlice;
  uint32_t k_off[4];
  uint32_t v_off[4];
  dma_offsets(lane, k_off, v_off);
  char* const wave_lds = lds + wave * kWaveLds;
  const uint32_t wave_dst = __builtin_amdgcn_readfirstlane(lds_addr_of(lds) + wave * kWaveLds);
  auto fetch = [&](int kb, int stage) {
    const uint32_t dst = wave_dst + stage * 2 * kSlice;
    dma_tile8(k_head + (size_t)kb * kTileBytes, k_off, dst);
    dma_tile8(v_head + (size_t)kb * kTileBytes, v_off, dst + kSlice);
  };

  const int seq_len = a.seq_lens ? a.seq_lens[bh / a.heads] : a.T;
  const int q0 = qb * kBlk + 32 * sub;  // the workgroup's first query row
  if (q0 >= seq_len) {
    store_empty<32, 256>(a, base, bh, q0);
    return;
  }
  // The diagonal goes first; its tiles are requested before the row's entries are read.
  if constexpr (!kGeneric) fetch(qb, 0);
  u32x4 qf[2][4];
  load_q(a, base, q0, seq_len, c16, g4, qf);
  Row<kRows> row(a, qb, bh, lane);
  const int n_blk = row.n_blk;

  // Operand reads of a slice: K tile t (keys 16t .. 16t+15 of the slice), V^T d-tile u.
  const int k_x = g4 ^ c16;
  const int v_x = 8 * (g4 & 1) + 2 * (c16 >> 2) + ((c16 & 3) >> 1);
  const char* k_rd = wave_lds + c16 * 256;
  const char* v_rd = wave_lds + kSlice + (4 * g4 + (c16 >> 2)) * 256 + 8 * (c16 & 1);
  u32x4 kop[2][4];
  auto k_read = [&](int stage) {
#pragma unroll
    for (int t = 0; t < 2; ++t) {
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) {
        kop[t][ks] = *(const u32x4*)(k_rd + stage * 2 * kSlice + t * 4096 + 16 * ((4 * ks) ^ k_x));
      }
    }
  };
  State s;
  const float scale = a.qk_scale;
  if constexpr (kGeneric) {
    if (n_blk > 0) fetch(row.key_block(0), 0);
  }
  // Q, the column chunk and the first K and V slices have landed (a real s_waitcnt: the compiler
  // then knows that no load of its own is outstanding inside the loop).
  __builtin_amdgcn_s_waitcnt(0x0F70);
  // Key blocks of the next two steps.
  int kb_next[2] = {kGeneric && n_blk > 0 ? row.key_block(0) : 0, n_blk > 1 ? row.key_block(1) : 0};
  if (n_blk > 1) fetch(kb_next[1], 1);
  if (n_blk > 0) k_read(0);

  // Step i, the operands of its K already in kop. Requests in flight, oldest first, eight each:
  // V(i), K(i+1), V(i+1). kMore: a step i + 2 exists; its K replaces K(i) during Q·K^T (whose
  // operands are in registers by then) and its V replaces V(i) during P·V.
  auto step = [&](auto diag_tag, auto more_tag, int i) {
    constexpr bool kDiag = decltype(diag_tag)::value;
    constexpr bool kMore = decltype(more_tag)::value;
    const int stage = i & 1;
    const bool next = kMore || i + 1 < n_blk;
    const uint32_t dst = wave_dst + stage * 2 * kSlice;
    const int kb = kDiag ? qb : kb_next[0];
    const int kb2 = kMore ? row.key_block(i + 2) : 0;
    kb_next[0] = kb_next[1];
    kb_next[1] = kb2;
    const char* k2 = k_head + (size_t)kb2 * kTileBytes;
    const char* v2 = v_head + (size_t)kb2 * kTileBytes;
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    if constexpr (kGeneric && !kDiag) {
      if (__builtin_expect(kb * kBlk >= seq_len, 0)) {  // all its keys are past seq_len: nothing but the requests to do
        if constexpr (kMore) {
          dma_tile8(k2, k_off, dst);
          USAGI_WAIT_VM(24);  // V(i) has landed: its slice can be written again
          dma_tile8(v2, v_off, dst + kSlice);
          USAGI_WAIT_VM(24);  // K(i+1) has landed
        } else if (next) {
          USAGI_WAIT_VM(8);
        } else {
          USAGI_WAIT_VM(0);  // V(i) has landed: O takes its place
        }
        if (next) k_read(stage ^ 1);
        return;
      }
    }

    floatx4 st[2][2];
#pragma unroll
    for (int qt = 0; qt < 2; ++qt) st[qt][0] = st[qt][1] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
#pragma unroll
      for (int t = 0; t < 2; ++t) {
#pragma unroll
        for (int qt = 0; qt < 2; ++qt) st[qt][t] = mfma_qk16<kBf16>(kop[t][ks], qf[qt][ks], st[qt][t]);
        if constexpr (kMore) dma_piece(k2, k_off, dst, 2 * ks + t);
      }
    }
    // V(i) has landed: its operands are read while the softmax runs.
    if constexpr (kMore) {
      USAGI_WAIT_VM(24);
    } else if (next) {
      USAGI_WAIT_VM(16);
    } else {
      USAGI_WAIT_VM(0);
    }
    half8 vop[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) vop[u] = v_fragment(v_rd + stage * 2 * kSlice + 16 * ((2 * u) ^ v_x));

    half8 pb[2][1];
    if constexpr (kDiag) {
      mask_diag<2>(st, 32 * sub, 32 * wave, c16, g4);
    } else if constexpr (kGeneric) {
      mask_generic<2>(st, kb, qb, seq_len, 32 * sub, 32 * wave, c16, g4);
    }
    softmax<2, kDiag>(st, s, scale, pb);

    // K(i+1) has landed: its operands are read while P·V runs.
    if (next) {
      if constexpr (kMore) {
        USAGI_WAIT_VM(16);
      } else {
        USAGI_WAIT_VM(8);
      }
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      k_read(stage ^ 1);
    }
    if constexpr (kBf16) {
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        u32x4 x = __builtin_bit_cast(u32x4, vop[u]);
#pragma unroll
        for (int w = 0; w < 4; ++w) x[w] = bf16x2_to_f16x2(x[w]);
        vop[u] = __builtin_bit_cast(half8, x);
      }
    }
    if constexpr (kDiag || kGeneric) {
      // V past seq_len may hold anything, and P = 0 does not cancel a NaN or an infinity there.
      const int n_keys = seq_len - kb * kBlk - 32 * wave;  // of this wave's 32
      if (__builtin_expect(n_keys < 32, 0)) {
        const int n = n_keys - 4 * g4;
        uint32_t keep[4];
#pragma unroll
        for (int w = 0; w < 4; ++w) {
          const int e = 16 * (w >> 1) + 2 * (w & 1);
          keep[w] = (e < n ? 0xffffu : 0u) | (e + 1 < n ? 0xffff0000u : 0u);
        }
#pragma unroll
        for (int u = 0; u < 8; ++u) {
          u32x4 x = __builtin_bit_cast(u32x4, vop[u]);
#pragma unroll
          for (int w = 0; w < 4; ++w) x[w] &= keep[w];
          vop[u] = __builtin_bit_cast(half8, x);
        }
      }
    }
    // On the diagonal a wave whose keys all lie above the rows is skipped.
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      if (!kDiag || wave <= sub) {
#pragma unroll
        for (int qt = 0; qt < 2; ++qt) {
          s.o[qt][u] = __builtin_amdgcn_mfma_f32_16x16x32_f16(vop[u], pb[qt][0], s.o[qt][u], 0, 0, 0);
        }
      }
      if constexpr (kMore) dma_piece(v2, v_off, dst + kSlice, u);
    }
  };

  using T_ = std::true_type;
  using F_ = std::false_type;
  int i = 0;
  if (row.has_diag) {
    if (n_blk > 2) {
      step(T_{}, T_{}, 0);
    } else {
      step(T_{}, F_{}, 0);
    }
    i = 1;
  }
  for (; i < n_blk - 2; ++i) step(F_{}, T_{}, i);
  for (; i < n_blk; ++i) step(F_{}, F_{}, i);
  merge_store<kBf16, 1, 4>(a, s, lds, kWaveLds, ml, base, bh, q0, seq_len, wave, c16, g4);
}

// ---------------------------------------------------------------------------------------------
// Eight waves: row group wave % kRG (32 rows), key group wave / kRG (128 / kKG keys).
// ---------------------------------------------------------------------------------------------
template <bool kBf16, int kRows, int kKG>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2)))
void bsa_wide_kernel(Args a) {
  constexpr bool kGeneric = kRows == kRowsGeneric;
  constexpr int kRG = 8 / kKG;
  constexpr int kR = 32 * kRG;          // query rows of a workgroup
  constexpr int kNT = kBlk / kKG / 16;  // 16-key tiles of a wave
  constexpr int kKS = kNT / 2;          // 32-key steps of its P·V
  // Two stages of a K and a V tile; at the end the eight waves' fp32 O, 16 KiB each.
  __shared__ __attribute__((aligned(1024))) char lds[4 * kTileBytes];
  __shared__ float2 ml[8][32];

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int c16 = lane & 15;
  const int g4 = lane >> 4;
  const int rg = wave % kRG;
  const int kg = wave / kRG;
  int sub, qb, bh;
  if (!work_of<kBlk / kR>(a, sub, qb, bh)) return;
  const size_t base = (size_t)bh * a.T * kHd;
  // A wave's DMA brings rows 16w .. 16w+15 of every tile.
  const char* k_head = (const char*)(a.k + base) + wave * 4096;
  const char* v_head = (const char*)(a.v + base) + wave * 4096;
  uint32_t k_off[4];
  uint32_t v_off[4];
  dma_offsets(lane, k_off, v_off);
  const uint32_t dst0 = __builtin_amdgcn_readfirstlane(lds_addr_of(lds) + wave * 4096);
  // bf16: the rows of V come into registers and go to LDS as fp16 (put_v), swizzled as the DMA of
  // fp16 inputs writes them, so that P·V runs on fp16 P and fp16 V.
  u32x4 vreg[4];
  auto load_v = [&](int kb, int i) {
    vreg[i] = *(const u32x4*)(v_head + (size_t)kb * kTileBytes + i * 1024 + lane * 16);
  };
  auto put_v = [&](int stage, int i) {
    u32x4 x = vreg[i];
#pragma unroll
    for (int w = 0; w < 4; ++w) x[w] = bf16x2_to_f16x2(x[w]);
    *(u32x4*)(lds + (2 * stage + 1) * kTileBytes + wave * 4096 + i * 1024 + v_off[i & 1]) = x;
  };
  auto fetch = [&](int kb, int stage) {
    const uint32_t dst = dst0 + stage * 2 * kTileBytes;
#pragma unroll
    for (int i = 0; i < 4; ++i) dma_piece(k_head + (size_t)kb * kTileBytes, k_off, dst, i);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if constexpr (kBf16) {
        load_v(kb, i);
      } else {
        dma_piece(v_head + (size_t)kb * kTileBytes, v_off, dst + kTileBytes, i);
      }
    }
  };

  const int seq_len = a.seq_lens ? a.seq_lens[bh / a.heads] : a.T;
  const int q0 = qb * kBlk + sub * kR;
  if (q0 >= seq_len) {
    store_empty<kR, 512>(a, base, bh, q0);
    return;
  }
  if constexpr (!kGeneric) fetch(qb, 0);
  u32x4 qf[2][4];
  load_q(a, base, q0 + 32 * rg, seq_len, c16, g4, qf);
  Row<kRows> row(a, qb, bh, lane);
  const int n_blk = row.n_blk;

  const int row0 = sub * kR + 32 * rg;   // the wave's first row of the query block
  const int key0 = kg * (kBlk / kKG);    // and its first key of a key block
  const int k_x = g4 ^ c16;
  const int v_x = 8 * (g4 & 1) + 2 * (c16 >> 2) + ((c16 & 3) >> 1);
  const char* k_rd0 = lds + (key0 + c16) * 256;
  const char* v_rd0 = lds + kTileBytes + (key0 + 4 * g4 + (c16 >> 2)) * 256 + 8 * (c16 & 1);
  State s;
  const float scale = a.qk_scale;
  if constexpr (kGeneric) {
    if (n_blk > 0) fetch(row.key_block(0), 0);
  }
  __builtin_amdgcn_s_waitcnt(0x0F70);
  if constexpr (kBf16) {
    if (n_blk > 0) {
#pragma unroll
      for (int n = 0; n < 4; ++n) put_v(0, n);
    }
  }

  int kb_next = kGeneric && n_blk > 0 ? row.key_block(0) : 0;  // key block of the next step
  // Step i: the tiles of step i + 1 (kMore) are requested during Q·K^T into the other stage, whose
  // readers all passed this step's barrier.
  auto step = [&](auto diag_tag, auto more_tag, int i) {
    constexpr bool kDiag = decltype(diag_tag)::value;
    constexpr bool kMore = decltype(more_tag)::value;
    const int stage = i & 1;
    const int kb = kDiag ? qb : kb_next;
    const int kb1 = kMore ? row.key_block(i + 1) : 0;
    kb_next = kb1;
    const char* k1 = k_head + (size_t)kb1 * kTileBytes;
    const char* v1 = v_head + (size_t)kb1 * kTileBytes;
    const uint32_t dst = dst0 + (stage ^ 1) * 2 * kTileBytes;
    USAGI_WAIT_VM(0);  // this wave's rows of K(i) and V(i) have landed (bf16: V(i) is in LDS as fp16)
    if constexpr (kDiag || kGeneric) {
      if (__builtin_expect((kb + 1) * kBlk > seq_len, 0)) {
        char* rows = lds + (2 * stage + 1) * kTileBytes + wave * 4096;
        const int n = seq_len - kb * kBlk - 16 * wave;
        // V past seq_len may hold anything, and P = 0 does not cancel a NaN or an infinity there.
#pragma unroll
        for (int r = 0; r < 16; r += 4) {
          if (r + g4 >= n) *(u32x4*)(rows + r * 256 + lane * 16) = u32x4{0, 0, 0, 0};
        }
      }
    }
    USAGI_BARRIER();
    if constexpr (kGeneric && !kDiag) {
      if (__builtin_expect(kb * kBlk >= seq_len, 0)) {  // all its keys are past seq_len: nothing but the next tiles to do
        if constexpr (kMore) {
          fetch(kb1, stage ^ 1);
          if constexpr (kBf16) {
#pragma unroll
            for (int n = 0; n < 4; ++n) put_v(stage ^ 1, n);
          }
        }
        return;
      }
    }

    // ---- S^T = K · Q^T: fragment f = kNT * ks + t, read four ahead.
    const char* k_rd = k_rd0 + stage * 2 * kTileBytes;
    const char* v_rd = v_rd0 + stage * 2 * kTileBytes;
    __builtin_amdgcn_s_setprio(1);
    floatx4 st[2][kNT];
#pragma unroll
    for (int qt = 0; qt < 2; ++qt) {
#pragma unroll
      for (int t = 0; t < kNT; ++t) st[qt][t] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
    }
    auto k_read = [&](int f) {
      return *(const u32x4*)(k_rd + (f % kNT) * 4096 + 16 * ((4 * (f / kNT)) ^ k_x));
    };
    constexpr int kF = 4 * kNT;
    u32x4 kop[4];
#pragma unroll
    for (int f = 0; f < 4; ++f) kop[f] = k_read(f);
#pragma unroll
    for (int f = 0; f < kF; ++f) {
      const u32x4 ka = kop[f & 3];
      if (f + 4 < kF) kop[f & 3] = k_read(f + 4);
#pragma unroll
      for (int qt = 0; qt < 2; ++qt) {
        st[qt][f % kNT] = mfma_qk16<kBf16>(ka, qf[qt][f / kNT], st[qt][f % kNT]);
      }
      if constexpr (kMore) {
        constexpr int kEvery = kF / 8;
        if (f % kEvery == kEvery - 1) {
          const int p = f / kEvery;
          if constexpr (kBf16) {
            if (p < 4) {
              load_v(kb1, p);
            } else {
              dma_piece(k1, k_off, dst, p - 4);
            }
          } else if (p < 4) {
            dma_piece(k1, k_off, dst, p);
          } else {
            dma_piece(v1, v_off, dst + kTileBytes, p - 4);
          }
        }
      }
    }
    __builtin_amdgcn_sched_group_barrier(0x100, 4, 1);
#pragma unroll
    for (int n = 0; n < kF - 4; ++n) {
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 1);
      __builtin_amdgcn_sched_group_barrier(0x008, 2, 1);
    }
    __builtin_amdgcn_sched_group_barrier(0x008, 8, 1);
    if constexpr (kDiag) {
      mask_diag<kNT>(st, row0, key0, c16, g4);
    } else if constexpr (kGeneric) {
      mask_generic<kNT>(st, kb, qb, seq_len, row0, key0, c16, g4);
    }
    __builtin_amdgcn_s_setprio(0);
    half8 pb[2][kKS];
    softmax<kNT, kDiag>(st, s, scale, pb);

    // ---- O^T += V^T · P^T, fragment g = 8ks + u read four ahead. On the diagonal the 32-key steps
    // above the wave's rows are skipped.
    __builtin_amdgcn_s_setprio(1);
    auto v_read = [&](int g) { return v_fragment(v_rd + (g >> 3) * 8192 + 16 * ((2 * (g & 7)) ^ v_x)); };
    constexpr int kG = 8 * kKS;
    half8 vop[4];
#pragma unroll
    for (int g = 0; g < 4; ++g) vop[g] = v_read(g);
#pragma unroll
    for (int g = 0; g < kG; ++g) {
      const half8 va = vop[g & 3];
      if (g + 4 < kG) vop[g & 3] = v_read(g + 4);
      if (!kDiag || key0 + 32 * (g >> 3) <= row0) {
#pragma unroll
        for (int qt = 0; qt < 2; ++qt) {
          s.o[qt][g & 7] = __builtin_amdgcn_mfma_f32_16x16x32_f16(va, pb[qt][g >> 3], s.o[qt][g & 7], 0, 0, 0);
        }
      }
      if constexpr (kBf16 && kMore) {
        if (g >= kG - 8 && g % 2 == 1) put_v(stage ^ 1, (g - kG + 8) / 2);
      }
    }
    if constexpr (!kDiag) {
      __builtin_amdgcn_sched_group_barrier(0x100, 8, 2);
#pragma unroll
      for (int n = 0; n < kG - 4; ++n) {
        __builtin_amdgcn_sched_group_barrier(0x008, 2, 2);
        __builtin_amdgcn_sched_group_barrier(0x100, 2, 2);
      }
      __builtin_amdgcn_sched_group_barrier(0x008, 8, 2);
    }
    __builtin_amdgcn_s_setprio(0);
  };

  using T_ = std::true_type;
  using F_ = std::false_type;
  int i = 0;
  if (row.has_diag) {
    if (n_blk > 1) {
      step(T_{}, T_{}, 0);
    } else {
      step(T_{}, F_{}, 0);
    }
    i = 1;
  }
  for (; i < n_blk - 1; ++i) step(F_{}, T_{}, i);
  if (i < n_blk) step(F_{}, F_{}, i);
  USAGI_BARRIER();  // every wave is done reading the tiles
  merge_store<kBf16, kRG, kKG>(a, s, lds, 16384, ml, base, bh, q0, seq_len, wave, c16, g4);
}

template <bool kBf16, int kRows>
SmallKernel kernel_of(int query_rows) {
  switch (query_rows) {
    case 32: return {reinterpret_cast<const void*>(&bsa_ksplit_kernel<kBf16, kRows>), 256};
    case 64: return {reinterpret_cast<const void*>(&bsa_wide_kernel<kBf16, kRows, 4>), 512};
    default: return {reinterpret_cast<const void*>(&bsa_wide_kernel<kBf16, kRows, 2>), 512};
  }
}

}  // namespace

SmallKernel usagi_bsa_small_kernel(bool bf16, int rows, int query_rows) {
  switch (rows) {
    case kRowsCsr: return bf16 ? kernel_of<true, kRowsCsr>(query_rows) : kernel_of<false, kRowsCsr>(query_rows);
    case kRowsWindow:
      return bf16 ? kernel_of<true, kRowsWindow>(query_rows) : kernel_of<false, kRowsWindow>(query_rows);
    default:
      return bf16 ? kernel_of<true, kRowsGeneric>(query_rows) : kernel_of<false, kRowsGeneric>(query_rows);
  }
}
