// CSR check on the GPU: the preconditions of the implicit-diagonal walk (usagi_bsa_check_csr), the
// window pattern the rows may spell out, and the length of every row, without copying the CSR to the
// host. A first call launches it ahead of the forward kernel, on the same stream, which it delays by its
// own time; the host waits for the result and reads it while the forward kernel runs.
//
// One wave per row, four rows in flight per workgroup; the time is the chain of dependent loads
// (row_ptr, column indices) of the few rows a wave gets: 4.8-6.6 us over 256 rows of 16 entries that are
// in the caches, 5.4-10.2 us for the first pass over a CSR of 32 to 2048 rows.
#include <hip/hip_runtime.h>

#include <stdint.h>

#include "bsa_internal.h"
#include "usagi_bsa.h"

namespace {

constexpr int kThreads = 256;
constexpr int kWaves = kThreads / 64;
constexpr int kMaxBlocks = USAGI_BSA_CHECK_MAX_BLOCKS;
constexpr int kMaxGroups = 1024;
constexpr int kFlagBits = USAGI_BSA_CHECK_FLAG_BITS;
constexpr int kMaxEntries = 0x7fffffff >> kFlagBits;  // above every row of kMaxBlocks full causal ones

struct CheckArgs {
  const int32_t* row_ptr;
  const int32_t* col_idx;
  const int32_t* seq_lens;  // or NULL: every row counts
  int32_t* result;
  int heads;
  int bh_count;
  int nqb;
  int max_nnz;
  int groups;
  int with_entries;  // the flag words hold the largest row end too
};

__global__ __launch_bounds__(kThreads) void bsa_check_kernel(CheckArgs a) {
  __shared__ uint32_t listed[kWaves][kMaxBlocks / 32];  // key blocks of the wave's row
  __shared__ int flags[kWaves];
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int nqb = a.nqb;
  const int n_rows = a.bh_count * nqb;
  auto in_list = [&](int rs, int re) { return 0 <= rs && rs < re && re <= a.max_nnz; };

  // The pattern is read off the last row of the first head: a run of `window` consecutive blocks that
  // ends at the diagonal, after a prefix 0 .. n_global-1.
  const int last = nqb - 1;
  int window = 0;
  int n_global = 0;
  {
    const int rs = a.row_ptr[last];
    const int re = a.row_ptr[nqb];
    if (in_list(rs, re)) {
      const int n = re - rs;
      const int32_t* c = a.col_idx + rs;
      window = n;
      for (int k0 = 0; k0 < n; k0 += 64) {
        const int k = k0 + lane;
        const uint64_t off = __ballot(k < n && c[n - 1 - k] != last - k);
        if (off) {
          window = k0 + __builtin_ctzll(off);
          break;
        }
      }
      n_global = n - window;
    }
  }

  int bad = 0;   // 1: a row before seq_len, 4: one at or past it, which the walk never reads
  int differs = window == 0;
  int entries = 0;  // largest end of a row
  for (int row = blockIdx.x * kWaves + wave; row < n_rows; row += a.groups * kWaves) {
    const int bh = row / nqb;
    const int qb = row - bh * nqb;
    const int32_t* rp = a.row_ptr + (size_t)bh * (nqb + 1) + qb;
    const int rs = rp[0];
    const int re = rp[1];
    const int bad_row = a.seq_lens && qb * USAGI_BSA_BLOCK >= a.seq_lens[bh / a.heads] ? 4 : 1;
    const bool listless = !in_list(rs, re) || (qb == 0 && rs != 0);
    if (lane == 0) a.result[a.groups + 2 + row] = listless && bad_row == 4 ? 0 : max(re - rs, 0);
    if (listless) {
      bad |= bad_row;
      differs = 1;
      continue;
    }
    entries = max(entries, re);
    const int n = re - rs;
    const int lo = max(qb - window + 1, 0);
    const int ng = min(n_global, lo);
    if (n != ng + (qb - lo + 1)) differs = 1;
    const int32_t* c = a.col_idx + (size_t)bh * a.max_nnz + rs;
    for (int w = lane; w < (nqb + 31) / 32; w += 64) listed[wave][w] = 0;
    // LDS operations of one wave complete in order: only the compiler has to keep theirs.
    __builtin_amdgcn_wave_barrier();
    bool wrong = false;
    for (int k = lane; k < n; k += 64) {
      const int kb = c[k];
      if (kb != (k < ng ? k : lo + (k - ng))) differs = 1;
      if (k == n - 1) {
        wrong |= kb != qb;
      } else if (kb < 0 || kb >= qb) {
        wrong = true;
      } else {
        wrong |= (atomicOr(&listed[wave][kb >> 5], 1u << (kb & 31)) >> (kb & 31)) & 1u;
      }
    }
    if (wrong) bad |= bad_row;
  }
  const int f = (__any(bad & 1) ? 1 : 0) | (__any(differs) ? 2 : 0) | (__any(bad & 4) ? 4 : 0);
  if (lane == 0) flags[wave] = min(entries, kMaxEntries) << kFlagBits | f;
  __syncthreads();
  if (threadIdx.x == 0) {
    int all = 0;
    int most = 0;
    for (int w = 0; w < kWaves; ++w) {
      all |= flags[w] & ((1 << kFlagBits) - 1);
      most = max(most, flags[w] >> kFlagBits);
    }
    a.result[blockIdx.x] = (a.with_entries ? most << kFlagBits : 0) | all;
    if (blockIdx.x == 0) {
      a.result[a.groups] = window;
      a.result[a.groups + 1] = n_global;
    }
  }
}

int launch_check(const int32_t* row_ptr, const int32_t* col_idx, const int32_t* seq_lens, int32_t batch,
                 int32_t heads, int32_t num_q_blocks, int32_t max_nnz, int32_t* result,
                 int32_t result_cap, void* stream, bool with_entries) {
  usagi_bsa_clear_error();
  if (!row_ptr || !result || batch <= 0 || heads <= 0 || num_q_blocks <= 0 || max_nnz < 0 ||
      (max_nnz > 0 && !col_idx))
    return usagi_bsa_fail(USAGI_BSA_EINVAL, "bad arguments");
  const int64_t bh = (int64_t)batch * heads;
  const int64_t rows = bh * num_q_blocks;
  if (num_q_blocks > kMaxBlocks || rows > 0x3fffffffLL)
    return usagi_bsa_fail(USAGI_BSA_EINVAL, "problem too large");
  CheckArgs a;
  a.row_ptr = row_ptr;
  a.col_idx = col_idx;
  a.seq_lens = seq_lens;
  a.heads = heads;
  a.with_entries = with_entries ? 1 : 0;
  a.result = result;
  a.bh_count = (int)bh;
  a.nqb = num_q_blocks;
  a.max_nnz = max_nnz;
  // Two rows per wave while the workgroups last.
  const int64_t want = (rows + 2 * kWaves - 1) / (2 * kWaves);
  a.groups = (int)(want < kMaxGroups ? want : kMaxGroups);
  if (result_cap < a.groups + 2 + rows)
    return usagi_bsa_fail(USAGI_BSA_EINVAL, "result_cap %d below %lld", (int)result_cap,
                          (long long)(a.groups + 2 + rows));
  void* params[] = {&a};
  const hipError_t err =
      hipLaunchKernel(reinterpret_cast<const void*>(&bsa_check_kernel), dim3((unsigned)a.groups),
                      dim3(kThreads), params, 0, static_cast<hipStream_t>(stream));
  if (err != hipSuccess) {
    usagi_bsa_fail((int)err, "kernel launch failed: %s", hipGetErrorString(err));
    return -1000 - (int)err;
  }
  return a.groups;
}

}  // namespace

extern "C" int usagi_bsa_check_csr_gpu(const int32_t* row_ptr, const int32_t* col_idx, int32_t batch,
                                       int32_t heads, int32_t num_q_blocks, int32_t max_nnz,
                                       int32_t* result, int32_t result_cap, void* stream) {
  return launch_check(row_ptr, col_idx, nullptr, batch, heads, num_q_blocks, max_nnz, result, result_cap,
                      stream, false);
}

extern "C" int usagi_bsa_check_csr_gpu_lens(const int32_t* row_ptr, const int32_t* col_idx,
                                            const int32_t* seq_lens, int32_t batch, int32_t heads,
                                            int32_t num_q_blocks, int32_t max_nnz, int32_t* result,
                                            int32_t result_cap, void* stream) {
  return launch_check(row_ptr, col_idx, seq_lens, batch, heads, num_q_blocks, max_nnz, result, result_cap,
                      stream, true);
}
