// block_copy.hip — rxmet_block_copy: widen or narrow the tensors of a call to whole unit tiles.
//
// Bound by launches: the tensors are small (a [3 x 100, 100] weight) except the states and their
// gradients [T, B, H], and one launch takes the place of a fill and one copy per block and tensor
// (a training step at T 61, B 50, I 23, H 100: 1280 - 1450 us with those, 590 us with four of
// these launches, host-bound both times).
// One thread per destination element, so that the stores are whole cache lines; the quotients
// come from multiplications (fast_div), since three divisions per element (some 60 vector
// operations) would cost more than the element's 8 bytes of traffic on the large tensors.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "rxmet_common.h"
#include "rxmet_layout.h"

namespace rxmet {
namespace {

constexpr int kThreads = 256;
constexpr int kMaxBlocks = 4096;                  // per job; a grid-stride loop takes the rest
constexpr int64_t kMaxElems = (int64_t(1) << 30);  // per part of a job, for the 31-bit quotients

// n / d for n < 2^31: floor((mulhi(n, m) + n) / 2^s), s = ceil(log2 d), m = floor(2^32 (2^s - d)
// / d) + 1 (Granlund and Montgomery); the sum stays below 2^32 because mulhi(n, m) <= n.
struct FastDiv {
  uint32_t d, m, s;
};

FastDiv fast_div(uint32_t d) {
  uint32_t s = 0;
  while ((uint64_t(1) << s) < d) ++s;
  return {d, static_cast<uint32_t>(((uint64_t(1) << 32) * ((uint64_t(1) << s) - d)) / d + 1), s};
}

struct Part {
  const float *src;
  float *dst;
  uint32_t n;  // destination elements
  uint32_t rows_src, cols_src;
  FastDiv cols, groups, rows;  // of dst
};

struct Parts {
  Part p[RXMET_BLOCK_JOBS];
};

__device__ __forceinline__ uint32_t quotient(uint32_t n, FastDiv f) {
  return (__umulhi(n, f.m) + n) >> f.s;
}

__global__ __launch_bounds__(kThreads) void block_copy(Parts parts) {
  const Part p = parts.p[blockIdx.y];
  const uint32_t step = gridDim.x * kThreads;
  for (uint32_t i = blockIdx.x * kThreads + threadIdx.x; i < p.n; i += step) {
    const uint32_t q0 = quotient(i, p.cols), c = i - q0 * p.cols.d;
    const uint32_t q1 = quotient(q0, p.groups), g = q0 - q1 * p.groups.d;
    const uint32_t a = quotient(q1, p.rows), r = q1 - a * p.rows.d;
    float v = 0.0f;
    if (r < p.rows_src && c < p.cols_src)
      v = p.src[((int64_t(a) * p.rows_src + r) * p.groups.d + g) * p.cols_src + c];
    p.dst[i] = v;
  }
}

int launch(const Parts &parts, int n, uint32_t most, hipStream_t s) {
  const uint32_t blocks = std::min<uint32_t>((most + kThreads - 1) / kThreads, kMaxBlocks);
  hipLaunchKernelGGL(block_copy, dim3(blocks, n), dim3(kThreads), 0, s, parts);
  RXMET_CHECK_LAUNCH();
  return 0;
}

}  // namespace
}  // namespace rxmet

using namespace rxmet;

extern "C" int rxmet_block_copy(int32_t n, const rxmet_block_job *jobs, void *stream) {
  clear_error();
  RXMET_CHECK_ARG(jobs != nullptr && n >= 1 && n <= RXMET_BLOCK_JOBS,
                  "block copy: 1 to 16 jobs");
  hipStream_t s = static_cast<hipStream_t>(stream);
  for (int k = 0; k < n; ++k) {
    const rxmet_block_job &j = jobs[k];
    RXMET_CHECK_ARG(j.outer >= 0 && j.rows_src >= 0 && j.rows_dst >= 0 && j.groups >= 0 &&
                        j.cols_src >= 0 && j.cols_dst >= 0 && j.reserved == 0,
                    "block copy: sizes must not be negative");
    const __int128 row = static_cast<__int128>(j.rows_dst) * j.groups * j.cols_dst;
    RXMET_CHECK_ARG(row <= kMaxElems, "block copy: one outer row holds too many elements");
    const bool reads = row > 0 && j.outer > 0 && j.rows_src > 0 && j.cols_src > 0;
    RXMET_CHECK_ARG(row == 0 || j.outer == 0 || (j.dst != nullptr && (!reads || j.src != nullptr)),
                    "block copy: src and dst must be non-null");
  }
  Parts parts;
  int used = 0;
  uint32_t most = 0;
  for (int k = 0; k < n; ++k) {
    const rxmet_block_job &j = jobs[k];
    const int64_t row = int64_t(j.rows_dst) * j.groups * j.cols_dst;
    const int64_t row_src = int64_t(j.rows_src) * j.groups * j.cols_src;
    if (row == 0) continue;
    const int64_t most_outer = kMaxElems / row;
    for (int64_t a = 0; a < j.outer; a += most_outer) {
      const uint32_t e = static_cast<uint32_t>(std::min(most_outer, j.outer - a) * row);
      parts.p[used++] = {j.src == nullptr ? nullptr : j.src + a * row_src, j.dst + a * row, e,
                         static_cast<uint32_t>(j.rows_src), static_cast<uint32_t>(j.cols_src),
                         fast_div(j.cols_dst), fast_div(j.groups), fast_div(j.rows_dst)};
      most = std::max(most, e);
      if (used == RXMET_BLOCK_JOBS) {
        if (int rc = launch(parts, used, most, s)) return rc;
        used = 0;
        most = 0;
      }
    }
  }
  return used ? launch(parts, used, most, s) : 0;
}
