// A fixed permutation of float32 values in two streaming passes (gfx950).
//
// The transposed matrix's weights in slot order are the CSR weights permuted:
// read slot by slot, every 4-byte weight is a cache line of its own from the
// last-level cache (N=166k, M=25M: 417 us for 100 MB).  Here the values first
// move, chunk by chunk of consecutive CSR edges, through LDS into per-bucket
// order, one bucket being a stretch of slots that fits LDS too; then each bucket
// is read back whole and dealt to its slots from LDS.  Both passes read and write
// memory in runs: at 25M edges a chunk's run for a bucket is about 26 values.  The
// two passes take 120 us there: 100 MB of values read and written in each, with the
// 16-bit tables 505 MB (4.2 TB/s).
#include <hip/hip_runtime.h>

#include "neurosim_hip_layout.h"
#include "ns_common.h"
#include "ns_host.h"

namespace ns {
namespace {

constexpr int kPermuteThreads = 1024;
constexpr int kPermuteWaves = kPermuteThreads / 64;

typedef float v4f __attribute__((ext_vector_type(4)));
typedef uint16_t v4u16 __attribute__((ext_vector_type(4)));

// One workgroup per chunk: the chunk's values to LDS in bucket order, then each
// bucket's run to its place in the workspace, a wavefront per run.  The runs'
// bounds come 64 at a time, one per lane, so that no run waits for its own.
__global__ __launch_bounds__(kPermuteThreads) void chunk_to_buckets_kernel(
    ns_blocked_permutation p, const float* values, float* workspace, int aligned) {
  extern __shared__ float held[];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int64_t base = static_cast<int64_t>(blockIdx.x) * p.chunk;
  const int count = static_cast<int>(min<int64_t>(p.chunk, p.n_edges - base));
  const int whole = aligned ? count & ~3 : 0;
  for (int i = 4 * tid; i < whole; i += 4 * kPermuteThreads) {
    const v4f x = *reinterpret_cast<const v4f*>(values + base + i);
    const v4u16 at = *reinterpret_cast<const v4u16*>(p.place + base + i);
#pragma unroll
    for (int k = 0; k < 4; ++k)
      if (at[k] < count) held[at[k]] = x[k];
  }
  for (int i = whole + tid; i < count; i += kPermuteThreads) {
    const int at = p.place[base + i];
    if (at < count) held[at] = values[base + i];
  }
  __syncthreads();
  const uint16_t* const starts = p.run_start + static_cast<int64_t>(blockIdx.x) * (p.n_buckets + 1);
  const int32_t* const targets = p.run_target + static_cast<int64_t>(blockIdx.x) * p.n_buckets;
  for (int b0 = wave * 64; b0 < p.n_buckets; b0 += kPermuteWaves * 64) {
    const int b = min(b0 + lane, p.n_buckets - 1);
    const int from = min<int>(starts[b], count), to = min<int>(starts[b + 1], count);
    const int target = targets[b];
    const int runs = min(64, p.n_buckets - b0);
    for (int r = 0; r < runs; ++r) {
      const int first = __builtin_amdgcn_readlane(from, r);
      const int last = __builtin_amdgcn_readlane(to, r);
      const int64_t out = __builtin_amdgcn_readlane(target, r);
      for (int i = first + lane; i < last; i += 64) {
        const int64_t at = out + (i - first);
        if (at >= 0 && at < p.n_edges) workspace[at] = held[i];
      }
    }
  }
}

// One workgroup per bucket: its values to LDS, then its slots.
__global__ __launch_bounds__(kPermuteThreads) void bucket_to_slots_kernel(
    ns_blocked_permutation p, const float* workspace, float* slots) {
  extern __shared__ float held[];
  const int tid = threadIdx.x;
  const int64_t start = max(p.bucket_start[blockIdx.x], 0);
  const int64_t end = min<int64_t>(p.bucket_start[blockIdx.x + 1], p.n_edges);
  const int count = static_cast<int>(min<int64_t>(max<int64_t>(end - start, 0), p.bucket));
  // From a 16-byte boundary of the workspace on, four values at a time.
  const int skip = static_cast<int>(start & 3);
  for (int i = 4 * tid; i < count + skip; i += 4 * kPermuteThreads) {
    const int64_t at = start - skip + i;
    if (at + 4 <= p.n_edges) {
      const v4f x = *reinterpret_cast<const v4f*>(workspace + at);
#pragma unroll
      for (int k = 0; k < 4; ++k)
        if (i + k >= skip && i + k - skip < count) held[i + k - skip] = x[k];
    } else {
      for (int k = 0; k < 4; ++k)
        if (i + k >= skip && i + k - skip < count) held[i + k - skip] = workspace[at + k];
    }
  }
  __syncthreads();
  const int64_t first = static_cast<int64_t>(blockIdx.x) * p.bucket;
  const int n = static_cast<int>(min<int64_t>(p.bucket, p.n_slots - first));
  for (int k = 4 * tid; k < n; k += 4 * kPermuteThreads) {
    const v4u16 from = *reinterpret_cast<const v4u16*>(p.slot_source + first + k);
    v4f out;
#pragma unroll
    for (int j = 0; j < 4; ++j) out[j] = from[j] < count ? held[from[j]] : 0.0f;
    *reinterpret_cast<v4f*>(slots + first + k) = out;
  }
}

}  // namespace
}  // namespace ns

using namespace ns;

extern "C" int ns_permute_blocked(const ns_blocked_permutation* permutation, const float* values,
                                  float* workspace, float* slots, void* stream) {
  clear_error();
  if (!permutation) return fail("a permutation is required");
  const ns_blocked_permutation& p = *permutation;
  if (p.n_edges < 0 || p.n_edges >= (int64_t{1} << 31)) return fail("n_edges must be in [0, 2^31)");
  if (p.n_slots < 0 || p.n_slots % 4 || p.n_slots >= (int64_t{1} << 32))
    return fail("n_slots must be a multiple of 4 in [0, 2^32)");
  for (const int32_t size : {p.chunk, p.bucket})
    if (size < 4 || size % 4 || size > NS_BLOCKED_MAX)
      return fail("chunks and buckets are a multiple of 4 from 4 to %d", NS_BLOCKED_MAX);
  if (p.n_chunks != (p.n_edges + p.chunk - 1) / p.chunk)
    return fail("the permutation has %d chunks for %lld edges", p.n_chunks, (long long)p.n_edges);
  if (p.n_buckets != (p.n_slots + p.bucket - 1) / p.bucket)
    return fail("the permutation has %d buckets for %lld slots", p.n_buckets, (long long)p.n_slots);
  if (p.n_slots == 0) return NS_OK;
  if (!p.bucket_start || !p.slot_source || !slots || !workspace)
    return fail("tables, workspace and slots are required");
  if (p.n_edges > 0 && (!p.place || !p.run_start || !p.run_target || !values))
    return fail("chunk tables and values are required");
  if (reinterpret_cast<uintptr_t>(slots) % 16 || reinterpret_cast<uintptr_t>(workspace) % 16 ||
      reinterpret_cast<uintptr_t>(p.slot_source) % 8 || reinterpret_cast<uintptr_t>(p.place) % 8)
    return fail("slots and workspace must be 16-byte, slot_source and place 8-byte aligned");
  if (overlaps(extent_of(workspace, 0, 1, 1, p.n_edges), extent_of(slots, 0, 1, 1, p.n_slots)) ||
      overlaps(extent_of(workspace, 0, 1, 1, p.n_edges), extent_of(values, 0, 1, 1, p.n_edges)) ||
      overlaps(extent_of(slots, 0, 1, 1, p.n_slots), extent_of(values, 0, 1, 1, p.n_edges)))
    return fail("values, workspace and slots must not overlap");
  const hipStream_t s = static_cast<hipStream_t>(stream);
  if (p.n_chunks > 0) {
    chunk_to_buckets_kernel<<<dim3(p.n_chunks), dim3(kPermuteThreads), p.chunk * 4, s>>>(
        p, values, workspace, reinterpret_cast<uintptr_t>(values) % 16 == 0);
    const hipError_t err = hipGetLastError();
    if (err != hipSuccess) return fail_launch("permutation", err);
  }
  bucket_to_slots_kernel<<<dim3(p.n_buckets), dim3(kPermuteThreads), p.bucket * 4, s>>>(
      p, workspace, slots);
  const hipError_t err = hipGetLastError();
  if (err != hipSuccess) return fail_launch("permutation", err);
  return NS_OK;
}
