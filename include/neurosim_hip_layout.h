/* Layout helpers of the gfx950 dendritic tick library: entry points that the
 * Python package's slot layouts call beside the tick's own (neurosim_hip.h).
 * Conventions (status codes, ns_last_error, caller's stream) are those of that
 * header. */
#ifndef NEUROSIM_HIP_LAYOUT_H
#define NEUROSIM_HIP_LAYOUT_H

#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

/* Most edges per chunk and slots per bucket of a blocked permutation. */
#define NS_BLOCKED_MAX 36864

/* A fixed permutation of M float32 values into n_slots slots, cut into chunks of
 * `chunk` consecutive sources and buckets of `bucket` consecutive slots (multiples
 * of 4 up to NS_BLOCKED_MAX, what one workgroup holds in LDS).  Within a chunk the values are ordered by bucket (and by
 * source within one); the workspace holds every bucket's values, chunk by chunk. */
typedef struct ns_blocked_permutation {
  int64_t n_edges, n_slots;    /* n_slots a multiple of 4 */
  int32_t chunk, bucket;
  int32_t n_chunks, n_buckets; /* ceil(n_edges / chunk), ceil(n_slots / bucket) */
  const uint16_t* place;       /* [n_edges]: the source's position in its chunk's order */
  const uint16_t* run_start;   /* [n_chunks][n_buckets + 1]: the chunk's runs in that order */
  const int32_t* run_target;   /* [n_chunks][n_buckets]: each run's place in the workspace */
  const int32_t* bucket_start; /* [n_buckets + 1]: each bucket's values in the workspace */
  const uint16_t* slot_source; /* [n_slots]: the slot's value within its bucket's values;
                                  0xFFFF: padding, zero */
} ns_blocked_permutation;

/* slots[k] = values[source of slot k] (0 for padding) through `workspace`
 * (float32[n_edges]); 16-byte aligned `slots`.  Every table entry is checked
 * against its bounds by the kernels. */
int ns_permute_blocked(const ns_blocked_permutation* permutation, const float* values,
                       float* workspace, float* slots, void* stream);

#ifdef __cplusplus
}
#endif

#endif  /* NEUROSIM_HIP_LAYOUT_H */
