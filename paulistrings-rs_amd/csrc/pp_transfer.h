// pp_transfer.h -- device halves of the bulk transfers (pp_transfer.hip): an upload's terms bucketed on the device,
// and a download's terms put into the canonical order there.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "pp_device.h"

namespace pp {

// The longest device bucket an upload lays out on the device (k_upload_rows orders a bucket's terms by counting, which
// grows with its square), and the largest reference bucket a download sorts in one workgroup's LDS (the keys, the
// coefficients and a 16-bit index per row: 84 KiB at W = 2, 104 KiB at W = 1).
constexpr uint32_t kUploadBucketRows = 2048;
// The most terms: a term's number, and the grid's threads past the last term, are 32-bit.
constexpr uint64_t kUploadTerms = 0xFFFFFFFFull - kBlock;
template <int W>
constexpr uint32_t kSortRows = W == 1 ? 4096u : 2048u;
constexpr uint32_t kSortParts = 256;  // device buckets one reference bucket may gather, or the other way round

// Terms as the host hands them over: term-major keys, x[i * W + w].
template <int W, typename T>
struct UploadArgs {
    const uint64_t* x;
    const uint64_t* z;
    const T* c;
    uint32_t n;
    const uint64_t* rows;  // hash rows
    int32_t bits;
    uint32_t num_buckets;
    uint32_t* bucket;  // per term: its bucket, and its place among the bucket's terms in order of arrival
    uint32_t* place;
    uint32_t* index;   // per column position: the term to put there, unordered within a bucket
    const uint64_t* start;
    uint32_t* len;
    uint64_t* ox;
    uint64_t* oz;
    T* oc;
    uint64_t ocap;
};

// The resident columns, read in the reference's order.  Both bucket counts are low bits of one hash: reference bucket
// rb holds the device buckets congruent to rb, or device bucket b (when there are fewer) the reference buckets
// congruent to b.
template <int W, typename T>
struct SortExportArgs {
    const uint64_t* x;
    const uint64_t* z;
    const T* c;
    uint64_t cap;
    const uint64_t* start;
    const uint32_t* len;
    uint32_t num_buckets;
    uint32_t ref_buckets;
    const uint64_t* rows;  // hash rows
    int32_t bits;          // device bucket bits
    uint32_t* ref_len;     // rows per reference bucket
    const uint64_t* ref_start;  // dense
    uint64_t* out_x;            // term-major
    uint64_t* out_z;
    T* out_c;
};

// Each nonzero term's bucket and place; len (zero before) counts them.
template <int W, typename T>
hipError_t launch_upload_count(hipStream_t st, const UploadArgs<W, T>& a);
// The terms into their buckets' segments, each bucket in the order the host gave them.
template <int W, typename T>
hipError_t launch_upload_rows(hipStream_t st, const UploadArgs<W, T>& a);
// ref_len (zero before) of a layout with fewer device buckets than reference buckets.
template <int W, typename T>
hipError_t launch_ref_counts(hipStream_t st, const SortExportArgs<W, T>& a);
// rows: the longest bucket of the coarser bucketing, at most kSortRows<W>.
template <int W, typename T>
hipError_t launch_sort_export(hipStream_t st, const SortExportArgs<W, T>& a, uint32_t rows);

}  // namespace pp
