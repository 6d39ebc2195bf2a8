// pp_transfer.hip -- the device halves of pp_sum_upload and pp_sum_download: bucketing a host's terms, and the
// reference's canonical order (bucket ascending, then the key's words; pauli_sum/storage.rs:285-295).
#include "pp_transfer.h"

namespace pp {

namespace {

template <int W>
__device__ __forceinline__ Key<W> term_key(const uint64_t* __restrict__ x, const uint64_t* __restrict__ z, uint64_t i) {
    Key<W> k;
    if constexpr (W == 2) {  // a term's two words in one 16-byte load (the arrays start 16-byte aligned)
        const ulonglong2 a = reinterpret_cast<const ulonglong2*>(x)[i], b = reinterpret_cast<const ulonglong2*>(z)[i];
        k.x[0] = a.x;
        k.x[1] = a.y;
        k.z[0] = b.x;
        k.z[1] = b.y;
    } else {
#pragma unroll
        for (int w = 0; w < W; ++w) {
            k.x[w] = x[i * W + w];
            k.z[w] = z[i * W + w];
        }
    }
    return k;
}

template <int W, typename T>
__global__ void __launch_bounds__(kBlock) k_upload_count(const UploadArgs<W, T> a) {
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= a.n) return;
    uint32_t b = 0xFFFFFFFFu, p = 0;
    if (a.c[i] != T(0)) {
        b = bucket_of<W>(term_key<W>(a.x, a.z, i), a.rows, a.bits);
        p = atomicAdd(&a.len[b], 1u);
    }
    a.bucket[i] = b;
    a.place[i] = p;
}

template <int W, typename T>
__global__ void __launch_bounds__(kBlock) k_upload_index(const UploadArgs<W, T> a) {
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= a.n) return;
    const uint32_t b = a.bucket[i];
    if (b != 0xFFFFFFFFu) a.index[a.start[b] + a.place[i]] = i;
}

// A workgroup per bucket: its terms' numbers, which arrived in the order of the count's atomics, ranked by counting the
// smaller ones (a bucket holds about 256), then each row gathered from the host's layout and written to its column
// position.  The layout is the same on every run: each bucket in the order of the host's arrays.  Counting beats a sort
// while buckets are short: 256 rows are 64 16-byte LDS broadcasts per thread.  2^20 two-word f64 terms go up in 2.3 ms,
// the bus and the copy into pinned memory being most of it, against 19.0 ms with the host's counting sort.
template <int W, typename T>
__global__ void __launch_bounds__(kBlock) k_upload_rows(const UploadArgs<W, T> a) {
    __shared__ __align__(16) uint32_t got[kUploadBucketRows];
    __shared__ uint32_t sorted[kUploadBucketRows];
    const uint32_t b = blockIdx.x;
    const uint32_t n = a.len[b];
    const uint64_t s = a.start[b];
    if (n == 0 || n > kUploadBucketRows) return;  // uniform (the host launches this for shorter buckets only)
    const uint32_t n4 = (n + 3u) & ~3u;
    for (uint32_t r = threadIdx.x; r < n4; r += kBlock) got[r] = r < n ? a.index[s + r] : 0xFFFFFFFFu;
    __syncthreads();
    for (uint32_t r = threadIdx.x; r < n; r += kBlock) {
        const uint32_t mine = got[r];
        uint32_t before = 0;
        for (uint32_t q = 0; q < n4; q += 4) {
            const uint4 v = *reinterpret_cast<const uint4*>(&got[q]);
            before += (v.x < mine) + (v.y < mine) + (v.z < mine) + (v.w < mine);
        }
        sorted[before] = mine;
    }
    __syncthreads();
    for (uint32_t r = threadIdx.x; r < n; r += kBlock) {
        const uint32_t i = sorted[r];
        store_key<W>(a.ox, a.oz, a.ocap, s + r, term_key<W>(a.x, a.z, i));
        a.oc[s + r] = a.c[i];
    }
}

// The reference bucket's bits above the device's, for a layout of fewer device buckets.
template <int W, typename T>
__device__ __forceinline__ uint32_t ref_part(const SortExportArgs<W, T>& a, const Key<W>& k, uint32_t parts) {
    uint32_t p = 0;
    for (uint32_t r = 0; (1u << r) < parts; ++r) p |= row_parity<W>(k, a.rows, a.bits + (int)r) << r;
    return p;
}

template <int W, typename T>
__global__ void __launch_bounds__(kBlock) k_ref_counts(const SortExportArgs<W, T> a) {
    __shared__ uint32_t count[kSortParts];
    const uint32_t b = blockIdx.x, parts = a.ref_buckets / a.num_buckets;
    for (uint32_t e = threadIdx.x; e < parts; e += kBlock) count[e] = 0u;
    __syncthreads();
    const uint32_t n = a.len[b];
    const uint64_t s = a.start[b];
    for (uint32_t r = threadIdx.x; r < n; r += kBlock)
        atomicAdd(&count[ref_part<W, T>(a, load_key<W>(a.x, a.z, a.cap, s + r), parts)], 1u);
    __syncthreads();
    for (uint32_t e = threadIdx.x; e < parts; e += kBlock) a.ref_len[b + e * a.num_buckets] = count[e];
}

// A workgroup per bucket of the coarser bucketing: its rows into LDS, a bitonic sort of 16-bit row indices by the
// reference bucket and the keys' words (x ascending, then z), and the rows written out term-major in that order.
// SPLIT: a device bucket of several reference buckets; else a reference bucket of one or more device buckets.
// Latency of LDS and barriers bounds it (55 stages for 1024 rows); a workgroup's neighbours on its compute unit fill
// the waits.  2^20 two-word f64 terms: a download of 2.6 ms, most of it the host's copies, against 13.4 ms when the
// host sorted.
template <int W, typename T, bool SPLIT>
__global__ void __launch_bounds__(512) k_sort_export(const SortExportArgs<W, T> a, uint32_t padded) {
    extern __shared__ __align__(16) unsigned char sort_lds[];
    uint64_t* const X = reinterpret_cast<uint64_t*>(sort_lds);  // [W][padded]
    uint64_t* const Z = X + (size_t)W * padded;
    T* const C = reinterpret_cast<T*>(Z + (size_t)W * padded);
    uint16_t* const order = reinterpret_cast<uint16_t*>(C + padded);
    uint8_t* const part = reinterpret_cast<uint8_t*>(order + padded);  // SPLIT only
    __shared__ uint32_t first[kSortParts + 1];
    const uint32_t b = blockIdx.x;
    const uint32_t coarse = SPLIT ? a.num_buckets : a.ref_buckets;
    const uint32_t parts = (SPLIT ? a.ref_buckets : a.num_buckets) / coarse;  // at most kSortParts
    const uint32_t tid = threadIdx.x, block = blockDim.x;
    for (uint32_t e = tid; e < parts; e += block) first[e + 1] = (SPLIT ? a.ref_len : a.len)[b + e * coarse];
    __syncthreads();
    if (tid == 0) {
        uint32_t acc = 0;
        first[0] = 0;
        for (uint32_t e = 1; e <= parts; ++e) {
            acc += first[e];
            first[e] = acc;
        }
    }
    __syncthreads();
    const uint32_t n = first[parts];
    if (n == 0 || n > padded) return;  // uniform
    uint32_t size = 2;
    while (size < n) size <<= 1;  // at most padded
    for (uint32_t i = tid; i < size; i += block) order[i] = (uint16_t)i;
    uint32_t e = 0;
    for (uint32_t i = tid; i < n; i += block) {
        uint64_t at = a.start[b] + i;
        if constexpr (!SPLIT) {
            while (first[e + 1] <= i) ++e;
            at = a.start[b + e * coarse] + (i - first[e]);
        }
        const Key<W> k = load_key<W>(a.x, a.z, a.cap, at);
        store_key<W>(X, Z, padded, i, k);
        C[i] = a.c[at];
        if constexpr (SPLIT) part[i] = (uint8_t)ref_part<W, T>(a, k, parts);
    }
    __syncthreads();
    // whether row i comes after row j (rows at or past n come last, in any order among themselves)
    auto after = [&](uint32_t i, uint32_t j) -> bool {
        if (i >= n || j >= n) return i >= n && j < n;
        if constexpr (SPLIT) {
            if (part[i] != part[j]) return part[i] > part[j];
        }
#pragma unroll
        for (int w = 0; w < W; ++w) {
            const uint64_t u = X[(size_t)w * padded + i], v = X[(size_t)w * padded + j];
            if (u != v) return u > v;
        }
#pragma unroll
        for (int w = 0; w < W; ++w) {
            const uint64_t u = Z[(size_t)w * padded + i], v = Z[(size_t)w * padded + j];
            if (u != v) return u > v;
        }
        return false;
    };
    for (uint32_t k = 2; k <= size; k <<= 1) {
        for (uint32_t d = k >> 1; d > 0; d >>= 1) {
            for (uint32_t t = tid; t < size / 2; t += block) {
                const uint32_t i = ((t & ~(d - 1u)) << 1) | (t & (d - 1u));
                const uint32_t j = i | d;
                const uint16_t u = order[i], v = order[j];
                const bool up = (i & k) == 0;
                if (up ? after(u, v) : after(v, u)) {
                    order[i] = v;
                    order[j] = u;
                }
            }
            __syncthreads();
        }
    }
    for (uint32_t i = tid; i < n; i += block) {
        const uint32_t r = order[i];
        uint64_t o = a.ref_start[b];  // out position o + i
        if constexpr (SPLIT) o = a.ref_start[b + part[r] * coarse] - first[part[r]];
        if constexpr (W == 2) {
            reinterpret_cast<ulonglong2*>(a.out_x)[o + i] = make_ulonglong2(X[r], X[padded + r]);
            reinterpret_cast<ulonglong2*>(a.out_z)[o + i] = make_ulonglong2(Z[r], Z[padded + r]);
        } else {
            a.out_x[o + i] = X[r];
            a.out_z[o + i] = Z[r];
        }
        a.out_c[o + i] = C[r];
    }
}

}  // namespace

static_assert(kUploadTerms + kBlock - 1 < 1ull << 32, "the grid's rounding and its thread numbers stay in 32 bits");

template <int W, typename T>
hipError_t launch_upload_count(hipStream_t st, const UploadArgs<W, T>& a) {
    if (a.n == 0) return hipSuccess;
    if (a.n > kUploadTerms) return hipErrorInvalidValue;
    hipLaunchKernelGGL((k_upload_count<W, T>), dim3((a.n + kBlock - 1) / kBlock), dim3(kBlock), 0, st, a);
    return hipGetLastError();
}

template <int W, typename T>
hipError_t launch_upload_rows(hipStream_t st, const UploadArgs<W, T>& a) {
    if (a.n == 0) return hipSuccess;
    if (a.n > kUploadTerms) return hipErrorInvalidValue;
    hipLaunchKernelGGL((k_upload_index<W, T>), dim3((a.n + kBlock - 1) / kBlock), dim3(kBlock), 0, st, a);
    hipLaunchKernelGGL((k_upload_rows<W, T>), dim3(a.num_buckets), dim3(kBlock), 0, st, a);
    return hipGetLastError();
}

template <int W, typename T>
hipError_t launch_ref_counts(hipStream_t st, const SortExportArgs<W, T>& a) {
    if (a.num_buckets == 0) return hipSuccess;
    if (a.ref_buckets < a.num_buckets || a.ref_buckets / a.num_buckets > kSortParts) return hipErrorInvalidValue;
    hipLaunchKernelGGL((k_ref_counts<W, T>), dim3(a.num_buckets), dim3(kBlock), 0, st, a);
    return hipGetLastError();
}

template <int W, typename T>
hipError_t launch_sort_export(hipStream_t st, const SortExportArgs<W, T>& a, uint32_t rows) {
    if (a.ref_buckets == 0 || rows == 0) return hipSuccess;
    const bool split = a.ref_buckets > a.num_buckets;
    if (rows > kSortRows<W> || (split ? a.ref_buckets / a.num_buckets : a.num_buckets / a.ref_buckets) > kSortParts)
        return hipErrorInvalidValue;
    uint32_t padded = 64;
    while (padded < rows) padded <<= 1;
    const size_t lds = (size_t)padded * (2 * W * sizeof(uint64_t) + sizeof(T) + sizeof(uint16_t) + (split ? 1 : 0));
    // a pair of rows per thread and stage up to 512 rows; larger buckets take 512 threads, since their LDS leaves
    // room for fewer workgroups
    const uint32_t block = padded <= 512 ? kBlock : 512;
    if (split)
        hipLaunchKernelGGL((k_sort_export<W, T, true>), dim3(a.num_buckets), dim3(block), lds, st, a, padded);
    else
        hipLaunchKernelGGL((k_sort_export<W, T, false>), dim3(a.ref_buckets), dim3(block), lds, st, a, padded);
    return hipGetLastError();
}

#define PP_TRANSFER_INSTANTIATE(W, T)                                                            \
    template hipError_t launch_upload_count<W, T>(hipStream_t, const UploadArgs<W, T>&);          \
    template hipError_t launch_upload_rows<W, T>(hipStream_t, const UploadArgs<W, T>&);           \
    template hipError_t launch_ref_counts<W, T>(hipStream_t, const SortExportArgs<W, T>&);         \
    template hipError_t launch_sort_export<W, T>(hipStream_t, const SortExportArgs<W, T>&, uint32_t);

PP_TRANSFER_INSTANTIATE(1, double)
PP_TRANSFER_INSTANTIATE(1, float)
PP_TRANSFER_INSTANTIATE(2, double)
PP_TRANSFER_INSTANTIATE(2, float)

}  // namespace pp
