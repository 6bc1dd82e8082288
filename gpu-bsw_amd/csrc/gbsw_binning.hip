// gbsw_binning.hip -- device-side length binning of a batch (batched form).
//
// Every pair gets a 15-bit key: its length class (or fine class), longest first (6 bits), then
// 511 - (longer length / 32) (9 bits, capped).  Sorting (key, pair index) yields the
// work order: classes of longer pairs first, inside a class the most rows first
// (longest-processing-time order for the persistent work queues), so the pairs of a
// wave have like column and step counts.  The order of pairs with one key is open: no
// result depends on it.  The reference has no counterpart: it launches pairs in input
// order (driver.cpp:176-185).
#include <algorithm>

#include <hip/hip_runtime.h>
#include <hipcub/hipcub.hpp>
#include <stdint.h>

#include "gbsw_kernels.hpp"

namespace gbsw {

__device__ __forceinline__ uint32_t sort_key(const PrepareArgs& a, int64_t p)
{
    const uint32_t la = (uint32_t)(a.ref_off[p + 1] - a.ref_off[p]);
    const uint32_t lb = (uint32_t)(a.qry_off[p + 1] - a.qry_off[p]);
    const uint32_t m = la < lb ? la : lb, M = la < lb ? lb : la;
    const uint32_t c = (uint32_t)(a.fine ? kFineClasses - 1 - fine_class((int)m) : kClasses - 1 - length_class((int)m));
    const uint32_t top = (1u << kRowBits) - 1u, r = M >> 5;
    return (c << kRowBits) | (top - (r < top ? r : top));
}

// Everything a job needs on the device before its kernels, in one launch: the small
// tables (read from pinned host memory), cleared status words, queues and split
// bookkeeping by the first `helpers` workgroups; and by the rest
//  - SMALL, up to kSmallSort pairs: the whole counting sort in one workgroup.  A
//    counter of 16 bits per key in LDS (51 KB); an atomic add gives a pair its rank
//    among those of its key, a scan of the counters every key's first place.
//  - otherwise the keys and pair indices for the radix sort, as far as there are pairs.
// Bound by latency.  Three copies, three clears, the keys and five sort kernels did this
// before, with launch gaps of 3 to 8 us between them: 82 us from the first to the
// alignment's start for 10,000 pairs (graph replay).  As one launch it took 37 us off a
// batch of 10,000 short reads (437 us) and 84 off a call of one read (399 us).
constexpr int kBins = kClasses << kRowBits;
constexpr int kSmallThreads = 1024, kSmallEach = kSmallSort / kSmallThreads;
constexpr int kScanEach = (kBins / 2 + kSmallThreads - 1) / kSmallThreads; // dwords (two counters) per thread
static_assert((kScanEach & 1) == 1, "an odd stride is free of bank conflicts");
static_assert(kSmallSort <= 32767, "ranks and places are 16-bit");

template <bool SMALL>
__global__ __launch_bounds__(SMALL ? kSmallThreads : 256) void k_prepare(PrepareArgs a)
{
    constexpr int T = SMALL ? kSmallThreads : 256;
    const int tid = threadIdx.x, b = blockIdx.x;
    if (b < a.helpers) {
        const int64_t step = (int64_t)a.helpers * T;
        for (int64_t x = (int64_t)b * T + tid; x < a.nsplit; x += step) a.split[x] = 0;
        if (b > 0) return;
        for (int x = tid; x < a.nsub; x += T) a.sub[x] = a.h_sub[x];
        for (int x = tid; x < 256; x += T) a.lut[x] = a.h_lut[x];
        for (int x = tid; x < a.alpha; x += T) a.colmax[x] = a.h_colmax[x];
        for (int x = tid; x < a.nstatus; x += T) a.status[x] = 0;
        for (int x = tid; x < a.nqueue; x += T) a.queue[x] = 0;
        return;
    }
    if constexpr (!SMALL) {
        const int64_t p = (int64_t)(b - a.helpers) * T + tid;
        if (p >= a.n) return;
        a.keys[p] = sort_key(a, p);
        a.vals[p] = (int32_t)p;
    } else {
        __shared__ uint32_t count[kScanEach * kSmallThreads];
        __shared__ uint32_t wave_sum[kSmallThreads / 64];
        for (int x = tid; x < kScanEach * kSmallThreads; x += T) count[x] = 0;
        __syncthreads();
        const int n = (int)a.n;
        uint32_t key[kSmallEach]; // key, then rank << 16
#pragma unroll
        for (int e = 0; e < kSmallEach; ++e)
            if (e * T + tid < n) key[e] = sort_key(a, e * T + tid);
#pragma unroll
        for (int e = 0; e < kSmallEach; ++e)
            if (e * T + tid < n) {
                const int sh = 16 * (int)(key[e] & 1u);
                const uint32_t old = atomicAdd(&count[key[e] >> 1], 1u << sh);
                key[e] |= ((old >> sh) & 0xFFFFu) << 16;
            }
        __syncthreads();
        // exclusive sums over the counters
        uint32_t mine = 0;
#pragma unroll
        for (int x = 0; x < kScanEach; ++x) {
            const uint32_t w = count[tid * kScanEach + x];
            mine += (w & 0xFFFFu) + (w >> 16);
        }
        uint32_t upto = mine;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const uint32_t v = (uint32_t)__shfl_up((int)upto, o);
            if ((tid & 63) >= o) upto += v;
        }
        if ((tid & 63) == 63) wave_sum[tid >> 6] = upto;
        __syncthreads();
        uint32_t at = upto - mine;
        for (int w = 0; w < (tid >> 6); ++w) at += wave_sum[w];
#pragma unroll
        for (int x = 0; x < kScanEach; ++x) {
            const uint32_t w = count[tid * kScanEach + x];
            count[tid * kScanEach + x] = at | (at + (w & 0xFFFFu)) << 16;
            at += (w & 0xFFFFu) + (w >> 16);
        }
        __syncthreads();
#pragma unroll
        for (int e = 0; e < kSmallEach; ++e)
            if (e * T + tid < n) {
                const uint32_t k = key[e] & 0xFFFFu;
                a.order[((count[k >> 1] >> (16 * (k & 1u))) & 0xFFFFu) + (key[e] >> 16)] = e * T + tid;
            }
    }
}

// Which byte values occur in the two buffers (16-byte aligned): bit b of word b / 32 of
// the workgroup's mask, in pinned host memory (no clearing before and no copy after).
// A flag per value in LDS, set by plain stores: lanes with one value write one address.
// (127 MB: 40 us; with a 256-bit mask per thread, set without indexing, it took 24
// instructions a byte and 100 us on twice the workgroups.)
__global__ __launch_bounds__(1024) void k_byte_presence(const uint8_t* p, uint64_t n, const uint8_t* p2, uint64_t n2,
                                                        uint32_t* masks)
{
    __shared__ uint32_t has[256];
    if (threadIdx.x < 256) has[threadIdx.x] = 0;
    __syncthreads();
    const uint64_t each = (uint64_t)blockDim.x * 16, stride = gridDim.x * each * 4;
    auto add = [&](const uint4& v) {
        const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
            for (int k = 0; k < 4; ++k) has[(w[q] >> (8 * k)) & 0xFFu] = 1;
    };
    auto scan = [&](const uint8_t* s, uint64_t len) {
        for (uint64_t i = blockIdx.x * each * 4 + threadIdx.x * 16; i < len; i += stride) {
            if (i + 3 * each + 16 <= len) {
                uint4 v[4];
#pragma unroll
                for (int k = 0; k < 4; ++k) v[k] = *(const uint4*)(s + i + k * each);
#pragma unroll
                for (int k = 0; k < 4; ++k) add(v[k]);
            } else {
                for (int k = 0; k < 4; ++k) {
                    const uint64_t at = i + k * each;
                    if (at + 16 <= len) add(*(const uint4*)(s + at));
                    else
                        for (uint64_t j = at; j < len; ++j) has[s[j]] = 1;
                }
            }
        }
    };
    scan(p, n);
    scan(p2, n2);
    __syncthreads();
    if (threadIdx.x < 256) {
        const uint64_t set = __ballot(has[threadIdx.x] != 0);
        if ((threadIdx.x & 31) == 0) masks[8 * blockIdx.x + threadIdx.x / 32] = (uint32_t)(set >> (threadIdx.x & 32));
    }
}

hipError_t byte_presence(const uint8_t* p, uint64_t n, const uint8_t* p2, uint64_t n2, uint32_t* masks,
                         hipStream_t stream)
{
    const unsigned blocks =
        (unsigned)std::max<uint64_t>(1, std::min<uint64_t>(kPresenceBlocks, (std::max(n, n2) + 65535) / 65536));
    hipLaunchKernelGGL(k_byte_presence, dim3(blocks), dim3(1024), 0, stream, p, n, p2, n2, masks);
    return hipGetLastError();
}

hipError_t prepare_job(const PrepareArgs& args, hipStream_t stream)
{
    PrepareArgs a = args;
    a.helpers = (int32_t)std::max<int64_t>(1, std::min<int64_t>(64, a.nsplit / 8192));
    if (a.order)
        hipLaunchKernelGGL(k_prepare<true>, dim3((unsigned)a.helpers + 1), dim3(kSmallThreads), 0, stream, a);
    else
        hipLaunchKernelGGL(k_prepare<false>, dim3((unsigned)(a.helpers + (a.keys ? (a.n + 255) / 256 : 0))), dim3(256), 0,
                           stream, a);
    return hipGetLastError();
}

// Stable LSD radix sort of (key, value) on bits [0, end_bit).  With temp == nullptr
// only the scratch size is returned in temp_bytes.
hipError_t sort_pairs(void* temp, size_t& temp_bytes, const uint32_t* kin, uint32_t* kout, const int32_t* vin,
                      int32_t* vout, int n, int end_bit, hipStream_t stream)
{
    return hipcub::DeviceRadixSort::SortPairs(temp, temp_bytes, kin, kout, vin, vout, n, 0, end_bit, stream);
}

} // namespace gbsw
