// fa_prim.hip -- scan and sort primitives used to turn per-query counts into
// NeighborList offsets and to order cluster labels: the library's own scan for
// up to four million counts, rocPRIM device algorithms beyond and for sorting.
#include <algorithm>
#include <cstring>

#include <rocprim/rocprim.hpp>

#include "fa_common.h"

namespace fa {

namespace {
struct widen
{
    __device__ __host__ uint64_t operator()(uint32_t v) const { return v; }
};

// ------------------------------------------------------------------ scan of up to kOwnScan counts
// Small and ordinary scans are bound by launches, not bytes: rocPRIM's scan is
// two, the 64-bit total two more, and clearing out[0] and copying the total to
// the host are three further commands.  Here each of up to kScanBlocks
// workgroups owns one contiguous part: scan_sums_kernel adds up the parts, and
// scan_parts_kernel scans its own part from the sum of the parts before it and
// writes the total (and up to two further words) to pinned host memory itself.
// Up to kScanSingle counts take the second kernel alone.  The input is read
// twice, so above kOwnScan (16 MiB) rocPRIM's single pass is the better one.
// No state outlives a call and nothing is cleared, so both can be captured.
// Offsets wrap at 32 bits, totals are summed in 64: callers refuse a list by
// its total before anything is sized from it.
// 250,000 points (a kNN list and its grid): nine commands fewer, 148 -> 138 us for the query and psi_6.
constexpr uint32_t kScanThreads = 512;
constexpr uint32_t kScanTile = kScanThreads * 8;
constexpr uint32_t kScanSingle = 2 * kScanTile;
constexpr uint32_t kScanBlocks = 512;
constexpr uint32_t kOwnScan = 1u << 22;

struct ScanParts
{
    uint32_t part, blocks; // counts per workgroup (a multiple of kScanTile), workgroups
};
ScanParts scan_parts(uint32_t n)
{
    ScanParts p;
    uint32_t const tiles = (n + kScanTile - 1) / kScanTile;
    p.part = n <= kScanSingle ? kScanSingle : (tiles + kScanBlocks - 1) / kScanBlocks * kScanTile;
    p.blocks = std::max(1u, (n + p.part - 1) / p.part);
    return p;
}

// sum of v over the workgroup, in every thread (s: kScanThreads / 64 words)
__device__ inline uint64_t block_sum(uint64_t v, uint64_t* s)
{
#pragma unroll
    for (int d = 32; d > 0; d >>= 1)
        v += __shfl_xor(static_cast<unsigned long long>(v), d);
    __syncthreads();
    if ((threadIdx.x & 63u) == 0)
        s[threadIdx.x >> 6] = v;
    __syncthreads();
    uint64_t r = 0;
#pragma unroll
    for (uint32_t w = 0; w < kScanThreads / 64; ++w)
        r += s[w];
    return r;
}

__global__ __launch_bounds__(kScanThreads) void scan_sums_kernel(const uint32_t* __restrict__ in, uint32_t n,
                                                                 uint32_t part, uint64_t* __restrict__ sums)
{
    __shared__ uint64_t s[kScanThreads / 64];
    uint32_t const beg = blockIdx.x * part, end = min(n - beg, part) + beg;
    uint64_t v = 0;
    for (uint32_t t = beg + threadIdx.x; t < end; t += kScanThreads)
        v += in[t];
    v = block_sum(v, s);
    if (threadIdx.x == 0)
        sums[blockIdx.x] = v;
}

// out[t] = sum of in[0 .. t), out[n] = the total; segments (nullable): out[t]
// where in[t] != 0, else 0.  host (nullable): the 64-bit total, then n_extra
// words of extra.
__global__ __launch_bounds__(kScanThreads) void scan_parts_kernel(const uint32_t* __restrict__ in, uint32_t n,
                                                                  uint32_t part, const uint64_t* __restrict__ sums,
                                                                  uint32_t* __restrict__ out,
                                                                  uint32_t* __restrict__ segments,
                                                                  uint64_t* __restrict__ host,
                                                                  const uint32_t* __restrict__ extra, int n_extra)
{
    __shared__ uint64_t s[kScanThreads / 64];
    __shared__ uint32_t s_wave[kScanThreads / 64];
    uint32_t const tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
    uint64_t first = 0, own = 0; // sum of the parts before this one; this thread's counts
    if (blockIdx.x)
    {
        for (uint32_t t = tid; t < blockIdx.x; t += kScanThreads)
            first += sums[t];
        first = block_sum(first, s);
    }
    uint32_t before = uint32_t(first); // offsets are 32 bits wide, the total is not
    uint32_t const beg = blockIdx.x * part, end = min(n - beg, part) + beg;
    for (uint32_t t0 = beg; t0 < end; t0 += kScanTile)
    {
        uint32_t const i0 = t0 + tid * 8;
        uint32_t v[8], sum = 0;
#pragma unroll
        for (uint32_t k = 0; k < 8; ++k)
        {
            v[k] = i0 + k < end ? in[i0 + k] : 0u;
            sum += v[k];
            own += v[k];
        }
        uint32_t incl = sum;
#pragma unroll
        for (int d = 1; d < 64; d <<= 1)
        {
            uint32_t const y = __shfl_up(incl, d);
            if (lane >= uint32_t(d))
                incl += y;
        }
        __syncthreads(); // the previous tile's s_wave has been read
        if (lane == 63u)
            s_wave[wave] = incl;
        __syncthreads();
        uint32_t base = 0, tile = 0;
#pragma unroll
        for (uint32_t w = 0; w < kScanThreads / 64; ++w)
        {
            base += w < wave ? s_wave[w] : 0u;
            tile += s_wave[w];
        }
        uint32_t x = before + base + (incl - sum);
#pragma unroll
        for (uint32_t k = 0; k < 8; ++k)
        {
            if (i0 + k < end)
            {
                out[i0 + k] = x;
                if (segments)
                    segments[i0 + k] = v[k] ? x : 0u;
            }
            x += v[k];
        }
        before += tile;
    }
    if (end != n) // the last part only from here on
        return;
    if (tid == 0)
        out[n] = before;
    if (!host)
        return;
    uint64_t const total = first + block_sum(own, s);
    if (tid == 0)
    {
        __hip_atomic_store(host, total, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        for (int k = 0; k < n_extra; ++k)
            __hip_atomic_store(reinterpret_cast<uint32_t*>(host + 1) + k, extra[k], __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_SYSTEM);
    }
}

// segments of a scanned list (lists beyond kOwnScan)
__global__ void scan_segments_kernel(const uint32_t* __restrict__ in, const uint32_t* __restrict__ out, uint32_t n,
                                     uint32_t* __restrict__ segments)
{
    uint32_t const t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t < n)
        segments[t] = in[t] ? out[t] : 0u;
}

// n > 0; sums: kScanBlocks words of device scratch
int own_scan(const uint32_t* d_in, uint32_t* d_out, uint32_t n, uint32_t* d_segments, uint64_t* host,
             const uint32_t* d_extra, int n_extra, uint64_t* sums)
{
    hipStream_t s = stream();
    ScanParts const p = scan_parts(n);
    if (p.blocks > 1)
        FA_KLAUNCH(scan_sums_kernel, dim3(p.blocks), dim3(kScanThreads), 0, s, d_in, n, p.part, sums);
    FA_KLAUNCH(scan_parts_kernel, dim3(p.blocks), dim3(kScanThreads), 0, s, d_in, n, p.part, sums, d_out, d_segments,
               host, d_extra, n_extra);
    FA_HIP(hipGetLastError());
    return FA_OK;
}
} // namespace

int exclusive_scan_u32(const uint32_t* d_in, uint32_t* d_out, uint32_t n, uint64_t* total, const uint32_t* d_extra,
                       uint32_t* h_extra, int n_extra, uint32_t* d_segments)
{
    int const extras = d_extra ? std::min(std::max(n_extra, 1), 2) : 0;
    size_t const extra_bytes = sizeof(uint32_t) * size_t(extras);
    hipStream_t s = stream();
    // Totals come back through pinned host memory; one synchronisation covers them.
    void* stage = nullptr;
    if (total || d_extra)
        if (int rc = readback_stage(2 * sizeof(uint64_t), &stage))
            return rc;
    uint64_t* h_stage = static_cast<uint64_t*>(stage);
    if (n > 0 && n <= kOwnScan)
    {
        void* sums = nullptr;
        if (int rc = scratch(0, sizeof(uint64_t) * kScanBlocks, &sums))
            return rc;
        if (int rc = own_scan(d_in, d_out, n, d_segments, h_stage, d_extra, extras, static_cast<uint64_t*>(sums)))
            return rc;
    }
    else
    {
        FA_HIP(hipMemsetAsync(d_out, 0, sizeof(uint32_t), s));
        if (h_stage)
            h_stage[0] = 0;
        if (n)
        {
            size_t bytes_scan = 0, bytes_red = 0;
            FA_HIP(rocprim::inclusive_scan(nullptr, bytes_scan, d_in, d_out + 1, size_t(n), rocprim::plus<uint32_t>(),
                                           s));
            auto it = rocprim::make_transform_iterator(d_in, widen());
            uint64_t* d_total = nullptr;
            FA_HIP(rocprim::reduce(nullptr, bytes_red, it, d_total, uint64_t(0), size_t(n), rocprim::plus<uint64_t>(),
                                   s));
            void* tmp = nullptr;
            if (int rc = scratch(0, bytes_scan + bytes_red + 512, &tmp))
                return rc;
            char* base = static_cast<char*>(tmp);
            d_total = reinterpret_cast<uint64_t*>(base);
            void* t_scan = base + 256;
            void* t_red = base + 256 + ((bytes_scan + 255) / 256) * 256;
            FA_HIP(rocprim::inclusive_scan(t_scan, bytes_scan, d_in, d_out + 1, size_t(n), rocprim::plus<uint32_t>(),
                                           s));
            if (d_segments)
                FA_KLAUNCH(scan_segments_kernel, dim3((n + 255) / 256), dim3(256), 0, s, d_in, d_out, n, d_segments);
            if (total)
            {
                FA_HIP(rocprim::reduce(t_red, bytes_red, it, d_total, uint64_t(0), size_t(n),
                                       rocprim::plus<uint64_t>(), s));
                FA_HIP(hipMemcpyAsync(h_stage, d_total, sizeof(uint64_t), hipMemcpyDeviceToHost, s));
            }
        }
        if (d_extra)
            FA_HIP(hipMemcpyAsync(h_stage + 1, d_extra, extra_bytes, hipMemcpyDeviceToHost, s));
    }
    if (!total && !d_extra)
        return FA_OK;
    FA_HIP(hipStreamSynchronize(s));
    if (total)
        *total = h_stage[0];
    if (d_extra)
        std::memcpy(h_extra, h_stage + 1, extra_bytes);
    return FA_OK;
}

namespace {
__global__ void zero_u32_kernel(uint32_t* __restrict__ d, uint64_t n)
{
    for (uint64_t t = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x; t < n; t += uint64_t(gridDim.x) * blockDim.x)
        d[t] = 0u;
}
} // namespace

int zero_u32(uint32_t* d, uint64_t n)
{
    if (n == 0)
        return FA_OK;
    uint64_t const blocks = std::min<uint64_t>((n + 255) / 256, 4096);
    FA_KLAUNCH(zero_u32_kernel, dim3(unsigned(blocks)), dim3(256), 0, stream(), d, n);
    FA_HIP(hipGetLastError());
    return FA_OK;
}

size_t scan_tmp_bytes(uint32_t n)
{
    size_t bytes = 0;
    if (n <= kOwnScan)
        return sizeof(uint64_t) * kScanBlocks + 256;
    uint32_t* dummy = nullptr;
    if (rocprim::inclusive_scan(nullptr, bytes, dummy, dummy, size_t(n), rocprim::plus<uint32_t>(), stream()) !=
        hipSuccess)
        return 0;
    return bytes + 256;
}

int exclusive_scan_u32_async(const uint32_t* d_in, uint32_t* d_out, uint32_t n, void* tmp, size_t tmp_bytes)
{
    if (n && n <= kOwnScan)
    {
        if (tmp_bytes < sizeof(uint64_t) * kScanBlocks)
            return fail(FA_ERR_RUNTIME, "scan storage too small");
        return own_scan(d_in, d_out, n, nullptr, nullptr, nullptr, 0, static_cast<uint64_t*>(tmp));
    }
    if (int rc = zero_u32(d_out, 1))
        return rc;
    if (n == 0)
        return FA_OK;
    size_t bytes = tmp_bytes;
    FA_HIP(rocprim::inclusive_scan(tmp, bytes, d_in, d_out + 1, size_t(n), rocprim::plus<uint32_t>(), stream()));
    return FA_OK;
}

int sort_u64(uint64_t* d_keys, uint32_t n)
{
    if (n < 2)
        return FA_OK;
    hipStream_t s = stream();
    size_t bytes = 0;
    FA_HIP(rocprim::radix_sort_keys(nullptr, bytes, d_keys, d_keys, size_t(n), 0, 64, s));
    void* tmp = nullptr;
    size_t const kb = size_t(n) * sizeof(uint64_t);
    if (int rc = scratch(1, bytes + kb + 256, &tmp))
        return rc;
    uint64_t* alt = reinterpret_cast<uint64_t*>(static_cast<char*>(tmp));
    void* t = static_cast<char*>(tmp) + ((kb + 255) / 256) * 256;
    FA_HIP(rocprim::radix_sort_keys(t, bytes, d_keys, alt, size_t(n), 0, 64, s));
    FA_HIP(hipMemcpyAsync(d_keys, alt, kb, hipMemcpyDeviceToDevice, s));
    return FA_OK;
}

} // namespace fa
