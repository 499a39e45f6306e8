// Rows [B,H,N] of narrow heads to rows filled up with zeros and back (the mixer's matrix-core kernels take head dims of 16, 32 and 64; the
// default models have 8).  Up to four arrays in one launch, each at strides of its own, so that k and v, or dk and dv, are one launch.
// Bound by its bytes.  torch fills the padded array and then copies into it element by element: mixer of 8 heads of 8, bf16,
// M=128: forward at N=200,000 146 -> 120 us, forward + backward under a mask at B=4, N=50,000 497 -> 412 us, at N=3000 310 -> 192 us (a
// dozen launches fewer).
#include <algorithm>

#include "common.hpp"

namespace flare {

namespace {

// One thread: one unit (16, 8, 4 or 2 bytes) of a destination row.  Rows are walked in the destination's memory order (the launcher
// sorts the three axes), source and destination then mostly share it.
// I: an unsigned type that holds the number of units (three 64-bit divisions a unit would cost more than its bytes).
template <typename U, typename I>
__global__ __launch_bounds__(256) void pad_rows_kernel(PadRowsArgs a)
{
    const PadRowsJob j = a.job[blockIdx.y];
    const I n1 = (I)a.n[1], n2 = (I)a.n[2], units = (I)a.dst_units, total = (I)a.n[0] * n1 * n2 * units;
    for (I i = (I)blockIdx.x * 256 + threadIdx.x; i < total; i += (I)gridDim.x * 256) {
        const I row = i / units, u = i - row * units, r2 = row / n2;
        const int64_t i2 = (int64_t)(row - r2 * n2), i0 = (int64_t)(r2 / n1), i1 = (int64_t)(r2 - (I)i0 * n1);
        U v{};
        if (u < (I)a.src_units) v = reinterpret_cast<const U*>(j.src + (i0 * j.ss[0] + i1 * j.ss[1] + i2 * j.ss[2]))[u];
        reinterpret_cast<U*>(j.dst + (i0 * j.ds[0] + i1 * j.ds[1] + i2 * j.ds[2]))[u] = v;
    }
}

}  // namespace

// widths and strides in bytes; the axes of every job in the same order
hipError_t launch_pad_rows(PadRowsArgs a, int64_t src_bytes, int64_t dst_bytes, hipStream_t st)
{
    // slowest axis of the first destination first
    for (int x = 0; x < 2; ++x)
        for (int y = 0; y + 1 < 3; ++y)
            if (a.job[0].ds[y] < a.job[0].ds[y + 1]) {
                std::swap(a.n[y], a.n[y + 1]);
                for (int k = 0; k < a.jobs; ++k) {
                    std::swap(a.job[k].ss[y], a.job[k].ss[y + 1]);
                    std::swap(a.job[k].ds[y], a.job[k].ds[y + 1]);
                }
            }
    uint64_t all = (uint64_t)src_bytes | (uint64_t)dst_bytes;
    for (int k = 0; k < a.jobs; ++k) {
        all |= reinterpret_cast<uintptr_t>(a.job[k].src) | reinterpret_cast<uintptr_t>(a.job[k].dst);
        for (int x = 0; x < 3; ++x)
            if (a.n[x] > 1) all |= (uint64_t)a.job[k].ss[x] | (uint64_t)a.job[k].ds[x];
    }
    const int unit = all % 16 == 0 ? 16 : all % 8 == 0 ? 8 : all % 4 == 0 ? 4 : 2;
    a.src_units = (int)(std::min(src_bytes, dst_bytes) / unit);
    a.dst_units = (int)(dst_bytes / unit);
    const int64_t total = a.n[0] * a.n[1] * a.n[2] * a.dst_units;
    const dim3 grid((unsigned)std::min<int64_t>((total + 255) / 256, 32 * (int64_t)device_cus()), (unsigned)a.jobs);
    const auto go = [&](auto u) {
        using U = decltype(u);
        if (total < (int64_t)1 << 31) hipLaunchKernelGGL((pad_rows_kernel<U, uint32_t>), grid, dim3(256), 0, st, a);
        else                          hipLaunchKernelGGL((pad_rows_kernel<U, uint64_t>), grid, dim3(256), 0, st, a);
    };
    switch (unit) {
        case 16: go(uint4{}); break;
        case 8:  go(uint2{}); break;
        case 4:  go(uint32_t{}); break;
        default: go(uint16_t{}); break;
    }
    return hipGetLastError();
}

}  // namespace flare
