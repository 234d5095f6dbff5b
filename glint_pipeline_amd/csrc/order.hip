// order.hip - a tick's meetings put in the order of their pairs on the
// device: one 64-bit key per meeting, sorted over the bits that ids have
// (rocPRIM, as the key-value flush and the meeting index sort).
#include <hip/hip_runtime.h>

#include <cstring>   // before rocPRIM, whose iterators use memset

#include <rocprim/device/device_radix_sort.hpp>

#include <algorithm>

#include "order.h"

namespace {

constexpr uint32_t kB = 256;

__global__ __launch_bounds__(kB) void k_order_keys(const glint_meeting *m, uint64_t n, uint32_t bits,
                                                   unsigned long long *keys, unsigned long long *vals)
{
    for (uint64_t i = blockIdx.x * (uint64_t)kB + threadIdx.x; i < n; i += (uint64_t)gridDim.x * kB) {
        const glint_meeting e = m[i];
        keys[i] = ((unsigned long long)e.pid_a << bits) | e.pid_b;
        vals[i] = ((unsigned long long)e.start << 32) | e.end;
    }
}

__global__ __launch_bounds__(kB) void k_order_write(glint_meeting *m, uint64_t n, uint32_t bits,
                                                    const unsigned long long *keys, const unsigned long long *vals)
{
    for (uint64_t i = blockIdx.x * (uint64_t)kB + threadIdx.x; i < n; i += (uint64_t)gridDim.x * kB) {
        const unsigned long long k = keys[i], v = vals[i];
        m[i] = glint_meeting{(uint32_t)(k >> bits), (uint32_t)(k & ((1ull << bits) - 1)), (uint32_t)(v >> 32),
                             (uint32_t)v};
    }
}

bool room(OrderWork &w, hipStream_t stream, uint64_t n)
{
    if (n <= w.cap) return true;
    order_free(w);
    const uint64_t cap = std::max<uint64_t>(1 << 16, n + n / 4);
    bool ok = true;
    for (int k = 0; k < 2; k++)
        ok = ok && hipMalloc((void **)&w.keys[k], 8 * cap) == hipSuccess &&
             hipMalloc((void **)&w.vals[k], 8 * cap) == hipSuccess;
    if (ok) {
        rocprim::double_buffer<unsigned long long> keys(w.keys[0], w.keys[1]), vals(w.vals[0], w.vals[1]);
        ok = rocprim::radix_sort_pairs(nullptr, w.tmp_bytes, keys, vals, (size_t)cap, 0, 60, stream) == hipSuccess &&
             hipMalloc(&w.tmp, std::max<size_t>(w.tmp_bytes, 256)) == hipSuccess;
    }
    if (!ok) {
        (void)hipGetLastError();
        order_free(w);
        return false;
    }
    w.cap = cap;
    return true;
}

}  // namespace

bool order_meetings(OrderWork &w, hipStream_t stream, glint_meeting *meetings, uint64_t n, uint32_t id_bits)
{
    if (id_bits > 30 || !room(w, stream, n)) return false;
    const uint32_t grid = (uint32_t)std::min<uint64_t>((n + kB - 1) / kB, 4096);
    rocprim::double_buffer<unsigned long long> keys(w.keys[0], w.keys[1]), vals(w.vals[0], w.vals[1]);
    size_t bytes = 0;
    if (rocprim::radix_sort_pairs(nullptr, bytes, keys, vals, (size_t)n, 0, 2 * id_bits, stream) != hipSuccess ||
        bytes > std::max<size_t>(w.tmp_bytes, 256))
        return false;
    k_order_keys<<<grid, kB, 0, stream>>>(meetings, n, id_bits, keys.current(), vals.current());
    if (rocprim::radix_sort_pairs(w.tmp, bytes, keys, vals, (size_t)n, 0, 2 * id_bits, stream) != hipSuccess)
        return false;
    k_order_write<<<grid, kB, 0, stream>>>(meetings, n, id_bits, keys.current(), vals.current());
    return hipGetLastError() == hipSuccess;
}

void order_free(OrderWork &w)
{
    for (int k = 0; k < 2; k++) {
        if (w.keys[k]) (void)hipFree(w.keys[k]);
        if (w.vals[k]) (void)hipFree(w.vals[k]);
    }
    if (w.tmp) (void)hipFree(w.tmp);
    w = OrderWork{};
}
