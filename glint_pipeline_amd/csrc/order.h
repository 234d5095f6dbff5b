// order.h - a tick's meetings put in the order of their pairs on the device.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>

#include "glint.h"

// Buffers of the sort, kept by a context between ticks and grown when a tick
// has more meetings than any before.
struct OrderWork {
    unsigned long long *keys[2] = {nullptr, nullptr}, *vals[2] = {nullptr, nullptr};
    void *tmp = nullptr;
    size_t tmp_bytes = 0;
    uint64_t cap = 0;
};

// Sorts the n meetings (distinct pairs of ids below 2^id_bits, id_bits <= 30)
// in place by (pid_a, pid_b), on the stream.  False if that could not be
// enqueued (no memory for the buffers, say): the meetings are as they were.
bool order_meetings(OrderWork &w, hipStream_t stream, glint_meeting *meetings, uint64_t n, uint32_t id_bits);
void order_free(OrderWork &w);
