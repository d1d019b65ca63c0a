// hb_schedule.h -- host rules of the union's schedule that need no device.
#pragma once

#include <algorithm>
#include <cstdint>

namespace hb {

// Precisions above 10: a wavefront reads a row of 4 KiB in about 0.7 us, so a hub of 10,000
// neighbours alone would take as long as the rest of the iteration.  Lists of more than
// `len` arcs are cut into tasks of `len`, each with a partial row of 2^p bytes of its own.
constexpr uint32_t kWideHub = 256;

// the tasks of a CSR's lists of more than `len` arcs
inline uint64_t wide_tasks(const uint32_t *off, uint32_t n, uint64_t len)
{
    uint64_t tasks = 0;
    for (uint32_t u = 0; u < n; ++u) {
        const uint64_t d = off[u + 1] - off[u];
        if (d > len) tasks += (d + len - 1) / len;
    }
    return tasks;
}

// Task length: kWideHub, doubled until the partial rows take no more than the two register
// buffers (or 1 GiB, for small graphs).  Without the bound they grow with the arcs: 65,536 nodes
// of 10,000 arcs at p = 16 would need 168 GB beside 17 GB of registers.  Longer tasks cost up to a
// sixth where they read few bytes each (8,192 nodes of 2,000 arcs at p = 14: 30.0 ms a run with
// tasks of 1,024, 25.9 with 256; 2,048 of 2,047 at p = 16: 16.9 and 19.3).
inline uint64_t wide_task_len(const uint32_t *off, uint32_t n, int p)
{
    const uint64_t most = std::max((uint64_t)n << (p + 1), (uint64_t)1 << 30) >> p;
    uint64_t len = kWideHub;
    while (wide_tasks(off, n, len) > most) len *= 2;
    return len;
}

}  // namespace hb
