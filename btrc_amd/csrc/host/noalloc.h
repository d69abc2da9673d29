// Sizes of btrc_hip_trace_closest_noalloc's scratch: the batch's ray counters,
// then the traversal's stack entries beyond the LDS part, [entry][lane].
#pragma once

#include <algorithm>
#include <cstddef>
#include <cstdint>

namespace btrc {

// 64 MiB holds the entries of 16 wavefronts per CU for a tree that needs 43 (a
// million triangles); 8 MiB held 2 (1M incoherent rays: 2.27 ms, now 0.44).
constexpr size_t NOALLOC_SCRATCH_BYTES = (size_t)64 << 20;
constexpr size_t NOALLOC_COUNTER_BYTES = 2048;
// Trees with more stack entries are refused, whatever the scratch could hold:
// the entry point's limit since its scratch was 8 MiB and one wavefront of 64
// lanes kept 16 of its 8-byte entries per lane in LDS.
constexpr int64_t NOALLOC_STACK_MAX = 16 + (((size_t)8 << 20) - NOALLOC_COUNTER_BYTES) / (64 * 8);

// bytes of one wavefront's entries; short_stack: entries in LDS
inline size_t noalloc_wave_bytes(int32_t stack, int32_t short_stack)
{
    return (size_t)std::max(0, stack - short_stack) * 64 * 8;
}

// wavefronts of a persistent grid of `grid` whose entries fit; 0: refused
inline int32_t noalloc_waves(int32_t stack, int32_t short_stack, int32_t grid)
{
    if(stack > NOALLOC_STACK_MAX)
        return 0;
    const size_t wave = noalloc_wave_bytes(stack, short_stack), room = NOALLOC_SCRATCH_BYTES - NOALLOC_COUNTER_BYTES;
    return wave == 0 ? grid : (int32_t)std::min<size_t>((size_t)grid, room / wave);
}

} // namespace btrc
