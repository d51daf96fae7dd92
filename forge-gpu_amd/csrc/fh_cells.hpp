// fh_cells.hpp -- per-cell entries straight from sorted keys, no scan and no clear: what the slots of
// the sorted keys and the empty cells between their runs write (cell_start of HashGrid::build and
// of the SPH rebuild, cell_start / cell_end of find_cell_boundaries).
#pragma once

#include "fh_internal.hpp"

namespace fh {

// CSR: the key in slot s starts its run when the key before it, pk, differs; slot s then owns
// cell_start[c] = s for the cells pk < c <= k (the empty cells before its own take its index: the
// first sorted index with key >= c), and the last slot also owns the cells after its key up to and
// including C, which take n.  These ranges partition 0..C, so every entry is written once; together
// they are the prefix sum of the per-cell counts of hashgrid.rs:102-106.  (find_cell_boundaries: the
// ranges are the empty cells pk < c < k, which take the sentinels.)
//
// A slot's wave writes its ranges except the blocks of kCellBlock cells (aligned, the last one
// ending at the last entry) that lie wholly inside one range: those are empty cells between two
// runs, and lanes of fill_empty_blocks write them.  Left to the slot, a long gap is one wave's
// serial store loop: a dam-break block of 1,048,576 particles in the lower part of 100^3 cells
// leaves ~680,000 cells behind its last key, and k_gather_resident took 312 us with them against
// 14 us now (k_cell_starts 304 -> 6 us).  What a slot keeps of a gap is at most two partial blocks.
constexpr uint32_t kCellBlock = 256;

// put(c, val) for the cells [lo, hi) (none if hi <= lo): short ranges by their lane, longer ones by
// the whole wave, which steps through offsets: a cell number near 2^32 would wrap around.
template <class Put>
__device__ __forceinline__ void fill_range(uint32_t lo, uint32_t hi, uint32_t val, int lane,
                                           Put&& put) {
    const uint32_t len = hi > lo ? hi - lo : 0u;
    const bool mine = len <= 8u;
    if (mine)
        for (uint32_t o = 0; o < len; o++) put(lo + o, val);
    uint64_t wide = __ballot(!mine);
    while (wide) {  // uniform
        const int l = __ffsll((unsigned long long)wide) - 1;
        wide &= wide - 1ull;
        const uint32_t wlo = (uint32_t)__shfl((int)lo, l, kWave);
        const uint32_t wlen = (uint32_t)__shfl((int)len, l, kWave);
        const uint32_t wv = (uint32_t)__shfl((int)val, l, kWave);
        // (wlen < 2 * kCellBlock: fill_cells leaves the whole blocks out)
        for (uint32_t o = (uint32_t)lane; o < wlen; o += kWave) put(wlo + o, wv);
    }
}
// The same without the whole blocks inside, of `entries` cells in all.
template <class Put>
__device__ __forceinline__ void fill_cells(uint32_t lo, uint32_t hi, uint32_t entries, uint32_t val,
                                           int lane, Put&& put) {
    const uint32_t first = (lo + kCellBlock - 1u) & ~(kCellBlock - 1u);  // may wrap past 2^32
    const uint32_t end = hi == entries ? hi : hi & ~(kCellBlock - 1u);
    const bool cut = first >= lo && first < end;  // whole blocks [first, end) are not ours
    fill_range(lo, cut ? first : hi, val, lane, put);
    if (__ballot(cut && end < hi) != 0ull) fill_range(cut ? end : hi, hi, val, lane, put);
}

// Blocks of kCellBlock cells, 16 lanes each: a block is written when it lies inside one slot's
// range (the rule fill_cells skips by): no key falls in it, or (LAST: a range includes its own
// slot's key) none before its last cell.  The
// first slot whose key is >= the block's first cell is searched with 16 probes per round: six
// dependent rounds for 4,194,304 keys, a third of the loads that 64 probes take in four.  These
// workgroups come first in the launch, so that the rounds overlap the slots' work (a grid with no
// long gap pays 0.8 us: 551,368 cells of 4,194,304 uniform points, k_csr_from_sorted 8.7 -> 9.5).
constexpr uint32_t kBlockLanes = 16, kGroupBlocks16 = 256 / kBlockLanes;
template <bool LAST, class Put>
__device__ __forceinline__ void fill_empty_blocks(uint32_t group, const uint32_t* __restrict__ keys,
                                                  uint32_t n, uint32_t entries, Put&& put) {
    const uint32_t b = group * kGroupBlocks16 + threadIdx.x / kBlockLanes;
    const uint32_t t = threadIdx.x % kBlockLanes, shift = (threadIdx.x & 63u) & ~(kBlockLanes - 1u);
    const bool live = b <= (entries - 1u) / kCellBlock;
    const uint32_t c0 = live ? b * kCellBlock : 0u;
    const uint32_t last = min(c0 + (kCellBlock - 1u), entries - 1u);
    uint32_t lo = 0, hi = live ? n : 0u;
    while (__ballot(lo < hi) != 0ull) {  // until every block of the wave has its slot
        const uint32_t step = (hi - lo + kBlockLanes - 1u) / kBlockLanes;
        const uint32_t i = lo + t * step;
        const bool less = i < hi && keys[min(i, n - 1u)] < c0;
        const uint32_t below =
            (uint32_t)__popcll((__ballot(less) >> shift) & ((1ull << kBlockLanes) - 1ull));
        hi = below ? min(hi, lo + below * step) : lo;
        lo += below ? (below - 1u) * step + 1u : 0u;
    }
    if (!live || (lo < n && (LAST ? keys[lo] < last : keys[lo] <= last))) return;
    for (uint32_t c = t; c <= last - c0; c += kBlockLanes) put(c0 + c, lo);
}
// Workgroups (256 threads) for the blocks of `entries` >= 1 cells.
inline uint32_t empty_block_groups(uint32_t entries) {
    return (entries - 1u) / (kGroupBlocks16 * kCellBlock) + 1u;
}

// launch(groups, fill_groups): the blocks of `entries` cells and the slots of n keys in one launch,
// or, where that would be 2^32 threads or more, in one each (more keys than one launch takes: refused).
template <class Launch>
hipError_t launch_cell_groups(uint32_t n, uint32_t entries, Launch&& launch) {
    constexpr uint32_t kMaxGroups = (1u << 24) - 1u;
    const uint32_t fill = empty_block_groups(entries), slots = n / 256u + (n % 256u != 0u);
    if (slots > kMaxGroups) return hipErrorInvalidConfiguration;
    if (fill + slots <= kMaxGroups) {
        launch(fill + slots, fill);
        return hipGetLastError();
    }
    launch(fill, fill);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    launch(slots, 0u);
    return hipGetLastError();
}

}  // namespace fh
