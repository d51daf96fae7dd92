// fh_grid.hip -- cell ranges and the 3x3x3 neighbour query for gfx950.  (The CSR cell_start
// of HashGrid::build comes from the sorted keys directly, k_csr_from_sorted in fh_sph.hip.)
//
//   k_boundaries   find_cell_boundaries (radix_sort.rs:229-317): one thread per sorted key marks
//                  the first / last index of its run and the empty cells before it.
//   k_nbr_stream   HashGrid::query_neighbors (hashgrid.rs:145-193) for every point of a built
//                  grid: the 3 x-adjacent cells of one (dy, dz) row are contiguous in the
//                  sorted order, so the 27-cell walk is 9 contiguous ranges visited in the
//                  reference's dz, dy, dx order.
#include "fh_cells.hpp"
#include "fh_internal.hpp"
#include "fh_stream.hpp"

namespace fh {

// ---------------------------------------------------------------------------------------------
__global__ void k_fill_u32(uint32_t* __restrict__ p, uint32_t value, uint32_t n) {
    uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = value;
}

hipError_t launch_fill_u32(fh_ctx* c, uint32_t* p, uint32_t value, uint32_t n) {
    if (n == 0) return hipSuccess;
    k_fill_u32<<<ceil_div(n, 256u), 256, 0, c->stream>>>(p, value, n);
    return hipGetLastError();
}

// radix_sort.rs:451-465, in one launch: the slots write the first and the end of their runs and the
// sentinels of the empty cells before them, and fill_empty_blocks the longer gaps (two fills of
// every cell and then the runs: 10 us for 300,007 keys of 1,000,000 cells, 7 us this way and two
// launches fewer).
__global__ __launch_bounds__(256) void k_boundaries(const uint32_t* __restrict__ keys, uint32_t n,
                                                    uint32_t C, uint32_t* __restrict__ cell_start,
                                                    uint32_t* __restrict__ cell_end,
                                                    uint32_t fill_groups) {
    const auto empty = [&](uint32_t c, uint32_t) {
        cell_start[c] = 0xFFFFFFFFu;
        cell_end[c] = 0u;
    };
    if (blockIdx.x < fill_groups) {
        fill_empty_blocks<false>(blockIdx.x, keys, n, C, empty);
        return;
    }
    const uint32_t s = (blockIdx.x - fill_groups) * 256u + threadIdx.x;
    const int lane = threadIdx.x & 63;
    uint32_t lo = 0, hi = 0, lo2 = 0, hi2 = 0;
    if (s < n) {
        const uint32_t k = keys[s];
        const uint32_t pk = s > 0u ? keys[s - 1u] : 0xFFFFFFFFu;  // "-1" before slot 0
        if (s == 0u || pk != k) {
            lo = min(s == 0u ? 0u : pk + 1u, C);  // pk < k: no wrap
            hi = min(k, C);
            if (k < C) cell_start[k] = s;
        }
        if (s == n - 1u || keys[s + 1u] != k) {
            if (k < C) cell_end[k] = s + 1u;
            if (s == n - 1u) {
                lo2 = k < C ? k + 1u : C;
                hi2 = C;
            }
        }
    }
    fill_cells(lo, hi, C, 0u, lane, empty);
    if (__ballot(lo2 < hi2) != 0ull) fill_cells(lo2, hi2, C, 0u, lane, empty);
}

hipError_t launch_boundaries(fh_ctx* c, const uint32_t* sorted_keys, uint32_t n,
                             uint32_t num_cells, uint32_t* cell_start, uint32_t* cell_end) {
    return launch_cell_groups(n, num_cells, [&](uint32_t groups, uint32_t fill) {
        k_boundaries<<<groups, 256, 0, c->stream>>>(sorted_keys, n, num_cells, cell_start, cell_end,
                                                    fill);
    });
}

// ---------------------------------------------------------------------------------------------
// Rust `f32 as i32` of an already floored value (NaN -> 0, saturating).
__device__ __forceinline__ int32_t rust_as_i32(float f) {
    if (f != f) return 0;
    if (f >= 2147483648.0f) return INT32_MAX;
    if (f <= -2147483648.0f) return INT32_MIN;
    return (int32_t)f;
}

struct Pos3 {
    float x, y, z;
};

// The point positions in sorted order (float4), so the query walks contiguous memory.  A
// gather through sorted_indices from the caller's three arrays would read three scattered
// words per point (a cache line each), and a scatter to the sorted slots (through the inverse
// permutation) writes partial cache lines twice (rank, then the float4); instead the points are
// packed once as float4 in their own order (k_pack_pos: coalesced reads and writes), and every
// sorted slot then reads one 16-byte record (k_gather_pos: coalesced sidx reads and writes, one
// scattered 16-byte read per point, mostly served from the MALL, which holds the packed copy).
__global__ __launch_bounds__(256) void k_pack_pos(const float* __restrict__ x,
                                                  const float* __restrict__ y,
                                                  const float* __restrict__ z, uint32_t stride,
                                                  uint32_t n, float4* __restrict__ packed) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const size_t o = (size_t)i * stride;
    packed[i] = make_float4(x[o], y[o], z[o], 0.0f);
}

__global__ __launch_bounds__(256) void k_gather_pos(const float4* __restrict__ packed,
                                                    const uint32_t* __restrict__ sidx,
                                                    uint32_t n, float4* __restrict__ spos) {
    const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= n) return;
    const uint32_t i = sidx[s];
    // a grid built over these n points holds a permutation of 0..n-1
    spos[s] = i < n ? packed[i] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
}

// The same straight from the caller's 12-byte records (x, y, z adjacent, stride 3): one scattered
// record per point as from the packed copy, without the pass that makes it (4,194,304 points: build and
// query 669 -> 637 us; three separate arrays would cost three lines per point).
__global__ __launch_bounds__(256) void k_gather_aos(const float* __restrict__ xyz,
                                                    const uint32_t* __restrict__ sidx, uint32_t n,
                                                    float4* __restrict__ spos) {
    const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= n) return;
    const uint32_t i = sidx[s];
    Pos3 p = {0.0f, 0.0f, 0.0f};
    if (i < n) p = ((const Pos3*)xyz)[i];
    spos[s] = make_float4(p.x, p.y, p.z, 0.0f);
}

// HashGrid::query_neighbors for every point of a built grid, with the neighbour candidates of 64
// consecutive sorted points staged through LDS (the wave candidate stream of fh_stream.hpp, one
// z-slab at a time, kQueryWin candidates per window: a slab's stream of uniform points, ~240
// candidates, mostly fits one window, so a lane's rows are rarely cut by a window edge and the
// row loops, which run as long as their longest lane, run once per slab).  A candidate is 12 bytes
// in LDS (16 put neighbouring cells' lanes on the same banks), and a window 384 of them: the
// query of 4,194,304 points 429 -> 405 us (256: 425, 320: 413, 448: 438).  Arithmetic is exactly
// the reference's (the library is built with -ffp-contract=off): diff = p_j - q, dist_sq =
// (dx*dx + dy*dy) + dz*dz, `<=` against radius*radius, weight coeff*diff*diff*diff summed in
// visiting order; each lane visits its own candidates in the reference's order (dz, dy, then
// ascending sorted index), so counts and weight sums are bit-identical to the CPU restatement.
// Points whose query cell lies outside the grid (the reference does not clamp it) take a
// per-lane walk around that cell afterwards.
#ifndef FH_QWIN
#define FH_QWIN 384
#endif
constexpr int kQueryWin = FH_QWIN;

// One candidate: a candidate beyond the radius adds 0 to the count and +0.0f to the weight sum,
// which starts at +0 and only grows, so w + 0.0f == w bit for bit and the sum over the
// candidates is the reference's sum over its neighbours.
__device__ __forceinline__ void nbr_pair(float px, float py, float pz, const float4& q,
                                         float radius_sq, float coeff, uint32_t& cnt, float& w) {
    const float dx = px - q.x, dy = py - q.y, dz = pz - q.z;
    const float dist_sq = dx * dx + dy * dy + dz * dz;
    const bool ok = dist_sq <= radius_sq;
    const float diff = radius_sq - dist_sq;
    const float t = coeff * diff * diff * diff;
    cnt += ok ? 1u : 0u;
    w += ok ? t : 0.0f;
}

__global__ __launch_bounds__(kWave) void k_nbr_stream(const float4* __restrict__ spos,
                                                      const uint32_t* __restrict__ sidx,
                                                      uint32_t n, GridDesc g,
                                                      const uint32_t* __restrict__ cell_start,
                                                      float radius_sq, float coeff,
                                                      uint32_t* __restrict__ counts,
                                                      float* __restrict__ wsum) {
    constexpr int kLoads = kQueryWin / kWave;
    __shared__ float s_p[3 * kQueryWin];  // x, y, z
    const int lane = threadIdx.x;
    // runs of consecutive sub-tiles on one XCD: neighbouring sub-tiles read mostly the same
    // candidate rows, which then stay in that XCD's L2
    const uint32_t s = xcd_chunked(blockIdx.x, gridDim.x) * kWave + (uint32_t)lane;
    const bool in = s < n;
    const float4 q = spos[in ? s : 0u];
    // the sort's (clamped) cell, and the reference's unclamped query cell
    const uint32_t cxc = cell_coord(q.x, g.ox, g.cs, g.nx);
    const uint32_t cyc = cell_coord(q.y, g.oy, g.cs, g.ny);
    const uint32_t czc = cell_coord(q.z, g.oz, g.cs, g.nz);
    const int64_t cxu = rust_as_i32(floorf((q.x - g.ox) / g.cs));
    const int64_t cyu = rust_as_i32(floorf((q.y - g.oy) / g.cs));
    const int64_t czu = rust_as_i32(floorf((q.z - g.oz) / g.cs));
    const bool inside = cxu == (int64_t)cxc && cyu == (int64_t)cyc && czu == (int64_t)czc;
    const uint32_t hr = cyc + czc * g.ny;  // home row of the sorted order
    const uint32_t x0 = cxc > 0u ? cxc - 1u : 0u;
    const uint32_t x1 = cxc + 1u < g.nx ? cxc + 1u : g.nx - 1u;
    uint32_t cnt = 0;
    float w = 0.0f;
    for (int dz = -1; dz <= 1; dz++) {  // uniform
        uint32_t b[3], e[3];
        const int nz = (int)czc + dz;
#pragma unroll
        for (int r = 0; r < 3; r++) {
            const int ny = (int)cyc + r - 1;
            b[r] = e[r] = 0u;
            if (in && nz >= 0 && nz < (int)g.nz && ny >= 0 && ny < (int)g.ny) {
                const uint32_t row = (uint32_t)ny * g.nx + (uint32_t)nz * g.nx * g.ny;
                b[r] = cell_start[row + x0];
                e[r] = min(cell_start[row + x1 + 1u], n);
            }
        }
        // a segment's row union runs from its first lane's begin to its last lane's end, which
        // holds because the lanes' clamped ranges grow along the row; an outside point keeps its
        // clamped ranges for the union and evaluates none of them (it is walked later)
        LightStream L;
        light_stream(L, b, e, hr, in, lane);
        if (!inside) {
#pragma unroll
            for (int r = 0; r < 3; r++) L.cnt[r] = 0u;
        }
        for (uint32_t w0 = 0; w0 < L.T; w0 += kQueryWin) {  // uniform
            uint32_t j[kLoads];
            window_indices<kQueryWin>(L, w0, lane, j);
            float4 v[kLoads];
#pragma unroll
            for (int k = 0; k < kLoads; k++) v[k] = spos[j[k]];
            __builtin_amdgcn_wave_barrier();
#pragma unroll
            for (int k = 0; k < kLoads; k++) {
                float* const o = s_p + 3 * (k * kWave + lane);
                o[0] = v[k].x;
                o[1] = v[k].y;
                o[2] = v[k].z;
            }
            __builtin_amdgcn_wave_barrier();
            // the rows in the reference's dy order (walking them longest first would change
            // the order of the weight sum)
#pragma unroll
            for (int r = 0; r < 3; r++) {
                const uint32_t jb = max(L.S[r], w0);
                const uint32_t je = min(L.S[r] + L.cnt[r], w0 + (uint32_t)kQueryWin);
                // two candidates per step of the LDS address
                // (the bounds are formed from the count, never before the buffer: an address
                // below the LDS buffer's start would wrap around in 32-bit LDS addressing)
                const uint32_t m = je > jb ? je - jb : 0u;
                const float* c = s_p + 3u * (jb - w0);
                const float* const ce = c + 3u * m;
                const float* const cu = c + 3u * (m & ~1u);
                while (c < cu) {
                    const float x0 = c[0], y0 = c[1], z0 = c[2];
                    const float x1 = c[3], y1 = c[4], z1 = c[5];
                    nbr_pair(x0, y0, z0, q, radius_sq, coeff, cnt, w);
                    nbr_pair(x1, y1, z1, q, radius_sq, coeff, cnt, w);
                    c += 6;
                }
                if (c < ce) nbr_pair(c[0], c[1], c[2], q, radius_sq, coeff, cnt, w);
            }
            __builtin_amdgcn_wave_barrier();
        }
    }
    if (in && !inside) {  // rare: the reference's walk around an unclamped query cell
        cnt = 0;
        w = 0.0f;
        const int64_t lx0 = cxu - 1 < 0 ? 0 : cxu - 1;
        const int64_t lx1 = cxu + 1 > (int64_t)g.nx - 1 ? (int64_t)g.nx - 1 : cxu + 1;
        for (int dz = -1; dz <= 1; dz++) {
            const int64_t nz = czu + dz;
            if (nz < 0 || nz >= (int64_t)g.nz) continue;
            for (int dy = -1; dy <= 1; dy++) {
                const int64_t ny = cyu + dy;
                if (ny < 0 || ny >= (int64_t)g.ny || lx0 > lx1) continue;
                const uint32_t row = (uint32_t)ny * g.nx + (uint32_t)nz * g.nx * g.ny;
                const uint32_t jb = cell_start[row + (uint32_t)lx0];
                const uint32_t je = min(cell_start[row + (uint32_t)lx1 + 1u], n);
                for (uint32_t j = jb; j < je; j++) {
                    const float4 p = spos[j];
                    nbr_pair(p.x, p.y, p.z, q, radius_sq, coeff, cnt, w);
                }
            }
        }
    }
    if (!in) return;
    const uint32_t i = sidx[s];
    if (i >= n) return;
    counts[i] = cnt;
    if (wsum) wsum[i] = w;
}

// Batched HashGrid::query_neighbors (hashgrid.rs:145-193): kQueryLanes lanes per query walk its nine
// row ranges together, kQueryStep * kQueryLanes candidates per step with all their loads in
// flight, and a ballot gives each neighbour its place, so the list keeps the reference's order.
// Eight lanes, two steps at a time: a row of ~21 candidates (30 neighbours within the radius) takes two.
//
// Positions come from a copy in slot order when the batch is large (k_sort_pos), where a row is a few
// contiguous lines; read through sorted_indices from the caller's arrays every candidate is a line
// (two more in three separate arrays), and a lane per query waits for them one after the other.
// 120,000 queries in 600,000 points: 333 us for a count or fill pass with a lane per query, 67 us
// with eight, the copy (11 us) included (83 while both ways to the positions shared a loop); 4, 16 and
// 32 lanes 110, 82 and 80 against those 83, and 94 with 16-byte positions: the rows' lines, which
// mostly miss a 4 MB L2, are what is left.
//
// The copy reads every point once, so it pays from a number of candidates per point on: 2.5, or, where
// the caller's positions themselves stay in the L2, 12.  2,000,000 points, 200,000 queries: 4
// neighbours each (2.6 candidates per point) 106 us against 145 in place; 2 (1.3) 114 against 104; 0.5
// (0.3) 95 against 64.  600,000 points, 30 neighbours: 7,000 queries (2.3) 38 against 34.  100,000
// points and queries: 3 neighbours (19) 30 against 33, 1 (6.4) 28 against 24.  Below kQueryCopyMin
// queries the extra launch would cost more than it gives.  Queries all over the grid meet 27 n / C
// candidates each, wherever the points are.  Where that is too few, but the queries are at least a
// kQueryFew-th of the points, they may all be where the points are (a fluid in a corner of its box):
// k_sort_pos counts the candidates of kQuerySamples of them and leaves its answer for k_query (5 us:
// 120,000 queries among 600,000 points in a 64th of the grid 72 us a pass, 263 in place).
// The points' number is the grid's own (cell_start[C]), read on the device; a grid of more points than
// the context holds is read in place.
// An id of that number or more (a grid over some of an array's points, an entry that no query comes
// near) is not followed by the copy, which leaves a NaN: its position is read where a query meets it.
constexpr uint32_t kQueryLanes = 8, kQueryStep = 2, kQueryCopyMin = 1024;
constexpr uint32_t kQueryCopyShare = 5, kQueryCacheShare = 24, kQueryCacheN = 1u << 18;
constexpr uint32_t kQueryFew = 32, kQuerySamples = 16;
struct QueryCopy {
    Pos3* spos;      // null: no copy (12 bytes: a row is a quarter fewer lines than with float4)
    uint32_t* ask;   // k_sort_pos' answer where query_rule asks for the samples
    uint32_t max_n;  // room of spos
    uint32_t nq;     // queries of the whole batch
    uint32_t C;      // cells
};
__device__ __forceinline__ uint32_t query_share(uint32_t n) {
    return n < kQueryCacheN ? kQueryCacheShare : kQueryCopyShare;
}
// Whether the batch reads from a copy: by kQueryCopyShare / 2 candidates per point of the grid.
enum : uint32_t { kInPlace, kCopied, kAsk };
__device__ __forceinline__ uint32_t query_rule(const QueryCopy& Q, uint32_t n) {
    if (!Q.spos || n > Q.max_n) return kInPlace;
    if ((uint64_t)Q.nq * 54u >= (uint64_t)Q.C * query_share(n)) return kCopied;
    return (uint64_t)Q.nq * kQueryFew >= n ? kAsk : kInPlace;
}

// The cell of a query (not clamped) and its row r = (dz + 1) * 3 + dy + 1 of the reference's walk.
struct QueryCell {
    int64_t cy, cz, x0, x1;
};
__device__ __forceinline__ QueryCell query_cell(float px, float py, float pz, const GridDesc& g) {
    const int64_t cx = rust_as_i32(floorf((px - g.ox) / g.cs));
    QueryCell c;
    c.cy = rust_as_i32(floorf((py - g.oy) / g.cs));
    c.cz = rust_as_i32(floorf((pz - g.oz) / g.cs));
    c.x0 = cx - 1 < 0 ? 0 : cx - 1;
    c.x1 = cx + 1 > (int64_t)g.nx - 1 ? (int64_t)g.nx - 1 : cx + 1;
    return c;
}
__device__ __forceinline__ void query_range(const QueryCell& c, uint32_t r, const GridDesc& g,
                                            const uint32_t* __restrict__ cstart, uint32_t n,
                                            uint32_t& b, uint32_t& e) {
    const int64_t nz = c.cz + (int64_t)(r / 3u) - 1, ny = c.cy + (int64_t)(r % 3u) - 1;
    b = e = 0u;
    if (nz < 0 || nz >= (int64_t)g.nz || ny < 0 || ny >= (int64_t)g.ny || c.x0 > c.x1) return;
    const uint32_t row = (uint32_t)ny * g.nx + (uint32_t)nz * g.nx * g.ny;
    e = min(cstart[row + (uint32_t)c.x1 + 1u], n);
    b = cstart[row + (uint32_t)c.x0];
}

__global__ __launch_bounds__(256) void k_sort_pos(const float* __restrict__ x,
                                                  const float* __restrict__ y,
                                                  const float* __restrict__ z, uint32_t stride,
                                                  GridDesc g,
                                                  const uint32_t* __restrict__ cstart,
                                                  const uint32_t* __restrict__ sidx,
                                                  const float* __restrict__ qx,
                                                  const float* __restrict__ qy,
                                                  const float* __restrict__ qz, uint32_t qstride,
                                                  QueryCopy Q) {
    const uint32_t n = cstart[Q.C];
    const uint32_t rule = query_rule(Q, n);
    if (rule == kInPlace) return;
    if (rule == kAsk) {  // the same count in every workgroup
        __shared__ uint32_t s_met;
        if (threadIdx.x < kWave) {
            uint32_t met = 0;
            if (threadIdx.x < kQuerySamples) {
                const size_t o = (size_t)((uint64_t)threadIdx.x * Q.nq / kQuerySamples) * qstride;
                const QueryCell c = query_cell(qx[o], qy[o], qz[o], g);
#pragma unroll
                for (uint32_t r = 0; r < 9u; r++) {
                    uint32_t b, e;
                    query_range(c, r, g, cstart, n, b, e);
                    met += e > b ? min(e - b, 1u << 22) : 0u;  // (no overflow: 144 rows)
                }
            }
#pragma unroll
            for (int d = 1; d < (int)kQuerySamples; d <<= 1)
                met += (uint32_t)__shfl_xor((int)met, d, kWave);
            if (threadIdx.x == 0u) s_met = met;
        }
        __syncthreads();
        const bool copy =
            2u * (uint64_t)s_met * Q.nq >= (uint64_t)kQuerySamples * query_share(n) * n;
        if (blockIdx.x == 0u && threadIdx.x == 0u) *Q.ask = copy ? 1u : 0u;
        if (!copy) return;
    }
    for (uint32_t s = blockIdx.x * 256u + threadIdx.x; s < n; s += gridDim.x * 256u) {
        const uint32_t i = sidx[s];
        const size_t at = (size_t)(i < n ? i : 0u) * stride;
        const float nan = __builtin_nanf("");
        Pos3 p = {x[at], y[at], z[at]};
        if (i >= n) p = Pos3{nan, nan, nan};
        Q.spos[s] = p;
    }
}

__global__ __launch_bounds__(256) void k_query(const float* __restrict__ x,
                                               const float* __restrict__ y,
                                               const float* __restrict__ z, uint32_t stride,
                                               GridDesc g, const uint32_t* __restrict__ cstart,
                                               const uint32_t* __restrict__ sidx,
                                               const float* __restrict__ qx,
                                               const float* __restrict__ qy,
                                               const float* __restrict__ qz, uint32_t qstride,
                                               uint32_t nq, float radius_sq,
                                               uint32_t* __restrict__ counts,
                                               const uint32_t* __restrict__ offsets,
                                               uint32_t* __restrict__ indices, QueryCopy Q) {
    const uint32_t t = threadIdx.x % kQueryLanes;
    const uint32_t shift = (threadIdx.x & 63u) & ~(kQueryLanes - 1u);
    const uint32_t qi = (blockIdx.x * 256u + threadIdx.x) / kQueryLanes;
    if (qi >= nq) return;  // whole groups
    const uint32_t n = cstart[Q.C];
    const uint32_t rule = query_rule(Q, n), asked = *Q.ask;
    const bool copied = rule == kCopied || (rule == kAsk && asked);  // uniform
    const size_t oq = (size_t)qi * qstride;
    const float px = qx[oq], py = qy[oq], pz = qz[oq];
    const QueryCell c = query_cell(px, py, pz, g);
    // lane t loads row t's range, and every lane the last one's
    uint32_t b0, e0, b8, e8;
    query_range(c, t, g, cstart, n, b0, e0);
    query_range(c, 8u, g, cstart, n, b8, e8);
    uint32_t cnt = 0;
    uint32_t* out = (offsets && indices) ? indices + offsets[qi] : nullptr;
    const uint32_t room = out ? offsets[qi + 1] - offsets[qi] : 0u;
    const auto row = [&](uint32_t r) {
        const uint32_t b = r < 8u ? (uint32_t)__shfl((int)b0, (int)r, (int)kQueryLanes) : b8;
        const uint32_t e = r < 8u ? (uint32_t)__shfl((int)e0, (int)r, (int)kQueryLanes) : e8;
        for (uint32_t j0 = b; j0 < e; j0 += kQueryStep * kQueryLanes) {  // uniform in the group
            float X[kQueryStep], Y[kQueryStep], Z[kQueryStep];
            bool read = !copied;
            if (copied) {
#pragma unroll
                for (uint32_t k = 0; k < kQueryStep; k++) {
                    const Pos3 p = Q.spos[min(j0 + k * kQueryLanes + t, e - 1u)];
                    X[k] = p.x;
                    Y[k] = p.y;
                    Z[k] = p.z;
                }
                static_assert(kQueryStep == 2, "one compare asks both candidates of a step");
                read = __builtin_isunordered(X[0], X[1]);  // (a point that is NaN reads the same again)
            }
            if (read) {
                uint32_t i[kQueryStep];
#pragma unroll
                for (uint32_t k = 0; k < kQueryStep; k++)
                    i[k] = sidx[min(j0 + k * kQueryLanes + t, e - 1u)];
#pragma unroll
                for (uint32_t k = 0; k < kQueryStep; k++) {
                    const size_t o = (size_t)i[k] * stride;
                    X[k] = x[o];
                    Y[k] = y[o];
                    Z[k] = z[o];
                }
            }
#pragma unroll
            for (uint32_t k = 0; k < kQueryStep; k++) {
                const uint32_t j = j0 + k * kQueryLanes + t;
                const float dx = X[k] - px, dy2 = Y[k] - py, dz2 = Z[k] - pz;
                const float dist_sq = dx * dx + dy2 * dy2 + dz2 * dz2;
                const bool hit = j < e && dist_sq <= radius_sq;
                const uint32_t m =
                    (uint32_t)(__ballot(hit) >> shift) & ((1u << kQueryLanes) - 1u);
                const uint32_t at = cnt + (uint32_t)__popc(m & ((1u << t) - 1u));
                if (hit && at < room) out[at] = sidx[j];
                cnt += (uint32_t)__popc(m);
            }
        }
    };
    // the rows in order: all nine, or, where more than three in eight of the wave's are empty, those
    // that hold points (uniform in the group; 100,000 queries of 0.3 neighbours 30 -> 21 us)
    const uint64_t held = __ballot(b0 < e0);
    if (__popcll(held) >= 40) {
        for (uint32_t r = 0; r < 9u; r++) row(r);
    } else {
        uint32_t rows = (uint32_t)(held >> shift) & ((1u << kQueryLanes) - 1u);
        rows |= b8 < e8 ? 1u << 8 : 0u;
        for (; rows; rows &= rows - 1u) row((uint32_t)__builtin_ctz(rows));
    }
    if (t == 0u) counts[qi] = cnt;
}

hipError_t launch_query(fh_ctx* c, const float* x, const float* y, const float* z,
                        uint32_t stride, const GridDesc& g, const uint32_t* cell_start,
                        const uint32_t* sorted_indices, const float* qx, const float* qy,
                        const float* qz, uint32_t qstride, uint32_t nq, float radius,
                        uint32_t* counts, const uint32_t* offsets, uint32_t* indices) {
    if (nq == 0) return hipSuccess;
    const QueryCopy Q{nq >= kQueryCopyMin ? (Pos3*)c->spos : nullptr, &c->ctl->query_copy, c->max_n,
                      nq, g.nx * g.ny * g.nz};
    if (Q.spos) {
        const uint32_t groups = ceil_div(c->max_n, 256u);
        k_sort_pos<<<groups < 2048u ? groups : 2048u, 256, 0, c->stream>>>(
            x, y, z, stride, g, cell_start, sorted_indices, qx, qy, qz, qstride, Q);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    constexpr uint32_t kChunk = 1u << 28;  // queries per launch: below 2^32 threads
    for (uint32_t q0 = 0; q0 < nq; q0 += min(kChunk, nq - q0)) {
        const uint32_t m = min(kChunk, nq - q0);
        const size_t o = (size_t)q0 * qstride;
        k_query<<<ceil_div(m, 256u / kQueryLanes), 256, 0, c->stream>>>(
            x, y, z, stride, g, cell_start, sorted_indices, qx + o, qy + o, qz + o, qstride, m,
            radius * radius, counts + q0, offsets ? offsets + q0 : nullptr, indices, Q);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

hipError_t launch_neighbor_query(fh_ctx* c, const float* x, const float* y, const float* z,
                                 uint32_t stride, uint32_t n, const GridDesc& g,
                                 const uint32_t* cell_start, const uint32_t* sorted_indices,
                                 float radius, uint32_t* counts, float* wsum) {
    if (n == 0) return hipSuccess;
    hipError_t e;
    if (stride == 3u && y == x + 1 && z == x + 2) {
        k_gather_aos<<<ceil_div(n, 256u), 256, 0, c->stream>>>(x, sorted_indices, n, c->spos);
    } else {
        // c->sout (3 float4 per point) is free between SPH calls: the packed copy goes there
        k_pack_pos<<<ceil_div(n, 256u), 256, 0, c->stream>>>(x, y, z, stride, n, c->sout);
        e = hipGetLastError();
        if (e != hipSuccess) return e;
        k_gather_pos<<<ceil_div(n, 256u), 256, 0, c->stream>>>(c->sout, sorted_indices, n, c->spos);
    }
    e = hipGetLastError();
    if (e != hipSuccess) return e;
    // Same float expressions as sph_density.rs:413-416 with h = radius.
    float h = radius;
    float h2 = h * h;
    float h9 = h2 * h2 * h2 * h2 * h;
    float coeff = 315.0f / (64.0f * 3.14159265f * h9);
    tbeg(c, KID_NBR);
    k_nbr_stream<<<ceil_div(n, (uint32_t)kWave), kWave, 0, c->stream>>>(
        c->spos, sorted_indices, n, g, cell_start, radius * radius, coeff, counts, wsum);
    tend(c, KID_NBR);
    return hipGetLastError();
}

}  // namespace fh
