// fh_sph.hip -- SPH density and fused pressure/viscosity passes for gfx950, plus the
// gravity / integrate / box modules.
//
// The passes run over the particles in cell-sorted order (gathered once per substep into
// float4 arrays), so a particle's 27-cell neighbourhood is 9 contiguous ranges of the same
// arrays -- the 3 x-adjacent cells of each (dy, dz) row -- and neighbour reads are coalesced
// and cache-friendly instead of the reference's gathers through sorted_idx into unsorted
// arrays (sph_density.rs:445-450).  Results are scattered back to the caller's arrays in
// original particle order, so FieldSet semantics are unchanged.
//
// Arithmetic follows the reference expressions term by term (the library is compiled with
// -ffp-contract=off and IEEE division / square root) and the neighbours of a particle are
// visited in the reference's order (dz, dy, dx, then ascending particle id within a cell), so
// density and velocity updates reproduce the CPU restatement of sph_density.rs:409-460 and
// sph_fused.rs:542-638.
#include "fh_cells.hpp"
#include "fh_internal.hpp"
#include "fh_stream.hpp"

namespace fh {

// Sorted-order copies of the state.  The sort's last pass wrote rank[i] = sorted slot of
// particle i; k_gather (particle order) writes spos[rank[i]] = (pos[i], bits of rank[i]) and
// svel[rank[i]] = (vel[i], bits of i) -- the caller's arrays are read in order and each
// particle costs two 16-byte stores, instead of six 4-byte reads from scattered lines.  The
// particle id in svel[.].w travels with the particle through later reorderings (co-located
// groups, resident substeps) and into the new state (k_finalize).
__global__ __launch_bounds__(256) void k_gather(
    const float* __restrict__ px, const float* __restrict__ py, const float* __restrict__ pz,
    const float* __restrict__ vx, const float* __restrict__ vy, const float* __restrict__ vz,
    const uint32_t* __restrict__ rank, uint32_t n, float4* __restrict__ spos,
    float4* __restrict__ svel) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const uint32_t r = rank[i];
    if (r >= n) return;  // never taken when the sort is consistent
    spos[r] = make_float4(px[i], py[i], pz[i], __uint_as_float(r));
    if (svel) svel[r] = make_float4(vx[i], vy[i], vz[i], __uint_as_float(i));
}

// Cell ranges, and (big != null) the candidate co-located groups: runs of at least
// kCollapseMin keys in which at least kGroupHits of kGroupSamples evenly spaced particles (over
// the first L of the run, L its length rounded down to a power of two) sit at the position of
// one of them.  Listed as (first slot, offset of that sample) -- the group pass counts the run
// and the members at that sample's position exactly -- and tagged with the epoch in
// cand_tag[cell] for the plan, which runs beside the group pass.
template <class Pos>
__device__ __forceinline__ void cell_starts_slot(uint32_t s, const uint32_t* __restrict__ skeys,
                                                 uint32_t n, uint32_t C,
                                                 uint32_t* __restrict__ cell_start, Pos pos,
                                                 uint2* __restrict__ big, uint32_t cap,
                                                 uint64_t* __restrict__ cand_tag, Control* ctl) {
    const int lane = threadIdx.x & 63;
    uint32_t lo = 0, hi = 0, lo2 = 0, hi2 = 0;
    bool cand = false;
    uint32_t k = 0;
    if (s < n) {
        k = skeys[s];
        const uint32_t pk = s > 0u ? skeys[s - 1u] : 0xFFFFFFFFu;  // "-1" before slot 0
        if (pk != k) {
            lo = pk + 1u;
            hi = min(k, C - 1u) + 1u;
            cand = big && s + kCollapseMin - 1u < n && skeys[s + kCollapseMin - 1u] == k;
        }
        if (s == n - 1u) {
            lo2 = min(k, C - 1u) + 1u;
            hi2 = C + 1u;
        }
    }
    const auto put = [&](uint32_t c, uint32_t v) { cell_start[c] = v; };
    fill_cells(lo, hi, C + 1u, s, lane, put);
    if (__ballot(lo2 < hi2) != 0ull) fill_cells(lo2, hi2, C + 1u, n, lane, put);
    // Rare: a run of at least kCollapseMin.  The whole wave takes each such run of its lanes in
    // turn: lane q < kGroupSamples loads sample q (one round trip for all 16); the middle sample
    // is tried first as the group's position, then each other in turn (a corner group can fill
    // all but the middle of a run).
    uint64_t todo = __ballot(cand);
    while (todo) {  // uniform
        const int l = __ffsll((unsigned long long)todo) - 1;
        todo &= todo - 1ull;
        const uint32_t rs = (uint32_t)__builtin_amdgcn_readlane((int)s, l);
        const uint32_t rk = (uint32_t)__builtin_amdgcn_readlane((int)k, l);
        uint32_t L = kCollapseMin;
        while (L < (1u << 30) && rs + 2u * L - 1u < n && skeys[rs + 2u * L - 1u] == rk) L *= 2u;
        uint32_t px = 0, py = 0, pz = 0;
        if ((uint32_t)lane < kGroupSamples) {
            const float4 v = pos(rs + ((uint32_t)lane * L) / kGroupSamples);
            px = __float_as_uint(v.x);
            py = __float_as_uint(v.y);
            pz = __float_as_uint(v.z);
        }
        uint32_t off = 0, hits = 0;
        for (uint32_t a = 0; a < kGroupSamples; a++) {  // uniform
            const uint32_t qa = a == 0u ? kGroupSamples / 2u : (a <= kGroupSamples / 2u ? a - 1u : a);
            const uint32_t ax = (uint32_t)__builtin_amdgcn_readlane((int)px, (int)qa);
            const uint32_t ay = (uint32_t)__builtin_amdgcn_readlane((int)py, (int)qa);
            const uint32_t az = (uint32_t)__builtin_amdgcn_readlane((int)pz, (int)qa);
            const uint32_t hq = (uint32_t)__popcll(__ballot((uint32_t)lane < kGroupSamples &&
                                                            px == ax && py == ay && pz == az));
            if (hits < kGroupHits) {
                hits = hq;
                off = (qa * L) / kGroupSamples;
            }
        }
        if (hits >= kGroupHits && lane == 0) {
            const uint32_t slot = atomicAdd(&ctl->big_count.v, 1u);
            if (slot < cap) big[slot] = make_uint2(rs, off);
            cand_tag[rk] = (uint64_t)ctl->epoch << 32;  // the plan: this cell may hold a group
        }
    }
}

// Position of sorted slot x for the samples of cell_starts_slot: from the sorted copy, or, in
// resident substeps (which build that copy in the same kernel), from the previous substep's
// state through the slot map.
struct SortedPos {
    const float4* __restrict__ spos;
    __device__ float4 operator()(uint32_t x) const { return spos[x]; }
};
struct ResidentPos {
    const float4* __restrict__ sout;
    const uint32_t* __restrict__ prev;
    uint32_t n;
    __device__ float4 operator()(uint32_t x) const { return sout[2u * min(prev[x], n - 1u)]; }
};

__global__ __launch_bounds__(256) void k_cell_starts(const uint32_t* __restrict__ skeys,
                                                     uint32_t n, uint32_t C,
                                                     uint32_t* __restrict__ cell_start,
                                                     const float4* __restrict__ spos,
                                                     uint2* __restrict__ big, uint32_t cap,
                                                     uint64_t* __restrict__ cand_tag,
                                                     Control* ctl, uint32_t fill_groups) {
    if (blockIdx.x < fill_groups) {
        fill_empty_blocks<true>(blockIdx.x, skeys, n, C + 1u,
                                [&](uint32_t c, uint32_t v) { cell_start[c] = v; });
        return;
    }
    cell_starts_slot((blockIdx.x - fill_groups) * blockDim.x + threadIdx.x, skeys, n, C, cell_start,
                     SortedPos{spos}, big, cap, cand_tag, ctl);
}

static hipError_t launch_cell_starts(fh_ctx* c, uint32_t cells, uint32_t n, bool list_big) {
    const uint32_t fill = empty_block_groups(cells + 1u);
    tbeg(c, KID_SCAN);
    k_cell_starts<<<fill + ceil_div(n, 256u), 256, 0, c->stream>>>(
        c->skeys, n, cells, c->cell_start, c->spos, list_big ? c->big : nullptr,
        ceil_div(c->max_n, 64u) + 1u, c->run_tag, c->ctl, fill);
    tend(c, KID_SCAN);
    return hipGetLastError();
}

hipError_t launch_gather(fh_ctx* c, const GridDesc& g, uint32_t cells, const float* px,
                         const float* py, const float* pz, const float* vx, const float* vy,
                         const float* vz, uint32_t n, bool with_vel, bool list_big) {
    (void)g;
    if (n == 0) return launch_fill_u32(c, c->cell_start, 0u, cells + 1u);
    tbeg(c, KID_GATHER);
    k_gather<<<ceil_div(n, 256u), 256, 0, c->stream>>>(px, py, pz, vx, vy, vz, c->rank, n,
                                                       c->spos, with_vel ? c->svel : nullptr);
    hipError_t e = hipGetLastError();
    tend(c, KID_GATHER);
    if (e != hipSuccess) return e;
    return launch_cell_starts(c, cells, n, list_big);
}

// Resident substeps: new slot r takes the state of previous slot prev[r] from c->sout (one
// 32-byte read: (x, y, z, rho), (vx, vy, vz, particle id)) and writes spos / svel in order;
// the same thread then does k_cell_starts' work for slot r.
__global__ __launch_bounds__(256) void k_gather_resident(
    const float4* __restrict__ sout, const uint32_t* __restrict__ prev, uint32_t n,
    float4* __restrict__ spos, float4* __restrict__ svel, const uint32_t* __restrict__ skeys,
    uint32_t C, uint32_t* __restrict__ cell_start, uint2* __restrict__ big, uint32_t cap,
    uint64_t* __restrict__ cand_tag, Control* ctl, uint32_t fill_groups) {
    if (blockIdx.x < fill_groups) {
        fill_empty_blocks<true>(blockIdx.x, skeys, n, C + 1u,
                                [&](uint32_t c, uint32_t v) { cell_start[c] = v; });
        return;
    }
    const uint32_t r = (blockIdx.x - fill_groups) * blockDim.x + threadIdx.x;
    if (r < n) {
        const uint32_t q = prev[r];
        if (q < n) {  // always, when the sort is consistent
            const float4 p = sout[2u * q], v = sout[2u * q + 1u];
            spos[r] = make_float4(p.x, p.y, p.z, __uint_as_float(r));
            svel[r] = v;
        }
    }
    cell_starts_slot(r, skeys, n, C, cell_start, ResidentPos{sout, prev, n}, big, cap, cand_tag,
                     ctl);
}

hipError_t launch_gather_resident(fh_ctx* c, uint32_t cells, uint32_t n) {
    if (n == 0) return launch_fill_u32(c, c->cell_start, 0u, cells + 1u);
    const uint32_t fill = empty_block_groups(cells + 1u);
    tbeg(c, KID_GATHER);
    k_gather_resident<<<fill + ceil_div(n, 256u), 256, 0, c->stream>>>(
        c->sout, c->sidx2, n, c->spos, c->svel, c->skeys, cells, c->cell_start, c->big,
        ceil_div(c->max_n, 64u) + 1u, c->run_tag, c->ctl, fill);
    tend(c, KID_GATHER);
    return hipGetLastError();
}

// CSR cell_start from keys the caller already sorted (hashgrid.rs:102-106 computes the same
// array as the prefix sum of per-cell counts): cell_start[c] = number of keys < c for
// c = 0..C, so keys >= C count in no cell.  Each slot fills the cells between the previous
// slot's key and its own (both clamped to C), the last slot the cells after its key; the
// filled ranges partition 0..C (whole empty blocks: fill_empty_blocks).
__global__ __launch_bounds__(256) void k_csr_from_sorted(const uint32_t* __restrict__ keys,
                                                         uint32_t n, uint32_t C,
                                                         uint32_t* __restrict__ cell_start,
                                                         uint32_t fill_groups) {
    if (blockIdx.x < fill_groups) {
        fill_empty_blocks<true>(blockIdx.x, keys, n, C + 1u,
                                [&](uint32_t c, uint32_t v) { cell_start[c] = v; });
        return;
    }
    const uint32_t s = (blockIdx.x - fill_groups) * blockDim.x + threadIdx.x;
    const int lane = threadIdx.x & 63;
    uint32_t lo = 0, hi = 0, lo2 = 0, hi2 = 0;
    if (s < n) {
        const uint32_t k = min(keys[s], C);
        const uint32_t lo_k = s > 0u ? min(keys[s - 1u], C) + 1u : 0u;  // "-1" before slot 0
        lo = lo_k;
        hi = lo_k <= k ? k + 1u : lo_k;
        if (s == n - 1u) {
            lo2 = k + 1u;
            hi2 = C + 1u;
        }
    }
    const auto put = [&](uint32_t c, uint32_t v) { cell_start[c] = v; };
    fill_cells(lo, hi, C + 1u, s, lane, put);
    if (__ballot(lo2 < hi2) != 0ull) fill_cells(lo2, hi2, C + 1u, n, lane, put);
}

hipError_t launch_csr_from_sorted(fh_ctx* c, const uint32_t* keys, uint32_t n, uint32_t cells,
                                  uint32_t* cell_start) {
    if (n == 0) return launch_fill_u32(c, cell_start, 0u, cells + 1u);
    return launch_cell_groups(n, cells + 1u, [&](uint32_t groups, uint32_t fill) {
        k_csr_from_sorted<<<groups, 256, 0, c->stream>>>(keys, n, cells, cell_start, fill);
    });
}

// Sorted-order state for the exact passes over a caller's grid (sorted_indices[s] = the particle in
// slot s): the same layout k_gather writes, plus the densities.  A malformed id is never written
// back; as a neighbour it reads particle 0 in the force pass, and is none in the unfused passes
// (SKIP_BAD: a NaN position passes no distance test), which also get rank[i], a slot of particle i.
template <bool SKIP_BAD>
__global__ __launch_bounds__(256) void k_gather_grid(
    const float* __restrict__ px, const float* __restrict__ py, const float* __restrict__ pz,
    const float* __restrict__ vx, const float* __restrict__ vy, const float* __restrict__ vz,
    const float* __restrict__ density, const uint32_t* __restrict__ sorted_indices, uint32_t n,
    float4* __restrict__ spos, float4* __restrict__ svel, float* __restrict__ srho,
    uint32_t* __restrict__ sidx, uint32_t* __restrict__ rank) {
    const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= n) return;
    const uint32_t i = sorted_indices[s];
    const bool ok = i < n;
    const uint32_t q = ok ? i : 0u;
    const float bad = __builtin_nanf("");
    spos[s] = SKIP_BAD && !ok ? make_float4(bad, bad, bad, 0.0f)
                              : make_float4(px[q], py[q], pz[q], __uint_as_float(s));
    if (SKIP_BAD && ok) rank[i] = s;
    svel[s] = make_float4(vx[q], vy[q], vz[q], __uint_as_float(q));
    srho[s] = density[q];
    sidx[s] = ok ? i : 0xFFFFFFFFu;
}

hipError_t launch_gather_grid(fh_ctx* c, const float* px, const float* py, const float* pz,
                              const float* vx, const float* vy, const float* vz,
                              const float* density, const uint32_t* sorted_indices, uint32_t n,
                              bool skip_bad) {
    if (n == 0) return hipSuccess;
    tbeg(c, KID_GATHER);
    const auto kernel = skip_bad ? k_gather_grid<true> : k_gather_grid<false>;
    kernel<<<ceil_div(n, 256u), 256, 0, c->stream>>>(px, py, pz, vx, vy, vz, density,
                                                     sorted_indices, n, c->spos, c->svel, c->srho,
                                                     c->sidx, c->rank);
    tend(c, KID_GATHER);
    return hipGetLastError();
}

// Binary position frame of the streaming runner (manifest_runner.rs:150-167 interleaves
// pos_x/y/z per particle; serve.rs:43-62 packs u32 frame, u32 count, then the f32 values,
// all little-endian -- the device's byte order).  Word w of the output is written by thread
// w (coalesced stores): words 0 and 1 are the header, word 2 + 3 i + a is component a of
// particle i.  The frame number is `frame`, or, when `counter` is non-NULL, *counter, which the
// kernel then increments (so a captured graph emits consecutive frame numbers).
__global__ __launch_bounds__(256) void k_pack_frame(const float* __restrict__ px,
                                                    const float* __restrict__ py,
                                                    const float* __restrict__ pz, uint32_t n,
                                                    uint32_t frame, uint32_t* counter,
                                                    uint32_t* __restrict__ out) {
    const uint64_t w = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const uint64_t words = 2ull + 3ull * n;
    if (w >= words) return;
    if (w < 2u) {
        if (w == 0u) {
            uint32_t f = frame;
            if (counter) {
                f = *counter;
                *counter = f + 1u;  // one thread of one workgroup: no other access in the launch
            }
            out[0] = f;
        } else {
            out[1] = n;
        }
        return;
    }
    const uint64_t t = w - 2u;
    const uint32_t i = (uint32_t)(t / 3u), a = (uint32_t)(t - 3u * (t / 3u));
    const float* src = a == 0u ? px : (a == 1u ? py : pz);
    out[w] = __float_as_uint(src[i]);
}

hipError_t launch_pack_frame(fh_ctx* c, const float* px, const float* py, const float* pz,
                             uint32_t n, uint32_t frame, uint32_t* counter, void* out) {
    const uint64_t words = 2ull + 3ull * n;
    k_pack_frame<<<(uint32_t)((words + 255u) / 256u), 256, 0, c->stream>>>(
        px, py, pz, n, frame, counter, (uint32_t*)out);
    return hipGetLastError();
}

// Clamped cell of a particle in the SPH kernels (sph_density.rs:421-426): grid origin 0.
struct Cell3 {
    int cx, cy, cz;
};
__device__ __forceinline__ Cell3 sph_cell(const float4& p, const GridDesc& g) {
    Cell3 c;
    c.cx = (int)cell_coord(p.x, 0.0f, g.cs, g.nx);
    c.cy = (int)cell_coord(p.y, 0.0f, g.cs, g.ny);
    c.cz = (int)cell_coord(p.z, 0.0f, g.cs, g.nz);
    return c;
}

// ---------------------------------------------------------------------------------------------
// Neighbour walk of the bit-exact passes: one wave per 64 consecutive sorted particles, each lane
// visiting its own candidates in the reference's order (dz, dy, dx, then ascending slot).  The
// candidates are staged through LDS a window at a time (the stream of fh_stream.hpp, one z-slab
// after the other), 12 bytes of position each, so that a candidate costs the wave three LDS dwords
// instead of a 16-byte gather per lane.
//
// For the passes whose pair terms hold IEEE divisions and square roots (~70 VALU instructions,
// and one lane in six is within h) a row is walked twice: first the distance test of up to 32
// candidates into a bit mask per lane, then the set bits.  In one loop every candidate that is a
// neighbour of any of the 64 lanes costs the whole wave the divisions: 216 times per particle of
// a dam-break block against ~54, the longest lane's hits.  262,144 particles of such a block: force
// pass 124 -> 64 us, density pass (one walk) 52 -> 35 us; 400,000: force pass 145 -> 106 us.
//
// The stream needs the lanes' ranges to grow along a home row and to be those of a grid built over
// these positions.  A wave that finds otherwise (a caller's grid of other positions), or whose
// stream is far longer than its lanes' ranges (sparse particles beside a dense row), walks its
// lanes' ranges in global memory instead: the same candidates in the same order.
// 320 candidates per window: 262,144 particles, force pass 64 us (256: 73, 384: 87, 192: 92; each
// further window is another round of loads, a larger one leaves fewer waves per SIMD).
constexpr int kExactWin = 320;
// (64 home rows of 3 unions of at most n candidates each: no 32-bit overflow of a stream's length)
constexpr uint32_t kExactStreamN = 1u << 24;
// A wave none of whose particles faces more candidates in a slab than this walks them in global memory
// too: a stream's set-up costs more than it saves, and of the force pass's velocities only the
// neighbours' are read.  262,000 particles: density pass, 0.3 per cell 24.2 (stream) and 18.8 us, 0.7
// 25.0 and 22.0, 1 25.5 and 23.4, 2 27.3 and 30.5; force pass, whose registers and LDS leave fewer waves
// to hide the loads, 0.1 per cell 33.2 and 27.8 us, 0.3 34.8 and 35.7, 1 43.4 and 59.3.
constexpr uint32_t kExactFewDensity = 16, kExactFewForce = 4;
struct ExactLds {
    float xyz[3 * (kExactWin + 4)];  // (a row's masked last step reads up to 3 candidates past it)
};

// The three row ranges of slab dz around cell c, clamped to n (empty outside the grid, and where a
// malformed grid has them inverted).
__device__ __forceinline__ void exact_ranges(const Cell3& c, bool live, const GridDesc& g,
                                             const uint32_t* __restrict__ cstart, uint32_t n,
                                             int dz, uint32_t b[3], uint32_t e[3]) {
    const uint32_t x0 = (uint32_t)(c.cx > 0 ? c.cx - 1 : 0);
    const uint32_t x1 = (uint32_t)(c.cx + 1 < (int)g.nx ? c.cx + 1 : (int)g.nx - 1);
    const int nz = c.cz + dz;
#pragma unroll
    for (int r = 0; r < 3; r++) {
        const int ny = c.cy + r - 1;
        b[r] = e[r] = 0u;
        if (live && nz >= 0 && nz < (int)g.nz && ny >= 0 && ny < (int)g.ny) {
            const uint32_t row = (uint32_t)ny * g.nx + (uint32_t)nz * g.nx * g.ny;
            e[r] = min(cstart[row + x1 + 1u], n);
            b[r] = min(cstart[row + x0], e[r]);
        }
    }
}

// Whether the wave's ranges can be laid out as a stream (uniform).
__device__ __forceinline__ bool exact_streams(const uint32_t b[3], const uint32_t e[3],
                                              uint32_t hr, bool in, int lane) {
    const uint32_t hp = (uint32_t)__shfl_up((int)hr, 1u, kWave);
    const bool same = in && lane > 0 && hp == hr;
    bool ok = !in || lane == 0 || hp <= hr;  // home rows in order: each is one run of lanes
#pragma unroll
    for (int r = 0; r < 3; r++) {
        const uint32_t bp = (uint32_t)__shfl_up((int)b[r], 1u, kWave);
        const uint32_t ep = (uint32_t)__shfl_up((int)e[r], 1u, kWave);
        ok = ok && (!same || (bp <= b[r] && ep <= e[r]));
    }
    return __ballot(!ok) == 0ull;
}

// Walks the neighbourhood of the lanes with `in` (consecutive from lane 0).  load(j): what the pass
// needs of sorted particle j beside its position (float4), store(slot, v): to window slot `slot`;
// row(p, w, m): m candidates, positions at p (12 bytes each), at window slot w on;
// one(j): a candidate in global memory.
template <class Load, class Store, class Row, class One>
__device__ __forceinline__ void exact_walk(ExactLds& lds, const float4* __restrict__ spos,
                                           uint32_t n, const GridDesc& g,
                                           const uint32_t* __restrict__ cstart, const Cell3& c,
                                           bool in, int lane, uint32_t few, Load&& load,
                                           Store&& store, Row&& row, One&& one) {
    const uint32_t hr = (uint32_t)c.cy + (uint32_t)c.cz * g.ny;
    for (int dz = -1; dz <= 1; dz++) {  // uniform
        uint32_t b[3], e[3];
        exact_ranges(c, in, g, cstart, n, dz, b, e);
        LightStream L;
        const uint32_t cand = (e[0] - b[0]) + (e[1] - b[1]) + (e[2] - b[2]);
        bool stream = n <= kExactStreamN && __ballot(cand > few) != 0ull &&
                      exact_streams(b, e, hr, in, lane);
        if (stream) {
            light_stream(L, b, e, hr, in, lane);
            const uint32_t w = wave_max(L.cnt[0] + L.cnt[1] + L.cnt[2]);
            stream = L.T <= 16u * w + 2048u;
        }
        if (!stream) {
#pragma unroll 1
            for (int r = 0; r < 3; r++)
                for (uint32_t j = b[r]; j < e[r]; j++) one(j);
            continue;
        }
        for (uint32_t w0 = 0; w0 < L.T; w0 += kExactWin) {  // uniform
            uint32_t j[kExactWin / kWave];
            window_indices<kExactWin>(L, w0, lane, j);
            float4 v[kExactWin / kWave], u[kExactWin / kWave];
#pragma unroll
            for (int k = 0; k < kExactWin / kWave; k++) {
                v[k] = spos[j[k]];
                u[k] = load(j[k]);
            }
            __builtin_amdgcn_wave_barrier();
#pragma unroll
            for (int k = 0; k < kExactWin / kWave; k++) {
                float* const o = lds.xyz + 3 * (k * kWave + lane);
                o[0] = v[k].x;
                o[1] = v[k].y;
                o[2] = v[k].z;
                store(k * kWave + lane, u[k]);
            }
            __builtin_amdgcn_wave_barrier();
#pragma unroll 1
            for (int r = 0; r < 3; r++) {  // in the reference's order
                const uint32_t S = r == 0 ? L.S[0] : (r == 1 ? L.S[1] : L.S[2]);
                const uint32_t cnt = r == 0 ? L.cnt[0] : (r == 1 ? L.cnt[1] : L.cnt[2]);
                const uint32_t jb = max(S, w0), je = min(S + cnt, w0 + (uint32_t)kExactWin);
                const uint32_t m = cnt && je > jb ? je - jb : 0u;
                row(lds.xyz + 3u * (jb - w0), jb - w0, m);
            }
            __builtin_amdgcn_wave_barrier();
        }
    }
}

// A candidate's squared distance with the reference's expressions (sph_fused.rs:594-597).
__device__ __forceinline__ float exact_r2(const float4& pi, float x, float y, float z) {
    const float djx = pi.x - x, djy = pi.y - y, djz = pi.z - z;
    return djx * djx + djy * djy + djz * djz;
}

// Which of m <= 32 candidates may lie within h: bit 31 - t for candidate t, from the sign of
// r2 - h2 (exact for every finite r2; the hit itself tests r2 again, so a NaN of either sign does
// no harm).
__device__ __forceinline__ uint32_t exact_mask(const float* __restrict__ p, uint32_t m,
                                               const float4& pi, float h2) {
    uint32_t mask = 0;
    const auto test = [&](const float* q) {
        const float d = exact_r2(pi, q[0], q[1], q[2]) - h2;
        mask = __builtin_amdgcn_alignbit(mask, __float_as_uint(d), 31);
    };
    const float* const pe = p + 3u * ((m + 3u) & ~3u);  // (up to 3 candidates past the row)
    while (p < pe) {
        test(p);
        test(p + 3);
        test(p + 6);
        test(p + 9);
        p += 12;
    }
    mask <<= (0u - m) & 28u;
    return m ? mask & ~(0x7FFFFFFFu >> (m - 1u)) : 0u;
}

// exact_walk's row for the passes with masks: hit(slot, p) for each candidate that may be within
// h, in order.
template <class Hit>
__device__ __forceinline__ void exact_hits(const float* __restrict__ p, uint32_t w, uint32_t m,
                                           const float4& pi, float h2, Hit&& hit) {
    for (uint32_t c = 0; __ballot(c < m) != 0ull; c += 32u) {  // uniform
        uint32_t mask = c < m ? exact_mask(p + 3u * c, min(m - c, 32u), pi, h2) : 0u;
        while (mask) {
            const uint32_t t = (uint32_t)__builtin_clz(mask);
            mask ^= 0x80000000u >> t;
            hit(w + c + t, p + 3u * (c + t));
        }
    }
}

// ---------------------------------------------------------------------------------------------
// Density: rho_i = sum_j mass*poly6*(h2 - r2)^3 over r2 < h2, self included.
__global__ __launch_bounds__(kWave) void k_density(const float4* __restrict__ spos,
                                                   const uint32_t* __restrict__ sidx, uint32_t n,
                                                   GridDesc g, const uint32_t* __restrict__ cstart,
                                                   float h2, float mc, float* __restrict__ srho,
                                                   float* __restrict__ density) {
    __shared__ ExactLds lds;
    const int lane = threadIdx.x;
    const uint32_t s = xcd_chunked(blockIdx.x, gridDim.x) * kWave + (uint32_t)lane;
    const bool in = s < n;
    const float4 pi = spos[in ? s : 0u];
    const Cell3 c = sph_cell(pi, g);
    float rho = 0.0f;
    // a candidate beyond h adds +0.0f, which changes no sum (they start at +0 and never become -0)
    const auto add = [&](float r2) {
        const float diff = h2 - r2;
        const float t = mc * diff * diff * diff;
        rho += r2 < h2 ? t : 0.0f;
    };
    exact_walk(
        lds, spos, n, g, cstart, c, in, lane, kExactFewDensity, [](uint32_t) { return float4{}; },
        [](int, const float4&) {},
        [&](const float* p, uint32_t, uint32_t m) {
            const float* const pu = p + 3u * (m & ~1u);
            while (p < pu) {
                const float ra = exact_r2(pi, p[0], p[1], p[2]);
                const float rb = exact_r2(pi, p[3], p[4], p[5]);
                add(ra);
                add(rb);
                p += 6;
            }
            if (m & 1u) add(exact_r2(pi, p[0], p[1], p[2]));
        },
        [&](uint32_t j) {
            const float4 q = spos[j];
            add(exact_r2(pi, q.x, q.y, q.z));
        });
    if (!in) return;
    srho[s] = rho;
    const uint32_t i = sidx[s];
    if (density && i < n) density[i] = rho;
}

hipError_t launch_density(fh_ctx* c, const SphArgs& a, const uint32_t* cell_start,
                          float* density_out) {
    if (a.n == 0) return hipSuccess;
    // Same float expressions as sph_density.rs:413-416; mass * coeff is the first product of
    // `mass * poly6_coeff * diff * diff * diff` (:453).
    float h2 = a.h * a.h;
    float h9 = h2 * h2 * h2 * h2 * a.h;
    float poly6 = 315.0f / (64.0f * 3.14159265f * h9);
    float mc = a.mass * poly6;
    tbeg(c, KID_DENSITY);
    k_density<<<ceil_div(a.n, (uint32_t)kWave), kWave, 0, c->stream>>>(
        c->spos, c->sidx, a.n, a.g, cell_start, h2, mc, c->srho, density_out);
    tend(c, KID_DENSITY);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------------------------
struct ForceConsts {
    float h, h2, mass, k, rho0, mu, gcoef, lcoef, dt;
    uint32_t flags;
    float gx, gy, gz;
    float mn[3], mx[3], e;
};

// Fused pressure + viscosity (sph_fused.rs:542-638) and the optional epilogue: gravity
// (gravity.rs:33), integrate with its non-finite guard (integrate.rs:23-29) and the box
// (box_collider.rs:37-46), written back through sidx to the caller's arrays.
// (5 waves per SIMD: left to itself the compiler takes 105 registers, for 4)
__global__ __launch_bounds__(kWave) __attribute__((amdgpu_waves_per_eu(5, 8))) void k_force(const float4* __restrict__ spos,
                                                 const float4* __restrict__ svel,
                                                 const float* __restrict__ srho,
                                                 const uint32_t* __restrict__ sidx, uint32_t n,
                                                 GridDesc g, const uint32_t* __restrict__ cstart,
                                                 ForceConsts K, float* __restrict__ px,
                                                 float* __restrict__ py, float* __restrict__ pz,
                                                 float* __restrict__ vx, float* __restrict__ vy,
                                                 float* __restrict__ vz,
                                                 float* __restrict__ accel) {
    __shared__ ExactLds lds;
    __shared__ float4 s_vr[kExactWin];  // velocity and density of the window's candidates
    const int lane = threadIdx.x;
    const uint32_t s = xcd_chunked(blockIdx.x, gridDim.x) * kWave + (uint32_t)lane;
    const bool in = s < n;
    const float4 pi = spos[in ? s : 0u];
    const float4 vi = svel[in ? s : 0u];
    const float rho_i = srho[in ? s : 0u];
    float ax = 0.0f, ay = 0.0f, az = 0.0f;
    float nvx = vi.x, nvy = vi.y, nvz = vi.z;
    const bool live = in && !(rho_i < 1e-6f);
    const float p_i = K.k * (rho_i - K.rho0);
    float pax = 0.0f, pay = 0.0f, paz = 0.0f;
    float vax = 0.0f, vay = 0.0f, vaz = 0.0f;
    const Cell3 c = sph_cell(pi, g);
    const auto pair = [&](float qx, float qy, float qz, float vjx, float vjy, float vjz,
                          float rho_j) {
        float djx = pi.x - qx;
        float djy = pi.y - qy;
        float djz = pi.z - qz;
        float r2 = djx * djx + djy * djy + djz * djz;
        if (r2 < K.h2 && r2 > 1e-12f && !(rho_j < 1e-6f)) {
            float r = sqrtf(r2);
            float diff = K.h - r;
            float p_j = K.k * (rho_j - K.rho0);
            float grad_scale = K.gcoef * diff * diff / r;
            float f_scale = -K.mass * (p_i + p_j) / (2.0f * rho_j) * grad_scale;
            pax += f_scale * djx;
            pay += f_scale * djy;
            paz += f_scale * djz;
            float lap = K.lcoef * diff;
            float v_scale = K.mu * K.mass / rho_j * lap;
            vax += v_scale * (vjx - vi.x);
            vay += v_scale * (vjy - vi.y);
            vaz += v_scale * (vjz - vi.z);
        }
    };
    exact_walk(
        lds, spos, n, g, cstart, c, in, lane, kExactFewForce,
        [&](uint32_t j) {
            const float4 v = svel[j];
            return make_float4(v.x, v.y, v.z, srho[j]);
        },
        [&](int slot, const float4& v) { s_vr[slot] = v; },
        [&](const float* p, uint32_t w, uint32_t m) {
            exact_hits(p, w, live ? m : 0u, pi, K.h2, [&](uint32_t slot, const float* q) {
                const float4 v = s_vr[slot];
                pair(q[0], q[1], q[2], v.x, v.y, v.z, v.w);
            });
        },
        [&](uint32_t j) {
            const float4 q = spos[j];
            if (live && exact_r2(pi, q.x, q.y, q.z) < K.h2) {
                const float4 v = svel[j];
                pair(q.x, q.y, q.z, v.x, v.y, v.z, srho[j]);
            }
        });
    if (!in) return;
    if (live) {
        float inv_rho = 1.0f / rho_i;
        ax = (pax + vax) * inv_rho;
        ay = (pay + vay) * inv_rho;
        az = (paz + vaz) * inv_rho;
        nvx = vi.x + ax * K.dt;
        nvy = vi.y + ay * K.dt;
        nvz = vi.z + az * K.dt;
    }
    const uint32_t i = sidx[s];
    if (i >= n) return;
    float npx = pi.x, npy = pi.y, npz = pi.z;
    if (K.flags & FH_EPI_GRAVITY) {
        nvx += K.gx * K.dt;
        nvy += K.gy * K.dt;
        nvz += K.gz * K.dt;
    }
    if (K.flags & FH_EPI_INTEGRATE) {
        if (!isfinite(nvx)) nvx = 0.0f;
        if (!isfinite(nvy)) nvy = 0.0f;
        if (!isfinite(nvz)) nvz = 0.0f;
        npx += nvx * K.dt;
        npy += nvy * K.dt;
        npz += nvz * K.dt;
    }
    if (K.flags & FH_EPI_BOX) {
        if (npx < K.mn[0]) { npx = K.mn[0]; nvx = fabsf(nvx) * K.e; }
        if (npx > K.mx[0]) { npx = K.mx[0]; nvx = -fabsf(nvx) * K.e; }
        if (npy < K.mn[1]) { npy = K.mn[1]; nvy = fabsf(nvy) * K.e; }
        if (npy > K.mx[1]) { npy = K.mx[1]; nvy = -fabsf(nvy) * K.e; }
        if (npz < K.mn[2]) { npz = K.mn[2]; nvz = fabsf(nvz) * K.e; }
        if (npz > K.mx[2]) { npz = K.mx[2]; nvz = -fabsf(nvz) * K.e; }
    }
    vx[i] = nvx;
    vy[i] = nvy;
    vz[i] = nvz;
    if (K.flags & (FH_EPI_INTEGRATE | FH_EPI_BOX)) {
        px[i] = npx;
        py[i] = npy;
        pz[i] = npz;
    }
    if (accel) {
        accel[i] = ax;
        accel[(size_t)n + i] = ay;
        accel[2 * (size_t)n + i] = az;
    }
}

hipError_t launch_force(fh_ctx* c, const SphArgs& a, const fh_epilogue* epi,
                        const uint32_t* cell_start, float* px, float* py, float* pz, float* vx,
                        float* vy, float* vz, float* accel) {
    if (a.n == 0) return hipSuccess;
    ForceConsts K;
    K.h = a.h;
    K.h2 = a.h * a.h;
    K.mass = a.mass;
    K.k = a.k;
    K.rho0 = a.rho0;
    K.mu = a.mu;
    // sph_fused.rs:552-555
    float h6 = K.h2 * K.h2 * K.h2;
    K.gcoef = -45.0f / (3.14159265f * h6);
    K.lcoef = 45.0f / (3.14159265f * h6);
    K.dt = a.dt;
    K.flags = epi ? epi->flags : 0u;
    K.gx = epi ? epi->gravity[0] : 0.0f;
    K.gy = epi ? epi->gravity[1] : 0.0f;
    K.gz = epi ? epi->gravity[2] : 0.0f;
    for (int q = 0; q < 3; q++) {
        K.mn[q] = epi ? epi->box_min[q] : 0.0f;
        K.mx[q] = epi ? epi->box_max[q] : 0.0f;
    }
    K.e = epi ? epi->restitution : 0.0f;
    tbeg(c, KID_FORCE);
    k_force<<<ceil_div(a.n, (uint32_t)kWave), kWave, 0, c->stream>>>(
        c->spos, c->svel, c->srho, c->sidx, a.n, a.g, cell_start, K, px, py, pz, vx, vy, vz, accel);
    tend(c, KID_FORCE);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------------------------
// Unfused modules (sph_pressure.rs:28-112, sph_viscosity.rs:27-106) over the caller's grid
// (cell_start[C+1], sorted_indices[n] left in the FieldSet by the density module), j == i skipped.
// The state is copied to slot order first (k_gather_grid), so that the walk is the exact passes'
// (exact_walk) instead of three scattered reads per candidate and lane; 150,001 particles: pressure
// 115 -> 51 us, viscosity 120 -> 48 us, the copy (7 us each) included.  The reference expressions are kept term by
// term (no contraction, IEEE division and square root) in the reference's order, so each velocity
// equals the CPU restatement's bit for bit.  Ranges and ids are clamped to n so a malformed grid
// cannot read out of bounds; a particle that a malformed grid holds twice is updated from one of
// its slots, one that it does not hold is walked from its own position.
struct UnfusedConsts {
    float h, h2, mass, k, rho0, mu, coef, dt;
    uint32_t n;
};

// sph_pressure.rs:34-111 (K.coef = -45 / (pi h^6)) and sph_viscosity.rs:34-105 (K.coef =
// 45 / (pi h^6)): one pass over the slots, one lane per slot.  Every neighbour's velocity is the
// copy's, the state before the pass; the particle's own in-place update goes to v.
template <bool VISC>
__global__ __launch_bounds__(kWave) __attribute__((amdgpu_waves_per_eu(5, 8))) void k_unfused(
    const float4* __restrict__ spos, const float4* __restrict__ svel,
    const float* __restrict__ srho, const uint32_t* __restrict__ sidx,
    const uint32_t* __restrict__ rank, const float* __restrict__ px, const float* __restrict__ py,
    const float* __restrict__ pz, const float* __restrict__ density, float* __restrict__ vx,
    float* __restrict__ vy, float* __restrict__ vz, const uint32_t* __restrict__ cstart,
    GridDesc g, UnfusedConsts K) {
    __shared__ ExactLds lds;
    __shared__ float4 s_vr[kExactWin];  // velocity and density of the window's candidates
    const int lane = threadIdx.x;
    const uint32_t s = xcd_chunked(blockIdx.x, gridDim.x) * kWave + (uint32_t)lane;
    const bool in = s < K.n;
    const uint32_t i = in ? sidx[s] : K.n;
    // (ranks are those of this call for every particle the grid holds)
    const bool own = i < K.n && rank[i] == s;
    float4 pi = spos[in ? s : 0u];
    float4 vi = svel[in ? s : 0u];
    float rho_i = srho[in ? s : 0u];
    float ax = 0.0f, ay = 0.0f, az = 0.0f;
    float p_i = K.k * (rho_i - K.rho0);
    const auto pair = [&](float qx, float qy, float qz, float vjx, float vjy, float vjz,
                          float rho_j) {
        float djx = pi.x - qx;
        float djy = pi.y - qy;
        float djz = pi.z - qz;
        float r2 = djx * djx + djy * djy + djz * djz;
        if (r2 < K.h2 && r2 > 1e-12f && !(rho_j < 1e-6f)) {
            float r = sqrtf(r2);
            if constexpr (VISC) {
                float lap = K.coef * (K.h - r);
                float scale = K.mu * K.mass / rho_j * lap;
                ax += scale * (vjx - vi.x);
                ay += scale * (vjy - vi.y);
                az += scale * (vjz - vi.z);
            } else {
                float diff = K.h - r;
                float p_j = K.k * (rho_j - K.rho0);
                float grad_scale = K.coef * diff * diff / r;
                float f_scale = -K.mass * (p_i + p_j) / (2.0f * rho_j) * grad_scale;
                ax += f_scale * djx;
                ay += f_scale * djy;
                az += f_scale * djz;
            }
        }
    };
    const auto update = [&](uint32_t t) {
        vx[t] = vi.x + (ax / rho_i) * K.dt;
        vy[t] = vi.y + (ay / rho_i) * K.dt;
        vz[t] = vi.z + (az / rho_i) * K.dt;
    };
    const bool live = own && !(rho_i < 1e-6f);
    exact_walk(
        lds, spos, K.n, g, cstart, sph_cell(pi, g), in, lane, kExactFewForce,
        [&](uint32_t j) {
            const float4 v = VISC ? svel[j] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            return make_float4(v.x, v.y, v.z, srho[j]);
        },
        [&](int slot, const float4& v) { s_vr[slot] = v; },
        [&](const float* p, uint32_t w, uint32_t m) {
            exact_hits(p, w, live ? m : 0u, pi, K.h2, [&](uint32_t slot, const float* q) {
                const float4 v = s_vr[slot];
                pair(q[0], q[1], q[2], v.x, v.y, v.z, v.w);
            });
        },
        [&](uint32_t j) {
            const float4 q = spos[j];
            if (live && exact_r2(pi, q.x, q.y, q.z) < K.h2) {
                const float4 v = svel[j];
                pair(q.x, q.y, q.z, v.x, v.y, v.z, srho[j]);
            }
        });
    if (live) update(i);
    // a particle that the grid does not hold (rank[s] is then no slot of it)
    const uint32_t rs = in ? rank[s] : 0u;
    if (in && !(rs < K.n && sidx[rs] == s) && !(density[s] < 1e-6f)) {
        rho_i = density[s];
        p_i = K.k * (rho_i - K.rho0);
        pi = make_float4(px[s], py[s], pz[s], 0.0f);
        vi = make_float4(vx[s], vy[s], vz[s], 0.0f);  // no slot, so no other thread writes them
        ax = ay = az = 0.0f;
        const Cell3 c = sph_cell(pi, g);
        for (int dz = -1; dz <= 1; dz++) {
            uint32_t b[3], e[3];
            exact_ranges(c, true, g, cstart, K.n, dz, b, e);
            for (int r = 0; r < 3; r++)
                for (uint32_t j = b[r]; j < e[r]; j++) {
                    const float4 q = spos[j], v = svel[j];
                    pair(q.x, q.y, q.z, v.x, v.y, v.z, srho[j]);
                }
        }
        update(s);
    }
}

hipError_t launch_unfused(fh_ctx* c, bool viscosity, const SphArgs& a, const float* px,
                          const float* py, const float* pz, float* vx, float* vy, float* vz,
                          const float* density, const uint32_t* cell_start,
                          const uint32_t* sorted_indices) {
    if (a.n == 0) return hipSuccess;
    UnfusedConsts K;
    K.h = a.h;
    K.h2 = a.h * a.h;
    K.mass = a.mass;
    K.k = a.k;
    K.rho0 = a.rho0;
    K.mu = a.mu;
    const float h6 = K.h2 * K.h2 * K.h2;  // sph_pressure.rs:47-50, sph_viscosity.rs:47-49
    K.coef = viscosity ? 45.0f / (3.14159265f * h6) : -45.0f / (3.14159265f * h6);
    K.dt = a.dt;
    K.n = a.n;
    const hipError_t e = launch_gather_grid(c, px, py, pz, vx, vy, vz, density, sorted_indices, a.n,
                                            true);
    if (e != hipSuccess) return e;
    const auto kernel = viscosity ? k_unfused<true> : k_unfused<false>;
    kernel<<<ceil_div(a.n, (uint32_t)kWave), kWave, 0, c->stream>>>(
        c->spos, c->svel, c->srho, c->sidx, c->rank, px, py, pz, density, vx, vy, vz, cell_start,
        a.g, K);
    return hipGetLastError();
}

// Copy of the grid of the last rebuild (CSR cell_start[C+1], sorted ids) into caller arrays:
// the FieldSet's u32 fields that the unfused modules read (sph_density.rs:44-74 keeps them).
__global__ __launch_bounds__(256) void k_copy_grid(const uint32_t* __restrict__ cs_in,
                                                   uint32_t cells1,
                                                   const uint32_t* __restrict__ si_in, uint32_t n,
                                                   uint32_t* __restrict__ cs_out,
                                                   uint32_t* __restrict__ si_out) {
    const uint32_t stride = gridDim.x * blockDim.x;
    for (uint32_t t = blockIdx.x * blockDim.x + threadIdx.x; t < cells1; t += stride)
        if (cs_out) cs_out[t] = cs_in[t];
    for (uint32_t t = blockIdx.x * blockDim.x + threadIdx.x; t < n; t += stride)
        if (si_out) si_out[t] = si_in[t];
}

hipError_t launch_copy_grid(fh_ctx* c, uint32_t cells, uint32_t n, uint32_t* cell_start,
                            uint32_t* sorted_indices) {
    if (!cell_start && !sorted_indices) return hipSuccess;
    uint32_t blocks = ceil_div(max(cells + 1u, n), 256u);
    if (blocks > 2048u) blocks = 2048u;
    k_copy_grid<<<blocks, 256, 0, c->stream>>>(c->cell_start, cells + 1u, c->sidx, n, cell_start,
                                               sorted_indices);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------------------------
// gravity.rs:31-34
__global__ void k_gravity(float* __restrict__ vx, float* __restrict__ vy, float* __restrict__ vz,
                          float gx, float gy, float gz, float dt, uint32_t n) {
    uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) {
        vx[i] += gx * dt;
        vy[i] += gy * dt;
        vz[i] += gz * dt;
    }
}

// integrate.rs:16-31
__global__ void k_integrate(float* __restrict__ px, float* __restrict__ py,
                            float* __restrict__ pz, float* __restrict__ vx,
                            float* __restrict__ vy, float* __restrict__ vz, float dt,
                            uint32_t n) {
    uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    float _vx = vx[i], _vy = vy[i], _vz = vz[i];
    if (!isfinite(_vx)) { _vx = 0.0f; vx[i] = 0.0f; }
    if (!isfinite(_vy)) { _vy = 0.0f; vy[i] = 0.0f; }
    if (!isfinite(_vz)) { _vz = 0.0f; vz[i] = 0.0f; }
    px[i] += _vx * dt;
    py[i] += _vy * dt;
    pz[i] += _vz * dt;
}

// box_collider.rs:26-47
__global__ void k_box(float* __restrict__ px, float* __restrict__ py, float* __restrict__ pz,
                      float* __restrict__ vx, float* __restrict__ vy, float* __restrict__ vz,
                      float mnx, float mny, float mnz, float mxx, float mxy, float mxz, float e,
                      uint32_t n) {
    uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    float x = px[i], y = py[i], z = pz[i], u = vx[i], v = vy[i], w = vz[i];
    if (x < mnx) { x = mnx; u = fabsf(u) * e; }
    if (x > mxx) { x = mxx; u = -fabsf(u) * e; }
    if (y < mny) { y = mny; v = fabsf(v) * e; }
    if (y > mxy) { y = mxy; v = -fabsf(v) * e; }
    if (z < mnz) { z = mnz; w = fabsf(w) * e; }
    if (z > mxz) { z = mxz; w = -fabsf(w) * e; }
    px[i] = x;
    py[i] = y;
    pz[i] = z;
    vx[i] = u;
    vy[i] = v;
    vz[i] = w;
}

hipError_t launch_gravity(fh_ctx* c, float* vx, float* vy, float* vz, uint32_t n, float gx,
                          float gy, float gz, float dt) {
    if (n == 0) return hipSuccess;
    k_gravity<<<ceil_div(n, 256u), 256, 0, c->stream>>>(vx, vy, vz, gx, gy, gz, dt, n);
    return hipGetLastError();
}

hipError_t launch_integrate(fh_ctx* c, float* px, float* py, float* pz, float* vx, float* vy,
                            float* vz, uint32_t n, float dt) {
    if (n == 0) return hipSuccess;
    k_integrate<<<ceil_div(n, 256u), 256, 0, c->stream>>>(px, py, pz, vx, vy, vz, dt, n);
    return hipGetLastError();
}

hipError_t launch_box(fh_ctx* c, float* px, float* py, float* pz, float* vx, float* vy,
                      float* vz, uint32_t n, const float* mn, const float* mx, float e) {
    if (n == 0) return hipSuccess;
    k_box<<<ceil_div(n, 256u), 256, 0, c->stream>>>(px, py, pz, vx, vy, vz, mn[0], mn[1], mn[2],
                                                    mx[0], mx[1], mx[2], e, n);
    return hipGetLastError();
}

}  // namespace fh
