// Tiled list straight from the cell list.  Tiles are runs of T = 512 or 256
// consecutive slots of the cell list, whose cells are stored in Morton order,
// so a tile covers a compact block of space whatever order the particles are
// in; slot s holds particle members[s].  Two kernels:
//
//   k_group_rows     one wavefront per group of 64 slots (group_walk.h): each
//                    particle's neighbors as numbers among the group's
//                    candidates, the candidates that any of them lists, and
//                    the group's cells;
//   k_tile_compact   one workgroup per tile: the union of its groups' cells
//                    (LDS hash, sorted into Morton order) numbers the tile's
//                    candidates; those that are listed get their ranks in the
//                    tile's neighbor set (jset) by a scan of their marks; a
//                    table per group turns its candidate numbers into ranks,
//                    and the columns of the tiled list are written through
//                    it, ordered by list length.
//
// A tile whose cells hold more candidates than LDS does, or whose neighbor
// set exceeds kTileCap - 1, reports it; the host then compacts the same rows
// into 256-column tiles, or uses the plain walk.
//
// 1M particles, 139 entries each: k_group_rows 0.56 ms, k_tile_compact 0.32 ms,
// against 1.27 ms for one kernel in which each lane walked its 27 cells from
// LDS and appended its hits serially (17 instructions per candidate).  The
// rows take 12,400 VALU instructions per 64 particles: 5,400 in the tests of
// 27 batches of 64 candidates, 3,500 in taking 139 entries out of the masks.
// At 60,000 particles (DPD, density 3) 46 + 37 us against 98, at 4,096 37 + 53
// against 100.
#include <type_traits>

#include "cells.h"
#include "device_common.h"
#include "group_walk.h"
#include "tiles.h"

namespace azp
{

// Candidates of one tile (two bytes of LDS each).  512-column tiles of 50
// particles a cell reach 6,600 (Yukawa, at a seventh of the system sizes), and
// must not fall to 256 columns for that: the FP64 pair kernel's workgroup is
// then 256 lanes, and one whose neighbors take more than half of the LDS has
// its CU to itself (225,000 particles, two types: 238 us against 216).  Tiles
// of colloids (7,000 to 9,500) are left to the plain walk and the hash build.
constexpr uint32_t kTileCand = 6656;
constexpr uint32_t kUnionCells = 512; // distinct non-empty cells around one tile
constexpr uint32_t kCellHash = 1024;  // open-addressing table of those cells

__device__ __forceinline__ uint32_t cell_hash(uint32_t c)
    {
    return (c * 2654435761u) >> 22; // 10 bits
    }

// Largest value over the 64 lanes of the wavefront (every lane gets it).
__device__ __forceinline__ uint32_t wave_max_u32(uint32_t v)
    {
    for (int off = 32; off > 0; off >>= 1)
        v = max(v, (uint32_t)__shfl_xor((int)v, off));
    return v;
    }

// Exclusive scan of one value per thread over the T-thread workgroup.
template<uint32_t T> __device__ __forceinline__ uint32_t tile_scan(uint32_t v, uint32_t* s_wave, uint32_t& total)
    {
    const uint32_t lane = threadIdx.x & 63u, w = threadIdx.x >> 6;
    uint32_t x = v;
    for (uint32_t off = 1; off < 64; off <<= 1)
        {
        const uint32_t y = (uint32_t)__shfl_up((int)x, off);
        if (lane >= off)
            x += y;
        }
    if (lane == 63u)
        s_wave[w] = x;
    __syncthreads();
    uint32_t base = 0, tot = 0;
    for (uint32_t k = 0; k < T / 64; ++k)
        {
        const uint32_t sw = s_wave[k];
        base += k < w ? sw : 0u;
        tot += sw;
        }
    __syncthreads();
    total = tot;
    return base + x - v;
    }

// OR over the wavefront.
__device__ __forceinline__ uint32_t wave_or(uint32_t v)
    {
    // rotations within rows of 16 lanes
    v |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x128, 0xf, 0xf, false);
    v |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x124, 0xf, 0xf, false);
    v |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x122, 0xf, 0xf, false);
    v |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x121, 0xf, 0xf, false);
    return (uint32_t)(lane_value((int)v, 0) | lane_value((int)v, 16) | lane_value((int)v, 32) | lane_value((int)v, 48));
    }

// The neighbors of each particle, by groups of 64 cell-list slots.  A column's
// mask words that are not empty wait in a ring in LDS, with the number of
// their first candidate; while some lane's ring is full, and at the end, every
// lane takes one entry per step from its own, and stores four (8 bytes) at a
// time: entries stored one by one
// to scattered rows cost a memory transaction each and took 0.4 of 0.63 ms,
// and draining whole buffers instead of keeping the ring took 0.70 ms.
constexpr uint32_t kGroupWaves = 4;
constexpr uint32_t kRowBuffer = 16; // a power of two

template<int ONEHOT> __global__ void __launch_bounds__(64 * kGroupWaves, 4) k_group_rows(const TileWalkArgs a)
    {
    __shared__ GroupLds s_group[kGroupWaves];
    __shared__ uint32_t s_mask[kGroupWaves][kRowBuffer * 64];
    __shared__ uint16_t s_first[kGroupWaves][kRowBuffer * 64];
    const uint32_t w = threadIdx.x >> 6, lane = threadIdx.x & 63u;
    const uint32_t group = xcd_logical_block() * kGroupWaves + w;
    if (group * 64u >= a.N)
        return; // the whole wavefront (no barrier below spans wavefronts)
    const uint32_t span = a.flags[kTileFlagSpan];
    GroupColumn me;
    me.slot = group * 64u + lane;
    me.valid = me.slot < a.N;
    me.i = me.valid ? a.g.members[me.slot] : 0u;
    me.cell = me.valid ? a.cell_of[me.i] : 0u;
    GroupGeom G;
#pragma unroll
    for (int k = 0; k < 3; ++k)
        {
        G.n[k] = a.grid.n[k];
        G.L[k] = a.box.L[k];
        G.Linv[k] = a.box.Linv[k];
        G.scale[k] = a.fx_scale[k];
        G.reach[k] = a.reach[k];
        }
    G.slip = a.slip;
    G.cell_base = 0u;
    me.c[0] = (int)(me.cell % (uint32_t)G.n[0]);
    me.c[1] = (int)((me.cell / (uint32_t)G.n[0]) % (uint32_t)G.n[1]);
    me.c[2] = (int)(me.cell / ((uint32_t)G.n[0] * (uint32_t)G.n[1]));
    me.fixed = a.g.cell_fixed[me.valid ? me.slot : 0u];
    if ((span & a.sizes) == a.sizes)
        return; // no tile size fits (tested here, behind the loads above)
    if (me.valid && (uint32_t)me.fixed.w >= a.g.ntypes)
        {
        const double4 p = a.g.pos[me.i];
        atomicOr(a.flags + kTileFlagBad, isfinite(p.x) && isfinite(p.y) && isfinite(p.z) ? 1u : 2u);
        }
    // cells and 64-candidate batches of the passes so far; a group that needs
    // more of either than there is room for reports it and stores nothing
    uint32_t ncell = 0, nbatch = 0, from = 0;
    uint32_t pushed = 0, taken = 0;   // words of the column put into its ring, taken from it
    uint32_t word = 0, base = 0;      // the rest of the last one taken
    uint32_t count = 0;               // entries of the column
    uint32_t four_low = 0, four_high = 0; // the last of them, the newest in the high bits
    bool room = true, direct = false;
    uint2* cells = a.group_cells + (size_t)group * a.group_cell_cap;
    uint32_t* const group_used = reinterpret_cast<uint32_t*>(a.group_used + (size_t)group * a.group_batch_cap);
    uint32_t* used = group_used;
    uint16_t* row = a.group_rows + (size_t)me.slot * a.max_neighbors;
    // one entry per lane and step until no lane's ring holds more than `keep`
    // words
    auto drain = [&](uint32_t keep, bool last) {
        while (__ballot(pushed - taken > keep || (last && word != 0u)) != 0ull)
            {
            const uint32_t at = (taken & (kRowBuffer - 1u)) * 64u + lane;
            const uint32_t v = s_mask[w][at], n = s_first[w][at];
            const bool advance = word == 0u && taken != pushed;
            word = advance ? v : word;
            base = advance ? n : base;
            taken += advance ? 1u : 0u;
            if (word != 0u)
                {
                const uint32_t entry = base + (uint32_t)__builtin_ctz(word);
                word &= word - 1u;
                four_low = __builtin_amdgcn_alignbit(four_high, four_low, 16);
                four_high = __builtin_amdgcn_alignbit(entry, four_high, 16);
                ++count;
                if ((count & 3u) == 0u && count <= a.max_neighbors)
                    *reinterpret_cast<uint2*>(row + count - 4u) = make_uint2(four_low, four_high);
                }
            }
    };
    auto begin = [&](uint32_t n, uint32_t total) {
        const uint32_t batches = (total + 63u) / 64u;
        room = room && ncell + n <= a.group_cell_cap && nbatch + batches <= a.group_batch_cap;
        if (room)
            for (uint32_t k = lane; k < n; k += 64)
                {
                const uint32_t first = s_group[w].first[k];
                const uint32_t next = k + 1 < n ? s_group[w].first[k + 1] : total;
                cells[ncell + k] = make_uint2(s_group[w].delta[k] + first, (first + nbatch * 64u) | ((next - first) << 16));
                }
        used = group_used + nbatch * 2u;
        from = nbatch * 64u;
        ncell += n;
        nbatch += batches;
    };
    auto emit = [&](uint32_t low, uint32_t high, uint32_t P, uint32_t, uint32_t) {
        if (!room)
            {
            count += (uint32_t)(__popc(low) + __popc(high));
            return;
            }
        const uint32_t any_low = wave_or(low), any_high = wave_or(high);
        if (lane < 2u)
            used[(P >> 5) + lane] = lane == 0u ? any_low : any_high;
        // room for two words (a lane reads back only what it wrote itself)
        drain(kRowBuffer - 2u, false);
        if (low != 0u)
            {
            const uint32_t at = (pushed++ & (kRowBuffer - 1u)) * 64u + lane;
            s_mask[w][at] = low;
            s_first[w][at] = (uint16_t)(from + P);
            }
        if (high != 0u)
            {
            const uint32_t at = (pushed++ & (kRowBuffer - 1u)) * 64u + lane;
            s_mask[w][at] = high;
            s_first[w][at] = (uint16_t)(from + P + 32u);
            }
    };
    uint64_t todo = __ballot(me.valid);
    while (todo != 0ull)
        todo &= ~group_pass<ONEHOT, false>(a.g, G, s_group[w], me, todo, group_anchor(todo), true, direct, begin, emit);
    drain(0u, true);
    // the entries after the last whole four
    if (me.valid && room && (count & 3u) != 0u && count <= a.max_neighbors)
        {
        const uint64_t four = ((uint64_t)four_high << 32 | four_low) >> (16u * (4u - (count & 3u)));
        *reinterpret_cast<uint2*>(row + (count & ~3u)) = make_uint2((uint32_t)four, (uint32_t)(four >> 32));
        }
    if (me.valid)
        {
        // a list longer than the capacity is truncated (and reported), so
        // consumers never read past the allocation
        a.n_neigh[me.i] = min(count, a.max_neighbors);
        if (count > a.max_neighbors)
            atomicMax(a.flags + kTileFlagOverflow, count);
        }
    if (lane == 0)
        {
        a.group_meta[group] = room ? make_uint2(ncell, nbatch | (direct ? 0x80000000u : 0u)) : make_uint2(0u, 0u);
        if (!room)
            {
            atomicMax(a.flags + kTileFlagCells, ncell);
            atomicMax(a.flags + kTileFlagBatches, nbatch);
            }
        }
    }

// Distinct neighbors, ranks and columns of each tile.
template<uint32_t T> __global__ void __launch_bounds__(T, T == 512 ? 4 : 2) k_tile_compact(const TileWalkArgs a)
    {
    constexpr uint32_t C = kTileCand;
    constexpr uint32_t G = T / 64u, NW = T / 64u;
    // hash of the union's cells: first slots, then (u16) candidate numbers;
    // the column sort's three arrays once the ranks are known
    __shared__ uint32_t s_hash[kCellHash + kCellHash / 2];
    __shared__ uint32_t s_gs[kUnionCells];      // first slot of each union cell
    __shared__ uint16_t s_off[kUnionCells + 2]; // its first candidate number
    __shared__ uint16_t s_mark[C];
    extern __shared__ uint64_t s_ucell[]; // union cells until the rank tables take their place
    __shared__ uint32_t s_wave[NW], s_nc[G], s_nb[G], s_base[G + 1];
    __shared__ uint32_t s_n, s_bad, s_direct;
    uint32_t* s_key = s_hash;
    uint16_t* s_val = reinterpret_cast<uint16_t*>(s_hash + kCellHash);
    uint16_t* s_table = reinterpret_cast<uint16_t*>(s_ucell);

    const uint32_t span = a.flags[kTileFlagSpan];
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
    const uint32_t t = xcd_logical_block();
    const uint32_t slot = t * T + tid;
    const bool active = slot < a.N;
    const uint32_t g0 = t * G, ng = min(G, (a.N + 63u) / 64u - g0);
    const uint32_t i = active ? a.g.members[slot] : 0u;

    // most tiles' candidates; the places after them are cleared where needed
    constexpr uint32_t kMarks = 12u * 512u;
    for (uint32_t k = tid; k < kCellHash; k += T)
        s_key[k] = 0xffffffffu;
    for (uint32_t k = tid; k < kMarks; k += T)
        s_mark[k] = 0u;
    if (tid == 0)
        s_n = s_bad = s_direct = 0u;
    __syncthreads();
    if (tid < ng)
        {
        const uint2 m = a.group_meta[g0 + tid];
        s_nc[tid] = m.x;
        s_nb[tid] = m.y & 0x7fffffffu;
        if (m.y & 0x80000000u)
            s_direct = 1u;
        }
    if (span & (T == 512u ? kTileSpan512 : kTileSpan256))
        return; // a tile of this size spans too many cells: the host sees the flag
    __syncthreads();
    if (tid == 0)
        {
        uint32_t b = 0;
        for (uint32_t g = 0; g < ng; ++g)
            {
            s_base[g] = b;
            b += s_nb[g] * 64u;
            }
        s_base[ng] = b;
        }
    // 1. the distinct cells of the groups
    for (uint32_t g = wave; g < ng; g += NW)
        for (uint32_t k = lane; k < s_nc[g]; k += 64)
            {
            const uint2 c = a.group_cells[(size_t)(g0 + g) * a.group_cell_cap + k];
            uint32_t hs = cell_hash(c.x), p = 0;
            for (; p < kCellHash; ++p)
                {
                const uint32_t prev = atomicCAS(&s_key[hs], 0xffffffffu, c.x);
                if (prev == 0xffffffffu)
                    {
                    const uint32_t u = atomicAdd(&s_n, 1u);
                    if (u < kUnionCells)
                        s_ucell[u] = ((uint64_t)c.x << 32) | (hs << 16) | (c.y >> 16);
                    break;
                    }
                if (prev == c.x)
                    break;
                hs = (hs + 1u) & (kCellHash - 1u);
                }
            if (p == kCellHash)
                s_bad = 1u;
            }
    __syncthreads();
    const uint32_t U = s_n, entries = s_base[ng];
    // every thread leaves together: the conditions are shared
    const uint32_t misfit = ((s_bad != 0u || U > kUnionCells) ? 1u : 0u) | (entries > kTileTableMax ? 2u : 0u);
    if (misfit != 0u || U == 0u || entries > a.table_cap)
        {
        if (tid == 0)
            {
            if (misfit == 0u && U != 0u)
                atomicMax(a.flags + kTileFlagTable, entries);
            atomicOr(a.flags + kTileFlagMisfit, misfit);
            a.tile_count[t] = 0u;
            }
        return;
        }

    // 2. in Morton order (ascending first slot): bitonic sort over the next
    // power of two
    uint32_t P2 = 1;
    while (P2 < U)
        P2 <<= 1;
    for (uint32_t k = U + tid; k < P2; k += T)
        s_ucell[k] = ~0ull;
    __syncthreads();
    if (P2 <= T)
        {
        // one key per thread; stages with a stride below 64 exchange keys
        // within the wavefront (no barrier), the others through LDS
        uint64_t key = tid < P2 ? s_ucell[tid] : ~0ull;
        for (uint32_t size = 2; size <= P2; size <<= 1)
            for (uint32_t stride = size >> 1; stride > 0; stride >>= 1)
                {
                uint64_t other;
                if (stride >= 64u)
                    {
                    __syncthreads();
                    if (tid < P2)
                        s_ucell[tid] = key;
                    __syncthreads();
                    other = tid < P2 ? s_ucell[tid ^ stride] : ~0ull;
                    }
                else
                    {
                    const uint32_t lo = (uint32_t)__shfl_xor((int)(uint32_t)key, (int)stride);
                    const uint32_t hi = (uint32_t)__shfl_xor((int)(uint32_t)(key >> 32), (int)stride);
                    other = ((uint64_t)hi << 32) | lo;
                    }
                // ascending blocks keep the smaller key at the lower position
                const bool lower = (tid & stride) == 0u, up = (tid & size) == 0u;
                key = (lower == up) ? min(key, other) : max(key, other);
                }
        __syncthreads();
        if (tid < P2)
            s_ucell[tid] = key;
        __syncthreads();
        }
    else
        {
        for (uint32_t size = 2; size <= P2; size <<= 1)
            for (uint32_t stride = size >> 1; stride > 0; stride >>= 1)
                {
                for (uint32_t e = tid; e < P2; e += T)
                    {
                    const uint32_t p = e ^ stride;
                    if (p > e)
                        {
                        const bool up = (e & size) == 0u;
                        const uint64_t x = s_ucell[e], y = s_ucell[p];
                        if ((x > y) == up)
                            {
                            s_ucell[e] = y;
                            s_ucell[p] = x;
                            }
                        }
                    }
                __syncthreads();
                }
        }

    // 3. candidate numbers
    constexpr uint32_t QC = kUnionCells / T;
    uint64_t cell[QC];
    uint32_t sum = 0;
#pragma unroll
    for (uint32_t q = 0; q < QC; ++q)
        {
        const uint32_t u = tid * QC + q;
        cell[q] = u < U ? s_ucell[u] : 0ull;
        sum += (uint32_t)cell[q] & 0xffffu;
        }
    uint32_t Mc;
    uint32_t run = tile_scan<T>(sum, s_wave, Mc);
    if (Mc > C)
        {
        if (tid == 0)
            {
            atomicOr(a.flags + kTileFlagMisfit, 2u);
            a.tile_count[t] = 0u;
            }
        return; // Mc is the same for every thread
        }
#pragma unroll
    for (uint32_t q = 0; q < QC; ++q)
        {
        const uint32_t u = tid * QC + q;
        if (u < U)
            {
            s_gs[u] = (uint32_t)(cell[q] >> 32);
            s_off[u] = (uint16_t)run;
            s_val[((uint32_t)cell[q] >> 16) & (kCellHash - 1u)] = (uint16_t)run;
            run += (uint32_t)cell[q] & 0xffffu;
            }
        }
    if (tid == 0)
        s_off[U] = (uint16_t)Mc;
    if (Mc > kMarks)
        for (uint32_t k = kMarks + tid; k < C; k += T)
            s_mark[k] = 0u;
    __syncthreads();

    // 4. each group's candidates by tile candidate number: a wavefront a
    // group, 16 lanes a cell, the next cell read ahead
    {
    const uint32_t g = min(wave, ng - 1u);
    const uint32_t n = wave < ng ? s_nc[g] : 0u;
    const uint2* src = a.group_cells + (size_t)(g0 + g) * a.group_cell_cap;
    uint32_t k = lane >> 4;
    uint2 next = k < n ? src[k] : make_uint2(0u, 0u);
    for (; k < n; k += 4u)
        {
        const uint2 c = next;
        if (k + 4u < n)
            next = src[k + 4u];
        uint32_t hs = cell_hash(c.x);
        while (s_key[hs] != c.x) // every cell was inserted
            hs = (hs + 1u) & (kCellHash - 1u);
        const uint32_t o = s_val[hs], first = s_base[g] + (c.y & 0xffffu), m = c.y >> 16;
        for (uint32_t q = tid & 15u; q < m; q += 16u)
            s_table[first + q] = (uint16_t)(o + q);
        }
    }
    __syncthreads();
    // 5. marks of the listed ones: a wavefront a group, two words (64
    // candidates) at a time, 64 words read at once
    {
    const uint32_t g = min(wave, ng - 1u);
    const uint32_t n = wave < ng ? 2u * s_nb[g] : 0u;
    const uint32_t* src = reinterpret_cast<const uint32_t*>(a.group_used + (size_t)(g0 + g) * a.group_batch_cap);
    for (uint32_t q0 = 0; q0 < n; q0 += 64u)
        {
        const uint32_t mine = q0 + lane < n ? src[q0 + lane] : 0u;
        const uint32_t m = min(64u, n - q0);
        for (uint32_t q = 0; q < m; q += 2u)
            {
            const uint32_t word = (uint32_t)__shfl((int)mine, (int)(q + (lane >> 5)));
            if ((word >> (lane & 31u)) & 1u)
                s_mark[s_table[s_base[g] + (q0 + q) * 32u + lane]] = 1u;
            }
        }
    }
    __syncthreads();
    // 6. ranks: exclusive scan of the marks, a run of them per thread; the
    // neighbor set
    uint32_t M = 0;
    auto rank = [&](auto per_thread) {
        constexpr uint32_t QM = decltype(per_thread)::value;
        uint32_t msum = 0;
#pragma unroll
        for (uint32_t q = 0; q < QM; ++q)
            msum += s_mark[tid * QM + q];
        uint32_t r = tile_scan<T>(msum, s_wave, M);
        if (M > kTileCap - 1)
            return;
        // the union cell of the thread's first candidate, then onwards
        uint32_t lo = 0, hi = U;
        while (hi - lo > 1u)
            {
            const uint32_t mid = (lo + hi) >> 1;
            if (s_off[mid] <= tid * QM)
                lo = mid;
            else
                hi = mid;
            }
#pragma unroll
        for (uint32_t q = 0; q < QM; ++q)
            {
            const uint32_t m = tid * QM + q;
            while (lo + 1u < U && s_off[lo + 1u] <= m)
                ++lo;
            if (s_mark[m] != 0u)
                {
                a.tile_jset[(size_t)t * kTileCap + r] = a.g.members[s_gs[lo] + (m - s_off[lo])];
                s_mark[m] = (uint16_t)(r << 4); // entries are 16 x rank
                ++r;
                }
            }
    };
    if (Mc <= kMarks)
        rank(std::integral_constant<uint32_t, kMarks / T>{});
    else
        rank(std::integral_constant<uint32_t, C / T>{});
    if (M > kTileCap - 1)
        {
        if (tid == 0)
            {
            atomicOr(a.flags + kTileFlagMisfit, 4u);
            a.tile_count[t] = 0u;
            }
        return; // M is the same for every thread
        }
    if (tid == 0)
        {
        a.tile_count[t] = M;
        atomicMax(a.flags + kTileFlagLargest, M);
        if (s_direct == 0u)
            atomicAdd(a.flags + kTileFlagRelative, 1u);
        }
    __syncthreads();
    // 7. the tables hold ranks from here on (places past a pass's last
    // candidate are never read: no mask has their bits)
    for (uint32_t x = tid; x < entries; x += T)
        s_table[x] = s_mark[min((uint32_t)s_table[x], C - 1u)];

    // 8. columns ordered by list length (longest first, ties by slot), so the
    // pair kernel's 64-lane wavefronts run lists of nearly equal length: a
    // bitonic sort of (length, slot) keys, one per thread, whose stages with
    // a stride below 64 exchange keys within the wavefront (no barrier)
    const uint32_t nn = active ? a.n_neigh[i] : 0u;
    uint32_t* s_sort = s_hash;
    uint32_t* s_who = s_sort + T;
    uint32_t* s_len = s_who + T;
    static_assert(3 * T <= kCellHash + kCellHash / 2, "the sort's arrays fit the hash's space");
    s_who[tid] = i;
    s_len[tid] = nn;
    uint32_t key = (min(nn, 0xffffu) << 16) | (0xffffu - tid);
    for (uint32_t size = 2; size <= T; size <<= 1)
        for (uint32_t stride = size >> 1; stride > 0; stride >>= 1)
            {
            uint32_t other;
            if (stride >= 64u)
                {
                __syncthreads();
                s_sort[tid] = key;
                __syncthreads();
                other = s_sort[tid ^ stride];
                }
            else
                other = (uint32_t)__shfl_xor((int)key, (int)stride);
            // the lower position of a pair keeps the larger key in a
            // descending block, the smaller in an ascending one
            const bool lower = (tid & stride) == 0u, down = (tid & size) == 0u;
            key = (lower == down) ? max(key, other) : min(key, other);
            }
    // column t T + tid holds the slot of the tid-th key: its writer is this
    // thread, so consecutive lanes store consecutive columns
    const uint32_t cslot = 0xffffu - (key & 0xffffu);
    __syncthreads();
    const uint32_t ci = s_who[cslot], cnn = s_len[cslot];
    const bool cactive = t * T + cslot < a.N;
    // the column wavefront's longest list, padded to whole steps of 8
    const uint32_t P = (wave_max_u32(cactive ? cnn : 0u) + 7u) & ~7u;
    if (!cactive)
        return;
    const uint32_t col = t * T + tid;
    a.tile_nn[col] = cnn;
    a.tile_order[col] = ci;
    a.tile_col[ci] = col;
    // 9. entries, two a word; the row is read in 16-byte chunks (8 entries),
    // four in flight.  A group without room stored no rows (its build is
    // repeated).
    const uint32_t g = cslot >> 6;
    const uint32_t have = s_nb[g] != 0u ? cnn : 0u;
    const uint16_t* tab = s_table + s_base[g];
    const uint4* row = reinterpret_cast<const uint4*>(a.group_rows + (size_t)(t * T + cslot) * a.max_neighbors);
    auto chunk_load = [&](uint32_t kc) { return kc < have ? row[kc / 8] : make_uint4(0u, 0u, 0u, 0u); };
    auto rank_of_entry = [&](uint32_t k, uint32_t word, uint32_t half) {
        return k < have ? (uint32_t)tab[(word >> (16u * half)) & 0xffffu] : M << 4; // 16 x rank
    };
    auto chunk_store = [&](uint32_t kc, uint4 ch) {
        if (kc >= P)
            return;
        const uint32_t w4[4] = {ch.x, ch.y, ch.z, ch.w};
#pragma unroll
        for (uint32_t w = 0; w < 4; ++w)
            a.tlist[(size_t)((kc >> 1) + w) * a.pitch + col]
                = rank_of_entry(kc + 2 * w, w4[w], 0u) | (rank_of_entry(kc + 2 * w + 1, w4[w], 1u) << 16);
    };
    for (uint32_t k0 = 0; k0 < P; k0 += 32)
        {
        const uint4 c0 = chunk_load(k0), c1 = chunk_load(k0 + 8);
        const uint4 c2 = chunk_load(k0 + 16), c3 = chunk_load(k0 + 24);
        chunk_store(k0, c0);
        chunk_store(k0 + 8, c1);
        chunk_store(k0 + 16, c2);
        chunk_store(k0 + 24, c3);
        }
    }

// Plain column list from a tiled list of the per-tile walk: lane i (a
// particle) reads its column tile_col[i]; entry k is jset[tile][rank],
// padding entries hold i up to the longest list of the 64 particles rounded
// up to 8.
__global__ void __launch_bounds__(64) k_tiles_to_plain(uint32_t N,
                                                       const uint32_t* __restrict__ n_neigh,
                                                       const uint32_t* __restrict__ tile_col,
                                                       uint32_t tile_size,
                                                       const uint32_t* __restrict__ tile_jset,
                                                       const uint32_t* __restrict__ tlist,
                                                       uint32_t pitch,
                                                       uint32_t* __restrict__ nlist)
    {
    const uint32_t i = blockIdx.x * 64u + threadIdx.x;
    const bool active = i < N;
    const uint32_t nn = active ? n_neigh[i] : 0u;
    uint32_t wmax = nn;
    for (int off = 32; off > 0; off >>= 1)
        wmax = max(wmax, (uint32_t)__shfl_xor((int)wmax, off));
    const uint32_t P = (wmax + 7u) & ~7u;
    if (!active)
        return;
    const uint32_t s = tile_col[i];
    const uint32_t* js = tile_jset + (size_t)(s / tile_size) * kTileCap;
    for (uint32_t k = 0; k < P; k += 2)
        {
        uint32_t w = 0;
        if (k < nn)
            w = tlist[(size_t)(k >> 1) * pitch + s];
        nlist[(size_t)k * pitch + i] = k < nn ? js[(w & 0xffffu) >> 4] : i;
        nlist[(size_t)(k + 1) * pitch + i] = k + 1 < nn ? js[w >> 20] : i;
        }
    }

// The launch arguments with t's arrays.
static TileWalkArgs tile_args(const TileList& t, const TileWalkArgs& args)
    {
    TileWalkArgs a = args;
    a.tile_nn = t.nn.ptr;
    a.tile_order = t.order_buf.ptr;
    a.tile_col = t.col.ptr;
    a.tile_count = t.count.ptr;
    a.tile_jset = t.jset.ptr;
    a.tlist = t.list.ptr;
    const size_t groups = ((size_t)args.N + 63) / 64;
    a.group_meta = t.groups.ptr;
    a.group_used = a.group_meta + groups;
    a.group_cells = a.group_used + groups * args.group_batch_cap;
    a.group_rows = t.group_rows.ptr;
    return a;
    }

int tiles_rows(TileList& t, const TileWalkArgs& args, bool uniform, hipStream_t s)
    {
    if (args.g.ntypes == 0 || args.g.ntypes > kTileWalkMaxTypes)
        return set_error(AZP_ERR_UNSUPPORTED, "the per-tile walk serves 1 to %u particle types", kTileWalkMaxTypes);
    const size_t groups = ((size_t)args.N + 63) / 64;
    AZP_TRY(t.groups.reserve(groups * (1 + (size_t)args.group_batch_cap + args.group_cell_cap)));
    AZP_TRY(t.group_rows.reserve((size_t)args.N * args.max_neighbors));
    const TileWalkArgs a = tile_args(t, args);
    const dim3 grid(grid_for(groups, kGroupWaves)), block(64 * kGroupWaves);
    if (uniform)
        hipLaunchKernelGGL(k_group_rows<0>, grid, block, 0, s, a);
    else if (a.g.ntypes <= 2)
        hipLaunchKernelGGL(k_group_rows<1>, grid, block, 0, s, a);
    else
        hipLaunchKernelGGL(k_group_rows<4>, grid, block, 0, s, a);
    AZP_LAUNCH_CHECK();
    return AZP_OK;
    }

int tiles_compact(TileList& t, uint32_t tile_size, const TileWalkArgs& args, hipStream_t s)
    {
    if (tile_size != 256 && tile_size != 512)
        return set_error(AZP_ERR_INVALID, "tile size %u must be 256 or 512", tile_size);
    if (args.table_cap < kTileTable || args.table_cap > kTileTableMax)
        return set_error(AZP_ERR_INVALID, "rank tables of %u entries", args.table_cap);
    const uint32_t ntiles = (args.N + tile_size - 1) / tile_size;
    const uint32_t words = (((args.max_neighbors + 7u) & ~7u) + 1u) / 2u;
    AZP_TRY(t.count.reserve(ntiles));
    AZP_TRY(t.jset.reserve((size_t)ntiles * kTileCap));
    AZP_TRY(t.list.reserve((size_t)words * args.pitch));
    AZP_TRY(t.nn.reserve(args.N));
    AZP_TRY(t.order_buf.reserve(args.N));
    AZP_TRY(t.col.reserve(args.N));
    const TileWalkArgs a = tile_args(t, args);
    // gfx950 gives a workgroup 160 KiB of LDS; the largest size on every launch
    // (a host-side attribute, no device work), so threads agree on it
    const size_t lds = (size_t)a.table_cap * sizeof(uint16_t);
    const void* kernel = tile_size == 512 ? reinterpret_cast<const void*>(&k_tile_compact<512>)
                                          : reinterpret_cast<const void*>(&k_tile_compact<256>);
    AZP_HIP(hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)(kTileTableMax * sizeof(uint16_t))));
    if (tile_size == 512)
        hipLaunchKernelGGL(k_tile_compact<512>, dim3(ntiles), dim3(512), lds, s, a);
    else
        hipLaunchKernelGGL(k_tile_compact<256>, dim3(ntiles), dim3(256), lds, s, a);
    AZP_LAUNCH_CHECK();
    t.ntiles = ntiles;
    t.order = t.order_buf.ptr;
    return AZP_OK;
    }

int tiles_to_plain(const TileList& t, uint32_t N, const uint32_t* d_n_neigh, uint32_t pitch, uint32_t* d_nlist,
                   hipStream_t s)
    {
    if (N == 0)
        return AZP_OK;
    if (!t.valid || !t.order)
        return set_error(AZP_ERR_STATE, "no tiled list of the per-tile walk to expand");
    hipLaunchKernelGGL(k_tiles_to_plain, dim3((N + 63) / 64), dim3(64), 0, s, N, d_n_neigh, t.col.ptr, t.size,
                       t.jset.ptr, t.list.ptr, pitch, d_nlist);
    AZP_LAUNCH_CHECK();
    return AZP_OK;
    }

} // namespace azp
