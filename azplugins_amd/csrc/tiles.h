// Tiled neighbor list: the full list of a block of particles (a tile)
// rewritten against the tile's own set of neighbors.
//
// A tile is a run of T = 512 or 256 columns.  Built by the per-tile walk
// (k_tile_walk.hip) the columns are the tile's cell-list slots reordered by
// list length, column s belonging to particle order[s]; built from a plain
// list (k_tiles.hip) column i is particle i.  The build collects the distinct
// neighbors of the tile's particles into jset[t][0..count[t]) and stores
// every list entry as 16 x its rank in that set (the byte offset of the
// neighbor's staged position in LDS), two entries per 32-bit word: word m of
// column s (at list[m * pitch + s]) holds entries 2m (low half) and 2m + 1
// (high half).  Columns are padded with 16 x count[t] (one past the last
// rank) up to their wavefront's longest list rounded up to 8.  The force
// kernel stages the tile's neighbor positions in LDS once (slot count[t]
// holds a dummy) and gathers from LDS, and the list stream shrinks from 4 to
// 2 bytes per entry.
#pragma once

#include <cstdint>

#include "azp_internal.h"
#include "cells.h"
#include "group_walk.h"

namespace azp
{

// Most LDS position slots per tile (distinct neighbors + the dummy slot):
// 3968 int4 = 62 KB, leaving room for the per-type-pair tables of up to 6
// types within a 64 KB workgroup allocation.
constexpr uint32_t kTileCap = 3968;

struct TileList
    {
    DeviceArray<uint32_t> count; // [ntiles]
    DeviceArray<uint32_t> jset;  // [ntiles * kTileCap]
    DeviceArray<uint32_t> list;  // [words * pitch]
    DeviceArray<uint32_t> flag;  // [0] largest distinct count above capacity, [1] largest count
    DeviceArray<uint32_t> nn;        // per-tile walk: list length of column s
    DeviceArray<uint32_t> order_buf; // per-tile walk: particle of column s
    DeviceArray<uint32_t> col;       // per-tile walk: column of particle i
    // per-tile walk, by group of 64 slots, in one allocation: how many cells
    // and batches, the candidates that any of its particles lists, its cells
    DeviceArray<uint2> groups;
    DeviceArray<uint16_t> group_rows; // the particles' rows
    // Tiles of the per-tile walk: a tile's columns are its cell-list slots
    // reordered by list length (longest first); column s belongs to particle
    // order[s] and has nn[s] entries.  Null for tiles of consecutive
    // particles (column i is particle i, counts in the list's n_neigh).
    const uint32_t* order = nullptr;
    uint32_t size = 0;           // columns per tile (0: no tiles)
    uint32_t slots = 0;          // LDS slots the force kernel needs: largest count + 1
    uint32_t ntiles = 0;
    bool valid = false;
    };

// Builds tiles of `tile_size` (256 or 512) particles from the full list in
// particle-major rows (entry k of particle i at d_rows[i * max_neighbors + k],
// max_neighbors a multiple of 8); `pitch` is the column pitch of the tiled
// list.
// Returns AZP_OK and sets t.valid when every tile fits kTileCap - 1 distinct
// neighbors; t.valid is false otherwise (the caller keeps the plain list).
// Synchronizes `stream` (reads two flag words through `h_flag`, pinned).
int tiles_build(TileList& t,
                uint32_t tile_size,
                uint32_t N,
                const uint32_t* d_n_neigh,
                const uint32_t* d_rows,
                uint32_t pitch,
                uint32_t max_neighbors,
                uint32_t* h_flag,
                hipStream_t stream);

// Flag words of a neighbor list's builds ([1] is the rebuild check, the last
// one the step kernel's).  Words 3 to 6 are the compaction's.
constexpr uint32_t kTileFlagOverflow = 0; // largest count above max_neighbors
constexpr uint32_t kTileFlagBad = 2;      // bad type (1) / position (2)
constexpr uint32_t kTileFlagMisfit = 3;   // a tile did not fit (1: cells, 2: candidates, 4: neighbor set)
constexpr uint32_t kTileFlagLargest = 4;  // largest neighbor-set size
constexpr uint32_t kTileFlagRelative = 5; // tiles tested on the matrix cores throughout
constexpr uint32_t kTileFlagTable = 6;    // most rank-table entries of a tile beyond table_cap
constexpr uint32_t kTileFlagCells = 7;    // most cells of a group beyond group_cell_cap
constexpr uint32_t kTileFlagBatches = 8;  // most batches of a group beyond group_batch_cap
constexpr uint32_t kTileFlagSpan = 9;     // sizes with a tile of more than kOwnCells cells (kTileSpan512, kTileSpan256)
constexpr uint32_t kTileFlags = 10;
constexpr uint32_t kFlagStep = kTileFlags; // the step kernel's rebuild check
constexpr uint32_t kTileSpan512 = 1, kTileSpan256 = 2;

// A tile whose slots span more cells than this (about four particles a cell
// or fewer at 512 slots) is left to the plain walk: its union outgrows the
// compaction's hash.
constexpr uint32_t kOwnCells = 128;

// Inputs and outputs of the per-tile walk (k_tile_walk.hip): the cell list
// (cell_of, members, the cell-ordered fixed-point copy) and the list radii;
// per-particle counts; the groups' rows as scratch; the slot-ordered tiled
// list as output.
struct TileWalkArgs
    {
    GroupArgs g;
    uint32_t N;
    DevBox box;
    float fx_scale[3]; // L / 2^32 per axis
    int reach[3];      // group_reach per axis
    float slip;        // group_slip
    CellGrid grid;
    const uint32_t* cell_of; // geometric cell of each particle
    uint32_t* n_neigh;       // by particle
    uint32_t max_neighbors;  // a multiple of 8
    uint32_t* flags;
    uint32_t pitch;
    uint32_t group_cell_cap, group_batch_cap, table_cap;
    uint32_t sizes; // kTileSpan512 | kTileSpan256: the tile sizes that this build may use
    // set by tiles_rows / tiles_compact
    uint2* group_cells;    // by group: first slot, first candidate | members << 16 of each cell
    uint2* group_used;     // by group and batch of 64 candidates
    uint16_t* group_rows;  // by slot: the candidate numbers of its entries
    uint2* group_meta;     // by group: cells, batches (high bit: direct tests)
    uint32_t* tile_nn;     // by column
    uint32_t* tile_order;  // particle of each column
    uint32_t* tile_col;    // column of each particle
    uint32_t* tile_count;
    uint32_t* tile_jset;
    uint32_t* tlist;
    };

// Rank-table entries (two bytes of LDS each) of a tile: with kTileTable two
// tiles share a CU (80 KiB each with the 22 KiB of the compaction's other
// arrays); a build whose tiles need more compacts again with room for them, up
// to one tile per CU.
constexpr uint32_t kTileTable = 29568;
constexpr uint32_t kTileTableMax = 69632;

// Most batches of a group the walk makes room for: a 256-column tile of four
// such groups fills the largest rank tables.
constexpr uint32_t kGroupBatchesMax = kTileTableMax / 64 / 4;
// Most cells it lists: a pass visits at most 27 for each column that it serves.
constexpr uint32_t kGroupCellsMax = 64 * 27;

// Enqueues the groups' rows (which no tile size enters) into t's arrays, sized
// here; nothing is done if the span flags rule out every size of args.sizes.
// `uniform`: one list radius for every type pair.
int tiles_rows(TileList& t, const TileWalkArgs& args, bool uniform, hipStream_t stream);

// Enqueues the tiled list with tiles of `tile_size` (256 or 512) particles from
// the rows; the caller reads args.flags afterwards and sets t.size / t.slots /
// t.valid when no misfit is flagged.
int tiles_compact(TileList& t, uint32_t tile_size, const TileWalkArgs& args, hipStream_t stream);

// Most particle types the per-tile walk serves.
constexpr uint32_t kTileWalkMaxTypes = 8;

// Enqueues the expansion of a valid tiled list of the per-tile walk into the
// plain column list (d_nlist[k * pitch + i], padding entries hold i).
int tiles_to_plain(const TileList& t, uint32_t N, const uint32_t* d_n_neigh, uint32_t pitch, uint32_t* d_nlist,
                   hipStream_t stream);

} // namespace azp
