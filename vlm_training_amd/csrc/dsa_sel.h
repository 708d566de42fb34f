// Blocks of rows staged in LDS whole and read row by row as lists name them (the compacted walks: dsa_tile_sel.hip, dsa_tile_selkv.hip).
#pragma once
#include "dsa_tile.h"

#define SEL_LOADERS 8                                    // waves that request them
// A block lies in groups of four rows, 1 KiB each, which one wave load fills: [64-byte column g of the row][row of the group][16-byte chunk
// w ^ x].  What a read adds for its column is an immediate.  x goes 0, 2, 3, 1 with the group's number modulo 4, so that each of these covers the
// 64 banks once: rows of different classes r & 15 at one chunk (row-wise operand of 32x32 tiles: a phase of a 16-byte read takes lanes 0-3, 12-15,
// 20-23, 24-27 or 4-11, 16-19, 28-31 of a half wave) or, of 16x16 tiles, sixteen of them at two neighbouring chunks; four rows of different
// r & 3 at four neighbouring chunks (transposed operand), or eight of two groups next to each other at two.
template <int ROWS>
struct SelBlock {
    static constexpr int D = 128, ROW_B = 2 * D, BYTES = ROWS * ROW_B;
    static constexpr int LOAD_ROWS = 1024 / ROW_B, LOADS = BYTES / 1024, LPW = LOADS / SEL_LOADERS;   // wave loads of a block
    static_assert(LOADS % SEL_LOADERS == 0 && SEL_LOADERS * LOAD_ROWS % 16 == 0, "a wave's loads are of rows of the same classes");
    __host__ __device__ static constexpr int mix(int group) { return (group ^ group >> 1) & 1 ? 2 | group >> 1 : group >> 1; }
    // of wave load p, the row a lane loads and its chunk
    __device__ __forceinline__ static int load_row(int p, int lane) { return p * LOAD_ROWS + (lane >> 2 & 3); }
    __device__ __forceinline__ static int load_chunk(int p, int lane) { return (lane >> 4) * 4 + ((lane & 3) ^ mix(p & 3)); }
    // where chunk 0 of row r lies; chunk 4 g + w of it: (entry(r) ^ (w << 4)) + COLUMN_B * g
    static constexpr int COLUMN_B = 256;
    __device__ __forceinline__ static int entry(int r) { return (r >> 2) * 1024 + (r & 3) * 64 + mix(r >> 2 & 3) * 16; }
};
// (may_alias: a list's entries are written as words and read by halves)
template <class T> __device__ __forceinline__ T lds_read(uint32_t at) {
    typedef T __attribute__((may_alias)) any;
    return *(__attribute__((address_space(3))) const any *)at;
}

