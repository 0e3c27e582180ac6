// Which tiles of rows a workgroup of networks_fused_kernel (dense_fused.hip) takes one after the other, and where the chunks of
// the packed weights lie: what it asks for ahead of need, a tile's first rows and weights, is found from here.
#pragma once

namespace khan {

constexpr int kFusedRows = 64;      // rows of a tile
constexpr int kFusedKC = 16;        // k per chunk of the weights = one matrix instruction deep
constexpr int kFusedParts = 2;      // half-precision parts per float32 operand
constexpr int kFusedK1 = 384, kFusedN1 = 128, kFusedN2 = 128, kFusedN3 = 64;

// Packed weights: per type the six matrices one after the other (layer 1 as stored as three matrices of 128 columns),
// each chunk by chunk of 16 k as [chunk][part][column][16 k] of half precision -- what a workgroup would otherwise split again
// for every tile of rows it takes, laid out so that a chunk's part is one contiguous run that the workgroup's
// threads copy 8 bytes each.
constexpr int kPackF1 = 0;                                                          // layer 1 transposed: 128 columns x 384
constexpr int kPackF2 = kPackF1 + kFusedParts * kFusedN1 * kFusedK1;                // layer 2 transposed: 128 x 128
constexpr int kPackF3 = kPackF2 + kFusedParts * kFusedN2 * kFusedN1;                // layer 3 transposed: 64 x 128
constexpr int kPackB1 = kPackF3 + kFusedParts * kFusedN3 * kFusedN2;                // layer 1 as stored: 384 columns x 128
constexpr int kPackB2 = kPackB1 + kFusedParts * kFusedK1 * kFusedN1;                // layer 2 as stored: 128 x 128
constexpr int kPackB3 = kPackB2 + kFusedParts * kFusedN1 * kFusedN2;                // layer 3 as stored: 128 x 64
constexpr int kPackPerType = kPackB3 + kFusedParts * kFusedN2 * kFusedN3;           // 294,912 half-precision values
constexpr int kPackBytes = 4 * kPackPerType * 2;

// bytes in front of chunk c of a type's matrix at `matrix` (kPackF1 ...) of `cols` columns x K, of its columns from 128
// `column_tile` on
constexpr int packed_chunk_at(int type, int matrix, int cols, int K, int column_tile, int c)
{
    return (type * kPackPerType + matrix + column_tile * kFusedParts * 128 * K + c * kFusedParts * cols * kFusedKC) * 2;
}

struct FusedTile {
    int tile, type, row0;      // its number, its rows' type and the first of them
};
// tile_end: running sum of the types' tiles
constexpr FusedTile fused_tile(const int (&tile_end)[4], int tile)
{
    const int type = (tile >= tile_end[0]) + (tile >= tile_end[1]) + (tile >= tile_end[2]);
    return {tile, type, (tile - (type == 0 ? 0 : type == 1 ? tile_end[0] : type == 2 ? tile_end[1] : tile_end[2])) * kFusedRows};
}
// The tile that a workgroup takes after `at`, or `at` itself where there is none.  Its first rows and weights are asked for ahead
// either way.  Where there is none those loads are to give zeros without going to memory: the lanes' own offsets take them past
// the end (kFusedSkip more), because the offset that all lanes share need not count in the hardware's check of the end.  (A
// branch around them, or loading the present tile's again, costs a launch of one tile a workgroup 1.1 us of 14.)
constexpr unsigned kFusedSkip = 1u << 30;
static_assert(kFusedSkip >= kPackBytes && kFusedSkip >= kFusedRows * kFusedK1 * 4 && kFusedSkip + kPackBytes < 1u << 31,
              "past the end of any weights and of a tile's rows, without overflow");
constexpr FusedTile fused_next(const int (&tile_end)[4], const FusedTile& at, int step)
{
    return step < tile_end[3] - at.tile ? fused_tile(tile_end, at.tile + step) : at;
}

}  // namespace khan
