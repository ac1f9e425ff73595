// Order of a packed matrix [N, K].  A feature tile (16 features) is a row of units of 1 KiB, 64 lanes of 16 bytes each: a k-step of 32 columns in
// bf16, two of e4m3, four of MXFP4.  Tiles lie in groups of 16 (256 features), and in a group blocks of two units do, tile by tile: the tiles' first blocks,
// their second ones, and so on.  Waves go through their tiles side by side, and what they ask for at a time is then a run of bytes, which is spread evenly over
// the memory channels; with whole tiles behind one another it is pieces 64 or 128 KiB apart, many of them of the same channels.  MI355X, reads alone of 67, 134
// and 235 MB by 1024 to 2048 waves: whole tiles 13.1, 24.3 and 36.9 us, groups of 16 12.3, 21.7 and 35.4 (of all tiles 12.0, 21.5 and 35.2, but then a panel's
// bytes lie all over the matrix).  Products of 16 rows and 16384 x 2048, 2048 x 8192: 14.6 -> 13.2, 9.5 -> 7.7 us; of 32 rows and 28672 x 4096, 4096 x 4096
// 39.4 -> 37.0, 9.2 -> 7.7.
// Matrices whose features or units do not come out even lie tile by tile, and so does MXFP4, a quarter of the bytes for as many columns: in groups of 16, products of 32 rows and
// 28672 x 4096 21.3 -> 23.0 us, of 16 rows and 6144 x 4096 10.4 -> 11.3; all matrices of an 8B or 1B layer together 0 to 2 % slower for 16 to 200 rows (e4m3 0 to 5 % faster).
#pragma once

constexpr int FRAG_GROUP = 16, FRAG_BLOCK = 2;

__host__ __device__ inline bool frag_grouped(long long N, int units, bool mxfp4) { return !mxfp4 && N % (16 * FRAG_GROUP) == 0 && units % FRAG_BLOCK == 0; }  // units: of a tile
// the place of a tile's first unit
__host__ __device__ inline long long frag_first(int tile, int units, bool grouped) {
  const unsigned int t = (unsigned int)tile;
  return grouped ? (long long)(t / FRAG_GROUP) * FRAG_GROUP * units + t % FRAG_GROUP * FRAG_BLOCK : (long long)t * units;
}
__host__ __device__ inline int frag_next(int units, bool grouped) { return grouped ? FRAG_BLOCK : units; }                       // from a tile's to the next one's, inside a group
__host__ __device__ inline int frag_stride(bool grouped) { return grouped ? FRAG_GROUP * FRAG_BLOCK : FRAG_BLOCK; }              // from a block to a tile's next one
// of unit u, behind the tile's first
__host__ __device__ inline long long frag_behind(int u, bool grouped) { return (long long)((unsigned int)u / FRAG_BLOCK) * frag_stride(grouped) + (unsigned int)u % FRAG_BLOCK; }
