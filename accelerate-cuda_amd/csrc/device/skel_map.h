/*
 * skel_map.h -- map / zipWith / generate / transform / backpermute.
 *
 * Takes the place of CodeGen/Mapping.hs:39-78 (map), CodeGen/IndexSpace.hs:47-83
 * (generate) and :96-141 (transform; backpermute is transform with the identity
 * function, CodeGen.hs:101).  After fusion all of them are "for every linear
 * index ix of the result, out[ix] = get(ix)", where `get` is the generated
 * fragment (an element function applied to delayed inputs, an index
 * permutation followed by a read, or a pure function of the index), so one
 * template serves the three entry points.
 *
 * Each thread handles ACC_UNROLL groups of ACC_VEC consecutive elements; a
 * full tile runs without bounds checks so that reads of manifest arrays and
 * the writes merge into 128-bit accesses, and the ACC_UNROLL independent
 * groups keep several of them in flight per lane.
 *
 * Generated definitions expected: ACC_ENTRY, ACC_ELT, ACC_ENV_PARAMS,
 * ACC_ENV_ASSUME, ACC_OUT_PARAMS, ACC_OUT_SIZE, ACC_GET(ix), ACC_BLOCK, ACC_VEC,
 * ACC_UNROLL, ACC_ALIGNED.
 */

#define ACC_TILE (ACC_BLOCK * ACC_VEC * ACC_UNROLL)

#ifndef ACC_MAP_TILED
#define ACC_MAP_TILED 0
#endif

#if ACC_MAP_TILED
/*
 * The same result produced in square tiles of its two innermost dimensions (ACC_FLAG_TILED, rank >= 2), for element
 * functions that read their sources ACROSS rows -- a transposing backpermute above all, where a run of consecutive
 * result elements reads one element of as many source rows (IndexSpace.hs:96-141 evaluates in runs whatever the
 * index function does).  A wave takes a tile of 32 x 32 elements, its lanes 8 across and 8 down with a block of 4 x 4
 * each: a row of the tile is written in a run of 128 bytes (Float32), and a source read along the tile's columns is
 * read in runs of 128 bytes too (the four elements a lane reads down a column are consecutive there, and so are the
 * eight lanes below one another).  (A workgroup that evaluates a tile of 64 x 64 down its columns, passes it through
 * LDS and writes it along its rows in runs of 256 bytes, lines in two pieces where they are, transposes no faster, and
 * neither do lanes with blocks of 8 x 8 or 2 x 2: 5003 x 3001 Float32 in 40 and 36 us against 31; whole lines do, below.)
 *
 * What bounds it: the memory side, once the index arithmetic is out of the way.  The place of every element is known
 * here before the fragment asks for it, so the compiler is told what `ix % shOut_0` and `ix / shOut_0` come to: it then
 * drops the fragment's divisions (two 64-bit ones an element, some 3000 instructions a lane) and sees that the four
 * elements down a column lie side by side in the source, which become one 128-bit access.
 *
 * Where the rows of the result are no whole cache lines, a run leaves a piece of a line at both ends, which the memory side
 * takes as a read and a write of the line if the pieces do not meet in time.  Large results of 4- and 8-byte elements
 * therefore go through LDS: a workgroup evaluates four tiles side by side, as ever, and writes of every row the lines that
 * begin within the first 96 (Float64: 112) columns -- the rest of its columns it has for the sake of the last line, and its
 * neighbour evaluates them again.  The lines leave in non-temporal stores.  Other such results are written as they stand:
 * the four waves take two tiles by two and a die takes one contiguous run of the workgroups, so that the pieces meet in
 * one L2.  Rows of whole lines have no pieces: their workgroups, four tiles side by side, are dealt out over the dies, and
 * in large matrices lie one below the other and go down strips of eight, so that the source too is read in longer runs.
 *
 * Transposes in us, before (pieces in every size, divisions gone; whole lines row after row) and now: 5003 x 3001 Float32
 * 30.4 / 20.7 on operands that the memory-side cache holds in part, 32.9 / 28.6 on those it does not (a copy 21.4); 8191^2
 * 152 / 104; 7001 x 2500 Float64 73 / 60; 3891 x 2048 18.5 / 15.7; 8192^2, in strips, 118 / 100; 4096^2 28.8 and 28.8.  Small
 * ones are the tiles at the ends, whose reads were waited for one by one behind a test and now are asked for at once:
 * 1001 x 999 6.4 / 5.0, thirty planes of 501 x 400 14.9 / 14.2, 100 x 101 x 102 turned 9.4 / 6.2.
 */
#ifndef ACC_TT
#define ACC_TT 4                                      /* a lane's block is ACC_TT x ACC_TT */
#endif
#define ACC_TSIDE (8 * ACC_TT)                        /* a wave's tile is ACC_TSIDE x ACC_TSIDE */
#define ACC_TILE_LINE (128 / ACC_TILE_ELT_BYTES)      /* elements of a cache line */
#define ACC_TILE_PITCH (ACC_BLOCK / ACC_WAVE * ACC_TSIDE + 4)

#define ACC_MAP_CAT2_(a, b) a##b
#define ACC_MAP_CAT_(a, b) ACC_MAP_CAT2_(a, b)
#define ACC_TILES_WHOLE 0
#define ACC_TILES_PIECES 1
#define ACC_TILES_LINES 2
#define ACC_TILES_ENTRY ACC_ENTRY
#define ACC_TILES_FORM ACC_TILES_WHOLE
#include "skel_map_tiles.h"
#undef ACC_TILES_ENTRY
#undef ACC_TILES_FORM
#define ACC_TILES_ENTRY ACC_MAP_CAT_(ACC_ENTRY, _pieces)
#define ACC_TILES_FORM ACC_TILES_PIECES
#include "skel_map_tiles.h"
#undef ACC_TILES_ENTRY
#undef ACC_TILES_FORM
#if ACC_TILE_LINES
#define ACC_TILES_ENTRY ACC_MAP_CAT_(ACC_ENTRY, _lines)
#define ACC_TILES_FORM ACC_TILES_LINES
#include "skel_map_tiles.h"
#undef ACC_TILES_ENTRY
#undef ACC_TILES_FORM
#endif

#else

extern "C" __global__ void __launch_bounds__(ACC_BLOCK)
ACC_ENTRY(ACC_ENV_PARAMS ACC_OUT_PARAMS ACC_GUARD_PARAM)
{
  ACC_GUARD_CHECK
  typedef ACC_ELT T;
  ACC_ENV_ASSUME
#if ACC_ALIGNED
  ACC_OUT_ASSUME(arrOut)
#endif
  auto get = [&](const Int64 ix) -> T { return (ACC_GET(ix)); };

  const Int64 n = (ACC_OUT_SIZE);
  const Int64 num_tiles = (n + ACC_TILE - 1) / ACC_TILE;

  for (Int64 tile = blockIdx.x; tile < num_tiles; tile += gridDim.x) {
    const Int64 base = tile * (Int64)ACC_TILE + (Int64)threadIdx.x * ACC_VEC;
    if ((tile + 1) * (Int64)ACC_TILE <= n) {
      T v[ACC_UNROLL][ACC_VEC];
#pragma unroll
      for (int u = 0; u < ACC_UNROLL; ++u)
#pragma unroll
        for (int k = 0; k < ACC_VEC; ++k) v[u][k] = get(base + u * (ACC_BLOCK * ACC_VEC) + k);
#pragma unroll
      for (int u = 0; u < ACC_UNROLL; ++u)
#pragma unroll
        for (int k = 0; k < ACC_VEC; ++k) ACC_PUT(arrOut, base + u * (ACC_BLOCK * ACC_VEC) + k, v[u][k]);
    } else {
#pragma unroll
      for (int u = 0; u < ACC_UNROLL; ++u)
#pragma unroll
        for (int k = 0; k < ACC_VEC; ++k) {
          const Int64 ix = base + u * (ACC_BLOCK * ACC_VEC) + k;
          if (ix < n) ACC_SET(arrOut, ix, get(ix));
        }
    }
  }
}

#endif   /* ACC_MAP_TILED */
