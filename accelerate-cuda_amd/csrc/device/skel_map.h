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
 * LDS and writes it along its rows -- runs of 256 bytes both ways, but the direction of the source fixed -- transposes
 * no faster, and neither do lanes with blocks of 8 x 8 or 2 x 2: 5003 x 3001 Float32 in 40 and 36 us against 31.)
 *
 * What bounds it: the memory side, once the index arithmetic is out of the way.  The place of every element is known
 * here before the fragment asks for it, so the compiler is told what `ix % shOut_0` and `ix / shOut_0` come to: it then
 * drops the fragment's divisions (two 64-bit ones an element, some 3000 instructions a lane) and sees that the four
 * elements down a column lie side by side in the source, which become one 128-bit access.  Where
 * the rows of the result are no whole cache lines, a run leaves a piece of a line at both ends: the four waves of a
 * workgroup then take two tiles by two and a die takes one contiguous run of the workgroups, so that the pieces meet in
 * one L2.  Rows of whole lines have no pieces; dealing their workgroups out over the dies, four tiles side by side, is
 * the faster order.  Transposes in us, dealt out with divisions / without / two by two on one die: 5003 x 3001 Float32
 * 46.5 / 37.1 / 31.0 (3.9 TB/s; 1.2 times the source is read, 1.08 times the result written); 4000 x 4000 31.9 / 28.1 /
 * 29.6; 8192 x 8192 125 / 118 / 131; 7001 x 2500 Float64 89.3 / - / 72.6.
 */
#ifndef ACC_TT
#define ACC_TT 4                                      /* a lane's block is ACC_TT x ACC_TT */
#endif
#define ACC_TSIDE (8 * ACC_TT)                        /* a wave's tile is ACC_TSIDE x ACC_TSIDE */

extern "C" __global__ void __launch_bounds__(ACC_BLOCK)
ACC_ENTRY(ACC_ENV_PARAMS ACC_OUT_PARAMS ACC_GUARD_PARAM)
{
  ACC_GUARD_CHECK
  typedef ACC_ELT T;
  ACC_ENV_ASSUME
  /* the element at `ix`, which is column `acc_c` of row `acc_r` of the result's rows taken as one list */
  auto acc_get_at = [&](const Int64 ix, const Int64 acc_r, const Int64 acc_c) -> T {
    __builtin_assume(ix % shOut_0 == acc_c);
    __builtin_assume(ix / shOut_0 == acc_r);
    return (ACC_GET(ix));
  };

  /* The tiles' second dimension is the second innermost one of the result, or one further out (ACC_TILE_H its
   * extent, ACC_TILE_MIDS the rows between neighbours along it: a volume turned so that its innermost
   * dimension becomes its outermost reads its source along that one).  What lies between that dimension and the
   * innermost (`mids` rows for every place along it) and outside it (`outers`) is walked tile by tile. */
  const Int64 w = shOut_0, h = ACC_TILE_H, mids = ACC_TILE_MIDS, stride = mids * w;
  const Int64 n = (ACC_OUT_SIZE);
  const Int64 outers = (h > 0 && stride > 0) ? n / (h * stride) : 0;
  const int lane = acc_lane();
  const int lx = lane & 7, ly = lane >> 3;
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  /* a workgroup's waves: two by two tiles, or side by side where the result is no taller than one and where its rows
   * are whole cache lines (the driver counts the workgroups by the same rule) */
  constexpr int WAVES = ACC_BLOCK / ACC_WAVE;
  const bool whole_lines = (w * ACC_TILE_ELT_BYTES) % 128 == 0;
  const int down = (WAVES % 2 == 0 && h > ACC_TSIDE && !whole_lines) ? 2 : 1, across = WAVES / down;
  const Int64 groups_x = (w + across * ACC_TSIDE - 1) / (across * ACC_TSIDE), groups_y = (h + down * ACC_TSIDE - 1) / (down * ACC_TSIDE);
  const Int64 groups = groups_x * groups_y * mids * outers;
  /* the quotient of numbers no larger than the array has elements: in 32 bits where it has fewer than 2^31 */
  const bool narrow = n < 0x7fffffff;
  auto divide = [&](const Int64 a, const Int64 b) -> Int64 {
    return narrow ? (Int64)((unsigned int)a / (unsigned int)b) : a / b;
  };

  for (Int64 group = whole_lines ? (Int64)blockIdx.x : acc_xcd_contiguous_block(); group < groups; group += gridDim.x) {
    const Int64 g1 = divide(group, groups_x), gx = group - g1 * groups_x;
    const Int64 plane = divide(g1, groups_y), gy = g1 - plane * groups_y;
    const Int64 outer = divide(plane, mids), mid = plane - outer * mids;
    const Int64 tx = gx * across + (down == 2 ? wave >> 1 : wave), ty = gy * down + (down == 2 ? wave & 1 : 0);
    const Int64 x = tx * ACC_TSIDE + lx * ACC_TT, y = ty * ACC_TSIDE + ly * ACC_TT;
    const Int64 row = (outer * h + y) * mids + mid, base = row * w + x;
    if ((tx + 1) * ACC_TSIDE <= w && (ty + 1) * ACC_TSIDE <= h) {
      T v[ACC_TT][ACC_TT];
      /* down the columns first: what a transposed source holds side by side */
#pragma unroll
      for (int k = 0; k < ACC_TT; ++k)
#pragma unroll
        for (int i = 0; i < ACC_TT; ++i) v[i][k] = acc_get_at(base + i * stride + k, row + i * mids, x + k);
#pragma unroll
      for (int i = 0; i < ACC_TT; ++i)
#pragma unroll
        for (int k = 0; k < ACC_TT; ++k) ACC_SET(arrOut, base + i * stride + k, v[i][k]);
    } else {
#pragma unroll
      for (int i = 0; i < ACC_TT; ++i)
#pragma unroll
        for (int k = 0; k < ACC_TT; ++k)
          if (x + k < w && y + i < h) ACC_SET(arrOut, base + i * stride + k, acc_get_at(base + i * stride + k, row + i * mids, x + k));
    }
  }
}

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
