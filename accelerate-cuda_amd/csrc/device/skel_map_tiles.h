/*
 * skel_map_tiles.h -- the map in tiles; included by skel_map.h once for each form of the result (ACC_TILES_FORM):
 *   whole    its rows are whole cache lines and it begins with one (<entry>)
 *   pieces   they are not: a tile's runs are written as they stand, and leave a piece of a line at both ends (<entry>_pieces)
 *   lines    the same results, of elements of 4 and 8 bytes, written in whole lines through LDS (<entry>_lines)
 */
extern "C" __global__ void __launch_bounds__(ACC_BLOCK)
ACC_TILES_ENTRY(ACC_ENV_PARAMS ACC_OUT_PARAMS ACC_GUARD_PARAM)
{
  ACC_GUARD_CHECK
  typedef ACC_ELT T;
  ACC_ENV_ASSUME
#if ACC_TILES_FORM == ACC_TILES_LINES
  __shared__ __align__(16) T acc_tile[ACC_TSIDE * ACC_TILE_PITCH];
#endif
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
  /* A workgroup's waves: side by side, the last ACC_TILE_LINE columns for the sake of the next workgroup's lines; or two
   * by two, side by side where the rows are whole cache lines or the result is no taller than one tile, and below one
   * another, down strips eight workgroups tall, in large matrices of whole lines.  (The driver counts the workgroups by the
   * same rule.) */
  constexpr int WAVES = ACC_BLOCK / ACC_WAVE;
  constexpr bool whole = ACC_TILES_FORM == ACC_TILES_WHOLE, lines = ACC_TILES_FORM == ACC_TILES_LINES;
  const bool strips = whole && n == w * h && n * ACC_TILE_ELT_BYTES >= ACC_TILE_STRIPS_FROM;
  const int down = lines || h <= ACC_TSIDE ? 1 : (strips ? WAVES : (WAVES % 2 == 0 && !whole ? 2 : 1)), across = WAVES / down;
  const int columns = across * ACC_TSIDE - (lines ? ACC_TILE_LINE : 0);
  const Int64 groups_x = (w + columns - 1) / columns, groups_y = (h + down * ACC_TSIDE - 1) / (down * ACC_TSIDE);
  const Int64 groups = groups_x * groups_y * mids * outers;
  /* the quotient of numbers no larger than the array has elements: in 32 bits where it has fewer than 2^31 */
  const bool narrow = n < 0x7fffffff;
  auto divide = [&](const Int64 a, const Int64 b) -> Int64 {
    return narrow ? (Int64)((unsigned int)a / (unsigned int)b) : a / b;
  };

  for (Int64 group = whole ? (Int64)blockIdx.x : acc_xcd_contiguous_block(); group < groups; group += gridDim.x) {
    /* row after row of groups, or down strips eight groups tall */
    const Int64 plane = divide(group, groups_x * groups_y), g = group - plane * (groups_x * groups_y);
    const Int64 strip = divide(g, groups_x * 8), g1 = g - strip * (groups_x * 8), tall = acc_min<Int64>(8, groups_y - strip * 8);
    const Int64 gx = strips ? divide(g1, tall) : g - divide(g, groups_x) * groups_x;
    const Int64 gy = strips ? strip * 8 + (g1 - gx * tall) : divide(g, groups_x);
    const Int64 outer = divide(plane, mids), mid = plane - outer * mids;
    const Int64 x0 = gx * columns, tx = down == 1 ? wave : (down == 2 ? wave >> 1 : 0), ty = gy * down + (down == 1 ? 0 : (down == 2 ? wave & 1 : wave));
    const Int64 x = x0 + tx * ACC_TSIDE + lx * ACC_TT, y = ty * ACC_TSIDE + ly * ACC_TT;
    const Int64 row = (outer * h + y) * mids + mid, base = row * w + x;
    /* what lies beyond the result is made from its last row or column and goes nowhere: a read under a test would be waited
     * for on the spot, one element after the other.  (Not in whole lines: only the last rows of the tiles meet an end there,
     * and the registers that sixteen such elements take cost the others more.) */
    auto acc_get_within = [&](const Int64 yy, const Int64 xx) -> T {
      const Int64 acc_c = acc_min<Int64>(xx, w - 1), acc_r = (outer * h + acc_min<Int64>(yy, h - 1)) * mids + mid;
      return acc_get_at(acc_r * w + acc_c, acc_r, acc_c);
    };
    (void)acc_get_within;
    const bool inside = x0 + (tx + 1) * ACC_TSIDE <= w && (ty + 1) * ACC_TSIDE <= h;
#if ACC_TILES_FORM == ACC_TILES_LINES
    /* through LDS, and out in whole lines: of every row the columns from the first line that begins at or beyond x0 to the
     * one that begins as far into the next workgroup's */
    __syncthreads();                                     /* (the turn before has been written out) */
    T v[ACC_TT][ACC_TT];
    if (inside) {
#pragma unroll
      for (int k = 0; k < ACC_TT; ++k)
#pragma unroll
        for (int i = 0; i < ACC_TT; ++i) v[i][k] = acc_get_at(base + i * stride + k, row + i * mids, x + k);
      /* (in this branch: reads that both branches end with become one read an element behind them) */
#pragma unroll
      for (int k = 0; k < ACC_TT; ++k)
#pragma unroll
        for (int i = 0; i < ACC_TT; ++i) acc_pin(v[i][k]);
    } else {
#pragma unroll
      for (int k = 0; k < ACC_TT; ++k)
#pragma unroll
        for (int i = 0; i < ACC_TT; ++i) v[i][k] = acc_get_within(y + i, x + k);
    }
#pragma unroll
    for (int i = 0; i < ACC_TT; ++i)
#pragma unroll
      for (int k = 0; k < ACC_TT; ++k) acc_tile[(ly * ACC_TT + i) * ACC_TILE_PITCH + (int)tx * ACC_TSIDE + lx * ACC_TT + k] = v[i][k];
    __syncthreads();
    const Int64 y0 = ty * ACC_TSIDE, rows = acc_min<Int64>(ACC_TSIDE, h - y0);
    const bool left = gx == 0, right = gx == groups_x - 1;
    T *const to0 = arrOut_0 + ((outer * h + y0) * mids + mid) * w + x0;            /* where the group begins */
    auto past = [&](const int r) -> int { return (int)((0 - (unsigned long long)(to0 + r * stride)) & 127u) / (int)sizeof(T); };
    if (!left && !right) {
      constexpr int VEC = 16 / (int)sizeof(T), PIECES = (WAVES * ACC_TSIDE - ACC_TILE_LINE) / VEC;
      typedef T piece_t __attribute__((ext_vector_type(VEC)));
      for (int e = (int)threadIdx.x; e < (int)rows * PIECES; e += ACC_BLOCK) {
        const int r = e / PIECES, c = past(r) + (e - r * PIECES) * VEC;
        if (x0 + c >= w) continue;                       /* (the array ends amid the next group's first line) */
        piece_t p;
#pragma unroll
        for (int k = 0; k < VEC; ++k) p[k] = acc_tile[r * ACC_TILE_PITCH + c + k];
        if (x0 + c + VEC <= w) __builtin_nontemporal_store(p, (piece_t *)(to0 + r * stride + c));
        else for (int k = 0; x0 + c + k < w; ++k) to0[r * stride + c + k] = p[k];
      }
    } else {
      for (int e = (int)threadIdx.x; e < (int)rows * (WAVES * ACC_TSIDE); e += ACC_BLOCK) {
        const int r = e / (WAVES * ACC_TSIDE), c = e - r * (WAVES * ACC_TSIDE), from = past(r);
        if ((left || c >= from) && (right || c < from + columns) && x0 + c < w) to0[r * stride + c] = acc_tile[r * ACC_TILE_PITCH + c];
      }
    }
#else
    if (inside) {
      T v[ACC_TT][ACC_TT];
      /* down the columns first: what a transposed source holds side by side */
#pragma unroll
      for (int k = 0; k < ACC_TT; ++k)
#pragma unroll
        for (int i = 0; i < ACC_TT; ++i) v[i][k] = acc_get_at(base + i * stride + k, row + i * mids, x + k);
#pragma unroll
      for (int i = 0; i < ACC_TT; ++i)
#pragma unroll
        for (int k = 0; k < ACC_TT; ++k) {
          if (strips && ACC_TILE_LINES) ACC_PUT(arrOut, base + i * stride + k, v[i][k]);
          else                          ACC_SET(arrOut, base + i * stride + k, v[i][k]);
        }
    } else if (whole) {
#pragma unroll
      for (int i = 0; i < ACC_TT; ++i)
#pragma unroll
        for (int k = 0; k < ACC_TT; ++k)
          if (x + k < w && y + i < h) ACC_SET(arrOut, base + i * stride + k, acc_get_at(base + i * stride + k, row + i * mids, x + k));
    } else {
      T v[ACC_TT][ACC_TT];
#pragma unroll
      for (int k = 0; k < ACC_TT; ++k)
#pragma unroll
        for (int i = 0; i < ACC_TT; ++i) v[i][k] = acc_get_within(y + i, x + k);
#pragma unroll
      for (int i = 0; i < ACC_TT; ++i)
#pragma unroll
        for (int k = 0; k < ACC_TT; ++k)
          if (x + k < w && y + i < h) ACC_SET(arrOut, base + i * stride + k, v[i][k]);
    }
#endif
  }
}
