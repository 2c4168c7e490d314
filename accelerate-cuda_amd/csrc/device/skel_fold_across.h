/*
 * skel_fold_across.h -- the fold along rows that lie across memory, neighbouring rows in neighbouring lanes; included by
 * skel_foldseg.h once for ACC_ACROSS_R rows a lane == 1 (<entry>_across) and once for as many as are 16 bytes of an
 * element narrower than that (<entry>_across_wide).
 *
 * A workgroup takes `chunk` lanes' rows side by side (a lane's rows lie `chunk` rows apart, so that every access of a
 * wave is one run whatever the element function reads besides), `subs` times over: each of those goes through one
 * piece of the rows, the pieces following one another, and the pieces' values meet in LDS, in order.  With too few rows
 * to fill the device so, the rows are cut into `split` of these runs of pieces, whose values <entry>_join puts together;
 * with split == 1 the workgroup writes the results itself.  Where rows are cut at all, a lane goes through its piece in
 * two halves side by side, joined at the end: twice the requests in flight, and shorter chains of rounding.  A row that
 * is not cut is folded in index order by one lane.
 *
 * What bounds it: the memory side, and the second launch where there is one (3 us).  Sums down the columns, us before
 * (one row a lane, every piece a part of its own for the second launch) and now: 20000 x 1000 Float32 20.9 / 18.3,
 * 200000 x 100 38.3 / 18.6, 262144 x 16 23.4 / 9.8, 100000 x 333 Float64 70.7 / 51.9 (5.1 TB/s); the product of two
 * 512 x 512 matrices as a fold 76 / 36.
 */
extern "C" __global__ void __launch_bounds__(ACC_BLOCK)
ACC_FS_CAT_(ACC_FOLDSEG_ENTRY, ACC_ACROSS_ENTRY)(ACC_ENV_PARAMS
                                                const Int64 shOut_0, ACC_OUT_ARRAY(arrOut),
                                                ACC_SEG_PARAMS,
                                                const Int64 split, ACC_ELT *__restrict__ part, int *__restrict__ part_ok,
                                                const int chunk, const int subs ACC_GUARD_PARAM)
{
  ACC_GUARD_CHECK
  typedef ACC_ELT T;
  constexpr int R = ACC_ACROSS_R;
  ACC_ENV_ASSUME
  auto get = ACC_GET_AT_ROW_COL;
  auto f   = [&](const T &x, const T &y) -> T { return (ACC_COMBINE(x, y)); };
  (void)shIn_1;
  const Int64 rows = shOut_0, len = shIn_0;
  /* (in bytes: an element type may have members with initialisers of their own) */
  __shared__ __align__(16) unsigned char s_raw[ACC_BLOCK * R * sizeof(T)];
  __shared__ int s_ok[ACC_BLOCK];
  T *s_val = (T *)s_raw;
#if ACC_HAS_SEED
  const T seed = (ACC_SEED);
#else
  const T seed = T();
#endif

  const Int64 lanes = (rows + R - 1) / R, chunks = (lanes + chunk - 1) / chunk;
  const int sub = (int)threadIdx.x / chunk, side = (int)threadIdx.x - sub * chunk;
  const Int64 pieces = split * subs, piece = (len + pieces - 1) / pieces;
  for (Int64 b = blockIdx.x; b < chunks * split; b += gridDim.x) {       /* (the same number of turns in every thread) */
    const Int64 run = b / chunks, first = (b - run * chunks) * chunk * R + side;
    const bool mine = sub < subs && first < rows;
    Int64 row[R];                                        /* past the last one: that one again, not written */
#pragma unroll
    for (int r = 0; r < R; ++r) row[r] = acc_min<Int64>(first + r * chunk, rows - 1);
    const Int64 k0 = acc_min<Int64>((run * subs + sub) * piece, len), k1 = acc_min<Int64>(k0 + piece, len);
    T v[R];
    bool ok = mine && k0 < k1;
    if (ok) {
      /* (from the right a row in one piece begins with the seed, x0 (+) (x1 (+) (... (x_last (+) z))), as the other
       * entries associate a row; from the left the seed comes last) */
      if (pieces == 1)       acc_across_piece<R, 1, ACC_FOLD_RIGHT && ACC_HAS_SEED, T>(get, f, row, k0, k1, seed, v);
      else if (k1 - k0 >= 4) acc_across_piece<R, 2, false, T>(get, f, row, k0, k1, seed, v);
      else                   acc_across_piece<R, 1, false, T>(get, f, row, k0, k1, seed, v);
    }
    /* the pieces of a row meet: neighbours in order, then neighbours of those */
    if (subs > 1) {
      __syncthreads();                                   /* (the turn before has read) */
      s_ok[threadIdx.x] = ok;
      if (ok) {
#pragma unroll
        for (int r = 0; r < R; ++r) s_val[threadIdx.x * R + r] = v[r];
      }
      for (int apart = 1; apart < subs; apart *= 2) {
        __syncthreads();
        const int other = (int)threadIdx.x + apart * chunk;
        if (sub < subs && (sub & (2 * apart - 1)) == 0 && sub + apart < subs && s_ok[other]) {
#pragma unroll
          for (int r = 0; r < R; ++r) {
            const T w = s_val[other * R + r];
            v[r] = ok ? f(v[r], w) : w;
            s_val[threadIdx.x * R + r] = v[r];
          }
          ok = true;
          s_ok[threadIdx.x] = 1;
        }
      }
    }
    if (!mine || sub != 0) continue;
    if (split > 1) {
#pragma unroll
      for (int r = 0; r < R; ++r) {
        if (first + r * chunk >= rows) break;
        if (ok) part[row[r] * split + run] = v[r];
        part_ok[row[r] * split + run] = ok;
      }
    } else {
#pragma unroll
      for (int r = 0; r < R; ++r) {
        if (first + r * chunk >= rows) break;
#if ACC_HAS_SEED
        /* ((x0 (+) x1) (+) ... x_last) (+) z; a row in one piece from the right has its seed already */
        ACC_PUT(arrOut, row[r], (ACC_FOLD_RIGHT && pieces == 1) ? v[r] : f(v[r], seed));
#else
        ACC_PUT(arrOut, row[r], v[r]);
#endif
      }
    }
  }
}
