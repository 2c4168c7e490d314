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
                                                const Int64 acc_split, ACC_ELT *__restrict__ acc_part, int *__restrict__ acc_part_ok,
                                                const int acc_chunk, const int acc_subs ACC_GUARD_PARAM)
{
  ACC_GUARD_CHECK
  typedef ACC_ELT T;
  constexpr int acc_R = ACC_ACROSS_R;
  ACC_ENV_ASSUME
  auto acc_get = ACC_GET_AT_ROW_COL;
  auto acc_f   = [&](const T &x, const T &y) -> T { return (ACC_COMBINE(x, y)); };
  (void)shIn_1;
  const Int64 acc_rows = shOut_0, acc_len = shIn_0;
  /* (in bytes: an element type may have members with initialisers of their own) */
  __shared__ __align__(16) unsigned char acc_s_raw[ACC_BLOCK * acc_R * sizeof(T)];
  __shared__ int acc_s_ok[ACC_BLOCK];
  T *acc_s_val = (T *)acc_s_raw;
#if ACC_HAS_SEED
  const T acc_seed = (ACC_SEED);
#else
  const T acc_seed = T();
#endif

  const Int64 lanes = (acc_rows + acc_R - 1) / acc_R, chunks = (lanes + acc_chunk - 1) / acc_chunk;
  const int sub = (int)threadIdx.x / acc_chunk, side = (int)threadIdx.x - sub * acc_chunk;
  const Int64 pieces = acc_split * acc_subs, piece = (acc_len + pieces - 1) / pieces;
  for (Int64 b = blockIdx.x; b < chunks * acc_split; b += gridDim.x) {       /* (the same number of turns in every thread) */
    const Int64 run = b / chunks, first = (b - run * chunks) * acc_chunk * acc_R + side;
    const bool mine = sub < acc_subs && first < acc_rows;
    Int64 row[acc_R];                                        /* past the last one: that one again, not written */
#pragma unroll
    for (int r = 0; r < acc_R; ++r) row[r] = acc_min<Int64>(first + r * acc_chunk, acc_rows - 1);
    const Int64 k0 = acc_min<Int64>((run * acc_subs + sub) * piece, acc_len), k1 = acc_min<Int64>(k0 + piece, acc_len);
    T v[acc_R];
    bool ok = mine && k0 < k1;
    if (ok) {
      /* (from the right a row in one piece begins with the seed, x0 (+) (x1 (+) (... (x_last (+) z))), as the other
       * entries associate a row; from the left the seed comes last) */
      if (pieces == 1)       acc_across_piece<acc_R, 1, ACC_FOLD_RIGHT && ACC_HAS_SEED, T>(acc_get, acc_f, row, k0, k1, acc_seed, v);
      else if (k1 - k0 >= 4) acc_across_piece<acc_R, 2, false, T>(acc_get, acc_f, row, k0, k1, acc_seed, v);
      else                   acc_across_piece<acc_R, 1, false, T>(acc_get, acc_f, row, k0, k1, acc_seed, v);
    }
    /* the pieces of a row meet: neighbours in order, then neighbours of those */
    if (acc_subs > 1) {
      __syncthreads();                                   /* (the turn before has read) */
      acc_s_ok[threadIdx.x] = ok;
      if (ok) {
#pragma unroll
        for (int r = 0; r < acc_R; ++r) acc_s_val[threadIdx.x * acc_R + r] = v[r];
      }
      for (int apart = 1; apart < acc_subs; apart *= 2) {
        __syncthreads();
        const int other = (int)threadIdx.x + apart * acc_chunk;
        if (sub < acc_subs && (sub & (2 * apart - 1)) == 0 && sub + apart < acc_subs && acc_s_ok[other]) {
#pragma unroll
          for (int r = 0; r < acc_R; ++r) {
            const T w = acc_s_val[other * acc_R + r];
            v[r] = ok ? acc_f(v[r], w) : w;
            acc_s_val[threadIdx.x * acc_R + r] = v[r];
          }
          ok = true;
          acc_s_ok[threadIdx.x] = 1;
        }
      }
    }
    if (!mine || sub != 0) continue;
    if (acc_split > 1) {
#pragma unroll
      for (int r = 0; r < acc_R; ++r) {
        if (first + r * acc_chunk >= acc_rows) break;
        if (ok) acc_part[row[r] * acc_split + run] = v[r];
        acc_part_ok[row[r] * acc_split + run] = ok;
      }
    } else {
#pragma unroll
      for (int r = 0; r < acc_R; ++r) {
        if (first + r * acc_chunk >= acc_rows) break;
#if ACC_HAS_SEED
        /* ((x0 (+) x1) (+) ... x_last) (+) z; a row in one piece from the right has its seed already */
        ACC_PUT(arrOut, row[r], (ACC_FOLD_RIGHT && pieces == 1) ? v[r] : acc_f(v[r], acc_seed));
#else
        ACC_PUT(arrOut, row[r], v[r]);
#endif
      }
    }
  }
}
