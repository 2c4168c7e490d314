/*
 * skel_stencil_flat.h -- 3-D stencils with taps in other planes, the lanes over the vectors of a plane.
 *
 * The strips of skel_stencil.h are 64 lanes of one row each: a row of 300 columns is two strips of 256 or three of 128,
 * of which a fifth of the lanes lie outside the volume, and every strip ends amid a cache line that another one writes the
 * rest of.  Here the lanes are laid over the vectors of a whole plane, row after row: a wave takes 62 consecutive vectors
 * wherever rows end among them, and one more at either end whose columns its neighbours ask for, so no lane is idle and
 * consecutive waves read and write consecutive memory.  A wave makes ACC_FLAT_PLANES planes of the result, written out; it
 * asks for the first ACC_FIRST planes it reads at once -- all of them for a stencil that reads few rows -- and for the others
 * one by one.
 *   - The columns left and right of a lane's vector come from the lanes beside it (DPP wave shifts), at the ends of a row
 *     from the boundary condition; under `wrap` those lanes read the other end of the row, the others all ask for one
 *     element.  (Taps two columns away are read by the lane itself, as all were: 300^3 with 7 points 51 us against 44.)
 *   - The boundary condition along rows and columns is worked out once: it is the offset within a plane that each of the
 *     lane's reads goes to, the same in every plane.
 *   - The last vector of a row ends where the row ends (it overlaps its neighbour, whose columns it produces a second
 *     time, the same values); the two hand each other what stands beside the other's columns.
 *   - A die takes an eighth of every plane, the same one, so that the rows that neighbouring planes share are in its L2, and
 *     all dies go through the volume together: what is in flight is a few planes, not the whole volume.  (Every die a run
 *     of planes of its own: 47 us instead of 44.)
 *
 * What bounds it: the memory side; a copy of the same bytes takes 36 us.  300^3 Float32, 7 points: 77 us in strips, 54.4 in
 * waves that walked through 8 planes and read the columns beside a vector themselves, 45.2 (4.8 TB/s) so; 27 points 97 /
 * 64 / 51; Float64 131 / 103 / 88 and 167 / 118 / 113; 150^3 15.0 / 8.7 / 7.1.  Planes a wave, all at once / one asked for
 * ahead: 2 49.7, 4 45.7 / 47.4, 8 - / 47.7; with 27 points 67.5, 58.4 / 57.5, - / 51.3.  Two rows a lane: 47.4, with 27
 * points the same.  Ordinary stores instead of non-temporal ones: 47.8.
 *
 * Generated definitions expected: those of skel_stencil.h, for ACC_STENCIL_RANK 3 and one source of one component, and
 * ACC_FLAT_PLANES, ACC_FLAT_SPREAD (waves of a plane for each die from which planes are dealt out over the dies); the planes of
 * source and result are smaller than 4 GB (the driver sees to it), the rows no shorter than a vector.
 */

#ifndef ACC_SVEC
#define ACC_SVEC 4
#endif
#define ACC_NR    (2 * ACC_RADIUS_Z + ACC_FLAT_PLANES)    /* planes a wave reads */
#define ACC_FIRST (2 * ACC_RADIUS_Z + 1 + ACC_PREFETCH) /* ... of them asked for at once */
#define ACC_WW    (ACC_SVEC + 2 * ACC_RADIUS_X)       /* row window of one lane */
#define ACC_NZ    (2 * ACC_RADIUS_Y + 1)              /* rows read of each */
#define ACC_GIVE  (ACC_RADIUS_X == 1 ? 1 : 0)         /* lanes hand each other the columns beside their own */
#define ACC_OWNED (ACC_WAVE - 2 * ACC_GIVE)           /* lanes whose columns are stored */

/* what is known of a vector's address */
#define ACC_FLAT_ALIGN(S) (ACC_ALIGNED ? (ACC_SVEC * sizeof(S) < 16 ? ACC_SVEC * sizeof(S) : 16) : alignof(S))

#define ACC_B_CLAMP 0
#define ACC_B_MIRROR 1
#define ACC_B_WRAP 2
#define ACC_B_CONSTANT 3

template <int MODE>
ACC_DEV int acc_flat_boundary(int i, const int sz)
{
  if (MODE == ACC_B_MIRROR) i = i < 0 ? -i : (i >= sz ? sz - (i - sz + 2) : i);
  if (MODE == ACC_B_WRAP)   i = i < 0 ? sz + i : (i >= sz ? i - sz : i);
  /* clamped in every mode: the maps assume the array spans the stencil; keep the address legal if not */
  return acc_max(0, acc_min(i, sz - 1));
}

/* the neighbouring lane's value; a lane that has no neighbour gets that of the wave's other end (what it makes of it is
 * dropped, but the element function is to see values of the array only) */
#define ACC_DPP_WAVE_ROL1 0x134
#define ACC_DPP_WAVE_ROR1 0x13C
template <int CTRL, typename S>
ACC_DEV S acc_flat_shift(const S &x)
{
  unsigned int s[acc_words<S>::n];
  __builtin_memcpy(s, &x, sizeof(S));
#pragma unroll
  for (int w = 0; w < acc_words<S>::n; ++w) s[w] = (unsigned int)__builtin_amdgcn_update_dpp(0, (int)s[w], CTRL, 0xf, 0xf, true);
  S r;
  __builtin_memcpy(&r, s, sizeof(S));
  return r;
}

/* the source as a lane sees it */
template <typename S, int MODE>
struct acc_flat_source {
  /* rows begin on 16-byte boundaries in an aligned instance: whole vectors then, unless a vector is longer than that */
  static constexpr bool WHOLE = ACC_ALIGNED && ACC_SVEC * sizeof(S) <= 16;
  struct row { S e[ACC_WW]; };
  struct __attribute__((aligned(ACC_FLAT_ALIGN(S)))) vec { S v[ACC_SVEC]; };
  static constexpr bool GIVE = ACC_GIVE != 0, ENDS = GIVE && MODE == ACC_B_WRAP;      /* ENDS: the other end of a row is read */
  static constexpr int SIDE = ACC_RADIUS_X > 0 ? ACC_RADIUS_X : 1;

  const char *base;
  Int64 plane_bytes;
  int d, z0;
  S outside;
  unsigned int row_at[ACC_NZ];         /* bytes from the start of a plane to each of the rows */
  unsigned int own;                    /* ... and from the start of a row to the vector and its neighbours */
  unsigned int left[SIDE], right[SIDE];
  unsigned int end_at[ENDS ? ACC_NZ : 1];
  unsigned int rows_in, left_in, right_in;         /* constant boundary: which of them lie inside */
  bool at_left, at_right;              /* the row begins, ends with this lane's vector */
  int rest;                            /* columns of the last vector that are not the one's before it, where that is not all of them */
  bool last, next_last;                /* ... this lane's vector, its right neighbour's is that one */
  row window[ACC_NR][ACC_NZ];
  S end[ENDS ? ACC_NR : 1][ENDS ? ACC_NZ : 1];

  ACC_DEV void place(const int x, const int y, const int w, const int h)
  {
    rows_in = left_in = right_in = 0;
    at_left = x == 0;
    at_right = x + ACC_SVEC == w;
    rest = WHOLE ? 0 : w % ACC_SVEC;
    last = rest != 0 && at_right && !at_left;
    next_last = rest != 0 && !at_right && x + 2 * ACC_SVEC > w;
#pragma unroll
    for (int p = 0; p < ACC_NZ; ++p) {
      const int gy = y - ACC_RADIUS_Y + p;
      row_at[p] = (unsigned int)acc_flat_boundary<MODE>(gy, h) * (unsigned int)w * (unsigned int)sizeof(S);
      rows_in |= (gy >= 0 && gy < h ? 1u : 0u) << p;
      /* (the lanes amid a row all ask for the plane's first element) */
      if (ENDS) end_at[p] = at_left ? row_at[p] + (unsigned int)(w - 1) * (unsigned int)sizeof(S) : (at_right ? row_at[p] : 0u);
    }
    own = (unsigned int)x * (unsigned int)sizeof(S);
#pragma unroll
    for (int j = 0; j < (GIVE ? 0 : ACC_RADIUS_X); ++j) {
      const int l = x - ACC_RADIUS_X + j, r = x + ACC_SVEC + j;
      left[j] = (unsigned int)acc_flat_boundary<MODE>(l, w) * (unsigned int)sizeof(S);
      right[j] = (unsigned int)acc_flat_boundary<MODE>(r, w) * (unsigned int)sizeof(S);
      left_in |= (l >= 0 ? 1u : 0u) << j;
      right_in |= (r < w ? 1u : 0u) << j;
    }
  }
  /* ask for the rows of plane z0 - rz + i (those that no tap of the stencil reads are not asked for: the compiler sees) */
  ACC_DEV void ask(const int i)
  {
    const char *plane = base + (Int64)acc_flat_boundary<MODE>(z0 - ACC_RADIUS_Z + i, d) * plane_bytes;
#pragma unroll
    for (int p = 0; p < ACC_NZ; ++p) {
      row &r = window[i][p];
      const vec v = *(const vec *)(plane + (row_at[p] + own));
#pragma unroll
      for (int k = 0; k < ACC_SVEC; ++k) r.e[ACC_RADIUS_X + k] = v.v[k];
#pragma unroll
      for (int j = 0; j < (GIVE ? 0 : ACC_RADIUS_X); ++j) {
        r.e[j] = *(const S *)(plane + (row_at[p] + left[j]));
        r.e[ACC_RADIUS_X + ACC_SVEC + j] = *(const S *)(plane + (row_at[p] + right[j]));
      }
      if (ENDS) end[i][p] = *(const S *)(plane + end_at[p]);
    }
  }
  /* what stands beside the lane's columns, and outside */
  ACC_DEV void settle(const int i)
  {
    const int gz = z0 - ACC_RADIUS_Z + i;
    const bool plane_in = MODE != ACC_B_CONSTANT || (gz >= 0 && gz < d);
#pragma unroll
    for (int p = 0; p < ACC_NZ; ++p) {
      row &r = window[i][p];
      const bool in = plane_in && (MODE != ACC_B_CONSTANT || ((rows_in >> p) & 1u));
#pragma unroll
      for (int k = 0; k < ACC_SVEC; ++k) r.e[ACC_RADIUS_X + k] = in ? r.e[ACC_RADIUS_X + k] : outside;
      if (GIVE) {
        const S *v = &r.e[ACC_RADIUS_X];
        /* what the neighbours get: the columns at the ends, or, where the last vector of a row overlaps the one before
         * it, those that stand beside the other's */
        S first = v[0], back = v[ACC_SVEC - 1];
        if (!WHOLE) {
          S to_left = v[ACC_SVEC - 1], to_right = v[0];                            /* (rest 1) */
#pragma unroll
          for (int k = 2; k < ACC_SVEC; ++k) {
            to_left = rest == k ? v[ACC_SVEC - k] : to_left;
            to_right = rest == k ? v[k - 1] : to_right;
          }
          first = last ? to_left : first;
          back = next_last ? to_right : back;
        }
        const S l = acc_flat_shift<ACC_DPP_WAVE_ROR1>(back), t = acc_flat_shift<ACC_DPP_WAVE_ROL1>(first);
        /* (the columns next to the first and the last: with one column a lane, where there are any, the neighbours hold them) */
        const S second = ACC_SVEC > 1 ? v[ACC_SVEC > 1 ? 1 : 0] : (at_right ? v[0] : t), last_but_one = ACC_SVEC > 1 ? v[ACC_SVEC > 1 ? ACC_SVEC - 2 : 0] : (at_left ? v[0] : l);
        const S beyond_l = MODE == ACC_B_CONSTANT ? outside : (MODE == ACC_B_WRAP ? end[ENDS ? i : 0][ENDS ? p : 0] : (MODE == ACC_B_MIRROR ? second : v[0]));
        const S beyond_r = MODE == ACC_B_CONSTANT ? outside : (MODE == ACC_B_WRAP ? (at_left ? v[0] : end[ENDS ? i : 0][ENDS ? p : 0]) : (MODE == ACC_B_MIRROR ? last_but_one : v[ACC_SVEC - 1]));
        r.e[0] = at_left ? beyond_l : l;
        r.e[ACC_WW - 1] = at_right ? beyond_r : t;
      } else {
#pragma unroll
        for (int j = 0; j < ACC_RADIUS_X; ++j) {
          if (MODE != ACC_B_CONSTANT) break;
          r.e[j] = (in && ((left_in >> j) & 1u)) ? r.e[j] : outside;
          r.e[ACC_RADIUS_X + ACC_SVEC + j] = (in && ((right_in >> j) & 1u)) ? r.e[ACC_RADIUS_X + ACC_SVEC + j] : outside;
        }
      }
    }
  }
};

struct acc_out_vec { ACC_ELT v[ACC_SVEC]; };

extern "C" __global__ void __launch_bounds__(ACC_BLOCK)
stencil(ACC_ENV_PARAMS ACC_OUT_PARAMS ACC_SRC1_PARAMS, const int acc_walk ACC_GUARD_PARAM)
{
  ACC_GUARD_CHECK
  typedef ACC_ELT T;
  ACC_ENV_ASSUME
  (void)acc_walk;
  const int acc_d = (int)shOut_2, acc_h = (int)shOut_1, acc_w = (int)shOut_0;
  /* (the driver counts the waves by the same numbers, all of them within 32 bits) */
  const unsigned int acc_vectors = ((unsigned int)acc_w + ACC_SVEC - 1) / ACC_SVEC, acc_per_plane = acc_vectors * (unsigned int)acc_h;
  const unsigned int acc_waves = (acc_per_plane + ACC_OWNED - 1) / ACC_OWNED;
  constexpr unsigned int acc_waves_of_block = ACC_BLOCK / ACC_WAVE;
  const unsigned int acc_mine = (unsigned int)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  unsigned int acc_run, acc_nth;                       /* which planes, and which wave of them */
  if (acc_waves >= 8 * ACC_FLAT_SPREAD) {
    /* a die takes an eighth of every plane, and all dies go through the planes together */
    const unsigned int acc_die = blockIdx.x % ACC_XCDS, acc_turn = blockIdx.x / ACC_XCDS;
    const unsigned int acc_blocks = ((acc_waves + ACC_XCDS - 1) / ACC_XCDS + acc_waves_of_block - 1) / acc_waves_of_block;
    const unsigned int acc_from = acc_waves * acc_die / ACC_XCDS, acc_to = acc_waves * (acc_die + 1) / ACC_XCDS;
    acc_run = acc_turn / acc_blocks;
    acc_nth = acc_from + (acc_turn - acc_run * acc_blocks) * acc_waves_of_block + acc_mine;
    if (acc_nth >= acc_to) return;                               /* whole wave leaves together */
  } else {
    /* planes of a few waves: a die takes one contiguous run of them */
    const unsigned int acc_number = (unsigned int)acc_xcd_contiguous_block() * acc_waves_of_block + acc_mine;
    acc_run = acc_number / acc_waves;
    acc_nth = acc_number - acc_run * acc_waves;
  }
  const int acc_z0 = (int)acc_run * ACC_FLAT_PLANES;
  if (acc_z0 >= acc_d) return;
  /* (lanes before the first and beyond the last vector of a plane do that one again, and store nothing) */
  const int acc_place = (int)(acc_nth * ACC_OWNED) + acc_lane() - ACC_GIVE;
  const bool acc_stores = (!ACC_GIVE || (acc_lane() > 0 && acc_lane() < ACC_WAVE - 1)) && acc_place < (int)acc_per_plane;
  const unsigned int acc_id = (unsigned int)acc_max(0, acc_min(acc_place, (int)acc_per_plane - 1));
  const int acc_y = (int)(acc_id / acc_vectors);
  const int acc_x = acc_min((int)(acc_id % acc_vectors) * ACC_SVEC, acc_w - ACC_SVEC);

#define ACC_DECLARE_A(c, CT, OUTSIDE, arg)                                                          \
  acc_flat_source<CT, ACC_BOUNDARY> acc_a##c;                                                       \
  acc_a##c.base = (const char *)arrStencil_##c;                                                     \
  acc_a##c.plane_bytes = (Int64)acc_h * acc_w * (Int64)sizeof(CT);                                  \
  acc_a##c.d = acc_d; acc_a##c.z0 = acc_z0; acc_a##c.outside = (CT)OUTSIDE;                         \
  acc_a##c.place(acc_x, acc_y, acc_w, acc_h);
  ACC_SRC1_COMPONENTS(ACC_DECLARE_A, 0)
#undef ACC_DECLARE_A
#define ACC_CALL_A(c, CT, OUTSIDE, call) acc_a##c.call;
#define ACC_EACH(call) do { ACC_SRC1_COMPONENTS(ACC_CALL_A, call) } while (0)
#pragma unroll
  for (int acc_i = 0; acc_i < acc_min(ACC_NR, ACC_FIRST); ++acc_i) ACC_EACH(ask(acc_i));
  __builtin_amdgcn_sched_barrier(0);                     /* (every request ahead of anything that waits for one) */
#pragma unroll
  for (int acc_i = 0; acc_i < 2 * ACC_RADIUS_Z; ++acc_i) ACC_EACH(settle(acc_i));

#pragma unroll
  for (int acc_z = 0; acc_z < ACC_FLAT_PLANES; ++acc_z) {
    if (acc_z0 + acc_z >= acc_d) return;                           /* the last run may be short */
    if (acc_z + ACC_FIRST < ACC_NR) ACC_EACH(ask(acc_z + ACC_FIRST));
    __builtin_amdgcn_sched_barrier(0);
    ACC_EACH(settle(acc_z + 2 * ACC_RADIUS_Z));
    acc_out_vec acc_res;
#pragma unroll
    for (int acc_k = 0; acc_k < ACC_SVEC; ++acc_k) {
#define ACC_WINDOW_READ(c, dz, dy, dx) acc_a##c.window[acc_z + ACC_RADIUS_Z + (dz)][ACC_RADIUS_Y + (dy)].e[ACC_RADIUS_X + acc_k + (dx)]
      ACC_STENCIL_TAPS1(ACC_WINDOW_READ)
#undef ACC_WINDOW_READ
      acc_res.v[acc_k] = (T)(ACC_STENCIL_FN);
    }
    if (!acc_stores) continue;
#define ACC_STORE_COMPONENT(c, CT)                                                                  \
    {                                                                                               \
      typedef CT acc_out_native __attribute__((ext_vector_type(ACC_SVEC)));                       \
      typedef acc_out_native acc_out_stored __attribute__((aligned(ACC_FLAT_ALIGN(CT))));         \
      char *plane = (char *)arrOut_##c + (Int64)(acc_z0 + acc_z) * ((Int64)acc_h * acc_w * (Int64)sizeof(CT)); \
      const unsigned int at = ((unsigned int)acc_y * (unsigned int)acc_w + (unsigned int)acc_x) * (unsigned int)sizeof(CT); \
      acc_out_native nv;                                                                          \
      _Pragma("unroll") for (int acc_k = 0; acc_k < ACC_SVEC; ++acc_k) nv[acc_k] = ACC_COMPONENT(acc_res.v[acc_k], c); \
      if (ACC_STENCIL_NT & 1) __builtin_nontemporal_store(nv, (acc_out_stored *)(plane + at));    \
      else                    *(acc_out_stored *)(plane + at) = nv;                               \
    }
    ACC_FOR_COMPONENTS(ACC_STORE_COMPONENT)
#undef ACC_STORE_COMPONENT
  }
#undef ACC_EACH
#undef ACC_CALL_A
}
