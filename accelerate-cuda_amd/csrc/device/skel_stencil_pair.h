/*
 * skel_stencil_pair.h -- several applications of a 2-D stencil in one launch, for a call that applies one many times
 * (acc_exec_stencil_iterate): what lies between them stays in registers, and most of the arrays' trips through memory are
 * gone.  Four, three and two (ACC_PAIR_LEVELS) are modules of their own, which are compiled at the same time: the three
 * in one took 1.4 s, a module takes 0.75.
 *
 * A wave owns a strip of columns, 64 vectors of ACC_SVEC less the outermost ones on either side, and `acc_walk` rows of the
 * result.  It walks down the source from as many rows above them as there are applications (times ry) to as many below,
 * ACC_AHEAD rows asked for ahead; every row it takes gives one row of each level -- the source, the first application's
 * result, the second's -- as soon as the 2 ry + 1 rows that one reads are there, and the last level's goes out.  Lanes hand
 * each other the columns beside their own (DPP wave shifts).  What the outermost lanes work out goes wrong one column
 * further in with every level; there are as many of them as that takes, and nothing of theirs is stored.  The last strip of
 * a row ends where the row ends (it overlaps its neighbour, whose columns it produces a second time, the same values).
 *
 * The boundary condition holds for every application, each at the edge of its own source: the row above the first row of a
 * level is the first one again under `clamp`, not what the stencil makes of rows above the array.  Waves at the left and
 * right edges put in place what their edge lanes' neighbours should have said (XEDGE), waves at the top and bottom the rows
 * outside, level by level, as the row arrives that stands for them (YEDGE).  (`wrap` is the exception: what stands left of
 * the array is its right end, and what stands above it its bottom, in between as well; such rows and columns are read and
 * worked out there.)
 *
 * Every second band of walks goes up from its last row instead of down from its first, so that of two walks that read
 * the same rows both begin or both end with them, at about the same time and in one L2 (a die takes one contiguous run of
 * the walks; walks at the upper and lower edge all go down).  All of them down, 8192 x 8192 Float32, 3 x 3: four
 * applications 119 us and now 116, three 112 and now 107; 5 points 118 / 114 and now 112 / 107; 5003 x 8000 75 / 72 and now
 * 70 / 66; 7001 x 5002 Float64 125 / 118 and now 123 / 116; arrays that the memory-side cache holds the same.
 *
 * What bounds it: memory -- waves that walk copy at 5.4 TB/s at best, 100 us for 8192 x 8192 Float32 -- with the vector
 * units close behind (15 instructions an element and application of 3 x 3, 105 us for four).  3 x 3 on 8192 x 8192
 * Float32: four applications 116 us and three 107, one by itself 88; two a launch, in strips that asked for all their rows
 * at once, 96.  Ten in a call, two of them by themselves: 884 us one a launch, 554 in pairs, 405 so.  Four, three, two and one by
 * itself: 3000 x 3000 Float32 27.1 / 20.9 / 16.2 / 15.9, Float64 33.2 / 25.9 / 22.3 / 27.1, 500 x 500 Float32 7.2 / 5.8 / 4.8 / 3.2
 * (launches count).  Two are there for calls of five and six on arrays that the memory-side cache holds: 3000 x 3000 Float64 77 /
 * 68.5 and 108 / 100 without and with them.  Walks of 28
 * rows: of 16 / 20 / 24 / 32 / 36 / 40 rows four take 126 / 121 / 119 / 117 / 120 / 118 us (4001 x 8191: 59 / 59 / 59 /
 * 61 / 59 / 61, and 59); shorter ones where the array would give too few waves (the driver's rule).  Six rows ahead instead
 * of three: the same.  Non-temporal stores: 8192 x 8192 the same, arrays that the memory-side cache holds a tenth slower.
 *
 * Generated definitions expected: ACC_PAIR_LEVELS and those of skel_stencil.h, for ACC_STENCIL_RANK 2, one source of one component of the
 * result's type, no arrays in the environment, taps at most one row and one column away; rows as long as a strip, or at
 * least as much longer as the outermost lanes of one side are wide; three rows or more.
 */

#ifndef ACC_SVEC
#define ACC_SVEC 4
#endif
#define ACC_RY ACC_RADIUS_Y
#define ACC_RX ACC_RADIUS_X
#define ACC_NR (2 * ACC_RY + 1)
#define ACC_WW (ACC_SVEC + 2 * ACC_RX)
#define ACC_AHEAD 3                                   /* rows asked for ahead; the walk is written out in as many steps */
static_assert(ACC_AHEAD % ACC_NR == 0, "windows and rows ahead come round together");
static_assert(ACC_RADIUS_X <= 1 && ACC_RADIUS_Y <= 1 && ACC_SVEC >= 2, "a lane hands its neighbours one column");

#define ACC_B_CLAMP 0
#define ACC_B_MIRROR 1
#define ACC_B_WRAP 2
#define ACC_B_CONSTANT 3

#define ACC_DPP_WAVE_ROL1 0x134
#define ACC_DPP_WAVE_ROR1 0x13C
/* the neighbouring lane's value; the lane that has no neighbour gets that of the wave's other end.  (What it makes of it is
 * dropped, but the element function sees nothing that is no value of the array: one that loops until its operands meet
 * need not end for a made-up zero.  A value kept for that lane takes a move: 8192 x 8192, ten applications, 404 us so, 410 with
 * it; 3000 x 3000 Float64 105 / 108.) */
template <int CTRL>
ACC_DEV ACC_ELT acc_pair_shift(const ACC_ELT &x)
{
  unsigned int s[acc_words<ACC_ELT>::n];
  __builtin_memcpy(s, &x, sizeof(ACC_ELT));
#pragma unroll
  for (int w = 0; w < acc_words<ACC_ELT>::n; ++w) s[w] = (unsigned int)__builtin_amdgcn_update_dpp(0, (int)s[w], CTRL, 0xf, 0xf, true);
  ACC_ELT r;
  __builtin_memcpy(&r, s, sizeof(ACC_ELT));
  return r;
}
struct acc_pair_own { ACC_ELT v[ACC_SVEC]; };
struct acc_pair_row { ACC_ELT e[ACC_WW]; };

template <int acc_levels>
ACC_DEV void acc_applications(ACC_OUT_PARAMS ACC_SRC1_PARAMS, const int acc_walk)
{
  typedef ACC_ELT T;
  constexpr int acc_outer = ACC_RX > 0 ? (acc_levels + ACC_SVEC - 1) / ACC_SVEC : 1;      /* lanes at either side whose columns go wrong, one more a level */
  constexpr int acc_owned = (ACC_WAVE - 2 * acc_outer) * ACC_SVEC;
  const int acc_h = (int)shOut_1, acc_w = (int)shOut_0;
  const int acc_me = acc_lane();
  const unsigned int acc_strips = ((unsigned int)acc_w + acc_owned - 1) / acc_owned;
  const unsigned int acc_number = (unsigned int)acc_xcd_contiguous_block() * (ACC_BLOCK / ACC_WAVE) +
                              (unsigned int)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int acc_y0 = (int)(acc_number / acc_strips) * acc_walk;
  if (acc_y0 >= acc_h) return;                                   /* whole wave leaves together */
  const int acc_y1 = acc_min(acc_y0 + acc_walk, acc_h);
  /* the last strip ends at the right edge, and the one before it leaves whole vectors for its outer lanes: a lane is
   * inside the array, or outside, with all its columns */
  const int acc_nth = (int)(acc_number % acc_strips), acc_last_x0 = acc_w - acc_owned;
  const int acc_x0 = acc_nth == (int)acc_strips - 1 ? acc_last_x0 : acc_min(acc_nth * acc_owned, acc_last_x0 - acc_outer * ACC_SVEC);
  const int acc_gx = acc_x0 + (acc_me - acc_outer) * ACC_SVEC;         /* this lane's first column */
  /* where it reads: its own columns; outside the array the other end of the row, or the nearest vector inside */
  const int acc_from = ACC_BOUNDARY == ACC_B_WRAP ? (acc_gx < 0 ? acc_gx + acc_w : (acc_gx >= acc_w ? acc_gx - acc_w : acc_gx)) : acc_max(0, acc_min(acc_gx, acc_w - ACC_SVEC));
  const bool acc_at_left = acc_gx == 0, acc_at_right = acc_gx + ACC_SVEC == acc_w;
  const bool acc_stores = acc_me >= acc_outer && acc_me < ACC_WAVE - acc_outer;
#define ACC_OUTSIDE_OF(c, CT, OUTSIDE, arg) const T acc_outside = (T)OUTSIDE;
  ACC_SRC1_COMPONENTS(ACC_OUTSIDE_OF, 0)
#undef ACC_OUTSIDE_OF

  auto acc_load = [&](const int y) -> acc_pair_own {         /* y inside the array */
    struct __attribute__((aligned(ACC_ALIGNED ? ACC_SVEC * sizeof(T) : alignof(T)))) vec { T v[ACC_SVEC]; };
    const vec own = *(const vec *)(arrStencil_0 + (Int64)y * acc_w + acc_from);
    acc_pair_own r;
#pragma unroll
    for (int acc_k = 0; acc_k < ACC_SVEC; ++acc_k) r.v[acc_k] = own.v[acc_k];
    return r;
  };
  /* a row with the columns beside each lane's own */
  auto acc_widen = [&](const acc_pair_own &own, auto xedge_c) -> acc_pair_row {
    constexpr bool xedge = decltype(xedge_c)::value && ACC_BOUNDARY != ACC_B_WRAP;
    acc_pair_row r;
#pragma unroll
    for (int acc_k = 0; acc_k < ACC_SVEC; ++acc_k) r.e[ACC_RX + acc_k] = own.v[acc_k];
    if (ACC_RX > 0) {
      T l = acc_pair_shift<ACC_DPP_WAVE_ROR1>(own.v[ACC_SVEC - 1]), t = acc_pair_shift<ACC_DPP_WAVE_ROL1>(own.v[0]);
      if (xedge) {
        const T beyond_l = ACC_BOUNDARY == ACC_B_CONSTANT ? acc_outside : own.v[ACC_BOUNDARY == ACC_B_MIRROR ? 1 : 0];
        const T beyond_r = ACC_BOUNDARY == ACC_B_CONSTANT ? acc_outside : own.v[ACC_BOUNDARY == ACC_B_MIRROR ? ACC_SVEC - 2 : ACC_SVEC - 1];
        l = acc_at_left ? beyond_l : l;
        t = acc_at_right ? beyond_r : t;
      }
      r.e[0] = l;
      r.e[ACC_WW - 1] = t;
    }
    return r;
  };
  auto acc_put = [&](const int y, const acc_pair_own &acc_res) {
    if (!acc_stores) return;
    typedef T acc_out_native __attribute__((ext_vector_type(ACC_SVEC)));
    typedef acc_out_native acc_out_stored __attribute__((aligned(ACC_ALIGNED ? ACC_SVEC * sizeof(T) : alignof(T))));
    acc_out_native nv;
#pragma unroll
    for (int acc_k = 0; acc_k < ACC_SVEC; ++acc_k) nv[acc_k] = acc_res.v[acc_k];
    acc_out_stored *dst = (acc_out_stored *)(arrOut_0 + (Int64)y * acc_w + acc_gx);
    if (ACC_STENCIL_NT & 1) __builtin_nontemporal_store(nv, dst);
    else                    *dst = nv;
  };

  auto acc_run = [&](auto xedge_c, auto acc_yedge_c, auto acc_up_c) {
    constexpr bool acc_yedge = decltype(acc_yedge_c)::value, acc_up = decltype(acc_up_c)::value;
    /* the row of the source that the walk begins with */
    const int acc_first = acc_up ? acc_y1 - 1 + acc_levels * ACC_RY : acc_y0 - acc_levels * ACC_RY;
    const int acc_rows = acc_y1 - acc_y0 + 2 * acc_levels * ACC_RY;  /* ... and how many it takes */
    /* the source's row that stands for row y, which may lie outside (what is asked for beyond the walk is not looked at) */
    auto acc_row_of = [&](const int y) -> int {
      if (acc_yedge && ACC_BOUNDARY == ACC_B_WRAP) return ((y % acc_h) + acc_h) % acc_h;
      return acc_yedge ? acc_max(0, acc_min(y, acc_h - 1)) : acc_up ? acc_max(0, y) : acc_min(y, acc_h - 1);
    };
    acc_pair_own acc_ahead[ACC_AHEAD];
    acc_pair_row acc_window[acc_levels][ACC_NR];                     /* of the source and of what lies between: the rows that the next application reads */
#pragma unroll
    for (int i = 0; i < ACC_AHEAD; ++i) acc_ahead[i] = acc_load(acc_row_of(acc_first + (acc_up ? -i : i)));
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int acc_l = 0; acc_l < acc_levels; ++acc_l)
#pragma unroll
      for (int i = 0; i < ACC_NR; ++i)
#pragma unroll
        for (int k = 0; k < ACC_WW; ++k) acc_window[acc_l][i].e[k] = acc_outside;

    for (int acc_base = 0; acc_base < acc_rows; acc_base += ACC_AHEAD) {
#pragma unroll
      for (int acc_u = 0; acc_u < ACC_AHEAD; ++acc_u) {
        const int acc_s = acc_base + acc_u;
        if (acc_s >= acc_rows) return;
        acc_pair_own acc_next = acc_ahead[acc_u];
        acc_ahead[acc_u] = acc_load(acc_row_of(acc_first + (acc_up ? -1 : 1) * (acc_s + ACC_AHEAD)));
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int acc_l = 0; acc_l < acc_levels; ++acc_l) {
          acc_pair_row (&acc_rows_of)[ACC_NR] = acc_window[acc_l];
          const int acc_newest = acc_u % ACC_NR, acc_before = (acc_u + 2 * ACC_NR - 1) % ACC_NR, acc_oldest = (acc_u + 1) % ACC_NR;
          acc_rows_of[acc_newest] = acc_widen(acc_next, xedge_c);
          if (acc_yedge && ACC_RY > 0 && ACC_BOUNDARY != ACC_B_WRAP) {
            /* the row above the first and the one below the last, of this level's own rows */
            const int y = acc_first + acc_s - acc_l * ACC_RY;
            if (ACC_BOUNDARY == ACC_B_CONSTANT) {
              if (y == 0 || y >= acc_h) {
#pragma unroll
                for (int k = 0; k < ACC_WW; ++k) {
                  if (y == 0) acc_rows_of[acc_before].e[k] = acc_outside;
                  else        acc_rows_of[acc_newest].e[k] = acc_outside;
                }
              }
            } else {
              if (ACC_BOUNDARY == ACC_B_CLAMP && y == 0) acc_rows_of[acc_before] = acc_rows_of[acc_newest];
              if (ACC_BOUNDARY == ACC_B_MIRROR && y == 1) acc_rows_of[acc_oldest] = acc_rows_of[acc_newest];
              if (y == acc_h) acc_rows_of[acc_newest] = acc_rows_of[ACC_BOUNDARY == ACC_B_MIRROR ? acc_oldest : acc_before];
            }
          }
          if (acc_s < 2 * (acc_l + 1) * ACC_RY) break;               /* the next level's first row that is wanted is not due yet */
          acc_pair_own acc_res;
#pragma unroll
          for (int acc_k = 0; acc_k < ACC_SVEC; ++acc_k) {
#define ACC_WINDOW_READ(c, dz, dy, dx) acc_rows_of[(acc_u + 1 + ACC_RY + (acc_up ? -(dy) : (dy))) % ACC_NR].e[ACC_RX + acc_k + (dx)]
            ACC_STENCIL_TAPS1(ACC_WINDOW_READ)
#undef ACC_WINDOW_READ
            acc_res.v[acc_k] = (T)(ACC_STENCIL_FN);
          }
          acc_next = acc_res;
          if (acc_l == acc_levels - 1) acc_put(acc_up ? acc_y1 - 1 - (acc_s - 2 * acc_levels * ACC_RY) : acc_y0 + acc_s - 2 * acc_levels * ACC_RY, acc_res);
        }
      }
    }
  };
  const bool acc_goes_up = ((acc_number / acc_strips) & 1) != 0;
  if (acc_y0 < acc_levels * ACC_RY || acc_y1 + acc_levels * ACC_RY > acc_h) acc_run(acc_bool<true>(), acc_bool<true>(), acc_bool<false>());
  else if (acc_x0 < acc_outer * ACC_SVEC || acc_x0 + acc_owned + acc_outer * ACC_SVEC > acc_w) acc_run(acc_bool<true>(), acc_bool<false>(), acc_bool<false>());
  else if (acc_goes_up) acc_run(acc_bool<false>(), acc_bool<false>(), acc_bool<true>());
  else acc_run(acc_bool<false>(), acc_bool<false>(), acc_bool<false>());
}

extern "C" __global__ void __launch_bounds__(ACC_BLOCK)
stencil(ACC_ENV_PARAMS ACC_OUT_PARAMS ACC_SRC1_PARAMS, const int acc_walk ACC_GUARD_PARAM)
{
  ACC_GUARD_CHECK
  acc_applications<ACC_PAIR_LEVELS>(shOut_1, shOut_0, arrOut_0, arrStencil_0, acc_walk);
}
