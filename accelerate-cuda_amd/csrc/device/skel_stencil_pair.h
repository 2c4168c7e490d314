/*
 * skel_stencil_pair.h -- two applications of a 2-D stencil in one launch, for a call that applies one many times
 * (acc_exec_stencil_iterate): what lies between the two stays in registers, and half of the arrays' trips through
 * memory are gone.
 *
 * A wave owns a strip of 62 vectors of ACC_SVEC columns and ACC_TILE_H rows of the result.  It reads the strip with one
 * vector more to either side and 2 ry rows more above and below, every row at once; its 64 lanes work out the rows in
 * between, 2 ry more than the result has, and from those the result.  Lanes hand each other the columns beside their own
 * (DPP wave shifts).  What the two outermost lanes work out is only right where it does not reach past them -- their
 * columns next to the strip, which is what their neighbours ask for -- and nothing of theirs is stored.  The last strip
 * of a row ends where the row ends (it overlaps its neighbour, whose columns it produces a second time, the same values).
 *
 * The boundary condition holds for both applications, each at the edge of its own source: the row above the first row
 * in between is the first one again under `clamp`, not what the stencil makes of rows above the array.  Waves at the left
 * and right edges put in place what their edge lanes' neighbours should have said (XEDGE), waves at the top and bottom
 * ask for the rows of every row in between by themselves (YEDGE).  (`wrap` is the exception along rows: what stands left
 * of the array is its right end, in between as well, and a lane outside the array reads and works it out there.)
 *
 * What bounds it: memory still, the vector units close behind (an element's two applications are some 45 instructions).
 * Ten applications of 3 x 3 to 8192 x 8192 Float32, two of them by themselves: 884 us one a launch, 558 so (a pair 96 us,
 * a single application 88); 4001 x 8191 464 / 263, 3000 x 3000 Float64 293 / 160 (the arrays stay in the memory-side
 * cache, which ordinary stores leave them in and non-temporal ones do not: 196), 300 x 300 42 / 30, where launches count.
 * Strips of 4 rows: of 2 / 3 / 6 / 8 rows 605 / 569 / 559 / 566 us and, on 300 x 300, 25 / 29 / 37 / 41.
 *
 * Generated definitions expected: those of skel_stencil.h, for ACC_STENCIL_RANK 2, one source of one component of the
 * result's type, no arrays in the environment, taps at most one row and one column away; rows as long as 62 vectors
 * or at least as 63.
 */

#ifndef ACC_SVEC
#define ACC_SVEC 4
#endif
#define ACC_RY ACC_RADIUS_Y
#define ACC_RX ACC_RADIUS_X
#define ACC_NR (2 * ACC_RY + 1)
#define ACC_WW (ACC_SVEC + 2 * ACC_RX)
#define ACC_OWNED (ACC_WAVE - 2)                      /* lanes whose columns are stored */
static_assert(ACC_RADIUS_X <= 1 && ACC_RADIUS_Y <= 1 && ACC_SVEC >= 2, "the outermost lanes supply one column");

#define ACC_B_CLAMP 0
#define ACC_B_MIRROR 1
#define ACC_B_WRAP 2
#define ACC_B_CONSTANT 3

ACC_DEV int acc_pair_boundary(int i, const int sz)
{
  if (ACC_BOUNDARY == ACC_B_MIRROR) i = i < 0 ? -i : (i >= sz ? sz - (i - sz + 2) : i);
  if (ACC_BOUNDARY == ACC_B_WRAP)   i = i < 0 ? sz + i : (i >= sz ? i - sz : i);
  /* clamped in every mode: the maps assume the array spans the stencil; keep the address legal if not */
  return acc_max(0, acc_min(i, sz - 1));
}

#define ACC_DPP_WAVE_SHL1 0x130
struct acc_pair_own { ACC_ELT v[ACC_SVEC]; };
struct acc_pair_row { ACC_ELT e[ACC_WW]; };

extern "C" __global__ void __launch_bounds__(ACC_BLOCK)
stencil(ACC_ENV_PARAMS ACC_OUT_PARAMS ACC_SRC1_PARAMS, const int acc_walk ACC_GUARD_PARAM)
{
  ACC_GUARD_CHECK
  typedef ACC_ELT T;
  ACC_ENV_ASSUME
  (void)acc_walk;
  const int acc_h = (int)shOut_1, acc_w = (int)shOut_0;
  const int acc_me = acc_lane();
  const unsigned int acc_strips = ((unsigned int)acc_w + ACC_OWNED * ACC_SVEC - 1) / (ACC_OWNED * ACC_SVEC);
  const unsigned int acc_number = (unsigned int)acc_xcd_contiguous_block() * (ACC_BLOCK / ACC_WAVE) +
                              (unsigned int)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int acc_y0 = (int)(acc_number / acc_strips) * ACC_TILE_H;
  if (acc_y0 >= acc_h) return;                                   /* whole wave leaves together */
  /* the last strip ends at the right edge, and the one before it leaves a whole vector for its outermost lane: the
   * outermost lanes are inside the array, or outside, with all their columns */
  const int acc_nth = (int)(acc_number % acc_strips), acc_last_x0 = acc_w - ACC_OWNED * ACC_SVEC;
  const int acc_x0 = acc_nth == (int)acc_strips - 1 ? acc_last_x0 : acc_min(acc_nth * (ACC_OWNED * ACC_SVEC), acc_last_x0 - ACC_SVEC);
  const int acc_gx = acc_x0 + (acc_me - 1) * ACC_SVEC;             /* this lane's first column */
  /* where it reads: its own columns; outside the array the other end of the row, or the nearest vector inside */
  const int acc_from = ACC_BOUNDARY == ACC_B_WRAP ? (acc_gx < 0 ? acc_gx + acc_w : (acc_gx >= acc_w ? acc_gx - acc_w : acc_gx)) : acc_max(0, acc_min(acc_gx, acc_w - ACC_SVEC));
  const bool acc_at_left = acc_gx == 0, acc_at_right = acc_gx + ACC_SVEC == acc_w;
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
  auto acc_all_outside = [&]() -> acc_pair_own {
    acc_pair_own r;
#pragma unroll
    for (int acc_k = 0; acc_k < ACC_SVEC; ++acc_k) r.v[acc_k] = acc_outside;
    return r;
  };
  /* a row with the columns beside each lane's own */
  auto acc_widen = [&](const acc_pair_own &own, auto xedge_c) -> acc_pair_row {
    constexpr bool xedge = decltype(xedge_c)::value && ACC_BOUNDARY != ACC_B_WRAP;
    acc_pair_row r;
#pragma unroll
    for (int acc_k = 0; acc_k < ACC_SVEC; ++acc_k) r.e[ACC_RX + acc_k] = own.v[acc_k];
    if (ACC_RX > 0) {
      T l = acc_wave_shift_up1(own.v[ACC_SVEC - 1]), t = acc_dpp<ACC_DPP_WAVE_SHL1, 0xf>(own.v[0], own.v[0]);
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
  /* one application: rows[0 .. 2 ry] are the rows it reads */
  auto acc_apply = [&](const acc_pair_row (&acc_rows)[ACC_NR]) -> acc_pair_own {
    acc_pair_own acc_res;
#pragma unroll
    for (int acc_k = 0; acc_k < ACC_SVEC; ++acc_k) {
#define ACC_WINDOW_READ(c, dz, dy, dx) acc_rows[ACC_RY + (dy)].e[ACC_RX + acc_k + (dx)]
      ACC_STENCIL_TAPS1(ACC_WINDOW_READ)
#undef ACC_WINDOW_READ
      acc_res.v[acc_k] = (T)(ACC_STENCIL_FN);
    }
    return acc_res;
  };
  auto acc_put = [&](const int y, const acc_pair_own &acc_res) {
    if (acc_me == 0 || acc_me == ACC_WAVE - 1) return;
    typedef T acc_out_native __attribute__((ext_vector_type(ACC_SVEC)));
    typedef acc_out_native acc_out_stored __attribute__((aligned(ACC_ALIGNED ? ACC_SVEC * sizeof(T) : alignof(T))));
    acc_out_native nv;
#pragma unroll
    for (int acc_k = 0; acc_k < ACC_SVEC; ++acc_k) nv[acc_k] = acc_res.v[acc_k];
    acc_out_stored *dst = (acc_out_stored *)(arrOut_0 + (Int64)y * acc_w + acc_gx);
    if (ACC_STENCIL_NT & 1) __builtin_nontemporal_store(nv, dst);
    else                    *dst = nv;
  };

  auto acc_run = [&](auto xedge_c, auto yedge_c) {
    constexpr bool yedge = decltype(yedge_c)::value;
    constexpr int READ_ROWS = ACC_TILE_H + 4 * ACC_RY, MID_ROWS = ACC_TILE_H + 2 * ACC_RY;
    acc_pair_own src[READ_ROWS];
    acc_pair_row above[ACC_NR], between[ACC_NR];
    if (!yedge) {
#pragma unroll
      for (int i = 0; i < READ_ROWS; ++i) src[i] = acc_load(acc_y0 - 2 * ACC_RY + i);
      __builtin_amdgcn_sched_barrier(0);                 /* (every request ahead of anything that waits for one) */
#pragma unroll
      for (int i = 0; i < ACC_NR - 1; ++i) above[i + 1] = acc_widen(src[i], xedge_c);
    }
#pragma unroll
    for (int m = 0; m < MID_ROWS; ++m) {
      acc_pair_own mid;
      if (!yedge) {
#pragma unroll
        for (int i = 0; i < ACC_NR - 1; ++i) above[i] = above[i + 1];
        above[ACC_NR - 1] = acc_widen(src[m + ACC_NR - 1], xedge_c);
        mid = acc_apply(above);
      } else {
        /* the row in between that the boundary condition puts here, and the rows that one is made of */
        const int want = acc_y0 - ACC_RY + m, at = acc_pair_boundary(want, acc_h);
#pragma unroll
        for (int i = 0; i < ACC_NR; ++i) {
          const int y = at - ACC_RY + i;
          const acc_pair_own read = acc_load(acc_pair_boundary(y, acc_h));
          above[i] = acc_widen((ACC_BOUNDARY == ACC_B_CONSTANT && (y < 0 || y >= acc_h)) ? acc_all_outside() : read, xedge_c);
        }
        mid = acc_apply(above);
        if (ACC_BOUNDARY == ACC_B_CONSTANT && (want < 0 || want >= acc_h)) mid = acc_all_outside();
      }
#pragma unroll
      for (int i = 0; i < ACC_NR - 1; ++i) between[i] = between[i + 1];
      between[ACC_NR - 1] = acc_widen(mid, xedge_c);
      const int y = acc_y0 + m - 2 * ACC_RY;
      if (m >= 2 * ACC_RY && (!yedge || y < acc_h)) acc_put(y, acc_apply(between));
    }
  };
  if (acc_y0 < 2 * ACC_RY || acc_y0 + ACC_TILE_H + 2 * ACC_RY > acc_h) acc_run(acc_bool<true>(), acc_bool<true>());
  else if (acc_x0 < ACC_SVEC || acc_x0 + (ACC_OWNED + 1) * ACC_SVEC > acc_w) acc_run(acc_bool<true>(), acc_bool<false>());
  else acc_run(acc_bool<false>(), acc_bool<false>());
}
