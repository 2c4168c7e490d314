/*
 * skel_stencil_flat.h -- 3-D stencils with taps in other planes, on volumes whose rows do not divide into strips.
 *
 * The strips of skel_stencil.h are 64 lanes of one row each: a row of 300 columns is two strips of 256 or three of 128,
 * of which a fifth of the lanes lie outside the volume, every strip ends amid a cache line that another one writes the
 * rest of, and what stands left and right of a strip is gathered for every plane anew.  Here the lanes are laid over the
 * vectors of a whole plane, row after row (bands of ACC_TZ rows): a wave takes 64 consecutive vectors wherever rows end
 * among them, so no lane is idle and consecutive waves read and write consecutive memory.  A wave walks through
 * `acc_walk` planes with the rows that its results read in registers, ACC_NZ rows side by side of 2 rz + 1 planes and
 * those asked for ahead, as the strips do.  What differs:
 *   - the columns left and right of a lane's vector are read by the lane itself, from the cache lines its neighbours
 *     read at the same time; no lane hands anything to another, so it does not matter where its neighbours are;
 *   - the boundary condition along rows and columns is worked out once, before the walk: it is the offset within a
 *     plane that each of the lane's reads goes to, the same in every plane;
 *   - the last vector of a row ends where the row ends (it overlaps its neighbour, whose columns it produces a second
 *     time, the same values).
 * The planes of a run that are read by the run before or after it, and the rows shared with the wave before or after,
 * come out of the L2: a die takes one contiguous run of the workgroups.
 *
 * What bounds it: the memory side.  7 points on 300^3 Float32, 216 MB: 77 us in strips, which read 1.86 and wrote 1.32
 * times what they had to; 54.6 us (4.0 TB/s) here, reading 1.11 and writing 1.06 times, with less than half the vector
 * instructions.  (The same launch on operands that the memory-side cache holds: 35 us.)  Non-temporal stores, a wave
 * through 8 planes, 57.1 us, ordinary ones 60.0; workgroups of 1024 64, of 64 63.
 *
 * Generated definitions expected: those of skel_stencil.h, for ACC_STENCIL_RANK 3 and one source; the planes of source
 * and result are smaller than 4 GB (the driver sees to it), the rows no shorter than a vector.
 */

#ifndef ACC_SVEC
#define ACC_SVEC 4
#endif
#define ACC_NR    (2 * ACC_RADIUS_Z + 1)              /* planes a result depends on */
#define ACC_RING  (ACC_NR + ACC_PREFETCH)             /* planes held in registers */
#define ACC_WW    (ACC_SVEC + 2 * ACC_RADIUS_X)       /* row window of one lane */
#define ACC_NZ    (2 * ACC_RADIUS_Y + ACC_TZ)         /* rows held side by side */

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

/* one component of the source as a lane sees it */
template <typename S, int MODE>
struct acc_flat_source {
  struct row { S e[ACC_WW]; };
  struct __attribute__((aligned(ACC_ALIGNED ? ACC_SVEC * sizeof(S) : alignof(S)))) vec { S v[ACC_SVEC]; };
  static constexpr int SIDE = ACC_RADIUS_X > 0 ? ACC_RADIUS_X : 1;

  const char *base;
  Int64 plane_bytes;
  int d, z0;
  S outside;
  unsigned int row_at[ACC_NZ];         /* bytes from the start of a plane to each of the rows */
  unsigned int own;                    /* ... and from the start of a row to the vector and its neighbours */
  unsigned int left[SIDE], right[SIDE];
  unsigned int rows_in, left_in, right_in;         /* constant boundary: which of them lie inside */
  row ring[ACC_NZ][ACC_RING];

  ACC_DEV void place(const int x, const int y, const int w, const int h)
  {
    rows_in = left_in = right_in = 0;
#pragma unroll
    for (int p = 0; p < ACC_NZ; ++p) {
      const int gy = y - ACC_RADIUS_Y + p;
      row_at[p] = (unsigned int)acc_flat_boundary<MODE>(gy, h) * (unsigned int)w * (unsigned int)sizeof(S);
      rows_in |= (gy >= 0 && gy < h ? 1u : 0u) << p;
    }
    own = (unsigned int)x * (unsigned int)sizeof(S);
#pragma unroll
    for (int j = 0; j < ACC_RADIUS_X; ++j) {
      const int l = x - ACC_RADIUS_X + j, r = x + ACC_SVEC + j;
      left[j] = (unsigned int)acc_flat_boundary<MODE>(l, w) * (unsigned int)sizeof(S);
      right[j] = (unsigned int)acc_flat_boundary<MODE>(r, w) * (unsigned int)sizeof(S);
      left_in |= (l >= 0 ? 1u : 0u) << j;
      right_in |= (r < w ? 1u : 0u) << j;
    }
  }
  /* plane z0 - rz + rho into ring slot `slot` */
  ACC_DEV void fetch(const int rho, const int slot)
  {
    const int gz = z0 - ACC_RADIUS_Z + rho;
    const char *plane = base + (Int64)acc_flat_boundary<MODE>(gz, d) * plane_bytes;
    const bool plane_in = MODE != ACC_B_CONSTANT || (gz >= 0 && gz < d);
#pragma unroll
    for (int p = 0; p < ACC_NZ; ++p) {
      row &r = ring[p][slot];
      const vec v = *(const vec *)(plane + (row_at[p] + own));
      const bool in = plane_in && (MODE != ACC_B_CONSTANT || ((rows_in >> p) & 1u));
#pragma unroll
      for (int k = 0; k < ACC_SVEC; ++k) r.e[ACC_RADIUS_X + k] = in ? v.v[k] : outside;
#pragma unroll
      for (int j = 0; j < ACC_RADIUS_X; ++j) {
        const S l = *(const S *)(plane + (row_at[p] + left[j])), t = *(const S *)(plane + (row_at[p] + right[j]));
        r.e[j] = (MODE != ACC_B_CONSTANT || (in && ((left_in >> j) & 1u))) ? l : outside;
        r.e[ACC_RADIUS_X + ACC_SVEC + j] = (MODE != ACC_B_CONSTANT || (in && ((right_in >> j) & 1u))) ? t : outside;
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
  const int acc_d = (int)shOut_2, acc_h = (int)shOut_1, acc_w = (int)shOut_0;
  /* (the driver counts the waves by the same numbers, all of them within 32 bits) */
  const unsigned int acc_vectors = ((unsigned int)acc_w + ACC_SVEC - 1) / ACC_SVEC, acc_bands = ((unsigned int)acc_h + ACC_TZ - 1) / ACC_TZ;
  const unsigned int acc_per_plane = acc_vectors * acc_bands, acc_waves = (acc_per_plane + ACC_WAVE - 1) / ACC_WAVE;
  const unsigned int acc_number = (unsigned int)acc_xcd_contiguous_block() * (ACC_BLOCK / ACC_WAVE) +
                              (unsigned int)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const unsigned int acc_run = acc_number / acc_waves;
  const int acc_z0 = (int)acc_run * acc_walk;
  if (acc_z0 >= acc_d) return;                                   /* whole wave leaves together */
  const int acc_planes = acc_min(acc_walk, acc_d - acc_z0);
  /* (lanes beyond the last vector of a plane do the last one again) */
  const unsigned int acc_id = acc_min<unsigned int>((acc_number - acc_run * acc_waves) * ACC_WAVE + (unsigned int)acc_lane(), acc_per_plane - 1);
  const int acc_y = (int)(acc_id / acc_vectors) * ACC_TZ;
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

  const int acc_total = acc_planes + 2 * ACC_RADIUS_Z;
#pragma unroll
  for (int acc_rho = 0; acc_rho < ACC_RING - 1; ++acc_rho) ACC_EACH(fetch(acc_min(acc_rho, acc_total - 1), acc_rho));
  __builtin_amdgcn_sched_barrier(0);                     /* (every request ahead of anything that waits for one) */

  for (int acc_zb = 0; acc_zb < acc_planes; acc_zb += ACC_RING) {
#pragma unroll
    for (int acc_s = 0; acc_s < ACC_RING; ++acc_s) {
      const int acc_z = acc_zb + acc_s;
      if (acc_z < acc_planes) {
        /* asked for without a test -- a load under a condition is waited for on the spot: past the end of the run the
         * last plane again, into a slot nothing reads any more */
        ACC_EACH(fetch(acc_min(acc_z + ACC_RING - 1, acc_total - 1), (acc_s + ACC_RING - 1) % ACC_RING));
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int acc_py = 0; acc_py < ACC_TZ; ++acc_py) {
          acc_out_vec acc_res;
#pragma unroll
          for (int acc_k = 0; acc_k < ACC_SVEC; ++acc_k) {
#define ACC_WINDOW_READ(c, dz, dy, dx) acc_a##c.ring[acc_py + ACC_RADIUS_Y + (dy)][(acc_s + ACC_RADIUS_Z + (dz)) % ACC_RING].e[ACC_RADIUS_X + acc_k + (dx)]
            ACC_STENCIL_TAPS1(ACC_WINDOW_READ)
#undef ACC_WINDOW_READ
            acc_res.v[acc_k] = (T)(ACC_STENCIL_FN);
          }
          if (ACC_TZ > 1 && acc_y + acc_py >= acc_h) continue;       /* the last band of rows may be short */
#define ACC_STORE_COMPONENT(c, CT)                                                                  \
          {                                                                                         \
            typedef CT acc_out_native __attribute__((ext_vector_type(ACC_SVEC)));                   \
            typedef acc_out_native acc_out_stored __attribute__((aligned(ACC_ALIGNED ? ACC_SVEC * sizeof(CT) : alignof(CT)))); \
            char *plane = (char *)arrOut_##c + (Int64)(acc_z0 + acc_z) * ((Int64)acc_h * acc_w * (Int64)sizeof(CT)); \
            const unsigned int at = ((unsigned int)(acc_y + acc_py) * (unsigned int)acc_w + (unsigned int)acc_x) * (unsigned int)sizeof(CT); \
            acc_out_native nv;                                                                      \
            _Pragma("unroll") for (int acc_k = 0; acc_k < ACC_SVEC; ++acc_k) nv[acc_k] = ACC_COMPONENT(acc_res.v[acc_k], c); \
            if (ACC_STENCIL_NT & 1) __builtin_nontemporal_store(nv, (acc_out_stored *)(plane + at)); \
            else                    *(acc_out_stored *)(plane + at) = nv;                           \
          }
          ACC_FOR_COMPONENTS(ACC_STORE_COMPONENT)
#undef ACC_STORE_COMPONENT
        }
      }
    }
  }
#undef ACC_EACH
#undef ACC_CALL_A
}
