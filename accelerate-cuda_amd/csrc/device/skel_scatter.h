/*
 * skel_scatter.h -- forward permutation whose combination is the new value (`permute const`):
 *
 *     out = defaults;   for every source index ix:   j = permutation(ix);
 *     unless j is `ignore`:   out[j] = get(ix)
 *
 * The scatter behind `filter`, behind every pass of a sort and behind any reordering (CodeGen/IndexSpace.hs:160-303
 * takes a lock per element for it, as for every permute).  Nothing is read from the result and nothing is locked; of
 * several sources on one target one wins whole, as under any order of the combinations.
 *
 * What bounds it: memory.  The source is read once (a lane takes single elements, a wave's worth side by side, so that
 * the elements of a compaction or of a sorting pass leave a wave as runs of neighbouring targets, which the memory
 * pipeline sends out as whole cache lines), and the stores are ordinary ones that meet in the L2 of the die: every
 * store with device scope goes through to memory by itself.
 *
 * Kernels:
 *   permute        a tile of ACC_BLOCK x ACC_BATCH sources per workgroup; `winner` as below, or NULL
 *   permute_claim  for an element that no single store covers -- a tuple, whose components are arrays of their own, or a
 *                  scalar wider than 8 bytes: every source's index into its target's word of `winner`, where one of them
 *                  stays; `permute` then stores the sources that find their own index there.  (`winner` need not be
 *                  cleared: what is looked at has been written in the same call.)
 *   permute_fill   the defaults into the result
 *   permute_small  all of it in one workgroup, for sources and results of at most ACC_SMALL elements
 *
 * A launch works on the sources [first, past); indices in `winner` count from `first`.
 *
 * The operands that the fragments read at the element's own index (ACC_OWN_*, all of them arrays at least `past` long)
 * are asked for ahead of everything else, for the whole batch: `filter` reads a place only where the element stays, and a
 * read behind such a test is waited for on the spot, one element after the other.  Everything else that the element
 * function reads is read for sources that stay only: what it makes of one that is dropped need not exist.
 *
 * Measured with the operands in HBM, 2^24 Int32 sources, defaults included, through the atomics template (stores of device
 * scope, a lane four elements side by side, reads behind tests) and now: half of them kept in order 64 us -> 49, a sorting
 * pass by 4 bits 146 -> 77, by 8 bits 356 -> 161, a random permutation 392 -> 286, all of them on 10 targets of 2^24 9.7 ms
 * -> 0.05; the scatter of `filter` (flag, place and value of 2^24 read, half stored) 98 -> 27, at 2^20 9.4 -> 4.0.  A lane
 * takes 8 elements (ACC_BATCH): 32 do the sorting pass by 8 bits in 123 us and the random permutation in 262, but the
 * scatter of `filter` in 32, and in 7.2 at 2^20, where they leave half of the device idle.  Pairs of Int32, two launches:
 * 115 / 218 / 595 / 1240 us.
 *
 * Generated definitions expected: ACC_ELT, ACC_NCOMP, ACC_FOR_COMPONENTS, ACC_ENV_PARAMS, ACC_ENV_ASSUME, ACC_OUT_PARAMS,
 * ACC_OUT_SIZE, ACC_GET(ix), ACC_PERMUTATION(ix), ACC_OWN_NAMES, ACC_OWN_FIELDS, ACC_OWN_LOAD(sv, ix), ACC_OWN_WITHIN(past),
 * ACC_GET_OWN(ix), ACC_GET_TOTAL, ACC_PERMUTATION_OWN(ix), ACC_BLOCK, ACC_BATCH, ACC_SMALL.
 */

#define ACC_TILE (ACC_BLOCK * ACC_BATCH)
#define ACC_AHEAD (ACC_GET_TOTAL && ACC_NCOMP == 1)               /* elements worked out with the targets */
#define ACC_CLAIMED (ACC_NCOMP > 1 || sizeof(ACC_ELT) > 8)       /* what no single store of at most 8 bytes writes */

/* What stands in a fragment for a read of an operand at the element's own index: `v`, asked for ahead of the tests, where
 * the array and the index named there are the element's own, as they are unless the fragment gives one of the names to
 * something of its own; there it is the read that was written. */
template <typename T, typename I>
ACC_DEV const T &acc_own_value(const T *a, const I ix, const T *own_a, const Int64 own_ix, const T &v)
{
  return a == own_a && (Int64)ix == own_ix ? v : a[ix];
}
template <typename A, typename I, typename T>
ACC_DEV decltype(auto) acc_own_value(const A &a, const I ix, const T *, const Int64, const T &) { return a[ix]; }

/* Names the kernels share.  A tile that reaches past the end reads the last source there (`in`): no test per element
 * stands in front of a read. */
#define ACC_SCATTER_NAMES                                                                                                           \
  typedef ACC_ELT T;                                                                                                                \
  ACC_ENV_ASSUME                                                                                                                    \
  struct acc_own { ACC_OWN_FIELDS };                                                                                                \
  auto acc_get      = [&](const Int64 ix) -> T { return (ACC_GET(ix)); };                                                           \
  auto acc_perm     = [&](const Int64 ix) -> Int64 { return (Int64)(ACC_PERMUTATION(ix)); };                                        \
  ACC_OWN_NAMES                                                                                                                     \
  auto acc_get_own  = [&](const Int64 ix, const acc_own &acc_sv) -> T { const Int64 acc_own_ix = ix; (void)acc_own_ix; (void)acc_sv; return (ACC_GET_OWN(ix)); }; \
  auto acc_perm_own = [&](const Int64 ix, const acc_own &acc_sv) -> Int64 { const Int64 acc_own_ix = ix; (void)acc_own_ix; (void)acc_sv; return (Int64)(ACC_PERMUTATION_OWN(ix)); }; \
  (void)acc_get; (void)acc_get_own;                                                                                                 \
  const Int64 acc_ntarget = (ACC_OUT_SIZE);                                                                                         \
  const Int64 acc_ix0 = acc_first + (Int64)blockIdx.x * ACC_TILE + threadIdx.x;                                                     \
  auto acc_in = [&](const int k) -> Int64 { return acc_min<Int64>(acc_ix0 + k * ACC_BLOCK, acc_past - 1); };

extern "C" __global__ void __launch_bounds__(ACC_BLOCK)
permute_claim(ACC_ENV_PARAMS ACC_OUT_PARAMS, const Int64 acc_first, const Int64 acc_past, unsigned int *__restrict__ acc_winner ACC_GUARD_PARAM)
{
  ACC_GUARD_CHECK
  ACC_SCATTER_NAMES
  Int64 j[ACC_BATCH];
  if (ACC_OWN_WITHIN(acc_past)) {
    acc_own sv[ACC_BATCH];
#pragma unroll
    for (int k = 0; k < ACC_BATCH; ++k) { ACC_OWN_LOAD(sv[k], acc_in(k)) }
#pragma unroll
    for (int k = 0; k < ACC_BATCH; ++k) j[k] = acc_perm_own(acc_in(k), sv[k]);
  } else {
#pragma unroll
    for (int k = 0; k < ACC_BATCH; ++k) j[k] = acc_perm(acc_in(k));
  }
#pragma unroll
  for (int k = 0; k < ACC_BATCH; ++k)
    if (acc_ix0 + k * ACC_BLOCK < acc_past && j[k] >= 0 && j[k] < acc_ntarget) acc_winner[j[k]] = (unsigned int)(acc_ix0 + k * ACC_BLOCK - acc_first);
}

extern "C" __global__ void __launch_bounds__(ACC_BLOCK)
permute(ACC_ENV_PARAMS ACC_OUT_PARAMS, const Int64 acc_first, const Int64 acc_past, const unsigned int *__restrict__ acc_winner ACC_GUARD_PARAM)
{
  ACC_GUARD_CHECK
  ACC_SCATTER_NAMES
  /* The element function of a source that is dropped may have no value -- the index it reads through may be any number.
   * One that only calculates with the source's own operands has (ACC_GET_TOTAL).  Of any other a lane that stores nothing
   * works out the element of a source of its wave that stays: behind a test every read would be waited for on the spot
   * (2^24 Int32 through an index, half of them kept in order: 65.6 us behind tests, 59 so). */
  Int64 j[ACC_BATCH];
  T x[ACC_BATCH];
  bool mine[ACC_BATCH];
#if ACC_AHEAD
  if (ACC_OWN_WITHIN(acc_past)) {
    acc_own sv[ACC_BATCH];
#pragma unroll
    for (int k = 0; k < ACC_BATCH; ++k) { ACC_OWN_LOAD(sv[k], acc_in(k)) }
#pragma unroll
    for (int k = 0; k < ACC_BATCH; ++k) {
      j[k] = acc_perm_own(acc_in(k), sv[k]);
      x[k] = acc_get_own(acc_in(k), sv[k]);
    }
  } else {
#pragma unroll
    for (int k = 0; k < ACC_BATCH; ++k) j[k] = acc_perm(acc_in(k));
#pragma unroll
    for (int k = 0; k < ACC_BATCH; ++k)
      if (j[k] >= 0 && j[k] < acc_ntarget) x[k] = acc_get(acc_in(k));
  }
#else
  acc_own sv[ACC_BATCH];
  const bool whole = ACC_OWN_WITHIN(acc_past);
  if (whole) {
    asm volatile("");          /* (a request shared with the other form would be made, and waited for, ahead of the branch) */
#pragma unroll
    for (int k = 0; k < ACC_BATCH; ++k) { ACC_OWN_LOAD(sv[k], acc_in(k)) }
#pragma unroll
    for (int k = 0; k < ACC_BATCH; ++k) j[k] = acc_perm_own(acc_in(k), sv[k]);
  } else {
#pragma unroll
    for (int k = 0; k < ACC_BATCH; ++k) j[k] = acc_perm(acc_in(k));
  }
#endif
#pragma unroll
  for (int k = 0; k < ACC_BATCH; ++k) mine[k] = acc_ix0 + k * ACC_BLOCK < acc_past && j[k] >= 0 && j[k] < acc_ntarget;
  if (ACC_CLAIMED) {
    unsigned int w[ACC_BATCH];
#pragma unroll
    for (int k = 0; k < ACC_BATCH; ++k) w[k] = acc_winner[mine[k] ? j[k] : 0];
#pragma unroll
    for (int k = 0; k < ACC_BATCH; ++k) mine[k] = mine[k] && w[k] == (unsigned int)(acc_ix0 + k * ACC_BLOCK - acc_first);
  }
#if !ACC_AHEAD
  Int64 stays = -1;
  acc_own of_stays;
#pragma unroll
  for (int k = ACC_BATCH - 1; k >= 0; --k) {
    const unsigned long long here = __ballot(mine[k]);
    if (here != 0ull) {
      const int lane = __builtin_ctzll(here);
      stays = acc_readlane(acc_in(k), lane);
      of_stays = acc_readlane(sv[k], lane);
    }
  }
  if (stays < 0) return;                                   /* (the whole wave) */
  if (whole) {
#pragma unroll
    for (int k = 0; k < ACC_BATCH; ++k)
      x[k] = ACC_GET_TOTAL ? acc_get_own(acc_in(k), sv[k]) : acc_get_own(mine[k] ? acc_in(k) : stays, mine[k] ? sv[k] : of_stays);
  } else {
#pragma unroll
    for (int k = 0; k < ACC_BATCH; ++k) x[k] = acc_get(mine[k] ? acc_in(k) : stays);
  }
#endif
#pragma unroll
  for (int k = 0; k < ACC_BATCH; ++k)
    if (mine[k]) ACC_SET(arrOut, j[k], x[k]);
}

/* `count` elements of one component, in 16-byte pieces where both arrays lie on such boundaries */
template <typename C>
ACC_DEV void acc_copy_component(C *__restrict__ dst, const C *__restrict__ src, const Int64 count, const Int64 lane, const Int64 lanes)
{
  typedef unsigned int acc_u4 __attribute__((ext_vector_type(4)));
  if (((((unsigned long long)dst) | ((unsigned long long)src)) & 15u) == 0u) {
    const Int64 bytes = count * (Int64)sizeof(C), pieces = bytes / 16;
    for (Int64 i = lane; i < pieces; i += lanes) ((acc_u4 *)dst)[i] = __builtin_nontemporal_load((const acc_u4 *)src + i);
    for (Int64 i = pieces * 16 + lane; i < bytes; i += lanes) ((unsigned char *)dst)[i] = ((const unsigned char *)src)[i];
  } else {
    for (Int64 i = lane; i < count; i += lanes) dst[i] = src[i];
  }
}

extern "C" __global__ void __launch_bounds__(256)
permute_fill(ACC_OUT_ARRAY(arrTo), ACC_CONST_ARRAY(arrFrom), const Int64 count ACC_GUARD_PARAM)
{
  ACC_GUARD_CHECK
  const Int64 lane = (Int64)blockIdx.x * 256 + threadIdx.x, lanes = (Int64)gridDim.x * 256;
#define ACC_COPY_ONE(c, type) acc_copy_component<type>(arrTo_##c, arrFrom_##c, count, lane, lanes);
  ACC_FOR_COMPONENTS(ACC_COPY_ONE)
}

/* One workgroup: the defaults, a wait until they have arrived, the sources.  Below a few thousand elements a call is
 * what its launches cost. */
extern "C" __global__ void __launch_bounds__(1024)
permute_small(ACC_ENV_PARAMS ACC_OUT_PARAMS, ACC_CONST_ARRAY(arrFrom), const int acc_copy, const Int64 acc_n ACC_GUARD_PARAM)
{
  ACC_GUARD_CHECK
  typedef ACC_ELT T;
  ACC_ENV_ASSUME
  __shared__ unsigned int acc_s_winner[ACC_CLAIMED ? ACC_SMALL : 1];
  auto acc_get  = [&](const Int64 ix) -> T { return (ACC_GET(ix)); };
  auto acc_perm = [&](const Int64 ix) -> Int64 { return (Int64)(ACC_PERMUTATION(ix)); };
  const Int64 acc_ntarget = (ACC_OUT_SIZE);
  const int tid = (int)threadIdx.x;
  constexpr int MOST = (ACC_SMALL + 1023) / 1024;
  Int64 j[MOST];
#pragma unroll
  for (int k = 0; k < MOST; ++k) {
    const Int64 ix = tid + k * 1024;
    j[k] = ix < acc_n ? acc_perm(ix) : -1;
    if (j[k] >= acc_ntarget) j[k] = -1;
    if (ACC_CLAIMED && j[k] >= 0) acc_s_winner[j[k]] = (unsigned int)ix;
  }
  if (acc_copy) {
#define ACC_COPY_SMALL(c, type) acc_copy_component<type>(arrOut_##c, arrFrom_##c, acc_ntarget, tid, 1024);
    ACC_FOR_COMPONENTS(ACC_COPY_SMALL)
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");       /* every wave's part has arrived before any wave stores over it */
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < MOST; ++k) {
    const Int64 ix = tid + k * 1024;
    if (j[k] < 0) continue;
    if (ACC_CLAIMED && acc_s_winner[j[k]] != (unsigned int)ix) continue;
    ACC_SET(arrOut, j[k], acc_get(ix));
  }
}
