"""Segmented folds and folds along rows of few segments, which are dealt out over more workgroups than one for every 256
of them: counts either side of a half, a quarter and an eighth of a workgroup's lanes and of several workgroups, segments
short and of several staged chunks, empty ones among them.  An operator that is associative and does not commute, from
either side, against the same chain in numpy (whole numbers, exact), and Float32 sums of segments of fewer than 128
elements, which are the sequential fold's in every bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

AFFINE = """
__device__ __forceinline__ Word32 affine16(Word32 x, Word32 y) {
  Word32 a1 = x >> 16, b1 = x & 0xffffu, a2 = y >> 16, b2 = y & 0xffffu;
  return (((a1 * a2) & 0xffffu) << 16) | ((a1 * b2 + b1) & 0xffffu);
}
"""
SEED = 0x00030005


def affine(x, y):
    a1, b1, a2, b2 = x >> 16, x & 0xffff, y >> 16, y & 0xffff
    return (((a1 * a2) & 0xffff) << 16) | ((a1 * b2 + b1) & 0xffff)


def chain(x, offs, f, seed):
    """f over every segment from the left, the seed last; all segments side by side"""
    a, b = offs[:-1], offs[1:]
    acc = np.full(len(a), seed, x.dtype)
    live = b > a
    acc[live] = x[a[live]]
    for k in range(1, int((b - a).max(initial=0))):
        live = b - a > k
        acc[live] = f(acc[live], x[a[live] + k])
    return np.where(b > a, f(acc, np.array(seed, x.dtype)), np.array(seed, x.dtype))


@pytest.fixture(scope="module")
def ctx():
    import acchip as A
    return A.Context(0)


COUNTS = (1, 31, 32, 33, 63, 64, 65, 127, 128, 129, 255, 256, 257, 513, 1000, 5003)


@pytest.mark.parametrize("knobs", ["foldseg.giants=0", "foldseg.giants=1", "foldseg.spread=1000,foldseg.spread_min=1"])
@pytest.mark.parametrize("right", [False, True])
def test_segments(ctx, right, knobs):
    import acchip as A
    with A.tuning(knobs, ctx):
        sk = ctx.skeleton(A.SKEL_FOLDSEG, "Word32", env=[(1, "Word32")], get="arrIn0_0[ix]", combine="affine16(x, y)", seed=str(SEED),
                          preamble=AFFINE, flags=A.FLAG_FOLD_RIGHT if right else 0, wait=True)
        fl = ctx.skeleton(A.SKEL_FOLDSEG, "float", env=[(1, "float")], get="arrIn0_0[ix]", combine="x + y", seed="0.5f", wait=True)
    rng = np.random.default_rng(11)
    for nseg in COUNTS:
        for mean in (2, 20, 100):
            print(nseg, mean, flush=True)
            lens = rng.poisson(mean, nseg).clip(0, 127)
            lens[rng.integers(0, nseg, 2)] = 0
            offs = np.concatenate([[0], np.cumsum(lens)]).astype(np.int64)
            x = rng.integers(0, 1 << 32, offs[-1] + 5, dtype=np.uint32)
            out, do = ctx.empty(nseg, np.uint32), ctx.array(offs.astype(np.int32))
            sk.foldseg([ctx.array(x)], len(x), do, out)
            assert np.array_equal(out.get(), chain(x, offs, affine, SEED)), (nseg, mean)
            if not right:
                y = rng.standard_normal(len(x)).astype(np.float32)
                outf = ctx.empty(nseg, np.float32)
                fl.foldseg([ctx.array(y)], len(y), do, outf)
                assert np.array_equal(outf.get(), chain(y, offs, lambda a, b: a + b, 0.5)), (nseg, mean)


@pytest.mark.parametrize("knobs", ["foldseg.giants=0", "foldseg.giants=1"])
@pytest.mark.parametrize("right", [False, True])
def test_long_stretches(ctx, right, knobs):
    """segments of which a staged chunk holds 256 elements or a little less or more, which the whole workgroup then folds, or
    several chunks, among short ones: such a stretch begins where the workgroup's chunks have it begin, so a sum of Float32
    has another association for another number of segments a workgroup, and is held to what any association may be off by"""
    import acchip as A
    with A.tuning(knobs, ctx):
        sk = ctx.skeleton(A.SKEL_FOLDSEG, "Word32", env=[(1, "Word32")], get="arrIn0_0[ix]", combine="affine16(x, y)", seed=str(SEED),
                          preamble=AFFINE, flags=A.FLAG_FOLD_RIGHT if right else 0, wait=True)
        fl = ctx.skeleton(A.SKEL_FOLDSEG, "float", env=[(1, "float")], get="arrIn0_0[ix]", combine="x + y", seed="0.5f", wait=True)
    rng = np.random.default_rng(15)
    for nseg in COUNTS[3:]:
        print(nseg, flush=True)
        lens = rng.poisson(20, nseg)
        at = rng.permutation(nseg)[:6]
        lens[at] = np.array([255, 256, 257, 511, 3000, 9001])[:len(at)]
        offs = np.concatenate([[0], np.cumsum(lens)]).astype(np.int64)
        x = rng.integers(0, 1 << 32, offs[-1] + 5, dtype=np.uint32)
        out, do = ctx.empty(nseg, np.uint32), ctx.array(offs.astype(np.int32))
        sk.foldseg([ctx.array(x)], len(x), do, out)
        assert np.array_equal(out.get(), chain(x, offs, affine, SEED)), nseg
        if not right:
            y = rng.standard_normal(len(x)).astype(np.float32)
            outf = ctx.empty(nseg, np.float32)
            fl.foldseg([ctx.array(y)], len(y), do, outf)
            c, m = (np.concatenate([[0], np.cumsum(v)])[offs] for v in (y.astype(np.float64), np.abs(y).astype(np.float64)))
            # (n additions in any order: n half units in the last place of the sum of the magnitudes)
            assert np.all(np.abs(outf.get() - (np.diff(c) + 0.5)) <= (lens + 1) * 2.0 ** -24 * (np.diff(m) + 0.5) + 1e-9), nseg


@pytest.mark.parametrize("right", [False, True])
def test_rows(ctx, right):
    import acchip as A
    sk = ctx.skeleton(A.SKEL_FOLD, "Word32", env=[(2, "Word32")], out_rank=1, get="arrIn0_0[ix]", combine="affine16(x, y)", seed=str(SEED),
                      preamble=AFFINE, flags=A.FLAG_FOLD_RIGHT if right else 0, wait=True)
    rng = np.random.default_rng(12)
    for rows in COUNTS:
        for w in (17, 32, 63, 127):
            print(rows, w, flush=True)
            x = rng.integers(0, 1 << 32, (rows, w), dtype=np.uint32)
            out = ctx.empty(rows, np.uint32)
            sk.fold([ctx.array(x)], (rows, w), out)
            assert np.array_equal(out.get(), chain(x.ravel(), np.arange(rows + 1) * w, affine, SEED)), (rows, w)


@pytest.mark.parametrize("right", [False, True])
@pytest.mark.parametrize("giants", [0, 1])
def test_beyond_2_31_elements(ctx, giants, right):
    """short segments of a source of more than 2^31 elements (none of them in memory: an element is its index), a last
    workgroup that has lanes without a segment"""
    import acchip as A
    rng = np.random.default_rng(13)
    nseg, last, first = (1 << 25) + 77, 90, (1 << 31) + 1005
    lens = rng.integers(0, 100, last)
    lens[last - 20], lens[last - 7] = 700, 0
    offs = np.full(nseg + 1, first, np.int64)
    offs[nseg - last + 1:] += np.cumsum(lens)
    print(nseg, first, flush=True)
    with A.tuning("foldseg.giants=%d" % giants, ctx):
        sk = ctx.skeleton(A.SKEL_FOLDSEG, "Int64", env=[], get="ix", combine="x + y", seed="5", seg_type="Int64",
                          flags=A.FLAG_FOLD_RIGHT if right else 0, wait=True)
    out = ctx.empty(nseg, np.int64)
    sk.foldseg([], int(offs[-1]) + 3, ctx.array(offs), out)
    got = out.get()
    assert np.all(got[:nseg - last] == 5)
    assert got[nseg - last:].tolist() == [5 + sum(range(int(a), int(b))) for a, b in zip(offs[nseg - last:-1], offs[nseg - last + 1:])]


def test_rows_beyond_2_31_elements(ctx):
    import acchip as A
    rows, w = (1 << 26) + 77, 33
    sk = ctx.skeleton(A.SKEL_FOLD, "Int64", env=[], out_rank=1, get="ix", combine="x + y", seed="0", wait=True)
    out = ctx.empty(rows, np.int64)
    print(rows, w, flush=True)
    sk.fold([], (rows, w), out)
    assert np.array_equal(out.get(), w * (w * np.arange(rows, dtype=np.int64)) + w * (w - 1) // 2)
