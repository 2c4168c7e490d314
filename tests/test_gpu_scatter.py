"""`permute const` (skel_scatter.h) at the sizes where it changes hands: one workgroup up to 4096 elements, tiles of 2048
sources, pieces of 16 bytes in the copy of the defaults.  Elements are stored unchanged, so results are exact."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TYPES = {"Int8": np.int8, "Word16": np.uint16, "Int32": np.int32, "float": np.float32, "Int64": np.int64}


@pytest.fixture(scope="module")
def A():
    import acchip
    return acchip


@pytest.fixture(scope="module")
def ctx(A):
    c = A.Context(0)
    yield c
    c.close()


class Part(object):
    """`count` elements of an array from element `off` on"""
    def __init__(self, arr, off, count):
        self.d = arr.desc(shape=(count,), offset_elems=off)

    def desc(self):
        return self.d


@pytest.mark.parametrize("n", [1, 63, 2047, 2048, 2049, 4096, 4097, 70001])
@pytest.mark.parametrize("ctype", list(TYPES))
def test_scalars(A, ctx, ctype, n):
    dt = TYPES[ctype]
    rng = np.random.default_rng(n)
    places = rng.permutation(n + 5)[:n].astype(np.int32)
    places[rng.random(n) < 0.3] = -1
    vals = rng.integers(0, 100, n).astype(dt)
    sk = ctx.skeleton(A.SKEL_PERMUTE, ctype, env=[(1, ctype), (1, "Int32")], out_rank=1, get="acc_stream(arrIn0_0, ix)", combine="x",
                      permutation="(acc_stream(arrIn1_0, ix) >= 0 ? (Int64)arrIn1_0[ix] : ACC_IGNORE)")
    for off in (0, 1):                                   # 16-byte pieces, single elements
        defaults = rng.integers(0, 100, n + 5 + off).astype(dt)
        out = ctx.array(np.full(n + 7 + off, 77, dt))
        sk.permute([ctx.array(vals), ctx.array(places)], n, Part(ctx.array(defaults), off, n + 5), Part(out, off, n + 5))
        want = np.full(n + 7 + off, 77, dt)
        want[off:off + n + 5] = defaults[off:]
        m = places >= 0
        want[off:][places[m]] = vals[m]
        assert np.array_equal(out.get(), want), (ctype, n, off)


@pytest.mark.parametrize("n", [1, 2049, 4096, 4097, 50001])
def test_tuples_win_whole(A, ctx, n):
    """three sources a target: the components of one of them, whichever"""
    rng = np.random.default_rng(n)
    places = rng.permutation(np.arange(n) // 3).astype(np.int32)
    nt = int(places.max()) + 2
    wide, small = rng.integers(0, 1 << 40, n).astype(np.int64), (np.arange(n) % 100).astype(np.int8)
    sk = ctx.skeleton(A.SKEL_PERMUTE, "Int64, Int8, Int32", env=[(1, "Int64"), (1, "Int8"), (1, "Int32")], out_rank=1,
                      get="acc_elt{arrIn0_0[ix], acc_stream(arrIn1_0, ix), (Int32)ix}", combine="acc_elt{x.a2, x.a1, x.a0}", permutation="(Int64)arrIn2_0[ix]")
    out = ctx.empty_tuple(nt, [np.int64, np.int8, np.int32])
    sk.permute([ctx.array(wide), ctx.array(small), ctx.array(places)], n,
               ctx.tuple_array(np.full(nt, 5, np.int64), np.full(nt, 6, np.int8), np.full(nt, -1, np.int32)), out)
    a2, a1, a0 = out.get()
    assert np.array_equal(places[a0[:-1]], np.arange(nt - 1)) and a0[-1] == -1 and a2[-1] == 5 and a1[-1] == 6
    assert np.array_equal(wide[a0[:-1]], a2[:-1]) and np.array_equal(small[a0[:-1]], a1[:-1])


@pytest.mark.parametrize("n", [3000, 9000])
def test_an_operand_shorter_than_the_source(A, ctx, n):
    """an array that the fragments read at their own index only below its end must not be read beyond it, and an empty
    one not at all; and a result that is its own defaults is not copied"""
    short = np.arange(n // 2 + 3, dtype=np.int32)
    m = short.size
    sk = ctx.skeleton(A.SKEL_PERMUTE, "Int32", env=[(1, "Int32"), (1, "Int32")], out_rank=1,
                      get="(ix < shIn0_0 ? arrIn0_0[ix] * 2 : (Int32)ix)", combine="x", permutation="(ix < shIn0_0 ? (Int64)acc_stream(arrIn1_0, ix) : ix)")
    out = ctx.array(np.full(n, -7, np.int32))
    sk.permute([ctx.array(short), ctx.array(short[::-1].copy())], n, out, out)
    want = np.arange(n, dtype=np.int32)
    want[:m] = 2 * short[::-1]
    assert np.array_equal(out.get(), want)
    empty = ctx.empty(0, np.int32)
    sk.permute([empty, empty], n, out, out)
    assert np.array_equal(out.get(), np.arange(n, dtype=np.int32))


@pytest.mark.parametrize("n", [3000, 9000])
@pytest.mark.parametrize("elt", ["Word8", "Int32", "Int32, Int8"])
def test_the_element_of_a_source_that_is_dropped_is_not_evaluated(A, ctx, elt, n):
    """a gather through an index that is only good where the source stays -- elsewhere it leads to elements in front of the
    ones meant, which are there -- and a mark wherever the element function is evaluated"""
    rng = np.random.default_rng(n)
    places = rng.permutation(n + 60).astype(np.int32)[:n]
    places[rng.random(n) < 0.4] = -1
    places[1000:2100] = -1                                             # (waves that keep nothing)
    kept = (places >= 0) & (places < n)
    through = np.where(kept, rng.integers(50, 100, n), rng.integers(0, 50, n)).astype(np.int32)
    values, marks = rng.integers(0, 100, 100).astype(np.int32), ctx.array(np.zeros(n, np.int32))
    comps = [t.strip() for t in elt.split(",")]
    value = "({ ((Int32 *)arrIn3_0)[ix] = 1; arrIn0_0[arrIn1_0[ix]]; })"
    get = "(%s)%s" % (comps[0], value) if len(comps) == 1 else "acc_elt{%s, (Int8)(ix %% 100)}" % value
    sk = ctx.skeleton(A.SKEL_PERMUTE, elt, env=[(1, "Int32")] * 4, out_rank=1, get=get, combine="x" if len(comps) == 1 else "acc_elt{x.a1, x.a0}",
                      permutation="(Int64)arrIn2_0[ix]")
    dts = [{"Word8": np.uint8, "Int32": np.int32, "Int8": np.int8}[t] for t in comps]
    make = (lambda k: ctx.array(np.full(n, k, dts[0]))) if len(comps) == 1 else (lambda k: ctx.tuple_array(*[np.full(n, k, d) for d in dts]))
    out = make(0)
    sk.permute([ctx.array(values), ctx.array(through), ctx.array(places), marks], n, make(77), out)
    assert np.array_equal(marks.get() != 0, kept)
    got = out.get() if len(comps) > 1 else [out.get()]
    want = np.full(n, 77, np.int64)
    want[places[kept]] = values[through[kept]]
    assert np.array_equal(got[0].astype(np.int64), want)
    if len(comps) > 1:
        want[places[kept]] = np.flatnonzero(kept) % 100
        assert np.array_equal(got[1].astype(np.int64), want)


@pytest.mark.parametrize("n", [4000, 70001])
def test_a_fragment_with_an_index_of_its_own(A, ctx, n):
    """`ix` inside the lambda is not the element's index"""
    rng = np.random.default_rng(n)
    a, b, places = rng.integers(0, 100, n).astype(np.int32), rng.permutation(n).astype(np.int32), rng.permutation(n).astype(np.int32)
    sk = ctx.skeleton(A.SKEL_PERMUTE, "Int32", env=[(1, "Int32")] * 3, out_rank=1, combine="x", permutation="(Int64)acc_stream(arrIn2_0, ix)",
                      get="[&](Int64 ix) { return arrIn0_0[ix]; }((Int64)arrIn1_0[ix]) * 1000 + arrIn0_0[ix]")
    out = ctx.empty(n, np.int32)
    sk.permute([ctx.array(a), ctx.array(b), ctx.array(places)], n, ctx.array(np.zeros(n, np.int32)), out)
    want = np.zeros(n, np.int32)
    want[places] = a[b] * 1000 + a
    assert np.array_equal(out.get(), want)
