"""Many applications of a 2-D stencil, two a launch (variants 10 and 11), at the sizes where the strips change form: rows of
one strip exactly, one column and one vector more, two strips; bands cut short, arrays thinner than a band and than what
two applications reach; operands off the 16-byte boundary; every count of applications up to two pairs of pairs and a
rest.  One application a launch is the reference: equal in every bit, in the result and in the result before it."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

BOX = [(a, b) for a in (-1, 0, 1) for b in (-1, 0, 1)]
CROSS = [(-1, 0), (0, -1), (0, 0), (0, 1), (1, 0)]
ROWS = [(-1, 0), (1, 0)]
COLUMNS = [(0, -1), (0, 0), (0, 1)]


@pytest.fixture(scope="module")
def ctx():
    import acchip as A
    return A.Context(0)


class _Part(object):
    def __init__(self, arr, shape, off):
        self.arr, self.d = arr, arr.desc(shape=shape, offset_elems=off)

    def desc(self):
        return self.d


@pytest.mark.parametrize("boundary", ["clamp", "mirror", "wrap", "constant"])
@pytest.mark.parametrize("ctype,dt,taps", [("float", np.float32, BOX), ("double", np.float64, CROSS), ("Int32", np.int32, BOX), ("Int64", np.int64, ROWS),
                                           ("float", np.float32, COLUMNS)])
def test_pairs_against_single_applications(ctx, boundary, ctype, dt, taps):
    import acchip as A
    whole = dt in (np.int32, np.int64)
    # (lopsided weights: a row or column out of place shows)
    fn = " + ".join("(%s)%s * t%d" % (ctype, (3 + 2 * k) if whole else repr(0.07 * (k + 1) - 0.2), k) for k in range(len(taps)))
    desc = dict(out_rank=2, taps=taps, boundary=boundary, stencil_fn=fn, boundary_constant="(%s)7" % ctype if boundary == "constant" else None)
    assert "skel_stencil_pair.h" in A.preview(A.make_desc(A.SKEL_STENCIL, ctype, **desc), 10)[1]
    twos = ctx.skeleton(A.SKEL_STENCIL, ctype, wait=True, **desc)
    with A.tuning("stencil.pair=0", ctx):
        ones = ctx.skeleton(A.SKEL_STENCIL, ctype, wait=True, **desc)
    own = 62 * (16 // np.dtype(dt).itemsize)
    rng = np.random.default_rng(6)
    for shape in ((3, own), (8, own + 1), (9, own + 4), (9, own + 5), (16, 2 * own), (17, 2 * own - 3), (33, 2 * own + 1), (12, 2 * own + 4),
                  (40, 3 * own + 7), (24, 3 * own - 1)):
        n = shape[0] * shape[1]
        for shift, iters in ((0, 5), (1, 5), (0, 9), (0, 4), (0, 7)):
            print(ctype, len(taps), boundary, shape, shift, iters, flush=True)
            x = rng.integers(-50, 50, n + shift).astype(dt)
            got = []
            for sk in (twos, ones):
                a, b = ctx.array(np.concatenate([x, np.full(3, 77, dt)])), ctx.array(np.full(n + shift + 3, 77, dt))
                pa, pb = _Part(a, shape, shift), _Part(b, shape, shift)
                res = sk.stencil_iterate(None, pa, pb, iters)
                got.append((res is pb, a.get(), b.get()))
            assert got[0][0] == got[1][0]
            assert np.array_equal(got[0][1], got[1][1]) and np.array_equal(got[0][2], got[1][2]), (shape, shift, iters)
