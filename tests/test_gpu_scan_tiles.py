"""Scans in the tile between the small and the large one (variants 4 and 5), on sizes round one and several of its tiles
and with ends anywhere in a vector; whole numbers against numpy, exact."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

KINDS = ("scanl", "scanl1", "scanl'", "scanr", "scanr1", "scanr'")
TILE = 256 * 12 * 4                                   # elements of Int32


@pytest.fixture(scope="module")
def ctx():
    import acchip as A
    return A.Context(0)


def expected(kind, x, seed):
    right = kind.startswith("scanr")
    v = x[::-1] if right else x
    run = np.cumsum(v, dtype=np.int64).astype(np.int64)
    if kind.endswith("1"):
        out, total = run, None
    else:
        full = np.concatenate([[0], run]) + seed
        out, total = (full[:-1], full[-1]) if kind.endswith("'") else (full, None)
    return (out[::-1] if right else out), total


@pytest.mark.parametrize("ctype,dt", [("Int32", np.int32), ("Int64", np.int64)])
@pytest.mark.parametrize("kind", KINDS)
def test_middle_tile(ctx, kind, ctype, dt):
    import acchip as A
    with A.tuning("scan.small_below_kb=1", ctx):
        sk = ctx.skeleton(A.SCAN_KINDS[kind], ctype, env=[(1, ctype)], get="arrIn0_0[ix]", combine="x + y", seed=None if kind.endswith("1") else "5", wait=True)
    desc = A.make_desc(A.SCAN_KINDS[kind], ctype, env=[(1, ctype)], get="arrIn0_0[ix]", combine="x + y", seed=None if kind.endswith("1") else "5")
    assert all("#define ACC_ROWS 12\n" in A.preview(desc, v)[1] for v in (4, 5))
    rng = np.random.default_rng(5)
    tile = TILE * 4 // np.dtype(dt).itemsize
    for n in (300, 1025, tile - 1, tile, tile + 1, tile + 3, 3 * tile + 2, 700 * tile + 5):
        for shift in ((0, 1) if n < 5 * tile else (0,)):         # (unaligned operands: variant 5)
            print(kind, ctype, n, shift, flush=True)
            x = rng.integers(-9, 16, n + shift).astype(dt)
            plus = 1 if kind in ("scanl", "scanr") else 0
            out = ctx.array(np.full(n + plus + 2, -777, dt))
            tot = ctx.array(np.array(-1, dt))
            src = ctx.array(x)
            sk.scan([_Part(src, shift, n)], n, out.desc(shape=(n + plus,)), tot if kind.endswith("'") else None)
            got = out.get()
            want, total = expected(kind, x[shift:], 5)
            assert np.array_equal(got[:n + plus], want.astype(dt)), (kind, n)
            assert np.all(got[n + plus:] == -777), "wrote past the end"
            if total is not None:
                assert int(tot.get().reshape(-1)[0]) == int(np.array(total).astype(dt))


class _Part(object):
    def __init__(self, arr, off, count):
        self.d = arr.desc(shape=(count,), offset_elems=off)

    def desc(self):
        return self.d
