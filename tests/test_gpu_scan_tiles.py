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


@pytest.mark.parametrize("ctype,dt", [("float", np.float32), ("double", np.float64)])
def test_the_tile_does_not_depend_on_what_was_called_before(ctx, ctype, dt):
    """An instance that has run nothing yet takes the same tile without allocations, and recorded into a graph, as
    acc_exec_scan does; so does one whose unaligned form was first wanted for an array of another size.  Sums of floating
    numbers tell the tile: what the first one holds is associated by its shape alone (further on by what the look-back
    finds finished, which differs from call to call)."""
    import ctypes as C

    import acchip as A
    size = np.dtype(dt).itemsize
    n, large = (20 << 20) // size + 3, (49 << 20) // size
    rng = np.random.default_rng(1)
    x = rng.standard_normal(large + 1).astype(dt)
    src, stream, first = ctx.array(x), ctx.stream(), TILE * 4 // size

    def fresh():
        return ctx.skeleton(A.SKEL_SCANL1, ctype, env=[(1, ctype)], get="arrIn0_0[ix]", combine="x + y", wait=True)
    for shift in (0, 1):
        usual = fresh()
        want, got, out = ctx.empty(n, dt), ctx.empty(n, dt), ctx.empty(large, dt)
        env = [_Part(src, shift, n)]
        usual.scan(env, n, want, stream=stream)
        sk = fresh()
        if shift:                                                  # (the unaligned form is loaded by a first call)
            sk.scan([_Part(src, shift, large)], large, out, stream=stream)
        print(ctype, shift, "without allocations", flush=True)
        sk.scan(env, n, got, stream=stream, noalloc=True)
        ctx.sync()
        assert np.array_equal(got.get()[:first], want.get()[:first]), shift
        # the other way round: a call of this size first
        sk = fresh()
        sk.scan(env, n, got, stream=stream)
        usual.scan([_Part(src, shift, large)], large, out, stream=stream)
        ctx.sync()
        ref = out.get()
        sk.scan([_Part(src, shift, large)], large, out, stream=stream, noalloc=True)
        ctx.sync()
        assert np.array_equal(out.get()[:first], ref[:first]), shift
    hip = C.CDLL("libamdhip64.so")
    hip.hipStreamBeginCapture.argtypes = [C.c_void_p, C.c_int]
    hip.hipStreamEndCapture.argtypes = [C.c_void_p, C.POINTER(C.c_void_p)]
    hip.hipGraphInstantiate.argtypes = [C.POINTER(C.c_void_p), C.c_void_p, C.c_void_p, C.c_void_p, C.c_size_t]
    hip.hipGraphLaunch.argtypes = [C.c_void_p, C.c_void_p]
    hip.hipGraphExecDestroy.argtypes = hip.hipGraphDestroy.argtypes = [C.c_void_p]
    usual, sk = fresh(), fresh()
    env = [_Part(src, 0, n)]
    want, got = ctx.empty(n, dt), ctx.empty(n, dt)
    graph, graph_exec = C.c_void_p(), C.c_void_p()
    ctx.sync()
    assert hip.hipStreamBeginCapture(stream, 2) == 0
    try:
        sk.scan(env, n, got, stream=stream, noalloc=True)
    finally:
        rc = hip.hipStreamEndCapture(stream, C.byref(graph))
    assert rc == 0 and graph.value and hip.hipGraphInstantiate(C.byref(graph_exec), graph, None, None, 0) == 0
    for replay in range(3):
        print(ctype, "replay", replay, flush=True)
        src.set(rng.standard_normal(large + 1).astype(dt))
        assert hip.hipGraphLaunch(graph_exec, stream) == 0
        usual.scan(env, n, want, stream=stream)
        ctx.sync()
        assert np.array_equal(got.get()[:first], want.get()[:first]) and np.allclose(got.get(), want.get(), rtol=0, atol=1e-2)
    hip.hipGraphExecDestroy(graph_exec)
    hip.hipGraphDestroy(graph)


class _Part(object):
    def __init__(self, arr, off, count):
        self.d = arr.desc(shape=(count,), offset_elems=off)

    def desc(self):
        return self.d
