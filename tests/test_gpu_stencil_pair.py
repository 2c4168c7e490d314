"""Many applications of a 2-D stencil, two to four a launch (variants 10 and 11), at the sizes where the strips change form:
rows of one strip exactly, one column and one vector more, two strips; walks cut short, arrays thinner than a walk and than
what a launch's applications reach; operands off the 16-byte boundary; counts of applications that split differently.  One
application a launch is the reference: equal in every bit, in the result and in the result before it."""
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


def strip(taps, dt, levels=4):
    """columns of a strip, as the kernel has them: the outermost lanes of either side, as many as go wrong, store nothing"""
    vec = 16 // np.dtype(dt).itemsize
    outer = -(-levels // vec) if any(dx for _, dx in taps) else 1
    return (64 - 2 * outer) * vec


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
    own = strip(taps, dt)
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


@pytest.mark.parametrize("boundary", ["clamp", "mirror", "wrap", "constant"])
@pytest.mark.parametrize("ctype,dt,taps", [("float", np.float32, BOX), ("double", np.float64, BOX), ("Int32", np.int32, CROSS), ("float", np.float32, COLUMNS)])
def test_walks_and_counts(ctx, boundary, ctype, dt, taps):
    """every count of applications whose launches split differently, walks that end amid the steps written out, inside the
    array and cut short by its end; one application a launch is the reference, bit by bit"""
    import acchip as A
    fn = " + ".join("(%s)%s * t%d" % (ctype, (3 + 2 * k) if dt == np.int32 else repr(0.07 * (k + 1) - 0.2), k) for k in range(len(taps)))
    desc = dict(out_rank=2, taps=taps, boundary=boundary, stencil_fn=fn, boundary_constant="(%s)7" % ctype if boundary == "constant" else None)
    with A.tuning("stencil.pair=0", ctx):
        ones = ctx.skeleton(A.SKEL_STENCIL, ctype, wait=True, **desc)
    own = strip(taps, dt)
    rng = np.random.default_rng(7)
    for walk, shape, counts in ((0, (29, 2 * own + 9), range(1, 15)), (28, (90, own + 24), (4, 9)), (5, (37, 2 * own - 8), (4, 9)), (1, (6, own + 16), (5, 9))):
        with A.tuning("stencil.pair_walk=%d" % walk, ctx):
            many = ctx.skeleton(A.SKEL_STENCIL, ctype, wait=True, **desc)
        for iters in counts:
            print(ctype, len(taps), boundary, walk, shape, iters, flush=True)
            x = rng.integers(-50, 50, shape).astype(dt)
            got = []
            for sk in (many, ones):
                a, b = ctx.array(x), ctx.array(np.full(shape, 77, dt))
                res = sk.stencil_iterate(None, a, b, iters)
                got.append((res is b, a.get(), b.get()))
            assert got[0][0] == got[1][0] and all(np.array_equal(got[0][k], got[1][k]) for k in (1, 2)), (walk, shape, iters)


@pytest.mark.parametrize("boundary", ["clamp", "wrap"])
@pytest.mark.parametrize("ctype,dt,taps", [("float", np.float32, BOX), ("double", np.float64, CROSS), ("Int32", np.int32, ROWS), ("Int64", np.int64, COLUMNS)])
def test_walks_that_go_up(ctx, boundary, ctype, dt, taps):
    """strips inside the array, whose every second walk goes up: walks shorter than what the launch reads beyond them, of as
    many rows as are asked for ahead and of one more, and a last one of a single row; equal to one application a launch"""
    import acchip as A
    fn = " + ".join("(%s)%s * t%d" % (ctype, (3 + 2 * k) if np.issubdtype(dt, np.integer) else repr(0.07 * (k + 1) - 0.2), k) for k in range(len(taps)))
    desc = dict(out_rank=2, taps=taps, boundary=boundary, stencil_fn=fn)
    with A.tuning("stencil.pair=0", ctx):
        ones = ctx.skeleton(A.SKEL_STENCIL, ctype, wait=True, **desc)
    own = strip(taps, dt)
    rng = np.random.default_rng(11)
    for walk, h in ((1, 16), (3, 31), (4, 33), (28, 141)):
        with A.tuning("stencil.pair_walk=%d" % walk, ctx):
            many = ctx.skeleton(A.SKEL_STENCIL, ctype, wait=True, **desc)
        for iters in (4, 9):                              # a three and one by itself; two fours and one
            print(ctype, len(taps), boundary, walk, h, iters, flush=True)
            x = rng.integers(-50, 50, (h, 4 * own + 9)).astype(dt)
            got = []
            for sk in (many, ones):
                a, b = ctx.array(x), ctx.array(np.full(x.shape, 77, dt))
                res = sk.stencil_iterate(None, a, b, iters)
                got.append((res is b, a.get(), b.get()))
            assert got[0][0] == got[1][0] and all(np.array_equal(got[0][k], got[1][k]) for k in (1, 2)), (walk, h, iters)


@pytest.mark.parametrize("boundary", ["clamp", "mirror", "wrap", "constant"])
@pytest.mark.parametrize("ctype,dt,taps", [("float", np.float32, BOX), ("double", np.float64, CROSS), ("Int32", np.int32, ROWS), ("Int64", np.int64, BOX)])
def test_two_a_launch(ctx, boundary, ctype, dt, taps):
    """arrays of 12 MB and a little more, from which on calls of five and six applications make two a launch: the widths at
    which the strips of two, of three and of four applications change form, and those that one of them cannot take"""
    import acchip as A
    whole = dt in (np.int32, np.int64)
    fn = " + ".join("(%s)%s * t%d" % (ctype, (3 + 2 * k) if whole else repr(0.07 * (k + 1) - 0.2), k) for k in range(len(taps)))
    desc = dict(out_rank=2, taps=taps, boundary=boundary, stencil_fn=fn, boundary_constant="(%s)7" % ctype if boundary == "constant" else None)
    many = ctx.skeleton(A.SKEL_STENCIL, ctype, wait=True, **desc)
    with A.tuning("stencil.pair=0", ctx):
        ones = ctx.skeleton(A.SKEL_STENCIL, ctype, wait=True, **desc)
    vec, esz = 16 // np.dtype(dt).itemsize, np.dtype(dt).itemsize
    widths = set()
    for levels in (2, 3, 4):
        own = strip(taps, dt, levels)
        outer = (64 - own // vec) // 2
        widths |= {own, own + 1, own + outer * vec - 1, own + outer * vec, 2 * own + 1}
    rng = np.random.default_rng(8)
    for w in sorted(widths):
        h = (12 << 20) // (w * esz) + 2
        x = rng.integers(-50, 50, (h, w)).astype(dt)
        for iters in (5, 6, 8, 10):
            print(ctype, len(taps), boundary, (h, w), iters, flush=True)
            got = []
            for sk in (many, ones):
                a, b = ctx.array(x), ctx.empty((h, w), dt)
                res = sk.stencil_iterate(None, a, b, iters)
                got.append((res is b, a.get(), b.get()))
            assert got[0][0] == got[1][0] and all(np.array_equal(got[0][k], got[1][k]) for k in (1, 2)), (h, w, iters)


@pytest.mark.parametrize("what,rank,shape", [("acc_pair_own", 2, (40, 300)), ("acc_flat_source", 3, (5, 7, 700))])
def test_a_form_that_cannot_be_built_leaves_the_call_to_another(ctx, what, rank, shape):
    """a preamble that takes a name which only this form's template has: the form does not compile, the others do"""
    import acchip as A
    taps = CROSS if rank == 2 else [(0, 0, 0), (-1, 0, 0), (1, 0, 0), (0, -1, 0), (0, 1, 0), (0, 0, -1), (0, 0, 1)]
    desc = dict(out_rank=rank, taps=taps, boundary="clamp", stencil_fn=" + ".join("%d * t%d" % (k + 2, k) for k in range(len(taps))))
    broken = A.make_desc(A.SKEL_STENCIL, "Int32", preamble="#define %s 1" % what, **desc)
    with pytest.raises(A.AccError):
        A.compile_source(A.preview(broken, 10 if rank == 2 else 8)[1])
    x = np.random.default_rng(2).integers(-50, 50, shape).astype(np.int32)
    got = []
    for preamble in (None, "#define %s 1" % what):
        sk = ctx.skeleton(A.SKEL_STENCIL, "Int32", preamble=preamble, wait=True, **desc)
        for _ in range(2):
            a, b = ctx.array(x), ctx.empty(shape, np.int32)
            if rank == 2:
                got.append(sk.stencil_iterate(None, a, b, 6).get())
            else:
                sk.stencil(None, a, b)
                got.append(b.get())
    assert all(np.array_equal(g, got[0]) for g in got)


@pytest.mark.parametrize("rank,shape", [(2, (40, 300)), (3, (5, 7, 700))])
def test_recorded_before_the_form_is_loaded(ctx, rank, shape):
    """under capture nothing is built: the graph holds the form that is there, and its results are the same"""
    import ctypes as C

    import acchip as A
    taps = CROSS if rank == 2 else [(0, 0, 0), (-1, 0, 0), (1, 0, 0), (0, -1, 0), (0, 1, 0), (0, 0, -1), (0, 0, 1)]
    desc = dict(out_rank=rank, taps=taps, boundary="mirror", stencil_fn=" + ".join("%d * t%d" % (k + 2, k) for k in range(len(taps))))
    sk = ctx.skeleton(A.SKEL_STENCIL, "Int32", wait=True, **desc)
    hip = C.CDLL("libamdhip64.so")
    hip.hipStreamBeginCapture.argtypes = [C.c_void_p, C.c_int]
    hip.hipStreamEndCapture.argtypes = [C.c_void_p, C.POINTER(C.c_void_p)]
    hip.hipGraphInstantiate.argtypes = [C.POINTER(C.c_void_p), C.c_void_p, C.c_void_p, C.c_void_p, C.c_size_t]
    hip.hipGraphLaunch.argtypes = [C.c_void_p, C.c_void_p]
    hip.hipGraphExecDestroy.argtypes = hip.hipGraphDestroy.argtypes = [C.c_void_p]
    stream, rng = ctx.stream(), np.random.default_rng(2)
    a, b = ctx.empty(shape, np.int32), ctx.empty(shape, np.int32)

    def call(x, y):
        if rank == 2:
            return sk.stencil_iterate(None, x, y, 5, stream=stream)
        sk.stencil(None, x, y, stream=stream)
        return y
    graph, graph_exec = C.c_void_p(), C.c_void_p()
    ctx.sync()
    assert hip.hipStreamBeginCapture(stream, 2) == 0
    try:
        res = call(a, b)
    finally:
        rc = hip.hipStreamEndCapture(stream, C.byref(graph))
    assert rc == 0 and graph.value and hip.hipGraphInstantiate(C.byref(graph_exec), graph, None, None, 0) == 0
    for replay in range(4):
        print(rank, "replay", replay, flush=True)
        x = rng.integers(-50, 50, shape).astype(np.int32)
        a.set(x)
        assert hip.hipGraphLaunch(graph_exec, stream) == 0
        ctx.sync()
        got = res.get()
        eager = call(ctx.array(x), ctx.empty(shape, np.int32))          # (the form is built and taken from here on)
        ctx.sync()
        assert np.array_equal(got, eager.get()), replay
    hip.hipGraphExecDestroy(graph_exec)
    hip.hipGraphDestroy(graph)


@pytest.mark.parametrize("ctype,dt", [("Int32", np.int32), ("double", np.float64)])
@pytest.mark.parametrize("rank,shape,iters", [(2, (40, 256), 9), (2, (31, 508), 4), (2, (12400, 256), 5), (3, (9, 30, 150), 1)])
def test_the_element_function_sees_values_of_the_array_only(ctx, ctype, dt, rank, shape, iters):
    """also where what it makes is dropped, in the lanes at the ends of a wave (2-D: by four, three and two applications a launch):
    the first zero it sees turns every later result into -1"""
    import acchip as A
    taps = BOX if rank == 2 else [(0, 0, 0), (-1, 0, 0), (1, 0, 0), (0, -1, 0), (0, 1, 0), (0, 0, -1), (0, 0, 1)]
    args = ", ".join("t%d" % k for k in range(len(taps)))
    pre = """__device__ int zero_seen;
__device__ __forceinline__ %s look(%s, %s centre) {
  if (%s) atomicOr(&zero_seen, 1);
  return __atomic_load_n(&zero_seen, __ATOMIC_RELAXED) ? (%s)-1 : centre;
}
""" % (ctype, ", ".join("%s t%d" % (ctype, k) for k in range(len(taps))), ctype, " || ".join("t%d == 0" % k for k in range(len(taps))), ctype)
    with A.tuning("stencil.flat=2,stencil.thin_3d=0", ctx):
        sk = ctx.skeleton(A.SKEL_STENCIL, ctype, out_rank=rank, taps=taps, boundary="clamp", preamble=pre,
                          stencil_fn="look(%s, t%d)" % (args, taps.index((0,) * rank)), wait=True)
    x = np.random.default_rng(4).integers(1, 50, shape).astype(dt)
    for _ in range(3):
        a, b = ctx.array(x), ctx.empty(shape, dt)
        if rank == 2:
            res = sk.stencil_iterate(None, a, b, iters)
        else:
            sk.stencil(None, a, b)
            res = b
        assert np.array_equal(res.get(), x)
