"""Maps in tiles (ACC_FLAG_TILED) at the sizes where the tiling changes form: one tile or two down a workgroup (32 and 33
rows), the last tile of either direction full, one short and one over, more workgroups than one die takes; index
fragments the compiler can resolve from the tile's place and ones it cannot.  The same map in runs is the oracle: moved
whole numbers, equal in every element."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

FORMS = {
    "transpose": "arrIn0_0[(ix % shOut_0) * shIn0_0 + (ix / shOut_0)]",
    "from_index": "arrIn0_0[acc_from_index<2>({shOut_1, shOut_0}, ix).i[1] * shIn0_0 + acc_from_index<2>({shOut_1, shOut_0}, ix).i[0]]",
    "mirrored": "arrIn0_0[((shOut_0 - 1 - ix % shOut_0)) * shIn0_0 + (shOut_1 - 1 - ix / shOut_0)] + (Int32)((ix + 1) % shOut_0)",
}


@pytest.fixture(scope="module")
def ctx():
    import acchip as A
    return A.Context(0)


@pytest.mark.parametrize("form", sorted(FORMS))
@pytest.mark.parametrize("shape", [(10, 33), (31, 64), (32, 65), (33, 63), (33, 129), (64, 64), (65, 127), (257, 511), (1000, 1003)])
def test_tiles_against_runs(ctx, form, shape):
    import acchip as A
    print("tiled map", form, shape, flush=True)
    h, w = shape
    src = ctx.array(np.random.default_rng(h * w).integers(-1000, 1000, (w, h)).astype(np.int32))
    results = []
    for flags in (A.FLAG_TILED, 0):
        sk = ctx.skeleton(A.SKEL_MAP, "Int32", env=[(2, "Int32")], out_rank=2, flags=flags, get=FORMS[form])
        out = ctx.array(np.full(h * w + 3, 77, np.int32))
        sk.map([src], out.desc(shape=(h, w)))
        results.append(out.get())
    assert np.array_equal(results[0], results[1])
    assert np.array_equal(results[0][-3:], [77, 77, 77])
    if form != "mirrored":
        assert np.array_equal(results[0][:-3].reshape(h, w), src.get().T)


@pytest.mark.parametrize("dim,shape", [(2, (33, 3, 65)), (2, (32, 2, 64)), (2, (70, 1, 40))])
def test_tiles_of_an_outer_dimension(ctx, dim, shape):
    """rank 3: the remainder and the quotient by the innermost extent where the tile's rows are not next to one another"""
    import acchip as A
    print("tiled map of rank 3", dim, shape, flush=True)
    frag = "(Int32)((ix % shOut_0) * 1000003 + (ix / shOut_0) * 7 + ix)"
    results = []
    for flags in (A.FLAG_TILED | A.FLAG_TILE_DIM(dim), 0):
        out = ctx.empty(shape, np.int32)
        ctx.skeleton(A.SKEL_GENERATE, "Int32", env=[], out_rank=3, flags=flags, get=frag).map([], out)
        results.append(out.get())
    assert np.array_equal(results[0], results[1])


@pytest.mark.parametrize("shape", [(70, 3, 65), (33, 40, 97), (5, 33, 130)])
@pytest.mark.parametrize("dim", [1, 2])
def test_volumes_in_whole_lines(ctx, dim, shape):
    import acchip as A
    frag = "(ix % shOut_0) * 1000003 + (ix / shOut_0) * 7 + ix"
    results = []
    with A.tuning("map.lines_from_mb=0", ctx):
        for flags in (A.FLAG_TILED | A.FLAG_TILE_DIM(dim), 0):
            out = ctx.empty(shape, np.int64)
            ctx.skeleton(A.SKEL_GENERATE, "Int64", env=[], out_rank=3, flags=flags, get=frag, wait=True).map([], out)
            results.append(out.get())
    assert np.array_equal(results[0], results[1])


def test_large_matrices_of_whole_lines(ctx):
    """down strips of workgroups, from 128 MB of result on: a last strip of one row of them, a last tile short"""
    import acchip as A
    sk = ctx.skeleton(A.SKEL_MAP, "Int32", env=[(2, "Int32")], out_rank=2, flags=A.FLAG_TILED, get=FORMS["transpose"], wait=True)
    for h, w in ((8 * 128 + 1, 32768), (32769, 1056), (8193, 4128)):
        x = np.arange(h * w, dtype=np.int32).reshape(w, h)
        out = ctx.array(np.full((h, w), 77, np.int32))
        sk.map([ctx.array(x)], out)
        assert np.array_equal(out.get(), x.T), (h, w)


@pytest.mark.parametrize("ctype,dt", [("Int32", np.int32), ("double", np.float64), ("Int16", np.int16)])
def test_tiles_in_whole_lines(ctx, ctype, dt):
    """results whose rows are no whole cache lines go out in lines: widths either side of what a workgroup writes, of whole
    lines, results that begin anywhere within a line"""
    import acchip as A
    get = FORMS["transpose"]
    with A.tuning("map.lines_from_mb=0", ctx):
        tiled, runs = [ctx.skeleton(A.SKEL_MAP, ctype, env=[(2, ctype)], out_rank=2, flags=f, get=get, wait=True) for f in (A.FLAG_TILED, 0)]
    lines = np.dtype(dt).itemsize >= 4
    assert ("#define ACC_TILE_LINES %d\n" % lines) in tiled.source(0)
    rng = np.random.default_rng(13)
    for h, w in [(10, 34), (33, 95), (32, 96), (31, 97), (40, 111), (33, 112), (33, 113), (100, 128), (33, 129), (65, 191), (64, 193), (35, 225), (1030, 160),
                 (1024, 64), (1056, 96), (300, 1001)]:
        x = rng.integers(-1000, 1000, (w, h)).astype(dt)
        src = ctx.array(x)
        for shift in (0, 1, 5, 31):
            print(ctype, h, w, shift, flush=True)
            for sk in (tiled, runs):
                out = ctx.array(np.full(h * w + shift + 3, 77, dt))
                sk.map([src], out.desc(shape=(h, w), offset_elems=shift))
                got = out.get()
                assert np.array_equal(got[shift:shift + h * w].reshape(h, w), x.T), (h, w, shift)
                assert np.all(got[:shift] == 77) and np.all(got[shift + h * w:] == 77), (h, w, shift)


@pytest.mark.parametrize("ctype,dt", [("Int32", np.int32), ("double", np.float64), ("Int16", np.int16)])
@pytest.mark.parametrize("lines_from", [0, 28])
def test_in_place(ctx, ctype, dt, lines_from):
    """the result is one of the operands, read where it is written: every element is evaluated once, so that none is made of
    what has been written already (an index that has been replaced by what it names, for instance)"""
    import acchip as A
    get = "(atomicAdd((int *)&arrIn2_0[ix], 1), (%s)(2 * arrIn0_0[ix] + %s))" % (ctype, FORMS["transpose"].replace("In0", "In1"))
    with A.tuning("map.lines_from_mb=%d" % lines_from, ctx):
        sk = ctx.skeleton(A.SKEL_MAP, ctype, env=[(2, ctype), (2, ctype), (2, "Int32")], out_rank=2, flags=A.FLAG_TILED, wait=True, get=get)
    rng = np.random.default_rng(14)
    for h, w in [(33, 97), (65, 193), (33, 128), (1030, 1001), (3001, 999), (2, 999)]:
        x, y = rng.integers(-9, 9, (w, h)).astype(dt), rng.integers(-9, 9, (h, w)).astype(dt)
        for shift in (0, 1):
            src, out, want = ctx.array(x), ctx.array(np.concatenate([np.full(shift, 7, dt), y.reshape(-1)])), y
            here, counts = out.desc(shape=(h, w), offset_elems=shift), ctx.array(np.zeros((h, w), np.int32))
            for turn in range(1, 4):
                print(ctype, h, w, shift, flush=True)
                sk.map([here, src, counts], here)
                want = 2 * want + x.T
                assert np.array_equal(out.get()[shift:].reshape(h, w), want) and np.all(out.get()[:shift] == 7), (h, w, shift)
                assert np.all(counts.get() == turn), (h, w, shift)
