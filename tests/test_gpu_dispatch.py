"""Which form a call takes, where the choice is a matter of time and not of the result: the fragments say which workgroup
evaluated an element, or how many there are."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    import acchip as A
    return A.Context(0)


@pytest.mark.parametrize("get", ["0", "(Int32)threadIdx.x * 0"])              # (the second might be a gather)
@pytest.mark.parametrize("nseg,mean,own", [
    # up to eight workgroups a compute unit: the fewest segments that leave one more than 1024 elements
    (1000, 64, 32), (1000, 16, 128), (60000, 30, 64), (65536, 100, 32),
    # more of them: no more chunks in all, half empty ones among them, or a third more of workgroups with one chunk
    (765249, 10, 256), (458496, 12, 256), (359769, 20, 128), (300000, 50, 256), (262143, 100, 128), (200000, 70, 32), (524287, 40, 64), (291628, 36, 64),
    (250000, 33, 64), (262143, 64, 32),
    # 32 a compute unit at most
    (1000000, 30, 256), (1 << 20, 32, 256)])
def test_segments_a_workgroup(ctx, nseg, mean, own, get):
    import acchip as A
    if get != "0":                       # a third more of one-chunk workgroups, and more than 20 a compute unit, only in a stream
        own = {200000: 128, 524287: 128, 291628: 256, 250000: 128, 262143: 128}.get(nseg, own)
    if ctx.props().compute_units != 256:
        pytest.skip("the counts are those of 256 compute units")
    sk = ctx.skeleton(A.SKEL_FOLDSEG, "Int32", env=[], get=get, combine="acc_max(acc_max(x, y), (Int32)blockIdx.x)", seed="-1", wait=True)
    out = ctx.empty(nseg, np.int32)
    sk.foldseg([], nseg * mean, ctx.array((np.arange(nseg + 1) * mean).astype(np.int32)), out)
    assert np.array_equal(out.get(), np.arange(nseg) // own)


SEVEN = [(0, 0, 0), (-1, 0, 0), (1, 0, 0), (0, -1, 0), (0, 1, 0), (0, 0, -1), (0, 0, 1)]
BOX = [(z, y, x) for z in (-1, 0, 1) for y in (-1, 0, 1) for x in (-1, 0, 1)]


@pytest.mark.parametrize("ctype,dt,taps,shape,strips", [
    # 512 MB of source and result at most
    ("Int32", np.int32, SEVEN, (60, 1024, 1024), False), ("Int32", np.int32, BOX, (60, 1000, 1000), False),
    # whole strips: planes far apart, or near each other
    ("Int32", np.int32, SEVEN, (131, 512, 1024), True), ("Int32", np.int32, SEVEN, (257, 512, 512), False), ("Int32", np.int32, BOX, (140, 512, 1024), False),
    ("Int32", np.int32, BOX, (150, 512, 1024), True), ("Int64", np.int64, BOX, (150, 512, 512), False), ("Int64", np.int64, SEVEN, (131, 512, 512), True),
    ("Int64", np.int64, BOX, (75, 512, 1024), True), ("Int32", np.int32, SEVEN, (400, 512, 512), True),
    # nearly whole ones, and rows that leave more of a strip outside
    ("Int32", np.int32, SEVEN, (70, 1000, 1000), True), ("Int32", np.int32, SEVEN, (45, 1580, 1000), False), ("Int32", np.int32, BOX, (45, 1580, 1000), True),
    ("Int32", np.int32, SEVEN, (80, 900, 970), False), ("Int64", np.int64, SEVEN, (66, 700, 760), True), ("Int64", np.int64, BOX, (66, 700, 760), False)])
def test_volumes_in_strips_or_by_vectors(ctx, ctype, dt, taps, shape, strips):
    import acchip as A
    print(ctype, len(taps), shape, flush=True)
    desc = dict(out_rank=3, taps=taps, boundary="clamp", stencil_fn="(%s)blockIdx.x + 0 * (%s)" % (ctype, " + ".join("t%d" % k for k in range(len(taps)))))
    src, got = ctx.empty(shape, dt), []
    out = ctx.empty(shape, dt)
    for knobs in ("stencil.flat=1", "stencil.flat=0", "stencil.flat=2"):
        with A.tuning(knobs, ctx):
            sk = ctx.skeleton(A.SKEL_STENCIL, ctype, wait=True, **desc)
        sk.stencil(None, src, out)
        got.append(out.get())
    alike = [np.mean(got[0] == g) for g in got[1:]]            # (a last strip that overlaps its neighbour: either number)
    assert alike[0 if strips else 1] > 0.98 and alike[1 if strips else 0] < 0.5, alike


@pytest.mark.parametrize("ctype,dt,degree,loop,lines", [("Int32", np.int32, 4, "", True), ("Int32", np.int32, 20, "", True), ("Int32", np.int32, 64, "", False), ("Int32", np.int32, 0, "for", False),
                                                        ("Int64", np.int64, 4, "", True), ("Int64", np.int64, 64, "", False), ("Int64", np.int64, 0, "while", False)])
def test_tiled_maps_in_lines_or_as_they_stand(ctx, ctype, dt, degree, loop, lines):
    """a result of no whole lines goes out in lines, for which a part of it is evaluated twice, unless its elements are dear"""
    import acchip as A
    h, w = 301, 1000
    loops = {"": "", "for": "for (int i = 0; i < 3; ++i) r = r * q + i; ", "while": "int i = 0; while (i < 3) { r = r * q + i; ++i; } "}[loop]
    calc = "[&]{ const %s q = arrIn0_0[(ix %% shOut_0) * shOut_1 + ix / shOut_0]; %s r = q; %s%sreturn r * 0 + (%s)blockIdx.x; }()" % (
        ctype, ctype, loops, "".join("r = (r ^ %d) * q + %d; " % (7 * i + 3, 1 + i) for i in range(degree)), ctype)
    # (a product by zero that is not seen through: the operands are read, the result says who made it)
    calc = calc.replace("r * 0", "(r == (%s)0x5a5a5a5b ? 1 : 0)" % ctype)
    src = ctx.array(np.random.default_rng(3).integers(0, 1000, (w, h)).astype(dt))
    got = []
    for knobs in ("map.lines_from_mb=0", "map.lines_from_mb=100000"):
        with A.tuning(knobs, ctx):
            sk = ctx.skeleton(A.SKEL_MAP, ctype, env=[(2, ctype)], out_rank=2, flags=A.FLAG_TILED, get=calc, wait=True)
        out = ctx.empty((h, w), dt)
        sk.map([src], out)
        got.append(out.get())
    assert np.array_equal(got[0], got[1]) != lines
