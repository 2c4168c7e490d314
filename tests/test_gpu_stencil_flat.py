"""3-D stencils with the lanes over the vectors of a plane (variants 8 and 9) at the sizes where that changes form: rows
of a whole number of vectors and not, a last band of one row, a last wave partly beyond the plane, one run of planes and
several, runs cut short, volumes thinner than the stencil's reach; every boundary condition.  The element-a-thread
template is the reference: the same operations in the same order on one element, equal in every bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

STAR = [(0, 0, 0), (-1, 0, 0), (1, 0, 0), (0, -1, 0), (0, 1, 0), (0, 0, -1), (0, 0, 1)]
BOX = [(a, b, c) for a in (-1, 0, 1) for b in (-1, 0, 1) for c in (-1, 0, 1)]
ODD = [(0, 0, 2), (-1, 1, -2), (1, 0, 1), (0, -1, 0)]                    # lopsided, two columns away
SHAPES = [(5, 7, 20), (3, 2, 17), (2, 1, 19), (17, 9, 33), (33, 16, 64), (40, 31, 101), (9, 130, 260), (70, 3, 258)]


@pytest.fixture(scope="module")
def ctx():
    import acchip as A
    return A.Context(0)


@pytest.mark.parametrize("boundary", ["clamp", "mirror", "wrap", "constant"])
@pytest.mark.parametrize("ctype,dt,taps", [("float", np.float32, STAR), ("float", np.float32, BOX), ("double", np.float64, STAR),
                                           ("Int32", np.int32, ODD), ("Int64", np.int64, BOX)])
def test_against_an_element_a_thread(ctx, boundary, ctype, dt, taps):
    import acchip as A
    fn = " + ".join("(%s)%d * t%d" % (ctype, 3 + k % 5, k) for k in range(len(taps)))
    desc = dict(out_rank=3, taps=taps, boundary=boundary, stencil_fn=fn, boundary_constant="(%s)7" % ctype if boundary == "constant" else None)
    assert "skel_stencil_flat.h" in A.preview(A.make_desc(A.SKEL_STENCIL, ctype, **desc), 8)[1]
    flat = ctx.skeleton(A.SKEL_STENCIL, ctype, wait=True, **desc)
    with A.tuning("stencil.nd=1,stencil.flat=0,stencil.thin_3d=1000000", ctx):
        each = ctx.skeleton(A.SKEL_STENCIL, ctype, wait=True, **desc)
    rng = np.random.default_rng(3)
    for shape in SHAPES:
        # (mirrored and wrapped taps are defined where the volume spans the stencil)
        if boundary in ("mirror", "wrap") and min(shape) < 3:
            continue
        n = int(np.prod(shape))
        for shift in (0, 1):                                             # operands off the 16-byte boundary: variant 9
            print(ctype, len(taps), boundary, shape, shift, flush=True)
            x = rng.integers(-50, 50, n + shift).astype(dt)
            src, got = ctx.array(x), []
            for sk in (flat, each):
                out = ctx.array(np.full(n + shift + 3, 77, dt))
                sk.stencil(None, _Part(src, shape, shift), _Part(out, shape, shift))
                got.append(out.get())
            assert np.array_equal(got[0], got[1]), (shape, shift)
            assert np.all(got[0][shift + n:] == 77) and np.all(got[0][:shift] == 77)


class _Part(object):
    def __init__(self, arr, shape, off):
        self.d = arr.desc(shape=shape, offset_elems=off)

    def desc(self):
        return self.d


@pytest.mark.parametrize("walk", [1, 2, 3, 4, 7, 8, 16])
@pytest.mark.parametrize("ctype,dt,taps", [("float", np.float32, BOX), ("double", np.float64, STAR), ("Int32", np.int32, ODD)])
def test_walks_through_several_planes(ctx, ctype, dt, taps, walk):
    """the last wave's planes are cut short: depths round one, two and three times the planes a wave makes, their number
    given"""
    import acchip as A
    fn = " + ".join("(%s)%d * t%d" % (ctype, 3 + k % 5, k) for k in range(len(taps)))
    desc = dict(out_rank=3, taps=taps, stencil_fn=fn)
    rng = np.random.default_rng(4)
    for boundary in ("clamp", "constant", "wrap"):
        desc.update(boundary=boundary, boundary_constant="(%s)7" % ctype if boundary == "constant" else None)
        with A.tuning("stencil.flat=2,stencil.thin_3d=0,stencil.flat_walk=%d" % walk, ctx):
            flat = ctx.skeleton(A.SKEL_STENCIL, ctype, wait=True, **desc)
        with A.tuning("stencil.nd=1", ctx):
            each = ctx.skeleton(A.SKEL_STENCIL, ctype, wait=True, **desc)
        for depth in sorted({max(3, d) for d in (walk - 1, walk, walk + 1, 2 * walk + 1, 3 * walk)}):
            for h, w in ((5, 22), (6, 131)):
                print(ctype, boundary, walk, depth, h, w, flush=True)
                src, got = ctx.array(rng.integers(-50, 50, (depth, h, w)).astype(dt)), []
                for sk in (flat, each):
                    out = ctx.empty((depth, h, w), dt)
                    sk.stencil(None, src, out)
                    got.append(out.get())
                assert np.array_equal(got[0], got[1]), (boundary, depth, h, w)


@pytest.mark.parametrize("shape", [(83, 84, 300), (160, 150, 150)])
@pytest.mark.parametrize("taps,planes,ahead", [(STAR, 4, 4), (BOX, 8, 1)])
def test_planes_a_wave_makes_by_itself(ctx, shape, taps, planes, ahead):
    """four, all asked for at once, where a result reads few rows, else eight with one asked for ahead, whatever the volume; a
    walk of 0 says the same"""
    import acchip as A
    desc = dict(out_rank=3, taps=taps, boundary="mirror", stencil_fn=" + ".join("%d * t%d" % (3 + k % 5, k) for k in range(len(taps))))
    for knobs in ("stencil.flat=1", "stencil.flat_walk=0"):
        with A.tuning(knobs, ctx):
            text = A.preview(A.make_desc(A.SKEL_STENCIL, "Int32", **desc), 8)[1]
        assert "#define ACC_FLAT_PLANES %d\n" % planes in text and "#define ACC_PREFETCH %d\n" % ahead in text
    flat = ctx.skeleton(A.SKEL_STENCIL, "Int32", wait=True, **desc)
    with A.tuning("stencil.nd=1", ctx):
        each = ctx.skeleton(A.SKEL_STENCIL, "Int32", wait=True, **desc)
    src, got = ctx.array(np.random.default_rng(4).integers(-50, 50, shape).astype(np.int32)), []
    for sk in (flat, each):
        out = ctx.empty(shape, np.int32)
        sk.stencil(None, src, out)
        got.append(out.get())
    assert np.array_equal(got[0], got[1])


@pytest.mark.parametrize("boundary", ["clamp", "mirror", "wrap", "constant"])
@pytest.mark.parametrize("ctype,dt,taps", [("float", np.float32, BOX), ("double", np.float64, STAR), ("Int32", np.int32, STAR)])
def test_planes_dealt_out_over_the_dies(ctx, boundary, ctype, dt, taps):
    """every length that a row's last vector can have, in planes of just less and just more than the eight waves a die from
    which every die takes a share of every plane, shares of unequal size among them"""
    import acchip as A
    fn = " + ".join("(%s)%d * t%d" % (ctype, 3 + k % 5, k) for k in range(len(taps)))
    desc = dict(out_rank=3, taps=taps, boundary=boundary, stencil_fn=fn, boundary_constant="(%s)7" % ctype if boundary == "constant" else None)
    with A.tuning("stencil.flat=2", ctx):
        flat = ctx.skeleton(A.SKEL_STENCIL, ctype, wait=True, **desc)
    with A.tuning("stencil.nd=1", ctx):
        each = ctx.skeleton(A.SKEL_STENCIL, ctype, wait=True, **desc)
    vec = 16 // np.dtype(dt).itemsize
    rng = np.random.default_rng(5)
    for d, h, w in [(5, 62, 64 * vec - k) for k in range(vec + 1)] + [(9, 66, 61 * vec - 1), (3, 71, 63 * vec + 1), (13, 131, 62 * vec)]:
        print(ctype, boundary, d, h, w, flush=True)
        src, got = ctx.array(rng.integers(-50, 50, (d, h, w)).astype(dt)), []
        for sk in (flat, each):
            out = ctx.array(np.full((d, h, w), 77, dt))
            sk.stencil(None, src, out)
            got.append(out.get())
        assert np.array_equal(got[0], got[1]), (d, h, w)


@pytest.mark.parametrize("boundary", ["clamp", "mirror", "wrap", "constant"])
@pytest.mark.parametrize("svec,ctype,dt,taps", [(1, "float", np.float32, BOX), (1, "double", np.float64, STAR), (2, "Int32", np.int32, STAR),
                                                (4, "double", np.float64, STAR), (8, "float", np.float32, STAR), (8, "Int64", np.int64, BOX)])
def test_columns_a_lane(ctx, boundary, svec, ctype, dt, taps):
    """as many as stencil.svec says: one, whose neighbours stand with other lanes where the boundary mirrors them, and more
    than 16 bytes of them, of which rows that begin on a 16-byte boundary need not be a whole number"""
    import acchip as A
    fn = " + ".join("(%s)%d * t%d" % (ctype, 3 + k % 5, k) for k in range(len(taps)))
    desc = dict(out_rank=3, taps=taps, boundary=boundary, stencil_fn=fn, boundary_constant="(%s)7" % ctype if boundary == "constant" else None)
    with A.tuning("stencil.flat=2,stencil.thin_3d=0,stencil.svec=%d" % svec, ctx):
        assert "skel_stencil_flat.h" in A.preview(A.make_desc(A.SKEL_STENCIL, ctype, **desc), 8)[1] or svec * np.dtype(dt).itemsize > 32
        flat = ctx.skeleton(A.SKEL_STENCIL, ctype, wait=True, **desc)
    with A.tuning("stencil.nd=1", ctx):
        each = ctx.skeleton(A.SKEL_STENCIL, ctype, wait=True, **desc)
    rng = np.random.default_rng(5)
    for d, h, w in ((5, 7, 20), (9, 5, 36), (3, 6, 61), (4, 62, 64), (6, 70, 130), (3, 3, 16), (4, 9, 260)):
        print(svec, ctype, boundary, d, h, w, flush=True)
        src, got = ctx.array(rng.integers(-50, 50, (d, h, w)).astype(dt)), []
        for sk in (flat, each):
            out = ctx.array(np.full((d, h, w), 77, dt))
            sk.stencil(None, src, out)
            got.append(out.get())
        assert np.array_equal(got[0], got[1]), (d, h, w)
