"""Folds along rows that lie across memory at the sizes where the work is cut otherwise: rows either side of a wave's lanes,
of several rows a lane and of the bound between the two entries; lengths that are not cut, cut into pieces of one
workgroup and of many, with pieces left empty.  An operator that is associative and does not commute, from either side,
against the same chain in numpy: whole numbers, exact."""
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


@pytest.fixture(scope="module")
def ctx():
    import acchip as A
    return A.Context(0)


@pytest.mark.parametrize("right", [False, True])
@pytest.mark.parametrize("seeded", [False, True])
def test_not_commutative(ctx, right, seeded):
    import acchip as A
    sk = ctx.skeleton(A.SKEL_FOLD if seeded else A.SKEL_FOLD1, "Word32", env=[(2, "Word32")], out_rank=1, get="arrIn0_0[acc_col * shIn0_0 + acc_row]",
                      combine="affine16(x, y)", seed=str(SEED) if seeded else None, preamble=AFFINE,
                      flags=A.FLAG_TILED | (A.FLAG_FOLD_RIGHT if right else 0), wait=True)
    rng = np.random.default_rng(8)
    for w in (1, 3, 63, 64, 65, 255, 256, 257, 4095, 4096, 4097):
        for h in (8, 16, 31, 32, 33, 35, 63, 67, 1025, 16 * 4 * 300 + 1):
            if w * h > 1 << 21:
                continue
            print("affine", "right" if right else "left", seeded, h, w, flush=True)
            m = rng.integers(0, 2**32, (h, w), dtype=np.uint64).astype(np.uint32)
            m[:, 0] |= 0x00010000
            out = ctx.array(np.full(w + 2, 77, np.uint32))
            sk.fold([ctx.array(m)], (w, h), out.desc(shape=(w,)))
            want = m[0].astype(np.uint64)
            for k in range(1, h):
                want = affine(want, m[k].astype(np.uint64))
            if seeded:
                want = affine(want, np.uint64(SEED))
            got = out.get()
            assert np.array_equal(got[:w], want.astype(np.uint32)), (h, w)
            assert np.array_equal(got[w:], [77, 77])


@pytest.mark.parametrize("ctype,dt", [("Int8", np.int8), ("Int64", np.int64), ("Int64, Int32, Int64", None)])
def test_element_sizes(ctx, ctype, dt):
    """four rows a lane of 1-byte elements, two of 8 bytes, one of a tuple"""
    import acchip as A
    tup = dt is None
    src_t, src_dt = ("Int32", np.int32) if tup else (ctype, dt)
    read = "arrIn0_0[acc_col * shIn0_0 + acc_row]"
    sk = ctx.skeleton(A.SKEL_FOLD, ctype, env=[(2, src_t)], out_rank=1, flags=A.FLAG_TILED, wait=True,
                      get="acc_elt{(Int64)%s, 1, (Int64)%s * 2}" % (read, read) if tup else read,
                      combine="acc_elt{x.a2 + y.a2, x.a1 + y.a1, x.a0 + y.a0}" if tup else "(%s)(x + y)" % ctype, seed="acc_elt{0, 0, 0}" if tup else "0")
    rng = np.random.default_rng(9)
    for h, w in ((9, 5), (40, 130), (700, 67), (5000, 300), (129, 4100)):
        print("sums", ctype, h, w, flush=True)
        m = rng.integers(-9, 10, (h, w)).astype(src_dt)
        total = m.sum(axis=0, dtype=np.int64)
        if tup:
            out = ctx.empty_tuple(w, [np.int64, np.int32, np.int64])
            sk.fold([ctx.array(m)], (w, h), out)
            a, b, c = out.get()
            assert np.array_equal(a, total) and np.array_equal(b, np.full(w, h)) and np.array_equal(c, 2 * total)
        else:
            out = ctx.empty(w, src_dt)
            sk.fold([ctx.array(m)], (w, h), out)
            assert np.array_equal(out.get(), total.astype(src_dt))
