"""Counts on more targets than whole elements fit LDS for (a row of 8-bit counts a workgroup, added up by permute_merge): as
many sources as give one row, a few, a whole number of the merge's batches and one row more or less; targets that end amid
a word, and few and many words for the merge's workgroups.  Against numpy, exact."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    import acchip as A
    return A.Context(0)


@pytest.mark.parametrize("waves", [4, 7, 16])
def test_rows(ctx, waves):
    import acchip as A
    with A.tuning("permute.narrow_from=100,permute.merge_waves=%d" % waves, ctx):
        sk = ctx.skeleton(A.SKEL_PERMUTE, "Int32", env=[(1, "Int32")], out_rank=1, get="1", combine="x + y", permutation="arrIn0_0[ix]",
                          combine_hint=A.COMBINE_ADD, wait=True)
    tile = sk.info().elements_per_block
    rng = np.random.default_rng(9)
    for bins in (127, 1000, 8193, 18754, 65535, 65536):
        for rows in (1, 2, 17, 63, 64, 65, 129, 255, 300):
            n = rows * tile - 5
            if n < 4 * bins:
                continue
            print(bins, rows, n, flush=True)
            keys = (rng.integers(0, bins, n) if rows % 2 else np.minimum(rng.zipf(1.3, n) - 1, bins - 1)).astype(np.int32)
            base = rng.integers(0, 1 << 20, bins).astype(np.int32)
            out = ctx.empty(bins, np.int32)
            sk.permute([ctx.array(keys)], n, ctx.array(base), out)
            assert np.array_equal(out.get(), base + np.bincount(keys, minlength=bins).astype(np.int32)), (bins, rows)
