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
