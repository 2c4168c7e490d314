"""`permute const` (skel_scatter.h) on the CPU: the generated kernels, compiled for the host and run a thread at a time
(`permute` and `permute_claim` have no barrier).  What is asked here is which reads a kernel makes, and a read that should
not be made is best made where memory is plain: the element function leaves a mark wherever it is evaluated."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
DEVICE = os.path.join(ROOT, "accelerate-cuda_amd", "csrc", "device")
CLANG = "/opt/rocm/llvm/bin/clang++"
TYPES = {"Int8": np.int8, "Int32": np.int32, "float": np.float32, "Int64": np.int64}

# what the kernels take from acc_hip_device.h, for one thread at a time
STUB = """
#pragma once
typedef signed char Int8; typedef short Int16; typedef int Int32; typedef long long Int64;
typedef unsigned char Word8; typedef unsigned short Word16; typedef unsigned int Word32; typedef unsigned long long Word64;
#define ACC_DEV static inline
#define ACC_IGNORE (-1LL)
#define ACC_GUARD_PARAM
#define ACC_GUARD_CHECK
#define __global__
#define __launch_bounds__(n)
#define __shared__ static
#define __syncthreads()
struct place { unsigned int x; };
static place blockIdx, threadIdx, gridDim;
template <bool B> struct acc_bool { static constexpr bool value = B; };
template <typename T> ACC_DEV T acc_min(T x, T y) { return x < y ? x : y; }
template <typename T> ACC_DEV T acc_max(T x, T y) { return x > y ? x : y; }
ACC_DEV unsigned long long __ballot(bool p) { return p ? 1 : 0; }         /* (a wave of one lane) */
template <typename T> ACC_DEV T acc_readlane(const T &v, int) { return v; }
template <typename T> ACC_DEV T acc_stream(const T *p, const Int64 ix) { return p[ix]; }
"""


@pytest.fixture(scope="module")
def A():
    import acchip
    return acchip


def scatter(A, tmp_path, elt, env, arrays, n, out, **fragments):
    """the call `permute`, preceded by permute_claim where the kernel wants it: `out` as it leaves it"""
    desc = A.make_desc(A.SKEL_PERMUTE, elt, env=[(1, t) for t in env], out_rank=1, **fragments)
    _, src = A.preview(desc, 1)
    comps = [t.strip() for t in elt.split(",")]
    names = ", ".join("shIn%d_0, arrIn%d_0" % (k, k) for k in range(len(env))) + ", shOut_0, "
    names += ", ".join("arrOut_%d" % c for c in range(len(comps) - 1, -1, -1))
    src += """
extern "C" void each_thread(ACC_ENV_PARAMS ACC_OUT_PARAMS, const Int64 n, unsigned int *winner)
{
  gridDim.x = (unsigned)((n + ACC_TILE - 1) / ACC_TILE);
  for (int pass = ACC_CLAIMED ? 0 : 1; pass < 2; ++pass)
    for (blockIdx.x = 0; blockIdx.x < gridDim.x; ++blockIdx.x)
      for (threadIdx.x = 0; threadIdx.x < ACC_BLOCK; ++threadIdx.x)
        if (pass) permute(%s, 0, n, winner);
        else      permute_claim(%s, 0, n, winner);
}
""" % (names, names)
    (tmp_path / "acc_hip_device.h").write_text(STUB)
    text = open(os.path.join(DEVICE, "skel_scatter.h")).read()
    wait = 'asm volatile("s_waitcnt vmcnt(0)" ::: "memory");'
    assert text.count(wait) == 1
    (tmp_path / "skel_scatter.h").write_text(text.replace(wait, ""))
    (tmp_path / "kernel.cpp").write_text(src)
    so = tmp_path / "kernel.so"
    subprocess.run([CLANG, "-x", "c++", "-std=c++17", "-O1", "-w", "-fPIC", "-shared", "-I", str(tmp_path), "-o", str(so), str(tmp_path / "kernel.cpp")],
                   check=True, capture_output=True)
    args = []
    for a in arrays:
        args += [C.c_int64(a.size), C.c_void_p(a.ctypes.data)]
    args.append(C.c_int64(out[0].size))
    args += [C.c_void_p(o.ctypes.data) for o in out]                     # highest component first
    winner = np.full(out[0].size, 0xffffffff, np.uint32)
    C.CDLL(str(so)).each_thread(*args, C.c_int64(n), C.c_void_p(winner.ctypes.data))
    return out


@pytest.mark.parametrize("whole", [True, False])
@pytest.mark.parametrize("elt", ["Int8", "Int32", "Int64", "Int32, Int8"])
def test_the_element_of_a_source_that_is_dropped_is_not_evaluated(A, tmp_path, elt, whole):
    """a gather through an index that is -1 where the source is dropped: by ACC_IGNORE, by a target beyond the result;
    with every operand as long as the source (asked for ahead of the tests) and with one that is shorter"""
    n = 5000
    rng = np.random.default_rng(n)
    comps = [t.strip() for t in elt.split(",")]
    places = rng.permutation(n + 60).astype(np.int32)[:n]                # 60 targets' worth lie beyond the result
    places[rng.random(n) < 0.4] = -1
    kept = (places >= 0) & (places < n)
    through = np.where(kept, rng.integers(0, 100, n), -1).astype(np.int32)
    values = rng.integers(0, 100, 100).astype(np.int32)
    marks = np.zeros(n, np.int32)
    length = np.zeros(n if whole else n - 1, np.int32)                   # read at its own index below its end only
    value = "({ ((Int32 *)arrIn3_0)[ix] = 1; const Int32 i = arrIn1_0[ix]; (i < 0 ? 99 : arrIn0_0[i]) + (ix < shIn4_0 ? arrIn4_0[ix] : 0); })"
    get = "(%s)%s" % (comps[0], value) if len(comps) == 1 else "acc_elt{%s, (Int8)(ix %% 100)}" % value
    out = [np.full(n, 77, TYPES[t]) for t in comps]
    scatter(A, tmp_path, elt, ["Int32"] * 5, [values, through, places, marks, length], n, out, get=get,
            combine="x" if len(comps) == 1 else "acc_elt{x.a1, x.a0}", permutation="(Int64)arrIn2_0[ix]")
    assert np.array_equal(marks != 0, kept)
    want = np.full(n, 77, np.int64)
    want[places[kept]] = values[through[kept]]
    assert np.array_equal(out[0].astype(np.int64), want)
    if len(comps) > 1:
        want[places[kept]] = np.flatnonzero(kept) % 100
        assert np.array_equal(out[1].astype(np.int64), want)


def test_which_element_functions_are_worked_out_ahead(A):
    """... of every source: those that cannot fail to have a value, whatever the source's own operands hold"""
    def total(get, **more):
        d = A.make_desc(A.SKEL_PERMUTE, "Int32", env=[(1, "Int32"), (1, "Int32")], out_rank=1, get=get, combine="x", permutation="(Int64)arrIn1_0[ix]", **more)
        return "#define ACC_GET_TOTAL 1\n" in A.preview(d)[1]
    for get in ("arrIn0_0[ix]", "(acc_stream(arrIn0_0, ix) * 3 + (Int32)ix)", "arrIn0_0[ix] > 0 ? arrIn1_0[ix] : -1", "(Int32)(1.5e-3f * (float)arrIn0_0[ix])"):
        assert total(get), get
    for get in ("arrIn0_0[arrIn1_0[ix]]", "arrIn0_0[ix + 1]", "arrIn0_0[0]", "arrIn0_0[ix] / arrIn1_0[ix]", "arrIn0_0[ix] % arrIn1_0[ix]", "abs(arrIn0_0[ix])",
                "({ Int32 a = arrIn0_0[ix]; while (a > 9) a -= arrIn1_0[ix]; a; })", "*(arrIn0_0 + arrIn1_0[ix])", "acc_stream(arrIn0_0, arrIn1_0[ix])"):
        assert not total(get), get
    assert not total("arrIn0_0[ix]", preamble="#define V 1")


def _next(a):
    return np.append(a[1:], 0)


REBOUND = [
    # (fragment, preamble, its value from the arrays a and b and the index i)
    ("[&](Int64 ix) { return arrIn0_0[ix]; }((Int64)arrIn1_0[ix])", None, lambda a, b, i: a[b]),
    ("[&](Int64 ix) { return acc_stream(arrIn0_0, ix) + arrIn1_0[ix]; }(ix / 2)", None, lambda a, b, i: a[i // 2] + b[i // 2]),
    ("({ Int32 s = arrIn1_0[ix]; for (Int64 ix = 0; ix < 3; ++ix) s += arrIn0_0[ix]; s; })", None, lambda a, b, i: b + a[:3].sum()),
    ("({ const unsigned char ix = 7; arrIn0_0[ix]; })", None, lambda a, b, i: 0 * i + a[7]),
    ("({ const Int32 *arrIn0_0 = arrIn1_0; arrIn0_0[ix]; })", None, lambda a, b, i: b),
    ("({ struct { const Int32 *arrIn0_0; } s = {arrIn1_0}; s.arrIn0_0[ix]; })", None, lambda a, b, i: b),
    ("({ const Int32 *p = &arrIn0_0[ix]; ix + 1 < shIn0_0 ? p[1] : 0; })", None, lambda a, b, i: _next(a)),
    ("({ auto &v = arrIn0_0[ix]; v + (3 & arrIn1_0[ix]); })", None, lambda a, b, i: a + (3 & b)),
    ("AT(arrIn1_0[ix]) + arrIn0_0[ix]", "#define AT(i) [&](Int64 ix) { return arrIn0_0[ix]; }(i)", lambda a, b, i: a[b] + a),
    ("arrIn0_0[ix] + first * past + copy", "static const Int32 first = 2, past = 3, copy = 4;", lambda a, b, i: a + 10),
    ("not_acc_stream(arrIn0_0, ix)", "ACC_DEV Int32 not_acc_stream(const Int32 *p, Int64 ix) { return p[ix] + 1; }", lambda a, b, i: a + 1),
]


@pytest.mark.parametrize("fragment,preamble,value", REBOUND)
@pytest.mark.parametrize("where", ["get", "permutation"])
def test_names_that_a_fragment_gives_to_something_of_its_own(A, tmp_path, fragment, preamble, value, where):
    n = 3000
    rng = np.random.default_rng(1)
    a, b = rng.integers(0, n, n).astype(np.int32), rng.permutation(n).astype(np.int32)
    places, want = rng.permutation(n).astype(np.int32), np.full(n, -5, np.int32)
    v = value(a, b, np.arange(n))
    out = [want.copy()]
    if where == "get":
        scatter(A, tmp_path, "Int32", ["Int32"] * 3, [a, b, places], n, out, get=fragment, combine="x", permutation="(Int64)arrIn2_0[ix]", preamble=preamble)
        want[places] = v
        assert np.array_equal(out[0], want)
    else:                                                    # (of several sources on one target any: they bring their target)
        scatter(A, tmp_path, "Int32", ["Int32"] * 2, [a, b], n, out, get=fragment, combine="x", permutation="(Int64)(%s)" % fragment, preamble=preamble)
        v = v[(v >= 0) & (v < n)]
        want[v] = v
        assert np.array_equal(out[0], want)


def test_reads_at_the_own_index_are_taken_ahead(A):
    """... of the fragments as the front end and the other code generators write them"""
    def own(get, **more):
        d = A.make_desc(A.SKEL_PERMUTE, "Int32", env=[(1, "Int32"), (2, ["Int32", "float"])], out_rank=1, get=get, combine="x", permutation="(Int64)arrIn0_0[ix]", **more)
        return [line for line in A.preview(d)[1].splitlines() if line.startswith("#define ACC_OWN_FIELDS")][0][len("#define ACC_OWN_FIELDS"):].split()
    assert own("arrIn0_0 [ ix ]") == ["Int32", "s0_0;"]
    assert own("(Int32)(acc_stream( arrIn1_1 ,ix ) * 2.0f) & 3 & arrIn1_0[ix]") == ["Int32", "s0_0;", "Int32", "s1_0;", "float", "s1_1;"]
    assert own("[&] { const Int32 v = arrIn1_0[ix]; return v * v; }()") == ["Int32", "s0_0;", "Int32", "s1_0;"]
    assert own("arrIn1_0[ix + 1] + arrIn1_0[(ix)]") == ["Int32", "s0_0;"]
    assert own("*(&arrIn1_0[ix])") == ["Int32", "s0_0;"] and own("1", preamble="#define V 1") == []
