"""Segmented folds (skel_foldseg.h) on the CPU: the generated kernel, compiled for the host, a thread a lane and one
workgroup.  What is asked here is where in a staged chunk a lane looks for its segment when the chunk lies beyond element
2^31 of the source, and a place outside the chunk is best looked at where memory is plain: every element of the chunk is
told from what surrounds it."""
import ctypes as C
import mmap
import os
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
DEVICE = os.path.join(ROOT, "accelerate-cuda_amd", "csrc", "device")
CLANG = "/opt/rocm/llvm/bin/clang++"

# what the kernel takes from acc_hip_device.h: one wave of 64 lanes, which meet at a barrier
STUB = """
#pragma once
#include <pthread.h>
#include <thread>
#include <vector>
typedef signed char Int8; typedef short Int16; typedef int Int32; typedef long long Int64;
typedef unsigned char Word8; typedef unsigned short Word16; typedef unsigned int Word32; typedef unsigned long long Word64;
#define ACC_DEV static inline
#define ACC_WAVE 64
#define ACC_GUARD_PARAM
#define ACC_GUARD_CHECK
#define __global__
#define __launch_bounds__(n)
#define __shared__ static
#define __HIP_MEMORY_SCOPE_WORKGROUP 3
struct place { unsigned int x; };
static place blockIdx, gridDim;
static thread_local place threadIdx;
static pthread_barrier_t meet;
static inline void __syncthreads() { pthread_barrier_wait(&meet); }
template <bool B> struct acc_bool { static constexpr bool value = B; };
template <typename T> ACC_DEV T acc_min(T x, T y) { return x < y ? x : y; }
template <typename T> ACC_DEV T acc_max(T x, T y) { return x > y ? x : y; }
template <typename T> ACC_DEV void acc_pin(T &) {}
ACC_DEV int acc_lane() { return (int)threadIdx.x; }
static unsigned long long votes;
ACC_DEV unsigned long long __ballot(bool p)
{
  if (acc_lane() == 0) votes = 0;
  __syncthreads();
  if (p) __atomic_fetch_or(&votes, 1ull << acc_lane(), __ATOMIC_RELAXED);
  __syncthreads();
  return votes;
}
template <typename T> struct acc_opt { T v; int ok; };
template <typename T> ACC_DEV acc_opt<T> acc_some(const T &v) { return {v, 1}; }
template <typename T> ACC_DEV acc_opt<T> acc_none() { return {T(), 0}; }
template <typename T, typename F> struct acc_lifted {
  F f;
  acc_opt<T> operator()(const acc_opt<T> &x, const acc_opt<T> &y) const { return !x.ok ? y : !y.ok ? x : acc_some(f(x.v, y.v)); }
};
template <typename T, typename F> ACC_DEV acc_lifted<T, F> acc_lift(F f) { return {f}; }
template <typename T, typename F> ACC_DEV acc_opt<T> acc_wave_reduce(acc_opt<T> x, const acc_lifted<T, F> &f)
{
  static acc_opt<T> of[ACC_WAVE];
  of[acc_lane()] = x;
  __syncthreads();
  acc_opt<T> all = of[0];
  for (int k = 1; k < ACC_WAVE; ++k) all = f(all, of[k]);
  __syncthreads();
  return all;
}
"""

CALL = """
extern "C" void one_workgroup(const Int64 nseg, ACC_ELT *out, const Int64 n, const Int64 *offsets)
{
  gridDim.x = 1;
  blockIdx.x = 0;
  pthread_barrier_init(&meet, nullptr, ACC_BLOCK);
  std::vector<std::thread> lanes;
  for (unsigned lane = 0; lane < ACC_BLOCK; ++lane)
    lanes.emplace_back([=] { threadIdx.x = lane; foldSeg(nseg, out, n, offsets); });
  for (std::thread &t : lanes) t.join();
}
"""
PLACE = """
extern "C" int place_in_chunk(Int64 ix, Int64 cs, Int64 ce) { return acc_place_in_chunk(ix, cs, ce); }
"""


@pytest.fixture(scope="module")
def A():
    import acchip
    return acchip


def build(A, tmp_path, more="", **fragments):
    """foldSeg of the generated source for the host: the template as far as its first entry goes"""
    with A.tuning("foldseg.block=64"):
        _, src = A.preview(A.make_desc(A.SKEL_FOLDSEG, "Int64", combine="x + y", seed="0", seg_type="Int64", **fragments), 1)
    (tmp_path / "acc_hip_device.h").write_text(STUB)
    text = open(os.path.join(DEVICE, "skel_foldseg.h")).read()
    entry, end = text.index("ACC_FOLDSEG_ENTRY(ACC_ENV_PARAMS"), "\n#if ACC_SEG_UNIFORM\n/* ---- short rows"
    assert text.count(end) == 1 and entry < text.index(end)
    (tmp_path / "skel_foldseg.h").write_text(text[:text.index(end)])
    (tmp_path / "kernel.cpp").write_text(src + CALL + more)
    so = tmp_path / "kernel.so"
    subprocess.run([CLANG, "-x", "c++", "-std=c++17", "-O1", "-w", "-fPIC", "-shared", "-pthread", "-I", str(tmp_path), "-o", str(so), str(tmp_path / "kernel.cpp")],
                   check=True, capture_output=True)
    return C.CDLL(str(so))


def fold(lib, offsets, n):
    """the segments' folds, worked out in a child: a read far outside the chunk would end the process"""
    offsets = np.asarray(offsets, np.int64)
    out = np.frombuffer(mmap.mmap(-1, 8 * (len(offsets) - 1)), np.int64)
    child = os.fork()
    if child == 0:
        lib.one_workgroup(C.c_int64(len(out)), C.c_void_p(out.ctypes.data), C.c_int64(n), C.c_void_p(offsets.ctypes.data))
        os._exit(0)
    assert os.waitpid(child, 0)[1] == 0
    return out


@pytest.mark.parametrize("right", [False, True])
@pytest.mark.parametrize("first", [0, (1 << 31) - 700, (1 << 31) + 5, 3 << 30, (1 << 32) - 9, (1 << 32) + 77, 11 << 30])
@pytest.mark.parametrize("nseg", [1, 40, 63, 64, 130])
def test_lanes_without_a_segment_fold_nothing(A, tmp_path_factory, first, nseg, right):
    """chunks anywhere in the source, fewer segments than lanes and a last turn of few: a lane that has none looks at no
    element and is no owner of a stretch that all of them fold (empty segments and such stretches among them)"""
    key = "right" if right else "left"
    if key not in _built:
        _built[key] = build(A, tmp_path_factory.mktemp(key), get="ix", flags=A.FLAG_FOLD_RIGHT if right else 0)
    rng = np.random.default_rng(nseg)
    lens = rng.integers(0, 60, nseg)
    lens[rng.integers(0, nseg)] = 700
    offsets = first + np.concatenate([[0], np.cumsum(lens)])
    got = fold(_built[key], offsets, int(offsets[-1]) + 3)
    want = [sum(range(int(a), int(b))) for a, b in zip(offsets[:-1], offsets[1:])]
    assert got.tolist() == want


_built = {}


def test_the_place_of_an_index_in_a_chunk(A, tmp_path):
    """an index before the chunk is its start and one behind it its end, however far away"""
    lib = build(A, tmp_path, PLACE, get="ix")
    lib.place_in_chunk.argtypes = [C.c_int64] * 3
    far = [0, 1, 2047, 2048, (1 << 31) - 1, 1 << 31, (1 << 31) + 2049, (1 << 32) - 1, 1 << 32, 5 << 31, 1 << 40]
    for cs in far:
        for length in (1, 2048):
            for ix in far + [cs + 1, cs + length, cs + length + 1, cs + (1 << 31) + 5, cs + (1 << 32) + 5]:
                assert lib.place_in_chunk(ix, cs, cs + length) == min(max(ix - cs, 0), length), (ix, cs, length)
