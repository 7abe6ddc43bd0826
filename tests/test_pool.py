"""The pool of idle device blocks (parrsb_amd/csrc/hip/runtime.hip) on the CPU:
the file holds no kernels, so it is compiled with g++ against a stand-in for
the runtime's allocator that counts bytes and fails beyond a capacity."""
import ctypes as C
import os
import subprocess
import threading

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIP = os.path.join(ROOT, "parrsb_amd", "csrc", "hip")

STAND_IN = r"""
#include "runtime.hpp"
#include <atomic>
#include <cstdlib>
#include <map>
#include <mutex>
static std::mutex mu;
static std::map<void *, size_t> blocks;
static size_t used, capacity = ~(size_t)0;
static int mallocs, frees, objects;
extern "C" {
hipError_t hipMalloc(void **p, size_t n) {
  std::lock_guard<std::mutex> l(mu);
  mallocs++;
  if (n > capacity - used) return hipErrorOutOfMemory;
  *p = malloc(1);
  blocks[*p] = n, used += n;
  return hipSuccess;
}
hipError_t hipFree(void *p) {
  std::lock_guard<std::mutex> l(mu);
  auto it = blocks.find(p);
  if (it == blocks.end()) abort();  // freed twice
  used -= it->second, blocks.erase(it), free(p), frees++;
  return hipSuccess;
}
hipError_t hipGetDevice(int *d) { *d = 0; return hipSuccess; }
hipError_t hipGetLastError(void) { return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t) { objects--; return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t) { objects--; return hipSuccess; }
hipError_t hipHostFree(void *) { objects--; return hipSuccess; }
static hipError_t drain = hipSuccess, query = hipErrorNotReady;
static int flag, sets_after, queries, syncs, yields;
static unsigned device_flags;
hipError_t hipStreamSynchronize(hipStream_t) { syncs++, flag = sets_after > 0; return drain; }
hipError_t hipStreamQuery(hipStream_t) {
  if (++queries == sets_after) flag = 1;
  return query;
}
hipError_t hipGetDeviceFlags(unsigned *f) { *f = device_flags; return hipSuccess; }
int sched_yield(void) { yields++; return 0; }
// waits for a flag set at the n-th query or by the synchronisation (0: never)
int t_await(unsigned flags, int n, int drains, int ended, int *out) {
  flag = queries = syncs = yields = 0, sets_after = n, device_flags = flags | hipDeviceMapHost;
  drain = drains ? hipSuccess : hipErrorUnknown, query = ended ? hipSuccess : hipErrorNotReady;
  const hipError_t e = rsb_await((hipStream_t)8, &flag, rsb_schedule());
  out[0] = queries, out[1] = syncs, out[2] = yields;
  return e;
}
int t_drain(int ok, int n, void **p) {
  drain = ok ? hipSuccess : hipErrorUnknown;
  return rsb_drain_release((hipStream_t)8, std::vector<const void *>(p, p + n));
}
void *t_malloc(size_t n) { void *p = nullptr; return rsb_pool_malloc(&p, n) == hipSuccess ? p : nullptr; }
void t_free(void *p) { (void)rsb_pool_free(p); }
void t_release(void *p) { rsb_pool_release(p); }
void t_settings(void) { rsb_pool_settings(); }
void t_tick(void) { rsb_pool_tick(0); }
void t_capacity(size_t n) { capacity = n; }
size_t t_used(void) { return used; }
int t_mallocs(void) { return mallocs; }
int t_give_streams(void) {
  const rsb_stream_set s{(hipStream_t)8, {(hipEvent_t)8, (hipEvent_t)8, (hipEvent_t)8, (hipEvent_t)8}, (int *)8};
  objects += 6;
  if (rsb_pool_give_streams(0, s)) return 1;
  rsb_destroy_streams(s);
  return 0;
}
int t_objects(void) { return objects; }
}
hipError_t rsb_dev_free(const void *p) { return rsb_pool_free(p); }
void rsb_dev_release(const void *p) { rsb_pool_release(p); }
"""


@pytest.fixture(scope="module")
def built(tmp_path_factory):
    d = tmp_path_factory.mktemp("pool")
    src = d / "stand_in.cpp"
    src.write_text(STAND_IN)
    so = d / "libpool.so"
    subprocess.run(["g++", "-std=c++17", "-O1", "-fPIC", "-shared", "-Wall", "-Wno-unused-result",
                    "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-I" + HIP,
                    "-I" + os.path.join(ROOT, "include"), "-x", "c++",
                    os.path.join(HIP, "runtime.hip"), str(src), "-o", str(so), "-lpthread"],
                   check=True)
    return so


@pytest.fixture()
def pool(built, tmp_path, monkeypatch):
    """A copy of its own for each test: the pool lives as long as the library."""
    monkeypatch.delenv("PARRSB_AMD_POOL_MB", raising=False)
    so = tmp_path / "libpool.so"
    so.write_bytes(built.read_bytes())
    L = C.CDLL(str(so), mode=os.RTLD_LOCAL | os.RTLD_NOW | getattr(os, "RTLD_DEEPBIND", 8))
    L.t_malloc.restype, L.t_malloc.argtypes = C.c_void_p, [C.c_size_t]
    L.t_free.argtypes = L.t_release.argtypes = [C.c_void_p]
    L.t_capacity.argtypes, L.t_used.restype = [C.c_size_t], C.c_size_t
    L.rsbgpu_release_memory.restype = C.c_longlong
    return L


MB = 1 << 20


def _stats(L):
    out = (C.c_int64 * 3)()
    assert L.rsbgpu_memory(0, out) == 0
    return list(out)


def test_idle_blocks_serve_again_and_go_back_on_request(pool):
    a = [pool.t_malloc(3 * MB) for _ in range(4)]
    assert _stats(pool) == [12 * MB, 0, 12 * MB]
    for p in a:
        pool.t_release(p)
    assert _stats(pool) == [0, 12 * MB, 12 * MB] and pool.t_used() == 12 * MB
    n = pool.t_mallocs()
    p = pool.t_malloc(3 * MB - 100)
    assert pool.t_mallocs() == n and p in a
    assert pool.t_give_streams() == 1 and pool.t_objects() == 6
    assert pool.rsbgpu_release_memory() == 9 * MB  # the block in use stays
    assert pool.t_used() == 3 * MB and _stats(pool) == [3 * MB, 0, 3 * MB]
    assert pool.t_objects() == 0
    pool.t_release(p)
    assert pool.rsbgpu_release_memory() == 3 * MB and pool.t_used() == 0
    assert pool.rsbgpu_release_memory() == 0


@pytest.mark.parametrize("mb", [0, 5, None])
def test_bound(pool, mb, monkeypatch):
    if mb is not None:
        monkeypatch.setenv("PARRSB_AMD_POOL_MB", str(mb))
    pool.t_settings()
    limit = (4096 if mb is None else mb) * MB
    unit = MB if mb is not None else 512 * MB
    for p in [pool.t_malloc(unit) for _ in range(12)]:
        pool.t_release(p)
    assert _stats(pool)[1] == min(limit, 12 * unit) == pool.t_used()
    assert pool.t_give_streams() == (0 if mb == 0 else 1)


def test_blocks_nobody_asks_for_go_back(pool):
    pool.t_release(pool.t_malloc(MB))
    for _ in range(16):
        pool.t_tick()
    assert _stats(pool)[1] == MB
    pool.t_tick()
    assert _stats(pool)[1] == 0 and pool.t_used() == 0


def test_memory_running_out_empties_the_pool(pool):
    pool.t_capacity(64 * MB)
    for p in [pool.t_malloc(8 * MB) for _ in range(6)]:
        pool.t_release(p)
    p = pool.t_malloc(60 * MB)
    assert p and pool.t_used() == 60 * MB and _stats(pool)[1] == 0
    assert not pool.t_malloc(60 * MB)


def test_a_block_that_fits_only_at_its_own_size(pool, monkeypatch):
    """Sizes are rounded up to an eighth of their power of two, unless only
    the exact size fits."""
    n = 8 * MB + 5
    pool.t_capacity(9 * MB - 1)
    p = pool.t_malloc(n)
    assert p and pool.t_used() == n and _stats(pool)[0] == n
    pool.t_release(p)
    assert pool.t_malloc(n - 3 * MB) == p and pool.t_used() == n  # up to twice the size serves
    pool.t_capacity(1 << 40)
    monkeypatch.setenv("PARRSB_AMD_MEM_LIMIT_MB", "10")
    pool.t_settings()
    assert not pool.t_malloc(2 * MB) and pool.t_malloc(MB)


@pytest.mark.parametrize("ok", [0, 1])
def test_blocks_of_a_stream_that_did_not_drain_stay_out(pool, ok):
    p = (C.c_void_p * 4)(pool.t_malloc(MB), None, pool.t_malloc(2 * MB), pool.t_malloc(MB))
    assert pool.t_drain(ok, 4, p) == ok
    assert _stats(pool)[:2] == [0, 4 * MB * ok] and pool.t_used() == 4 * MB * ok


AUTO, SPIN, YIELD, BLOCKING = 0, 1, 2, 4
NOT_READY, UNKNOWN = 600, 999


@pytest.mark.parametrize("flags", [AUTO, SPIN, YIELD, BLOCKING])
def test_the_host_waits_as_the_schedule_flags_ask(pool, flags):
    out = (C.c_int * 3)()
    assert pool.t_await(flags, 3, 1, 0, out) == 0
    queries, syncs, yields = out
    if flags == BLOCKING:  # asleep in the runtime, not looking
        assert (queries, syncs, yields) == (0, 1, 0)
        assert pool.t_await(flags, 0, 1, 0, out) == NOT_READY
        assert pool.t_await(flags, 3, 0, 0, out) == UNKNOWN
    else:
        assert queries == 3 and syncs == 0 and (yields > 1000) == (flags == YIELD)
        # a stream that ends without setting the flag
        assert pool.t_await(flags, 0, 1, 1, out) == NOT_READY and out[0] == 1


def test_threads(pool):
    def work(k):
        for i in range(300):
            p = [pool.t_malloc((1 + (i * 7 + k * 3 + j) % 9) * 4096) for j in range(5)]
            for q in p[:4]:
                pool.t_release(q)
            pool.t_free(p[4])
            if i % 50 == 0:
                pool.rsbgpu_release_memory()
            pool.t_tick()
    ts = [threading.Thread(target=work, args=(k,)) for k in range(6)]
    for t in ts:
        t.start()
    for t in ts:
        t.join(60)
    assert not any(t.is_alive() for t in ts)
    assert _stats(pool)[0] == 0
    pool.rsbgpu_release_memory()
    assert pool.t_used() == 0
