"""Calls on a bank whose HIP calls fail: an update leaves the bank as it was,
a batched route without memory goes query by query.

The route library's host code runs here against a stand-in for the HIP
runtime (device memory is host memory, kernels do not run except that row
placement and eviction set norms and ids), which can be told to fail the
n-th call of a function from now on."""

import subprocess
import sys

import pytest

from graftrepository_amd import _lib

RUNTIME = r"""
#include <math.h>
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>
typedef struct { uint32_t x, y, z; } dim3;
static char fail_name[64];
static int fail_in;
void fake_fail(const char* name, int nth) { snprintf(fail_name, 64, "%s", name); fail_in = nth; }
int fake_failed(void) { return fail_in == 0; }
static int last;
static int fails(const char* name) {
  if (strcmp(name, fail_name) != 0 || fail_in == 0 || --fail_in > 0) return 0;
  return last = 2;
}
#define CALL(name) if (fails(#name)) return 2
static size_t pinned, device;
static int pins;
int fake_pins(void) { return pins; }
size_t fake_pinned(void) { return pinned; }
size_t fake_device(void) { return device; }
static void* take(size_t n, size_t* sum) {
  size_t* p = calloc(1, n + 64);
  *p = n;
  *sum += n;
  return p + 8;
}
static int give(void* q, size_t* sum) {
  if (q) { size_t* p = (size_t*)q - 8; *sum -= *p; free(p); }
  return 0;
}
int hipMalloc(void** p, size_t n) { CALL(hipMalloc); *p = take(n, &device); return 0; }
int hipHostMalloc(void** p, size_t n, unsigned f) { CALL(hipHostMalloc); ++pins; *p = take(n, &pinned); return 0; }
int hipFree(void* p) { return give(p, &device); }
int hipHostFree(void* p) { return give(p, &pinned); }
int hipHostGetDevicePointer(void** d, void* h, unsigned f) { *d = h; return 0; }
int hipMemcpyAsync(void* d, const void* s, size_t n, int k, void* q) { CALL(hipMemcpyAsync); memcpy(d, s, n); return 0; }
int hipMemcpy(void* d, const void* s, size_t n, int k) { memcpy(d, s, n); return 0; }
int hipMemsetAsync(void* d, int v, size_t n, void* q) { memset(d, v, n); return 0; }
int hipGetDevice(int* d) { *d = 0; return 0; }
int hipSetDevice(int d) { return 0; }
/* LDS a block may have (hipDeviceAttributeSharedMemPerBlockOptin), and the
   device clock's kHz (hipDeviceAttributeWallClockRate) */
int hipDeviceGetAttribute(int* v, int a, int d) {
  *v = a == 75 ? 163840 : (a == 10017 ? 100000 : 0);
  return *v == 0;
}
int hipStreamCreateWithFlags(void** s, unsigned f) { *s = malloc(1); return 0; }
int hipStreamDestroy(void* s) { free(s); return 0; }
int hipStreamSynchronize(void* s) { return 0; }
int hipStreamWaitEvent(void* s, void* e, unsigned f) { return 0; }
int hipEventCreate(void** e) { *e = malloc(1); return 0; }
int hipEventCreateWithFlags(void** e, unsigned f) { *e = malloc(1); return 0; }
int hipEventDestroy(void* e) { free(e); return 0; }
int hipEventRecord(void* e, void* s) { CALL(hipEventRecord); return 0; }
int hipEventSynchronize(void* e) { return 0; }
int hipEventQuery(void* e) { return 0; }
int hipEventElapsedTime(float* ms, void* a, void* b) { *ms = 1.0f; return 0; }
int hipFuncSetAttribute(const void* f, int a, int v) { return 0; }
int hipGetLastError(void) { const int e = last; last = 0; return e; }
const char* hipGetErrorString(int e) { return "stand-in failure"; }
static struct { const void* host; const char* name; void* object; } kernels[4096];
static int n_kernels;
void** __hipRegisterFatBinary(const void* d) { return malloc(sizeof(void*)); }
void __hipUnregisterFatBinary(void** m) {}
void __hipRegisterFunction(void** m, const void* host, char* dev, const char* name, unsigned t,
                           void* a, void* b, void* c, void* d, int* e) {
  kernels[n_kernels].host = host;
  kernels[n_kernels].object = m;
  kernels[n_kernels++].name = strdup(name);
}
void __hipRegisterVar(void** m, void* v, char* h, char* d, int e, size_t n, int c, int g) {}
static struct { dim3 g, b; size_t lds; void* s; } pushed;
int __hipPushCallConfiguration(dim3 g, dim3 b, size_t lds, void* s) {
  pushed.g = g; pushed.b = b; pushed.lds = lds; pushed.s = s;
  return 0;
}
int __hipPopCallConfiguration(dim3* g, dim3* b, size_t* lds, void** s) {
  *g = pushed.g; *b = pushed.b; *lds = pushed.lds; *s = pushed.s;
  return 0;
}
/* a number per code object: that of kernel i, its name at *name; -1 past the last */
int64_t fake_kernel(int i, const char** name) {
  if (i >= n_kernels) return -1;
  *name = kernels[i].name;
  return (int64_t)kernels[i].object;
}
static float* norms;
static uint64_t* ids;
static uint64_t end_tick[4];
void fake_ticks(uint64_t a, uint64_t b, uint64_t c, uint64_t d) {
  end_tick[0] = a; end_tick[1] = b; end_tick[2] = c; end_tick[3] = d;
}
#define ARG(i, T) (*(T*)args[i])
int hipLaunchKernel(const void* f, dim3 g, dim3 b, void** args, size_t lds, void* s) {
  const char* name = "";
  for (int i = 0; i < n_kernels; ++i) if (kernels[i].host == f) name = kernels[i].name;
  CALL(hipLaunchKernel);
  if (strstr(name, "mla_place_rows_kernel")) {
    const uint64_t* slots = ARG(5, const uint64_t*);
    const uint64_t* from = ARG(6, const uint64_t*);
    norms = ARG(9, float*);
    ids = ARG(10, uint64_t*);
    for (uint64_t r = 0; r < ARG(1, uint64_t); ++r) {
      const uint64_t slot = slots ? slots[r] : ARG(7, uint64_t) + r;
      norms[slot] = 1.0f;
      ids[slot] = from ? from[r] : slot;
    }
  }
  if (strstr(name, "mla_route_kernel") && ARG(11, unsigned*)) {
    /* no node found; the blocks' flags, and their ticks as told */
    for (unsigned i = 0; i < g.x; ++i) {
      for (int j = 0; j < ARG(9, int); ++j) {
        uint32_t* e = ARG(10, uint32_t*) + 4 * (i * ARG(9, int) + j);
        e[0] = 0x7fc00000u;
        e[1] = 0x80000000u | ARG(12, unsigned);
        e[2] = e[3] = ~0u;
      }
      ARG(11, unsigned*)[i] = ARG(12, unsigned);
      uint64_t** stamps = (uint64_t**)args[13];
      if (stamps[0] && i == 0) { stamps[0][0] = 1000; stamps[0][1] = ARG(12, unsigned); }
      if (stamps[1]) stamps[1][i] = i < 4 ? end_tick[i] : end_tick[3];
    }
  }
  if (strstr(name, "mla_evict_kernel")) {
    for (uint64_t r = 0; r < ARG(1, uint64_t); ++r) {
      ARG(2, float*)[ARG(0, const uint64_t*)[r]] = NAN;
      ARG(3, uint64_t*)[ARG(0, const uint64_t*)[r]] = ~0ull;
    }
  }
  return 0;
}
/* ids of the slots below n whose norm is a number, in slot order */
uint64_t fake_live(uint64_t n, uint64_t* out) {
  uint64_t k = 0;
  for (uint64_t i = 0; i < n; ++i) if (norms[i] == norms[i]) out[k++] = ids[i];
  return k;
}
"""

# run in a process of its own: loading the stand-in first binds the library to it
PRELUDE = r"""
import ctypes, sys
hip = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
for f in (hip.fake_live, hip.fake_pinned, hip.fake_device):
    f.restype = ctypes.c_uint64
import numpy as np
from graftrepository_amd import MlaNodeBank
CAP = 20_032

def fail(name, nth=1):
    hip.fake_fail(name.encode(), nth)

def device_ids():
    out = np.empty(CAP, np.uint64)
    n = hip.fake_live(ctypes.c_uint64(CAP), out.ctypes.data_as(ctypes.c_void_p))
    return sorted(out[:n].tolist())

def refused(call, *args):
    try:
        call(*args)
    except RuntimeError:
        assert hip.fake_failed()
        return
    raise AssertionError("the call did not fail")

def state(bank):
    i = bank.info()
    return i["live"], i["epoch"], i["slots_in_use"], device_ids()
"""


@pytest.fixture(scope="module")
def runtime(tmp_path_factory):
    d = tmp_path_factory.mktemp("hip")
    (d / "hip.c").write_text(RUNTIME)
    subprocess.run(["gcc", "-O1", "-shared", "-fPIC", "-w", str(d / "hip.c"), "-o", str(d / "hip.so"), "-lm"],
                   check=True)
    return d / "hip.so"


def run(runtime, body):
    root = _lib.PKG.parent
    subprocess.run([sys.executable, "-c", PRELUDE + body, str(runtime)], check=True, cwd=root, timeout=120)


def test_a_failure_is_reported_once(runtime):
    run(runtime, r"""
with MlaNodeBank(np.ones((100, 32), np.float32), capacity=CAP) as bank:
    fail("hipHostMalloc")
    refused(bank.evict, np.asarray([5, 7], np.uint64))
    bank.evict(np.asarray([5, 7], np.uint64))  # its launch succeeds
    assert state(bank)[0] == 98
""")
APPEND = r"""
COUNT, WHAT, NTH = {count}, "{what}", {nth}
rows = np.ones((100, 288), np.float32)
new = np.ones((COUNT, 288), np.float32)
ids = np.arange(COUNT, dtype=np.uint64) + 1000
with MlaNodeBank(rows, capacity=CAP) as bank:
    bank.evict(np.asarray([3, 50, 98, 99], np.uint64))  # holes and a tail
    before = state(bank)
    assert before[0] == 96 and before[2] == 98
    fail(WHAT, NTH)
    refused(bank.append, new, ids)
    assert state(bank) == before, (state(bank)[:3], before[:3])
    bank.append(new, ids)  # not "already live"
    after = state(bank)
    assert after[0] == 96 + COUNT and after[1] == before[1] + 1 and after[2] == 96 + COUNT
    assert after[3] == sorted(before[3] + ids.tolist())
    bank.evict(ids)
    assert state(bank)[3] == before[3] and state(bank)[0] == 96
"""


# 2,000 rows: placed from the stage in parts; 9,000: through the copy engine
@pytest.mark.parametrize("count,what,nth", [
    (2_000, "hipHostMalloc", 1), (2_000, "hipLaunchKernel", 1), (2_000, "hipLaunchKernel", 3),
    (9_000, "hipHostMalloc", 1), (9_000, "hipMalloc", 1), (9_000, "hipMemcpyAsync", 1),
    (9_000, "hipLaunchKernel", 1)])
def test_failed_append_changes_nothing(runtime, count, what, nth):
    run(runtime, APPEND.format(count=count, what=what, nth=nth))


def test_failed_evict_changes_nothing(runtime):
    run(runtime, r"""
with MlaNodeBank(np.ones((100, 32), np.float32), capacity=CAP) as bank:
    for what in ("hipHostMalloc", "hipLaunchKernel"):
        before = state(bank)
        fail(what)
        refused(bank.evict, np.asarray([5, 7], np.uint64))
        assert state(bank) == before
        bank.evict(np.asarray([5, 7], np.uint64))
        assert state(bank)[0] == before[0] - 2
        bank.append(np.ones((2, 32), np.float32), np.asarray([5, 7], np.uint64))
""")


# an update whose event cannot be recorded waits for its kernels instead
def test_update_without_its_event(runtime):
    run(runtime, r"""
with MlaNodeBank(np.ones((100, 32), np.float32), capacity=CAP) as bank:
    fail("hipEventRecord")
    bank.evict(np.asarray([5, 7], np.uint64))
    assert hip.fake_failed()
    fail("hipEventRecord")
    bank.append(np.ones((2, 32), np.float32), np.asarray([200, 201], np.uint64))
    assert hip.fake_failed()
    assert state(bank)[0] == 100 and state(bank)[3] == sorted([i for i in range(100) if i not in (5, 7)] + [200, 201])
""")


# each buffer of the batched route in turn; the ring screen takes 200 bf16 queries
@pytest.mark.parametrize("dtype,nq,buffers", [("f32", 8, 2), ("bf16", 200, 4)])
def test_batched_route_without_memory(runtime, dtype, nq, buffers):
    run(runtime, f"""
import os
os.environ["GRM_HIP_BLOCKING_SYNC"] = "1"  # kernels do not run: no flags
dtype, nq = "{dtype}", {nq}
rows = np.ones((20_000, 64), np.float32 if dtype == "f32" else np.uint16)
q = np.ones((nq, 64), rows.dtype)
for nth in range(1, {buffers} + 2):
    with MlaNodeBank(rows, dtype=dtype) as bank:
        bank.route(q[:1], 3, query_dtype=dtype)  # the single-query route's buffers
        bank.route(np.ones((nq, 64), rows.dtype), 3, query_dtype=dtype, warmup=nq - 1)
        assert bank.route_stats()["batched"] == 0
        fail("hipMalloc", nth)
        bank.route(q, 3, query_dtype=dtype)
        stats = bank.route_stats()
        if nth <= {buffers}:
            assert hip.fake_failed() and stats["batched"] == 0, (nth, stats)
        else:
            assert not hip.fake_failed() and stats["batched"] == nq, (nth, stats)
""")


# Block 0 stamps the start (tick 1000 of a 100 MHz clock); a short block of
# another XCD may have ended by then
@pytest.mark.parametrize("ticks,us", [((1600, 1500, 1700, 1400), 7.0), ((1600, 900, 1500, 999), 6.0),
                                      ((999, 900, 1, 999), None)])
def test_blocks_that_end_before_the_start_stamp(runtime, ticks, us):
    run(runtime, f"""
with MlaNodeBank(np.ones((200, 32), np.float32)) as bank:  # 4 blocks
    hip.fake_ticks(*(ctypes.c_uint64(t) for t in {ticks}))
    q = np.ones((1, 32), np.float32)
    for _ in range(2):
        try:
            ms = bank.route(q, 3).device_ms
        except RuntimeError:
            assert {us} is None
        else:
            assert abs(ms * 1e3 - {us}) < 1e-3
""")


# Pinned allocations are most of a first call's cost on a new bank: the
# query's, the results' and one for flags, stamps and ticks
@pytest.mark.parametrize("nq,timed", [(1, False), (1, True), (8, False), (8, True)])
def test_pinned_allocations_of_a_first_route(runtime, nq, timed):
    run(runtime, f"""
with MlaNodeBank(np.ones((20_000, 64), np.float32)) as bank:
    hip.fake_ticks(*(ctypes.c_uint64(2000),) * 4)
    before = hip.fake_pins()
    try:
        bank.route(np.ones(({nq}, 64), np.float32), 3, timed={timed})
    except RuntimeError as e:  # the merge kernel does not run here
        assert {nq} > 1 and "completion flags" in str(e)
    assert hip.fake_pins() - before == 3
""")


# ... sized for the call, and for a larger one when that comes; without
# memory for it the call is refused and the next one is as before
def test_marks_grow_with_the_calls(runtime):
    run(runtime, r"""
import os
os.environ["GRM_HIP_MLA_BATCH_MIN"] = "1000"
with MlaNodeBank(np.ones((20_000, 64), np.float32)) as bank:
    hip.fake_ticks(*(ctypes.c_uint64(2000),) * 4)
    q = np.ones((40, 64), np.float32)
    before = hip.fake_pinned()
    bank.route(q[:1], 3)
    assert hip.fake_pinned() - before < 32_768
    for nq in (16, 1, 40):  # 157 blocks a query
        assert abs(bank.route(q[:nq], 3).device_ms - 0.01) < 1e-6
with MlaNodeBank(np.ones((20_000, 64), np.float32)) as bank:
    bank.route(q[:1], 3)
    fail("hipHostMalloc", 3)  # after the query's and the results'
    refused(bank.route, q, 3)
    bank.route(q[:1], 3)
    bank.route(q, 3)
""")


# A bank's first route loads the code object its kernels are in: the screens'
# probe forms, which only tests reach, are not in that one
def test_probe_forms_have_a_code_object_of_their_own(runtime):
    run(runtime, r"""
hip.fake_kernel.restype = ctypes.c_int64
import graftrepository_amd
graftrepository_amd.load()
name, kernels = ctypes.c_char_p(), []
while (o := hip.fake_kernel(len(kernels), ctypes.byref(name))) != -1:
    kernels.append((name.value, o))
def objects(form, *words):
    return {o for n, o in kernels if form in n and any(w in n for w in words)}
screens = (b"mla_batch_ring_kernel", b"mla_batch_stream_kernel")
probe, routes = objects(b"Lb1E", *screens), objects(b"Lb0E", *screens)
assert len(probe) == len(routes) == 1
assert routes == objects(b"", b"mla_route_kernel") and probe.isdisjoint(routes)
""")


# large appends share one pinned stage and its device copy
def test_memory_held_after_large_appends(runtime):
    run(runtime, r"""
rows = np.ones((9_000, 288), np.float32)
ids = np.arange(9_000, dtype=np.uint64) + 1000
size = 9_000 * (288 * 4 + 16)
with MlaNodeBank(np.ones((100, 288), np.float32), capacity=CAP) as bank:
    bank.append(rows[:10], ids[:10] + 20_000)  # the small updates' stages
    bank.evict(ids[:10] + 20_000)
    pinned, device = hip.fake_pinned(), hip.fake_device()
    for _ in range(2):
        bank.append(rows, ids)
        bank.append(rows, ids + 50_000)
        bank.evict(ids)
        bank.evict(ids + 50_000)
    assert hip.fake_pinned() - pinned <= size + 2 * 9_000 * 8
    assert hip.fake_device() - device <= size
    assert device_ids() == list(range(100))
""")
