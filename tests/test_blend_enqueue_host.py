"""What a blend enqueues, without a GPU: the library runs in a process of its own on a stand-in for the HIP
runtime that writes down every kernel launch instead of making it.

A blend of a frame of at most 8192 tiles is two launches, one that ranks the tiles into a table kept per
(device, stream) and one that reads it.  Whatever another thread enqueues on the stream, no launch may
write the table between the two."""
import json
import os
import subprocess
import sys

import pytest

from flashgs_amd import cabi

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

# The tile ranking is the launch of one workgroup of 1024 threads: (ranges, num_tiles, table).  A blend takes ranges
# first and the table as its 15th argument.  The launch that ranks takes its time, so that a thread that
# does not wait for it gets in.
RUNTIME = r"""
#include <pthread.h>
#include <stddef.h>
#include <stdlib.h>
#include <unistd.h>

typedef struct { unsigned x, y, z; } dim3;
typedef struct { int ranks; void *stream, *ranges, *table; } Launch;

static Launch launches[256];
static int count, capturing, no_memory;
static pthread_mutex_t lock = PTHREAD_MUTEX_INITIALIZER;
static __thread dim3 pushed_grid, pushed_block;
static __thread void *pushed_stream;

int hipGetDevice(int *device) { *device = 0; return 0; }
int hipDeviceGetAttribute(int *value, int attribute, int device) { (void)attribute; (void)device; *value = 256; return 0; }
int hipGetLastError(void) { return 0; }
int hipMalloc(void **p, size_t bytes) { *p = no_memory ? NULL : malloc(bytes); return *p ? 0 : 2; }
int hipGetSymbolAddress(void **p, const void *symbol) { *p = (void *)symbol; return 0; }
int hipStreamIsCapturing(void *stream, int *status) { (void)stream; *status = capturing; return 0; }

int __hipPushCallConfiguration(dim3 grid, dim3 block, size_t lds, void *stream)
{
    (void)lds;
    pushed_grid = grid; pushed_block = block; pushed_stream = stream;
    return 0;
}

int __hipPopCallConfiguration(dim3 *grid, dim3 *block, size_t *lds, void **stream)
{
    *grid = pushed_grid; *block = pushed_block; *lds = 0; *stream = pushed_stream;
    return 0;
}

int hipLaunchKernel(const void *function, dim3 grid, dim3 block, void **args, size_t lds, void *stream)
{
    (void)function; (void)lds;
    const int ranks = grid.x == 1 && block.x == 1024;
    pthread_mutex_lock(&lock);
    if (count < 256) {
        Launch *l = &launches[count++];
        l->ranks = ranks;
        l->stream = stream;
        l->ranges = *(void **)args[0];
        l->table = *(void **)args[ranks ? 2 : 14];
    }
    pthread_mutex_unlock(&lock);
    if (ranks) usleep(20000);
    return 0;
}

void stand_in_set(int is_capturing, int is_out_of_memory) { capturing = is_capturing; no_memory = is_out_of_memory; }
int stand_in_launches(Launch *out)
{
    pthread_mutex_lock(&lock);
    const int n = count;
    for (int i = 0; i < n; i++) out[i] = launches[i];
    count = 0;
    pthread_mutex_unlock(&lock);
    return n;
}
"""

PROGRAM = r"""
import ctypes as C, json, sys, threading

class Launch(C.Structure):
    _fields_ = [("ranks", C.c_int), ("stream", C.c_void_p), ("ranges", C.c_void_p), ("table", C.c_void_p)]

hip = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)         # in front of the runtime that the library links
lib = C.CDLL(sys.argv[2])
calls, capturing, no_memory = json.loads(sys.argv[3]), int(sys.argv[4]), int(sys.argv[5])
lib.fgs_blend.argtypes = [C.c_int] * 4 + [C.c_void_p] * 9
lib.fgs_last_error.restype = C.c_char_p
bg = (C.c_float * 3)()
start = threading.Barrier(len(calls))
status = []

def blends(bx, by, w, h, ranges, stream, times):
    start.wait()
    for _ in range(times):
        status.append(lib.fgs_blend(bx, by, w, h, 256, 256, 256, 256, ranges, C.addressof(bg), 256, None, stream))

hip.stand_in_set(capturing, no_memory)
threads = [threading.Thread(target=blends, args=c) for c in calls]
for t in threads: t.start()
for t in threads: t.join()
found = (Launch * 256)()
n = hip.stand_in_launches(found)
print(json.dumps({"status": status, "launches": [[f.ranks, f.stream, f.ranges, f.table] for f in found[:n]]}))
"""


@pytest.fixture(scope="module")
def runtime(tmp_path_factory):
    where = tmp_path_factory.mktemp("runtime")
    source, library = where / "runtime.c", where / "libruntime.so"
    source.write_text(RUNTIME)
    subprocess.check_call(["gcc", "-O1", "-shared", "-fPIC", "-pthread", str(source), "-o", str(library)])
    return str(library)


def enqueued(runtime, calls, capturing=False, no_memory=False):
    """Launches [ranks, stream, ranges, table] of threads that each blend (bx, by, width, height, ranges, stream, times)."""
    done = subprocess.run([sys.executable, "-c", PROGRAM, runtime, cabi.LIB_PATH, json.dumps(calls), str(int(capturing)),
                           str(int(no_memory))], capture_output=True, text=True, timeout=120, cwd=ROOT)
    assert done.returncode == 0, done.stderr[-2000:]
    found = json.loads(done.stdout.splitlines()[-1])
    assert found["status"] == [0] * sum(c[-1] for c in calls)
    return found["launches"]


@pytest.mark.parametrize("block", [(16, 16), (32, 16), (32, 32)])
def test_threads_that_blend_on_one_stream_read_their_own_ranking(runtime, block):
    calls = [[*block, 640, 360, 0x10000, 0x70, 4], [*block, 1000, 700, 0x20000, 0x70, 4], [*block, 320, 200, 0x30000, 0x70, 4]]
    launches = enqueued(runtime, calls)
    assert len(launches) == 24
    ranked = {}                     # table -> whose lists it ranks
    for ranks, _, ranges, table in launches:
        assert table
        if ranks:
            ranked[table] = ranges
        else:
            assert ranked[table] == ranges, "a blend reads the ranking of another thread's lists"


@pytest.mark.parametrize("block", [(16, 16), (32, 32)])
def test_blends_on_different_streams_have_tables_of_their_own(runtime, block):
    launches = enqueued(runtime, [[*block, 640, 360, 0x10000, 0x70, 2], [*block, 640, 360, 0x20000, 0x80, 2]])
    tables = {stream: {t for _, s, _, t in launches if s == stream} for stream in (0x70, 0x80)}
    assert len(launches) == 8 and all(len(t) == 1 for t in tables.values()) and tables[0x70] != tables[0x80]


@pytest.mark.parametrize("block", [(16, 16), (32, 16), (32, 32)])
def test_captured_blends_hold_no_table(runtime, block):
    launches = enqueued(runtime, [[*block, 640, 360, 0x10000, 0x70, 2]], capturing=True)
    assert launches == [[0, 0x70, 0x10000, None]] * 2


@pytest.mark.parametrize("block", [(16, 16), (32, 16), (32, 32)])
def test_blends_without_memory_for_a_table_go_unranked(runtime, block):
    launches = enqueued(runtime, [[*block, 640, 360, 0x10000, 0x70, 2]], no_memory=True)
    assert launches == [[0, 0x70, 0x10000, None]] * 2
