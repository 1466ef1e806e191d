"""Which launches take part in starting the long lists of a large frame first, without a GPU: the library runs in a process
of its own on a stand-in for the HIP runtime that writes down every kernel launch instead of making it.

From 65536 tiles and 3 * 2^20 pairs on, fgs_render's launch that marks the tile ranges lists the tiles whose lists are long in a
table kept per (device, stream), which the blend behind it reads."""
import json
import os
import subprocess
import sys

import pytest

from flashgs_amd import cabi

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

# tile_ranges_sampled_kernel has the table as its fifth argument, blend_kernel the table as its 15th and the one of the next frame as its 16th.
# The launch that marks ranges takes its time, so that a thread that does not wait for it gets in.
RUNTIME = r"""
#include <pthread.h>
#include <stddef.h>
#include <stdlib.h>
#include <unistd.h>

typedef struct { unsigned x, y, z; } dim3;
typedef struct { size_t function, stream, ranges, table, next, groups; int marks; } Launch;

static Launch launches[256];
static int count, capturing, no_memory;
static pthread_mutex_t lock = PTHREAD_MUTEX_INITIALIZER;
static __thread dim3 pushed_grid, pushed_block;
static __thread void *pushed_stream;

int hipGetDevice(int *device) { *device = 0; return 0; }
int hipDeviceGetAttribute(int *value, int attribute, int device) { (void)attribute; (void)device; *value = 256; return 0; }
int hipGetLastError(void) { return 0; }
int hipMalloc(void **p, size_t bytes) { *p = no_memory ? NULL : malloc(bytes); return *p ? 0 : 2; }
int hipStreamIsCapturing(void *stream, int *status) { (void)stream; *status = capturing; return 0; }
int hipThreadExchangeStreamCaptureMode(int *mode) { (void)mode; return 0; }

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
    (void)block; (void)lds;
    const int marks = *(int *)args[0] >= 1000000;       /* the pair count; a blend has the ranges there, below that here */
    pthread_mutex_lock(&lock);
    if (count < 256) {
        Launch *l = &launches[count++];
        l->function = (size_t)function;
        l->stream = (size_t)stream;
        l->marks = marks;
        l->ranges = *(size_t *)args[marks ? 2 : 0];
        l->table = *(size_t *)args[marks ? 4 : 14];
        l->next = marks ? 0 : *(size_t *)args[15];
        l->groups = grid.x;
    }
    pthread_mutex_unlock(&lock);
    if (marks) usleep(20000);
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
    _fields_ = [(n, C.c_size_t) for n in ("function", "stream", "ranges", "table", "next", "groups")] + [("marks", C.c_int)]

hip = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)         # in front of the runtime that the library links
lib = C.CDLL(sys.argv[2])
calls, capturing, no_memory = json.loads(sys.argv[3]), int(sys.argv[4]), int(sys.argv[5])
lib.fgs_render_f32.argtypes = [C.c_int] * 5 + [C.c_void_p] * 10
lib.fgs_tile_ranges.argtypes = [C.c_int] * 5 + [C.c_void_p] * 3
lib.fgs_blend.argtypes = [C.c_int] * 4 + [C.c_void_p] * 9
bg = (C.c_float * 3)()
start = threading.Barrier(len(calls))
status = []

def frames(how, bx, by, w, h, pairs, ranges, stream, times):
    start.wait()
    for _ in range(times):
        if how == "render":
            status.append(lib.fgs_render_f32(bx, by, pairs, w, h, 256, 256, 256, 256, 256, ranges, C.addressof(bg), 256, None, stream))
        else:
            status.append(lib.fgs_tile_ranges(bx, by, pairs, w, h, 256, ranges, stream))
            status.append(lib.fgs_blend(bx, by, w, h, 256, 256, 256, 256, ranges, C.addressof(bg), 256, None, stream))

hip.stand_in_set(capturing, no_memory)
threads = [threading.Thread(target=frames, args=c) for c in calls]
for t in threads: t.start()
for t in threads: t.join()
found = (Launch * 256)()
n = hip.stand_in_launches(found)
print(json.dumps({"status": status, "launches": [{f: getattr(l, f) for f, _ in Launch._fields_} for l in found[:n]]}))
"""

FRAME = [16, 16, 7680, 4320, 14_000_000]                # a frame that lists: a seventh of a SIMD's entries is 1953
A, B = 0x10000, 0x20000                                 # addresses of ranges


@pytest.fixture(scope="module")
def runtime(tmp_path_factory):
    where = tmp_path_factory.mktemp("runtime")
    source, library = where / "runtime.c", where / "libruntime.so"
    source.write_text(RUNTIME)
    subprocess.check_call(["gcc", "-O1", "-shared", "-fPIC", "-pthread", str(source), "-o", str(library)])
    return str(library)


def enqueued(runtime, calls, capturing=False, no_memory=False):
    """Launches of threads that each make frames (how, bx, by, width, height, pairs, ranges, stream, times)."""
    done = subprocess.run([sys.executable, "-c", PROGRAM, runtime, cabi.LIB_PATH, json.dumps(calls), str(int(capturing)),
                           str(int(no_memory))], capture_output=True, text=True, timeout=120, cwd=ROOT)
    assert done.returncode == 0, done.stderr[-2000:]
    found = json.loads(done.stdout.splitlines()[-1])
    assert not any(found["status"])
    return found["launches"]


def test_only_frames_that_list_pay_for_the_listing(runtime):
    """Frames of fewer tiles, of fewer pairs, of so many that no list is long for it, and the operators one by one: the launch that marks their
    ranges is one that knows no table, and their blend has no workgroups in front."""
    listing = enqueued(runtime, [["render", *FRAME, A, 0x70, 1]])
    assert [l["marks"] for l in listing] == [1, 0]
    assert listing[0]["table"] and listing[0]["table"] == listing[1]["table"]
    plain = enqueued(runtime, [["operators", *FRAME, A, 0x70, 1]])
    distance = lambda launches: launches[0]["function"] - launches[1]["function"]       # of the two kernels, wherever the library was loaded
    assert not any(l["table"] for l in plain) and distance(plain) != distance(listing)
    assert listing[1]["groups"] == plain[1]["groups"] + 512
    for frame in ([16, 16, 3840, 2160, 8_000_000], [16, 16, 7680, 4320, 110_000_000]):
        render = enqueued(runtime, [["render", *frame, A, 0x70, 1]])
        assert not any(l["table"] for l in render) and distance(render) == distance(plain)


def test_threads_that_render_on_one_stream_read_the_lists_of_their_own_frame(runtime):
    launches = enqueued(runtime, [["render", *FRAME, A, 0x70, 6], ["render", *FRAME, B, 0x70, 6]])
    assert len(launches) == 24
    listed, cleared = {}, set()
    for i, l in enumerate(launches):
        if l["marks"]:
            assert i == 0 or l["table"] in cleared, "the table of a frame was cleared by the blend of the one before"
            listed[l["table"]] = l["ranges"]
        else:
            assert listed[l["table"]] == l["ranges"], "a blend reads the lists of another thread's frame"
            assert l["next"] != l["table"]
            cleared = {l["next"]}
    assert len(listed) == 2


def test_renders_on_different_streams_have_tables_of_their_own(runtime):
    launches = enqueued(runtime, [["render", *FRAME, A, 0x70, 3], ["render", *FRAME, B, 0x80, 3]])
    tables = {s: {l["table"] for l in launches if l["stream"] == s} for s in (0x70, 0x80)}
    assert len(launches) == 12 and all(len(t) == 2 for t in tables.values()) and not tables[0x70] & tables[0x80]


@pytest.mark.parametrize("why", ["capturing", "no_memory"])
@pytest.mark.parametrize("block", [(16, 16), (32, 16), (32, 32)])
def test_no_table_under_capture_or_without_memory(runtime, why, block):
    launches = enqueued(runtime, [["render", *block, 16384, 8192, 14_000_000, A, 0x70, 2]], **{why: True})
    assert [l["marks"] for l in launches] == [1, 0] * 2 and not any(l["table"] or l["next"] for l in launches)
