"""What fgs_sort_render enqueues, without a GPU: the library runs in a process of its own on a stand-in for the HIP runtime that
writes down every kernel launch, by the kernel's name, instead of making it.

The ranking of a small frame's tiles and the long lists of a large one are written by launches of the sort, into tables kept per
(device, stream), and read by the blend of the same call."""
import json
import os
import subprocess
import sys

import pytest

from flashgs_amd import cabi

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

# Of every kernel that writes or reads a table: the argument that holds its ranges, the one that holds the table and where in that argument
# (a pointer's number) it stands.  A launch that writes a table takes its time, so that a thread that does not wait for it gets in.
RUNTIME = r"""
#include <pthread.h>
#include <stddef.h>
#include <stdlib.h>
#include <string.h>
#include <unistd.h>

typedef struct { unsigned x, y, z; } dim3;
typedef struct { int kind; size_t stream, ranges, table, next; } Launch;
enum { kRanks = 1, kLists = 2, kBlends = 3 };

static struct { const void *function; char name[160]; } kernels[512];
static Launch launches[1024];
static int kernel_count, launched[512], count, capturing, no_memory, failing, asked;
static pthread_mutex_t lock = PTHREAD_MUTEX_INITIALIZER;
static __thread dim3 pushed_grid, pushed_block;
static __thread void *pushed_stream;

void **__hipRegisterFatBinary(const void *data) { static void *module; (void)data; return &module; }
void __hipUnregisterFatBinary(void **module) { (void)module; }
void __hipRegisterVar(void **m, void *v, char *h, char *d, int e, size_t s, int c, int g) { (void)m; (void)v; (void)h; (void)d; (void)e; (void)s; (void)c; (void)g; }
void __hipRegisterFunction(void **module, const void *function, char *host, const char *name, unsigned limit, void *tid, void *bid, dim3 *block, dim3 *grid, int *size)
{
    (void)module; (void)host; (void)limit; (void)tid; (void)bid; (void)block; (void)grid; (void)size;
    if (kernel_count < 512) {
        kernels[kernel_count].function = function;
        strncpy(kernels[kernel_count++].name, name, 159);
    }
}

int hipGetDevice(int *device) { asked++; *device = 0; return 0; }
int hipDeviceGetAttribute(int *value, int attribute, int device) { (void)attribute; (void)device; asked++; *value = 256; return 0; }
int hipGetLastError(void) { const int failed = failing; failing = 0; return failed; }
const char *hipGetErrorString(int error) { (void)error; return "made to fail"; }
int hipMalloc(void **p, size_t bytes) { asked++; *p = no_memory ? NULL : malloc(bytes); return *p ? 0 : 2; }
int hipGetSymbolAddress(void **p, const void *symbol) { *p = (void *)symbol; return 0; }
int hipStreamIsCapturing(void *stream, int *status) { (void)stream; asked++; *status = capturing; return 0; }
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
    (void)grid; (void)block; (void)lds;
    const char *name = "";
    if (failing) return 1;
    for (int i = 0; i < kernel_count; i++) {
        if (kernels[i].function != function) continue;
        name = kernels[i].name;
        __sync_fetch_and_add(&launched[i], 1);
    }
    Launch l = { 0, (size_t)stream, 0, 0, 0 };
    if (strstr(name, "tile_scatter_kernel")) {                  /* (TileRanking) */
        l.kind = kRanks; l.table = *(size_t *)args[9];
    } else if (strstr(name, "segment_sort_general_kernel")) {   /* (TileRanking) */
        l.kind = kRanks; l.table = *(size_t *)args[15];
    } else if (strstr(name, "tile_order_kernel")) {
        l.kind = kRanks; l.ranges = *(size_t *)args[0]; l.table = *(size_t *)args[2];
    } else if (strstr(name, "segment_sort_wave_kernel")) {      /* (TileNotes) */
        l.kind = kLists; l.ranges = ((size_t *)args[16])[0]; l.table = ((size_t *)args[16])[1];
    } else if (strstr(name, "tile_ranges_sampled_kernel")) {
        l.kind = kLists; l.ranges = *(size_t *)args[2]; l.table = *(size_t *)args[4];
    } else if (strstr(name, "blend_kernel")) {
        l.kind = kBlends; l.ranges = *(size_t *)args[0]; l.table = *(size_t *)args[14];
        if (!strstr(name, "shared")) l.next = *(size_t *)args[15];
    }
    if (l.kind && (l.table || l.kind == kBlends)) {
        pthread_mutex_lock(&lock);
        if (count < 1024) launches[count++] = l;
        pthread_mutex_unlock(&lock);
        if (l.kind != kBlends) usleep(20000);
    }
    return 0;
}

void stand_in_set(int is_capturing, int is_out_of_memory) { capturing = is_capturing; no_memory = is_out_of_memory; }
void stand_in_fail(void) { failing = 1; }
int stand_in_asked(void) { const int n = asked; asked = 0; return n; }
int stand_in_launches_of(const char *part)
{
    int n = 0;
    for (int i = 0; i < kernel_count; i++) if (strstr(kernels[i].name, part)) n += launched[i];
    return n;
}
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
    _fields_ = [("kind", C.c_int)] + [(n, C.c_size_t) for n in ("stream", "ranges", "table", "next")]

hip = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)         # in front of the runtime that the library links
lib = C.CDLL(sys.argv[2])
threads_of, capturing, no_memory = json.loads(sys.argv[3]), int(sys.argv[4]), int(sys.argv[5])
lib.fgs_sort_render.argtypes = [C.c_int] * 5 + [C.c_void_p, C.c_size_t] + [C.c_void_p] * 11 + [C.c_int, C.c_void_p]
lib.fgs_sort_gaussian.argtypes = [C.c_int] * 5 + [C.c_void_p, C.c_size_t] + [C.c_void_p] * 5
lib.fgs_render_f32.argtypes = [C.c_int] * 5 + [C.c_void_p] * 10
lib.fgs_get_sort_buffer_size.restype = C.c_size_t
lib.fgs_last_error.restype = C.c_char_p
bg = (C.c_float * 3)()
start = threading.Barrier(len(threads_of))
results = [[] for _ in threads_of]

def frames(mine, calls):
    start.wait()
    for how, bx, by, w, h, pairs, ranges, stream in calls:
        hip.stand_in_asked()
        room = lib.fgs_get_sort_buffer_size(pairs)
        if how.endswith("fails"): hip.stand_in_fail()             # up to the first time that the library looks
        if how == "sort":
            rc = lib.fgs_sort_gaussian(pairs, w, h, bx, by, 256, room, 256, 256, 256, 256, stream)
        elif how.startswith("render"):
            rc = lib.fgs_render_f32(bx, by, pairs, w, h, 256, 256, 256, 256 + 4 * (how == "render misaligned keys"), 256, ranges, C.addressof(bg),
                                    None if how == "render without image" else 256, None, stream)
        else:
            space = {"misaligned": 256 + 8, "no space": None}.get(how, 256)
            rc = lib.fgs_sort_render(bx, by, pairs, w, h, space, room - (how == "short of room"), 256, 256, None if how == "no keys" else 256, 256,
                                     256, 256, 256, ranges, C.addressof(bg), 256, None, 0, stream)
        results[mine].append([rc, hip.stand_in_asked() if len(threads_of) == 1 else None])

hip.stand_in_set(capturing, no_memory)
threads = [threading.Thread(target=frames, args=c) for c in enumerate(threads_of)]
for t in threads: t.start()
for t in threads: t.join()
found = (Launch * 1024)()
n = hip.stand_in_launches(found)
noting, plain = (hip.stand_in_launches_of(b"segment_sort_wave_kernelILi16ELb1ELb%dEE" % notes) for notes in (1, 0))
print(json.dumps({"noting": noting, "plain": plain, "results": results, "launches": [{f: getattr(l, f) for f, _ in Launch._fields_} for l in found[:n]]}))
"""

RANKS, LISTS, BLENDS = 1, 2, 3
LONG = [16, 16, 7680, 4320, 14_000_000]                 # a frame that lists its long lists
A, B = 0x10000, 0x20000                                 # addresses of ranges
REFUSED = {"short of room": cabi.FGS_E_WORKSPACE, "misaligned": cabi.FGS_E_INVALID, "no space": cabi.FGS_E_INVALID, "no keys": cabi.FGS_E_INVALID}


@pytest.fixture(scope="module")
def runtime(tmp_path_factory):
    where = tmp_path_factory.mktemp("runtime")
    source, library = where / "runtime.c", where / "libruntime.so"
    source.write_text(RUNTIME)
    subprocess.check_call(["gcc", "-O1", "-shared", "-fPIC", "-pthread", str(source), "-o", str(library)])
    return str(library)


def enqueued(runtime, threads, capturing=False, no_memory=False, count_segments=False):
    """(status and calls of the runtime, but for launches, of every frame; launches that write or read a table) of threads
    that each make frames (how, bx, by, width, height, pairs, ranges, stream).  count_segments: how often the first segment launch was the one
    that writes ranges and lists, and how often the one that does not."""
    done = subprocess.run([sys.executable, "-c", PROGRAM, runtime, cabi.LIB_PATH, json.dumps(threads), str(int(capturing)),
                           str(int(no_memory))], capture_output=True, text=True, timeout=120, cwd=ROOT)
    assert done.returncode == 0, done.stderr[-2000:]
    found = json.loads(done.stdout.splitlines()[-1])
    if count_segments:
        return found["noting"], found["plain"]
    return found["results"], found["launches"]


def check_turns(launches):
    """Every launch that lists finds the table that it lists in cleared by the blend in front of it, and the blend behind it reads that one."""
    cleared, listed = None, None
    for l in launches:
        if l["kind"] == LISTS:
            assert cleared is None or l["table"] == cleared, "the table still holds the lists of an earlier frame"
            listed = l
        elif l["kind"] == BLENDS:
            assert listed and l["table"] == listed["table"] and l["ranges"] == listed["ranges"], "a blend reads the lists of another frame"
            assert l["next"] and l["next"] != l["table"]
            cleared, listed = l["next"], None


@pytest.mark.parametrize("how", sorted(REFUSED))
@pytest.mark.parametrize("frame", [[16, 16, 1280, 720, 200_000], LONG])
def test_a_refused_call_asks_the_runtime_for_nothing(runtime, how, frame):
    """... and uses up no turn of the tables of long lists: the next frame's is the one that the last blend cleared."""
    calls = [["sort_render", *frame, A, 0x70], [how, *frame, A, 0x70], ["sort_render", *frame, A, 0x70], [how, *frame, A, 0x70],
             ["render", *frame, A, 0x70]]
    results, launches = enqueued(runtime, [calls])
    assert [r for r, _ in results[0]] == [0, REFUSED[how], 0, REFUSED[how], 0]
    assert [asked for _, asked in results[0]][1::2] == [0, 0]
    if frame is LONG:
        assert [l["kind"] for l in launches] == [LISTS, BLENDS] * 3
        check_turns(launches)


@pytest.mark.parametrize("how, code", [("render without image", cabi.FGS_E_INVALID), ("render misaligned keys", cabi.FGS_E_INVALID),
                                       ("render fails", cabi.FGS_E_HIP), ("sort_render fails", cabi.FGS_E_HIP)])
def test_a_frame_without_a_blend_uses_up_no_turn(runtime, how, code):
    """Refused, or ended by an error before its blend: nothing of it is enqueued, and the next frame lists in the table that was cleared last."""
    calls = [["sort_render", *LONG, A, 0x70], [how, *LONG, B, 0x70], ["render", *LONG, A, 0x70], [how, *LONG, B, 0x70], ["sort_render", *LONG, A, 0x70]]
    results, launches = enqueued(runtime, [calls])
    assert [r for r, _ in results[0]] == [0, code, 0, code, 0]
    assert [l["kind"] for l in launches] == [LISTS, BLENDS] * 3
    check_turns(launches)


RANKED = [16, 16, 1920, 1080]                           # ranked: by the scatter, by the last launch of the sort, or by a launch of its own
PAIRS = {"by the scatter": 200_000, "by the last launch": 5_000_000, "by itself": 1000}


def check_tables(launches):
    """The last launch that wrote a blend's table belongs to the blend's own frame.  Frames of one thread have one address of ranges; a ranking that
    the sort makes knows none, but a frame's launches stand together."""
    ranked = {}
    for l in launches:
        if l["kind"] == RANKS:
            assert l["table"] not in ranked, "another frame's ranking between a ranking and the blend that reads it"
            ranked[l["table"]] = l["ranges"]
        else:
            assert l["kind"] == BLENDS and l["table"] in ranked
            assert ranked.pop(l["table"]) in (0, l["ranges"])
    assert not ranked


@pytest.mark.parametrize("first", sorted(PAIRS))
@pytest.mark.parametrize("second", sorted(PAIRS) + ["render"])
def test_threads_that_sort_and_render_on_one_stream_read_their_own_ranking(runtime, first, second):
    one = [["sort_render", *RANKED, PAIRS[first], A, 0x70]] * 4
    other = [["render", *RANKED, 200_000, B, 0x70] if second == "render" else ["sort_render", *RANKED, PAIRS[second], B, 0x70]] * 4
    results, launches = enqueued(runtime, [one, other])
    assert not any(rc for thread in results for rc, _ in thread)
    assert len(launches) == 16
    check_tables(launches)


@pytest.mark.parametrize("other", ["sort_render", "render"])
def test_threads_that_sort_and_render_on_one_stream_read_their_own_long_lists(runtime, other):
    results, launches = enqueued(runtime, [[["sort_render", *LONG, A, 0x70]] * 6, [[other, *LONG, B, 0x70]] * 6])
    assert not any(rc for thread in results for rc, _ in thread)
    assert len(launches) == 24 and len({l["table"] for l in launches}) == 2
    check_turns(launches)


def test_frames_on_different_streams_have_tables_of_their_own(runtime):
    calls = [[["sort_render", *frame, ranges, stream]] * 3 for stream, ranges in ((0x70, A), (0x80, B)) for frame in (LONG, [*RANKED, 200_000])]
    results, launches = enqueued(runtime, calls)
    assert not any(rc for thread in results for rc, _ in thread)
    tables = {s: {l["table"] for l in launches if l["stream"] == s} for s in (0x70, 0x80)}
    assert len(launches) == 24 and all(len(t) == 3 for t in tables.values()) and not tables[0x70] & tables[0x80]


@pytest.mark.parametrize("why", ["capturing", "no_memory"])
@pytest.mark.parametrize("frame", [LONG] + [[*RANKED, pairs] for pairs in PAIRS.values()])
def test_no_table_under_capture_or_without_memory(runtime, why, frame):
    results, launches = enqueued(runtime, [[["sort_render", *frame, A, 0x70]] * 2], **{why: True})
    assert not any(rc for rc, _ in results[0])
    assert [l["kind"] for l in launches] == [BLENDS] * 2 and not any(l["table"] or l["next"] for l in launches)


@pytest.mark.parametrize("frame", [LONG, [16, 16, 1920, 1080, 200_000], [16, 16, 7680, 4320, 100_000]])
def test_a_sort_by_itself_does_not_pay_for_the_ranges(runtime, frame):
    """... and the call that needs them has the launch that writes them."""
    assert enqueued(runtime, [[["sort", *frame, A, 0x70]] * 3 + [["sort_render", *frame, A, 0x70]] * 2], count_segments=True) == (2, 3)
