"""The order in which threads that share a stream enqueue the launches of a call, with the HIP runtime's launch calls
replaced by ones that write down who called (no GPU)."""
import shutil
import subprocess
import sys

import pytest

# Stands in front of libamdhip64 in the symbol lookup of libbhi_hip.so: notes the calling thread, and lets others run.
RECORDER = r"""
#include <pthread.h>
#include <unistd.h>
static _Thread_local int who;
static int order[4096], n;
static pthread_mutex_t m = PTHREAD_MUTEX_INITIALIZER;
typedef struct { unsigned x, y, z; } dim3_t;
int __hipPushCallConfiguration(dim3_t g, dim3_t b, unsigned long s, void* st) { return 0; }
int __hipPopCallConfiguration(dim3_t* g, dim3_t* b, unsigned long* s, void** st) { return 0; }
int hipGetLastError(void) { return 0; }
int hipLaunchKernel(const void* f, dim3_t g, dim3_t b, void** a, unsigned long s, void* st) {
    pthread_mutex_lock(&m);
    if (n < 4096) order[n++] = who;
    pthread_mutex_unlock(&m);
    usleep(200);
    return 0;
}
void i_am(int w) { who = w; }
int launches(int* out) { for (int i = 0; i < n; ++i) out[i] = order[i]; return n; }
"""

CALLS = r"""
import ctypes, sys, threading
recorder = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
lib = ctypes.CDLL(sys.argv[2])
class Member(ctypes.Structure):
    _fields_ = [("A_rem", ctypes.c_void_p), ("A_exp", ctypes.c_void_p), ("exp_words", ctypes.c_int64), ("Y", ctypes.c_void_p),
                ("offsets", ctypes.c_void_p), ("table", ctypes.c_void_p), ("table_bytes", ctypes.c_int64), ("header", ctypes.c_void_p),
                ("bias", ctypes.c_void_p), ("M", ctypes.c_int32), ("reserved", ctypes.c_int32), ("residual", ctypes.c_void_p)]
at = 1 << 20                                   # an address that nothing reads: no kernel runs
def calls(who, name, table_bytes, rows):
    m = Member(at, at, 1 << 20, at, at, at, table_bytes, at, None, 256, 0, None)
    recorder.i_am(who)
    for _ in range(20):
        rc = getattr(lib, name)(ctypes.byref(m), ctypes.c_void_p(at), 1, 512, rows, ctypes.c_void_p(at), ctypes.c_int64(1 << 30), None)
        assert rc == 0, (name, rc)
threads = [threading.Thread(target=calls, args=a) for a in
           ((1, "bhi_wide_bf16_huffman", 8192, 40), (2, "bhi_wide_bf16_huffman", 8192, 200), (3, "bhi_wide_bf16_ans", 1024, 640))]
[t.start() for t in threads]
[t.join() for t in threads]
out = (ctypes.c_int * 4096)()
n = recorder.launches(out)
print(*out[:n])
"""


@pytest.mark.skipif(shutil.which("gcc") is None, reason="needs a C compiler")
def test_the_launches_of_a_wide_product_stay_together(tmp_path):
    """pack_x_kernel and wide_kernel hand X over in the stream's workspace: nobody else's launch may come in between."""
    from bf16_huffman_infer_amd import _lib
    source, recorder = tmp_path / "recorder.c", tmp_path / "recorder.so"
    source.write_text(RECORDER)
    subprocess.run(["gcc", "-O1", "-shared", "-fPIC", "-o", str(recorder), str(source), "-lpthread"], check=True)
    done = subprocess.run([sys.executable, "-c", CALLS, str(recorder), _lib.LIB_PATH], capture_output=True, text=True, timeout=120)
    assert done.returncode == 0, done.stderr
    order = [int(v) for v in done.stdout.split()]
    assert len(order) == 3 * 20 * 2 and set(order) == {1, 2, 3}, order
    assert order[0::2] == order[1::2], order
