"""The library's per-stream scratch (scratch_get, nelisp-gpu_amd/csrc/
nlg_runtime.hip) against a stand-in for the few HIP calls that it makes, in a
process of its own and without a GPU: an allocation that is refused leaves no
error behind, which the next launch check would report as its own, and one made
while another stream is being captured asks for the relaxed mode; the per-thread
stream's handle names another stream, and so another scratch, in every thread."""
import os
import subprocess
import sys
import tempfile

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

FAKE = r'''
#include <stdlib.h>
typedef int hipError_t;
int refuse, last;                      /* the thread's last error */
static hipError_t ret(int e) { if (e) last = e; return e; }
int mode;                              /* of the thread: 0 global, 2 relaxed */
hipError_t hipThreadExchangeStreamCaptureMode(int *m) { int o = mode; mode = *m; *m = o; return ret(0); }
hipError_t hipMalloc(void **p, size_t n) {
  if (mode != 2) return ret(900);      /* another stream is being captured */
  if (refuse) return ret(2);           /* hipErrorOutOfMemory */
  *p = malloc(n);
  return ret(0);
}
hipError_t hipFree(void *p) { free(p); return ret(0); }
hipError_t hipMemsetAsync(void *p, int v, size_t n, void *st) { return ret(0); }
hipError_t hipGetLastError(void) { int e = last; last = 0; return e; }
hipError_t hipStreamIsCapturing(void *st, int *status) { *status = 0; return ret(0); }
'''

PROGRAM = r'''
import ctypes as C, sys
fake = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)  # found before libamdhip64's
lib = C.CDLL(sys.argv[2])
get, get_try = lib._Z11nlg_scratchmP12ihipStream_t, lib._Z15nlg_scratch_trymP12ihipStream_ti
get.restype = get_try.restype = C.c_void_p
get.argtypes, get_try.argtypes = [C.c_size_t, C.c_void_p], [C.c_size_t, C.c_void_p, C.c_int]
refuse, last = C.c_int.in_dll(fake, "refuse"), C.c_int.in_dll(fake, "last")
for slot in (1, 2, 3):
    refuse.value = 1
    assert get_try(5 << 20, 0x1000, slot) is None
    assert last.value == 0, (slot, last.value)
    refuse.value = 0
    p = get_try(5 << 20, 0x1000, slot)
    assert p and get_try(1 << 20, 0x1000, slot) == p  # kept, per stream and slot
    assert get_try(1 << 20, 0x2000, slot) not in (None, p)
import threading  # hipStreamPerThread (2) is another stream in every thread
mine, other = get_try(1 << 20, 2, 3), []
t = threading.Thread(target=lambda: other.extend(get_try(1 << 20, 2, 3) for _ in range(2)))
t.start()
t.join()
assert mine and other[0] and other[0] == other[1] != mine == get_try(1 << 20, 2, 3)
refuse.value = 1
assert get(5 << 20, 0x1000) is None and last.value == 0
lib.nlg_last_error.restype = C.c_char_p
assert C.c_int.in_dll(fake, "mode").value == 0  # given back
assert b"hipMalloc" in lib.nlg_last_error()
print("ok")
'''


def test_a_refused_scratch_leaves_no_error():
    lib = os.path.join(ROOT, "nelisp-gpu_amd", "lib", "libnlgpu.so")
    with tempfile.TemporaryDirectory() as t:
        src, so = os.path.join(t, "fake.c"), os.path.join(t, "libfake.so")
        with open(src, "w") as f:
            f.write(FAKE)
        subprocess.run(["gcc", "-shared", "-fPIC", "-O1", src, "-o", so], check=True)
        r = subprocess.run([sys.executable, "-c", PROGRAM, so, lib], capture_output=True, text=True)
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stdout + r.stderr
