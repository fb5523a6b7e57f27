"""The backend's workspace (hipb_gemm_ws) against a device allocator of the
test's own: what it grows to, frees, keeps for graphs and does without."""
import ctypes
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")
MIB = 1 << 20

# Takes the place of the runtime's calls inside the library built here.
STUB = r"""
#include <hip/hip_runtime_api.h>
size_t stub_free = 0;            /* bytes left */
int stub_mallocs, stub_frees, stub_syncs, stub_capturing;
static size_t size[64];
static char at[64];
hipError_t hipMalloc(void **p, size_t n)
{
    stub_mallocs++;
    if (n > stub_free)
        return hipErrorOutOfMemory;
    for (int i = 0; i < 64; i++)
        if (!size[i]) {
            size[i] = n;
            stub_free -= n;
            *p = at + i;
            return hipSuccess;
        }
    return hipErrorOutOfMemory;
}
hipError_t hipFree(void *p)
{
    stub_frees++;
    stub_free += size[(char *)p - at];
    size[(char *)p - at] = 0;
    return hipSuccess;
}
hipError_t hipGetLastError(void) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t s) { stub_syncs++; return hipSuccess; }
hipError_t hipStreamIsCapturing(hipStream_t s, hipStreamCaptureStatus *st)
{
    *st = stub_capturing ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
    return hipSuccess;
}
"""


@pytest.fixture(scope="module")
def so(tmp_path_factory):
    d = tmp_path_factory.mktemp("ws")
    (d / "stub.c").write_text(STUB)
    pkg = os.path.join(ROOT, "i.sam3.opencl_amd")
    if not os.path.isdir(os.path.join(pkg, "_obj")):
        pytest.skip("no object files (build.py leaves them beside the library)")
    objs = [os.path.join(pkg, "_obj", f) for f in sorted(os.listdir(os.path.join(pkg, "_obj")))
            if f.endswith(".o") and f != "hip_backend.o"]
    subprocess.run(["gcc", "-shared", "-fPIC", "-O1", "-std=gnu11", "-w", "-Wl,-Bsymbolic",
                    "-D__HIP_PLATFORM_AMD__", "-I" + os.path.join(ROOT, "include"),
                    "-I" + os.path.join(pkg, "csrc"), "-I" + os.path.join(ROCM, "include"),
                    os.path.join(pkg, "csrc", "hip_backend.c"), str(d / "stub.c"), "-o",
                    str(d / "ws.so")] + objs +
                   ["-L" + os.path.join(ROCM, "lib"), "-lamdhip64", "-lpthread", "-lm",
                    "-lstdc++", "-Wl,-rpath," + os.path.join(ROCM, "lib")], check=True)
    lib = ctypes.CDLL(str(d / "ws.so"))
    lib.hipb_gemm_ws.restype = ctypes.c_void_p
    lib.hipb_gemm_ws.argtypes = [ctypes.c_void_p, ctypes.c_size_t]
    return lib


class Ws:
    def __init__(self, so, free):
        import sam3_hip
        self.so, self.b = so, sam3_hip.HipbBackend()
        for n in ("mallocs", "frees", "syncs", "capturing"):
            setattr(self, n, ctypes.c_int.in_dll(so, "stub_" + n))
            getattr(self, n).value = 0
        self.free = ctypes.c_size_t.in_dll(so, "stub_free")
        self.free.value = free

    def get(self, n):
        return self.so.hipb_gemm_ws(ctypes.byref(self.b), n)


def test_grows_and_frees(so):
    """Twice the size at each growth; the outgrown block goes back after the
    stream is done with it."""
    w = Ws(so, 1 << 40)
    p = w.get(MIB)
    assert p and w.b.gemm_ws_bytes == 32 * MIB
    assert w.get(32 * MIB) == p and w.mallocs.value == 1
    assert w.get(33 * MIB) and w.b.gemm_ws_bytes == 64 * MIB
    assert w.b.gemm_ws_count == 1 and w.frees.value == 1 and w.syncs.value == 1
    assert w.get(500 * MIB) and w.b.gemm_ws_bytes == 500 * MIB
    assert w.free.value == (1 << 40) - 500 * MIB
    assert w.get(0) is None and w.get((8 << 30) + 1) is None
    assert w.get(7 << 30) and w.b.gemm_ws_bytes == 7 << 30
    assert w.get(8 << 30) and w.b.gemm_ws_bytes == 8 << 30   # not twice
    w.so.hipFree(ctypes.c_void_p(w.b.gemm_ws[0]))


def test_graphs_keep_theirs(so):
    """A workspace that a graph of the library was captured with outlives its
    growth; a capture neither grows it nor, when it is the caller's, gets it."""
    w = Ws(so, 1 << 40)
    p = w.get(40 * MIB)
    w.b.capture = 1
    assert w.get(10 * MIB) == p and w.get(41 * MIB) is None
    w.b.capture = 0
    w.capturing.value = 1
    assert w.get(10 * MIB) is None
    w.capturing.value = 0
    q = w.get(50 * MIB)
    assert q != p and w.b.gemm_ws_count == 2 and w.frees.value == 0
    r = w.get(200 * MIB)   # no graph holds q
    assert r and w.b.gemm_ws_count == 2 and w.frees.value == 1
    assert w.b.gemm_ws[0] == p
    for i in range(2):
        w.so.hipFree(ctypes.c_void_p(w.b.gemm_ws[i]))


def test_short_of_memory(so):
    """What is asked for where its double cannot be had, nothing where that
    cannot either, and no allocation on each of the calls that follow."""
    w = Ws(so, 100 * MIB)
    assert w.get(40 * MIB) and w.b.gemm_ws_bytes == 40 * MIB
    w.b.gemm_ws_held = 1
    assert w.get(50 * MIB) and w.b.gemm_ws_bytes == 50 * MIB   # 80 do not fit beside 40
    n = w.mallocs.value
    assert w.get(70 * MIB) is None and w.mallocs.value == n + 2
    for _ in range(20):
        assert w.get(70 * MIB) is None
    assert w.mallocs.value == n + 2
    w.free.value += 1 << 30
    got = [w.get(70 * MIB) for _ in range(64)]
    assert got[-1] and w.mallocs.value == n + 3
