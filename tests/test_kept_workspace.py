"""The workspace bd_cholesky keeps between calls, on the host: bd_potrf.hip is
compiled for the CPU and linked to a stand-in for the HIP runtime whose device
memory is a table of address ranges.  The stand-in hands the first free
addresses out again, as a device does, numbers its allocations, and can lose
all of them at once (hipDeviceReset).  Its launchers note whether the factor's
workspace is memory that the library holds."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "brownian_dynamics_cuda_amd", "csrc")
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"

FAKE = r"""
#include <hip/hip_runtime.h>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include "bd_hip.h"
#include "bd_kernels.h"

namespace {
struct Range { size_t bytes; unsigned long long id; bool ours; };
std::map<size_t, Range> live;
unsigned long long ids = 0;
size_t room = (size_t)1 << 40;  // largest allocation that succeeds
bool library = true;            // who allocates
hipError_t last = hipSuccess;
hipError_t err(hipError_t e) { if (e != hipSuccess) last = e; return e; }
hipStream_t capturing = nullptr;  // the stream under capture: no allocation, no wait meanwhile
int launches = 0, dead_used = 0, foreign_used = 0, foreign_freed = 0, dead_freed = 0;
}  // namespace

extern "C" {
hipError_t hipMalloc(void **p, size_t n) {
    if (capturing) return err(hipErrorStreamCaptureUnsupported);
    if (n > room) return err(hipErrorOutOfMemory);
    size_t at = 4096;
    for (auto &r : live) {
        if (r.first >= at + n) break;
        at = (r.first + r.second.bytes + 4095) / 4096 * 4096;
    }
    live[at] = {n, ++ids, library};
    *p = (void *)at;
    return hipSuccess;
}
hipError_t hipFree(void *p) {
    if (capturing) return err(hipErrorStreamCaptureUnsupported);
    auto it = live.find((size_t)p);
    if (it == live.end()) { dead_freed++; return err(hipErrorInvalidValue); }
    if (!it->second.ours) foreign_freed++;
    live.erase(it);
    return hipSuccess;
}
hipError_t hipPointerGetAttribute(void *data, hipPointer_attribute a, hipDeviceptr_t p) {
    if (a != HIP_POINTER_ATTRIBUTE_BUFFER_ID) return err(hipErrorInvalidValue);
    for (auto &r : live)
        if ((size_t)p >= r.first && (size_t)p < r.first + r.second.bytes) {
            *(unsigned long long *)data = r.second.id;
            return hipSuccess;
        }
    return err(hipErrorInvalidValue);
}
hipError_t hipGetDevice(int *d) { *d = 0; return hipSuccess; }
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t, int) { *v = 256; return hipSuccess; }
hipError_t hipGetLastError() { hipError_t e = last; last = hipSuccess; return e; }
const char *hipGetErrorString(hipError_t) { return "error"; }
hipError_t hipMemcpyAsync(void *d, const void *, size_t n, hipMemcpyKind, hipStream_t) { memset(d, 0, n); return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return capturing ? err(hipErrorStreamCaptureUnsupported) : hipSuccess; }
hipError_t hipStreamIsCapturing(hipStream_t q, hipStreamCaptureStatus *s) {
    *s = capturing && q == capturing ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
    return hipSuccess;
}
hipError_t hipGetSymbolAddress(void **p, const void *s) { *p = (void *)s; return hipSuccess; }
void **__hipRegisterFatBinary(const void *) { static void *h; return &h; }
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
void __hipRegisterFunction(void **, const void *, char *, const char *, unsigned, void *, void *, void *, void *, int *) {}
}

namespace bd {
void set_last_error(const char *) {}
size_t split_bytes(int ld, int nb) { return (size_t)ld * nb * 512; }
int chol_panel_tiles(const CholWork &c) { return c.mpad / 64 >= 60 ? 8 : 0; }
void launch_pack(const double *, int, const CholWork &c, hipStream_t) {
    launches++;
    const size_t a = (size_t)c.A, n = (size_t)c.mpad * c.mpad * sizeof(double);
    for (auto &r : live)
        if (a >= r.first && a + n <= r.first + r.second.bytes) {
            foreign_used += !r.second.ours;
            return;
        }
    dead_used++;
}
void launch_diag(const CholWork &, int, bool, hipStream_t) { launches++; }
void launch_cholesky(const CholWork &, hipStream_t, MarkFn, void *, hipEvent_t, int) { launches++; }
void launch_unpark(const CholWork &, double *, int, hipStream_t) { launches++; }
}  // namespace bd

static double host[1];
static int factor(int m, hipStream_t q = nullptr) {
    int neg = -1;
    return bd_cholesky(m, host, m, host, m, BD_CHOL_FP64, &neg, q);
}
static void device_reset() { live.clear(); }
static void *foreign(size_t bytes) {
    void *p = nullptr;
    library = false;
    (void)hipMalloc(&p, bytes);
    library = true;
    return p;
}
#define CHECK(x) do { if (!(x)) { printf("line %d: %s\n", __LINE__, #x); return 1; } } while (0)
#define SOUND() CHECK(!dead_used && !foreign_used && !foreign_freed && !dead_freed)
"""

SCENES = {
    "kept": r"""
    CHECK(factor(700) == BD_OK && live.size() == 1);
    const auto id = live.begin()->second.id;
    CHECK(factor(100) == BD_OK && factor(700) == BD_OK);
    CHECK(live.size() == 1 && live.begin()->second.id == id);   // the same one throughout
    CHECK(factor(1500) == BD_OK && live.size() == 1 && live.begin()->second.id != id);  // a larger one in its place
    CHECK(factor(7000) == BD_OK && live.empty());   // 392 MB and more: none is kept
    CHECK(factor(64) == BD_OK && live.size() == 1);
    CHECK(bd_cholesky_release() == BD_OK && live.empty());
    CHECK(bd_cholesky_release() == BD_OK);
    SOUND();
""",
    "memory runs out": r"""
    room = (size_t)3968 * 3968 * 8 + ((size_t)63 * 4096 + 32 + 64 * 64 * 64) * 8;
    CHECK(factor(3968) == BD_OK);      // without room for the packed tiles
    room = 1 << 20;
    CHECK(factor(3969) == BD_E_HIP);
    CHECK(last == hipSuccess || hipGetLastError() == hipErrorOutOfMemory);
    room = (size_t)1 << 40;
    CHECK(factor(3969) == BD_OK);
    SOUND();
""",
    "stream under capture": r"""
    capturing = (hipStream_t)4096;
    CHECK(factor(700, capturing) == BD_E_HIP && launches == 0 && live.empty());
    capturing = nullptr;
    (void)hipGetLastError();
    CHECK(factor(700) == BD_OK && live.size() == 1);
    launches = 0;
    capturing = (hipStream_t)4096;
    CHECK(factor(700, capturing) == BD_E_HIP);
    CHECK(launches == 0);           // refused before anything is on the stream
    capturing = nullptr;
    CHECK(live.size() == 1);
    CHECK(bd_cholesky_release() == BD_OK && live.empty());   // and nothing lost
    SOUND();
""",
    "device reset": r"""
    CHECK(factor(700) == BD_OK && live.size() == 1);
    device_reset();
    CHECK(factor(700) == BD_OK && live.size() == 1);
    SOUND();
    device_reset();
    CHECK(bd_cholesky_release() == BD_OK);
    CHECK(hipGetLastError() == hipSuccess);
    SOUND();
""",
    "device reset, the addresses in other hands": r"""
    CHECK(factor(700) == BD_OK && live.size() == 1);
    device_reset();
    void *p = foreign((size_t)1 << 30);
    CHECK(factor(700) == BD_OK && live.count((size_t)p));
    SOUND();
    device_reset();
    p = foreign((size_t)1 << 30);
    CHECK(bd_cholesky_release() == BD_OK && live.count((size_t)p));
    CHECK(factor(900) == BD_OK && live.count((size_t)p));
    SOUND();
""",
}


@pytest.fixture(scope="module")
def potrf(tmp_path_factory):
    if not os.path.exists(HIPCC):
        pytest.skip("hipcc not available")
    d = tmp_path_factory.mktemp("potrf")
    obj = d / "potrf.o"
    r = subprocess.run([HIPCC, "-x", "hip", "--cuda-host-only", "-fPIC", "-std=c++17", "-O1", "-I" + os.path.join(ROOT, "include"),
                        "-c", os.path.join(CSRC, "bd_potrf.hip"), "-o", str(obj)], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-2000:]
    und = subprocess.run(["nm", "-u", str(obj)], capture_output=True, text=True, check=True).stdout.split()
    fat = "".join('extern "C" { char %s[64]; }\n' % s for s in und if s.startswith("__hip_fatbin"))
    return d, obj, fat


@pytest.mark.parametrize("scene", list(SCENES))
def test_workspace(scene, potrf):
    d, obj, fat = potrf
    name = "".join(c if c.isalnum() else "_" for c in scene)
    src, exe = d / f"{name}.cpp", d / name
    src.write_text(FAKE + fat + "int main() {\n" + SCENES[scene] + '    puts("ok");\n    return 0;\n}\n')
    r = subprocess.run([HIPCC, "-x", "hip", "--cuda-host-only", "-fPIC", "-std=c++17", "-O1", "-I" + CSRC,
                        "-I" + os.path.join(ROOT, "include"), "-c", str(src), "-o", str(exe) + ".o"],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-3000:]
    r = subprocess.run(["g++", str(exe) + ".o", str(obj), "-o", str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-3000:]
    out = subprocess.run([str(exe)], capture_output=True, text=True)
    assert out.stdout.strip() == "ok", out.stdout + out.stderr


def test_release_from_python():
    """The user's call that gives the kept workspaces back; without a GPU there
    are none, and it is no error."""
    from brownian_dynamics_cuda_amd import engine as E
    assert E.release_cholesky_workspace() is None
