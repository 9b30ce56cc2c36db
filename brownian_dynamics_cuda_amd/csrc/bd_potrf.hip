// bd_potrf.hip -- the blocked Cholesky factor of a caller's matrix in
// device memory: the library's replacement of cusolverDnDpotrf +
// Cholesky_Decomposition_mod (func_cuda.cu:3513-3534, 614-630), with the
// CPU rule of func.cpp:806-836 for a negative pivot (|f|, counted) instead
// of cuSOLVER's failure code.  The factor itself is the one the step uses
// (bd_chol.hip); this file only moves the caller's matrix into the
// factor's padded storage and the factor back out.
#include <hip/hip_runtime.h>

#include <cstdarg>
#include <cstdio>
#include <mutex>
#include <string>
#include <utility>

#include "../../include/bd_hip.h"
#include "bd_kernels.h"

using namespace bd;

namespace {

int fail(int code, const char *fmt, ...) {
    char buf[512];
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(buf, sizeof buf, fmt, ap);
    va_end(ap);
    set_last_error(buf);
    return code;
}

#define POTRF_CHK(x)                                                                      \
    do {                                                                                  \
        hipError_t e_ = (x);                                                              \
        if (e_ != hipSuccess)                                                             \
            return fail(BD_E_HIP, "%s: %s (%s:%d)", #x, hipGetErrorString(e_), __FILE__, \
                        __LINE__);                                                        \
    } while (0)

int check_args(int m, const double *D, int ldd, const double *L, int ldl, int mode) {
    if (m < 1) return fail(BD_E_ARG, "m must be >= 1 (got %d)", m);
    if (!D || !L) return fail(BD_E_ARG, "D and L are required");
    if (ldd < m || ldl < m) return fail(BD_E_ARG, "leading dimensions must be >= m");
    if (D == L && ldd != ldl) return fail(BD_E_ARG, "in place needs ldd == ldl");
    if (mode != BD_CHOL_FP64 && mode != BD_CHOL_FP32 && mode != BD_CHOL_BF16)
        return fail(BD_E_ARG, "unsupported chol_mode %d", mode);
    return BD_OK;
}

int cus_of_current_device() {
    int dev = 0, ncu = 256;
    if (hipGetDevice(&dev) == hipSuccess) {
        int v = 0;
        if (hipDeviceGetAttribute(&v, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess && v > 0) ncu = v;
    }
    return ncu;
}

CholWork work_of(int m, int mode) {
    CholWork c{};
    c.m = m;
    c.mpad = (m + 63) / 64 * 64;
    c.ld = c.mpad;
    c.mode = mode;
    return c;
}

// Work of one factor in the workspace at ws (doubles): the padded matrix
// (mpad x mpad), the inverses of the diagonal factors (one 64x64 tile per
// block column and one of scratch) and the negative-pivot counter; behind these, where packed,
// the packed panel tiles of the super-panels (pack_bytes, 0 for a matrix that
// has none).
size_t workspace_doubles(int m) {
    const size_t mpad = ((size_t)m + 63) / 64 * 64;
    return mpad * mpad + (mpad / 64 + 1) * 64 * 64 + 32;
}

size_t pack_bytes(int m, int mode) {
    const CholWork c = work_of(m, mode);
    const int nb = chol_panel_tiles(c);
    return nb ? split_bytes(c.ld, nb) : 0;
}

int run_factor(int m, const double *D, int ldd, double *L, int ldl, int mode, int *neg, hipStream_t q,
               double *ws, bool packed) {
    CholWork c = work_of(m, mode);
    c.A = ws;
    c.Linv = ws + (size_t)c.mpad * c.mpad;
    c.neg = reinterpret_cast<int *>(c.Linv + (size_t)(c.mpad / 64 + 1) * 64 * 64);
    c.Lp = ws + workspace_doubles(m);
    if (packed) {
        c.sp = c.Lp + kPanelDoubles;
        c.sp_nb = chol_panel_tiles(c);
    }
    c.ncu = cus_of_current_device();
    c.split_tiles = c.ncu * 19 / 10;
    launch_pack(D, ldd, c, q);
    launch_diag(c, 0, true, q);
    launch_cholesky(c, q);
    launch_unpark(c, L, ldl, q);
    POTRF_CHK(hipGetLastError());
    int h = 0;
    POTRF_CHK(hipMemcpyAsync(&h, c.neg, sizeof(int), hipMemcpyDeviceToHost, q));
    POTRF_CHK(hipStreamSynchronize(q));
    if (neg) *neg = h;
    return BD_OK;
}

constexpr int kMaxDevices = 64;

// The workspace of the last bd_cholesky call on each device, kept for the
// next one: hipMalloc and hipFree took 360 of the 1240 us of a 3001-row factor.
// A call takes the workspace out and puts it back when its stream is done with
// it, so calls that overlap (threads, streams) never share one, and at most one
// workspace of at most kKeepBytes stays per device.  It is given back by
// bd_cholesky_release, by a call that needs a larger one and when an allocation
// of the library fails.  A device reset takes every allocation with it, and the
// addresses may belong to another one by the next call: a kept workspace is used
// or freed only if its address still holds the allocation it was kept as (by the
// number the runtime gives each; 0.3 us).
constexpr size_t kKeepBytes = (size_t)256 << 20;
struct Workspace {
    void *ptr;
    size_t bytes;
    unsigned long long id;
};
std::mutex g_kept_mu;
Workspace g_kept[kMaxDevices] = {};

// the runtime's number of the allocation at p, 0 where there is none
unsigned long long allocation_id(void *p) {
    unsigned long long id = 0;
    if (p && hipPointerGetAttribute(&id, HIP_POINTER_ATTRIBUTE_BUFFER_ID, p) == hipSuccess) return id;
    if (p) (void)hipGetLastError();
    return 0;
}

Workspace exchange_kept(int dev, Workspace w) {
    if (dev < 0 || dev >= kMaxDevices) return w;
    std::lock_guard<std::mutex> lock(g_kept_mu);
    std::swap(g_kept[dev], w);
    return w;
}

// the kept workspace out of its place, none if it is gone
Workspace take_kept(int dev) {
    const Workspace w = exchange_kept(dev, {});
    return w.ptr && allocation_id(w.ptr) == w.id ? w : Workspace{};
}

// at least bytes on the current device dev: the kept workspace if it is large
// enough, else a new one in its place
hipError_t take_workspace(int dev, size_t bytes, Workspace *w) {
    *w = take_kept(dev);
    if (w->bytes >= bytes) return hipSuccess;
    if (w->ptr) (void)hipFree(w->ptr);
    *w = {nullptr, bytes, 0};
    const hipError_t e = hipMalloc(&w->ptr, bytes);
    if (e != hipSuccess) *w = {};
    else w->id = allocation_id(w->ptr);
    return e;
}
hipError_t give_workspace(int dev, Workspace w, bool keep) {
    if (keep && w.id && w.bytes <= kKeepBytes) {
        w = exchange_kept(dev, w);
        // another call's, put back meanwhile
        if (w.ptr && allocation_id(w.ptr) != w.id) return hipSuccess;
    }
    return w.ptr ? hipFree(w.ptr) : hipSuccess;
}

// Workspace of bd_cholesky_noalloc: a static device array of the library,
// sized for matrices of up to kNoallocMaxM rows (33 block columns; the
// 2082-row tensor of the 100-nucleosome fiber fits): 36.8 MB that every GPU
// the library runs on holds until the process ends.  Host code never uses
// the array's name as an address: the device address comes from
// hipGetSymbolAddress, once per device, and is kept in g_scratch.
constexpr int kNoallocMaxM = BD_CHOLESKY_NOALLOC_MAX_M;
constexpr size_t kNoallocDoubles =
    (size_t)kNoallocMaxM * kNoallocMaxM + (size_t)(kNoallocMaxM / 64 + 1) * 64 * 64 + 32;
static __device__ __align__(256) double scratch[kNoallocDoubles];

std::mutex g_scratch_mu;
double *g_scratch[kMaxDevices] = {};

int scratch_of_current_device(double **out) {
    int dev = 0;
    POTRF_CHK(hipGetDevice(&dev));
    if (dev < 0 || dev >= kMaxDevices) return fail(BD_E_ARG, "device ordinal %d out of range", dev);
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (!g_scratch[dev]) {
        void *ptr = nullptr;
        const hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !ptr)
            return fail(BD_E_HIP, "hipGetSymbolAddress(scratch) on device %d: %s", dev, hipGetErrorString(e));
        g_scratch[dev] = static_cast<double *>(ptr);
    }
    *out = g_scratch[dev];
    return BD_OK;
}

}  // namespace

bool bd::release_workspaces() {
    bool any = false;
    for (int dev = 0; dev < kMaxDevices; dev++) {
        const Workspace w = take_kept(dev);
        if (!w.ptr) continue;
        any = true;
        (void)hipFree(w.ptr);
    }
    return any;
}

extern "C" {

int bd_cholesky(int m, const double *D, int ldd, double *L, int ldl, int mode, int *neg, void *stream) {
    int r = check_args(m, D, ldd, L, ldl, mode);
    if (r) return r;
    hipStream_t q = static_cast<hipStream_t>(stream);
    // under capture nothing may be allocated, freed or waited for: refused here,
    // before launches are on the stream and a workspace is out of its place
    hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
    POTRF_CHK(hipStreamIsCapturing(q, &capture));
    if (capture != hipStreamCaptureStatusNone) return fail(BD_E_HIP, "bd_cholesky: the stream is being captured");
    int dev = 0;
    POTRF_CHK(hipGetDevice(&dev));
    Workspace ws{};
    // without room for the packed panel tiles the factor does without them
    const size_t pack = pack_bytes(m, mode), bytes = (workspace_doubles(m) + (pack ? kPanelDoubles : 0)) * sizeof(double);
    const bool packed = pack && take_workspace(dev, bytes + pack, &ws) == hipSuccess;
    if (!packed) {
        if (pack) (void)hipGetLastError();
        POTRF_CHK(take_workspace(dev, bytes, &ws));
    }
    r = run_factor(m, D, ldd, L, ldl, mode, neg, q, static_cast<double *>(ws.ptr), packed);
    // a call that failed may have left work on the stream: nothing is kept
    const hipError_t e = give_workspace(dev, ws, r == BD_OK);
    if (r) return r;
    if (e != hipSuccess) return fail(BD_E_HIP, "hipFree: %s", hipGetErrorString(e));
    return BD_OK;
}

int bd_cholesky_release(void) {
    release_workspaces();
    return BD_OK;
}

int bd_cholesky_noalloc(int m, const double *D, int ldd, double *L, int ldl, int mode, int *neg, void *stream) {
    int r = check_args(m, D, ldd, L, ldl, mode);
    if (r) return r;
    if (m > kNoallocMaxM)
        return fail(BD_E_CAPACITY, "m=%d exceeds the static workspace of bd_cholesky_noalloc (at most %d rows)", m,
                    kNoallocMaxM);
    double *ws = nullptr;
    r = scratch_of_current_device(&ws);
    if (r) return r;
    return run_factor(m, D, ldd, L, ldl, mode, neg, static_cast<hipStream_t>(stream), ws, false);
}

}  // extern "C"
