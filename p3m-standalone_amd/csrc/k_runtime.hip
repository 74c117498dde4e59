// HIP runtime wrappers of the internal C ABI: streams, events, memory,
// small utility kernels.
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdio>
#include <cstring>

#include "k_internal.hpp"

static thread_local char g_err[512];

extern "C" const char *p3mk_error(void) { return g_err; }

int p3mk_fail(int code, const char *what, int hip_code) {
    if (hip_code != 0)
        std::snprintf(g_err, sizeof(g_err), "%s: %s", what,
                      hipGetErrorString((hipError_t)hip_code));
    else
        std::snprintf(g_err, sizeof(g_err), "%s", what);
    return code;
}

int p3mk_launch_check(const char *what) {
    hipError_t e = hipGetLastError();
    if (e != hipSuccess)
        return p3mk_fail(P3MK_EDEVICE, what, (int)e);
    return P3MK_OK;
}

struct p3mk_queue {
    hipStream_t stream;
    hipEvent_t ev[P3MK_NUM_EVENTS];
    // optional ring of event sets: set k receives the events of the k-th
    // step after p3mk_ring_start, so the stage times of several steps can be
    // read after they all ran
    hipEvent_t *ring = nullptr;
    int ring_sets = 0;
    int ring_pos = 0;
};

static void ring_free(p3mk_queue *q) {
    if (q->ring) {
        for (int i = 0; i < q->ring_sets * P3MK_NUM_EVENTS; i++)
            (void)hipEventDestroy(q->ring[i]);
        delete[] q->ring;
    }
    q->ring = nullptr;
    q->ring_sets = q->ring_pos = 0;
}

hipStream_t p3mk_stream(p3mk_queue *q) { return q ? q->stream : (hipStream_t)0; }

extern "C" int p3mk_device_check(void) {
    int n = 0;
    hipError_t e = hipGetDeviceCount(&n);
    if (e != hipSuccess || n < 1)
        return p3mk_fail(P3MK_ENODEVICE, "no HIP device available", e == hipSuccess ? 0 : (int)e);
    return P3MK_OK;
}

extern "C" int p3mk_queue_create(p3mk_queue **out) {
    int rc = p3mk_device_check();
    if (rc != P3MK_OK)
        return rc;
    p3mk_queue *q = new (std::nothrow) p3mk_queue;
    if (!q)
        return p3mk_fail(P3MK_ENOMEM, "queue allocation failed", 0);
    hipError_t e = hipStreamCreateWithFlags(&q->stream, hipStreamNonBlocking);
    if (e != hipSuccess) {
        delete q;
        return p3mk_fail(P3MK_EDEVICE, "hipStreamCreate", (int)e);
    }
    for (int i = 0; i < P3MK_NUM_EVENTS; i++) {
        e = hipEventCreate(&q->ev[i]);
        if (e != hipSuccess) {
            for (int j = 0; j < i; j++)
                (void)hipEventDestroy(q->ev[j]);
            (void)hipStreamDestroy(q->stream);
            delete q;
            return p3mk_fail(P3MK_EDEVICE, "hipEventCreate", (int)e);
        }
    }
    *out = q;
    return P3MK_OK;
}

extern "C" void p3mk_queue_destroy(p3mk_queue *q) {
    if (!q)
        return;
    (void)hipStreamSynchronize(q->stream);
    ring_free(q);
    for (int i = 0; i < P3MK_NUM_EVENTS; i++)
        (void)hipEventDestroy(q->ev[i]);
    (void)hipStreamDestroy(q->stream);
    delete q;
}

extern "C" int p3mk_queue_sync(p3mk_queue *q) {
    hipError_t e = hipStreamSynchronize(q->stream);
    if (e != hipSuccess)
        return p3mk_fail(P3MK_EDEVICE, "hipStreamSynchronize", (int)e);
    return P3MK_OK;
}

extern "C" int p3mk_record(p3mk_queue *q, int slot) {
    if (slot < 0 || slot >= P3MK_NUM_EVENTS)
        return p3mk_fail(P3MK_EINVAL, "event slot out of range", 0);
    hipError_t e = hipEventRecord(q->ev[slot], q->stream);
    if (e != hipSuccess)
        return p3mk_fail(P3MK_EDEVICE, "hipEventRecord", (int)e);
    if (q->ring && q->ring_pos < q->ring_sets) {
        e = hipEventRecord(q->ring[q->ring_pos * P3MK_NUM_EVENTS + slot], q->stream);
        if (e != hipSuccess)
            return p3mk_fail(P3MK_EDEVICE, "hipEventRecord", (int)e);
    }
    return P3MK_OK;
}

extern "C" int p3mk_ring_start(p3mk_queue *q, int nsets) {
    if (nsets < 0)
        return p3mk_fail(P3MK_EINVAL, "negative ring size", 0);
    hipError_t e = hipStreamSynchronize(q->stream);
    if (e != hipSuccess)
        return p3mk_fail(P3MK_EDEVICE, "hipStreamSynchronize", (int)e);
    ring_free(q);
    if (nsets == 0)
        return P3MK_OK;
    q->ring = new (std::nothrow) hipEvent_t[(size_t)nsets * P3MK_NUM_EVENTS];
    if (!q->ring)
        return p3mk_fail(P3MK_ENOMEM, "event ring allocation failed", 0);
    for (int i = 0; i < nsets * P3MK_NUM_EVENTS; i++) {
        e = hipEventCreate(&q->ring[i]);
        if (e != hipSuccess) {
            for (int j = 0; j < i; j++)
                (void)hipEventDestroy(q->ring[j]);
            delete[] q->ring;
            q->ring = nullptr;
            return p3mk_fail(P3MK_EDEVICE, "hipEventCreate", (int)e);
        }
    }
    q->ring_sets = nsets;
    q->ring_pos = 0;
    return P3MK_OK;
}

extern "C" void p3mk_ring_advance(p3mk_queue *q) {
    if (q->ring && q->ring_pos < q->ring_sets)
        q->ring_pos++;
}

extern "C" int p3mk_ring_filled(p3mk_queue *q) { return q->ring ? q->ring_pos : 0; }

extern "C" int p3mk_ring_elapsed_ms(p3mk_queue *q, int set, int a, int b, float *ms) {
    if (!q->ring || set < 0 || set >= q->ring_pos || a < 0 || b < 0 || a >= P3MK_NUM_EVENTS ||
        b >= P3MK_NUM_EVENTS)
        return p3mk_fail(P3MK_EINVAL, "event ring slot out of range", 0);
    hipError_t e = hipEventElapsedTime(ms, q->ring[set * P3MK_NUM_EVENTS + a],
                                       q->ring[set * P3MK_NUM_EVENTS + b]);
    if (e != hipSuccess)
        return p3mk_fail(P3MK_EDEVICE, "hipEventElapsedTime", (int)e);
    return P3MK_OK;
}

extern "C" int p3mk_elapsed_ms(p3mk_queue *q, int a, int b, float *ms) {
    if (a < 0 || b < 0 || a >= P3MK_NUM_EVENTS || b >= P3MK_NUM_EVENTS)
        return p3mk_fail(P3MK_EINVAL, "event slot out of range", 0);
    hipError_t e = hipEventElapsedTime(ms, q->ev[a], q->ev[b]);
    if (e != hipSuccess)
        return p3mk_fail(P3MK_EDEVICE, "hipEventElapsedTime", (int)e);
    return P3MK_OK;
}

extern "C" int p3mk_alloc(void **p, size_t bytes) {
    *p = nullptr;
    if (bytes == 0)
        return P3MK_OK;
    hipError_t e = hipMalloc(p, bytes);
    if (e != hipSuccess) {
        *p = nullptr;
        (void)hipGetLastError(); // reported here, not by the next launch check
        return p3mk_fail(P3MK_ENOMEM, "hipMalloc", (int)e);
    }
    return P3MK_OK;
}

extern "C" void p3mk_release(void *p) {
    if (p)
        (void)hipFree(p);
}

extern "C" int p3mk_alloc_host(void **p, size_t bytes) {
    *p = nullptr;
    if (bytes == 0)
        return P3MK_OK;
    hipError_t e = hipHostMalloc(p, bytes, hipHostMallocDefault);
    if (e != hipSuccess) {
        *p = nullptr;
        return p3mk_fail(P3MK_ENOMEM, "hipHostMalloc", (int)e);
    }
    return P3MK_OK;
}

extern "C" void p3mk_release_host(void *p) {
    if (p)
        (void)hipHostFree(p);
}

static int copy(void *dst, const void *src, size_t bytes, hipMemcpyKind k, p3mk_queue *q) {
    if (bytes == 0)
        return P3MK_OK;
    hipError_t e = hipMemcpyAsync(dst, src, bytes, k, q->stream);
    if (e != hipSuccess)
        return p3mk_fail(P3MK_EDEVICE, "hipMemcpyAsync", (int)e);
    return P3MK_OK;
}

extern "C" int p3mk_copy_h2d(void *dst, const void *src, size_t bytes, p3mk_queue *q) {
    return copy(dst, src, bytes, hipMemcpyHostToDevice, q);
}
extern "C" int p3mk_copy_d2h(void *dst, const void *src, size_t bytes, p3mk_queue *q) {
    return copy(dst, src, bytes, hipMemcpyDeviceToHost, q);
}
extern "C" int p3mk_copy_d2d(void *dst, const void *src, size_t bytes, p3mk_queue *q) {
    return copy(dst, src, bytes, hipMemcpyDeviceToDevice, q);
}

__global__ void k_axpy(size_t n, double a, const double *__restrict__ x, double *__restrict__ y) {
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    const size_t stride = (size_t)gridDim.x * blockDim.x;
    for (; i < n; i += stride)
        y[i] += a * x[i];
}

extern "C" int p3mk_axpy(size_t n, double a, const double *x, double *y, p3mk_queue *q) {
    if (n == 0)
        return P3MK_OK;
    size_t blocks = (n + 255) / 256;
    if (blocks > 8192)
        blocks = 8192;
    hipLaunchKernelGGL(k_axpy, dim3((unsigned)blocks), dim3(256), 0, q->stream, n, a, x, y);
    return p3mk_launch_check("axpy");
}

// p: the 16-byte unit each range begins in; the range is [lo, hi) from there
struct FillRanges {
    unsigned char *p[P3MK_MAX_RANGES];
    unsigned long long hi[P3MK_MAX_RANGES], first[P3MK_MAX_RANGES + 1]; // first unit of each
    unsigned char lo[P3MK_MAX_RANGES];
};

__global__ void k_fill_many(FillRanges r, int k) {
    const unsigned long long stride = (unsigned long long)gridDim.x * blockDim.x;
    const uint4 z = make_uint4(0u, 0u, 0u, 0u);
    for (unsigned long long u = (unsigned long long)blockIdx.x * blockDim.x + threadIdx.x; u < r.first[k];
         u += stride) {
        int s = 0;
#pragma unroll
        for (int j = 1; j < P3MK_MAX_RANGES; j++)
            s += (j < k && u >= r.first[j]) ? 1 : 0;
        unsigned char *base = r.p[0];
        unsigned long long lo = r.lo[0], hi = r.hi[0], first = r.first[0];
#pragma unroll
        for (int j = 1; j < P3MK_MAX_RANGES; j++)
            if (s == j) {
                base = r.p[j];
                lo = r.lo[j];
                hi = r.hi[j];
                first = r.first[j];
            }
        const unsigned long long at = (u - first) * 16;
        if (at >= lo && at + 16 <= hi) {
            *reinterpret_cast<uint4 *>(base + at) = z;
        } else { // a range's first or last unit
            for (unsigned long long b = at > lo ? at : lo; b < at + 16 && b < hi; b += 4)
                *reinterpret_cast<unsigned int *>(base + b) = 0u;
        }
    }
}

// One launch for all the buffers a force evaluation starts from zero (a
// launch each, and one more for a size that is no multiple of 16 bytes, were
// a third of a small system's launches).  A range may begin at any word: the
// callers' force arrays and the parts of one array are 8-byte aligned.
extern "C" int p3mk_fill_zero_many(int k, const p3mk_range *ranges, p3mk_queue *q) {
    FillRanges r = {};
    int n = 0;
    unsigned long long units = 0;
    for (int j = 0; j < k; j++) {
        if (ranges[j].bytes == 0)
            continue;
        const unsigned long long p = (unsigned long long)ranges[j].p, lo = p % 16;
        if (n == P3MK_MAX_RANGES || ranges[j].bytes % 4 != 0 || p % 4 != 0)
            return p3mk_fail(P3MK_EINVAL, "zero fill: too many ranges, or one not of whole words", 0);
        r.p[n] = (unsigned char *)ranges[j].p - lo;
        r.lo[n] = (unsigned char)lo;
        r.hi[n] = lo + ranges[j].bytes;
        r.first[n] = units;
        units += (r.hi[n] + 15) / 16;
        n++;
    }
    if (n == 0)
        return P3MK_OK;
    for (int j = n; j <= P3MK_MAX_RANGES; j++)
        r.first[j] = units;
    const unsigned blocks = (unsigned)(units > 8192ull * 256 ? 8192 : (units + 255) / 256);
    hipLaunchKernelGGL(k_fill_many, dim3(blocks), dim3(256), 0, q->stream, r, n);
    return p3mk_launch_check("fill_zero");
}

extern "C" int p3mk_fill_zero(void *p, size_t bytes, p3mk_queue *q) {
    const p3mk_range r = {p, bytes};
    return p3mk_fill_zero_many(1, &r, q);
}

// The reference's sum (common.c:315-319): f_k + f_r rounded, then added to f.
__global__ void k_finish_forces(int n, const int *__restrict__ pos, const double *__restrict__ fs, int add_fr,
                                int add_f, const double *__restrict__ fk, double *__restrict__ fr,
                                double *__restrict__ f) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n)
        return;
    const long p = fs != nullptr ? pos[i] : 0;
#pragma unroll
    for (int d = 0; d < 3; d++) {
        const long j = (long)d * n + i;
        double r = add_fr ? fr[j] : 0.0;
        if (fs != nullptr)
            r += fs[(long)d * n + p];
        fr[j] = r;
        const double s = fk[j] + r;
        f[j] = add_f ? f[j] + s : s;
    }
}

extern "C" int p3mk_finish_forces(int n, const int *pos, const double *fs, int add_fr, int add_f,
                                  const double *fk, double *fr, double *f, p3mk_queue *q) {
    if (n <= 0)
        return P3MK_OK;
    hipLaunchKernelGGL(k_finish_forces, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, q->stream, n, pos, fs,
                       add_fr, add_f, fk, fr, f);
    return p3mk_launch_check("finish forces");
}

__global__ void k_check_positions(int n, double lo, double hi, const double *__restrict__ x,
                                  const double *__restrict__ y, const double *__restrict__ z,
                                  int *bad) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    int b = 0;
    if (i < n) {
        const double v[3] = {x[i], y[i], z[i]};
        for (int d = 0; d < 3; d++)
            b |= !(v[d] >= lo && v[d] < hi);
    }
    // one atomic per wavefront
    unsigned long long m = __ballot(b);
    if ((threadIdx.x & 63) == 0 && m)
        atomicAdd(bad, (int)__popcll(m));
}

extern "C" int p3mk_check_positions(int n, double lo, double hi, const double *x, const double *y,
                                    const double *z, int *bad, int *scratch, p3mk_queue *q) {
    *bad = 0;
    if (n <= 0)
        return P3MK_OK;
    int rc = p3mk_fill_zero(scratch, sizeof(int), q);
    if (rc)
        return rc;
    hipLaunchKernelGGL(k_check_positions, dim3((n + 255) / 256), dim3(256), 0, q->stream, n, lo,
                       hi, x, y, z, scratch);
    rc = p3mk_launch_check("check_positions");
    if (rc)
        return rc;
    rc = p3mk_copy_d2h(bad, scratch, sizeof(int), q);
    if (rc)
        return rc;
    return p3mk_queue_sync(q);
}

struct p3mk_graph {
    hipGraph_t graph;
    hipGraphExec_t exec;
};

extern "C" int p3mk_capture_begin(p3mk_queue *q) {
    hipError_t e = hipStreamBeginCapture(q->stream, hipStreamCaptureModeThreadLocal);
    if (e != hipSuccess)
        return p3mk_fail(P3MK_EDEVICE, "hipStreamBeginCapture", (int)e);
    return P3MK_OK;
}

extern "C" int p3mk_capture_end(p3mk_queue *q, p3mk_graph **out) {
    *out = nullptr;
    hipGraph_t g = nullptr;
    hipError_t e = hipStreamEndCapture(q->stream, &g);
    if (e != hipSuccess)
        return p3mk_fail(P3MK_EDEVICE, "hipStreamEndCapture", (int)e);
    p3mk_graph *pg = new (std::nothrow) p3mk_graph;
    if (!pg) {
        (void)hipGraphDestroy(g);
        return p3mk_fail(P3MK_ENOMEM, "graph allocation", 0);
    }
    pg->graph = g;
    e = hipGraphInstantiate(&pg->exec, g, nullptr, nullptr, 0);
    if (e != hipSuccess) {
        (void)hipGraphDestroy(g);
        delete pg;
        return p3mk_fail(P3MK_EDEVICE, "hipGraphInstantiate", (int)e);
    }
    *out = pg;
    return P3MK_OK;
}

extern "C" int p3mk_graph_launch(p3mk_graph *g, p3mk_queue *q) {
    hipError_t e = hipGraphLaunch(g->exec, q->stream);
    if (e != hipSuccess)
        return p3mk_fail(P3MK_EDEVICE, "hipGraphLaunch", (int)e);
    return P3MK_OK;
}

extern "C" void p3mk_graph_destroy(p3mk_graph *g) {
    if (!g)
        return;
    (void)hipGraphExecDestroy(g->exec);
    (void)hipGraphDestroy(g->graph);
    delete g;
}
