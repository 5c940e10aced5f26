// Device, context, memory and event entry points of libgip_hip.
#include <cstdio>
#include <cstring>

#include "gip_internal.h"

namespace gip {

thread_local std::string g_last_error;

int set_error(int code, const std::string &msg) {
    g_last_error = msg;
    return code;
}

int hip_fail(hipError_t e, const char *what) {
    return set_error(e == hipErrorOutOfMemory ? GIP_ENOMEM : GIP_EHIP,
                     std::string(what) + ": " + hipGetErrorString(e));
}

// gip_sync's kernel after a published result: the host waits for its number
// as for the result's, so it does not pay for draining what the result's wait
// left (dot and gip_sync 21.6 -> 18.3 us, with the stream drained by both
// 17.8; a step of 46^3 in two partitions, whose halo exchanges call it, 10.5
// -> 7.3 ms).  With the stream drained since, the runtime's own wait is the
// cheaper one (an idle stream 0.4 us against 6.1).
__global__ void k_seq(uint64_t *flag, uint64_t seq) { publish_seq(flag, seq); }

hipError_t drain(gip_ctx *c) {
    const hipError_t e = hipStreamSynchronize(c->stream);
    if (e == hipSuccess) c->published = false;
    return e;
}

int wait_published(gip_ctx *c, const uint64_t *flag, uint64_t want) {
    const hipStream_t st = c->stream;
    c->published = true;
    if (seq_reached(flag, want)) return GIP_OK;
    // a captured kernel does not run: refused as a wait for the stream is,
    // which also ends the capture (asked while the kernel runs)
    if (capturing(st)) {
        const hipError_t e = hipStreamSynchronize(st);
        return e != hipSuccess ? hip_fail(e, "a result under stream capture")
                               : set_error(GIP_EHIP, "a result cannot be waited for under stream capture");
    }
    const int rc = wait_seq(flag, want, [&]() {
        const hipError_t e = hipStreamQuery(st);
        return e == hipErrorNotReady ? -1 : (int)e;
    });
    if (rc == WAIT_OK) return GIP_OK;
    if (rc == WAIT_MISSING) return set_error(GIP_EHIP, "a kernel's result did not arrive");
    return hip_fail((hipError_t)(rc - 1), "waiting for a kernel's result");
}

int reduce_grid(int n) {
    int g = (n + kBlock * 4 - 1) / (kBlock * 4);
    if (g < 1) g = 1;
    if (g > kMaxRedBlocks) g = kMaxRedBlocks;
    return g;
}

}  // namespace gip

using namespace gip;

struct gip_event {
    hipEvent_t ev;
    int device;
};

extern "C" {

const char *gip_last_error(void) { return g_last_error.c_str(); }

int gip_device_count(int *count) {
    if (!count) return set_error(GIP_EINVAL, "count is null");
    GIP_HIP_TRY(hipGetDeviceCount(count));
    return GIP_OK;
}

int gip_init(int device, gip_ctx **out) {
    if (!out) return set_error(GIP_EINVAL, "ctx out pointer is null");
    *out = nullptr;
    int n = 0;
    GIP_HIP_TRY(hipGetDeviceCount(&n));
    if (device < 0 || device >= n) return set_error(GIP_EINVAL, "device index out of range");
    GIP_HIP_TRY(hipSetDevice(device));
    gip_ctx *c = new (std::nothrow) gip_ctx();
    if (!c) return set_error(GIP_ENOMEM, "context allocation failed");
    c->device = device;
    hipDeviceProp_t prop;
    GIP_HIP_TRY(hipGetDeviceProperties(&prop, device));
    c->num_cu = prop.multiProcessorCount;
    // default-priority, non-blocking stream
    hipError_t e = hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking);
    if (e == hipSuccess) e = hipMalloc(&c->d_partials, sizeof(double) * kMaxRedBlocks * 4);
    if (e == hipSuccess) e = hipHostMalloc(&c->h_result, sizeof(double) * kHostBlock, hipHostMallocCoherent);
    if (e == hipSuccess) e = hipHostGetDevicePointer((void **)&c->h_result_dev, c->h_result, 0);
    if (e == hipSuccess) std::memset(c->h_result, 0, sizeof(double) * kHostBlock);
    if (e == hipSuccess) e = hipStreamSynchronize(c->stream);
    if (e != hipSuccess) {
        int rc = hip_fail(e, "context setup");
        gip_finalize(c);
        return rc;
    }
    int rc = pcg_scratch_setup(device);  // the no-alloc solve's scratch on this device
    if (rc) {
        gip_finalize(c);
        return rc;
    }
    *out = c;
    return GIP_OK;
}

int gip_finalize(gip_ctx *c) {
    if (!c) return GIP_OK;
    hipSetDevice(c->device);
    if (c->stream) hipStreamSynchronize(c->stream);
    if (c->d_partials) hipFree(c->d_partials);
    if (c->h_result) hipHostFree(c->h_result);
    if (c->stream) hipStreamDestroy(c->stream);
    delete c;
    return GIP_OK;
}

int gip_use_device(int device) {
    GIP_HIP_TRY(hipSetDevice(device));
    return GIP_OK;
}

int gip_sync(gip_ctx *c) {
    if (!c) return set_error(GIP_EINVAL, "null context");
    if (!c->published || capturing(c->stream)) {
        GIP_HIP_TRY(drain(c));
        return GIP_OK;
    }
    uint64_t want;
    {
        std::lock_guard<std::mutex> lock(c->sync_mu);
        want = ++c->sync_seq;
        k_seq<<<1, 1, 0, c->stream>>>(reinterpret_cast<uint64_t *>(c->h_result_dev + kSyncSlot), want);
        GIP_LAUNCH_CHECK("gip_sync");
    }
    return wait_published(c, reinterpret_cast<const uint64_t *>(c->h_result + kSyncSlot), want);
}

void *gip_stream(gip_ctx *c) { return c ? (void *)c->stream : nullptr; }

int gip_malloc(gip_ctx *c, size_t bytes, void **dptr) {
    if (!c || !dptr) return set_error(GIP_EINVAL, "null argument");
    *dptr = nullptr;
    GIP_HIP_TRY(hipSetDevice(c->device));
    GIP_HIP_TRY(hipMalloc(dptr, bytes ? bytes : 1));
    return GIP_OK;
}

int gip_free(gip_ctx *c, void *dptr) {
    if (!c) return set_error(GIP_EINVAL, "null context");
    if (!dptr) return GIP_OK;
    GIP_HIP_TRY(drain(c));
    GIP_HIP_TRY(hipFree(dptr));
    return GIP_OK;
}

int gip_memcpy_h2d(gip_ctx *c, void *dst, const void *src, size_t bytes) {
    if (!c || (bytes && (!dst || !src))) return set_error(GIP_EINVAL, "null argument");
    if (!bytes) return GIP_OK;
    GIP_HIP_TRY(hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, c->stream));
    GIP_HIP_TRY(drain(c));  // the host buffer may be reused at return
    return GIP_OK;
}

int gip_memcpy_d2h(gip_ctx *c, void *dst, const void *src, size_t bytes) {
    if (!c || (bytes && (!dst || !src))) return set_error(GIP_EINVAL, "null argument");
    if (!bytes) return GIP_OK;
    GIP_HIP_TRY(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, c->stream));
    GIP_HIP_TRY(drain(c));
    return GIP_OK;
}

int gip_memcpy_d2d(gip_ctx *c, void *dst, const void *src, size_t bytes) {
    if (!c || (bytes && (!dst || !src))) return set_error(GIP_EINVAL, "null argument");
    if (!bytes) return GIP_OK;
    GIP_HIP_TRY(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToDevice, c->stream));
    return GIP_OK;
}

int gip_event_create(gip_ctx *c, gip_event **ev) {
    if (!c || !ev) return set_error(GIP_EINVAL, "null argument");
    gip_event *e = new (std::nothrow) gip_event();
    if (!e) return set_error(GIP_ENOMEM, "event allocation failed");
    e->device = c->device;
    hipError_t r = hipEventCreate(&e->ev);
    if (r != hipSuccess) {
        delete e;
        return hip_fail(r, "hipEventCreate");
    }
    *ev = e;
    return GIP_OK;
}

int gip_event_record(gip_ctx *c, gip_event *ev) {
    if (!c || !ev) return set_error(GIP_EINVAL, "null argument");
    GIP_HIP_TRY(hipEventRecord(ev->ev, c->stream));
    return GIP_OK;
}

int gip_event_elapsed_ms(gip_event *a, gip_event *b, float *ms) {
    if (!a || !b || !ms) return set_error(GIP_EINVAL, "null argument");
    GIP_HIP_TRY(hipEventSynchronize(b->ev));
    GIP_HIP_TRY(hipEventElapsedTime(ms, a->ev, b->ev));
    return GIP_OK;
}

int gip_event_destroy(gip_event *ev) {
    if (!ev) return GIP_OK;
    hipEventDestroy(ev->ev);
    delete ev;
    return GIP_OK;
}

}  // extern "C"
