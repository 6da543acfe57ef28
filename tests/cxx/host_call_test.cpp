/*
 * Host-pointer calls whose launches fail, without a GPU: the shim's source is
 * compiled in and the HIP calls it makes are replaced by these, which keep
 * "device" memory on the host, launch nothing and can fail a chosen launch.
 * A call that fails at any of its launches writes nothing to its output, as
 * the reference's (src/quantized_matvec.cpp:196-223 validates first and fails
 * whole), and the next call is served.
 */
#include "../../my-inference-engine_amd/csrc/qmv_shim.cpp"

#include <cstdio>
#include <vector>

namespace {
int g_launches = 0, g_fail_at = -1; /* count of launches; the one that fails */
hipError_t g_launch_error = hipSuccess;
} // namespace

extern "C" {
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDevice(int *d) { *d = 0; return hipSuccess; }
hipError_t hipMalloc(void **p, size_t n) { *p = calloc(1, n); return hipSuccess; }
hipError_t hipFree(void *p) { free(p); return hipSuccess; }
hipError_t hipHostMalloc(void **p, size_t n, unsigned) { *p = calloc(1, n); return hipSuccess; }
hipError_t hipHostFree(void *p) { free(p); return hipSuccess; }
hipError_t hipHostGetDevicePointer(void **d, void *h, unsigned) { *d = h; return hipSuccess; }
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t) { memcpy(d, s, n); return hipSuccess; }
hipError_t hipMemsetAsync(void *d, int v, size_t n, hipStream_t) { memset(d, v, n); return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) { *s = (hipStream_t)calloc(1, 8); return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus *c) { *c = hipStreamCaptureStatusNone; return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { *e = (hipEvent_t)calloc(1, 8); return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t __hipPushCallConfiguration(dim3, dim3, size_t, hipStream_t) { return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3 *, dim3 *, size_t *, hipStream_t *) { return hipSuccess; }
hipError_t hipLaunchKernel(const void *, dim3, dim3, void **, size_t, hipStream_t)
{
    g_launch_error = g_launches++ == g_fail_at ? hipErrorLaunchFailure : hipSuccess;
    return g_launch_error;
}
hipError_t hipGetLastError()
{
    const hipError_t e = g_launch_error;
    g_launch_error = hipSuccess;
    return e;
}
}

int main()
{
    const int rows = 3000, cols = 512, batch = 170; /* six launches, 2.4 MB */
    std::vector<unsigned char> w((size_t)rows * cols / 32 * 34);
    QmvTensorView v = {};
    v.data = w.data();
    v.ggml_type = QMV_GGML_TYPE_Q8_0;
    v.dimension_count = 2;
    v.dimensions[0] = cols;
    v.dimensions[1] = rows;
    v.dimensions[2] = v.dimensions[3] = 1;
    v.element_count = (uint64_t)rows * cols;
    v.block_elements = 32;
    v.block_bytes = 34;
    v.block_count = v.element_count / 32;
    std::vector<float> in((size_t)batch * cols, 1.0f), out((size_t)batch * rows);
    const auto call = [&]() {
        g_launches = 0;
        std::fill(out.begin(), out.end(), 7.0f);
        return qmv_tensor_matmul_f32(&v, in.data(), cols, batch, out.data(), rows);
    };
    if (call() != 1) { /* uploads the tensor as well */
        printf("the first call failed: %s\n", qmv_last_error());
        return 1;
    }
    if (call() != 1) return 1;
    const int launches = g_launches;
    if (launches < 6) {
        printf("%d launches: not a call of several\n", launches);
        return 1;
    }
    int failures = 0;
    for (g_fail_at = 0; g_fail_at < launches; ++g_fail_at) {
        const int ok = call();
        size_t written = 0;
        for (float o : out) written += o != 7.0f;
        if (ok || written) {
            ++failures;
            printf("launch %d of %d fails: the call returns %d, %zu outputs written\n", g_fail_at, launches, ok, written);
        }
    }
    g_fail_at = -1;
    if (call() != 1 || out[0] != 0.0f || out.back() != 0.0f) {
        ++failures;
        printf("the call after a failure is not served\n");
    }
    printf("%d launches, %d failures\n", launches, failures);
    return failures != 0;
}
