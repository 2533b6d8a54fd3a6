// zant_model_predict_host gives the caller's input buffer back only when its upload has been waited for, also where a later step fails (host
// code only: the HIP calls that it makes are this program's own).  Prints "ok" when it does.
#include <cstdio>
#include <cstdlib>
#include <cstring>

#include "common.h"
#include "zant_hip.h"

static bool uploading = false;            // an upload from the caller's buffer may still read it
static int fail_download = 0;             // 1: cannot be enqueued, 2: its wait fails once
static bool wait_fails = false;

extern "C" {
hipError_t hipMalloc(void **p, size_t n) { return (*p = std::calloc(1, n)) ? hipSuccess : hipErrorOutOfMemory; }
hipError_t hipFree(void *p) { std::free(p); return hipSuccess; }
hipError_t hipMemsetAsync(void *p, int v, size_t n, hipStream_t) { std::memset(p, v, n); return hipSuccess; }
hipError_t hipMemcpyAsync(void *to, const void *from, size_t n, hipMemcpyKind kind, hipStream_t) {
    if (kind == hipMemcpyDeviceToHost && fail_download == 1) return hipErrorInvalidValue;
    std::memcpy(to, from, n);
    if (kind == hipMemcpyHostToDevice) uploading = true;
    if (kind == hipMemcpyDeviceToHost && fail_download == 2) wait_fails = true;
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) {
    if (wait_fails) { wait_fails = false; return hipErrorUnknown; }
    uploading = false;
    return hipSuccess;
}
}

int main() {
    zant_ctx ctx;
    ctx.num_cus = 256;
    zant_model *m = nullptr;
    const int64_t in[4] = {2, 3, 4, 5}, out[2] = {6, 20};
    if (zant_model_create(&ctx, &m) != ZANT_OK) return 1;
    const int x = zant_model_input(m, ZANT_F32, in, 4, 1.0f, 0), y = x < 0 ? x : zant_model_reshape(m, x, out, 2);
    if (x < 0 || y < 0 || zant_model_finalize(m) != ZANT_OK) { std::printf("model: %d %d\n", x, y); return 1; }
    float a[120], b[120] = {};
    for (int i = 0; i < 120; ++i) a[i] = float(i);
    for (fail_download = 0; fail_download <= 2; ++fail_download) {
        uploading = false;
        const int rc = zant_model_predict_host(m, a, b);
        if ((rc == ZANT_OK) != (fail_download == 0)) { std::printf("failure %d: returns %d\n", fail_download, rc); return 1; }
        if (uploading) { std::printf("failure %d: returns while the upload may read the buffer\n", fail_download); return 1; }
        if (!fail_download && std::memcmp(a, b, sizeof(a)) != 0) { std::puts("wrong result"); return 1; }
    }
    std::puts("ok");
    std::fflush(stdout);
    std::_Exit(0);  // (the model's memory is this program's)
}
