// xnor_nn_hip_forward_pass (xnor_nn_amd/csrc/api.hip) on the CPU, with stand-ins for the launches and
// for the runtime: two threads run passes on one descriptor, each with a resource table and a stream of
// its own, and every launch of a pass has to go to that pass's stream.  Usage: pass_stream_check CASE.
#include <chrono>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <string>
#include <thread>

#include "plan.hpp"
#include "xnor_nn_hip.h"

namespace {
bool matrix_cores = true;
std::atomic<int> launches{0}, strays{0};
thread_local hipStream_t own = nullptr;

hipError_t launched(hipStream_t s) {
    launches++;
    if (s != own) strays++;
    std::this_thread::sleep_for(std::chrono::microseconds(20)); // the other thread asks for the lock
    return hipSuccess;
}
} // namespace

namespace xnor_hip {
void binarize_plan(Plan &) {}
void mfma_plan(Plan &g) { g.use_mfma = matrix_cores; }
int pick_q(int, int) { return 4; }
hipError_t launch_binarize_data(const Plan &, const float *, uint32_t *, float *, hipStream_t s,
        const KernelEvents &) { return launched(s); }
hipError_t launch_mean_abs(const Plan &, const float *, float *, hipStream_t s) { return launched(s); }
bool weights_join_binarize(const Plan &) { return false; }
hipError_t launch_binarize_data_and_weights(const Plan &, const float *, uint32_t *, float *, const float *,
        uint32_t *, uint32_t *, float *, int32_t *, hipStream_t s) { return launched(s); }
hipError_t launch_box_filter(const Plan &, const float *, float *, hipStream_t s) { return launched(s); }
hipError_t launch_plain_read(const void *, size_t, hipStream_t s, const KernelEvents &) {
    return launched(s);
}
hipError_t launch_binarize_weights(const Plan &, const float *, uint32_t *, uint32_t *, float *, int32_t *,
        hipStream_t s) { return launched(s); }
hipError_t launch_convolution(const Plan &, const uint32_t *, const uint32_t *, const float *,
        const float *, const int32_t *, float *, int32_t *, hipStream_t s, const KernelEvents &) {
    return launched(s);
}
int weights_float_parts() { return 1; }
hipError_t launch_weights_float(const float *, float *, size_t, float *, hipStream_t s) {
    return launched(s);
}
hipError_t weights_float_scratch(float **) { return hipSuccess; }
hipError_t launch_convolution_mfma(const Plan &, const uint32_t *, const uint32_t *, const float *,
        const float *, float *, int32_t *, const float *, float *, hipStream_t s, const KernelEvents &) {
    return launched(s);
}
hipError_t launch_mfma_only(int, int, hipStream_t s) { return launched(s); }
hipError_t launch_forward_small(const Plan &, const float *, uint32_t *, float *, const uint32_t *,
        const float *, float *, float *, hipStream_t s) { return launched(s); }
const char *convolution_kernel_name(const Plan &) { return ""; }
const char *binarize_kernel_name(const Plan &) { return ""; }
const char *weights_kernel_name(const Plan &) { return ""; }
Memory memory_of(const void *) { return Memory::device; }
HostIo::~HostIo() {}
bool HostIo::move(hipStream_t, const char *, Memory, size_t, char *, char *, Memory, size_t, const char *,
        bool (*)(void *), void *) { return false; }
void host_io_descriptor_created() {}
void host_io_descriptor_destroyed() {}
} // namespace xnor_hip

extern "C" {
hipError_t hipMalloc(void **p, size_t n) { *p = malloc(n); return hipSuccess; }
hipError_t hipFree(void *p) { free(p); return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipGetDevice(int *d) { *d = 0; return hipSuccess; }
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t, int) { *v = 256; return hipSuccess; }
hipError_t hipMemcpyAsync(void *, const void *, size_t, hipMemcpyKind, hipStream_t) {
    return hipErrorUnknown;
}
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipErrorUnknown; }
hipError_t hipEventCreate(hipEvent_t *) { return hipErrorUnknown; }
hipError_t hipEventCreateWithFlags(hipEvent_t *, unsigned) { return hipErrorUnknown; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipErrorUnknown; }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *, hipEvent_t, hipEvent_t) { return hipErrorUnknown; }
}

int main(int argc, char **argv) {
    const std::string name = argc > 1 ? argv[1] : "";
    matrix_cores = name != "popcount kernel";
    const int weights = name == "old weights" ? 0 : XNOR_NN_HIP_NEW_WEIGHTS;
    xnor_nn_convolution_t c;
    if (xnor_nn_init_convolution(&c, xnor_nn_algorithm_bcast, xnor_nn_data_format_nchw,
                xnor_nn_weights_format_oihw, xnor_nn_data_format_nchw, 1, 32, 32, 8, 8, 3, 3, 1, 1, 1, 1)
            != xnor_nn_success)
        return 1;
    if (name != "one pass" && xnor_nn_hip_set_stage_fusion(&c, 0) != xnor_nn_success) return 1;
    std::atomic<int> failed{0};
    auto passes = [&](int number) {
        static char streams[2];
        own = reinterpret_cast<hipStream_t>(&streams[number]);
        xnor_nn_resources_t res = {};
        float weight = 0.f, in = 0.f, out = 0.f;
        if (xnor_nn_allocate_resources(&c, res) != xnor_nn_success) { failed++; return; }
        res[xnor_nn_resource_user_weights] = &weight;
        for (int i = 0; i < 200; i++)
            if (xnor_nn_hip_forward_pass(&c, res, &in, &out, own,
                        XNOR_NN_HIP_DEVICE_POINTERS | XNOR_NN_HIP_ON_STREAM | weights) != xnor_nn_success)
                failed++;
        xnor_nn_free_resources(res);
    };
    std::thread a(passes, 0), b(passes, 1);
    a.join();
    b.join();
    xnor_nn_destroy_convolution(&c);
    if (failed || strays || launches < 2 * 200 * 2) {
        printf("%d calls failed, %d of %d launches on the other thread's stream\n", failed.load(),
                strays.load(), launches.load());
        return 1;
    }
    printf("ok\n");
    return 0;
}
