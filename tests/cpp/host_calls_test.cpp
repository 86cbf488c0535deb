// Host-side checks of the library without a GPU: this program defines the HIP runtime calls that
// libipic_gpu.so makes (its own definitions take precedence over the runtime's), runs no kernel,
// notes what is queued and allocated, and can refuse a launch.
//
//   host_calls_test --failed-step   after a step that fails with work queued, a call that hands out
//                                   device pointers waits for that work
//   host_calls_test --create        what creating a context allocates
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <initializer_list>

#include "ipic_gpu.h"

namespace {
int launches = 0, refuse = 0, error = 0, device_allocs = 0, pinned_allocs = 0;
bool queued = false;
}  // namespace

extern "C" {
struct Dim3 { unsigned x, y, z; };
int hipGetDevice(int* d) { *d = 0; return 0; }
int hipDeviceGetAttribute(int* v, int, int) { *v = 256; return 0; }
int hipMalloc(void** p, size_t n) { *p = std::calloc(1, n); ++device_allocs; return *p ? 0 : 2; }
int hipFree(void* p) { std::free(p); return 0; }
int hipHostMalloc(void** p, size_t n, unsigned) { *p = std::calloc(1, n); ++pinned_allocs; return *p ? 0 : 2; }
int hipHostFree(void* p) { std::free(p); return 0; }
int hipMemcpy(void* d, const void* s, size_t n, int) { std::memcpy(d, s, n); return 0; }
int hipMemcpyAsync(void* d, const void* s, size_t n, int, void*) { std::memcpy(d, s, n); queued = true; return 0; }
int hipMemsetAsync(void* d, int v, size_t n, void*) { std::memset(d, v, n); queued = true; return 0; }
int hipStreamCreateWithFlags(void** s, unsigned) { *s = std::malloc(1); return 0; }
int hipStreamDestroy(void* s) { std::free(s); return 0; }
int hipStreamSynchronize(void*) { queued = false; return 0; }
int hipEventCreate(void** e) { *e = std::malloc(1); return 0; }
int hipEventDestroy(void* e) { std::free(e); return 0; }
int hipEventRecord(void*, void*) { return 0; }
int hipEventSynchronize(void*) { return 0; }
int hipEventElapsedTime(float* ms, void*, void*) { *ms = 0; return 0; }
int hipGetLastError() { const int e = error; error = 0; return e; }
const char* hipGetErrorString(int) { return "refused"; }
int hipLaunchKernel(const void*, Dim3, Dim3, void**, size_t, void*) {
    if (++launches == refuse) return error = 719;
    queued = true;
    return 0;
}
int __hipPushCallConfiguration(Dim3, Dim3, size_t, void*) { return 0; }
int __hipPopCallConfiguration(Dim3* g, Dim3* b, size_t* n, void** s) {
    *g = *b = Dim3{1, 1, 1};
    *n = 0;
    *s = nullptr;
    return 0;
}
void** __hipRegisterFatBinary(const void*) { static void* h; return &h; }
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void*, char*, const char*, unsigned, void*, void*, void*, void*, int*) {}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
}

namespace {

ipic_ctx* make(int substeps) {
    ipic_desc d{};
    d.nspecies = 1;
    for (int k = 0; k < 3; ++k) {
        d.n[k] = 8;
        d.cell_width[k] = 1.0;
    }
    d.dt = 0.1;
    d.c = 1.0;
    d.species[0].q = d.species[0].qom = -1.0;
    d.field_substeps = substeps;
    ipic_ctx* c = nullptr;
    if (ipic_gpu_create(&d, &c) != 0) {
        std::printf("create: %s\n", ipic_gpu_last_error(nullptr));
        std::exit(1);
    }
    return c;
}

int failed_step() {
    int failed = 0;
    for (int substeps : {0, 1, 2})
        for (int at = 1;; ++at) {  // refuse the first, second, ... launch of the step
            ipic_ctx* c = make(substeps);
            launches = 0;
            refuse = at;
            ipic_step_stats st{};
            const int rc = ipic_gpu_step(c, 2, &st);
            refuse = 0;
            bool left = false;
            if (rc != 0) {
                ++failed;
                ipic_field_state fs{};
                const int rv = ipic_gpu_field_state(c, &fs);
                left = rv == 0 && queued;
            }
            ipic_gpu_destroy(c);
            if (left) {
                std::printf("%d substeps, launch %d refused: the view is given out with work queued\n", substeps, at);
                return 1;
            }
            if (rc == 0) break;  // the step has fewer launches
        }
    std::printf("%d failed steps\n", failed);
    return failed > 10 ? 0 : 1;
}

int create() {
    int device[2];
    for (int substeps : {1, 2}) {
        device_allocs = pinned_allocs = 0;
        ipic_gpu_destroy(make(substeps));
        device[substeps - 1] = device_allocs;
        if (pinned_allocs != 1) {
            std::printf("%d pinned allocations\n", pinned_allocs);
            return 1;
        }
    }
    std::printf("%d and %d device allocations\n", device[0], device[1]);
    return device[0] == device[1] ? 0 : 1;
}

}  // namespace

int main(int argc, char** argv) {
    if (argc == 2 && !std::strcmp(argv[1], "--failed-step")) return failed_step();
    if (argc == 2 && !std::strcmp(argv[1], "--create")) return create();
    return 2;
}
