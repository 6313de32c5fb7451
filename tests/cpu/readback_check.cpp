/*
 * readback_check.cpp -- pic_readback.hip on the CPU, over a stand-in for the
 * few runtime calls it makes: two devices, whose memory is the host's, copies
 * that happen when their event or stream is waited for, an event that belongs to
 * the device current at its creation, and a wait that can be made to fail.
 *
 *   device    a context on the device that is not current
 *   failed    a call that fails leaves the caller's array as it was
 *   waiting   a call that waits for a long kernel leaves the CPUs alone
 */
#include <sys/resource.h>

#include <chrono>
#include <cstdio>
#include <cstring>
#include <map>
#include <string>
#include <thread>
#include <vector>

#include "pic_ctx.h"

struct ihipStream_t {
    int dev;
};
struct ihipEvent_t {
    int dev;
};

namespace {
struct Copy {
    void *dst;
    const void *src;
    size_t n;
};
std::vector<Copy> queued;
int current = 0;
bool fail = false;
int kernel_ms = 0;   /* what the first wait takes */

hipError_t drain() {
    std::this_thread::sleep_for(std::chrono::milliseconds(kernel_ms));
    kernel_ms = 0;
    if (fail) {
        queued.clear();
        return hipErrorUnknown;
    }
    for (const Copy &c : queued) std::memcpy(c.dst, c.src, c.n);
    queued.clear();
    return hipSuccess;
}
}  // namespace

extern "C" {
hipError_t hipGetDevice(int *d) {
    *d = current;
    return hipSuccess;
}
hipError_t hipSetDevice(int d) {
    if (d < 0 || d > 1) return hipErrorInvalidDevice;
    current = d;
    return hipSuccess;
}
hipError_t hipGetLastError(void) { return hipSuccess; }
hipError_t hipPointerGetAttributes(hipPointerAttribute_t *a, const void *) {
    a->type = hipMemoryTypeUnregistered;
    return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t n, unsigned) {
    *p = new char[n];
    return hipSuccess;
}
hipError_t hipHostFree(void *p) {
    delete[] (char *)p;
    return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) {
    *e = new ihipEvent_t{current};
    return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t e) {
    delete e;
    return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
    return e->dev == s->dev ? hipSuccess : hipErrorInvalidHandle;
}
hipError_t hipEventSynchronize(hipEvent_t) { return drain(); }
hipError_t hipStreamSynchronize(hipStream_t) { return drain(); }
hipError_t hipMemcpy(void *dst, const void *src, size_t n, hipMemcpyKind) {
    std::memcpy(dst, src, n);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void *dst, const void *src, size_t n, hipMemcpyKind, hipStream_t) {
    queued.push_back({dst, src, n});
    return hipSuccess;
}
}

namespace picx {
thread_local char g_hip_err[256];
int record_hip(hipError_t, const char *) { return PIC_ERR_HIP; }
}  // namespace picx

namespace {
int bad = 0;
void expect(bool ok, const char *what) {
    if (ok) return;
    std::printf("%s\n", what);
    bad = 1;
}

struct Box {
    ihipStream_t stream;
    pic_ctx c;
    explicit Box(int dev) : stream{dev} {
        c.dev = dev;
        c.stream = &stream;
        picx::readback_attach();
    }
    ~Box() { picx::readback_detach(); }
};

/* more than the ring holds, and no whole number of chunks */
constexpr long N = 3'000'001;

int device() {
    std::vector<int> src(N), dst(N, -1);
    for (long k = 0; k < N; k++) src[k] = (int)(k * 2654435761u);
    Box a(0), b(1);
    for (Box *x : {&b, &a, &b}) {
        dst.assign(N, -1);
        expect(picx::readback(&x->c, dst.data(), src.data(), N, picx::ReadAs::i32) == PIC_SUCCESS,
               "a context on the device that is not current cannot be read");
        expect(dst == src, "values differ");
        expect(current == 0, "the caller's current device changed");
    }
    return bad;
}

int failed() {
    const std::vector<double> src(N, 1.0);
    Box a(0);
    for (long n : {N, 300'000L}) {   /* through the ring, and one chunk */
        for (picx::ReadAs as : {picx::ReadAs::f64, picx::ReadAs::f32_to_f64}) {
            std::vector<double> dst(n, -1.0);
            fail = true;
            expect(picx::readback(&a.c, dst.data(), src.data(), n, as) == PIC_ERR_HIP,
                   "a failed copy is not reported");
            fail = false;
            expect(dst == std::vector<double>(n, -1.0), "a failed call wrote into the array");
            expect(picx::readback(&a.c, dst.data(), src.data(), n, picx::ReadAs::f64) == PIC_SUCCESS &&
                       dst == std::vector<double>(n, 1.0), "the next call does not read");
        }
    }
    return bad;
}

double cpu_seconds() {
    rusage r;
    getrusage(RUSAGE_SELF, &r);
    return r.ru_utime.tv_sec + r.ru_stime.tv_sec +
           1e-6 * (r.ru_utime.tv_usec + r.ru_stime.tv_usec);
}

int waiting() {
    const std::vector<double> src(N, 1.0);
    std::vector<double> dst(N, -1.0);
    Box a(0);
    kernel_ms = 1000;
    const double before = cpu_seconds();
    expect(picx::readback(&a.c, dst.data(), src.data(), N, picx::ReadAs::f64) == PIC_SUCCESS &&
               dst == src, "values differ");
    expect(cpu_seconds() - before < 0.5, "half a second of CPU time while a kernel runs");
    return bad;
}
}  // namespace

int main(int argc, char **argv) {
    const std::map<std::string, int (*)()> checks = {{"device", device}, {"failed", failed}, {"waiting", waiting}};
    return argc == 2 && checks.count(argv[1]) ? checks.at(argv[1])() : 2;
}
