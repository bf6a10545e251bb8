// HostIo (xnor_nn_amd/csrc/host_io.hip) on the CPU: its host code as it is, linked with these
// stand-ins for the HIP runtime.  A stream is a thread that works through a queue; the transfer
// kernel is replaced by what it does.  Usage: host_io_check CASE; prints what is wrong, if anything.
#include <time.h>

#include <atomic>
#include <chrono>
#include <condition_variable>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <deque>
#include <functional>
#include <map>
#include <mutex>
#include <string>
#include <thread>
#include <vector>

#include "host_io.hpp"

namespace {

// ---- the stream ---------------------------------------------------------------------------
struct Stream {
    std::mutex mu;
    std::condition_variable more, idle;
    std::deque<std::function<void()>> todo;
    bool busy = false, stop = false;
    std::thread worker{[this] { work(); }};
    void work() {
        std::unique_lock<std::mutex> l(mu);
        for (;;) {
            more.wait(l, [this] { return stop || !todo.empty(); });
            if (todo.empty()) return;
            auto f = std::move(todo.front());
            todo.pop_front();
            busy = true;
            l.unlock();
            f();
            l.lock();
            busy = false;
            if (todo.empty()) idle.notify_all();
        }
    }
    void put(std::function<void()> f) {
        std::lock_guard<std::mutex> l(mu);
        todo.push_back(std::move(f));
        more.notify_one();
    }
    void sync() {
        std::unique_lock<std::mutex> l(mu);
        idle.wait(l, [this] { return todo.empty() && !busy; });
    }
    bool done() {
        std::lock_guard<std::mutex> l(mu);
        return todo.empty() && !busy;
    }
    ~Stream() {
        { std::lock_guard<std::mutex> l(mu); stop = true; more.notify_all(); }
        worker.join();
    }
};
Stream *stream_of(hipStream_t s) { return reinterpret_cast<Stream *>(s); }

// ---- memory -------------------------------------------------------------------------------
std::mutex mem_mu;
std::map<const char *, size_t> host_blocks; // pinned, the library's and the user's
size_t host_bytes = 0, host_bytes_most = 0;
std::atomic<long> host_allocations_left{1 << 30};
std::atomic<int> launches{0}, engine_copies{0};
std::atomic<bool> fail_queries{false}, capturing{false};

bool in_pinned(const char *p) {
    std::lock_guard<std::mutex> l(mem_mu);
    auto it = host_blocks.upper_bound(p);
    if (it == host_blocks.begin()) return false;
    --it;
    return p < it->first + it->second;
}

thread_local struct { dim3 grid, block; size_t lds; hipStream_t stream; } config;

} // namespace

extern "C" {
char __hip_fatbin[16];
void **__hipRegisterFatBinary(const void *) { static void *h; return &h; }
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *, char *, const char *, unsigned, void *, void *,
        void *, void *, int *) {}
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t lds, hipStream_t s) {
    config = {g, b, lds, s};
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *lds, hipStream_t *s) {
    *g = config.grid, *b = config.block, *lds = config.lds, *s = config.stream;
    return hipSuccess;
}
// link_copy_kernel(from, to, n, waiting, flag, arrived)
hipError_t hipLaunchKernel(const void *, dim3, dim3, void **args, size_t, hipStream_t s) {
    launches++;
    const char *from = *static_cast<const char **>(args[0]);
    char *to = *static_cast<char **>(args[1]);
    const size_t n = *static_cast<size_t *>(args[2]);
    uint32_t *flag = *static_cast<uint32_t **>(args[4]);
    const uint32_t arrived = *static_cast<uint32_t *>(args[5]);
    stream_of(s)->put([=] {
        memcpy(to, from, 16 * n);
        if (flag) __atomic_store_n(flag, arrived, __ATOMIC_RELEASE);
    });
    return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t bytes, unsigned) {
    if (host_allocations_left-- <= 0) return hipErrorOutOfMemory;
    if (posix_memalign(p, 4096, bytes) != 0) return hipErrorOutOfMemory;
    std::lock_guard<std::mutex> l(mem_mu);
    host_blocks[static_cast<char *>(*p)] = bytes;
    host_bytes += bytes;
    if (host_bytes > host_bytes_most) host_bytes_most = host_bytes;
    return hipSuccess;
}
hipError_t hipHostFree(void *p) {
    {
        std::lock_guard<std::mutex> l(mem_mu);
        auto it = host_blocks.find(static_cast<char *>(p));
        if (it == host_blocks.end()) abort();
        host_bytes -= it->second;
        host_blocks.erase(it);
    }
    free(p);
    return hipSuccess;
}
hipError_t hipMalloc(void **p, size_t bytes) { return (*p = malloc(bytes)) ? hipSuccess : hipErrorOutOfMemory; }
hipError_t hipFree(void *p) { free(p); return hipSuccess; }
hipError_t hipMemsetAsync(void *p, int v, size_t n, hipStream_t s) {
    stream_of(s)->put([=] { memset(p, v, n); });
    return hipSuccess;
}
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus *c) {
    *c = capturing ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
    return hipSuccess;
}
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipStreamQuery(hipStream_t s) {
    return fail_queries ? hipErrorUnknown : stream_of(s)->done() ? hipSuccess : hipErrorNotReady;
}
hipError_t hipStreamSynchronize(hipStream_t s) { stream_of(s)->sync(); return hipSuccess; }
hipError_t hipMemcpyAsync(void *to, const void *from, size_t n, hipMemcpyKind, hipStream_t s) {
    engine_copies++;
    stream_of(s)->put([=] { memcpy(to, from, n); });
    return hipSuccess;
}
hipError_t hipPointerGetAttributes(hipPointerAttribute_t *a, const void *p) {
    memset(a, 0, sizeof *a);
    a->type = in_pinned(static_cast<const char *>(p)) ? hipMemoryTypeHost : hipMemoryTypeUnregistered;
    return hipSuccess;
}
}

namespace {

std::atomic<int> wrong{0};
void check(bool ok, const char *what, size_t a = 0, size_t b = 0) {
    if (ok) return;
    printf("wrong: %s (%zu, %zu)\n", what, a, b);
    wrong++;
}

// The user's memory: pageable or pinned, at an odd address if asked for.
struct Tensor {
    std::vector<char> plain;
    char *at = nullptr, *pin = nullptr;
    size_t bytes;
    Tensor(size_t n, bool pinned, size_t shift = 0) : bytes(n) {
        if (pinned) {
            void *p = nullptr;
            if (hipHostMalloc(&p, n + shift + 16, 0) != hipSuccess) abort();
            pin = static_cast<char *>(p);
            at = pin + shift;
        } else {
            plain.resize(n + shift + 16);
            at = plain.data() + shift;
        }
    }
    ~Tensor() { if (pin) (void)hipHostFree(pin); }
};

unsigned char pattern(size_t i, unsigned seed) { return (unsigned char)((i * 2654435761u + seed) >> 13); }

double processor_seconds() { // of all threads
    timespec t;
    clock_gettime(CLOCK_PROCESS_CPUTIME_ID, &t);
    return t.tv_sec + 1e-9 * t.tv_nsec;
}
thread_local double run_seconds = 0; // of the last pass's call

// One pass: in_bytes in, every output byte an input byte (inverted) or a pattern, out_bytes out.
// expect: what run() has to return.
void pass(xnor_hip::HostIo &io, Stream &stream, size_t in_bytes, size_t out_bytes, unsigned seed,
        bool pin_in = false, bool pin_out = false, size_t shift = 0, bool expect = true) {
    Tensor in(in_bytes, pin_in, shift), out(out_bytes, pin_out, shift);
    std::vector<char> dev_in((in_bytes + 15) & ~(size_t)15), dev_out((out_bytes + 15) & ~(size_t)15);
    for (size_t i = 0; i < in_bytes; i++) in.at[i] = (char)pattern(i, seed);
    memset(out.at, 0x5A, out_bytes + 8);
    bool computed = false;
    const double before = processor_seconds();
    const bool ok = io.run(reinterpret_cast<hipStream_t>(&stream), in.at,
            xnor_hip::memory_of(in.at), in_bytes, dev_in.data(), out.at,
            xnor_hip::memory_of(out.at), out_bytes, dev_out.data(), [&] {
        computed = true;
        char *from = dev_in.data(), *to = dev_out.data();
        stream.put([=] {
            for (size_t i = 0; i < out_bytes; i++)
                to[i] = in_bytes ? (char)~from[i % in_bytes] : (char)pattern(i, seed);
        });
        return true;
    });
    run_seconds = processor_seconds() - before;
    check(ok == expect, "result of run", in_bytes, out_bytes);
    check(expect == false || computed, "compute was not called", in_bytes, out_bytes);
    if (!ok) return;
    if (out_bytes == 0) { // returns when the input has arrived
        for (size_t i = 0; i < in_bytes; i++)
            if (dev_in[i] != (char)pattern(i, seed)) { check(false, "input byte", in_bytes, i); return; }
        return;
    }
    for (size_t i = 0; i < out_bytes; i++) {
        const char want = in_bytes ? (char)~(char)pattern(i % in_bytes, seed) : (char)pattern(i, seed);
        if (out.at[i] != want) { check(false, "output byte", out_bytes, i); return; }
    }
    for (size_t i = 0; i < 8; i++) check(out.at[out_bytes + i] == 0x5A, "byte behind the output", out_bytes, i);
}

constexpr size_t MB = 1 << 20;

void pinned_tensors() {
    Stream stream;
    xnor_hip::HostIo io;
    pass(io, stream, 9 * MB + 12, 5 * MB + 4, 1, true, true, 4);
    check(launches == 0, "transfers through the library's buffers", launches);
    check(engine_copies == 2, "transfers in place", engine_copies);
    pass(io, stream, 9 * MB + 12, 0, 2, true, true, 4);
    pass(io, stream, 0, 5 * MB + 4, 3, true, true);
    check(launches == 0, "transfers through the library's buffers", launches);
    check(engine_copies == 4, "transfers in place", engine_copies);
    for (int which = 0; which < 4; which++)
        for (size_t n : {(size_t)4, 3 * MB + 20})
            pass(io, stream, n, 2 * MB - 8, 4 + which, which & 1, which & 2, 12);
}

void sizes() {
    Stream stream;
    xnor_hip::HostIo io;
    const size_t some[] = {0, 1, 4, 15, 16, MB / 4 - 1, MB / 4, MB / 4 + 1, MB / 2, 2 * MB - 4, 2 * MB,
                           2 * MB + 4, 5 * MB + 12, 16 * MB, 16 * MB + 4, 41 * MB + 8};
    unsigned seed = 0;
    for (size_t in : some)
        for (size_t out : some)
            if (in + out > 0 && in + out < 60 * MB) {
                seed++;
                pass(io, stream, in, out, seed, false, false, seed % 16);
            }
}

// The memory held is that of a pass's blocks, whatever the size of the tensors, and goes from pass to
// pass and from descriptor to descriptor.
void bounded() {
    Stream stream;
    for (int i = 0; i < 3; i++) {
        xnor_hip::HostIo io;
        pass(io, stream, 100 * MB, 60 * MB, i);
        pass(io, stream, 60 * MB, 0, i);
        pass(io, stream, 0, 70 * MB, i);
    }
    check(host_bytes_most <= 33 * MB, "pinned bytes at most", host_bytes_most);
}

// Without memory to pin the runtime copies; with some the blocks there are have to do.
void no_pinned_memory() {
    Stream stream;
    for (long left = 0; left < 6; left++) {
        xnor_hip::HostIo io;
        host_allocations_left = left;
        for (int i = 0; i < 3; i++) pass(io, stream, 9 * MB + 4, 7 * MB + 8, left + i);
        check(left >= 2 || engine_copies == 6 * (left + 1), "passes by the runtime", left, engine_copies);
        host_allocations_left = 1 << 30;
        xnor_hip::host_io_descriptor_destroyed(); // the blocks go back to the system
        xnor_hip::host_io_descriptor_created();
    }
}

void threads() {
    std::vector<std::thread> all;
    for (unsigned t = 0; t < 4; t++)
        all.emplace_back([t] {
            Stream stream;
            for (int i = 0; i < 6; i++) {
                xnor_hip::HostIo io;
                for (int j = 0; j < 3; j++) pass(io, stream, (3 + 5 * t + i) * MB + 4, 6 * MB - 4 * t, t + j);
            }
        });
    for (std::thread &t : all) t.join();
}

// A pass behind other work on the stream does not spend that time spinning.
void busy_stream() {
    Stream stream;
    xnor_hip::HostIo io;
    for (size_t in : {0 * MB, 9 * MB, 30 * MB})
        for (size_t out : {0 * MB, 9 * MB, 30 * MB}) {
            if (in + out == 0) continue;
            pass(io, stream, in, out, 1);
            const double alone = run_seconds;
            stream.put([] { std::this_thread::sleep_for(std::chrono::milliseconds(400)); });
            pass(io, stream, in, out, 2);
            check(run_seconds < alone + 0.1, "processor milliseconds behind 400 of other work",
                    (size_t)(1e3 * run_seconds), (size_t)(1e3 * alone));
        }
}

// A stream that has failed, and one that is being captured, end the call.
void refused() {
    Stream stream;
    xnor_hip::HostIo io;
    pass(io, stream, 3 * MB, MB, 1);
    capturing = true;
    const int before = launches;
    pass(io, stream, 3 * MB, MB, 2, false, false, 0, false);
    check(launches == before, "launches under capture", launches - before);
    capturing = false;
    fail_queries = true;
    stream.put([] { std::this_thread::sleep_for(std::chrono::milliseconds(300)); });
    pass(io, stream, 3 * MB, MB, 3, false, false, 0, false);
    fail_queries = false;
    pass(io, stream, 3 * MB, MB, 4);
}

} // namespace

int main(int argc, char **argv) {
    const std::map<std::string, void (*)()> cases = {
        {"pinned tensors", pinned_tensors}, {"sizes", sizes}, {"bounded", bounded},
        {"no pinned memory", no_pinned_memory}, {"threads", threads}, {"refused", refused},
        {"busy stream", busy_stream}};
    auto it = cases.find(argc > 1 ? argv[1] : "");
    if (it == cases.end()) {
        for (auto &c : cases) printf("%s\n", c.first.c_str());
        return 2;
    }
    xnor_hip::host_io_descriptor_created();
    it->second();
    xnor_hip::host_io_descriptor_destroyed();
    check(host_bytes == 0, "pinned bytes left behind", host_bytes);
    if (!wrong) printf("ok\n");
    return wrong ? 1 : 0;
}
