// See host_io.hpp.
#include "host_io.hpp"

#include <algorithm>
#include <atomic>
#include <cstring>
#include <memory>
#include <mutex>
#include <system_error>
#include <thread>

#if !defined(__HIP_DEVICE_COMPILE__)
#include <emmintrin.h>
#endif

namespace xnor_hip {

namespace {

// Bytes of one transfer over the link at most, and at either end of the call, where nothing else
// is under way while a piece is copied between the user's memory and the pinned buffer.
constexpr size_t PIECE = 2 << 20, END_PIECE = 256 << 10;
constexpr size_t SLICE = 256 << 10; // bytes a thread copies at a time
// Tensors in pinned memory go straight to a copy engine from this size on, smaller ones through the
// pinned buffers like any other (us a pass, in place / through the buffers, both tensors pinned:
// 0.26 + 0.17 MB 46 / 46, 0.5 + 0.35 MB 56 / 63, 8.3 + 5.5 MB 286 / 360, 66 + 44 MB 2004 / 2326;
// one of them, 0.26 MB in 50 / 45, 66 MB in 2179 / 2317).
constexpr size_t PINNED_DIRECT = 256 << 10;
constexpr size_t POOL_MOST = 256u << 20;

typedef uint32_t v4u __attribute__((ext_vector_type(4)));

// n 16-byte units from pinned to device memory or back; then, with a flag (pinned), *flag = 1 for
// the host to see that all of them have arrived.  Bound by the link, which sixteen workgroups
// saturate (51 GB/s; with 64 the flush per workgroup costs more, 47).  `waiting` counts workgroups
// and is left at 0.
__global__ __launch_bounds__(256)
void link_copy_kernel(const v4u *__restrict__ from, v4u *__restrict__ to, const size_t n,
        uint32_t *__restrict__ waiting, uint32_t *__restrict__ flag) {
    const size_t stride = (size_t)gridDim.x * 256;
    size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    for (; i + 3 * stride < n; i += 4 * stride) {
        const v4u a = from[i], b = from[i + stride], c = from[i + 2 * stride],
                  d = from[i + 3 * stride];
        to[i] = a;
        to[i + stride] = b;
        to[i + 2 * stride] = c;
        to[i + 3 * stride] = d;
    }
    for (; i < n; i += stride) to[i] = from[i];
    if (flag == nullptr) return; // the stream orders what follows
    __syncthreads();
    if (threadIdx.x == 0) {
        __threadfence_system(); // out of this XCD's L2
        if (atomicAdd(waiting, 1u) == gridDim.x - 1) {
            *waiting = 0;
            __threadfence_system();
            __hip_atomic_store(flag, 1u, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
        }
    }
}

// ---- pinned buffers -------------------------------------------------------------------------
struct Pinned { char *at; size_t bytes; };
std::mutex pool_mu;
std::vector<Pinned> pool; // free ones
size_t pool_bytes = 0;
int descriptors = 0;

char *pinned_get(size_t bytes, size_t *got) {
    {
        std::lock_guard<std::mutex> lock(pool_mu);
        int best = -1;
        for (size_t i = 0; i < pool.size(); i++)
            if (pool[i].bytes >= bytes && pool[i].bytes <= 4 * bytes
                    && (best < 0 || pool[i].bytes < pool[best].bytes))
                best = (int)i;
        if (best >= 0) {
            const Pinned p = pool[best];
            pool.erase(pool.begin() + best);
            pool_bytes -= p.bytes;
            *got = p.bytes;
            return p.at;
        }
    }
    void *p = nullptr;
    if (hipHostMalloc(&p, bytes, hipHostMallocPortable) != hipSuccess) {
        (void)hipGetLastError();
        return nullptr;
    }
    *got = bytes;
    return static_cast<char *>(p);
}

// True for memory that the copy engines read and write in place (the user pinned it).
bool pinned(const void *p) {
    hipPointerAttribute_t attr;
    if (hipPointerGetAttributes(&attr, p) == hipSuccess) return attr.type == hipMemoryTypeHost;
    (void)hipGetLastError(); // plain host memory: clear the sticky error
    return false;
}

void pinned_put(char *at, size_t bytes) {
    if (at == nullptr) return;
    {
        std::lock_guard<std::mutex> lock(pool_mu);
        if (descriptors > 0 && pool_bytes + bytes <= POOL_MOST) {
            pool.push_back({at, bytes});
            pool_bytes += bytes;
            return;
        }
    }
    (void)hipHostFree(at);
}

#if !defined(__HIP_DEVICE_COMPILE__)
inline void relax() { _mm_pause(); }

// Into the pinned buffer past the caches: nobody on this side reads it again, and ordinary stores
// would read every line before they write it (8.3 MB with three helpers: the whole pass
// 391 -> 372 us, 23 MB: 701 -> 564).  `to` is 16-byte aligned.
void copy_streaming(char *to, const char *from, size_t bytes) {
    size_t i = 0;
    for (; i + 64 <= bytes; i += 64) {
        const __m128i *s = reinterpret_cast<const __m128i *>(from + i);
        __m128i *d = reinterpret_cast<__m128i *>(to + i);
        const __m128i v0 = _mm_loadu_si128(s), v1 = _mm_loadu_si128(s + 1),
                      v2 = _mm_loadu_si128(s + 2), v3 = _mm_loadu_si128(s + 3);
        _mm_stream_si128(d, v0);
        _mm_stream_si128(d + 1, v1);
        _mm_stream_si128(d + 2, v2);
        _mm_stream_si128(d + 3, v3);
    }
    memcpy(to + i, from + i, bytes - i);
    _mm_sfence();
}
#else // (the device pass parses the host code and runs none of it)
inline void relax() {}
void copy_streaming(char *, const char *, size_t) {}
#endif

// What the copying threads share.
struct Work {
    const char *src;
    char *pin_in;
    size_t in_bytes;
    char *dst;
    const char *pin_out;
    size_t out_bytes;
    std::atomic<size_t> next_in{0}, next_out{0}; // bytes handed out to threads
    std::atomic<size_t> out_ready{0};            // output bytes that have reached pin_out
    std::atomic<size_t> out_done{0};             // ... and the user's memory
    std::unique_ptr<std::atomic<bool>[]> slice_in; // input slices that have reached pin_in
    std::atomic<bool> stop{false};

    bool copy_in_slice() {
        size_t at = next_in.load(std::memory_order_relaxed);
        do {
            if (at >= in_bytes) return false;
        } while (!next_in.compare_exchange_weak(at, std::min(at + SLICE, in_bytes)));
        copy_streaming(pin_in + at, src + at, std::min(SLICE, in_bytes - at));
        slice_in[at / SLICE].store(true, std::memory_order_release);
        return true;
    }
    bool copy_out_slice() {
        size_t at = next_out.load(std::memory_order_relaxed), end;
        do {
            const size_t ready = out_ready.load(std::memory_order_acquire);
            if (at >= ready) return false;
            end = std::min(at + SLICE, ready);
        } while (!next_out.compare_exchange_weak(at, end));
        memcpy(dst + at, pin_out + at, end - at);
        out_done.fetch_add(end - at, std::memory_order_release);
        return true;
    }
    void help() { // until every byte has been handed out
        while (!stop.load(std::memory_order_relaxed)) {
            if (copy_in_slice() || copy_out_slice()) continue;
            if (next_in.load(std::memory_order_relaxed) >= in_bytes
                    && next_out.load(std::memory_order_relaxed) >= out_bytes)
                return;
            relax();
        }
    }
};

} // namespace

void host_io_descriptor_created() {
    std::lock_guard<std::mutex> lock(pool_mu);
    descriptors++;
}

void host_io_descriptor_destroyed() {
    std::vector<Pinned> all;
    {
        std::lock_guard<std::mutex> lock(pool_mu);
        if (--descriptors > 0) return;
        all.swap(pool);
        pool_bytes = 0;
    }
    for (const Pinned &p : all) (void)hipHostFree(p.at);
}

HostIo::~HostIo() {
    pinned_put(pin_in_, pin_in_bytes_);
    pinned_put(pin_out_, pin_out_bytes_);
    pinned_put(reinterpret_cast<char *>(flags_), flag_bytes_);
    if (waiting_ != nullptr) (void)hipFree(waiting_);
}

bool HostIo::prepare(size_t in_bytes, size_t out_bytes, size_t flags) {
    auto want = [](char *&at, size_t &have, size_t bytes) {
        bytes = (bytes + 4095) & ~(size_t)4095;
        if (have >= bytes) return true;
        pinned_put(at, have);
        have = 0;
        at = pinned_get(bytes, &have);
        return at != nullptr;
    };
    char *f = reinterpret_cast<char *>(flags_);
    const bool ok = want(pin_in_, pin_in_bytes_, in_bytes)
        && want(pin_out_, pin_out_bytes_, out_bytes) && want(f, flag_bytes_, flags * 4);
    flags_ = reinterpret_cast<uint32_t *>(f);
    if (!ok) return false;
    memset(flags_, 0, flags * 4);
    if (waiting_ == nullptr) {
        if (hipMalloc((void **)&waiting_, sizeof(uint32_t)) != hipSuccess) return false;
        if (hipMemset(waiting_, 0, sizeof(uint32_t)) != hipSuccess) return false;
    }
    return true;
}

bool HostIo::run(hipStream_t stream, const char *src, size_t in_bytes, char *dev_in, char *dst,
        size_t out_bytes, const char *dev_out, const std::function<bool()> &compute) {
    // what the user has pinned needs no copy on this side
    const bool direct_in = in_bytes >= PINNED_DIRECT && pinned(src);
    const bool direct_out = out_bytes >= PINNED_DIRECT && pinned(dst);
    const size_t staged_in = direct_in ? 0 : in_bytes, staged_out = direct_out ? 0 : out_bytes;
    // output pieces end at multiples of 16 bytes, the last ones get smaller
    std::vector<size_t> out_ends;
    for (size_t at = 0; at < staged_out;) {
        const size_t left = staged_out - at;
        size_t n = left <= END_PIECE ? left : std::min(PIECE, std::max(END_PIECE, left / 2));
        if (n < left) n &= ~(size_t)15;
        out_ends.push_back(at += n);
    }
    // raised by the last input piece when nothing returns
    const size_t last_flag = out_ends.size();
    if (!prepare(staged_in, staged_out, out_ends.size() + 1)) {
        (void)hipGetLastError();
        return false;
    }
    Work w;
    w.src = src;
    w.pin_in = pin_in_;
    w.in_bytes = staged_in;
    w.dst = dst;
    w.pin_out = pin_out_;
    w.out_bytes = staged_out;
    const size_t slices = (staged_in + SLICE - 1) / SLICE;
    w.slice_in.reset(new std::atomic<bool>[slices ? slices : 1]);
    for (size_t i = 0; i < slices; i++) w.slice_in[i] = false;
    bool ok = !direct_in
        || hipMemcpyAsync(dev_in, src, in_bytes, hipMemcpyHostToDevice, stream) == hipSuccess;
    auto send = [&](const void *from, void *to, size_t bytes, uint32_t *flag) {
        const size_t n = (bytes + 15) / 16;
        hipLaunchKernelGGL(link_copy_kernel, dim3((unsigned)std::min<size_t>((n + 255) / 256, 16)),
                dim3(256), 0, stream, static_cast<const v4u *>(from), static_cast<v4u *>(to), n,
                waiting_, flag);
        ok = ok && hipGetLastError() == hipSuccess;
    };
    // Helpers share the copying; starting one takes the caller 10 us, which a megabyte or two of
    // copying pays for (8.3 + 5.5 MB with 0, 1, 2, 3 helpers: 500, 396, 383, 372 us).
    std::vector<std::thread> helpers;
    const size_t total = staged_in + staged_out;
    int helpers_wanted = total >= (8u << 20) ? 3 : total >= (4u << 20) ? 2 : total >= (2u << 20) ? 1 : 0;
    size_t sent = 0, ready = 0; // input bytes on their way; slices in the pinned buffer, from the front
    bool computed = false;
    size_t first_out = 0;
    size_t idle = 0;
    while (ok) {
        while (ready < slices && w.slice_in[ready].load(std::memory_order_acquire)) ready++;
        const size_t have = std::min(ready * SLICE, staged_in);
        // pieces grow with what has already been sent: the link starts early
        if (sent < have && (have == staged_in || have - sent >= std::min(PIECE, std::max(sent, END_PIECE)))) {
            const size_t n = std::min(PIECE, have - sent);
            const bool last = sent + n == staged_in;
            send(pin_in_ + sent, dev_in + sent, n, last && out_bytes == 0 ? flags_ + last_flag : nullptr);
            sent += n;
            continue;
        }
        if (!computed && sent == staged_in) {
            ok = compute();
            computed = true;
            for (size_t i = 0, at = 0; ok && i < out_ends.size(); at = out_ends[i++])
                send(dev_out + at, pin_out_ + at, out_ends[i] - at, flags_ + i);
            if (direct_out)
                ok = ok && hipMemcpyAsync(dst, dev_out, out_bytes, hipMemcpyDeviceToHost, stream)
                        == hipSuccess;
            continue;
        }
        if (computed && first_out < out_ends.size()
                && __atomic_load_n(&flags_[first_out], __ATOMIC_ACQUIRE) != 0) {
            w.out_ready.store(out_ends[first_out++], std::memory_order_release);
            continue;
        }
        for (; helpers_wanted > 0 && (sent > 0 || computed); helpers_wanted--) { // (the link is busy)
            try {
                helpers.emplace_back([&w] { w.help(); });
            } catch (const std::system_error &) { // none to be had: the caller copies alone
                helpers_wanted = 1;
            }
        }
        if (w.copy_in_slice() || w.copy_out_slice()) {
            idle = 0;
            continue;
        }
        if (computed && w.out_done.load(std::memory_order_acquire) == staged_out
                && (staged_in == 0 || out_bytes > 0
                    || __atomic_load_n(&flags_[last_flag], __ATOMIC_ACQUIRE) != 0))
            break;
        relax();
        // nothing to do but wait for a flag: a kernel that failed raises none
        if (++idle % (1 << 16) == 0) {
            const hipError_t e = hipStreamQuery(stream);
            ok = e == hipSuccess || e == hipErrorNotReady;
        }
    }
    w.stop = true;
    for (std::thread &t : helpers) t.join();
    // the copy engines raise no flag; and after a failure nothing of this call may still use the
    // pinned buffers
    if (direct_in || direct_out || !ok) {
        if (hipStreamSynchronize(stream) != hipSuccess) ok = false;
        if (!ok) (void)hipGetLastError();
    }
    return ok;
}

} // namespace xnor_hip
