// See host_io.hpp.
#include "host_io.hpp"

#include <algorithm>
#include <atomic>
#include <chrono>
#include <cstring>
#include <exception>
#include <mutex>
#include <thread>

#if !defined(__HIP_DEVICE_COMPILE__)
#include <emmintrin.h>
#endif

namespace xnor_hip {

namespace {

// Bytes a thread copies at a time; transfers over the link are whole slices, up to a block of them.
constexpr size_t SLICE = 256 << 10;
constexpr size_t BLOCK_SLICES = 8, BLOCK = BLOCK_SLICES * SLICE;
// Blocks of pinned memory that one direction of a pass goes through, in turn, and that are kept for
// later passes.
constexpr size_t RING_BLOCKS = 8, RING_SLICES = RING_BLOCKS * BLOCK_SLICES;
constexpr size_t POOL_BLOCKS = 128;
constexpr size_t FLAG_BYTES = 256; // of a pass's flags
// Tensors in pinned memory go straight to a copy engine from this size on, smaller ones through the
// pinned buffers like any other (us a pass, in place / through the buffers, both tensors pinned:
// 0.26 + 0.17 MB 46 / 46, 0.5 + 0.35 MB 56 / 63, 8.3 + 5.5 MB 286 / 360, 66 + 44 MB 2004 / 2326;
// one of them, 0.26 MB in 50 / 45, 66 MB in 2179 / 2317).
constexpr size_t PINNED_DIRECT = 256 << 10;

typedef uint32_t v4u __attribute__((ext_vector_type(4)));

// n 16-byte units from pinned to device memory or back; then, with a flag (pinned), *flag = arrived
// for the host to see that all of them are there.  Bound by the link, which sixteen workgroups
// saturate (51 GB/s; with 64 the flush per workgroup costs more, 47).  `waiting` counts workgroups
// and is left at 0.
__global__ __launch_bounds__(256)
void link_copy_kernel(const v4u *__restrict__ from, v4u *__restrict__ to, const size_t n,
        uint32_t *__restrict__ waiting, uint32_t *__restrict__ flag, const uint32_t arrived) {
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
            __hip_atomic_store(flag, arrived, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
        }
    }
}

// ---- pinned memory --------------------------------------------------------------------------
std::mutex pool_mu;
int descriptors = 0;

// Pinned pieces of one size that nobody uses.
template <size_t BYTES, size_t MOST>
struct Pool {
    char *piece[MOST];
    size_t pieces = 0;

    char *take() {
        {
            std::lock_guard<std::mutex> lock(pool_mu);
            if (pieces > 0) return piece[--pieces];
        }
        void *p = nullptr;
        if (hipHostMalloc(&p, BYTES, hipHostMallocPortable) == hipSuccess)
            return static_cast<char *>(p);
        (void)hipGetLastError();
        return nullptr;
    }
    void give(char *p) {
        {
            std::lock_guard<std::mutex> lock(pool_mu);
            if (descriptors > 0 && pieces < MOST) {
                piece[pieces++] = p;
                return;
            }
        }
        (void)hipHostFree(p);
    }
    void clear() { // under the lock
        while (pieces > 0) (void)hipHostFree(piece[--pieces]);
    }
};
Pool<BLOCK, POOL_BLOCKS> block_pool;
Pool<FLAG_BYTES, POOL_BLOCKS> flag_pool;

// The blocks of one direction of a pass, used in turn.  Slice i of the tensor lies in place
// i % slices().
struct Ring {
    char *block[RING_BLOCKS];
    size_t blocks = 0;

    Ring() = default;
    Ring(const Ring &) = delete;
    ~Ring() {
        while (blocks > 0) block_pool.give(block[--blocks]);
    }
    // As many blocks as the bytes fill, or as many as there are to be had; false without any.
    bool take(size_t bytes) {
        const size_t want = std::min((bytes + BLOCK - 1) / BLOCK, RING_BLOCKS);
        while (blocks < want && (block[blocks] = block_pool.take()) != nullptr) blocks++;
        return blocks > 0;
    }
    size_t slices() const { return blocks * BLOCK_SLICES; }
    char *slice(size_t i) const {
        return block[i / BLOCK_SLICES % blocks] + i % BLOCK_SLICES * SLICE;
    }
};

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

// One wait for something that arrives by itself, in turns: each call of turn() is one look later.
// Looks without a pause for as long as `spin` (what an ordinary pass waits is shorter than that, and a
// sleeping thread is woken 60 us late), then sleeps a sixteenth of the time waited so far between
// looks: behind 53 ms of other work on the stream a pass took its four threads 213 ms of processor time.
class Wait {
public:
    explicit Wait(std::chrono::microseconds spin) : spin_(spin) {}
    void over() { turns_ = 0; }
    bool turn() { // true after a sleep
        if (turns_++ == 0) since_ = std::chrono::steady_clock::now();
        relax();
        if (turns_ % 16 != 0) return false;
        const auto waited = std::chrono::steady_clock::now() - since_;
        if (waited < spin_) return false;
        std::this_thread::sleep_for(std::min<std::chrono::steady_clock::duration>(
                waited / 16, std::chrono::microseconds(500)));
        turns_ = 15; // (the next turn sleeps again)
        return true;
    }

private:
    const std::chrono::steady_clock::duration spin_;
    std::chrono::steady_clock::time_point since_;
    unsigned turns_ = 0;
};
constexpr std::chrono::microseconds SPIN_CALLER(2000), SPIN_HELPER(300);

// What the copying threads share.  All counts are slices from the front of a tensor.
struct Work {
    Ring in, out;
    uint32_t *flags = nullptr; // pinned, raised by the transfer kernels
    const char *src = nullptr;
    char *dst = nullptr;
    size_t in_bytes = 0, out_bytes = 0, in_slices = 0, out_slices = 0;
    std::atomic<size_t> next_in{0}, next_out{0}; // handed out to threads
    std::atomic<size_t> in_room{0};              // may be copied into the ring
    std::atomic<size_t> out_there{0};            // have reached the ring
    // the last slice (its number + 1) that has been copied into a place of the ring, or out of it
    std::atomic<size_t> in_copied[RING_SLICES], out_copied[RING_SLICES];
    std::atomic<bool> stop{false};

    Work() {
        for (size_t i = 0; i < RING_SLICES; i++) in_copied[i] = out_copied[i] = 0;
    }
    ~Work() {
        if (flags != nullptr) flag_pool.give(reinterpret_cast<char *>(flags));
    }
    bool copy_in_slice() {
        size_t i = next_in.load(std::memory_order_relaxed);
        do {
            if (i >= in_room.load(std::memory_order_acquire)) return false;
        } while (!next_in.compare_exchange_weak(i, i + 1));
        copy_streaming(in.slice(i), src + i * SLICE, std::min(SLICE, in_bytes - i * SLICE));
        in_copied[i % in.slices()].store(i + 1, std::memory_order_release);
        return true;
    }
    bool copy_out_slice() {
        size_t i = next_out.load(std::memory_order_relaxed);
        do {
            if (i >= out_there.load(std::memory_order_acquire)) return false;
        } while (!next_out.compare_exchange_weak(i, i + 1));
        memcpy(dst + i * SLICE, out.slice(i), std::min(SLICE, out_bytes - i * SLICE));
        out_copied[i % out.slices()].store(i + 1, std::memory_order_release);
        return true;
    }
    void help() { // until every slice has been handed out
        Wait wait(SPIN_HELPER);
        while (!stop.load(std::memory_order_relaxed)) {
            if (copy_in_slice() || copy_out_slice()) {
                wait.over();
                continue;
            }
            if (next_in.load(std::memory_order_relaxed) >= in_slices
                    && next_out.load(std::memory_order_relaxed) >= out_slices)
                return;
            wait.turn();
        }
    }
};

} // namespace

Memory memory_of(const void *p) {
    hipPointerAttribute_t attr;
    if (hipPointerGetAttributes(&attr, p) != hipSuccess) {
        (void)hipGetLastError(); // plain host memory: clear the sticky error
        return Memory::pageable;
    }
    return attr.type == hipMemoryTypeDevice || attr.type == hipMemoryTypeManaged ? Memory::device
        : attr.type == hipMemoryTypeHost ? Memory::pinned : Memory::pageable;
}

void host_io_descriptor_created() {
    std::lock_guard<std::mutex> lock(pool_mu);
    descriptors++;
}

void host_io_descriptor_destroyed() {
    std::lock_guard<std::mutex> lock(pool_mu);
    if (--descriptors > 0) return;
    block_pool.clear();
    flag_pool.clear();
}

HostIo::~HostIo() {
    if (waiting_ != nullptr) (void)hipFree(waiting_);
}

// Device memory that the transfer kernels need.
bool HostIo::prepare(hipStream_t stream) {
    if (waiting_ != nullptr) return true;
    // (cleared on the stream of the kernels that count in it)
    if (hipMalloc((void **)&waiting_, sizeof(uint32_t)) == hipSuccess
            && hipMemsetAsync(waiting_, 0, sizeof(uint32_t), stream) == hipSuccess)
        return true;
    (void)hipGetLastError();
    if (waiting_ != nullptr) (void)hipFree(waiting_);
    waiting_ = nullptr;
    return false;
}

bool HostIo::move(hipStream_t stream, const char *src, Memory src_memory, size_t in_bytes,
        char *dev_in, char *dst, Memory dst_memory, size_t out_bytes, const char *dev_out,
        bool (*compute)(void *), void *context) {
    hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(stream, &capture) != hipSuccess)
        (void)hipGetLastError(); // (no later call should report it)
    else if (capture != hipStreamCaptureStatusNone)
        return false; // nothing would arrive before the graph runs
    // Directions that the runtime copies by itself: what the user has pinned needs no copy on this
    // side, and without pinned memory of our own the runtime's staging has to do.
    Work w;
    bool direct_in = in_bytes >= PINNED_DIRECT && src_memory == Memory::pinned;
    bool direct_out = out_bytes >= PINNED_DIRECT && dst_memory == Memory::pinned;
    if ((in_bytes > 0 && !direct_in) || (out_bytes > 0 && !direct_out)) {
        if (prepare(stream)) w.flags = reinterpret_cast<uint32_t *>(flag_pool.take());
        const bool ready = w.flags != nullptr;
        if (ready) memset(w.flags, 0, FLAG_BYTES);
        if (in_bytes > 0 && !direct_in) direct_in = !(ready && w.in.take(in_bytes));
        if (out_bytes > 0 && !direct_out) direct_out = !(ready && w.out.take(out_bytes));
    }
    w.src = src;
    w.dst = dst;
    w.in_bytes = direct_in ? 0 : in_bytes;
    w.out_bytes = direct_out ? 0 : out_bytes;
    w.in_slices = (w.in_bytes + SLICE - 1) / SLICE;
    w.out_slices = (w.out_bytes + SLICE - 1) / SLICE;
    size_t in_room = std::min(w.in_slices, w.in.slices());
    w.in_room = in_room;
    const size_t half_ring = std::max<size_t>(w.in.blocks / 2, 1) * BLOCK_SLICES;
    // slices of the input and of the output that have arrived
    uint32_t *const in_flag = w.flags, *const out_flag = w.flags + FLAG_BYTES / 8;
    bool ok = !direct_in
        || hipMemcpyAsync(dev_in, src, in_bytes, hipMemcpyHostToDevice, stream) == hipSuccess;
    auto send = [&](const void *from, void *to, size_t bytes, uint32_t *flag, size_t arrived) {
        const size_t n = (bytes + 15) / 16;
        hipLaunchKernelGGL(link_copy_kernel, dim3((unsigned)std::min<size_t>((n + 255) / 256, 16)),
                dim3(256), 0, stream, static_cast<const v4u *>(from), static_cast<v4u *>(to), n,
                waiting_, flag, (uint32_t)arrived);
        ok = ok && hipGetLastError() == hipSuccess;
    };
    // Helpers share the copying; starting one takes the caller 10 us, which a megabyte or two of
    // copying pays for (8.3 + 5.5 MB with 0, 1, 2, 3 helpers: 500, 396, 383, 372 us).
    std::thread helpers[3];
    int started = 0;
    const size_t total = w.in_bytes + w.out_bytes;
    int helpers_wanted = total >= (8u << 20) ? 3 : total >= (4u << 20) ? 2 : total >= (2u << 20) ? 1 : 0;
    size_t in_there = 0, in_sent = 0; // input slices in the ring; on their way
    // output slices on their way; in the ring; in the user's memory
    size_t out_sent = 0, out_there = 0, out_done = 0;
    bool computed = false;
    Wait wait(SPIN_CALLER);
    while (ok) {
        while (in_there < w.in_slices && w.in_copied[in_there % w.in.slices()].load(
                        std::memory_order_acquire) == in_there + 1)
            in_there++;
        // pieces grow with what has already been sent: the link starts early
        const size_t in_block = BLOCK_SLICES - in_sent % BLOCK_SLICES; // to the end of the block
        const size_t in_have = std::min(in_there - in_sent, in_block);
        if (in_have > 0 && (in_there == w.in_slices
                    || in_have >= std::min(in_block, std::max<size_t>(in_sent, 1)))) {
            const size_t at = in_sent * SLICE, end = in_sent + in_have;
            // its half of the ring is waited for, or the call's end is (a flag with every piece
            // costs a pass with 266 MB of input 1.4 %)
            const bool told = (end % half_ring == 0 && end - half_ring + w.in.slices() < w.in_slices)
                || (end == w.in_slices && out_bytes == 0);
            send(w.in.slice(in_sent), dev_in + at, std::min(in_have * SLICE, w.in_bytes - at),
                    told ? in_flag : nullptr, end);
            in_sent = end;
            continue;
        }
        if (in_room < w.in_slices) {
            const size_t room = std::min<size_t>(w.in_slices,
                    w.in.slices() + __atomic_load_n(in_flag, __ATOMIC_ACQUIRE));
            // (told when it changes: the helpers read it)
            if (room != in_room) w.in_room.store(in_room = room, std::memory_order_release);
        }
        if (!computed && in_sent == w.in_slices) {
            ok = compute(context);
            computed = true;
            if (direct_out)
                ok = ok && hipMemcpyAsync(dst, dev_out, out_bytes, hipMemcpyDeviceToHost, stream)
                        == hipSuccess;
            continue;
        }
        while (out_done < w.out_slices && w.out_copied[out_done % w.out.slices()].load(
                        std::memory_order_acquire) == out_done + 1)
            out_done++;
        if (computed && out_sent < w.out_slices) { // the last pieces get smaller
            const size_t room = BLOCK_SLICES - out_sent % BLOCK_SLICES; // to the end of the block
            size_t n = std::min(room, std::max<size_t>((w.out_slices - out_sent) / 2, 1));
            if (n > 1 && n + 1 == room) n = room; // (no piece for a slice left in the block)
            if (out_sent + n <= out_done + w.out.slices()) {
                const size_t at = out_sent * SLICE;
                send(dev_out + at, w.out.slice(out_sent), std::min(n * SLICE, w.out_bytes - at),
                        out_flag, out_sent + n);
                out_sent += n;
                continue;
            }
        }
        if (out_there < out_sent) {
            const size_t there = __atomic_load_n(out_flag, __ATOMIC_ACQUIRE);
            if (there != out_there)
                w.out_there.store(out_there = there, std::memory_order_release);
        }
        for (; helpers_wanted > 0 && (in_sent > 0 || computed); helpers_wanted--) { // (the link is busy)
            try {
                helpers[started] = std::thread([&w] { w.help(); });
                started++;
            } catch (const std::exception &) { // none to be had: the caller copies alone
                helpers_wanted = 1;
            }
        }
        if (w.copy_in_slice() || w.copy_out_slice()) {
            wait.over();
            continue;
        }
        if (computed && out_done == w.out_slices
                && (w.in_slices == 0 || out_bytes > 0
                    || __atomic_load_n(in_flag, __ATOMIC_ACQUIRE) == w.in_slices))
            break;
        // nothing to do but wait for a flag: a kernel that failed raises none
        if (wait.turn()) {
            const hipError_t e = hipStreamQuery(stream);
            ok = e == hipSuccess || e == hipErrorNotReady;
        }
    }
    w.stop = true;
    for (int i = 0; i < started; i++) helpers[i].join();
    // The runtime's copies raise no flag; and after a failure nothing of this call may still use
    // the blocks (if even that cannot be waited for, they are not used again).
    if (direct_in || direct_out || !ok) {
        if (hipStreamSynchronize(stream) != hipSuccess) {
            ok = false;
            w.in.blocks = w.out.blocks = 0;
            w.flags = nullptr;
        }
        if (!ok) (void)hipGetLastError();
    }
    return ok;
}

} // namespace xnor_hip
