// Host tensors in and out of the device, piece by piece.
//
// A pageable buffer handed to hipMemcpyAsync goes through the runtime's own staging at 32 (in)
// and 18 GB/s (out).  Here the bytes go through blocks of pinned memory: the calling thread and up
// to three helpers copy slices between the user's memory and the blocks while a small kernel moves
// the pieces that are ready over the link (a kernel reaches 51 GB/s on pinned memory and costs a
// launch, where a copy engine costs 9 us per transfer), and flags in pinned memory tell the host
// what has come back (no stream or event to wait for).  A tensor that the user has pinned is moved
// by a copy engine, in place; where no memory can be pinned the runtime's staging takes over.  What
// bounds it is the link, in and then out.  Sending results back while input still arrives was built
// with a second stream and is not used: two kernels together move 76 GB/s, but what ties the
// streams together (events, or the host) cost more than that gained.
// AlexNet conv4, minibatch 32, 8.3 MB in and 5.5 MB out: 605 -> 375 us per forward pass.
#pragma once

#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

#include <type_traits>

namespace xnor_hip {

// Where a user's tensor lies: a kernel can use it in place (device or managed memory), the copy
// engines can, or neither.
enum class Memory { device, pinned, pageable };
Memory memory_of(const void *p); // asks the driver: 0.4 us

class HostIo {
public:
    HostIo() = default;
    ~HostIo();
    HostIo(const HostIo &) = delete;
    HostIo &operator=(const HostIo &) = delete;

    // Copies in_bytes from src to dev_in, has compute() enqueue the kernels on the stream, and
    // copies out_bytes from dev_out to dst (either tensor may be null with 0 bytes; neither lies on
    // the device).  The device buffers hold a multiple of 16 bytes.  Returns when dst is written, or without a dst when
    // the input has arrived; false on a HIP failure.
    template <class F>
    bool run(hipStream_t stream, const char *src, Memory src_memory, size_t in_bytes, char *dev_in,
            char *dst, Memory dst_memory, size_t out_bytes, const char *dev_out, F &&compute) {
        return move(stream, src, src_memory, in_bytes, dev_in, dst, dst_memory, out_bytes, dev_out,
                [](void *f) { return (bool)(*static_cast<std::remove_reference_t<F> *>(f))(); },
                &compute);
    }

private:
    uint32_t *waiting_ = nullptr; // device: workgroups of the transfer under way
    bool prepare(hipStream_t stream);
    bool move(hipStream_t stream, const char *src, Memory src_memory, size_t in_bytes,
            char *dev_in, char *dst, Memory dst_memory, size_t out_bytes, const char *dev_out,
            bool (*compute)(void *), void *context);
};

// A pass borrows its pinned blocks of 2 MB, at most eight for each direction, and gives them back
// for the next one, whichever descriptor's it is (allocating one takes most of a millisecond).  256
// MB at most are kept, and returned to the system when the last descriptor goes.
void host_io_descriptor_created();
void host_io_descriptor_destroyed();

} // namespace xnor_hip
