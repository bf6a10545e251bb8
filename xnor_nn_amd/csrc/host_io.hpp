// Host tensors in and out of the device, piece by piece.
//
// A pageable buffer handed to hipMemcpyAsync goes through the runtime's own staging at 32 (in)
// and 18 GB/s (out).  Here the bytes go through pinned buffers of this library: the calling
// thread and up to three helpers copy slices between the user's memory and the pinned buffers while a small
// kernel moves the pieces that are ready over the link (a kernel reaches 51 GB/s on pinned
// memory and costs a launch, where a copy engine costs 9 us per transfer), and flags in pinned
// memory tell the host what has come back (no stream or event to wait for).  A tensor that the
// user has pinned is moved by a copy engine, in place.  What bounds it is
// the link, in and then out.  Sending results back while input still arrives was built with a
// second stream and is not used: two kernels together move 76 GB/s, but what ties the streams
// together (events, or the host) cost more than that gained.
// AlexNet conv4, minibatch 32, 8.3 MB in and 5.5 MB out: 605 -> 375 us per forward pass.
#pragma once

#include <functional>

#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

namespace xnor_hip {

class HostIo {
public:
    HostIo() = default;
    ~HostIo();
    HostIo(const HostIo &) = delete;
    HostIo &operator=(const HostIo &) = delete;

    // Copies in_bytes from src to dev_in, has compute() enqueue the kernels on the stream, and
    // copies out_bytes from dev_out to dst (either tensor may be null with 0 bytes).  The device
    // buffers hold a multiple of 16 bytes.  Returns when dst is written, or without a dst when
    // the input has arrived; false on a HIP failure.
    bool run(hipStream_t stream, const char *src, size_t in_bytes, char *dev_in, char *dst,
            size_t out_bytes, const char *dev_out, const std::function<bool()> &compute);

private:
    char *pin_in_ = nullptr, *pin_out_ = nullptr;
    size_t pin_in_bytes_ = 0, pin_out_bytes_ = 0;
    uint32_t *flags_ = nullptr;   // pinned: one per piece of a call, raised by its transfer
    size_t flag_bytes_ = 0;
    uint32_t *waiting_ = nullptr; // device: workgroups of the transfer under way
    bool prepare(size_t in_bytes, size_t out_bytes, size_t flags);
};

// Pinned buffers are kept for the next descriptor that needs one (allocating one takes
// milliseconds), 256 MB at most, and given back to the system when the last descriptor goes.
void host_io_descriptor_created();
void host_io_descriptor_destroyed();

} // namespace xnor_hip
