// Host-side plumbing of the calls that are not launches alone: scratch memory in stream order, pageable host buffers
// to and from the device, and a float handed from a kernel to the waiting host.
#pragma once
#include <mutex>

#include "common.hpp"

namespace bitnet {

// Device scratch of one call, taken and given back in the order of `stream`: nobody waits for the device, and the next
// call on the stream finds the memory again.  hipMalloc + hipFree of 4.4 MB take 27 us; from the pool 1 to 2 us.  The
// pool (one per device) keeps at most 64 MiB that nobody uses, the runtime gives the rest back.
class StreamScratch {
public:
    StreamScratch() = default;
    StreamScratch(const StreamScratch &) = delete;
    StreamScratch &operator=(const StreamScratch &) = delete;
    ~StreamScratch() { give_back(); }
    int alloc(size_t bytes, hipStream_t stream);
    // Behind the last launch that uses it.  Ahead of a wait for the stream, whose work then hides the 12 us this takes the host.
    void give_back()
    {
        if (ptr) (void)hipFreeAsync(ptr, stream_);
        ptr = nullptr;
    }
    void *ptr = nullptr;

private:
    hipStream_t stream_ = nullptr;
};

// Pageable host memory to the device through pinned chunks: the host copies a chunk, a kernel pulls it over the link while
// the host copies the next.  (4.4 MB: the link alone takes 85 us, the host's copy 56 us; one after the other, as the
// runtime does it, 138 us.  hipMemcpyAsync and an event per chunk cost the host more than they hide.)  What follows on the
// stream sees the data; the object holds the chunks, and `src` must stay, until the stream has passed them: done() after the
// caller's own synchronisation, or the destructor, which waits.  One upload at a time has the chunks; others, small ones, and all of
// them where pinned memory is not to be had, take the runtime's path.
class Upload {
public:
    Upload() = default;
    Upload(const Upload &) = delete;
    Upload &operator=(const Upload &) = delete;
    ~Upload();
    int copy(void *dst, const void *src, size_t bytes, hipStream_t stream);
    void done();

private:
    std::unique_lock<std::mutex> ring_;
    hipStream_t stream_ = nullptr;
    bool reading_ = false;
};
// The other way: returns with `dst` complete.  `scalar` (optional): one device float that comes along, into *scalar_host.
// (4.4 MB into pageable memory through hipMemcpy: 250 us.)
int download(void *dst, const void *src, size_t bytes, const float *scalar, float *scalar_host, hipStream_t stream);
// Up to MOST separate pieces of device memory moved by one launch (a copy through the runtime costs the host 5 to 6 us each:
// twelve requests gathered and scattered again, 130 us of a batch).
struct Pieces {
    static constexpr int MOST = 32;
    float *dst[MOST];
    const float *src[MOST];
    unsigned count[MOST];  // floats
};
hipError_t launch_move_pieces(const Pieces &pieces, int n, hipStream_t stream);
// How long the chunks (4 MiB a process) live: made by the first copy that wants them, given back when a last layer is destroyed
// and nothing was copied since the last layer before it was.  Making and freeing them takes 45 to 85 us, which a program that makes
// a layer, loads it, saves it and drops it, one after the other, does not pay each time (a GGUF tensor of 640 x 2560 through all
// four: 125 us with the chunks given back each time, 84 so; 2560 x 2560: 255 and 168; 6912 x 2560: 500 and 470).
void staging_retain();
void staging_release();

// A reduction's result for the waiting host, without a copy and a stream synchronisation behind it (about 12 us
// together): every workgroup of the launch stores its partial result and the ticket as one 8-byte word into pinned memory,
// and the host polls the words and combines them.  No atomics: 640 workgroups meeting in two device words took 12 us.
class HostParts {
public:
    static constexpr int MOST = 256;  // workgroups of one launch
    HostParts() = default;
    HostParts(const HostParts &) = delete;
    HostParts &operator=(const HostParts &) = delete;
    ~HostParts();
    int acquire();
    // Waits for `count` words and hands each lower half to `each`; a launch that never answers is an error.
    template <typename F>
    int wait(hipStream_t stream, int count, F &&each)
    {
        for (int i = 0; i < count; ++i) {
            unsigned bits = 0;
            int rc = wait_one(stream, i, &bits);
            if (rc != BITNET_HIP_OK) return rc;
            each(bits);
        }
        return BITNET_HIP_OK;
    }
    unsigned long long *answers = nullptr;  // device address of the pinned words
    unsigned ticket = 0;                    // what the upper half of an answer must hold

private:
    int wait_one(hipStream_t stream, int index, unsigned *bits);
    int slot_ = -1, device_ = 0;
    int spins_ = 0;
};

}  // namespace bitnet
