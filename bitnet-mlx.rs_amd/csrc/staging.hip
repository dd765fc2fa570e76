// Scratch pools, pinned staging and host-visible results (see staging.hpp).
#include "staging.hpp"

#include <cstring>
#include <mutex>
#include <thread>

namespace bitnet {

namespace {

constexpr int MAX_DEVICES = 64;
constexpr size_t POOL_KEEP_BYTES = (size_t)64 << 20;

int current_device(int *device)
{
    BITNET_HIP_TRY(hipGetDevice(device));
    if (*device < 0 || *device >= MAX_DEVICES)
        return fail(BITNET_HIP_UNSUPPORTED, "device ordinal %d is beyond the %d this library keeps state for", *device, MAX_DEVICES);
    return BITNET_HIP_OK;
}

std::mutex pool_lock;
hipMemPool_t pools[MAX_DEVICES] = {};

int scratch_pool(hipMemPool_t *pool)
{
    int device = 0;
    int rc = current_device(&device);
    if (rc != BITNET_HIP_OK) return rc;
    std::lock_guard<std::mutex> guard(pool_lock);
    if (!pools[device]) {
        hipMemPoolProps props = {};
        props.allocType = hipMemAllocationTypePinned;
        props.location.type = hipMemLocationTypeDevice;
        props.location.id = device;
        hipMemPool_t made = nullptr;
        BITNET_HIP_TRY(hipMemPoolCreate(&made, &props));
        uint64_t keep = POOL_KEEP_BYTES;
        hipError_t e = hipMemPoolSetAttribute(made, hipMemPoolAttrReleaseThreshold, &keep);
        if (e != hipSuccess) {
            (void)hipMemPoolDestroy(made);
            return fail(BITNET_HIP_DEVICE_ERROR, "scratch pool: %s", hipGetErrorString(e));
        }
        pools[device] = made;
    }
    *pool = pools[device];
    return BITNET_HIP_OK;
}

// ---- pinned chunks ----
constexpr size_t CHUNK = (size_t)1 << 20;
constexpr int CHUNKS = 4;
constexpr size_t RING_MIN_BYTES = (size_t)256 << 10;  // below, one copy through the runtime is as fast

struct Ring {
    std::mutex lock;  // held by the copy that uses the chunks, and while they are made or freed
    uint8_t *base = nullptr, *on_device = nullptr;
    float *scalar = nullptr, *scalar_on_device = nullptr;  // behind the chunks
    hipEvent_t passed[CHUNKS] = {};
    int device = -1;
    bool used = false;  // since the last layer of some time before was destroyed

    void drop()
    {
        for (hipEvent_t &e : passed) {
            if (e) (void)hipEventDestroy(e);
            e = nullptr;
        }
        if (base) (void)hipHostFree(base);
        base = on_device = nullptr;
        device = -1;
    }
    // False where there is no pinned memory to be had: the copy then goes through the runtime, which needs none of ours.
    bool prepare()
    {
        int now = 0;
        if (hipGetDevice(&now) != hipSuccess) return false;
        if (base && device == now) return true;
        drop();
        void *mapped = nullptr;
        hipError_t e = hipHostMalloc(reinterpret_cast<void **>(&base), CHUNK * CHUNKS + 256, hipHostMallocDefault);
        if (e != hipSuccess) base = nullptr;
        else e = hipHostGetDevicePointer(&mapped, base, 0);
        for (hipEvent_t &ev : passed)
            if (e == hipSuccess) e = hipEventCreateWithFlags(&ev, hipEventDisableTiming);
        if (e != hipSuccess) {
            drop();
            (void)hipGetLastError();
            return false;
        }
        on_device = static_cast<uint8_t *>(mapped);
        scalar = reinterpret_cast<float *>(base + CHUNK * CHUNKS);
        scalar_on_device = reinterpret_cast<float *>(on_device + CHUNK * CHUNKS);
        device = now;
        return true;
    }
};
Ring ring;

// Takes the chunks for a copy of `bytes` at the device address `device_side`, where they pay and are there to be had.
bool take_ring(std::unique_lock<std::mutex> &mine, size_t bytes, const void *device_side)
{
    if (bytes < RING_MIN_BYTES || (reinterpret_cast<uintptr_t>(device_side) & 15) != 0 || !mine.try_lock()) return false;
    if (ring.prepare()) return ring.used = true;
    mine.unlock();
    return false;
}

std::mutex users_lock;
size_t users = 0;

// Moves `bytes` between the two memories, four 16-byte loads a thread in flight (dst and src 16-byte aligned; the last bytes one by
// one).  Bound by the link.
__global__ __launch_bounds__(256) void move_kernel(uint8_t *dst, const uint8_t *src, size_t bytes, const float *scalar, float *scalar_out)
{
    const size_t first = (size_t)blockIdx.x * 256 + threadIdx.x, stride = (size_t)gridDim.x * 256, whole = bytes >> 4;
    const uint4 *s4 = reinterpret_cast<const uint4 *>(src);
    uint4 *d4 = reinterpret_cast<uint4 *>(dst);
    size_t i = first;
    for (; i + 3 * stride < whole; i += 4 * stride) {
        uint4 v[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] = s4[i + j * stride];
#pragma unroll
        for (int j = 0; j < 4; ++j) d4[i + j * stride] = v[j];
    }
    for (; i < whole; i += stride) d4[i] = s4[i];
    for (size_t b = 16 * whole + first; b < bytes; b += stride) dst[b] = src[b];
    if (first == 0 && scalar) *scalar_out = *scalar;
}

hipError_t launch_move(uint8_t *dst, const uint8_t *src, size_t bytes, const float *scalar, float *scalar_out, hipStream_t stream)
{
    const size_t blocks = (bytes + 16383) / 16384;  // 16 KiB a workgroup: one batch of loads
    launch_kernel(move_kernel, dim3((unsigned)(blocks ? blocks : 1)), dim3(256), 0, stream, dst, src, bytes, scalar, scalar_out);
    return hipGetLastError();
}

// Piece blockIdx.y, 4096 floats a workgroup.
__global__ __launch_bounds__(256) void move_pieces_kernel(Pieces p)
{
    float *dst = p.dst[blockIdx.y];
    const float *src = p.src[blockIdx.y];
    const size_t count = p.count[blockIdx.y], begin = (size_t)blockIdx.x * 4096;
    if (begin >= count) return;
    const size_t end = begin + 4096 < count ? begin + 4096 : count;
    size_t i = begin + threadIdx.x;
    if (((reinterpret_cast<uintptr_t>(dst) | reinterpret_cast<uintptr_t>(src)) & 15) == 0) {
        const size_t whole = end & ~(size_t)3;
        for (size_t c = begin + 4 * (size_t)threadIdx.x; c < whole; c += 1024)
            *reinterpret_cast<float4 *>(dst + c) = *reinterpret_cast<const float4 *>(src + c);
        i = whole + threadIdx.x;
    }
    for (; i < end; i += 256) dst[i] = src[i];
}

// The host's copy of a chunk.  Both sides are cold (the link's data comes from memory, a caller's buffer is read or written
// once), so the stores bypass the cache: 27 us a MiB on the box measured, against 37 for memcpy; the link takes 19.
void stream_copy(uint8_t *dst, const uint8_t *src, size_t bytes)
{
    typedef long long v2ll __attribute__((vector_size(16), aligned(1)));
    typedef long long v2ll_aligned __attribute__((vector_size(16)));
    size_t i = 0;
    if ((reinterpret_cast<uintptr_t>(dst) & 15) == 0) {
        for (; i + 64 <= bytes; i += 64) {
            __builtin_prefetch(src + i + 2048, 0, 0);
            const v2ll *from = reinterpret_cast<const v2ll *>(src + i);
            const v2ll a = from[0], b = from[1], c = from[2], d = from[3];
            v2ll_aligned *to = reinterpret_cast<v2ll_aligned *>(dst + i);
            __builtin_nontemporal_store((v2ll_aligned)a, to);
            __builtin_nontemporal_store((v2ll_aligned)b, to + 1);
            __builtin_nontemporal_store((v2ll_aligned)c, to + 2);
            __builtin_nontemporal_store((v2ll_aligned)d, to + 3);
        }
        __atomic_thread_fence(__ATOMIC_SEQ_CST);  // in memory before a launch that reads it is enqueued
    }
    memcpy(dst + i, src + i, bytes - i);
}

// ---- results the host polls ----
constexpr int SLOTS = 64;  // calls that may wait at the same time; each holds one until its answer is there

struct SlotState {
    volatile unsigned long long *host = nullptr;
    unsigned long long *on_device = nullptr;
    unsigned tickets[SLOTS] = {};
    bool taken[SLOTS] = {};
};
std::mutex slots_lock;
SlotState slots[MAX_DEVICES];

int prepare_slots(SlotState &st)
{
    if (st.host) return BITNET_HIP_OK;
    constexpr size_t bytes = (size_t)SLOTS * HostParts::MOST * sizeof(unsigned long long);  // 128 KiB
    void *host = nullptr, *on_device = nullptr;
    BITNET_HIP_TRY(hipHostMalloc(&host, bytes, hipHostMallocDefault));
    hipError_t e = hipHostGetDevicePointer(&on_device, host, 0);
    if (e != hipSuccess) {
        (void)hipHostFree(host);
        return fail(BITNET_HIP_DEVICE_ERROR, "pinned result words: %s", hipGetErrorString(e));
    }
    memset(host, 0, bytes);
    st.on_device = static_cast<unsigned long long *>(on_device);
    st.host = static_cast<volatile unsigned long long *>(host);
    return BITNET_HIP_OK;
}

}  // namespace

hipError_t launch_move_pieces(const Pieces &pieces, int n, hipStream_t stream)
{
    unsigned most = 0;
    for (int i = 0; i < n; ++i) most = pieces.count[i] > most ? pieces.count[i] : most;
    if (most == 0) return hipSuccess;
    launch_kernel(move_pieces_kernel, dim3(most / 4096 + (most % 4096 != 0), (unsigned)n), dim3(256), 0, stream, pieces);
    return hipGetLastError();
}

int StreamScratch::alloc(size_t bytes, hipStream_t stream)
{
    hipMemPool_t pool = nullptr;
    int rc = scratch_pool(&pool);
    if (rc != BITNET_HIP_OK) return rc;
    hipError_t e = hipMallocFromPoolAsync(&ptr, bytes ? bytes : 1, pool, stream);
    if (e != hipSuccess) {
        ptr = nullptr;
        return fail(BITNET_HIP_MEMORY_ERROR, "scratch of %zu bytes: %s", bytes, hipGetErrorString(e));
    }
    stream_ = stream;
    return BITNET_HIP_OK;
}

int Upload::copy(void *dst, const void *src, size_t bytes, hipStream_t stream)
{
    std::unique_lock<std::mutex> mine(ring.lock, std::defer_lock);
    stream_ = stream;
    reading_ = true;
    if (!take_ring(mine, bytes, dst)) {
        BITNET_HIP_TRY(hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, stream));
        return BITNET_HIP_OK;
    }
    ring_ = std::move(mine);
    const size_t chunks = (bytes + CHUNK - 1) / CHUNK;
    hipError_t e = hipSuccess;
    for (size_t c = 0; c < chunks && e == hipSuccess; ++c) {
        const int slot = (int)(c % CHUNKS);
        const size_t at = c * CHUNK, part = bytes - at < CHUNK ? bytes - at : CHUNK;
        if (c >= CHUNKS) e = hipEventSynchronize(ring.passed[slot]);
        if (e != hipSuccess) break;
        stream_copy(ring.base + (size_t)slot * CHUNK, static_cast<const uint8_t *>(src) + at, part);
        e = launch_move(static_cast<uint8_t *>(dst) + at, ring.on_device + (size_t)slot * CHUNK, part, nullptr, nullptr, stream);
        if (e == hipSuccess && c + CHUNKS < chunks) e = hipEventRecord(ring.passed[slot], stream);
    }
    if (e != hipSuccess) return fail(BITNET_HIP_DEVICE_ERROR, "host to device copy of %zu bytes: %s", bytes, hipGetErrorString(e));
    return BITNET_HIP_OK;
}

void Upload::done()
{
    reading_ = false;
    if (ring_.owns_lock()) ring_.unlock();
}

Upload::~Upload()
{
    // the caller's buffer, and the chunks for their next user, must outlive what the link still reads
    if (reading_) (void)hipStreamSynchronize(stream_);
}

int download(void *dst, const void *src, size_t bytes, const float *scalar, float *scalar_host, hipStream_t stream)
{
    std::unique_lock<std::mutex> mine(ring.lock, std::defer_lock);
    if (!take_ring(mine, bytes, src)) {
        if (scalar) BITNET_HIP_TRY(hipMemcpyAsync(scalar_host, scalar, sizeof(float), hipMemcpyDeviceToHost, stream));
        BITNET_HIP_TRY(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, stream));
        BITNET_HIP_TRY(hipStreamSynchronize(stream));
        return BITNET_HIP_OK;
    }
    hipError_t e = hipSuccess;
    const size_t chunks = (bytes + CHUNK - 1) / CHUNK;
    auto part_of = [&](size_t c) { return c + 1 < chunks ? CHUNK : bytes - c * CHUNK; };
    auto request = [&](size_t c) {
        const int slot = (int)(c % CHUNKS);
        e = launch_move(ring.on_device + (size_t)slot * CHUNK, static_cast<const uint8_t *>(src) + c * CHUNK, part_of(c),
                        c == 0 ? scalar : nullptr, ring.scalar_on_device, stream);
        if (e == hipSuccess) e = hipEventRecord(ring.passed[slot], stream);
    };
    for (size_t c = 0; c < chunks && c < CHUNKS && e == hipSuccess; ++c) request(c);
    for (size_t c = 0; c < chunks && e == hipSuccess; ++c) {
        const int slot = (int)(c % CHUNKS);
        e = hipEventSynchronize(ring.passed[slot]);
        if (e != hipSuccess) break;
        if (c == 0 && scalar) *scalar_host = *ring.scalar;
        stream_copy(static_cast<uint8_t *>(dst) + c * CHUNK, ring.base + (size_t)slot * CHUNK, part_of(c));
        if (c + CHUNKS < chunks) request(c + CHUNKS);
    }
    if (e != hipSuccess) {
        (void)hipStreamSynchronize(stream);  // nothing of this copy is left in the chunks
        return fail(BITNET_HIP_DEVICE_ERROR, "device to host copy of %zu bytes: %s", bytes, hipGetErrorString(e));
    }
    return BITNET_HIP_OK;
}

void staging_retain()
{
    std::lock_guard<std::mutex> guard(users_lock);
    ++users;
}

void staging_release()
{
    std::lock_guard<std::mutex> guard(users_lock);
    if (--users == 0) {
        std::lock_guard<std::mutex> idle(ring.lock);
        if (!ring.used) ring.drop();
        ring.used = false;
    }
}

int HostParts::acquire()
{
    int rc = current_device(&device_);
    if (rc != BITNET_HIP_OK) return rc;
    SlotState &st = slots[device_];
    for (;;) {
        {
            std::lock_guard<std::mutex> guard(slots_lock);
            rc = prepare_slots(st);
            if (rc != BITNET_HIP_OK) return rc;
            for (int i = 0; i < SLOTS && slot_ < 0; ++i)
                if (!st.taken[i]) slot_ = i;
            if (slot_ >= 0) {
                st.taken[slot_] = true;
                ticket = ++st.tickets[slot_];
                answers = st.on_device + (size_t)slot_ * MOST;
                return BITNET_HIP_OK;
            }
        }
        std::this_thread::yield();  // 64 other threads are waiting for theirs; each gives its slot back
    }
}

int HostParts::wait_one(hipStream_t stream, int index, unsigned *bits)
{
    const volatile unsigned long long *word = slots[device_].host + (size_t)slot_ * MOST + index;
    unsigned long long v = *word;
    // a launch this short answers within some tens of microseconds; behind a longer queue, let the runtime wait
    for (; (unsigned)(v >> 32) != ticket && spins_ < 20000; ++spins_) {
        __builtin_ia32_pause();
        v = *word;
    }
    if ((unsigned)(v >> 32) != ticket) {
        BITNET_HIP_TRY(hipStreamSynchronize(stream));
        v = *word;
        if ((unsigned)(v >> 32) != ticket) return fail(BITNET_HIP_KERNEL_ERROR, "the reduction kernel left no result");
    }
    *bits = (unsigned)v;
    return BITNET_HIP_OK;
}

HostParts::~HostParts()
{
    if (slot_ < 0) return;
    std::lock_guard<std::mutex> guard(slots_lock);
    slots[device_].taken[slot_] = false;
}

}  // namespace bitnet
