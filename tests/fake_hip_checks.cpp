// Host-side checks of the library and of its C++ mirror against a stand-in for the HIP runtime: no GPU, no kernel runs.  The
// functions below take the place of the runtime's (the executable's symbols come first), keep device memory on the heap, write down
// what is called in which order, and can be told to fail.  Each check is named on the command line; `kernels M K N` prints the
// kernels that M token rows through a K -> N layer launch, by forward and by matmul on quantised rows; `step M LAYERS HIDDEN FFN KV_HEADS
// HEAD_DIM` how many launches of a decoder's step quantise their rows once a die.
#include <hip/hip_runtime.h>

#include <cxxabi.h>

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <map>
#include <string>
#include <utility>
#include <vector>

#include "../bitnet-mlx.rs_amd/host/bitlinear.hpp"

namespace fake {
struct Call {
    std::string name;
    hipStream_t stream;
    hipStreamCaptureMode mode;  // of the thread, when it called
};
std::vector<Call> calls;
hipStreamCaptureMode thread_mode = hipStreamCaptureModeGlobal;
hipError_t host_malloc_answer = hipSuccess, launch_answer = hipSuccess;
int copies_until_failure = -1;  // a copy that fails has moved half of its bytes
hipStream_t capturing = nullptr;
uintptr_t next_handle = 1;

hipError_t note(const char *name, hipStream_t stream = nullptr, hipError_t answer = hipSuccess)
{
    calls.push_back({name, stream, thread_mode});
    return answer;
}
std::map<const void *, std::string> &kernel_names()  // filled while the library is loaded
{
    static std::map<const void *, std::string> names;
    return names;
}
std::vector<std::string> kernels;  // launched, in order
size_t count(const std::string &name)
{
    size_t n = 0;
    for (const Call &c : calls) n += c.name == name;
    return n;
}
// the position of the last call of this name on this stream, or -1
long last(const std::string &name, hipStream_t stream)
{
    for (long i = (long)calls.size() - 1; i >= 0; --i)
        if (calls[i].name == name && calls[i].stream == stream) return i;
    return -1;
}
// The launches that quantise rows once a die, as far as their flags go (gemv_die.hip): a launch must find none of its rows' flags up, puts them
// up, and takes down those it is given to clear.  What is launched while the stream is captured does so when the graph is replayed.
struct DieLaunch {
    uint64_t *flags, *clear, tag;
    unsigned stride, m, halves;
};
size_t die_launches = 0, stale_flags = 0;
uint64_t last_tag = 0;
constexpr unsigned DIES = 16;
void run(const DieLaunch &l)
{
    for (unsigned die = 0; die < DIES; ++die)
        for (unsigned row = 0; row < l.m; ++row) {
            if (l.flags) {
                stale_flags += l.flags[die * l.stride + row] == l.tag;
                l.flags[die * l.stride + row] = l.tag;
            }
        }
    for (unsigned die = 0; l.clear && die < 8 * l.halves; ++die) memset(l.clear + die * l.stride, 0, l.m * sizeof(uint64_t));
    die_launches += l.flags != nullptr;
    if (l.flags) last_tag = l.tag;
}
std::vector<DieLaunch> captured;
std::map<const void *, std::vector<DieLaunch>> graphs;  // by graph and by executable graph
void launched(const std::string &name, void **args, hipStream_t s)
{
    DieLaunch l = {};
    if (name.find("gemv_die_kernel") != std::string::npos) {
        const char *last = static_cast<const char *>(args[10]) + 192;  // the block behind those of the three projections: q, a_scale, flags, ...
        memcpy(&l.flags, last + 16, 3 * sizeof(uint64_t));
        memcpy(&l.stride, last + 40, sizeof(unsigned));
        memcpy(&l.halves, last + 60, sizeof(unsigned));
        l.m = *static_cast<unsigned *>(args[6]) & 0xffffu;
    } else if (name.find("clear_die_flags_kernel") != std::string::npos) {
        l = {nullptr, *static_cast<uint64_t **>(args[0]), 0, *static_cast<unsigned *>(args[1]), *static_cast<unsigned *>(args[2]), DIES / 8};
    } else {
        return;
    }
    if (s && s == capturing) captured.push_back(l);
    else run(l);
}
int launches_until_failure = -1;  // the launch that fails is queued all the same, and the error is there for whoever asks next
hipError_t pending = hipSuccess;
hipError_t copy(void *dst, const void *src, size_t bytes)
{
    if (copies_until_failure == 0) {
        memcpy(dst, src, bytes / 2);
        return hipErrorInvalidValue;
    }
    if (copies_until_failure > 0) --copies_until_failure;
    memcpy(dst, src, bytes);
    return hipSuccess;
}
template <class T>
hipError_t make(T *out)
{
    *out = reinterpret_cast<T>(next_handle++ << 4);
    return hipSuccess;
}
}  // namespace fake

extern "C" {
hipError_t hipGetSymbolAddress(void **p, const void *) { static char held[1 << 21]; *p = held; return hipSuccess; }
hipError_t hipGetDevice(int *d) { *d = 0; return hipSuccess; }
hipError_t hipGetLastError() { return fake::pending != hipSuccess ? std::exchange(fake::pending, hipSuccess) : fake::launch_answer; }
const char *hipGetErrorString(hipError_t) { return "as told"; }
hipError_t hipFuncSetAttribute(const void *, hipFuncAttribute, int) { return hipSuccess; }

hipError_t hipMalloc(void **p, size_t n) { *p = calloc(1, n); return hipSuccess; }
hipError_t hipFree(void *p) { free(p); return fake::note("hipFree"); }
hipError_t hipHostMalloc(void **p, size_t n, unsigned)
{
    *p = fake::host_malloc_answer == hipSuccess ? aligned_alloc(256, (n + 255) / 256 * 256) : nullptr;
    return fake::note("hipHostMalloc", nullptr, fake::host_malloc_answer);
}
hipError_t hipHostFree(void *p) { free(p); return fake::note("hipHostFree"); }
hipError_t hipHostGetDevicePointer(void **d, void *h, unsigned) { *d = h; return hipSuccess; }
hipError_t hipMemPoolCreate(hipMemPool_t *p, const hipMemPoolProps *) { return fake::make(p); }
hipError_t hipMemPoolSetAttribute(hipMemPool_t, hipMemPoolAttr, void *) { return hipSuccess; }
hipError_t hipMallocFromPoolAsync(void **p, size_t n, hipMemPool_t, hipStream_t) { return hipMalloc(p, n); }
hipError_t hipMallocAsync(void **p, size_t n, hipStream_t) { return hipMalloc(p, n); }
hipError_t hipFreeAsync(void *p, hipStream_t) { free(p); return hipSuccess; }

hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind) { (void)fake::note("hipMemcpy"); return fake::copy(d, s, n); }
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t st)
{
    (void)fake::note("hipMemcpyAsync", st);
    return fake::copy(d, s, n);
}
hipError_t hipMemset(void *d, int v, size_t n) { memset(d, v, n); return fake::note("hipMemset"); }

hipError_t hipDeviceSynchronize() { return fake::note("hipDeviceSynchronize"); }
hipError_t hipStreamSynchronize(hipStream_t s) { return fake::note("hipStreamSynchronize", s); }
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) { (void)fake::note("hipStreamCreate"); return fake::make(s); }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { return fake::make(e); }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t s) { return fake::note("hipEventRecord", s); }
hipError_t hipEventSynchronize(hipEvent_t) { return fake::note("hipEventSynchronize"); }

hipError_t hipThreadExchangeStreamCaptureMode(hipStreamCaptureMode *m) { std::swap(*m, fake::thread_mode); return hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t s, hipStreamCaptureMode) { fake::capturing = s; fake::captured.clear(); return fake::note("hipStreamBeginCapture", s); }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t *g)
{
    fake::capturing = nullptr;
    (void)fake::make(g);
    fake::graphs[*g] = fake::captured;
    return hipSuccess;
}
hipError_t hipStreamIsCapturing(hipStream_t s, hipStreamCaptureStatus *st)
{
    *st = s && s == fake::capturing ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
    return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t *g, hipGraph_t of, hipGraphNode_t *, char *, size_t)
{
    (void)fake::make(g);
    fake::graphs[*g] = fake::graphs[of];
    return fake::note("hipGraphInstantiate");
}
hipError_t hipGraphLaunch(hipGraphExec_t g, hipStream_t s)
{
    for (const fake::DieLaunch &l : fake::graphs[g]) fake::run(l);
    return fake::note("hipGraphLaunch", s);
}
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return fake::note("hipGraphExecDestroy"); }

hipError_t __hipPushCallConfiguration(dim3, dim3, size_t, hipStream_t s) { return fake::note("configure", s); }
hipError_t __hipPopCallConfiguration(dim3 *, dim3 *, size_t *, hipStream_t *s) { *s = fake::calls.back().stream; return hipSuccess; }
hipError_t hipLaunchKernel(const void *f, dim3, dim3, void **args, size_t, hipStream_t s)
{
    fake::kernels.push_back(fake::kernel_names()[f]);
    fake::launched(fake::kernels.back(), args, s);
    if (fake::launches_until_failure >= 0 && fake::launches_until_failure-- == 0) fake::pending = hipErrorLaunchFailure;
    return fake::note("launch", s, fake::launch_answer);
}
void __hipRegisterFunction(void **, const void *f, char *, const char *name, unsigned, void *, void *, void *, void *, int *)
{
    char *plain = abi::__cxa_demangle(name, nullptr, nullptr, nullptr);
    fake::kernel_names()[f] = plain ? plain : name;
    free(plain);
}
}

namespace {

using namespace bitnet;
int failures = 0;
#define CHECK(cond) \
    do { \
        if (!(cond)) { std::printf("FAIL line %d: %s\n", __LINE__, #cond); ++failures; } \
    } while (0)

const hipStream_t side = reinterpret_cast<hipStream_t>(0x1000);

// The mirror's quantisers read on the null stream what a kernel on the caller's stream leaves: they wait for that stream first.
void mirror_waits_for_the_stream_it_was_given()
{
    auto x = DeviceTensor::from_vec(std::vector<float>(64 * 64, 1.0f), {64, 64}).unwrap();
    for (hipStream_t s : {side, hipStream_t(nullptr)}) {
        fake::calls.clear();
        CHECK(absmax_quantize_activations(x, std::nullopt, s).is_ok());
        long launched = fake::last("launch", s), waited = fake::last("hipStreamSynchronize", s);
        CHECK(launched >= 0 && launched < waited && fake::last("hipMemcpy", nullptr) > waited);
        fake::calls.clear();
        CHECK(BitNetWeightQuantizer().quantize(x, s).is_ok());
        launched = fake::last("launch", s), waited = fake::last("hipStreamSynchronize", s);
        CHECK(launched >= 0 && launched < waited && fake::count("hipMemcpy") == 3 && fake::last("hipMemcpy", nullptr) == waited + 3);
    }
}

// Nothing that the mirror enqueues on the null stream may still write a result that a kernel on the caller's stream fills.
void mirror_leaves_nothing_on_the_null_stream()
{
    auto ready = [] { return fake::last("hipMemset", nullptr) <= fake::last("hipStreamSynchronize", nullptr); };
    fake::calls.clear();
    auto x = DeviceTensor::zeros({40, 64}).unwrap();
    CHECK(ready());
    BitLinearConfig c;
    c.in_features = c.out_features = 64;
    auto layer = BitLinear::create(c, "layer").unwrap();
    CHECK(layer->update_weights(std::vector<float>(64 * 64, 0.5f), 64, 64).is_ok());
    fake::calls.clear();
    CHECK(layer->forward(x, nullptr, side).is_ok() && fake::count("launch") > 0 && ready());
    FeedForwardNetwork net;
    net.up_proj = net.gate_proj = net.down_proj = layer;
    fake::calls.clear();
    CHECK(net.forward(x, side).is_ok() && fake::count("launch") > 0 && ready());
}

// A GGUF tensor whose bytes do not reach the device leaves the layer with the weights it had.
void failed_gguf_copy_leaves_the_layer_whole()
{
    const size_t n = 32, k = 64, codes = n * k / 4;
    for (int on_device : {0, 1})
        for (int layout : {BITNET_HIP_LAYOUT_OUT_IN, BITNET_HIP_LAYOUT_IN_OUT}) {
            bitnet_hip_bitlinear *layer = nullptr;
            CHECK(bitnet_hip_bitlinear_create(k, n, 0, &layer) == BITNET_HIP_OK);
            const std::vector<uint8_t> held(codes, 0x61), data(8 + codes, 0x22);
            CHECK(bitnet_hip_bitlinear_set_weights_packed(layer, held.data(), codes, 0.5f, 0, nullptr) == BITNET_HIP_OK);
            fake::copies_until_failure = on_device;  // of a device tensor, the header's copy succeeds
            const size_t rows = layout == BITNET_HIP_LAYOUT_OUT_IN ? n : k, cols = n + k - rows;
            fake::calls.clear();
            CHECK(bitnet_hip_bitlinear_set_weights_gguf(layer, data.data(), data.size(), rows, cols, layout, on_device, nullptr, nullptr,
                                                        nullptr) != BITNET_HIP_OK);
            fake::copies_until_failure = -1;
            CHECK(fake::count("launch") == 0);
            std::vector<uint8_t> back(codes);
            CHECK(bitnet_hip_bitlinear_get_quantized(layer, nullptr, back.data(), codes) == BITNET_HIP_OK && back == held);
            bitnet_hip_bitlinear_destroy(layer);
        }
}

// Without pinned memory, layers are loaded and saved through the runtime's own copies.
void loads_and_saves_without_pinned_memory()
{
    const size_t n = 1024, k = 2048, codes = n * k / 4;  // more than the chunks are made for
    bitnet_hip_bitlinear *layer = nullptr;
    CHECK(bitnet_hip_bitlinear_create(k, n, 0, &layer) == BITNET_HIP_OK);
    std::vector<uint8_t> held(codes), back(codes);
    for (size_t i = 0; i < codes; ++i) held[i] = (uint8_t)(i * 7);
    fake::host_malloc_answer = hipErrorOutOfMemory;
    CHECK(bitnet_hip_bitlinear_set_weights_packed(layer, held.data(), codes, 0.5f, 0, nullptr) == BITNET_HIP_OK);
    CHECK(bitnet_hip_bitlinear_get_quantized(layer, nullptr, back.data(), codes) == BITNET_HIP_OK && back == held);
    CHECK(fake::count("hipHostMalloc") > 0);
    fake::host_malloc_answer = hipSuccess;
    // and through the chunks once there is some: a launch moves what is copied here otherwise
    fake::calls.clear();
    CHECK(bitnet_hip_bitlinear_set_weights_packed(layer, held.data(), codes, 0.5f, 0, nullptr) == BITNET_HIP_OK);
    CHECK(fake::count("hipHostMalloc") == 1 && fake::count("hipMemcpyAsync") == 0);
    bitnet_hip_bitlinear_destroy(layer);
}

// Loading from host memory waits for the stream once, at the end; and also where a launch behind the copy fails, since the
// caller's buffer is free on return.
void loads_wait_for_the_stream_once()
{
    for (size_t n : {size_t(64), size_t(1024)}) {  // through the runtime's copy, and through the chunks
        const size_t k = 2048, codes = n * k / 4;
        bitnet_hip_bitlinear *layer = nullptr;
        CHECK(bitnet_hip_bitlinear_create(k, n, 0, &layer) == BITNET_HIP_OK);
        const std::vector<uint8_t> data(8 + codes, 0x22);
        const std::vector<float> latent(n * k, 0.5f);
        const auto packed = [&] { return bitnet_hip_bitlinear_set_weights_packed(layer, data.data(), codes, 0.5f, 0, side); };
        const auto base3 = [&] { return bitnet_hip_bitlinear_set_weights_base3(layer, data.data(), (n * k + 4) / 5, 0.5f, 0, side); };
        const auto gguf = [&] {
            return bitnet_hip_bitlinear_set_weights_gguf(layer, data.data(), data.size(), n, k, BITNET_HIP_LAYOUT_OUT_IN, 0, nullptr, nullptr, side);
        };
        const auto f32 = [&] {
            return bitnet_hip_bitlinear_set_weights_f32(layer, latent.data(), n, k, BITNET_HIP_LAYOUT_OUT_IN, 0, BITNET_HIP_TERNARY_ABSMEAN_ROUNDCLIP, 0.5f, side);
        };
        const std::vector<std::function<int()>> loads = {packed, base3, gguf, f32};
        for (const auto &load : loads)
            for (hipError_t answer : {hipSuccess, hipErrorLaunchFailure}) {
                fake::calls.clear();
                fake::launch_answer = answer;
                CHECK((load() == BITNET_HIP_OK) == (answer == hipSuccess));
                fake::launch_answer = hipSuccess;
                CHECK(fake::count("hipStreamSynchronize") == 1);
                CHECK(fake::last("hipStreamSynchronize", side) > fake::last("launch", side));
                CHECK(fake::last("hipStreamSynchronize", side) > fake::last("hipMemcpyAsync", side));
            }
        bitnet_hip_bitlinear_destroy(layer);
    }
}

bitnet_hip_decoder *decoder_with_weights(size_t layers, size_t hidden, size_t ffn, size_t tokens = 4, size_t kv_heads = 2, size_t head_dim = 16)
{
    bitnet_hip_decoder *dec = nullptr;
    CHECK(bitnet_hip_decoder_create(layers, hidden, ffn, hidden / head_dim, kv_heads, head_dim, 1e-5f, BITNET_HIP_SUM_BLOCK256, tokens, &dec) == BITNET_HIP_OK);
    const std::vector<uint8_t> codes(hidden * (hidden > ffn ? hidden : ffn) / 4, 0x22);
    for (size_t l = 0; l < layers; ++l)
        for (int p = 0; p < 7; ++p) {
            bitnet_hip_bitlinear *layer = nullptr;
            CHECK(bitnet_hip_decoder_projection(dec, l, p, &layer) == BITNET_HIP_OK);
            CHECK(bitnet_hip_bitlinear_set_weights_packed(layer, codes.data(), codes.size(), 0.5f, 0, nullptr) == BITNET_HIP_OK);
        }
    return dec;
}

// A step that comes a third time is recorded from two blocks on, and one of large blocks (above 74 M weights) from twelve on.
void steps_worth_a_recording()
{
    const struct {
        size_t layers, hidden, ffn, blocks;
        bool recorded;
    } steps[] = {{2, 64, 64, 1, false}, {2, 64, 64, 2, true}, {11, 2048, 10600, 11, true}, {12, 2048, 10700, 11, false}, {12, 2048, 10700, 12, true}};
    for (const auto &t : steps) {
        bitnet_hip_decoder *dec = decoder_with_weights(t.layers, t.hidden, t.ffn);
        std::vector<float> x(t.hidden), out(t.hidden);
        fake::calls.clear();
        for (int times = 0; times < 3; ++times)
            CHECK(bitnet_hip_decoder_decode_layers(dec, 0, t.blocks, x.data(), 1, out.data(), nullptr, nullptr, side) == BITNET_HIP_OK);
        CHECK(fake::count("hipGraphLaunch") == (t.recorded ? 1 : 0));
        bitnet_hip_decoder_destroy(dec);
    }
}

// Recording a step that repeats, and giving up an old recording, leave a capture of another thread alone: what is no plain launch
// runs outside the global mode's rule, nothing waits for the whole device, and the thread's own mode is back afterwards.
void recording_a_step_leaves_other_captures_alone()
{
    bitnet_hip_decoder *dec = decoder_with_weights(2, 64, 64);
    std::vector<float> x(64), outs(8 * 64);
    const auto step = [&](int i) { CHECK(bitnet_hip_decoder_decode(dec, x.data(), 1, outs.data() + 64 * i, nullptr, nullptr, side) == BITNET_HIP_OK); };
    fake::calls.clear();
    for (int i = 0; i < 4; ++i)  // as many recordings as are kept
        for (int times = 0; times < 3; ++times) step(i);
    CHECK(fake::count("hipGraphInstantiate") == 4 && fake::count("hipGraphLaunch") == 4);
    for (int times = 0; times < 64; ++times) step(1 + times % 3);  // replays that earn another recording
    for (int times = 0; times < 3; ++times) step(5);
    CHECK(fake::count("hipGraphInstantiate") == 5 && fake::count("hipGraphExecDestroy") == 1);
    CHECK(fake::count("hipDeviceSynchronize") == 0);
    bool waited = false;
    for (const fake::Call &c : fake::calls) {
        if (c.name == "hipStreamCreate" || c.name == "hipStreamBeginCapture" || c.name == "hipGraphInstantiate" || c.name == "hipGraphExecDestroy")
            CHECK(c.mode == hipStreamCaptureModeRelaxed);
        if (c.name == "hipGraphLaunch") waited = false;
        if (c.name == "hipEventSynchronize") waited = true;
        if (c.name == "hipGraphExecDestroy") CHECK(waited);
    }
    CHECK(fake::thread_mode == hipStreamCaptureModeGlobal);
    bitnet_hip_decoder_destroy(dec);
}

// No launch of a step that quantises rows once a die finds a flag of an earlier launch up: not after steps of other sizes, in a replay, nor
// behind a step that failed after any of its launches, whether its flags could be cleared at once or not.  A step has no launch that does nothing
// but clear flags, also where an odd number of its launches use them.
void steps_find_their_flags_down()
{
    for (size_t layers : {1, 2, 3}) {
        bitnet_hip_decoder *dec = decoder_with_weights(layers, 512, 1408, 64);
        std::vector<float> x(64 * 512), out(64 * 512), other(64 * 512);
        const auto step = [&](size_t m, std::vector<float> &to, size_t end) {
            return bitnet_hip_decoder_decode_layers(dec, 0, end, x.data(), m, to.data(), nullptr, nullptr, side);
        };
        fake::die_launches = fake::stale_flags = 0;
        fake::kernels.clear();
        for (size_t m : {9, 33, 16, 3, 64, 17, 64})
            for (int times = 0; times < 4; ++times) CHECK(step(m, out, layers) == BITNET_HIP_OK);
        for (const std::string &name : fake::kernels) CHECK(name.find("clear_die_flags") == std::string::npos);
        bitnet_hip_decoder_graph *graph = nullptr;
        CHECK(bitnet_hip_decoder_graph_create(dec, 0, layers, x.data(), 12, out.data(), nullptr, nullptr, &graph) == BITNET_HIP_OK);
        CHECK(bitnet_hip_decoder_graph_launch(graph, side) == BITNET_HIP_OK && fake::die_launches > 0 && fake::stale_flags == 0);
        for (int at = 0; at < (int)(4 * layers); ++at)
            for (int clear_fails : {0, 1}) {
                fake::launches_until_failure = at;
                if (clear_fails) fake::launch_answer = hipErrorLaunchFailure;  // every launch then reports an error, the first one already
                CHECK(step(48, other, layers) != BITNET_HIP_OK);
                fake::launches_until_failure = -1;
                fake::launch_answer = fake::pending = hipSuccess;
                fake::stale_flags = 0;
                if (at % 3 == 0) CHECK(bitnet_hip_decoder_graph_launch(graph, side) == BITNET_HIP_OK);
                if (at % 3 == 1) CHECK(step(17, out, layers) == BITNET_HIP_OK);
                CHECK(step(40, other, 1) == BITNET_HIP_OK && step(64, other, layers) == BITNET_HIP_OK);
                CHECK(fake::stale_flags == 0);
            }
        fake::die_launches = 0;
        CHECK(step(48, other, layers) == BITNET_HIP_OK && fake::die_launches > 0);  // the launches on dies are not given up
        bitnet_hip_decoder_graph_destroy(graph);
        bitnet_hip_decoder_destroy(dec);
    }
}

// At two tokens gate and up are quantised on the dies unless the launch without that has just a workgroup for every compute unit.
void two_tokens_on_dies()
{
    const struct {
        size_t ffn;
        bool taken;
    } steps[] = {{6912, true}, {7680, true}, {7936, false}, {8192, false}, {8448, true}};
    for (const auto &t : steps) {
        bitnet_hip_decoder *dec = decoder_with_weights(2, 2560, t.ffn);
        std::vector<float> x(2 * 2560), out(2 * 2560);
        fake::die_launches = 0;
        CHECK(bitnet_hip_decoder_decode(dec, x.data(), 2, out.data(), nullptr, nullptr, side) == BITNET_HIP_OK);
        CHECK(fake::die_launches == (t.taken ? 2 : 0));
        CHECK(bitnet_hip_decoder_decode_layers(dec, 0, 1, x.data(), 2, out.data(), nullptr, nullptr, side) == BITNET_HIP_OK);
        CHECK(fake::die_launches == (t.taken ? 2 : 0));  // one alone has no other launch to clear its flags
        bitnet_hip_decoder_destroy(dec);
    }
}

// Layers made, loaded and dropped one after the other share the pinned chunks; they are given back once layers come and go unloaded.
void chunks_outlive_a_layer_that_used_them()
{
    const size_t n = 1024, k = 2048, codes = n * k / 4;
    const std::vector<uint8_t> data(codes, 0x22);
    const auto layer = [&](bool load) {
        bitnet_hip_bitlinear *l = nullptr;
        CHECK(bitnet_hip_bitlinear_create(k, n, 0, &l) == BITNET_HIP_OK);
        if (load) CHECK(bitnet_hip_bitlinear_set_weights_packed(l, data.data(), codes, 0.5f, 0, nullptr) == BITNET_HIP_OK);
        bitnet_hip_bitlinear_destroy(l);
    };
    for (int round = 1; round <= 2; ++round) {
        for (int i = 0; i < 3; ++i) layer(true);
        CHECK((int)fake::count("hipHostMalloc") == round && (int)fake::count("hipHostFree") == round - 1);
        layer(false);
        CHECK((int)fake::count("hipHostMalloc") == round && (int)fake::count("hipHostFree") == round);
    }
}

// The header of a GGUF tensor in device memory is read behind the work of the caller's stream, as the codes are.
void gguf_header_is_read_in_stream_order()
{
    const size_t n = 32, k = 64;
    const std::vector<uint8_t> data(8 + n * k / 4, 0x22);
    bitnet_hip_bitlinear *layer = nullptr;
    CHECK(bitnet_hip_bitlinear_create(k, n, 0, &layer) == BITNET_HIP_OK);
    fake::calls.clear();
    CHECK(bitnet_hip_bitlinear_set_weights_gguf(layer, data.data(), data.size(), n, k, BITNET_HIP_LAYOUT_OUT_IN, 1, nullptr, nullptr, side) ==
          BITNET_HIP_OK);
    CHECK(fake::count("hipMemcpy") == 0 && fake::count("hipMemcpyAsync") == 2);
    CHECK(fake::calls[0].name == "hipMemcpyAsync" && fake::calls[0].stream == side);
    CHECK(fake::calls[1].name == "hipStreamSynchronize" && fake::calls[1].stream == side);
    bitnet_hip_bitlinear_destroy(layer);
}

// A call of several tokens on short rows is one launch in which every workgroup quantises, which saves host time.  Recorded into a
// caller's graph it is the two launches that the GPU is faster with, as long as the caller gave scratch for them.
void recorded_calls_on_short_rows()
{
    const struct {
        size_t m, k, n;
        bool norm;
        size_t recorded;  // launches
    } calls[] = {{16, 2048, 2560, false, 2}, {40, 2048, 5120, false, 2}, {16, 1280, 2560, false, 2}, {256, 1536, 512, false, 2}, {16, 1024, 2560, true, 2},
                 {128, 512, 512, true, 2},   {9, 1280, 2560, false, 1},  {512, 2048, 512, false, 1}, {16, 1024, 2560, false, 1}, {512, 1024, 512, false, 1},
                 {9, 1024, 2560, true, 1},   {1, 2048, 2560, false, 1}};
    for (const auto &t : calls) {
        bitnet_hip_bitlinear *layer = nullptr;
        CHECK(bitnet_hip_bitlinear_create(t.k, t.n, 0, &layer) == BITNET_HIP_OK);
        const std::vector<uint8_t> codes(t.n * t.k / 4, 0x22);
        CHECK(bitnet_hip_bitlinear_set_weights_packed(layer, codes.data(), codes.size(), 0.5f, 0, nullptr) == BITNET_HIP_OK);
        auto x = DeviceTensor::zeros({t.m, t.k}).unwrap(), out = DeviceTensor::zeros({t.m, t.n}).unwrap(), ones = DeviceTensor::zeros({t.k}).unwrap();
        const size_t dims[2] = {t.m, t.k}, full = bitnet_hip_bitlinear_workspace_size(layer, t.m);
        const float *gamma = t.norm ? ones.data() : nullptr;
        std::vector<uint8_t> ws(full);
        float *const outs[1] = {out.data()};
        const auto launches = [&](size_t given) {
            fake::calls.clear();
            CHECK(bitnet_hip_bitlinear_forward(layer, x.data(), dims, 2, gamma, 1e-5f, BITNET_HIP_SUM_BLOCK256, nullptr, out.data(), given ? ws.data() : nullptr,
                                               given, nullptr, nullptr, nullptr, side) == BITNET_HIP_OK);
            const size_t one = fake::count("launch");
            fake::calls.clear();
            CHECK(bitnet_hip_bitlinear_forward_multi(&layer, 1, x.data(), t.m, gamma, 1e-5f, BITNET_HIP_SUM_BLOCK256, outs, given ? ws.data() : nullptr, given,
                                                     side) == BITNET_HIP_OK);
            CHECK(fake::count("launch") == one);
            return one;
        };
        const auto static_scratch = [&] {
            fake::calls.clear();
            CHECK(bitnet_hip_bitlinear_forward_noalloc(layer, x.data(), dims, 2, gamma, 1e-5f, BITNET_HIP_SUM_BLOCK256, nullptr, out.data(), side) == BITNET_HIP_OK);
            return fake::count("launch");
        };
        const auto scratch = [&](hipStream_t s) { return bitnet_hip_bitlinear_forward_scratch_on(&layer, 1, x.data(), t.m, gamma, BITNET_HIP_SUM_BLOCK256, s); };
        CHECK(launches(full) == 1 && launches(0) == 1 && static_scratch() == 1 && scratch(side) == 0);
        fake::capturing = side;
        CHECK(launches(full) == t.recorded && launches(full - 1) == 1 && launches(0) == 1 && static_scratch() == t.recorded);
        CHECK(scratch(side) == (t.recorded == 2 ? full : 0) && scratch(nullptr) == 0);
        fake::capturing = nullptr;
        bitnet_hip_bitlinear_destroy(layer);
    }
}

// A call on dies gives its flags a tag that no call before it had, since they lie in whatever memory the workspace is; it needs room for them, and
// is two launches where a replay would find them up, or where the result lies over the rows.
void calls_on_dies()
{
    bitnet_hip_bitlinear *layer = nullptr;
    const size_t m = 16, k = 4096, full = 2 * k * k / 4;
    CHECK(bitnet_hip_bitlinear_create(k, k, 0, &layer) == BITNET_HIP_OK);
    const std::vector<uint8_t> codes(k * k / 4, 0x22);
    CHECK(bitnet_hip_bitlinear_set_weights_packed(layer, codes.data(), codes.size(), 0.5f, 0, nullptr) == BITNET_HIP_OK);
    auto x = DeviceTensor::zeros({m + 1, k}).unwrap(), out = DeviceTensor::zeros({m, k}).unwrap();
    const size_t dims[2] = {m, k}, plain = bitnet_hip_bitlinear_workspace_size(layer, m);
    const size_t wanted = bitnet_hip_bitlinear_forward_scratch_on(&layer, 1, x.data(), m, nullptr, BITNET_HIP_SUM_BLOCK256, side);
    CHECK(wanted > plain && wanted < full);
    std::vector<uint8_t> ws(full);
    const auto launches = [&](size_t given, float *to) {
        fake::calls.clear();
        fake::die_launches = 0;
        CHECK(bitnet_hip_bitlinear_forward(layer, x.data(), dims, 2, nullptr, 1e-5f, BITNET_HIP_SUM_BLOCK256, nullptr, to, given ? ws.data() : nullptr, given, nullptr,
                                           nullptr, nullptr, side) == BITNET_HIP_OK);
        return fake::count("launch");
    };
    CHECK(launches(wanted, out.data()) == 1 && fake::die_launches == 1);
    const uint64_t tag = fake::last_tag;
    CHECK(launches(full, out.data()) == 1 && fake::die_launches == 1 && fake::last_tag != tag && tag >> 63 == 1 && fake::last_tag >> 63 == 1);
    CHECK(launches(wanted - 1, out.data()) == 2 && launches(plain, out.data()) == 2 && launches(0, out.data()) == 2);
    fake::capturing = side;
    CHECK(bitnet_hip_bitlinear_forward_scratch_on(&layer, 1, x.data(), m, nullptr, BITNET_HIP_SUM_BLOCK256, side) == plain);
    CHECK(launches(full, out.data()) == 2);
    fake::capturing = nullptr;
    for (float *over : {x.data(), x.data() + k, x.data() + (m - 1) * k})
        CHECK(launches(full, over) == 2 && fake::die_launches == 0);
    CHECK(launches(full, x.data()) == 2 && launches(0, x.data()) == 2);
    bitnet_hip_bitlinear_destroy(layer);
}

// The launches for few tokens that quantise in every workgroup do not take a result over the rows either, whatever scratch the caller was told of.
void results_over_the_rows()
{
    for (const auto &t : {std::pair<size_t, size_t>{1, 2560}, {1, 8192}, {1, 7424}, {2, 1024}, {8, 2560}, {32, 512}}) {
        bitnet_hip_bitlinear *layer = nullptr;
        CHECK(bitnet_hip_bitlinear_create(t.second, t.second, 0, &layer) == BITNET_HIP_OK);
        const std::vector<uint8_t> codes(t.second * t.second / 4, 0x22);
        CHECK(bitnet_hip_bitlinear_set_weights_packed(layer, codes.data(), codes.size(), 0.5f, 0, nullptr) == BITNET_HIP_OK);
        auto x = DeviceTensor::zeros({t.first, t.second}).unwrap(), out = DeviceTensor::zeros({t.first, t.second}).unwrap();
        const size_t dims[2] = {t.first, t.second};
        CHECK(bitnet_hip_bitlinear_forward_scratch(layer, x.data(), t.first, nullptr, BITNET_HIP_SUM_BLOCK256) == 0);
        uint8_t byte[1];
        for (float *to : {out.data(), x.data()})
            for (size_t given : {0, 1}) {
                const size_t launches = to == x.data() ? 2 : 1;
                fake::calls.clear();
                CHECK(bitnet_hip_bitlinear_forward(layer, x.data(), dims, 2, nullptr, 1e-5f, BITNET_HIP_SUM_BLOCK256, nullptr, to, given ? byte : nullptr, given,
                                                   nullptr, nullptr, nullptr, side) == BITNET_HIP_OK);
                CHECK(fake::count("launch") == launches);
                fake::calls.clear();
                CHECK(bitnet_hip_bitlinear_forward_multi(&layer, 1, x.data(), t.first, nullptr, 1e-5f, BITNET_HIP_SUM_BLOCK256, &to, given ? byte : nullptr, given,
                                                         side) == BITNET_HIP_OK);
                CHECK(fake::count("launch") == launches);
                fake::calls.clear();
                CHECK(bitnet_hip_bitlinear_forward_noalloc(layer, x.data(), dims, 2, nullptr, 1e-5f, BITNET_HIP_SUM_BLOCK256, nullptr, to, side) == BITNET_HIP_OK);
                CHECK(fake::count("launch") == launches);
            }
        bitnet_hip_bitlinear_destroy(layer);
    }
}

// A workspace holds the quantised rows and nothing that no kernel reads: workspace_size is what a call of two launches uses.
void a_workspace_is_what_a_call_uses()
{
    for (size_t m : {97, 256, 300})
        for (size_t k : {4096, 6900}) {
            bitnet_hip_bitlinear *layer = nullptr;
            CHECK(bitnet_hip_bitlinear_create(k, 2560, 0, &layer) == BITNET_HIP_OK);
            auto x = DeviceTensor::zeros({1024}).unwrap();
            const size_t used = bitnet_hip_bitlinear_forward_scratch(layer, x.data(), m, nullptr, BITNET_HIP_SUM_BLOCK256);
            CHECK(used != 0 && bitnet_hip_bitlinear_workspace_size(layer, m) == used);
            bitnet_hip_bitlinear_destroy(layer);
        }
}

struct Check {
    const char *name;
    void (*run)();
};
const Check checks[] = {
    {"mirror_waits_for_the_stream_it_was_given", mirror_waits_for_the_stream_it_was_given},
    {"mirror_leaves_nothing_on_the_null_stream", mirror_leaves_nothing_on_the_null_stream},
    {"failed_gguf_copy_leaves_the_layer_whole", failed_gguf_copy_leaves_the_layer_whole},
    {"loads_and_saves_without_pinned_memory", loads_and_saves_without_pinned_memory},
    {"loads_wait_for_the_stream_once", loads_wait_for_the_stream_once},
    {"steps_worth_a_recording", steps_worth_a_recording},
    {"recording_a_step_leaves_other_captures_alone", recording_a_step_leaves_other_captures_alone},
    {"steps_find_their_flags_down", steps_find_their_flags_down},
    {"two_tokens_on_dies", two_tokens_on_dies},
    {"chunks_outlive_a_layer_that_used_them", chunks_outlive_a_layer_that_used_them},
    {"gguf_header_is_read_in_stream_order", gguf_header_is_read_in_stream_order},
    {"recorded_calls_on_short_rows", recorded_calls_on_short_rows},
    {"calls_on_dies", calls_on_dies},
    {"results_over_the_rows", results_over_the_rows},
    {"a_workspace_is_what_a_call_uses", a_workspace_is_what_a_call_uses},
};

}  // namespace

int main(int argc, char **argv)
{
    if (argc == 5 && std::string(argv[1]) == "kernels") {
        const size_t m = std::strtoul(argv[2], nullptr, 10), k = std::strtoul(argv[3], nullptr, 10), n = std::strtoul(argv[4], nullptr, 10);
        // no kernel runs and no weights are copied in: buffers of a few bytes stand for the matrices, aligned as the real ones
        bitnet_hip_bitlinear *layer = nullptr;
        auto some = DeviceTensor::zeros({1024}).unwrap();
        const size_t dims[2] = {m, k};
        if (bitnet_hip_bitlinear_create(k, n, 0, &layer) != BITNET_HIP_OK) return 3;
        if (bitnet_hip_bitlinear_set_weights_f32(layer, some.data(), n, k, BITNET_HIP_LAYOUT_OUT_IN, 1, BITNET_HIP_TERNARY_ABSMEAN_ROUNDCLIP, 0.5f, side) != BITNET_HIP_OK)
            return 3;
        const auto print = [](const char *call) {
            for (const std::string &name : fake::kernels) std::printf("%s: %s\n", call, name.c_str());
            fake::kernels.clear();
        };
        fake::kernels.clear();
        if (bitnet_hip_bitlinear_forward(layer, some.data(), dims, 2, nullptr, 1e-5f, BITNET_HIP_SUM_BLOCK256, nullptr, some.data(), nullptr, 0, nullptr, nullptr,
                                         nullptr, side) != BITNET_HIP_OK)
            return 3;
        print("forward");
        const int8_t *rows = reinterpret_cast<const int8_t *>(some.data());
        const int32_t *sums = reinterpret_cast<const int32_t *>(some.data());
        if (bitnet_hip_bitlinear_matmul(layer, rows, sums, m, some.data(), nullptr, nullptr, some.data(), side) != BITNET_HIP_OK) return 3;
        print("matmul");
        return 0;
    }
    if (argc == 8 && std::string(argv[1]) == "step") {
        size_t v[6];
        for (int i = 0; i < 6; ++i) v[i] = std::strtoul(argv[2 + i], nullptr, 10);
        bitnet_hip_decoder *dec = decoder_with_weights(v[1], v[2], v[3], v[0], v[4], v[5]);
        std::vector<float> x(v[0] * v[2]), out(v[0] * v[2]);
        if (failures || bitnet_hip_decoder_decode(dec, x.data(), v[0], out.data(), nullptr, nullptr, side) != BITNET_HIP_OK) return 3;
        std::printf("%zu\n", fake::die_launches);
        return 0;
    }
    for (const Check &c : checks) {
        if (argc == 2 && std::string(argv[1]) != c.name) continue;
        if (argc == 1) { std::printf("%s\n", c.name); continue; }
        c.run();
        std::printf("%s: %d failed\n", c.name, failures);
        return failures ? 1 : 0;
    }
    return argc == 1 ? 0 : 2;
}
