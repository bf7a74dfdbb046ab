// Network graph, device tensor management and the forward loop.
#include "engine.h"
#include "range.h"

#include <immintrin.h>

#include <algorithm>
#include <chrono>
#include <cstring>
#include <limits>
#include <map>
#include <mutex>
#include <vector>

namespace fynhip {

void fail(int code, const char* fmt, ...) {
    char buf[1024];
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(buf, sizeof(buf), fmt, ap);
    va_end(ap);
    throw Error(code, buf);
}

// ---------------------------------------------------------------------------------------------
// Layer base
// ---------------------------------------------------------------------------------------------
Layer::Layer(Net* n, const fyn_layer_desc& desc) : d(desc), net(n) {}

Act Layer::act() const {
    // LayerBuilderTempl::getFlags (base/layerbuilder.h:445-493): RELU and LEAKY_RELU both set PRE_RELU,
    // the leak value distinguishes them (gpu/gpulayerbase.cpp:775-802).
    // Kernels may evaluate the activation branch-free as min(hi, max(lo, x)) + leak * min(x, 0); the
    // fields are normalised for that here.
    const float inf = std::numeric_limits<float>::infinity();
    Act a{ACT_NONE, 0.f, -inf, inf};
    if (d.flags & FYN_FLAG_PRE_RELU) {
        a.lo = 0.f;
        if (d.leaky_relu != 0.f) {
            a.kind = ACT_LEAKY;
            a.leak = d.leaky_relu;
        } else {
            a.kind = ACT_RELU;
        }
    } else if (d.flags & FYN_FLAG_PRE_CLIP) {
        a.kind = ACT_CLIP;
        a.lo = d.clip_low;
        a.hi = d.clip_high;
    }
    return a;
}

void Layer::port_shape(int port, int& c, int& h, int& w, int& pad) const {
    if (port == 0) {
        c = d.in_channels;
        h = d.height;
        w = d.width;
        pad = d.input_padding;
    } else {  // residual: same net size as the output (base/layerbase.h:266-274)
        c = oc;
        h = oh;
        w = ow;
        pad = d.residual_padding;
    }
}

const Tensor& Layer::tin(int port) const { return net->tensors[in[port]]; }
const Tensor& Layer::tout() const { return net->tensors[out]; }

// ---------------------------------------------------------------------------------------------
// Streams.  All streams of a device are created together, when the library first needs one there, and are leased to
// networks afterwards.  Measured on this runtime: streams created after the process has launched its first hipGraph
// overlap each other badly (four ResNet-50 instances side by side: 3000 frames/s instead of 4700), whereas streams
// that exist by then are unaffected by later graph launches.  Leasing also keeps the stream count of a process that
// builds and destroys many networks constant.  Streams are never destroyed; a network that finds none free gets a
// new one.  The first kMainStreams entries serve networks' own streams, the rest their copy streams.
//
// The process has a few hardware queues (4 by default) and a stream is tied to one of them when it is created; kernels
// of two streams that share a queue never overlap, whatever else is idle.  Which streams share one is up to the runtime
// (and to the streams that the application made before), so it is found out once, when the streams are created: a stream
// whose kernel never ran at the same time as a busy one's shares its queue.  A lease then takes a stream of the queue
// that has the fewest leases.  Four ResNet-50 instances side by side with one other network alive: 154 us per frame where
// two of them shared a queue, 108 us where each had its own.
// ---------------------------------------------------------------------------------------------
namespace {
struct DeviceStreams {
    std::vector<hipStream_t> streams;
    std::vector<char> leased;
    std::vector<int> queue;   // streams with equal numbers share a hardware queue
    std::map<int, uint64_t> last;   // queue -> when a stream of it was leased last
    uint64_t leases = 0;
};
constexpr size_t kMainStreams = 8, kCopyStreams = 8;
std::mutex g_streams_mu;
std::map<int, DeviceStreams> g_streams;

__global__ void occupy_kernel(unsigned long long ticks, unsigned long long* span) {
    const unsigned long long t0 = wall_clock64();
    unsigned long long t = t0;
    while (t - t0 < ticks) t = wall_clock64();
    span[0] = t0;
    span[1] = t;
}

// Fills ds.queue: every stream's kernel is run beside one of each queue known so far.
void find_queues(DeviceStreams& ds) {
    const size_t n = ds.streams.size();
    ds.queue.assign(n, 0);
    unsigned long long* span = nullptr;   // [stream][start, end]
    if (hipHostMalloc(reinterpret_cast<void**>(&span), n * 2 * sizeof(*span), hipHostMallocDefault) != hipSuccess) {
        (void)hipGetLastError();
        return;
    }
    const unsigned long long ticks = 5000;   // 50 us of the 100 MHz clock: longer than it takes to launch two kernels
    auto run = [&](size_t i, unsigned long long t) { hipLaunchKernelGGL(occupy_kernel, dim3(1), dim3(1), 0, ds.streams[i], t, span + 2 * i); };
    for (size_t i = 0; i < n; i++) run(i, 1);   // (a stream's first launch takes longer)
    for (size_t i = 0; i < n; i++) (void)hipStreamSynchronize(ds.streams[i]);
    std::vector<size_t> first;   // one stream of each queue
    for (size_t j = 0; j < n; j++) {
        size_t q = 0;
        for (; q < first.size(); q++) {
            run(first[q], ticks);
            run(j, ticks);
            (void)hipStreamSynchronize(ds.streams[first[q]]);
            (void)hipStreamSynchronize(ds.streams[j]);
            if (span[2 * j] >= span[2 * first[q] + 1]) break;   // one behind the other
        }
        if (q == first.size()) first.push_back(j);
        ds.queue[j] = (int)q;
    }
    (void)hipHostFree(span);
    FYN_HIP(hipGetLastError());
}

hipStream_t lease_stream(int device, bool copy) {
    std::lock_guard<std::mutex> lk(g_streams_mu);
    DeviceStreams& ds = g_streams[device];
    if (ds.streams.empty()) {
        for (size_t i = 0; i < kMainStreams + kCopyStreams; i++) {
            hipStream_t st = nullptr;
            if (i < kMainStreams) FYN_HIP(hipStreamCreate(&st));
            else FYN_HIP(hipStreamCreateWithFlags(&st, hipStreamNonBlocking));
            ds.streams.push_back(st);
            ds.leased.push_back(0);
        }
        find_queues(ds);
    }
    std::map<int, int> count;
    for (size_t i = 0; i < ds.streams.size(); i++) count[ds.queue[i]] += ds.leased[i];
    // (equal counts: the queue whose last lease is longest ago, so that networks made together get queues of their own)
    auto better = [&](int a, int b) { return count[a] != count[b] ? count[a] < count[b] : ds.last[a] < ds.last[b]; };
    const size_t lo = copy ? kMainStreams : 0, hi = copy ? kMainStreams + kCopyStreams : kMainStreams;
    size_t best = hi;
    for (size_t i = lo; i < hi; i++)
        if (!ds.leased[i] && (best == hi || better(ds.queue[i], ds.queue[best]))) best = i;
    if (best < hi) {
        ds.leased[best] = 1;
        ds.last[ds.queue[best]] = ++ds.leases;
        return ds.streams[best];
    }
    hipStream_t st = nullptr;   // all taken: one more, destroyed again when it comes back
    if (copy) FYN_HIP(hipStreamCreateWithFlags(&st, hipStreamNonBlocking));
    else FYN_HIP(hipStreamCreate(&st));
    return st;
}

void return_stream(int device, hipStream_t st) {
    if (!st) return;
    std::lock_guard<std::mutex> lk(g_streams_mu);
    DeviceStreams& ds = g_streams[device];
    for (size_t i = 0; i < ds.streams.size(); i++)
        if (ds.streams[i] == st) {
            ds.leased[i] = 0;
            return;
        }
    (void)hipStreamDestroy(st);   // an overflow stream
}
}  // namespace

// ---------------------------------------------------------------------------------------------
// Fixed staging area for read-backs that must not allocate (Net::copy_result_static).  One array per GPU, part of the
// loaded code object and held until the process ends.  In host code the array's name is only a handle for
// hipGetSymbolAddress; the address it yields on each device is what kernels and copies receive.
// ---------------------------------------------------------------------------------------------
static __device__ __align__(256) __attribute__((used)) float scratch[FYN_STATIC_SCRATCH_FLOATS];
namespace {
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
float* g_scratch_ptr[kMaxDevices] = {};

// The calling thread's current device must be `device`.
float* static_scratch(int device) {
    if (device < 0 || device >= kMaxDevices) fail(FYN_ERR_DEVICE, "device %d beyond the %d devices the fixed staging area covers", device, kMaxDevices);
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (!g_scratch_ptr[device]) {
        float* p = nullptr;
        FYN_HIP(hipGetSymbolAddress(reinterpret_cast<void**>(&p), HIP_SYMBOL(scratch)));
        if (!p) fail(FYN_ERR_DEVICE, "no device address for the fixed staging area on device %d", device);
        g_scratch_ptr[device] = p;
    }
    return g_scratch_ptr[device];
}
}  // namespace

// ---------------------------------------------------------------------------------------------
// Net
// ---------------------------------------------------------------------------------------------
extern "C" char** environ;

void Switches::read() {
    v_.clear();
    for (char** e = environ; e && *e; e++) {
        if (strncmp(*e, "FYNHIP_", 7) != 0) continue;
        const char* eq = strchr(*e, '=');
        if (eq) v_[std::string(*e, eq - *e)] = std::string(eq + 1);
    }
}
const char* Switches::get(const char* name) const {
    auto it = v_.find(name);
    return it == v_.end() ? nullptr : it->second.c_str();
}

Net::Net(int dev, int stor) : device(dev), storage(stor) {
    sw.read();
    if (stor != FYN_STORAGE_F32 && stor != FYN_STORAGE_F16) fail(FYN_ERR_INVALID, "unknown storage type %d", stor);
    int count = 0;
    FYN_HIP(hipGetDeviceCount(&count));
    if (dev < 0 || dev >= count) fail(FYN_ERR_DEVICE, "device %d not present (%d devices)", dev, count);
    FYN_HIP(hipSetDevice(dev));
    stream = lease_stream(dev, false);
    HostPool::network_created();
    try {
        // resolved here, where the caller may still allocate: looking the symbol up loads the code object on this device
        static_scratch_ = static_scratch(dev);
        unsigned* const words = static_cast<unsigned*>(dev_alloc(256));
        signal_.create(words);
        upload_words_ = words + 32;   // (a line of their own)
        feed_ = signal_.feed();
        // (where the runtime is told to finish a launch before the call returns, the frame is copied first)
        for (const char* e : {"HIP_LAUNCH_BLOCKING", "CUDA_LAUNCH_BLOCKING", "AMD_SERIALIZE_KERNEL"})
            if (const char* v = getenv(e)) feed_ahead_ = feed_ahead_ && (!*v || *v == '0');
        if (const char* v = sw.get("FYNHIP_FEED_GIVE_UP")) feed_give_up_ = (unsigned)atoi(v);   // (tests)
    } catch (...) {
        release_all();
        throw;
    }
}

void Net::release_all() {
    if (stream) (void)hipStreamSynchronize(stream);
    for (void* p : allocs_) (void)hipFree(p);
    allocs_.clear();
    signal_.destroy();   // (the stream is idle: the areas that waited for the word are free)
    return_stream(device, stream);
    HostPool::network_gone();
}

Net::~Net() {
    (void)hipSetDevice(device);
    try {
        async_end();
    } catch (...) {
    }
    if (stream) (void)hipStreamSynchronize(stream);
    if (graph_exec_) (void)hipGraphExecDestroy(graph_exec_);
    if (graph_) (void)hipGraphDestroy(graph_);
    for (auto& kv : layers) {
        if (kv.second->ev0) (void)hipEventDestroy(kv.second->ev0);
        if (kv.second->ev1) (void)hipEventDestroy(kv.second->ev1);
    }
    layers.clear();
    release_all();
}

void* Net::dev_alloc(size_t bytes, bool zero) {
    void* p = nullptr;
    if (bytes == 0) bytes = 16;
    FYN_HIP(hipMalloc(&p, bytes));
    allocs_.push_back(p);
    alloc_calls_++;
    alloc_bytes_ += bytes;
    if (zero) {
        launch_fill_zero(p, bytes, stream);
        FYN_HIP(hipGetLastError());
    }
    return p;
}

void Net::dev_free(void* p) {
    auto it = std::find(allocs_.begin(), allocs_.end(), p);
    if (it == allocs_.end()) return;
    FYN_HIP(hipStreamSynchronize(stream));
    allocs_.erase(it);
    (void)hipFree(p);
}

void Net::dev_free_many(const std::vector<void*>& ptrs) {
    bool synced = false;
    for (void* p : ptrs) {
        auto it = std::find(allocs_.begin(), allocs_.end(), p);
        if (it == allocs_.end()) continue;
        if (!synced) {
            FYN_HIP(hipStreamSynchronize(stream));
            synced = true;
        }
        allocs_.erase(it);
        (void)hipFree(p);
    }
}

float* Net::staging(size_t floats) {
    if (floats > staging_floats_) {
        FYN_HIP(hipStreamSynchronize(stream));
        // the old area stays owned by allocs_ and is released with the net
        staging_ = static_cast<float*>(dev_alloc(floats * sizeof(float), false));
        staging_floats_ = floats;
    }
    return staging_;
}

Layer* Net::layer(int number) {
    auto it = layers.find(number);
    if (it == layers.end()) fail(FYN_ERR_NOTFOUND, "no layer with number %d", number);
    return it->second.get();
}

void Net::add_layer(const fyn_layer_desc& d) {
    if (is_setup) fail(FYN_ERR_STATE, "cannot add layers after setup");
    // LayerFactory::pushBuilder (base/layerfactory.cpp:67-76)
    if (d.number < 0) fail(FYN_ERR_INVALID, "Must identify each layer with a valid number (found %d in the builder)", d.number);
    if (layers.count(d.number)) fail(FYN_ERR_DUPLICATE, "Trying to insert a layer on a position that is already taken (%d)", d.number);
    std::unique_ptr<Layer> l(create_layer(this, d));   // may throw: nothing is registered then
    layers[d.number] = std::move(l);
}

void Net::add_custom_layer(const fyn_layer_desc& d, const fyn_custom_layer& impl) {
    if (is_setup) fail(FYN_ERR_STATE, "cannot add layers after setup");
    if (d.number < 0) fail(FYN_ERR_INVALID, "Must identify each layer with a valid number (found %d in the builder)", d.number);
    if (layers.count(d.number)) fail(FYN_ERR_DUPLICATE, "Trying to insert a layer on a position that is already taken (%d)", d.number);
    std::unique_ptr<Layer> l(create_custom_layer(this, d, impl));
    layers[d.number] = std::move(l);
}

void Net::connect(int out_layer, int in_layer, int port) {
    if (is_setup) fail(FYN_ERR_STATE, "cannot connect layers after setup");
    Layer* src = layer(out_layer);
    Layer* dst = layer(in_layer);
    if (port < 0 || port >= dst->num_ports())
        fail(FYN_ERR_INVALID, "layer %s has no input port %d", dst->d.name, port);
    if (!(in_layer > out_layer))
        fail(FYN_ERR_INVALID, "layer %s (%d) cannot feed layer %s (%d): execution is in ascending number", src->d.name,
             out_layer, dst->d.name, in_layer);
    if (dst->in[port] != -1) return;  // already connected (BufferManager::checkIOMatch returns no match)
    // I/O match (base/buffermanager.cpp:462-492): same geometry on both sides of the edge.  The reference compares
    // textures, four channels each, not channel counts: a consumer may name up to three channels more or fewer
    // than were produced (the style-transfer samples download 4 channels of a 3-channel result,
    // samples/samplenetworks/stylenet3x3.cpp:175,180).  Channels beyond the produced ones read as zero.
    int c, h, w, pad;
    dst->port_shape(port, c, h, w, pad);
    if ((c + 3) / 4 != (src->oc + 3) / 4 || h != src->oh || w != src->ow || pad != src->d.output_padding)
        fail(FYN_ERR_INVALID,
             "Inputs/outputs do not match (I/O) for layers %s and %s: producer %dx%dx%d pad %d, consumer port %d wants "
             "%dx%dx%d pad %d",
             dst->d.name, src->d.name, src->oc, src->oh, src->ow, src->d.output_padding, port, c, h, w, pad);
    // tensors are created lazily: the producer's output tensor id
    if (src->out == -1) {
        if (!src->has_own_output()) {
            fail(FYN_ERR_INVALID, "layer %s has no output that can be connected", src->d.name);
        }
        Tensor t;
        t.producer = src->d.number;
        tensors.push_back(t);
        src->out = (int)tensors.size() - 1;
    }
    dst->in[port] = src->out;
    tensors[src->out].last_reader = std::max(tensors[src->out].last_reader, in_layer);
}

void Net::setup() {
    if (is_setup) fail(FYN_ERR_STATE, "network is already set up");
    FYN_HIP(hipSetDevice(device));
    // 1. tensors: external inputs for unconnected ports, outputs for every layer
    for (auto& kv : layers) {
        Layer* l = kv.second.get();
        for (int p = 0; p < l->num_ports(); p++) {
            if (l->in[p] != -1) continue;
            Tensor t;
            t.producer = -1;
            t.locked = true;
            t.last_reader = l->d.number;
            tensors.push_back(t);
            l->in[p] = (int)tensors.size() - 1;
            int c, h, w, pad;
            l->port_shape(p, c, h, w, pad);
            TView& v = tensors.back().v;
            v.c = c; v.h = h; v.w = w; v.pad = pad; v.cp = channel_pitch(c); v.f16 = f16();
        }
        if (l->has_own_output()) {
            if (l->out == -1) {
                Tensor t;
                t.producer = l->d.number;
                t.locked = true;  // nobody consumes it: it is a network output
                tensors.push_back(t);
                l->out = (int)tensors.size() - 1;
            }
            if (l->d.type == FYN_LAYER_UPLOAD) tensors[l->out].locked = true;  // filled from the host
            TView& v = tensors[l->out].v;
            v.c = l->oc; v.h = l->oh; v.w = l->ow; v.pad = l->d.output_padding; v.cp = channel_pitch(l->oc); v.f16 = f16();
        } else {
            // pass-through (download): output aliases the input, which must survive
            l->out = l->in[0];
            tensors[l->out].locked = true;
        }
    }
    keep_projection_inputs(this);
    const auto kept = keep_block_inputs(this);
    // 2. device buffers.  Liveness rule of BufferManager::findTexture (base/buffermanager.cpp:512-525)
    //    restated for in-order stream execution: a buffer can take layer N's output when every reader of
    //    its current tenant has a number < N; only buffers of identical geometry are shared so that the
    //    zero halo written at allocation stays valid.
    for (auto& kv : layers) {
        Layer* l = kv.second.get();
        for (int p = 0; p < l->num_ports(); p++) {
            Tensor& t = tensors[l->in[p]];
            if (t.buffer == -1 && t.producer == -1) {
                DevBuffer b;
                b.bytes = t.v.bytes();
                b.ptr = dev_alloc(b.bytes);
                b.locked = true;
                buffers.push_back(b);
                t.buffer = (int)buffers.size() - 1;
                t.v.ptr = b.ptr;
            }
        }
        if (!l->has_own_output()) continue;
        Tensor& t = tensors[l->out];
        int found = -1;
        if (reuse_buffers && !t.locked) {
            for (size_t i = 0; i < buffers.size(); i++) {
                DevBuffer& b = buffers[i];
                if (!b.locked && b.free_after < l->d.number && b.h == t.v.h && b.w == t.v.w && b.pad == t.v.pad &&
                    b.cp == t.v.cp && b.f16 == t.v.f16) {
                    found = (int)i;
                    break;
                }
            }
        }
        if (found == -1) {
            DevBuffer b;
            b.bytes = t.v.bytes();
            b.ptr = dev_alloc(b.bytes);
            b.h = t.v.h; b.w = t.v.w; b.pad = t.v.pad; b.cp = t.v.cp; b.f16 = t.v.f16;
            buffers.push_back(b);
            found = (int)buffers.size() - 1;
        }
        DevBuffer& b = buffers[found];
        b.locked = t.locked;
        b.free_after = std::max(t.last_reader, l->d.number);
        t.buffer = found;
        t.v.ptr = b.ptr;
        t.written = t.producer;
    }
    for (auto i = kept.rbegin(); i != kept.rend(); ++i) tensors[i->first].last_reader = i->second;
    // pass-through layers were given the tensor id only; nothing else to do for them
    assign_range_words();
    // 3. per-layer setup (weight packing, kernel selection)
    for (auto& kv : layers) {
        kv.second->setup();
        kv.second->set_up = true;
    }
    fuse_depthwise_layers(this);
    fuse_projection_layers(this);
    fuse_batchnorm_layers(this);
    // (a layer that computes what stands behind it keeps its own launch, which the last three ask for)
    fuse_function_layers(this);
    fuse_concat_layers(this);
    fuse_argmax_layers(this);
    fuse_block_layers(this);
    fuse_pair_layers(this);
    fuse_head_layers(this);
    assign_range_resets();
    poison_lds_ = sw.get("FYNHIP_POISON_LDS") != nullptr;
    FYN_HIP(hipStreamSynchronize(stream));
    is_setup = true;
}

bool Net::alone(int tensor, int from, int to) const {
    const Tensor& t = tensors[tensor];
    for (const Tensor& o : tensors)
        if (&o != &t && o.buffer == t.buffer && o.written <= to && std::max(o.last_reader, o.producer) >= from) return false;
    return true;
}

// Value ranges (range.h), fp32 storage only.  A tensor gets a word when whoever writes it keeps the word up to date:
// tensors fed from the host (set_input and the frame pipeline clear and raise the word themselves) and the outputs of
// layers whose kernels do (tracks_range()).
void Net::assign_range_words() {
    if (f16() || sw.get("FYNHIP_NO_RANGE_TRACKING") || sw.get("FYNHIP_FORCE_DIRECT_CONV") || tensors.empty()) return;
    amax_dev_ = static_cast<unsigned*>(dev_alloc(tensors.size() * RANGE_WORDS * sizeof(unsigned), true));
    for (size_t i = 0; i < tensors.size(); i++) {
        Tensor& t = tensors[i];
        bool tracked = t.producer == -1;
        if (t.producer >= 0) {
            Layer* pl = layer(t.producer);
            tracked = pl->d.type == FYN_LAYER_UPLOAD || pl->tracks_range();
        }
        if (tracked) t.amax = amax_dev_ + i * RANGE_WORDS;
    }
}

// A word raised during a forward pass must read 0 again before the tensor's producer runs in the next pass.  The
// clearing is given to a convolution kernel that runs after the tensor's last reader (kernels of one stream run one
// after the other, so nothing else touches the word at that time): the first such layer behind the last reader,
// wrapping around to the layers in front of the producer.  take(layer, word) says whether the layer's launch has room for
// the word; the result are the tensors for which none has.
template <class Take>
std::vector<int> Net::place_range_resets(Take&& take) const {
    std::vector<int> lost;
    for (size_t i = 0; i < tensors.size(); i++) {
        const Tensor& t = tensors[i];
        if (!t.amax || t.producer < 0 || layers.at(t.producer)->d.type == FYN_LAYER_UPLOAD) continue;   // (an upload's: cleared where it is written from the host)
        const int last = std::max(t.last_reader, t.producer);
        bool done = false;
        // layers behind the last reader, in execution order ...
        for (auto& kv : layers)
            if (kv.first > last && take(kv.second.get(), t.amax)) { done = true; break; }
        // ... then the layers in front of the launch that writes it (they run in the next pass, before it)
        if (!done)
            for (auto& kv : layers)
                if (kv.first < t.written && take(kv.second.get(), t.amax)) { done = true; break; }
        if (!done) lost.push_back((int)i);
    }
    return lost;
}

int Net::words_without_reset() const {
    if (!amax_dev_) return 0;
    std::map<const Layer*, int> room;
    for (auto& kv : layers) room[kv.second.get()] = kv.second->reset_room();
    return (int)place_range_resets([&](Layer* l, unsigned*) { return room[l]-- > 0; }).size();
}

// A tensor for which no layer is found loses its word.
void Net::assign_range_resets() {
    if (!amax_dev_) return;
    const std::vector<int> lost = place_range_resets([](Layer* l, unsigned* word) { return l->add_range_reset(word); });
    for (int i : lost) tensors[i].amax = nullptr;
    if (!lost.empty()) {
        // layers copied the word addresses into their kernel arguments during setup: let them look again
        for (auto& kv : layers) kv.second->setup_ranges();
    }
}

void Net::dump_layer(Layer* l) {
    // Engine::enableIntermediateOutput (base/engine.cpp:174-181,602-604): <name>_<seq>.bin, CHW fp32
    if (!l->has_own_output()) return;
    const TView& v = l->tout().v;
    std::vector<float> host((size_t)v.c * v.h * v.w);
    copy_result(l->d.number, host.data(), 0);
    char path[1024];
    snprintf(path, sizeof(path), "%s/%s_%llu.bin", dump_dir.c_str(), l->d.name, (unsigned long long)seq);
    FILE* f = fopen(path, "wb");
    if (!f) fail(FYN_ERR_INVALID, "cannot write %s", path);
    fwrite(host.data(), sizeof(float), host.size(), f);
    fclose(f);
}

void Net::run_layers(bool with_events) {
    for (auto& kv : layers) {
        Layer* l = kv.second.get();
        if (with_events) {
            if (!l->ev0) {
                FYN_HIP(hipEventCreate(&l->ev0));
                FYN_HIP(hipEventCreate(&l->ev1));
            }
            FYN_HIP(hipEventRecord(l->ev0, stream));
        }
        if (poison_lds_ && launch_poison_lds(stream) != 0) fail(FYN_ERR_DEVICE, "LDS fill failed");
        l->forward(stream);
        FYN_HIP(hipGetLastError());
        if (with_events) FYN_HIP(hipEventRecord(l->ev1, stream));
        if (!dump_dir.empty()) dump_layer(l);
    }
}

void Net::collect_timings() {
    if (!events_pending_) return;
    for (auto& kv : layers) {
        Layer* l = kv.second.get();
        if (!l->ev0) continue;
        float ms = 0.f;
        if (hipEventElapsedTime(&ms, l->ev0, l->ev1) == hipSuccess) {
            l->ms_total += ms;
            l->runs++;
        }
    }
    events_pending_ = false;
}

void Net::forward(uint64_t* seq_out) {
    if (!is_setup) fail(FYN_ERR_STATE, "forward() called on a network that was not set up");
    FYN_HIP(hipSetDevice(device));
    seq++;
    if (seq_out) *seq_out = seq;
    const bool plain = timings || !dump_dir.empty();
    if (graph_enabled_ && !plain) {
        if (!graph_exec_) {
            FYN_HIP(hipStreamBeginCapture(stream, hipStreamCaptureModeThreadLocal));
            try {
                run_layers(false);
            } catch (...) {
                hipGraph_t g = nullptr;
                (void)hipStreamEndCapture(stream, &g);
                if (g) (void)hipGraphDestroy(g);
                throw;
            }
            FYN_HIP(hipStreamEndCapture(stream, &graph_));
            FYN_HIP(hipGraphInstantiate(&graph_exec_, graph_, nullptr, nullptr, 0));
        }
        FYN_HIP(hipGraphLaunch(graph_exec_, stream));
        return;
    }
    if (timings) {
        FYN_HIP(hipStreamSynchronize(stream));
        collect_timings();
    }
    run_layers(timings);
    events_pending_ = timings;
}

void Net::finish() {
    FYN_HIP(hipSetDevice(device));
    if (events_pending_) {
        FYN_HIP(hipStreamSynchronize(stream));
        collect_timings();
        return;
    }
    const HostDone done = signal_.next();
    launch_tell_host(done, stream);
    FYN_HIP(hipGetLastError());
    signal_.wait(done.value, stream);
}

// Behind launches that use the caller's memory or an area on loan: a failure is reported when none of them runs any more.
void Net::check_queued() {
    const hipError_t e = hipGetLastError();
    if (e == hipSuccess) return;
    (void)hipStreamSynchronize(stream);
    fail(FYN_ERR_DEVICE, "launch failed: %s", hipGetErrorString(e));
}

void Net::count_area(size_t bytes, size_t& most) {
    if (bytes <= most) return;
    most = bytes;
    alloc_calls_++;
    alloc_bytes_ += bytes;
}

// Page-locked memory for a result on its way to the caller's, on loan for one call.
HostLoan Net::out_area(size_t floats) {
    const size_t bytes = floats * sizeof(float);
    HostLoan l(bytes);
    count_area(bytes, out_most_);
    return l;
}

void Net::use_graph(bool enable) {
    graph_enabled_ = enable;
    if (!enable && graph_exec_) {
        FYN_HIP(hipStreamSynchronize(stream));
        (void)hipGraphExecDestroy(graph_exec_);
        (void)hipGraphDestroy(graph_);
        graph_exec_ = nullptr;
        graph_ = nullptr;
    }
}

const Tensor& Net::input_tensor(int layer_no, int port) {
    if (!is_setup) fail(FYN_ERR_STATE, "set_input() before setup()");
    Layer* l = layer(layer_no);
    if (l->d.type == FYN_LAYER_UPLOAD) return l->tout();
    if (port < 0 || port >= l->num_ports()) fail(FYN_ERR_INVALID, "layer %s has no input port %d", l->d.name, port);
    const Tensor& t = l->tin(port);
    if (t.producer != -1) fail(FYN_ERR_INVALID, "input port %d of layer %s is fed by layer %d", port, l->d.name, t.producer);
    return t;
}

size_t Net::input_floats(int layer_no, int port) {
    const TView& v = input_tensor(layer_no, port).v;
    return (size_t)v.c * v.h * v.w;
}

void Net::async_sizes(size_t* in_floats, size_t* out_floats) const {
    if (slots_.empty()) fail(FYN_ERR_STATE, "no frame pipeline is active");
    *in_floats = async_in_floats_;
    *out_floats = async_out_floats_;
}

// A result in pieces: while the link moves one, the host copies the one before.  Pieces below a megabyte are not worth
// their launches (4 us each).
static size_t piece_pixels(size_t npix, size_t bytes) {
    const size_t pieces = std::min<size_t>(12, std::max<size_t>(1, bytes / (1280u << 10)));
    return std::max<size_t>(4, ((npix + pieces - 1) / pieces + 3) & ~size_t(3));
}

// How soon a workgroup looks again for pixels that are not there: not before a copy at 80 GB/s (10 ns a tick; four cores of
// the host this was measured on reach 100) could have brought them.  Behind a slower copy it looks again after the time
// that the rest would take at that rate, so the rate decides how many looks there are and not how long a frame takes.
static constexpr float kTicksPerByte = 1.f / 800.f;

// A frame into its tensor.  Host memory: the converting launch is queued first and takes the pixels as the host puts them
// into page-locked memory (HostFeed), so that launch latency, copy and transfer overlap: 3.8 MB in 90 us instead of 135 for
// two copies with a launch behind each.
void Net::upload(const float* data, int order, const TView& v, unsigned* amax) {
    const size_t npix = (size_t)v.h * v.w, plane = (npix + 31) & ~size_t(31);
    const bool planes = order == FYN_ORDER_CHANNELWISE;
    const Memory kind = memory_of(data);
    const UploadRange range{amax, upload_words_};
    if (kind == Memory::Device) {
        float* st = staging(plane * v.c);
        for (int c = 0; c < (planes ? v.c : 1); c++)
            FYN_HIP(hipMemcpyAsync(st + c * plane, data + c * npix, npix * (planes ? 1 : v.c) * sizeof(float), hipMemcpyDefault, stream));
        if (planes) launch_chw_to_tensor(st, plane, v, range, HostFeed{}, HostDone{}, true, stream);
        else launch_hwc_to_tensor(st, v, range, HostFeed{}, HostDone{}, true, stream);
        FYN_HIP(hipGetLastError());
        FYN_HIP(hipStreamSynchronize(stream));   // the caller's buffer is borrowed for this call only
        return;
    }
    // Page-locked memory may be the target of the application's work on the default stream, which the network's stream runs
    // behind: the host reads when that has ended.  (The pool's blocks hold results that have been waited for.)
    if (kind == Memory::PageLocked && !HostPool::contains(data, npix * v.c * sizeof(float))) {
        const HostDone done = signal_.next();
        launch_tell_host(done, stream);
        check_queued();
        signal_.wait(done.value, stream);
    }
    // (a caller that never waits is held at a few frames)
    const size_t bytes = plane * v.c * sizeof(float);
    unsigned& before = uploads_told_[upload_no_++ % kUploads];
    if (before) signal_.wait(before, stream);
    size_t under_way = 0;   // (areas of earlier frames that their launches still read)
    for (unsigned told : uploads_told_) under_way += told && !signal_.reached(told);
    HostLoan area(bytes, true);
    count_area(bytes, in_most_[under_way]);
    float* st = area.floats();
    // pieces: a small one first, so that the launch has something to do when it starts; multiples of 32 pixels (whole lines)
    HostCopy copies;   // (made before the loan ends, whatever happens)
    std::vector<std::pair<size_t, size_t>> pieces;   // copies made, pixels complete
    const size_t most = std::max<size_t>(4096, (256u << 10) / (v.c * sizeof(float)) & ~size_t(31));
    size_t step = most / 8 & ~size_t(31);
    for (size_t p0 = 0; p0 < npix;) {
        const size_t p1 = std::min(npix, p0 + step);
        for (int c = 0; c < (planes ? v.c : 1); c++)
            copies.add(st + (planes ? c * plane + p0 : p0 * v.c), data + (planes ? c * npix + p0 : p0 * v.c), (p1 - p0) * (planes ? 1 : v.c) * sizeof(float));
        pieces.push_back({copies.mark(), p1});
        p0 = p1;
        step = std::min(most, step * 2);
    }
    auto launch = [&](const HostFeed& feed) {
        const HostDone done = signal_.next();
        if (planes) launch_chw_to_tensor(st, plane, v, range, feed, done, false, stream);
        else launch_hwc_to_tensor(st, v, range, feed, done, false, stream);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) {
            // (one that is not running will not tell, and one that is runs to its end once the frame is there)
            copies.upto(copies.mark());
            if (feed.word) __atomic_store_n(&feed.word->ready, feed.base + (unsigned)npix, __ATOMIC_RELEASE);
            (void)hipStreamSynchronize(stream);
            fail(FYN_ERR_DEVICE, "converting a frame failed: %s", hipGetErrorString(e));
        }
        before = done.value;
        area.used_until(signal_, done.value);
    };
    copies.start();
    if (!feed_ahead_) {
        copies.upto(copies.mark());
        launch(HostFeed{});
        return;
    }
    const HostFeed feed{feed_, feed_base_, (float)v.c * (float)sizeof(float) * kTicksPerByte, feed_give_up_};
    feed_base_ += (unsigned)npix;
    launch(feed);
    for (const auto& piece : pieces) {
        copies.upto(piece.first);
        __atomic_store_n(&feed_->ready, feed.base + (unsigned)piece.second, __ATOMIC_RELEASE);
    }
    __atomic_thread_fence(__ATOMIC_SEQ_CST);   // (the progress has been told before the look)
    if (__atomic_load_n(&feed_->late, __ATOMIC_RELAXED)) {   // a slow source, a stopped process: the frame is complete now
        signal_.wait(before, stream);
        feed_->late = 0;
        launch(HostFeed{});
    }
}

void Net::set_input(int layer_no, int port, const float* data, int order) {
    if (!is_setup) fail(FYN_ERR_STATE, "set_input() before setup()");
    if (!data) fail(FYN_ERR_INVALID, "null input buffer");
    FYN_HIP(hipSetDevice(device));
    const Tensor& t = input_tensor(layer_no, port);
    if (order != FYN_ORDER_CHANNELWISE && order != FYN_ORDER_GPU_SHALLOW) fail(FYN_ERR_UNSUPPORTED, "input order %d not supported for upload", order);
    upload(data, order, t.v, t.amax);
}

// What a layer hands out: its output tensor; a layer that only passes its input on (download) may name up to three
// channels more or fewer than were produced, inside the same group of four (the extra ones are zero).
static TView result_view(Layer* l) {
    TView v = l->tout().v;
    if (!l->has_own_output()) v.c = std::min(l->oc, v.cp);
    return v;
}

// CHW planes of a tensor into the caller's memory.  Memory that the GPU reaches (HostPool) is written by the converting
// launch itself; anything else is filled from the staging area piece by piece, behind the launches that fill that.
void Net::download_planes(const TView& v, int include_padding, float* out) {
    const size_t npix = include_padding ? (size_t)v.hp() * v.wp() : (size_t)v.h * v.w, bytes = npix * v.c * sizeof(float);
    if (!host_memory(out)) {
        float* st = staging(npix * v.c);
        launch_tensor_to_chw(v, st, npix, include_padding, 0, npix, HostDone{}, true, stream);
        check_queued();
        FYN_HIP(hipMemcpyAsync(out, st, bytes, hipMemcpyDefault, stream));
        FYN_HIP(hipStreamSynchronize(stream));
        return;
    }
    if (HostPool::contains(out, bytes)) {
        const HostDone done = signal_.next();
        launch_tensor_to_chw(v, out, npix, include_padding, 0, npix, done, false, stream);
        check_queued();
        signal_.wait(done.value, stream);
        return;
    }
    const size_t plane = npix < 64 ? npix : (npix + 3) & ~size_t(3);
    HostLoan loan = out_area(plane * v.c);
    float* st = loan.floats();
    const size_t step = piece_pixels(npix, bytes);
    const unsigned first = signal_.last() + 1;
    for (size_t p0 = 0; p0 < npix; p0 += step) {
        const HostDone done = signal_.next();
        launch_tensor_to_chw(v, st, plane, include_padding, p0, std::min(npix, p0 + step), done, false, stream);
        loan.used_until(signal_, done.value);
    }
    check_queued();
    unsigned value = first;
    for (size_t p0 = 0; p0 < npix; p0 += step) {
        const size_t p1 = std::min(npix, p0 + step);
        signal_.wait(value++, stream);
        HostCopy copies;
        for (int c = 0; c < v.c; c++) copies.add(out + c * npix + p0, st + c * plane + p0, (p1 - p0) * sizeof(float));
        copies.start();
    }
}

// The same for interleaved pixels of pc floats.
void Net::download_pixels(const TView& v, int pc, float* out) {
    const size_t npix = (size_t)v.h * v.w, bytes = npix * pc * sizeof(float);
    // (a pixel is one store of up to sixteen bytes)
    const bool host = host_memory(out), direct = host && (reinterpret_cast<size_t>(out) & 15) == 0 && HostPool::contains(out, bytes);
    HostLoan loan = host && !direct ? out_area(npix * pc) : HostLoan();
    float* st = direct ? out : host ? loan.floats() : staging(npix * pc);
    const size_t step = host && !direct ? piece_pixels(npix, bytes) : npix;
    const unsigned first = signal_.last() + 1;
    for (size_t p0 = 0; p0 < npix; p0 += step) {
        const HostDone done = signal_.next();
        launch_tensor_to_hwc(v, st, pc, p0, std::min(npix, p0 + step), done, false, stream);
        loan.used_until(signal_, done.value);
    }
    check_queued();
    unsigned value = first;
    for (size_t p0 = 0; p0 < npix; p0 += step) {
        signal_.wait(value++, stream);
        if (host && !direct) memcpy(out + p0 * pc, st + p0 * pc, (std::min(npix, p0 + step) - p0) * pc * sizeof(float));
    }
    if (!host) {
        FYN_HIP(hipMemcpyAsync(out, st, bytes, hipMemcpyDefault, stream));
        FYN_HIP(hipStreamSynchronize(stream));
    }
}

// Indices and values of an arg-max layer, either of them where it is wanted.
void Net::download_argmax(const int* idx_dev, const TView& v, int32_t* idx, float* val) {
    const size_t n = (size_t)v.h * v.w, area = (n + 63) & ~size_t(63);
    if (!idx && !val) return finish();
    const bool direct = (!idx || (host_memory(idx) && HostPool::contains(idx, n * 4))) && (!val || (host_memory(val) && HostPool::contains(val, n * 4)));
    const bool host = (!idx || host_memory(idx)) && (!val || host_memory(val));
    HostLoan loan = host && !direct ? out_area(2 * area) : HostLoan();
    float* st = direct ? nullptr : host ? loan.floats() : staging(2 * area);
    int* di = !idx ? nullptr : direct ? idx : reinterpret_cast<int*>(st);
    float* dv = !val ? nullptr : direct ? val : st + area;
    const HostDone done = signal_.next();
    launch_argmax_to_host(idx_dev, v, di, dv, 0, n, done, stream);
    loan.used_until(signal_, done.value);
    check_queued();
    signal_.wait(done.value, stream);
    if (direct) return;
    if (idx) FYN_HIP(host ? (memcpy(idx, di, n * 4), hipSuccess) : hipMemcpy(idx, di, n * 4, hipMemcpyDefault));
    if (val) FYN_HIP(host ? (memcpy(val, dv, n * 4), hipSuccess) : hipMemcpy(val, dv, n * 4, hipMemcpyDefault));
}

void Net::copy_result(int layer_no, float* chw, int include_padding) {
    if (!is_setup) fail(FYN_ERR_STATE, "copy_result() before setup()");
    FYN_HIP(hipSetDevice(device));
    download_planes(result_view(layer(layer_no)), include_padding, chw);
}

void Net::copy_result_static(int layer_no, float* chw, int include_padding) {
    if (!is_setup) fail(FYN_ERR_STATE, "copy_result() before setup()");
    if (!chw) fail(FYN_ERR_INVALID, "null result buffer");
    FYN_HIP(hipSetDevice(device));
    Layer* l = layer(layer_no);
    const TView v = result_view(l);
    const size_t n = include_padding ? (size_t)v.c * v.hp() * v.wp() : (size_t)v.c * v.h * v.w;
    if (n > (size_t)FYN_STATIC_SCRATCH_FLOATS)
        fail(FYN_ERR_INVALID, "result of layer %s (%d) has %zu floats, the fixed staging area holds %zu: use fyn_layer_copy_result",
             l->d.name, l->d.number, n, (size_t)FYN_STATIC_SCRATCH_FLOATS);
    // every element of [0, n) is written by the conversion kernel: nothing of an earlier call is read
    launch_tensor_to_chw(v, static_scratch_, include_padding ? (size_t)v.hp() * v.wp() : (size_t)v.h * v.w, include_padding, 0,
                         include_padding ? (size_t)v.hp() * v.wp() : (size_t)v.h * v.w, HostDone{}, true, stream);
    FYN_HIP(hipGetLastError());
    FYN_HIP(hipMemcpyAsync(chw, static_scratch_, n * sizeof(float), hipMemcpyDefault, stream));
    FYN_HIP(hipStreamSynchronize(stream));
}

static void deep_tiling(int channels, int& tx, int& ty) {
    // CPUBufferShape::computeDeepTiling (cpu/cpubuffershape.cpp:430-448)
    const int tiles = (channels + 3) / 4;
    int best = 1 << 30;
    tx = tiles;
    ty = 1;
    for (int y = 1; y <= tiles; y++)
        for (int x = y; x <= tiles; x++)
            if (x * y >= tiles) {
                const int cost = (x - y) + (x * y - tiles);
                if (cost < best) {
                    best = cost;
                    tx = x;
                    ty = y;
                }
            }
}

void Net::get_output(int layer_no, float* data, int order) {
    if (!is_setup) fail(FYN_ERR_STATE, "get_output() before setup()");
    FYN_HIP(hipSetDevice(device));
    Layer* l = layer(layer_no);
    const TView v = result_view(l);
    if (order == FYN_ORDER_CHANNELWISE) {
        copy_result(layer_no, data, 0);
    } else if (order == FYN_ORDER_GPU_SHALLOW) {
        if (v.c > 4) fail(FYN_ERR_UNSUPPORTED, "GPU_SHALLOW download holds at most 4 channels per texel (layer has %d)", v.c);
        download_pixels(v, v.c == 3 ? 4 : v.c, data);  // rendered textures are RGBA (base/buffermanager.cpp:478-483)
    } else if (order == FYN_ORDER_GPU_DEEP) {
        // tiled RGBA buffer, tile t at grid (t % tx, t / tx), padding shared between tiles
        // (gpu/deep/deeptiler.cpp:63-110)
        std::vector<float> chw((size_t)v.c * v.h * v.w);
        copy_result(layer_no, chw.data(), 0);
        int tx, ty;
        deep_tiling(v.c, tx, ty);
        const int pad = v.pad;
        const int dw = tx * (v.w + pad) + pad, dh = ty * (v.h + pad) + pad;
        memset(data, 0, (size_t)dw * dh * 4 * sizeof(float));
        for (int ch = 0; ch < v.c; ch++) {
            const int t = ch / 4, comp = ch % 4, gx = t % tx, gy = t / tx;
            for (int y = 0; y < v.h; y++)
                for (int x = 0; x < v.w; x++)
                    data[(((size_t)(pad + gy * (v.h + pad) + y)) * dw + pad + gx * (v.w + pad) + x) * 4 + comp] =
                        chw[((size_t)ch * v.h + y) * v.w + x];
        }
    } else {
        fail(FYN_ERR_INVALID, "unknown buffer order %d", order);
    }
}

void Net::time_forward(int iters, float* ms) {
    if (!is_setup) fail(FYN_ERR_STATE, "time_forward() before setup()");
    FYN_HIP(hipSetDevice(device));
    hipEvent_t a, b;
    FYN_HIP(hipEventCreate(&a));
    FYN_HIP(hipEventCreate(&b));
    const bool t = timings;
    timings = false;
    FYN_HIP(hipEventRecord(a, stream));
    for (int i = 0; i < iters; i++) forward(nullptr);
    FYN_HIP(hipEventRecord(b, stream));
    FYN_HIP(hipEventSynchronize(b));
    timings = t;
    FYN_HIP(hipEventElapsedTime(ms, a, b));
    (void)hipEventDestroy(a);
    (void)hipEventDestroy(b);
}

void Net::time_steps(int iters, float* ms_each) {
    if (!is_setup) fail(FYN_ERR_STATE, "time_steps() before setup()");
    if (iters > 65536) fail(FYN_ERR_INVALID, "at most 65536 steps per call");
    FYN_HIP(hipSetDevice(device));
    // one event after every forward pass, all queued without waiting; differences of consecutive events are the steps
    std::vector<hipEvent_t> ev((size_t)iters + 1, nullptr);
    const bool t = timings;
    timings = false;
    try {
        for (auto& e : ev) FYN_HIP(hipEventCreate(&e));
        FYN_HIP(hipEventRecord(ev[0], stream));
        for (int i = 0; i < iters; i++) {
            forward(nullptr);
            FYN_HIP(hipEventRecord(ev[(size_t)i + 1], stream));
        }
        FYN_HIP(hipEventSynchronize(ev[(size_t)iters]));
        for (int i = 0; i < iters; i++) FYN_HIP(hipEventElapsedTime(&ms_each[i], ev[(size_t)i], ev[(size_t)i + 1]));
    } catch (...) {
        timings = t;
        (void)hipStreamSynchronize(stream);
        for (auto e : ev) if (e) (void)hipEventDestroy(e);
        throw;
    }
    timings = t;
    for (auto e : ev) (void)hipEventDestroy(e);
}

void Net::weights_changed() {
    if (!graph_exec_) return;
    FYN_HIP(hipSetDevice(device));
    FYN_HIP(hipStreamSynchronize(stream));
    (void)hipGraphExecDestroy(graph_exec_);
    (void)hipGraphDestroy(graph_);
    graph_exec_ = nullptr;
    graph_ = nullptr;
}

void Net::time_layer(int layer_no, int iters, float* ms) {
    if (!is_setup) fail(FYN_ERR_STATE, "time_layer() before setup()");
    FYN_HIP(hipSetDevice(device));
    Layer* l = layer(layer_no);
    // The launches are captured into one hipGraph so that host-side dispatch gaps do not enter the
    // measurement; the events bracket the graph on the network's stream.
    hipGraph_t g = nullptr;
    hipGraphExec_t ge = nullptr;
    FYN_HIP(hipStreamBeginCapture(stream, hipStreamCaptureModeThreadLocal));
    try {
        for (int i = 0; i < iters; i++) l->forward(stream);
    } catch (...) {
        (void)hipStreamEndCapture(stream, &g);
        if (g) (void)hipGraphDestroy(g);
        throw;
    }
    FYN_HIP(hipStreamEndCapture(stream, &g));
    FYN_HIP(hipGraphInstantiate(&ge, g, nullptr, nullptr, 0));
    hipEvent_t a, b;
    FYN_HIP(hipEventCreate(&a));
    FYN_HIP(hipEventCreate(&b));
    FYN_HIP(hipGraphLaunch(ge, stream));  // warm-up
    FYN_HIP(hipEventRecord(a, stream));
    FYN_HIP(hipGraphLaunch(ge, stream));
    FYN_HIP(hipEventRecord(b, stream));
    FYN_HIP(hipEventSynchronize(b));
    FYN_HIP(hipGetLastError());
    FYN_HIP(hipEventElapsedTime(ms, a, b));
    (void)hipEventDestroy(a);
    (void)hipEventDestroy(b);
    (void)hipGraphExecDestroy(ge);
    (void)hipGraphDestroy(g);
}

// ---------------------------------------------------------------------------------------------
// Frame pipeline (the counterpart of the reference engine's asynchronous mode, base/engine.cpp:386-683, with
// its two upload/download buffer sets, gpu/uploadlayer.h:74).  Two forms:
//   overlapped   for one network with large frames:
//                up stream    page-locked slot -> device staging slot (copy engine), piece by piece behind the host's copy
//                main stream  staging -> input tensor, all layers, output tensor -> device staging slot
//                down stream  device staging slot -> page-locked slot (copy engine).  The copy is made as one of rows with
//                gaps between them: some versions of the runtime carry out plain copies to the host with a kernel, and
//                every workgroup of such a kernel keeps a CU for the 90 us of a frame from layers that need it whole.
//                The streams are not joined by events: while a queue of the GPU waits for another one's signal, every
//                launch on the main stream starts about a microsecond later (18 launches beside a copy each way: 173 us
//                without events, 219 with them).  A thread of the pipeline's own joins them: it lets the launch that
//                converts the frame go on when the upload has ended (HostFeed; in a running pipeline that is long before
//                the launch's turn), sends the result on its way when the last launch has told so, and delivers it.
//   in place     everything on the network's stream, the layout kernels reading and writing the page-locked slots over
//                the link: networks that run side by side overlap each other's transfers, and where the transfers of a
//                frame are short (1 MB) nothing is gained by streams of their own.
// There is one slot more than frames that may be in flight between two calls: submit() queues its frame first and
// sees to the delivery of the one that has to leave afterwards, so that the GPU has the next frame in its queue.
// ---------------------------------------------------------------------------------------------
static constexpr size_t kRowGap = 256;   // bytes between the rows of an overlapped download

void Net::async_begin(int in_layer, int in_port, int in_order, int out_layer, int out_order, int depth, bool copy_streams) {
    if (!is_setup) fail(FYN_ERR_STATE, "async_begin() before setup()");
    if (!slots_.empty()) fail(FYN_ERR_STATE, "frame pipeline is already active");
    if (depth < 1 || depth > kMaxDepth) fail(FYN_ERR_INVALID, "pipeline depth %d out of range (1..%d)", depth, kMaxDepth);
    FYN_HIP(hipSetDevice(device));
    Layer* li = layer(in_layer);
    if (li->d.type == FYN_LAYER_UPLOAD) {
        async_in_ = &li->tout();
    } else {
        if (in_port < 0 || in_port >= li->num_ports()) fail(FYN_ERR_INVALID, "layer %s has no input port %d", li->d.name, in_port);
        async_in_ = &li->tin(in_port);
        if (async_in_->producer != -1) fail(FYN_ERR_INVALID, "input port %d of layer %s is fed by layer %d", in_port, li->d.name, async_in_->producer);
    }
    async_out_ = &layer(out_layer)->tout();
    async_out_view_ = result_view(layer(out_layer));
    const TView& vi = async_in_->v;
    const TView& vo = async_out_view_;
    if (in_order != FYN_ORDER_CHANNELWISE && in_order != FYN_ORDER_GPU_SHALLOW) fail(FYN_ERR_UNSUPPORTED, "input order %d not supported for upload", in_order);
    if (out_order == FYN_ORDER_GPU_SHALLOW) {
        if (vo.c > 4) fail(FYN_ERR_UNSUPPORTED, "GPU_SHALLOW download holds at most 4 channels per texel (layer has %d)", vo.c);
        async_out_floats_ = (size_t)vo.h * vo.w * (vo.c == 3 ? 4 : vo.c);
    } else if (out_order == FYN_ORDER_CHANNELWISE) {
        async_out_floats_ = (size_t)vo.c * vo.h * vo.w;
    } else {
        fail(FYN_ERR_UNSUPPORTED, "output order %d not supported by the frame pipeline", out_order);
    }
    async_in_floats_ = (size_t)vi.c * vi.h * vi.w;
    async_in_plane_ = ((size_t)vi.h * vi.w + 3) & ~size_t(3);
    async_in_order_ = in_order;
    async_out_order_ = out_order;
    async_own_streams_ = copy_streams && (async_in_floats_ + async_out_floats_) * sizeof(float) > (1u << 20);
    async_depth_ = depth;
    const size_t in_bytes = async_in_plane_ * vi.c * sizeof(float), out_bytes = async_out_floats_ * sizeof(float);
    if (async_own_streams_) {
        up_stream_ = lease_stream(device, true);
        down_stream_ = lease_stream(device, true);
        const size_t rows = std::max<size_t>(4, (out_bytes + (1u << 20) - 1) >> 20);
        async_row_ = (out_bytes / rows + 255 + 1) & ~size_t(255);
        async_rows_ = (out_bytes + async_row_ - 1) / async_row_;
    }
    slots_ = std::vector<AsyncSlot>(depth + 1);
    const size_t pin_out_bytes = async_own_streams_ ? async_rows_ * (async_row_ + kRowGap) : out_bytes;
    for (size_t i = 0; i < slots_.size(); i++) {
        AsyncSlot& s = slots_[i];
        s.pin_in = static_cast<float*>(HostPool::acquire(in_bytes, false, true));
        s.pin_out = static_cast<float*>(HostPool::acquire(pin_out_bytes, false));
        count_area(in_bytes, slot_in_most_[i]);
        count_area(pin_out_bytes, slot_out_most_[i]);
        if (!async_own_streams_) continue;
        FYN_HIP(hipMalloc(reinterpret_cast<void**>(&s.dev_in), in_bytes));
        FYN_HIP(hipMalloc(reinterpret_cast<void**>(&s.dev_out), async_rows_ * async_row_));
        alloc_calls_ += 2;
        alloc_bytes_ += in_bytes + async_rows_ * async_row_;
    }
    if (async_own_streams_) {
        carry_end_ = carry_stale_ = false;
        carry_error_ = nullptr;
        uploads_ = 0;
        async_pixels_ = (size_t)vi.h * vi.w;
        async_feed_ = static_cast<FeedWord*>(HostPool::acquire(sizeof(FeedWord), false));
        *async_feed_ = FeedWord{};
        carrier_ = std::thread([this] { carry(); });
    }
}

constexpr size_t kPipelineShared = 1u << 20;   // copies of a pipeline from this size on are shared with the helper threads

// The caller's memory takes what a slot's download left in page-locked memory.
static void add_rows(HostCopy& copies, float* to, const float* from, size_t bytes, size_t row, size_t gap) {
    for (size_t o = 0, r = 0; o < bytes; o += row, r++)
        copies.add(reinterpret_cast<char*>(to) + o, reinterpret_cast<const char*>(from) + r * (row + gap), std::min(row, bytes - o));
}

void Net::async_complete(AsyncSlot& s) {
    if (async_own_streams_) {
        for (int i = 0; i < 4096 && s.busy.load(std::memory_order_acquire); i++) _mm_pause();
        for (;;) {
            {
                std::unique_lock<std::mutex> lk(carry_mu_);
                carry_done_.wait(lk, [&] { return !s.busy.load(std::memory_order_acquire) || carry_error_ || carry_stale_; });
                if (carry_error_) std::rethrow_exception(carry_error_);
                if (!carry_stale_) return;
            }
            async_again();
        }
    }
    if (!s.busy) return;
    signal_.wait(s.value, stream);
    if (s.user_out) {
        HostCopy out;
        const size_t bytes = async_out_floats_ * sizeof(float);
        add_rows(out, s.user_out, s.pin_out, bytes, bytes, 0);
        out.start(kPipelineShared);
    }
    s.busy = false;
}

// A frame's conversion, layers and result, on the network's stream.
void Net::queue_frame(AsyncSlot& s) {
    const TView &vi = async_in_->v, &vo = async_out_view_;
    const size_t opix = (size_t)vo.h * vo.w;
    const float* src = async_own_streams_ ? s.dev_in : s.pin_in;
    float* dst = async_own_streams_ ? s.dev_out : s.pin_out;
    const UploadRange range{async_in_->amax, upload_words_};
    if (async_in_order_ == FYN_ORDER_CHANNELWISE) launch_chw_to_tensor(src, async_in_plane_, vi, range, HostFeed{}, HostDone{}, async_own_streams_, stream);
    else launch_hwc_to_tensor(src, vi, range, HostFeed{}, HostDone{}, async_own_streams_, stream);
    forward(nullptr);
    const HostDone done = signal_.next();
    if (async_out_order_ == FYN_ORDER_CHANNELWISE) launch_tensor_to_chw(vo, dst, opix, 0, 0, opix, done, async_own_streams_, stream);
    else launch_tensor_to_hwc(vo, dst, vo.c == 3 ? 4 : vo.c, 0, opix, done, async_own_streams_, stream);
    FYN_HIP(hipGetLastError());
    s.value = done.value;
}

// A frame was computed before its upload had arrived (the process was stopped while the frame's launches waited): it and
// the ones behind it are computed again.  The pipeline's thread leaves them alone until then; a frame keeps its slot, and
// so its place in device memory, until its result has been delivered.
void Net::async_again() {
    FYN_HIP(hipStreamSynchronize(up_stream_));
    FYN_HIP(hipStreamSynchronize(stream));
    async_feed_->late = 0;   // (no launch waits any more)
    for (AsyncSlot* s : carried_) queue_frame(*s);
    std::lock_guard<std::mutex> lk(carry_mu_);
    carry_stale_ = false;
}

// Whether the copies on a stream of the pipeline's are through (asked: an event would occupy a queue of the GPU).
static bool copies_made(hipStream_t st) {
    const hipError_t e = hipStreamQuery(st);
    if (e != hipErrorNotReady) FYN_HIP(e);
    return e == hipSuccess;
}

// The pipeline's thread.  Results leave in the order of submission; while one is being copied to the caller, the next is
// sent on its way and uploads are reported.
void Net::carry() {
    try {
        FYN_HIP(hipSetDevice(device));
        unsigned uploaded = 0;       // uploads reported
        AsyncSlot* sent = nullptr;   // its download is under way
        auto front = [&]() -> AsyncSlot* {
            std::lock_guard<std::mutex> lk(carry_mu_);
            return carried_.empty() ? nullptr : carried_.front();
        };
        auto turn = [&](bool idle) {
            const unsigned n = uploads_.load(std::memory_order_acquire);
            if (n != uploaded && copies_made(up_stream_)) {   // (all of the n frames' copies: they had been queued)
                __atomic_store_n(&async_feed_->ready, n * (unsigned)async_pixels_, __ATOMIC_RELEASE);
                uploaded = n;
            }
            if (!idle || carry_stale_) return;
            AsyncSlot* s = front();
            if (s && signal_.reached(s->value)) {
                if (__atomic_load_n(&async_feed_->late, __ATOMIC_ACQUIRE)) {
                    std::lock_guard<std::mutex> lk(carry_mu_);
                    carry_stale_ = true;
                    carry_done_.notify_all();
                    return;
                }
                FYN_HIP(hipMemcpy2DAsync(s->pin_out, async_row_ + kRowGap, s->dev_out, async_row_, async_row_, async_rows_, hipMemcpyDeviceToHost, down_stream_));
                sent = s;
            }
        };
        auto since = std::chrono::steady_clock::now();
        for (;;) {
            {
                std::unique_lock<std::mutex> lk(carry_mu_);
                if (carry_end_ && carry_stale_) return;   // (computing them again has failed)
                if (carried_.empty() && uploaded == uploads_.load(std::memory_order_acquire)) {
                    carry_more_.wait(lk, [&] { return carry_end_ || !carried_.empty() || uploaded != uploads_.load(std::memory_order_acquire); });
                    if (carry_end_ && carried_.empty()) return;
                    since = std::chrono::steady_clock::now();
                }
            }
            turn(!sent);
            if (!sent || !copies_made(down_stream_)) {
                for (int i = 0; i < 48; i++) _mm_pause();
                if (sent) continue;
                const auto waited = std::chrono::steady_clock::now() - since;
                if (waited > std::chrono::milliseconds(5)) std::this_thread::sleep_for(std::chrono::microseconds(20));   // (long frames)
                if (waited > std::chrono::seconds(1) && !carry_stale_) {   // something may have failed
                    AsyncSlot* s = front();
                    if (s && copies_made(stream) && !signal_.reached(s->value)) fail(FYN_ERR_DEVICE, "a launch ended without telling so");
                    since = std::chrono::steady_clock::now();
                }
                continue;
            }
            AsyncSlot* s = sent;
            sent = nullptr;
            {
                std::lock_guard<std::mutex> lk(carry_mu_);
                carried_.pop_front();
            }
            {
                HostCopy out;
                add_rows(out, s->user_out, s->pin_out, async_out_floats_ * sizeof(float), async_row_, kRowGap);
                out.start(kPipelineShared);
                for (size_t m = 1; m <= out.mark(); m++) {
                    turn(!sent);
                    out.upto(m);
                }
            }
            since = std::chrono::steady_clock::now();
            std::lock_guard<std::mutex> lk(carry_mu_);
            s->busy.store(false, std::memory_order_release);
            carry_done_.notify_all();
        }
    } catch (...) {
        std::lock_guard<std::mutex> lk(carry_mu_);
        carry_error_ = std::current_exception();
        carry_done_.notify_all();
    }
}

void Net::async_submit(const float* in, float* out, uint64_t* ticket) {
    if (slots_.empty()) fail(FYN_ERR_STATE, "async_submit() without async_begin()");
    if (!in || !out) fail(FYN_ERR_INVALID, "null frame buffer");
    FYN_HIP(hipSetDevice(device));
    AsyncSlot& s = slots_[async_seq_ % slots_.size()];
    async_complete(s);
    const TView& vi = async_in_->v;
    const size_t npix = (size_t)vi.h * vi.w;
    const bool planes = async_in_order_ == FYN_ORDER_CHANNELWISE;
    {
        HostCopy copies;
        if (planes)
            for (int c = 0; c < vi.c; c++) copies.add(s.pin_in + c * async_in_plane_, in + c * npix, npix * sizeof(float));
        else copies.add(s.pin_in, in, async_in_floats_ * sizeof(float));
        copies.start(kPipelineShared);
        if (async_own_streams_) {
            // (the copy engine follows in pieces of two megabytes and more)
            const size_t all = (planes ? async_in_plane_ * vi.c : async_in_floats_) * sizeof(float);
            const size_t pieces = std::max<size_t>(1, std::min<size_t>(8, all >> 21)), marks = copies.mark();
            size_t sent = 0;
            for (size_t m = 1; m <= pieces; m++) {
                copies.upto(marks * m / pieces);
                const size_t to = m == pieces ? all : copies.end_of(marks * m / pieces) - reinterpret_cast<char*>(s.pin_in);
                FYN_HIP(hipMemcpyAsync(reinterpret_cast<char*>(s.dev_in) + sent, reinterpret_cast<char*>(s.pin_in) + sent, to - sent, hipMemcpyHostToDevice, up_stream_));
                sent = to;
            }
        }
    }
    if (async_own_streams_) {
        const HostFeed feed{async_feed_, uploads_.load() * (unsigned)npix, 0.f, feed_give_up_};
        {
            std::lock_guard<std::mutex> lk(carry_mu_);
            uploads_++;
            carry_more_.notify_one();
        }
        if (feed_ahead_) launch_await_feed(feed, npix, stream);
        else FYN_HIP(hipStreamSynchronize(up_stream_));
    }
    queue_frame(s);
    s.user_out = out;
    s.busy = true;
    s.ticket = ++async_seq_;
    if (async_own_streams_) {
        std::lock_guard<std::mutex> lk(carry_mu_);
        carried_.push_back(&s);
        carry_more_.notify_one();
    }
    if (ticket) *ticket = s.ticket;
    if (async_seq_ > (uint64_t)async_depth_) async_complete(slots_[(async_seq_ - async_depth_ - 1) % slots_.size()]);
}

void Net::async_wait(uint64_t ticket) {
    if (slots_.empty()) fail(FYN_ERR_STATE, "async_wait() without async_begin()");
    FYN_HIP(hipSetDevice(device));
    if (ticket == 0 || ticket > async_seq_) fail(FYN_ERR_INVALID, "unknown frame ticket %llu", (unsigned long long)ticket);
    // frames complete in submission order: deliver everything up to the requested one
    for (uint64_t t = (async_seq_ > slots_.size() ? async_seq_ - slots_.size() + 1 : 1); t <= ticket; t++) {
        AsyncSlot& s = slots_[(t - 1) % slots_.size()];
        if (s.busy && s.ticket == t) async_complete(s);
    }
}

void Net::async_end() {
    if (slots_.empty()) return;
    (void)hipSetDevice(device);
    std::exception_ptr error;
    try {
        for (uint64_t t = (async_seq_ > slots_.size() ? async_seq_ - slots_.size() + 1 : 1); t <= async_seq_; t++) {
            AsyncSlot& s = slots_[(t - 1) % slots_.size()];
            if (s.busy && s.ticket == t) async_complete(s);
        }
    } catch (...) {
        error = std::current_exception();
    }
    if (carrier_.joinable()) {
        {
            std::lock_guard<std::mutex> lk(carry_mu_);
            carry_end_ = true;
            carry_more_.notify_one();
        }
        carrier_.join();
        carried_.clear();
        carry_error_ = nullptr;
    }
    if (stream) (void)hipStreamSynchronize(stream);
    if (up_stream_) (void)hipStreamSynchronize(up_stream_);
    if (down_stream_) (void)hipStreamSynchronize(down_stream_);
    for (AsyncSlot& s : slots_) {
        HostPool::release(s.pin_in);
        HostPool::release(s.pin_out);
        if (s.dev_in) (void)hipFree(s.dev_in);
        if (s.dev_out) (void)hipFree(s.dev_out);
    }
    HostPool::release(async_feed_);
    async_feed_ = nullptr;
    slots_.clear();
    return_stream(device, up_stream_);
    return_stream(device, down_stream_);
    up_stream_ = down_stream_ = nullptr;
    async_seq_ = 0;
    if (error) std::rethrow_exception(error);
}

}  // namespace fynhip
