// Host-side engine: network graph, device tensors, layer objects.  This is the part of the
// reference's base/ + gpu/ host code that survives the move from OpenGL to HIP:
//   LayerFactory / GPULayerFactoryBackend   -> Net::add_layer          (base/layerfactory.cpp, gpu/gpulayerfactory.cpp)
//   BufferManager                           -> Net::connect / assign_buffers (base/buffermanager.cpp)
//   NeuralNetwork / Engine (sync branch)    -> Net::setup / forward / finish (base/neuralnetwork.cpp, base/engine.cpp)
//   GPULayerBase subclasses                 -> Layer subclasses in layer_classes.h and layers.cpp
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <cstdarg>
#include <cstdio>
#include <deque>
#include <exception>
#include <map>
#include <memory>
#include <mutex>
#include <stdexcept>
#include <string>
#include <thread>
#include <vector>

#include "../../include/fynhip.h"
#include "host_io.h"
#include "kernels.h"

namespace fynhip {

// Error carried up to the C ABI (the reference throws FynException, common/fynexception.h).
struct Error : public std::runtime_error {
    int code;
    Error(int c, const std::string& m) : std::runtime_error(m), code(c) {}
};
[[noreturn]] void fail(int code, const char* fmt, ...) __attribute__((format(printf, 2, 3)));

#define FYN_HIP(call)                                                                              \
    do {                                                                                           \
        hipError_t e_ = (call);                                                                    \
        if (e_ != hipSuccess) ::fynhip::fail(FYN_ERR_DEVICE, "%s failed: %s (%s:%d)", #call,       \
                                             hipGetErrorString(e_), __FILE__, __LINE__);           \
    } while (0)

struct Tensor {
    TView v{};
    int producer = -1;     // layer number writing it (-1: external input)
    int written = -1;      // layer in whose launch that happens: the producer, or a layer in front that computes it as well
    int last_reader = -1;  // highest layer number in whose launch it is read
    bool locked = false;   // never reused (network outputs, external inputs)
    int buffer = -1;       // index into Net::buffers_
    unsigned* amax = nullptr;   // value-range word (range.h) when a producer keeps it, else null
};

struct DevBuffer {
    void* ptr = nullptr;
    size_t bytes = 0;
    int h = 0, w = 0, pad = 0, cp = 0, f16 = 0;  // geometry key (reuse only between identical geometries)
    int free_after = -1;                          // highest reader of the current tenant
    bool locked = false;
};

class Net;

// The FYNHIP_* environment switches (tests, experiments, tuning cache), read once when a network is created: nothing on
// a launch path, and nothing during a later setup or weight load, looks at the environment again.
class Switches {
  public:
    void read();                               // every variable of the environment whose name begins with FYNHIP_
    const char* get(const char* name) const;   // the value, or nullptr when the variable was not set (like getenv)
    bool on(const char* name) const { return get(name) != nullptr; }
  private:
    std::map<std::string, std::string> v_;
};

class Layer {
  public:
    Layer(Net* net, const fyn_layer_desc& d);
    virtual ~Layer() {}
    fyn_layer_desc d;
    Net* net;
    std::vector<int> in;  // tensor id per input port, -1 = not connected
    int out = -1;         // tensor id
    int oc = 0, oh = 0, ow = 0;  // output net shape

    virtual int num_ports() const { return (d.flags & FYN_FLAG_RESIDUAL_INPUT) ? 2 : 1; }
    // shape of the tensor expected on an input port (channels, h, w, padding)
    virtual void port_shape(int port, int& c, int& h, int& w, int& pad) const;
    virtual bool has_own_output() const { return true; }
    virtual size_t weight_floats() const { return 0; }
    virtual void load_weights(const float*) { fail(FYN_ERR_INVALID, "layer %s (%d) takes no weights", d.name, d.number); }
    virtual void setup() {}
    virtual void forward(hipStream_t s) = 0;
    virtual std::string info() const { return "none"; }
    // value ranges (range.h): whether this layer's kernels raise the word of their output tensor, and whether they can
    // take on clearing another tensor's word (true: taken)
    virtual bool tracks_range() const { return false; }
    virtual bool add_range_reset(unsigned*) { return false; }
    virtual int reset_room() const { return 0; }   // how many words it could still take
    virtual void setup_ranges() {}   // (re)reads the words of the layer's tensors into its kernel arguments
    // a sigmoid or tanh layer: its arguments, for the layer in front that computes it as well (computed_by), else null
    virtual const FuncParams* pointwise() const { return nullptr; }
    virtual void computed_by(int) {}
    Act act() const;
    const Tensor& tin(int port) const;
    const Tensor& tout() const;
    bool set_up = false;
    // timing
    hipEvent_t ev0 = nullptr, ev1 = nullptr;
    float ms_total = 0.f;
    int runs = 0;
};

class Net {
  public:
    Net(int device, int storage);
    Switches sw;
    ~Net();
    void add_layer(const fyn_layer_desc& d);
    void add_custom_layer(const fyn_layer_desc& d, const fyn_custom_layer& impl);
    void connect(int out_layer, int in_layer, int port);
    void setup();
    void forward(uint64_t* seq);
    void finish();
    Layer* layer(int number);
    void set_input(int layer, int port, const float* data, int order);
    const Tensor& input_tensor(int layer, int port);     // what set_input writes: an upload layer's output or an unconnected port
    size_t input_floats(int layer, int port);            // floats that set_input reads from the host buffer
    void async_sizes(size_t* in_floats, size_t* out_floats) const;   // per frame, of the active frame pipeline
    void copy_result(int layer, float* chw, int include_padding);
    void copy_result_static(int layer, float* chw, int include_padding);   // through the fixed staging area, no allocation
    void get_output(int layer, float* data, int order);
    void copy_argmax(int layer, int32_t* idx, float* val);
    void time_forward(int iters, float* ms);
    void time_steps(int iters, float* ms_each);
    // A captured forward pass holds kernel arguments by value (among them the power of two that undoes a layer's weight
    // pre-scaling): after a weight load on a set-up network the next forward() captures again.
    void weights_changed();
    void time_layer(int layer, int iters, float* ms);
    void use_graph(bool enable);
    // frame pipeline: upload of frame i+1 and download of frame i-1 overlap the layers of frame i
    void async_begin(int in_layer, int in_port, int in_order, int out_layer, int out_order, int depth, bool copy_streams);
    void async_submit(const float* in, float* out, uint64_t* ticket);
    void async_wait(uint64_t ticket);
    void async_end();

    int device;
    int storage;  // fyn_storage
    bool f16() const { return storage == FYN_STORAGE_F16; }
    bool is_setup = false;
    bool timings = false;
    bool reuse_buffers = true;
    // Layers fused into their neighbour's launch (fuse_depthwise_layers) run that way only in passes that neither time
    // nor dump single layers, and only in networks whose intermediate tensors may share buffers.
    bool fusion_on() const { return reuse_buffers && !timings && dump_dir.empty(); }
    // ... those that write the tensors in between where buffers aren't shared (the blocks and pairs that don't are not formed there)
    bool joined_on() const { return !timings && dump_dir.empty(); }
    std::string dump_dir;
    hipStream_t stream = nullptr;
    std::map<int, std::unique_ptr<Layer>> layers;  // ascending number = execution order
    std::vector<Tensor> tensors;
    std::vector<DevBuffer> buffers;
    uint64_t seq = 0;

    // Whether a tensor's buffer is the tensor's alone from layer `from` through layer `to`: no other tensor in it is
    // written by the launch of one of them, nor read by it.  Asked before a launch is made to write the tensor earlier
    // than its producer, or to read it later than its last reader; whoever does so enters it in `written` or
    // `last_reader`, which is what the next one to ask finds.
    bool alone(int tensor, int from, int to) const;
    // Tensors whose value-range word no launch would clear as things stand: they go without one (assign_range_resets).  A
    // fusion that takes launches away asks before and behind.
    int words_without_reset() const;
    void read_until(int tensor, int layer_no) { tensors[tensor].last_reader = std::max(tensors[tensor].last_reader, layer_no); }

    // device allocations owned by the net
    void* dev_alloc(size_t bytes, bool zero = true);
    void dev_free(void* p);   // setup-time only (waits for the stream)
    void dev_free_many(const std::vector<void*>& ptrs);   // the same for several areas, one wait
    float* staging(size_t floats);  // fp32 staging area in device memory, for callers whose buffers lie there

  private:
    struct AsyncSlot {
        float *pin_in = nullptr, *pin_out = nullptr, *dev_in = nullptr, *dev_out = nullptr;
        unsigned value = 0;   // what the stream's word reads when the frame's launches are through (in place: pin_out is filled then)
        float* user_out = nullptr;
        uint64_t ticket = 0;
        std::atomic<bool> busy{false};
    };
    std::vector<AsyncSlot> slots_;
    hipStream_t up_stream_ = nullptr, down_stream_ = nullptr;
    const Tensor* async_in_ = nullptr;
    const Tensor* async_out_ = nullptr;
    bool async_own_streams_ = true;
    int async_depth_ = 0;
    size_t async_row_ = 0, async_rows_ = 0;   // bytes of a row and rows of an overlapped download
    TView async_out_view_{};   // what the output layer hands out (a download layer may name other channel counts)
    int async_in_order_ = 0, async_out_order_ = 0;
    size_t async_in_floats_ = 0, async_out_floats_ = 0, async_in_plane_ = 0;   // (planes lie on multiples of four floats)
    uint64_t async_seq_ = 0;
    void async_complete(AsyncSlot& s);
    // overlapped pipelines: the thread that delivers results, and the frames handed to it
    std::thread carrier_;
    std::mutex carry_mu_;
    std::condition_variable carry_more_, carry_done_;
    std::deque<AsyncSlot*> carried_;
    std::exception_ptr carry_error_;
    std::atomic<unsigned> uploads_{0};     // frames whose upload has been queued
    FeedWord* async_feed_ = nullptr;       // pixels of them that have arrived in device memory
    size_t async_pixels_ = 0;              // of a frame
    bool carry_end_ = false;
    std::atomic<bool> carry_stale_{false};   // the result at the front was computed before its frame had arrived
    void carry();
    void async_again();
    void queue_frame(AsyncSlot& s);
    void run_layers(bool with_events);
    void release_all();
    void collect_timings();
    void dump_layer(Layer* l);
    std::vector<void*> allocs_;
  public:
    // allocations made for this network since it was created: calls of hipMalloc, and page-locked areas in use beyond
    // what was in use at once before (the pool may have had them); bytes asked for
    size_t alloc_calls_ = 0, alloc_bytes_ = 0;
  private:
    float* staging_ = nullptr;
    size_t staging_floats_ = 0;
    static constexpr unsigned kUploads = 4;   // areas of uploads that may be waiting for their launch
    static constexpr int kMaxDepth = 8;       // of a frame pipeline
    // largest page-locked areas so far: of an upload with so many others under way, of a read-back, of a pipeline's slots
    size_t in_most_[kUploads] = {}, out_most_ = 0, slot_in_most_[kMaxDepth + 1] = {}, slot_out_most_[kMaxDepth + 1] = {};
    unsigned uploads_told_[kUploads] = {}, upload_no_ = 0;
    HostSignal signal_;
    FeedWord* feed_ = nullptr;          // progress of the host's copies into the input area
    unsigned feed_base_ = 0;            // ... when all frames so far have been copied
    bool feed_ahead_ = true;            // uploads are launched ahead of the copy
    unsigned feed_give_up_ = kFeedGiveUp;
    unsigned* upload_words_ = nullptr;  // UploadRange::words of the network's stream
    HostLoan out_area(size_t floats);
    void count_area(size_t bytes, size_t& most);   // an area counts as an allocation when it is larger than any before in its place
    void check_queued();
    void upload(const float* data, int order, const TView& v, unsigned* amax);
    void download_planes(const TView& v, int include_padding, float* out);
    void download_pixels(const TView& v, int pc, float* out);
    void download_argmax(const int* idx_dev, const TView& v, int32_t* idx, float* val);
    float* static_scratch_ = nullptr;   // this device's address of the fixed staging area
    unsigned* amax_dev_ = nullptr;      // one value-range word per tensor
    void assign_range_words();
    template <class Take>
    std::vector<int> place_range_resets(Take&& take) const;   // (which launch clears which word: engine.cpp)
    void assign_range_resets();
    hipGraph_t graph_ = nullptr;
    hipGraphExec_t graph_exec_ = nullptr;
    bool graph_enabled_ = false;
    bool events_pending_ = false;
    bool poison_lds_ = false;           // FYNHIP_POISON_LDS: fill the LDS with NaN patterns in front of every layer
};

Layer* create_layer(Net* net, const fyn_layer_desc& d);
void fuse_batchnorm_layers(Net* net);   // after every layer's setup(): batch-norm layers that their readers (K-resident convolutions) can apply while staging
void keep_projection_inputs(Net* net);    // before buffers are assigned: inputs of such projections live until the layer that may compute them has run
void fuse_projection_layers(Net* net);   // after every layer's setup(): 1x1 shortcut projections that the 1x1 layer adding them can compute in its own launch
std::vector<std::pair<int, int>> keep_block_inputs(Net* net);   // ... and, while they are assigned, inputs of bottlenecks until their last layer, which may compute them, has run; (tensor, its last reader)
void fuse_block_layers(Net* net);        // after the other passes on convolutions: a 1x1, a 3x3 and a 1x1 layer in one launch
void fuse_pair_layers(Net* net);         // ... two 3x3 layers between tensors of few channels in one launch
void fuse_head_layers(Net* net);         // ... a 9x9 layer on an image and the 3x3 layer with a step of two behind it
void fuse_depthwise_layers(Net* net);   // after every layer's setup(): depthwise 3x3 layers that their 1x1 reader can compute itself
void fuse_function_layers(Net* net);   // after every layer's setup(): sigmoid / tanh layers that the row-rolling convolution in front of them can apply to what it stores
void fuse_concat_layers(Net* net);   // after every layer's setup(): bilinear scale layers in front of concatenations and batch-norm layers behind them
void fuse_argmax_layers(Net* net);   // after every layer's setup(): arg-max layers that the streaming 1x1 convolution in front of them can compute
Layer* create_custom_layer(Net* net, const fyn_layer_desc& d, const fyn_custom_layer& impl);

}  // namespace fynhip
