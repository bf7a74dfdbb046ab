// Graph-rewrite passes run once when a network is set up: layers whose work a neighbouring convolution launch can
// take over (depthwise convolutions, 1x1 projections of a residual branch, plain batch-norm layers) are folded into
// that launch, subject to the liveness of the tensors whose reads or writes move to another layer's slot.
#include <algorithm>
#include <cmath>
#include <cstring>

#include "layer_classes.h"

namespace fynhip {

// Depthwise 3x3 -> pointwise 1x1 (the second half of an inverted-residual block) as one launch.  Where the pointwise
// layer runs the K-resident form on 4x4 tiles and is the depthwise layer's only reader, its staging waves can compute
// the depthwise layer for the tile instead of fetching that layer's output (conv_kr16_kernel, DWS): every workgroup of
// a tile -- one per block of 16 or 32 output channels -- repeats the depthwise arithmetic for its tile, which costs
// less than a launch as long as the blocks are few.  Both ways are timed; the depthwise layer's tensor is not written
// when the fused way is taken, so the fusion is tied to buffer reuse (a caller who switches reuse off wants every
// layer's tensor) and is left out of passes that time or dump single layers.
void fuse_depthwise_layers(Net* net) {
    if (net->sw.get("FYNHIP_NO_DW_FUSION") || !net->reuse_buffers) return;
    std::map<int, int> readers;
    for (auto& kv : net->layers)
        for (int t : kv.second->in)
            if (t >= 0) readers[t]++;
    const char* at = net->sw.get("FYNHIP_AUTOTUNE");
    // First the other half of the block: a 1x1 layer (expand) whose only reader is the depthwise layer.  Every expanded
    // channel depends on the 1x1 layer's input only, so a workgroup can compute the window of the expanded tensor that
    // its tile of the depthwise layer needs (conv_e16dw_kernel); the expanded tensor is then never written.
    for (auto& kv : net->layers) {
        if (net->sw.get("FYNHIP_NO_EDW_FUSION")) break;
        DwConvLayer* dw = dynamic_cast<DwConvLayer*>(kv.second.get());
        if (!dw || dw->dil != 1 || (dw->stride != 1 && dw->stride != 2) || dw->p.res.ptr || dw->p.in.cp % 8 != 0 || dw->p.in.cp != dw->p.out.cp || dw->p.in.f16 != dw->p.out.f16)
            continue;
        const Tensor& t = net->tensors[dw->in[0]];
        if (t.producer < 0 || t.locked || readers[dw->in[0]] != 1) continue;
        ConvLayer* ex = dynamic_cast<ConvLayer*>(net->layer(t.producer));
        if (!ex || ex->k != 1 || ex->stride != 1 || ex->dil != 1 || ex->clamp || ex->frac_shift || ex->direct || (ex->d.flags & FYN_FLAG_RESIDUAL_INPUT)) continue;
        const TView& in_v = ex->tin(0).v;
        // (the launch writes the depthwise layer's output in the 1x1 layer's place in the order, while it reads its own input)
        if (!net->alone(dw->out, ex->d.number, dw->d.number)) continue;
        if (in_v.f16 != dw->p.out.f16 || ex->d.in_channels != in_v.cp || ex->tout().v.cp != dw->p.in.cp || ex->oc % 4 != 0 ||
            !conv_e16dw_supported(in_v.cp, (in_v.cp + 31) / 32, dw->stride))
            continue;
        ConvP16Params q{};
        q.in = in_v.ptr; q.in_hp = in_v.hp(); q.in_wp = in_v.wp(); q.in_cp = in_v.cp;
        q.stride = 1; q.in_y0 = q.in_x0 = in_v.pad;
        q.cin_chunks = (in_v.cp + 31) / 32;
        q.mfrags = (ex->oc + 15) / 16;
        q.f16 = in_v.f16 ? 1 : 0;
        q.scale = ex->scale_dev; q.bias = ex->bias_dev;
        q.acc_mul = 1.f;
        q.act = ex->act();
        q.dw_hp = ex->oh; q.dw_wp = ex->ow;
        q.out = dw->p.out.ptr; q.out_wp = dw->p.out.wp(); q.out_cp = dw->p.out.cp; q.out_off_y = q.out_off_x = dw->p.out.pad;
        q.npos_y = dw->p.out.h; q.npos_x = dw->p.out.w;
        q.tiles_x = (q.npos_x + 3) / 4; q.tiles_y = (q.npos_y + 3) / 4;
        q.dw_w = dw->w_dev; q.dw_scale = dw->scale_dev; q.dw_bias = dw->bias_dev;
        q.dw_cp = dw->p.in.cp; q.dw_stride = dw->stride; q.dw_act = dw->p.act;
        const size_t halves = (size_t)q.mfrags * q.cin_chunks * (q.f16 ? 1 : 2) * 64 * 8;
        void* const wp = net->dev_alloc(halves * 2, true);
        q.wpack = wp;
        bool pick = true;
        char key[200];
        snprintf(key, sizeof(key), "edw:%d:%dto%d:%dx%d:s%d", q.f16, in_v.cp, ex->oc, ex->oh, ex->ow, dw->stride);
        // (q.wm = 2: a workgroup per 16 expanded channels instead of 64, for layers with few tiles; by rule when nothing is timed)
        q.wm = (q.tiles_x * q.tiles_y * ((q.dw_cp + 63) / 64) < 128) ? 2 : 0;
        if (const char* e = net->sw.get("FYNHIP_EDW_NARROW")) q.wm = atoi(e) ? 2 : 0;
        int cached[3] = {0, 0, 0};
        if (net->sw.get("FYNHIP_FORCE_DW_FUSION") || net->sw.get("FYNHIP_EDW_NARROW")) {
        } else if (tune_cache_triple(net, key, cached)) {
            pick = cached[0] != 0;
            q.wm = cached[1];
        } else if (!(at && at[0] == '0')) {
            float t_fused = 1e30f, t_two = 1e30f;
            int best_wm = 0;
            for (int rep = 0; rep < 3; rep++) {
                for (int wm : {0, 2}) {
                    ConvP16Params c = q;
                    c.wm = wm;
                    const float t = time_calls(net, [&]() {
                        if (launch_conv_e16dw(c, net->stream) != 0) fail(FYN_ERR_DEVICE, "1x1 + depthwise convolution launch failed while tuning");
                    }, 10);
                    if (t < t_fused) { t_fused = t; best_wm = wm; }
                }
                t_two = std::min(t_two, time_calls(net, [&]() {
                    ex->run(net->stream);
                    launch_dwconv3x3(dw->p, net->stream);
                }, 10));
            }
            if (net->sw.get("FYNHIP_TUNE_VERBOSE"))
                fprintf(stderr, "[tune] 1x1 %d to %d at %dx%d + depthwise 3x3 (step %d): one launch (blocks of %d channels) %.1f us, two %.1f us\n", in_v.cp, ex->oc, ex->oh,
                        ex->ow, dw->stride, best_wm == 2 ? 16 : 64, t_fused * 1e3f, t_two * 1e3f);
            // (a near tie goes to the single launch: it leaves the expanded tensor unwritten, which a timing loop that
            // finds everything in the caches does not reward)
            pick = t_fused < t_two * 1.05f;
            q.wm = best_wm;
            tune_cache_store_triple(net, key, pick ? 1 : 0, best_wm, 0);
        }
        if (!pick) {
            net->dev_free(wp);
            continue;
        }
        ex->edw = q;
        ex->edw_wpack_dev = wp;
        ex->edw_fused = true;
        ex->edw_dw_no = dw->d.number;
        dw->fused_into = ex->d.number;
        net->tensors[dw->out].written = ex->d.number;
        ex->pack_edw();
    }
    for (auto& kv : net->layers) {
        ConvLayer* pw = dynamic_cast<ConvLayer*>(kv.second.get());
        if (!pw || !pw->takes_depthwise()) continue;
        const Tensor& t = net->tensors[pw->in[0]];
        if (t.producer < 0 || t.locked || readers[pw->in[0]] != 1) continue;
        DwConvLayer* dw = dynamic_cast<DwConvLayer*>(net->layer(t.producer));
        if (dw && dw->fused_into >= 0) continue;   // (already part of the 1x1 layer in front of it)
        if (!dw || dw->dil != 1 || (dw->stride != 1 && dw->stride != 2) || dw->p.res.ptr || dw->p.in.cp % 8 != 0 || dw->p.in.cp != dw->p.out.cp ||
            dw->p.in.f16 != dw->p.out.f16 || dw->p.out.f16 != pw->pp.f16 || dw->p.out.cp != pw->pp.in_cp)
            continue;
        // (the launch reads the depthwise layer's input in the 1x1 layer's place in the order, while it writes that layer's output)
        if (!net->alone(dw->in[0], dw->d.number, pw->d.number)) continue;
        ConvP16Params& f = pw->dw_fields;
        f.dw_in = dw->p.in.ptr; f.dw_w = dw->w_dev; f.dw_scale = dw->scale_dev; f.dw_bias = dw->bias_dev;
        f.dw_hp = dw->p.in.hp(); f.dw_wp = dw->p.in.wp(); f.dw_cp = dw->p.in.cp;
        f.dw_y0 = f.dw_x0 = dw->p.in.pad - 1;
        f.dw_stride = dw->stride; f.dw_act = dw->p.act;
        const ConvP16Params q = pw->with_depthwise();
        if (pw->d16 ? !conv_d16_dw_supported(q.cin_chunks, q.dw_stride) : (conv_kr16_lds_bytes(q, 1) == 0 || conv_kr16_lds_bytes(q, 1) > 160 * 1024)) continue;
        bool pick = true;
        char key[200];
        snprintf(key, sizeof(key), "dwpw:%d:%dx%dx%d:s%d:to%d:fm%d:d%d", q.f16, dw->p.in.cp, dw->p.in.h, dw->p.in.w, dw->stride, pw->oc, q.wm, pw->d16 ? 1 : 0);
        if (net->sw.get("FYNHIP_FORCE_DW_FUSION")) {
        } else if (tune_cache_flag(net, key, &pick)) {
        } else if (!(at && at[0] == '0')) {
            float t_fused = 1e30f, t_two = 1e30f;
            for (int rep = 0; rep < 3; rep++) {
                t_fused = std::min(t_fused, time_calls(net, [&]() {
                    if (pw->launch_with_depthwise(q, net->stream) != 0) fail(FYN_ERR_DEVICE, "1x1 convolution with a depthwise layer in front: launch failed while tuning");
                }, 10));
                t_two = std::min(t_two, time_calls(net, [&]() {
                    launch_dwconv3x3(dw->p, net->stream);
                    if (pw->launch_own(net->stream) != 0) fail(FYN_ERR_DEVICE, "1x1 convolution launch failed while tuning");
                }, 10));
            }
            if (net->sw.get("FYNHIP_TUNE_VERBOSE"))
                fprintf(stderr, "[tune] depthwise 3x3 (step %d) on %d channels at %dx%d + 1x1 to %d: one launch %.1f us, two %.1f us\n", dw->stride, dw->p.in.cp,
                        dw->p.in.h, dw->p.in.w, pw->oc, t_fused * 1e3f, t_two * 1e3f);
            pick = t_fused < t_two;
            tune_cache_store_flag(net, key, pick);
        }
        if (!pick) continue;
        pw->dw_fused = true;
        pw->dw_layer_no = dw->d.number;
        dw->fused_into = pw->d.number;
        net->read_until(dw->in[0], pw->d.number);
    }
}

// The projection that layer `c` could compute itself (fuse_projection_layers below), by the graph alone: `c` a 1x1 layer
// without step that adds, unactivated, the result of a 1x1 layer nothing else reads.
static ConvLayer* projection_of(Net* net, ConvLayer* c) {
    if (!c || c->k != 1 || c->stride != 1 || c->dil != 1 || c->clamp || c->frac_shift || c->direct || !(c->d.flags & FYN_FLAG_RESIDUAL_INPUT) ||
        (c->d.flags & FYN_FLAG_RELU_ON_RESIDUAL) || c->in.size() < 2 || c->in[1] < 0 || c->in[0] == c->in[1])
        return nullptr;
    const Tensor& rt = net->tensors[c->in[1]];
    if (rt.producer < 0 || rt.locked) return nullptr;
    int readers = 0;
    for (auto& kv : net->layers)
        for (int t : kv.second->in) readers += t == c->in[1];
    if (readers != 1) return nullptr;
    ConvLayer* pr = dynamic_cast<ConvLayer*>(net->layer(rt.producer));
    if (!pr || pr->k != 1 || pr->dil != 1 || pr->clamp || pr->frac_shift || pr->direct || (pr->d.flags & FYN_FLAG_RESIDUAL_INPUT) || pr->oc != c->oc ||
        pr->d.number >= c->d.number || pr->in.empty() || pr->in[0] < 0)
        return nullptr;
    return pr;
}
// Before buffers are assigned: the input of such a projection stays whole until the layer that may compute it has run
// (a few more buffers in networks with such pairs, whether the pair is joined in the end or not).
void keep_projection_inputs(Net* net) {
    if (net->sw.get("FYNHIP_NO_PROJECTION_FUSION") || !net->reuse_buffers) return;
    for (auto& kv : net->layers) {
        ConvLayer* c = dynamic_cast<ConvLayer*>(kv.second.get());
        ConvLayer* pr = projection_of(net, c);
        if (!pr) continue;
        net->read_until(pr->in[0], c->d.number);
    }
}
// A 1x1 projection (a residual block's shortcut convolution) whose only reader adds it to its own 1x1 convolution: both
// are sums over channels at the same output position, so they run as ONE reduction over two tensors on the K-resident
// form -- the projection's chunks behind the layer's own, each weight row carrying its layer's folded scale -- and the
// projection's tensor is never written.  Conditions: both 1x1 without dilation on tensors of one storage type, the same
// activation on fetch, no activation on the residual, the projection's input still whole when the reader runs, and a
// compiled variant for the joint chunk count; timed against the two launches.
void fuse_projection_layers(Net* net) {
    if (net->sw.get("FYNHIP_NO_PROJECTION_FUSION") || net->sw.get("FYNHIP_NO_P16_CONV") || net->sw.get("FYNHIP_NO_KR16_CONV") || !net->reuse_buffers) return;
    const char* at = net->sw.get("FYNHIP_AUTOTUNE");
    for (auto& kv : net->layers) {
        ConvLayer* c = dynamic_cast<ConvLayer*>(kv.second.get());
        ConvLayer* pr = projection_of(net, c);
        if (!pr || c->dw_fused || c->edw_fused || c->bn_fused || pr->dw_fused || pr->edw_fused || pr->bn_fused || pr->pj_fused || pr->pj_into >= 0) continue;
        const Tensor& rt = net->tensors[c->in[1]];
        const Act a1 = c->act(), a2 = pr->act();
        if (a1.kind != a2.kind || a1.lo != a2.lo || a1.hi != a2.hi || a1.leak != a2.leak) continue;
        const TView& v1 = c->tin(0).v;
        const TView& v2 = pr->tin(0).v;
        const TView& ov = c->tout().v;
        if (v1.f16 != ov.f16 || v2.f16 != ov.f16 || rt.v.f16 != ov.f16 || c->d.in_channels != v1.cp || pr->d.in_channels != v2.cp || v1.cp % 8 != 0 || v2.cp % 8 != 0 ||
            v1.cp < 8 || v2.cp < 8 || c->oc % 4 != 0 || c->oc < 8 || ov.cp < c->oc || c->oh * c->ow > 4096)
            continue;
        if (!net->alone(pr->in[0], pr->d.number, c->d.number)) continue;   // (the projection's input must still hold its values when the reader runs)
        const int n1 = (v1.cp + 31) / 32, n2 = (v2.cp + 31) / 32;
        ConvP16Params q{};
        q.in = v1.ptr; q.out = ov.ptr;
        q.in_hp = v1.hp(); q.in_wp = v1.wp(); q.in_cp = v1.cp;
        q.stride = 1; q.in_y0 = q.in_x0 = v1.pad;
        q.in2 = v2.ptr; q.in2_hp = v2.hp(); q.in2_wp = v2.wp(); q.in2_cp = v2.cp;
        q.in2_stride = pr->stride; q.in2_y0 = q.in2_x0 = v2.pad; q.in2_chunk0 = n1;
        q.npos_y = c->oh; q.npos_x = c->ow;
        q.out_wp = ov.wp(); q.out_cp = ov.cp; q.out_off_y = q.out_off_x = ov.pad;
        q.f16 = ov.f16 ? 1 : 0;
        q.acc_mul = 1.f;
        q.act = a1;
        q.tile_h = q.tile_w = 4;
        q.tiles_x = (c->ow + 3) / 4; q.tiles_y = (c->oh + 3) / 4;
        q.rcp_tiles_x = 1.0f / (float)q.tiles_x;
        q.pos_groups = q.tiles_x * q.tiles_y;
        // (the last pixel either tensor is read at lies inside it)
        if ((c->oh - 1) * pr->stride + v2.pad >= v2.hp() || (c->ow - 1) * pr->stride + v2.pad >= v2.wp()) continue;
        // the joint chunk count, rounded up to the next one a variant is compiled for (the chunks behind both tensors read as zero)
        int chunks = 0;
        for (int n = (n1 + n2 + 3) / 4 * 4; n <= 64 && !chunks; n += 4) {
            ConvP16Params t = q;
            t.cin_chunks = n; t.wm = 1; t.cout_blocks = (c->oc + 15) / 16; t.mfrags = t.cout_blocks;
            if (conv_kr16_lds_bytes(t, 1) != 0) chunks = n;
        }
        if (!chunks) continue;
        q.cin_chunks = chunks;
        std::vector<ConvP16Params> cands;
        for (int fm : {1, 2}) {
            if (fm == 2 && c->oc % 32 != 0 && c->oc % 32 <= 16) continue;
            ConvP16Params t = q;
            t.wm = fm;
            t.cout_blocks = (c->oc + 16 * fm - 1) / (16 * fm);
            t.mfrags = t.cout_blocks * fm;
            const size_t lds = conv_kr16_lds_bytes(t, 1);
            if (lds == 0 || lds > 160 * 1024 || (long long)t.pos_groups * t.cout_blocks > 65535) continue;
            cands.push_back(t);
        }
        if (cands.empty()) continue;
        const size_t halves = (size_t)((c->oc + 31) / 32 * 2) * 4 * (chunks / 4) * (q.f16 ? 1 : 2) * 64 * 8;
        void* const wp = net->dev_alloc(halves * 2, true);
        float* const sc = static_cast<float*>(net->dev_alloc(c->padded * sizeof(float), true));
        float* const bi = static_cast<float*>(net->dev_alloc(c->padded * sizeof(float), true));
        for (ConvP16Params& t : cands) { t.wpack = wp; t.scale = sc; t.bias = bi; }
        int pick = 0;
        bool win = true;
        char key[200];
        snprintf(key, sizeof(key), "pj:%d:%dand%dto%d:%dx%d:s%d", q.f16, v1.cp, v2.cp, c->oc, c->oh, c->ow, pr->stride);
        int cached[3] = {0, 0, 0};
        if (net->sw.get("FYNHIP_FORCE_PROJECTION_FUSION")) {
        } else if (tune_cache_triple(net, key, cached)) {
            win = cached[0] != 0;
            for (size_t i = 0; i < cands.size(); i++)
                if (cands[i].wm == cached[1]) pick = (int)i;
        } else if (!(at && at[0] == '0')) {
            float t_fused = 1e30f, t_two = 1e30f;
            for (int rep = 0; rep < 3; rep++) {
                for (size_t i = 0; i < cands.size(); i++) {
                    const float t = time_calls(net, [&]() {
                        if (launch_conv_kr16(cands[i], 1, net->stream) != 0) fail(FYN_ERR_DEVICE, "1x1 convolution over two tensors: launch failed while tuning");
                    }, 10);
                    if (t < t_fused) { t_fused = t; pick = (int)i; }
                }
                t_two = std::min(t_two, time_calls(net, [&]() {
                    pr->run(net->stream);
                    c->run(net->stream);
                }, 10));
            }
            if (net->sw.get("FYNHIP_TUNE_VERBOSE"))
                fprintf(stderr, "[tune] 1x1 on %d channels + 1x1 projection on %d (step %d) to %d at %dx%d: one launch %.1f us, two %.1f us\n", v1.cp, v2.cp, pr->stride, c->oc,
                        c->oh, c->ow, t_fused * 1e3f, t_two * 1e3f);
            win = t_fused < t_two;
            tune_cache_store_triple(net, key, win ? 1 : 0, cands[pick].wm, 0);
        }
        if (!win) {
            net->dev_free(wp); net->dev_free(sc); net->dev_free(bi);
            continue;
        }
        c->pj = cands[pick];
        c->pj_wpack_dev = wp; c->pj_scale_dev = sc; c->pj_bias_dev = bi;
        c->pj_fused = true;
        c->pj_layer_no = pr->d.number;
        pr->pj_into = c->d.number;
        net->read_until(pr->in[0], c->d.number);   // (its value-range word is cleared behind its last reader)
        c->pack_two_sources();
    }
}

// Batch-norm layers whose readers can apply them: a plain x * scale + bias (no activation, no residual input) between
// tensors of one geometry without a halo, read only by convolution layers on the K-resident or the LDS-free 1x1 form, as
// their data input.  Each reader then fetches from the batch-norm layer's input and applies scale and bias per channel
// before its own activation; the layer's output is never written and its launch is gone (the reference's ResNet-50 sample graph has one such layer in
// front of most blocks).  The input tensor must still hold its values when the last reader runs: no tensor produced
// between the batch-norm layer and that reader may live in the same buffer.
void fuse_batchnorm_layers(Net* net) {
    if (net->sw.get("FYNHIP_NO_BN_FUSION") || !net->reuse_buffers) return;
    for (auto& kv : net->layers) {
        BatchNormLayer* bn = dynamic_cast<BatchNormLayer*>(kv.second.get());
        if (!bn || bn->p.res.ptr || bn->p.act.kind != ACT_NONE) continue;
        const Tensor& x = net->tensors[bn->in[0]];
        const Tensor& y = net->tensors[bn->out];
        // (no halo: around the layer's output it holds zeros, which scale and bias applied to the input's halo would not give)
        if (y.locked || x.v.pad != 0 || y.v.pad != 0 || x.v.h != y.v.h || x.v.w != y.v.w || x.v.cp != y.v.cp || x.v.f16 != y.v.f16 || x.v.c != y.v.c) continue;
        std::vector<ConvLayer*> readers;
        bool all = true;
        int last = -1;
        for (auto& kr : net->layers) {
            Layer* l = kr.second.get();
            for (size_t port = 0; port < l->in.size(); port++) {
                if (l->in[port] != bn->out) continue;
                ConvLayer* c = dynamic_cast<ConvLayer*>(l);
                if (!c || port != 0 || !c->takes_batchnorm() || c->d.number <= bn->d.number) { all = false; continue; }
                readers.push_back(c);
                last = std::max(last, c->d.number);
            }
        }
        if (!all || readers.empty()) continue;
        if (!net->alone(bn->in[0], bn->d.number, last)) continue;
        for (ConvLayer* c : readers) {
            c->bn_fused = true;
            c->bn_layer_no = bn->d.number;
            c->bn_in = x.v.ptr; c->bn_mul = bn->scale_dev; c->bn_add = bn->bias_dev;
        }
        bn->fused_into = readers.front()->d.number;
        net->read_until(bn->in[0], last);   // (its value-range word is cleared behind its last reader)
    }
}

// The convolution in front of layer `l` that nothing else reads and that adds nothing itself.
static ConvLayer* alone_in_front(Net* net, const ConvLayer* l) {
    if (l->in.empty() || l->in[0] < 0) return nullptr;
    const Tensor& t = net->tensors[l->in[0]];
    if (t.producer < 0 || t.locked) return nullptr;
    int readers = 0;
    for (auto& kv : net->layers)
        for (int i : kv.second->in) readers += i == l->in[0];
    ConvLayer* p = readers == 1 ? dynamic_cast<ConvLayer*>(net->layer(t.producer)) : nullptr;
    return p && !(p->d.flags & FYN_FLAG_RESIDUAL_INPUT) && p->d.number < l->d.number && !p->in.empty() && p->in[0] >= 0 ? p : nullptr;
}
static bool plain_conv(const ConvLayer* l, int k) { return l && l->k == k && l->stride == 1 && l->dil == 1 && !l->frac_shift && !l->direct && !l->wide; }
// The bottleneck that ends with layer `c`, by the graph alone: a 1x1 layer, a 3x3 layer that alone reads it, and `c`, a 1x1
// layer that alone reads that one; no step, no dilation, nothing between them.
static bool block_of(Net* net, const ConvLayer* c, ConvLayer*& a, ConvLayer*& b) {
    if (!plain_conv(c, 1)) return false;
    b = alone_in_front(net, c);
    if (!plain_conv(b, 3) || b->clamp) return false;
    a = alone_in_front(net, b);
    return plain_conv(a, 1) && a->oh == c->oh && a->ow == c->ow && b->oh == c->oh && b->ow == c->ow;
}
// The 3x3 layer `a` that the 3x3 layer `c` alone reads, both with the same rule at the frame's edge.
static bool pair_of(Net* net, const ConvLayer* c, ConvLayer*& a) {
    if (!plain_conv(c, 3)) return false;
    a = alone_in_front(net, c);
    return plain_conv(a, 3) && a->clamp == c->clamp && a->oh == c->oh && a->ow == c->ow;
}
// The 9x9 layer `a` on an image that `c`, a 3x3 layer with a step of two, alone reads.
static bool head_of(Net* net, const ConvLayer* c, ConvLayer*& a) {
    if (!c || c->k != 3 || c->stride != 2 || c->dil != 1 || c->frac_shift || c->direct || c->wide || (c->d.flags & FYN_FLAG_RESIDUAL_INPUT)) return false;
    a = alone_in_front(net, c);
    if (!plain_conv(a, 9) || a->clamp != c->clamp || a->oc > 32 || c->oc > 64 || a->d.in_channels > 4) return false;
    const int from = net->tensors[a->in[0]].producer;   // (a frame from the host or the application: its value-range word is never lost)
    return from < 0 || net->layer(from)->d.type == FYN_LAYER_UPLOAD;
}
// What says which compiled variant computes a bottleneck: the next chunk count that there is one for (the channels behind the
// tensor read as zero).  False: none does.
static bool block_variant(const ConvLayer* a, const ConvLayer* b, const ConvLayer* c, bool bn, bool proj, ConvB16Params& q) {
    static const float some = 0.f;   // (whether the batch-norm layer is there is all that counts)
    const TView &iv = a->tin(0).v, &ov = c->tout().v;
    q.in_mul = q.in_add = bn ? &some : nullptr;
    q.proj = proj ? 1 : 0;
    q.f16 = ov.f16 ? 1 : 0;
    q.in_cp = iv.cp; q.out_cp = ov.cp;
    q.mid = std::max(a->oc, b->oc) <= 64 ? 4 : (std::max(a->oc, b->oc) + 15) / 16;
    if (q.mid > 4 && q.mid < 8) q.mid = 8;   // (channels behind a layer's count have zero weights, scales and biases)
    q.tiles_x = (c->ow + 3) / 4; q.tiles_y = (c->oh + 3) / 4;
    for (q.chunks = (iv.cp + 31) / 32; q.chunks <= 16 && conv_b16_weight_frags(q) == 0; q.chunks++) {}
    // (32-bit offsets)
    return conv_b16_weight_frags(q) != 0 && (long long)q.tiles_x * q.tiles_y <= 4096 && (long long)iv.hp() * iv.wp() * iv.cp <= (1ll << 30);
}
// ... and a pair: the compiled tile heights (indices of conv_c16_variant).
static std::vector<int> pair_variants(const ConvLayer* a, const ConvLayer* c) {
    std::vector<int> out;
    const TView &iv = a->tin(0).v, &mv = a->tout().v, &ov = c->tout().v;
    for (int i = 0; i < conv_c16_count(); i++) {
        int f16, groups, fr, th;
        conv_c16_variant(i, &f16, &groups, &fr, &th);
        if (f16 == (ov.f16 ? 1 : 0) && iv.cp == 8 * groups && mv.cp == iv.cp && ov.cp <= 16 * fr && (long long)((c->ow + 15) / 16) * ((c->oh + th - 1) / th) <= (1 << 20)) out.push_back(i);
    }
    return out;
}
// While buffers are assigned, the input of a block or pair that a variant is compiled for is read until its last layer has run,
// which may compute all of it (the tensors' last readers as they were: whether the layers are joined is not known yet).  A
// head's input is the frame, whose buffer nobody shares.
std::vector<std::pair<int, int>> keep_block_inputs(Net* net) {
    std::vector<std::pair<int, int>> were;
    if (!net->reuse_buffers || net->sw.get("FYNHIP_NO_P16_CONV")) return were;
    auto keep = [&](int tensor, int layer_no) {
        were.push_back({tensor, net->tensors[tensor].last_reader});
        net->read_until(tensor, layer_no);
    };
    for (auto& kv : net->layers) {
        ConvLayer *c = dynamic_cast<ConvLayer*>(kv.second.get()), *a = nullptr, *b = nullptr;
        if (!c) continue;
        if (!net->sw.get("FYNHIP_NO_PAIR_FUSION") && pair_of(net, c, a) && !pair_variants(a, c).empty()) keep(a->in[0], c->d.number);
        if (net->sw.get("FYNHIP_NO_BLOCK_FUSION") || !block_of(net, c, a, b)) continue;
        const int x = a->in[0], from = net->tensors[x].producer;
        const BatchNormLayer* bn = from < 0 ? nullptr : dynamic_cast<BatchNormLayer*>(net->layer(from));   // (which the block may apply)
        ConvB16Params q{};
        if (block_variant(a, b, c, false, false, q) || (projection_of(net, c) && block_variant(a, b, c, false, true, q))) keep(x, c->d.number);
        if (bn && !bn->in.empty() && bn->in[0] >= 0 && block_variant(a, b, c, true, false, q)) keep(bn->in[0], c->d.number);
    }
    return were;
}
// (tests: whoever forces a form of a layer wants to see that form)
static bool single_form_forced(const Net* net) {
    for (const char* form : {"FYNHIP_FORCE_PROJECTION_FUSION", "FYNHIP_FORCE_KR16_CONV", "FYNHIP_KR16_FM", "FYNHIP_FORCE_D16_CONV", "FYNHIP_D16_BLOCKS", "FYNHIP_FORCE_P16_CONV", "FYNHIP_P16_TILE",
                             "FYNHIP_FORCE_G16_CONV", "FYNHIP_G16_FRAGS", "FYNHIP_FORCE_P16N_CONV", "FYNHIP_P16N_ROWS", "FYNHIP_FORCE_KSPLIT", "FYNHIP_CONV_TILE", "FYNHIP_CONV_KC",
                             "FYNHIP_CONV_KC_MAX", "FYNHIP_CONV_PD"})
        if (net->sw.get(form)) return true;
    return false;
}
// Whether the layers `front` can go into the launch of layer `last`, which then reads tensor x: the words of value ranges
// that their launches clear need another launch to do so.
static bool words_survive(Net* net, const std::vector<ConvLayer*>& front, int last, int x) {
    const int reader = net->tensors[x].last_reader, lost = net->words_without_reset();
    for (ConvLayer* l : front) l->blk_into = last;
    net->read_until(x, last);
    const int then = net->words_without_reset();
    for (ConvLayer* l : front) l->blk_into = -1;
    net->tensors[x].last_reader = reader;
    return then <= lost;
}
// Bottlenecks (conv_b16.hip) as one launch in the place of their last layer, timed against the launches they run as now:
// with the batch-norm layer in front that the first layer applies, or the projection that the last one adds.
void fuse_block_layers(Net* net) {
    if (net->sw.get("FYNHIP_NO_BLOCK_FUSION") || net->sw.get("FYNHIP_NO_P16_CONV") || !net->reuse_buffers) return;
    if (!net->sw.get("FYNHIP_FORCE_BLOCK_FUSION") && single_form_forced(net)) return;
    const char* at = net->sw.get("FYNHIP_AUTOTUNE");
    for (auto& kv : net->layers) {
        ConvLayer *c = dynamic_cast<ConvLayer*>(kv.second.get()), *a = nullptr, *b = nullptr;
        if (!c || !block_of(net, c, a, b)) continue;
        if (a->blk_fused) continue;   // (the last layer of a block in front: its launch writes what this one's first layer would have to compute)
        if (a->dw_fused || a->edw_fused || a->pj_fused || a->pj_into >= 0 || b->bn_fused || c->bn_fused || c->dw_fused || c->edw_fused || c->fn_layer_no >= 0 || c->argmax_tail.idx) continue;
        const TView &iv = a->tin(0).v, &ov = c->tout().v;
        if (iv.f16 != ov.f16 || a->tout().v.f16 != ov.f16 || b->tout().v.f16 != ov.f16 || iv.cp % 8 != 0 || iv.cp < 8 || ov.cp % 4 != 0 || a->d.in_channels > iv.cp || c->oc > ov.cp ||
            b->d.in_channels != a->oc || c->d.in_channels != b->oc)
            continue;
        // (positions beside the first layer's output are zeros behind the second layer's activation as well)
        if (b->act().lo > 0.f || b->act().hi < 0.f) continue;
        ConvLayer* pr = nullptr;
        ConvB16Params q{};
        if (c->d.flags & FYN_FLAG_RESIDUAL_INPUT) {
            if (c->in.size() < 2 || c->in[1] < 0 || c->in[1] == c->in[0]) continue;
            const TView& rv = c->tin(1).v;
            if (rv.f16 != ov.f16) continue;
            pr = projection_of(net, c);
            const Act x = a->act(), y = pr ? pr->act() : x;
            if (pr && (pr->stride != 1 || pr->in[0] != a->in[0] || a->bn_fused || pr->bn_fused || x.kind != y.kind || x.lo != y.lo || x.hi != y.hi || x.leak != y.leak || pr->d.in_channels > iv.cp ||
                       net->tensors[c->in[1]].v.f16 != ov.f16 || net->sw.get("FYNHIP_NO_PROJECTION_FUSION")))
                pr = nullptr;
            if (!pr) {
                if (c->pj_fused || rv.cp < ov.cp || rv.cp % 4 != 0) continue;
                q.res = rv.ptr; q.res_wp = rv.wp(); q.res_cp = rv.cp; q.res_off = rv.pad;
                q.res_relu = (c->d.flags & FYN_FLAG_RELU_ON_RESIDUAL) ? 1 : 0;
            }
            q.res_scale = ((c->d.flags & FYN_FLAG_BATCHNORM_ON_RESIDUAL) && (c->d.flags & FYN_FLAG_POST_BATCHNORM)) ? 1 : 0;
        }
        // (the launch reads the block's input in the last layer's place in the order)
        int x = a->in[0];
        if (a->bn_fused) x = net->layer(a->bn_layer_no)->in[0];
        if (!net->alone(x, a->d.number, c->d.number)) continue;
        std::vector<ConvLayer*> front = {a, b};
        if (pr) front.push_back(pr);
        if (!words_survive(net, front, c->d.number, x)) continue;
        const ConvLayer* L[4] = {a, b, c, pr};
        for (int i = 0; i < 4; i++) {
            if (!L[i]) continue;
            q.scale[i] = L[i]->scale_dev; q.bias[i] = L[i]->bias_dev;
            q.acc_mul[i] = 1.f;
        }
        if (!block_variant(a, b, c, a->bn_fused, pr != nullptr, q)) continue;
        q.in = a->bn_fused ? a->bn_in : iv.ptr;
        q.in_mul = a->bn_fused ? a->bn_mul : nullptr; q.in_add = a->bn_fused ? a->bn_add : nullptr;
        q.out = ov.ptr;
        q.act[0] = a->act(); q.act[1] = b->act(); q.act[2] = c->act();
        q.in_hp = iv.hp(); q.in_wp = iv.wp(); q.in_off = iv.pad;
        q.h = c->oh; q.w = c->ow;
        q.out_wp = ov.wp(); q.out_off = ov.pad;
        q.rcp_tiles_x = 1.0f / (float)q.tiles_x;
        const size_t halves = conv_b16_weight_frags(q) * (q.f16 ? 1 : 2) * 64 * 8;
        void* const wp = net->dev_alloc(halves * 2, true);
        q.wpack = wp;
        // (untimed, us, one launch / apart.  In one round of workgroups it is ahead whatever the channels: fp32 56x56 256 to 64 to 64 to
        // 256 9.8 / 15.9, 64 to 32 to 32 to 64 9.1 / 13.2, 16 to 8 9.1 / 13.3, 7x7 9.0 / 10.7, 8.6 / 10.5, 8.7 / 13.3.  A second one costs
        // a launch of narrow fp32 layers more than the three: 72x72 64 to 32 16.5 / 13.8, 128 to 32 16.8 / 14.9, but 128 to 64 16.8 / 18.1,
        // 256 to 64 17.9 / 21.7; fp16 64 to 32 8.4 / 10.1.  256 to 64 at 96x96 25.0 / 24.7)
        const int tiles = q.tiles_x * q.tiles_y;
        bool pick = q.mid == 4 && (tiles <= 256 || (tiles <= 400 && (q.f16 || std::max(a->oc, b->oc) > 32)));
        char key[200];
        snprintf(key, sizeof(key), "blk:%d:%dto%dto%dto%d:%dx%d:r%d:b%d", q.f16, iv.cp, a->oc, b->oc, c->oc, c->oh, c->ow, pr ? 2 : q.res ? 1 : 0, a->bn_fused ? 1 : 0);
        if (net->sw.get("FYNHIP_FORCE_BLOCK_FUSION")) pick = true;
        else if (tune_cache_flag(net, key, &pick)) {
        } else if (!(at && at[0] == '0')) {
            float t_one = 1e30f, t_apart = 1e30f;
            for (int rep = 0; rep < 3; rep++) {
                t_one = std::min(t_one, time_calls(net, [&]() {
                    if (launch_conv_b16(q, net->stream) != 0) fail(FYN_ERR_DEVICE, "bottleneck launch failed while tuning");
                }, 10));
                t_apart = std::min(t_apart, time_calls(net, [&]() {
                    a->forward_alone(net->stream);
                    b->forward_alone(net->stream);
                    if (pr) pr->forward_alone(net->stream);
                    c->forward_alone(net->stream);
                }, 10));
            }
            if (net->sw.get("FYNHIP_TUNE_VERBOSE"))
                fprintf(stderr, "[tune] bottleneck %d to %d to %d to %d at %dx%d%s: one launch %.1f us, apart %.1f us\n", iv.cp, a->oc, b->oc, c->oc, c->oh, c->ow, pr ? " with its projection" : "", t_one * 1e3f,
                        t_apart * 1e3f);
            // (a near tie goes to the single launch.  512 to 128 to 128 to 512 on fp16 tensors, one launch / apart: 10.9 / 10.4 us at 24x24,
            // 10.9 / 10.5 at 28x28, 11.0 / 10.7 at 32x32.  A ResNet-50's frame with its three such blocks joined / apart, images of
            // 192, 224 and 256: four instances side by side 88 / 91, 99 / 102, 109 / 113 us, passes queued launch by launch 231 / 238, 237 / 243,
            // 236 / 249, a host frame by itself 272 / 277, 278 / 281, 285 / 289; on the other side a captured graph 215 / 212, 220 / 217,
            // 222 / 218, two instances 131 / 129, 138 / 136, 146 / 143, one stream of frames 223 / 221, 230 / 228, 238 / 236)
            pick = t_one < t_apart * 1.05f;
            tune_cache_store_flag(net, key, pick);
        }
        if (!pick) {
            net->dev_free(wp);
            continue;
        }
        c->blk = q;
        c->blk_wpack_dev = wp;
        c->blk_fused = true;
        c->blk_layers[0] = a->d.number; c->blk_layers[1] = b->d.number; c->blk_layers[2] = pr ? pr->d.number : -1;
        for (ConvLayer* l : front) l->blk_into = c->d.number;
        net->read_until(x, c->d.number);   // (its value-range word is cleared behind its last reader)
        c->pack_block();
    }
}

// The first two layers of a style-transfer net (conv_a16.hip) as one launch in the place of the second, timed against their own
// launches (us, 3 to 32 to 64 channels, one launch / apart): fp32 tensors 384x384 19 / 25, 512x624 26 / 39, 1920x1080 123 / 209;
// fp16 256x256 7.7 / 9.7, 512x624 14 / 29, 1920x1080 60 / 88; 3 to 12 to 20 channels, fp32, 256x256 9.8 / 12, 512x624 19 / 36,
// 1024x1024 43 / 67.  Where the tensor in between is written as well, 512x624 32 / 39, 1920x1080 145 / 211, fp16 71 / 90.  Untimed it
// is taken wherever the first layer is in its form on rows of sixteen positions: ahead at all of these.
void fuse_head_layers(Net* net) {
    if (net->sw.get("FYNHIP_NO_HEAD_FUSION") || net->sw.get("FYNHIP_NO_P16_CONV")) return;
    const bool forced = net->sw.get("FYNHIP_FORCE_HEAD_FUSION") != nullptr;
    if (!forced && single_form_forced(net)) return;
    const char* at = net->sw.get("FYNHIP_AUTOTUNE");
    for (auto& kv : net->layers) {
        ConvLayer *c = dynamic_cast<ConvLayer*>(kv.second.get()), *a = nullptr;
        if (!head_of(net, c, a) || a->blk_into >= 0 || c->blk_into >= 0 || c->fn_layer_no >= 0) continue;
        const TView &iv = a->tin(0).v, &mv = a->tout().v, &ov = c->tout().v;
        if (iv.f16 != ov.f16 || mv.f16 != ov.f16 || iv.cp != 4 || mv.cp > 32 || mv.cp % (mv.f16 ? 8 : 4) != 0 || ov.cp > 64 || ov.cp % 8 != 0 || a->d.in_channels > iv.cp || c->d.in_channels != a->oc || a->oh < 2 || a->ow < 2 || c->oh != a->oh / 2 ||
            c->ow != a->ow / 2)
            continue;
        // (the form whose weights and schedule the launch takes for the first layer; with fp32 tensors its fp8 correction terms too)
        if (!a->p16 || !a->c4 || a->pp.tile_w != 16 || (!iv.f16 && (!a->tin(0).amax || !conv_p16c4_uses_fp8(a->pp, 9)))) continue;
        if (c->clamp && (iv.pad || mv.pad)) continue;
        if ((long long)iv.hp() * iv.wp() * iv.cp > (1ll << 30)) continue;   // (32-bit offsets)
        // (positions beside a layer's input are zeros behind its activation as well)
        if (a->act().lo > 0.f || a->act().hi < 0.f || c->act().lo > 0.f || c->act().hi < 0.f) continue;
        const int x = a->in[0];
        if (!net->alone(x, a->d.number, c->d.number) || !words_survive(net, {a}, c->d.number, x)) continue;
        ConvA16Params q{};
        q.in = iv.ptr; q.in_hp = iv.hp(); q.in_wp = iv.wp(); q.in_off = iv.pad;
        q.in_amax = a->tin(0).amax;
        q.wpack[0] = a->p16_wpack_dev; q.mfrags0 = a->pp.mfrags;
        q.h = a->oh; q.w = a->ow; q.h2 = c->oh; q.w2 = c->ow;
        int rows, cols;
        conv_a16_tile(&rows, &cols);
        q.tiles_x = (q.w2 + cols - 1) / cols; q.tiles_y = (q.h2 + rows - 1) / rows;
        if (!net->reuse_buffers) {   // (every tensor stays readable: the launch writes the one in between as well)
            q.mid = mv.ptr; q.mid_wp = mv.wp(); q.mid_off = mv.pad;
            q.tiles_x = (q.w + 2 * cols - 1) / (2 * cols); q.tiles_y = (q.h + 2 * rows - 1) / (2 * rows);
        }
        q.rcp_tiles_x = 1.0f / (float)q.tiles_x;
        q.groups = std::min(q.tiles_x * q.tiles_y, 256);   // (one workgroup per CU)
        const ConvLayer* L[2] = {a, c};
        for (int i = 0; i < 2; i++) {
            q.scale[i] = L[i]->scale_dev; q.bias[i] = L[i]->bias_dev;
            q.acc_mul[i] = 1.f;
            q.act[i] = L[i]->act();
        }
        q.mid_cp = mv.cp;
        q.clamp = c->clamp ? 1 : 0;
        q.small = mv.cp <= 16 && ov.cp <= 32 ? 1 : 0;
        q.out = ov.ptr; q.out_cp = ov.cp; q.out_wp = ov.wp(); q.out_off = ov.pad;
        q.plain_stores = net->sw.get("FYNHIP_PLAIN_STORES") ? 1 : 0;
        q.f16 = ov.f16 ? 1 : 0;
        void* const wp = net->dev_alloc((size_t)(q.small ? (q.f16 ? 10 + 12 : 20) : 36 * (q.f16 ? 1 : 2)) * 1024, true);
        q.wpack[1] = wp;
        if (q.small && q.f16) {
            q.wpack[0] = static_cast<const unsigned char*>(wp) + 10 * 1024;
            q.mfrags0 = 1;
        }
        bool pick = true;
        char key[200];
        snprintf(key, sizeof(key), "head:%d:%dto%dto%d:%dx%d:e%d:k%d", q.f16, a->d.in_channels, a->oc, c->oc, a->oh, a->ow, q.clamp, q.mid ? 1 : 0);
        if (forced || tune_cache_flag(net, key, &pick)) {
        } else if (!(at && at[0] == '0')) {
            float t_one = 1e30f, t_apart = 1e30f;
            for (int rep = 0; rep < 3; rep++) {
                t_one = std::min(t_one, time_calls(net, [&]() {
                    if (launch_conv_a16(q, net->stream) != 0) fail(FYN_ERR_DEVICE, "launch of a 9x9 and a 3x3 layer failed while tuning");
                }, 10));
                t_apart = std::min(t_apart, time_calls(net, [&]() {
                    a->forward_alone(net->stream);
                    c->forward_alone(net->stream);
                }, 10));
            }
            if (net->sw.get("FYNHIP_TUNE_VERBOSE"))
                fprintf(stderr, "[tune] 9x9 %d to %d and 3x3 to %d with a step of two at %dx%d%s: one launch %.1f us, apart %.1f us\n", a->d.in_channels, a->oc, c->oc, a->oh, a->ow,
                        q.mid ? ", the tensor in between written" : "", t_one * 1e3f, t_apart * 1e3f);
            pick = t_one < t_apart;
            tune_cache_store_flag(net, key, pick);
        }
        if (!pick) {
            net->dev_free(wp);
            continue;
        }
        c->head = q;
        c->head_wpack_dev = wp;
        c->head_fused = true;
        c->head_layer = a->d.number;
        a->blk_into = c->d.number;
        net->read_until(x, c->d.number);
        c->pack_head();
    }
}

// Pairs of 3x3 layers between tensors of few channels (conv_c16.hip) as one launch in the place of the second.
void fuse_pair_layers(Net* net) {
    if (net->sw.get("FYNHIP_NO_PAIR_FUSION") || net->sw.get("FYNHIP_NO_P16_CONV") || !net->reuse_buffers) return;
    const bool forced = net->sw.get("FYNHIP_FORCE_PAIR_FUSION") != nullptr;
    if (!forced && single_form_forced(net)) return;
    const char* at = net->sw.get("FYNHIP_AUTOTUNE");
    const int want_th = net->sw.get("FYNHIP_PAIR_ROWS") ? atoi(net->sw.get("FYNHIP_PAIR_ROWS")) : 0;   // (tests: that tile height)
    for (auto& kv : net->layers) {
        ConvLayer *c = dynamic_cast<ConvLayer*>(kv.second.get()), *a = nullptr;
        if (!c || !pair_of(net, c, a) || a->blk_into >= 0 || c->blk_into >= 0 || a->pair_fused || a->fn_layer_no >= 0 || c->fn_layer_no >= 0) continue;
        const TView &iv = a->tin(0).v, &mv = a->tout().v, &ov = c->tout().v;
        if (iv.f16 != ov.f16 || mv.f16 != ov.f16 || iv.cp % 8 != 0 || mv.cp != iv.cp || ov.cp % 4 != 0 || a->d.in_channels > iv.cp || c->oc > ov.cp || c->d.in_channels != a->oc) continue;
        // (positions beside a layer's input are zeros behind its activation as well, or repeat the edge)
        if (!c->clamp && (a->act().lo > 0.f || a->act().hi < 0.f || c->act().lo > 0.f || c->act().hi < 0.f)) continue;
        if (c->clamp && (iv.pad != 0 || mv.pad != 0)) continue;
        if ((long long)iv.hp() * iv.wp() * iv.cp > (1ll << 30)) continue;   // (32-bit offsets)
        ConvC16Params q{};
        if (c->d.flags & FYN_FLAG_RESIDUAL_INPUT) {
            if (c->in.size() < 2 || c->in[1] < 0 || c->in[1] == c->in[0]) continue;
            const TView& rv = c->tin(1).v;
            if (rv.f16 != ov.f16 || rv.cp < ov.cp || rv.cp % 4 != 0) continue;
            q.res = rv.ptr; q.res_wp = rv.wp(); q.res_cp = rv.cp; q.res_off = rv.pad;
            q.res_relu = (c->d.flags & FYN_FLAG_RELU_ON_RESIDUAL) ? 1 : 0;
            q.res_scale = ((c->d.flags & FYN_FLAG_BATCHNORM_ON_RESIDUAL) && (c->d.flags & FYN_FLAG_POST_BATCHNORM)) ? 1 : 0;
        }
        // (the launch reads the pair's input in the second layer's place in the order)
        const int x = a->in[0];
        if (!net->alone(x, a->d.number, c->d.number) || !words_survive(net, {a}, c->d.number, x)) continue;
        const ConvLayer* L[2] = {a, c};
        for (int i = 0; i < 2; i++) {
            q.scale[i] = L[i]->scale_dev; q.bias[i] = L[i]->bias_dev;
            q.acc_mul[i] = 1.f;
            q.act[i] = L[i]->act();
        }
        q.in = iv.ptr; q.in_hp = iv.hp(); q.in_wp = iv.wp(); q.in_cp = iv.cp; q.in_off = iv.pad;
        q.h = c->oh; q.w = c->ow;
        q.clamp = c->clamp ? 1 : 0;
        q.out = ov.ptr; q.out_wp = ov.wp(); q.out_cp = ov.cp; q.out_off = ov.pad;
        q.groups = iv.cp / 8;
        q.f16 = ov.f16 ? 1 : 0;
        q.tiles_x = (q.w + 15) / 16; q.rcp_tiles_x = 1.0f / (float)q.tiles_x;
        std::vector<ConvC16Params> cands;
        size_t halves = 0;
        for (int i : pair_variants(a, c)) {
            int f16, groups, fr, th;
            conv_c16_variant(i, &f16, &groups, &fr, &th);
            if (want_th && th != want_th) continue;
            ConvC16Params t = q;
            t.th = th;
            t.tiles_y = (q.h + th - 1) / th;
            cands.push_back(t);
            int shares = 0;
            const int steps = conv_c16_steps(t, &shares);
            halves = std::max(halves, (size_t)2 * fr * shares * steps * (q.f16 ? 1 : 2) * 64 * 8);
        }
        if (cands.empty()) continue;
        void* const wp = net->dev_alloc(halves * 2, true);
        for (ConvC16Params& t : cands) t.wpack = wp;
        // (untimed: the tallest tiles that give half of the CUs a workgroup, on as many positions as are two rounds of the tallest
        // at most.  One launch / apart, fp32: 12x16 7.9 / 8.3 us, 156x128 12.0 / 16.3, 256x256 -- 688 tiles of six rows -- 32.0 / 29.2)
        int pick = 0;
        for (size_t i = 0; i < cands.size(); i++)
            if (cands[i].tiles_x * cands[i].tiles_y >= 128) pick = (int)i;
        if (!forced && (cands.back().tiles_x * cands.back().tiles_y > 512 || cands[0].tiles_x * cands[0].tiles_y < 64)) pick = -1;
        char key[200];
        snprintf(key, sizeof(key), "pair:%d:%dto%dto%d:%dx%d:r%d:e%d", q.f16, iv.cp, a->oc, c->oc, c->oh, c->ow, q.res ? 1 : 0, q.clamp);
        if (want_th || tune_cache_pick(net, key, cands.size(), forced, [&](size_t i, int b, int) { return cands[i].th == b; }, &pick)) {
        } else if (!(at && at[0] == '0')) {
            float t_one = 1e30f, t_apart = 1e30f;
            for (int rep = 0; rep < 3; rep++) {
                for (size_t i = 0; i < cands.size(); i++) {
                    const float t = time_calls(net, [&]() {
                        if (launch_conv_c16(cands[i], net->stream) != 0) fail(FYN_ERR_DEVICE, "launch of two 3x3 layers failed while tuning");
                    }, 10);
                    if (t < t_one) { t_one = t; pick = (int)i; }
                }
                t_apart = std::min(t_apart, time_calls(net, [&]() {
                    a->forward_alone(net->stream);
                    c->forward_alone(net->stream);
                }, 10));
            }
            if (net->sw.get("FYNHIP_TUNE_VERBOSE"))
                fprintf(stderr, "[tune] 3x3 %d to %d to %d at %dx%d: one launch (%d rows) %.1f us, apart %.1f us\n", iv.cp, a->oc, c->oc, c->oh, c->ow, cands[pick].th, t_one * 1e3f, t_apart * 1e3f);
            // (a tenth: on a few rows of tiles, where both ways are a chain of latencies, the frame does not show a smaller lead.  40 to 40
            // to 40, one launch / apart, and the frame of the sample net with its pairs joined / apart, us: fp32 12x16 7.9 / 8.3, 43.9 / 42.8;
            // 24x32 8.1 / 8.6, 44.1 / 43.1; 33x50 8.1 / 8.8, 45.5 / 45.0; 48x64 8.2 / 9.3, 47.0 / 47.3; 80x80 8.2 / 11.4, 55.9 / 61.0; fp16 24x32
            // 6.4 / 6.5, 35.0 / 34.8; 33x50 6.5 / 7.4, 35.6 / 37.0; 48x64 6.5 / 7.6, 36.7 / 39.3.  At 192x256, where the tiles take more than a
            // round, the timings tie, 22.5 / 22.3, and the frame with them within 1 %, 153.6 / 155.4; fp16 15.9 / 16.5, 104.8 / 105.8)
            const bool win = t_one < t_apart * 0.9f;
            tune_cache_store_triple(net, key, win ? 1 : 0, cands[pick].th, 0);
            if (!win && !forced) pick = -1;
        }
        if (pick < 0) {
            net->dev_free(wp);
            continue;
        }
        c->pair = cands[pick];
        c->pair_wpack_dev = wp;
        c->pair_fused = true;
        c->pair_layer = a->d.number;
        a->blk_into = c->d.number;
        net->read_until(x, c->d.number);
        c->pack_pair();
    }
}

// A sigmoid or tanh layer whose input comes from a convolution in the row-rolling form and goes nowhere else (the end of
// the style-net samples): the convolution applies it to what it stores, into the layer's own tensor.  The launch writes
// that tensor in the convolution's place in the order, earlier than its buffer was handed over for.
void fuse_function_layers(Net* net) {
    if (net->sw.get("FYNHIP_NO_FUNCTION_FUSION") || !net->reuse_buffers) return;
    std::map<int, int> readers;
    for (auto& kv : net->layers)
        for (int t : kv.second->in)
            if (t >= 0) readers[t]++;
    for (auto& kv : net->layers) {
        Layer* f = kv.second.get();
        const FuncParams* p = f->pointwise();
        if (!p) continue;
        const Tensor& t = net->tensors[f->in[0]];
        const Tensor& o = net->tensors[f->out];
        if (t.producer < 0 || t.locked || readers[f->in[0]] != 1) continue;
        ConvLayer* c = dynamic_cast<ConvLayer*>(net->layer(t.producer));
        if (!c || !c->rows || o.v.f16 != t.v.f16 || o.v.cp != 4 || t.v.cp != 4 || o.v.h != t.v.h || o.v.w != t.v.w) continue;
        if (!net->alone(f->out, c->d.number, f->d.number)) continue;
        c->fn_layer_no = f->d.number;
        c->fn_params = *p;
        f->computed_by(c->d.number);
        net->tensors[f->out].written = c->d.number;
    }
}


}  // namespace fynhip
