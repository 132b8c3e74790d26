// Encoder-stack handle behind the C ABI (et_model_*): assembles the C++ class
// layer (Linear / Attention / SkipLayerNorm / Encoder, include/et/*.h) from host
// weights the way the reference's example does (example/main.cu:24-182), chains
// the layers (example/main.cu:175-177) and replays the whole stack as one HIP
// graph.
#include <algorithm>
#include <array>
#include <memory>
#include <string>
#include <vector>

#include "et/Encoder.h"
#include "et/weights.hpp"

namespace {

using et::stream_t;

struct ILayer {
    virtual ~ILayer() = default;
    virtual et::LayerBuffers buffers() = 0;  // its own; the forwards below are given those they shall use
    virtual void forward(const et::LayerBuffers &b, half *out, half *src, stream_t stream) = 0;
    virtual void enable_mixed() = 0;
    virtual void forward_mixed(const et::LayerBuffers &b, float *out32, half *out16, const float *src32, half *src16, stream_t stream) = 0;
    virtual bool split_ok() const = 0;
    virtual void enable_split() = 0;
    virtual bool enable_fused_qkv(const half *gamma, const half *beta) = 0;
    virtual const half *norm2_gamma() const = 0;
    virtual const half *norm2_beta() const = 0;
    virtual et::SplitSum forward_split(const et::LayerBuffers &b, const et::SplitSum *in, const float *x32, half *x16, stream_t stream) = 0;
    virtual void finish_split(float *out32, half *out16, const et::SplitSum &s, stream_t stream) = 0;
    virtual bool chain_parts(et::ChainParts &p) = 0;
    virtual void chain_qkv_first(const et::LayerBuffers &b, half *x16, stream_t stream) = 0;
    virtual void chain_attention(const et::LayerBuffers &b, stream_t stream) = 0;
    virtual et::AttnState &attn() = 0;
    virtual bool local_weights(et_layer_weights &w) = 0;
    virtual bool local_qkv(et_layer_weights &w) = 0;
    virtual bool dense_weights(et_span (&w)[4]) = 0;
    virtual float epsilon(int k) const = 0;
};

template <typename EncoderT> struct LayerOf final : ILayer {
    std::unique_ptr<EncoderT> enc;
    explicit LayerOf(std::unique_ptr<EncoderT> e) : enc(std::move(e)) {}
    et::LayerBuffers buffers() override { return enc->buffers(); }
    void forward(const et::LayerBuffers &b, half *out, half *src, stream_t stream) override { enc->forward_f16_in(b, out, src, stream); }
    void enable_mixed() override { enc->enable_mixed(); }
    void forward_mixed(const et::LayerBuffers &b, float *out32, half *out16, const float *src32, half *src16, stream_t stream) override {
        enc->forward_mixed_in(b, out32, out16, src32, src16, stream);
    }
    bool split_ok() const override { return enc->split_ok(); }
    void enable_split() override { enc->enable_split(); }
    bool enable_fused_qkv(const half *gamma, const half *beta) override { return enc->enable_fused_qkv(gamma, beta); }
    const half *norm2_gamma() const override { return enc->norm2_gamma(); }
    const half *norm2_beta() const override { return enc->norm2_beta(); }
    et::SplitSum forward_split(const et::LayerBuffers &b, const et::SplitSum *in, const float *x32, half *x16, stream_t stream) override {
        return enc->forward_split_in(b, in, x32, x16, stream);
    }
    void finish_split(float *out32, half *out16, const et::SplitSum &s, stream_t stream) override {
        enc->finish_split(out32, out16, s, stream);
    }
    bool chain_parts(et::ChainParts &p) override { return enc->chain_parts(p); }
    void chain_qkv_first(const et::LayerBuffers &b, half *x16, stream_t stream) override { enc->chain_qkv_first_in(b, x16, stream); }
    void chain_attention(const et::LayerBuffers &b, stream_t stream) override { enc->chain_attention_in(b, stream); }
    et::AttnState &attn() override { return enc->attention(); }
    bool local_weights(et_layer_weights &w) override { return enc->local_weights(w); }
    bool local_qkv(et_layer_weights &w) override { return enc->local_qkv(w); }
    bool dense_weights(et_span (&w)[4]) override { return enc->dense_weights(w); }
    float epsilon(int k) const override { return enc->epsilon(k); }
};
struct LayerPackDeleter {
    void operator()(et_layer_pack_s *p) const { (void)et_encoder_layer_pack_destroy(p); }
};

// One weight matrix as handed over by the caller (host memory).
struct HostMatrix {
    enum Kind { None, Bsr16, Dense } kind = None;
    std::vector<int> row_ptr, column;
    std::vector<half> data;  // tiles [ntile][256] or dense [out][in]
    std::vector<half> bias;
};

struct HostLayer {
    std::array<HostMatrix, 4> w;  // ET_W_QKV, ET_W_O, ET_W_FF1, ET_W_FF2
    std::array<std::vector<half>, 2> gamma, beta;
};

using tile_attn_cfg = Attention_config<tile_mat, tile_mat, tile_mat, tile_mat, OTF_attn_full, true, false>;
using dense_attn_cfg = Attention_config<base_mat, base_mat, base_mat, base_mat, OTF_attn_full, true, false>;

struct Dims {
    int out, in;
};

}  // namespace

struct et_model_s {
    et_model_desc desc{};
    std::shared_ptr<Model_t> model;
    std::vector<HostLayer> host;
    std::vector<std::unique_ptr<ILayer>> layers;
    // layer i writes ring slot i % kRing, layer i + 1 reads it; a slot is written again kRing layers on
    static constexpr int kRing = 4;
    std::unique_ptr<et::DeviceBuffer<half>> pp[kRing];
    std::unique_ptr<et::DeviceBuffer<float>> pp32[kRing];  // mixed precision: the residual stream between layers
    std::unique_ptr<et::DeviceBuffer<half>> warm;      // result of the eager pass that precedes a capture
    std::vector<int> lens;   // empty = no padding
    std::vector<half> mask;  // empty = no additive mask
    bool finalized = false;
    bool split = false;  // mixed precision with SkipLayerNorm folded into the projections
    bool fused_qkv = false;  // and the QKV projection of every layer after the first inside its attention kernel
    // split, with everything between two attention kernels in one launch (et_encoder_chain_f32):
    // one description per layer and the barrier counters of all layers, cleared at the start of a forward
    bool chain = false;
    std::vector<et_chain_desc> chain_desc;
    std::unique_ptr<et::DeviceBuffer<int>> chain_sync;
    // everything between two attention kernels in one token-local launch (et_encoder_layer_f32), or in two with
    // several workgroups to a token strip: one pack per layer, the residual between layers, the shares of a strip.  mixed =
    // 0: shares for every layer, which may run on streams of their own (et_model_forward_layer); a whole forward keeps to
    // the first, which stays in the caches (six layers of 768, 528 rows: 309 us, 318 with a buffer a layer)
    std::vector<std::unique_ptr<et_layer_pack_s, LayerPackDeleter>> local;
    std::unique_ptr<et::DeviceBuffer<float>> local_x[2];
    std::vector<std::unique_ptr<et::DeviceBuffer<float>>> local_shares;
    std::vector<std::unique_ptr<et::DeviceBuffer<int>>> local_join;  // words at which the parts of a strip meet, a buffer for each of the shares
    float *shares(int layer) const { return local_shares.empty() ? nullptr : local_shares[(size_t)layer]->get(); }

    stream_t own_stream = nullptr;
    et_graph graph = nullptr;
    const void *graph_in = nullptr;
    void *graph_out = nullptr;

    int rows() const { return desc.batch * desc.seq_len; }
    Dims dims(int which) const {
        switch (which) {
            case ET_W_QKV: return {2 * desc.kdim + desc.vdim, desc.emdim};
            case ET_W_O: return {desc.emdim, desc.vdim};
            case ET_W_FF1: return {desc.dimFF, desc.emdim};
            default: return {desc.emdim, desc.dimFF};
        }
    }
    // The buffers layer i runs in as part of et_model_forward.  A whole forward keeps to those of one layer, with separate
    // launches of two: what it touches decides how much of the weights stays in the memory-side cache (256 MB) from one
    // forward to the next.  12 layers of BERT-base at 80 %, 64 x 128 tokens 1007 -> 860 us (a set a layer is 0.75 GB),
    // BERT-large 4 x 512 1352 -> 1165, 16 x 128 dense 1022 -> 992; 8 x 128 with two more models run in between 457 -> 396.
    // (Separate launches in one set: 16 x 128 dense 980, but 2 x 128 under mixed = 0 370 where two sets take 361.)
    et::LayerBuffers stack_buffers(int i) const {
        et::LayerBuffers b = layers[(size_t)(local.empty() ? i % 2 : 0) % layers.size()]->buffers();
        if (!ahead.empty()) b.ahead = ahead[(size_t)i].data(), b.nahead = (int)ahead[(size_t)i].size();
        return b;
    }
    std::vector<std::vector<et_span>> ahead;  // of every layer (plan_ahead), or none
    void drop_graph() {
        if (graph) (void)et_graph_destroy(graph);
        graph = nullptr;
    }
    ~et_model_s() {
        drop_graph();
        if (own_stream) (void)et_stream_destroy(own_stream);
    }
};

namespace {

template <typename Fn> int guarded(Fn fn) {
    try {
        return fn();
    } catch (const et::Error &e) {
        et_set_last_error(e.what());
        return e.status();
    } catch (const std::exception &e) {
        et_set_last_error(e.what());
        return ET_ERR_INVALID_ARG;
    }
}

template <typename MAT> std::unique_ptr<Linear<MAT>> make_linear(const HostMatrix &m, Dims d, int rows);

template <> std::unique_ptr<Linear<tile_mat>> make_linear<tile_mat>(const HostMatrix &m, Dims d, int rows) {
    tile_mat w(m.row_ptr, m.column, m.data, d.in / 16);
    et::require(w.blk_row_num == d.out / 16, "BSR weight: row_ptr length does not match the output width");
    return std::make_unique<Linear<tile_mat>>(d.in, d.out, std::move(w), m.bias.data(), rows);
}

template <> std::unique_ptr<Linear<base_mat>> make_linear<base_mat>(const HostMatrix &m, Dims d, int rows) {
    return std::make_unique<Linear<base_mat>>(d.in, d.out, base_mat(m.data), m.bias.data(), rows);
}

template <typename MAT, typename attn_cfg, typename ACT>
std::unique_ptr<ILayer> build_layer(et_model_s &m, const HostLayer &h) {
    // the layer body of Encoder<Encoder_config<attn_cfg, MAT, MAT, ACT>> without that class's own choice of
    // precision: the model's `mixed` field decides here which buffers a layer gets
    using enc_t = et::EncoderLayer<Attention<attn_cfg>, Linear<MAT>, Linear<MAT>, ACT>;
    const int rows = m.rows();
    auto lqkv = make_linear<MAT>(h.w[ET_W_QKV], m.dims(ET_W_QKV), rows);
    auto lo = make_linear<MAT>(h.w[ET_W_O], m.dims(ET_W_O), rows);
    auto attn = std::make_unique<Attention<attn_cfg>>(std::move(lqkv), std::move(lo), m.model, m.desc.batch);
    attn->set_causal(m.desc.causal != 0);
    auto ln1 = std::make_unique<SkipLayerNorm>(h.gamma[0].data(), h.beta[0].data(), m.desc.emdim, m.desc.eps);
    auto ln2 = std::make_unique<SkipLayerNorm>(h.gamma[1].data(), h.beta[1].data(), m.desc.emdim, m.desc.eps);
    auto l1 = make_linear<MAT>(h.w[ET_W_FF1], m.dims(ET_W_FF1), rows);
    auto l2 = make_linear<MAT>(h.w[ET_W_FF2], m.dims(ET_W_FF2), rows);
    auto enc = std::make_unique<enc_t>(std::move(attn), std::move(ln1), std::move(ln2), std::move(l1),
                                       std::move(l2), m.model);
    return std::make_unique<LayerOf<enc_t>>(std::move(enc));
}

template <typename MAT, typename attn_cfg> std::unique_ptr<ILayer> build_layer_act(et_model_s &m, const HostLayer &h) {
    if (m.desc.act == ET_ACT_RELU) return build_layer<MAT, attn_cfg, RELU_OP>(m, h);
    return build_layer<MAT, attn_cfg, GELU_OP>(m, h);
}

void apply_attention_state(et_model_s &m) {
    for (auto &l : m.layers) {
        l->attn().set_lens(m.lens.empty() ? nullptr : m.lens.data());
        l->attn().set_mask(m.mask.empty() ? nullptr : m.mask.data());
    }
}

void check_layer_index(const et_model_s *m, int layer) {
    et::require(m != nullptr, "et_model: NULL handle");
    et::require(layer >= 0 && layer < m->desc.nlayer, "et_model: layer index out of range");
}

// Mixed precision: the binary16 input is widened once, every layer hands the next one its result
// in both forms (binary32 residual, binary16 operand), the last one writes binary16 to `out`.
// The same with SkipLayerNorm folded into the neighbouring projections (five launches per layer):
// every layer hands the next one its un-normalised binary32 result with its row sums.
// The descriptions of the chain launches, or false when some layer has no such form.  Layer i's
// launch holds its output projection and FFN and layer i + 1's QKV projection.
bool build_chain(et_model_s &m) {
    const int n = (int)m.layers.size();
    std::vector<et::ChainParts> parts((size_t)n);
    for (int i = 0; i < n; i++)
        if (!m.layers[(size_t)i]->chain_parts(parts[(size_t)i])) return false;
    m.chain_sync = std::make_unique<et::DeviceBuffer<int>>((size_t)n * ET_CHAIN_SYNC_WORDS);
    m.chain_desc.assign((size_t)n, et_chain_desc{});
    for (int i = 0; i < n; i++) {
        const et::ChainParts &p = parts[(size_t)i];
        et_chain_desc &d = m.chain_desc[(size_t)i];
        d.o = p.o;
        d.bias_o = et::f16(p.bias_o);
        d.Z = et::f16(p.Z);
        if (i > 0) {  // the residual is LayerNorm2 of the previous layer's sum, formed from the statistics
                      // this layer's QKV projection left
            const et::ChainParts &q = parts[(size_t)i - 1];
            d.resid = q.V2;
            d.resid_fin = p.fin_in;
            d.resid_gamma = et::f16(q.gamma2);
            d.resid_beta = et::f16(q.beta2);
        }  // i == 0: resid16 = the model's input, set at run time
        d.V1 = p.V1;
        d.stats1 = p.stats1;
        d.up = p.up;
        d.bias_up = et::f16(p.bias_up);
        d.gamma1 = et::f16(p.gamma1);
        d.beta1 = et::f16(p.beta1);
        d.eps1 = p.eps1;
        d.fin1 = p.fin1;
        d.H = et::f16(p.H);
        d.act = p.act;
        d.down = p.down;
        d.bias_down = et::f16(p.bias_down);
        d.V2 = p.V2;
        d.stats2 = p.stats2;
        if (i + 1 < n) {
            const et::ChainParts &nx = parts[(size_t)i + 1];
            d.qkv = nx.qkv;
            d.bias_qkv = et::f16(nx.bias_qkv);
            d.gamma2 = et::f16(p.gamma2);
            d.beta2 = et::f16(p.beta2);
            d.eps2 = p.eps2;
            d.fin2 = nx.fin_in;
            d.QKV = et::f16(nx.QKV);
        }
        d.T = m.rows();
        d.sync = reinterpret_cast<uint32_t *>(m.chain_sync->get()) + (size_t)i * ET_CHAIN_SYNC_WORDS;
        et_chain_desc probe = d;
        if (i == 0) probe.resid16 = d.Z;  // any pointer: only the shapes are looked at
        if (et_encoder_chain_supported(&probe) != 1) return false;
    }
    return true;
}

// Two launches per layer: the attention kernel, and one chain launch for everything up to the next
// layer's QKV projection.
void run_layers_chain(et_model_s &m, half *out, half *in, stream_t stream) {
    const int n = (int)m.layers.size();
    etChk(et_fill_i32(m.chain_sync->get(), m.chain_sync->size, 0, stream));
    m.layers[0]->chain_qkv_first(m.layers[0]->buffers(), in, stream);
    et::SplitSum carry;
    for (int i = 0; i < n; i++) {
        m.layers[(size_t)i]->chain_attention(m.layers[(size_t)i]->buffers(), stream);
        et_chain_desc d = m.chain_desc[(size_t)i];
        if (i == 0) d.resid16 = et::f16(in);
        int groups2 = 0;
        etChk(et_encoder_chain_f32(&d, &groups2, stream));
        carry.v = d.V2;
        carry.stats = d.stats2;
        carry.groups = groups2;
    }
    // the last layer's sum is normalised by its second LayerNorm
    et::ChainParts last;
    (void)m.layers[(size_t)n - 1]->chain_parts(last);
    carry.gamma = last.gamma2;
    carry.beta = last.beta2;
    carry.eps = last.eps2;
    m.layers[(size_t)n - 1]->finish_split(nullptr, out, carry, stream);
}

// true when every chain launch of the last forward ran as it must (blocking)
bool chain_ran_clean(et_model_s &m, std::string &why) {
    const int n = (int)m.layers.size();
    for (int i = 0; i < n; i++) {
        int gave_up = 0, misplaced = 0;
        etChk(et_encoder_chain_status(m.chain_desc[(size_t)i].sync, &gave_up, &misplaced));
        if (gave_up || misplaced) {
            why = "layer " + std::to_string(i) + ": " + std::to_string(gave_up) + " workgroups gave up at a barrier, " +
                  std::to_string(misplaced) + " ran on another XCD than the rest of their group";
            return false;
        }
    }
    return true;
}

// How a stack divides a token strip: token rows of a workgroup over 16, and workgroups that share a strip; mt == 0: the
// separate launches are faster.
struct LocalPlan {
    int mt = 0, parts = 1;
};
// Every workgroup streams the kept tiles of the output projection and its share of the others at about 112 KiB/us.  Sharing a
// strip costs a meeting of its parts and half a microsecond a part, more where an XCD has many strips (fitted at 768 wide, 60 to
// 95 % sparsity, 128 to 2048 rows, shared strips in one launch): the number of parts that makes the sum least, while there is a
// compute unit for every workgroup of an XCD; beyond eight the shares cost more than they save (128 rows at 60 %, four layers:
// 134 us with 8, 144 with 12).  Above 256 strips of 16 rows a workgroup takes 32.
// Which stacks run it: time of the separate launches over that of these, stacks of two and of six layers (whose ratios differ
// by 0.05 in the mean: what the first layer's projection takes), 384 to 1024 wide with an FFN of four times the width, 512 to 800
// with 208 to 768 hidden features, 20 to 95 % sparsity, 16 to 1024 rows, and 768 wide with the QKV projection inside the attention
// kernel (four launches, 128 to 1024 rows: 0.93 - 1.33).  "half" is at most half of the tiles kept (denser layers run dense
// GEMMs beside), us the estimate above; of 3036 stacks the lines take the better form or one within 3 % for all but 98, 0.3 % from
// it on average.  On the side that takes the token-local launches, and on the other:
//  binary32 residual:
//   more than 16.5 KiB of tiles a feature                                0.66 - 1.13
//   257 rows and more                      1.01 - 1.68
//   193 to 256: half, to 18 us             0.97 - 1.31   above           0.95 - 1.03;  denser 1.03 - 1.51
//   144 to 192: to 32 us                   0.96 - 1.49
//   112 and 128 (the separate launches have a strip for each XCD):
//     half, to 13.5 us                     0.97 - 1.27   above           0.93 - 1.06
//       FFN narrower than the model, to 6.5  1.03 - 1.26 above           0.94 - 1.14
//     denser, to 20.5 us                   1.04 - 1.40   above           0.89 - 0.96
//   fewer: half                            0.98 - 2.23
//     denser, to 18.5 us                   0.95 - 1.36   above           0.77 - 1.05
//  binary16 between layers (mixed = 0):
//   above 4096 rows up to 18 KiB of tiles a feature 1.07 - 1.98, 1024 wide unpruned (24) 0.78
//   257 rows and more: half                0.98 - 1.57
//     denser, to 11 KiB of tiles a feature 0.95 - 1.43   above           0.74 - 1.15
//   FFN narrower than the model: 144 to 240 rows, to 15 us 0.90 - 1.31, up to 64, to 12 us 0.93 - 1.41, others, to 6.5 us
//                                          0.99 - 1.22;  above 0.91 - 0.97, 0.78 - 0.96, 0.81 - 1.07
//   256: to 12.5 us                        0.93 - 1.17   above           0.84 - 1.03
//   193 to 240: to 20.5 us                 0.93 - 1.34   above           0.89 - 1.15
//   144 to 192: to 23 us                   0.90 - 1.39   above           0.91 - 1.06
//   128: up to 512 wide, to 11 us          0.97 - 1.14   above           0.92 - 0.94
//     wider, to 6.5 us                     0.93 - 1.06   above           0.69 - 1.01
//   112: to 14.6 us                        0.85 - 1.23   above           0.70 - 0.97
//   fewer: half                            0.94 - 2.25
//     denser, to 13 us                     0.96 - 1.19   above           0.69 - 1.25
//  A single layer has no projection behind it to run in the launch: at 112 and 128 rows, to 5 us 0.97 - 1.07, above 0.84 - 0.96.
LocalPlan plan_local(const et_model_s &m) {
    LocalPlan p;
    const et_model_desc &d = m.desc;
    double kib[4] = {0, 0, 0, 0};  // of a layer, on average
    for (const HostLayer &h : m.host)
        for (int w = 0; w < 4; w++) {
            if (h.w[(size_t)w].kind != HostMatrix::Bsr16) return p;
            kib[w] += 0.5 * (double)h.w[(size_t)w].column.size() / (double)m.host.size();
        }
    const int rows = m.rows(), strips = (rows + 15) / 16, per_xcd = (strips + 7) / 8;
    const double shared = kib[ET_W_QKV] + kib[ET_W_FF1] + kib[ET_W_FF2], kept = kib[ET_W_O] + shared;
    const double all = (4.0 * d.emdim + 2.0 * d.dimFF) * d.emdim / 512.0;  // KiB of all tiles
    if (strips > 256) {
        if (d.mixed || kept <= 18.0 * d.emdim) p.mt = 2;
        return p;
    }
    double best = 0;
    for (int parts = 1; parts <= std::min(8, d.dimFF / 16) && parts * per_xcd <= 32; parts++) {
        const double us = (kib[ET_W_O] + shared / parts) / 112.0 + (parts > 1 ? 0.5 + (0.45 + 0.045 * per_xcd) * parts : 0.0);
        if (parts == 1 || us < best) {
            best = us;
            p.parts = parts;
        }
    }
    const bool half = kept <= 0.5 * all, narrow = d.dimFF < d.emdim;
    bool on;
    if (d.mixed == 0) {
        if (strips > 16) on = half || kept <= 11.0 * d.emdim;
        else if (narrow) on = best <= (strips > 8 && strips < 16 ? 15.0 : strips <= 4 ? 12.0 : 6.5);
        else if (strips > 8) on = best <= (strips == 16 ? 12.5 : strips > 12 ? 20.5 : 23.0);
        else if (strips > 6) on = best <= (strips == 7 ? 14.6 : d.emdim <= 512 ? 11.0 : 6.5);
        else on = half || best <= 13.0;
    } else if (kept > 16.5 * d.emdim) on = false;
    else if (strips > 16) on = true;
    else if (strips > 8) on = best <= (strips > 12 && half ? 18.0 : 32.0);
    else if (strips > 6) on = best <= (!half ? 20.5 : narrow ? 6.5 : 13.5);
    else on = half || best <= 18.5;
    if (m.host.size() == 1 && (strips == 7 || strips == 8)) on = on && best <= 5.0;
    p.mt = on ? 1 : 0;
    return p;
}

// The packs of the token-local launches; leaves m.local empty where a layer has no such form.
void build_local(et_model_s &m) {
    const LocalPlan plan = plan_local(m);
    const et_model_desc &d = m.desc;
    const int n = (int)m.layers.size(), ldq = 2 * d.kdim + d.vdim;
    if (plan.mt == 0 || d.kdim != d.emdim || d.vdim != d.emdim || et_encoder_layer_supported(m.rows(), d.emdim, d.dimFF, ldq) != 1) return;
    std::vector<std::unique_ptr<et_layer_pack_s, LayerPackDeleter>> packs;
    for (int i = 0; i < n; i++) {
        et_layer_weights w{};
        if (!m.layers[(size_t)i]->local_weights(w) || (i + 1 < n && !m.layers[(size_t)i + 1]->local_qkv(w))) return;
        et_layer_pack_s *p = nullptr;
        const auto create = d.mixed ? et_encoder_layer_pack_create : et_encoder_layer_pack_create_projecting;
        const int s = create(&w, m.rows(), d.emdim, d.dimFF, i + 1 < n ? ldq : 0, plan.mt, plan.parts, &p);
        if (s == ET_ERR_UNSUPPORTED) return;
        etChk(s);
        packs.emplace_back(p);
    }
    const size_t elems = (size_t)m.rows() * d.emdim;
    if (d.mixed)
        for (auto &b : m.local_x) b = std::make_unique<et::DeviceBuffer<float>>(elems);
    if (plan.parts > 1)
        for (int i = 0; i < (d.mixed ? 1 : n); i++) m.local_shares.push_back(std::make_unique<et::DeviceBuffer<float>>(elems * plan.parts));
    int joins = 0;
    if (plan.parts > 1) etChk(et_encoder_layer_joins(packs[0].get(), &joins));
    for (size_t i = 0; joins && i < m.local_shares.size(); i++) {
        const std::vector<int> zero((size_t)(m.rows() + 15) / 16, 0);
        m.local_join.push_back(std::make_unique<et::DeviceBuffer<int>>(zero.data(), zero.size()));
    }
    m.local = std::move(packs);
}

// Weights that a layer's launches read, asked for by its attention kernel (et_mha_fused_ahead_f16): the streams of the
// token-local launches, or O, FFN and the next QKV of a dense layer.  For a model whose weights and activations do not stay
// in the memory-side cache from one forward to the next, and enough token rows that the attention takes about as long as the
// requests.  us, off / on: 12 layers of BERT-base at 80 %, 64 x 128 tokens, three models in turn 990 / 890, one model again and
// again 855 / 856; BERT-large at 90 %, 4 x 512 1349 / 1238, 1172 / 1171; 16 x 128 dense 1017 / 997, 996 / 992; 32 x 128 dense one
// model 1685 / 1612.  On the other side of the lines: 8 x 128 at 80 % (70 MB in all) 394 / 401, 384 / 392; 4 x 128 dense 604 / 619.
void plan_ahead(et_model_s &m) {
    const size_t n = m.layers.size();
    const et_model_desc &d = m.desc;
    const int ldq = 2 * d.kdim + d.vdim;
    std::vector<std::vector<et_span>> ahead(n);
    double bytes = 0;
    for (size_t i = 0; i < n; i++) {
        et_span w[4], next[4];
        if (!m.local.empty()) {
            ahead[i].resize(1);
            etChk(et_encoder_layer_pack_streams(m.local[i].get(), ahead[i].data()));
        } else if (m.layers[i]->dense_weights(w)) {
            ahead[i] = {w[1], w[2], w[3]};
            if (i + 1 < n && m.layers[i + 1]->dense_weights(next)) ahead[i].push_back(next[0]);
        } else {
            return;
        }
        for (const et_span &s : ahead[i]) bytes += (double)s.bytes;
    }
    // a row of what the forward writes: binary16 projections and results, the binary32 residual and shares
    const int parts = m.local_shares.empty() ? 0 : (int)(m.local_shares[0]->size / ((size_t)m.rows() * d.emdim));
    const double row = m.local.empty() ? 4.0 * (ldq + d.vdim + 3 * d.emdim + d.dimFF) : 2.0 * (ldq + d.vdim) + (8.0 + 4.0 * parts) * d.emdim;
    if (m.rows() >= 2048 && bytes + row * m.rows() >= 96.0 * (1 << 20)) m.ahead = std::move(ahead);
}

// The token-local launches read and write up to 16 bytes at a time; input and result at another address (which the
// separate launches take) pass through buffers of the layer that these launches leave alone.
bool local_aligned(const half *p) { return (reinterpret_cast<std::uintptr_t>(p) & 15) == 0; }
void copy_rows(et_model_s &m, half *to, const half *from, stream_t stream) {
    etChk(et_memcpy_d2d(to, from, (std::size_t)m.rows() * m.desc.emdim * sizeof(half), stream));
}
half *local_input(et_model_s &m, const et::LayerBuffers &b, half *in, stream_t stream) {
    if (local_aligned(in)) return in;
    copy_rows(m, b.attn, in, stream);
    return b.attn;
}
half *local_result(const et::LayerBuffers &b, half *out) { return local_aligned(out) ? out : b.ffn; }

// The token-local launches of layer i; `k`: the shares it runs with.
void run_local(et_model_s &m, int i, int k, const half *z, const float *x32, const half *x16, float *x32_out, half *out16, half *qkv, stream_t stream) {
    const ILayer &l = *m.layers[(size_t)i];
    if (m.local_join.empty())
        etChk(et_encoder_layer_f32(m.local[(size_t)i].get(), et::f16(z), x32, et::f16(x16), x32_out, et::f16(out16), et::f16(qkv), m.shares(k),
                                   m.desc.act, l.epsilon(0), l.epsilon(1), stream));
    else
        etChk(et_encoder_layer_joined_f32(m.local[(size_t)i].get(), et::f16(z), x32, et::f16(x16), x32_out, et::f16(out16), et::f16(qkv), m.shares(k),
                                          reinterpret_cast<uint32_t *>(m.local_join[(size_t)k]->get()), 4000, m.desc.act, l.epsilon(0),
                                          l.epsilon(1), stream));
}

// One layer from binary16 to binary16, as et_model_forward under mixed = 0 chains it (`chained`: behind the layer before it)
// and et_model_forward_layer issues it.  The token-local launches take the layer's input and leave its result in binary16,
// and the next layer's QKV made from the result as they round it; a layer that runs alone makes its QKV from its input with
// the same products, so that it does the same whether the one before it ran in the same call or not, and leaves the next
// one's where its own was read: it touches no buffer of another layer.
void run_layer_f16(et_model_s &m, int i, half *out, half *in, bool chained, stream_t stream) {
    ILayer &l = *m.layers[(size_t)i];
    const et::LayerBuffers b = chained ? m.stack_buffers(i) : l.buffers();
    if (m.local.empty()) return l.forward(b, out, in, stream);
    if (i == 0) l.chain_qkv_first(b, in, stream);
    half *x = local_input(m, b, in, stream), *to = local_result(b, out);
    if (i > 0 && !chained) etChk(et_encoder_layer_project_f16(m.local[(size_t)i - 1].get(), et::f16(x), et::f16(b.qkv), stream));
    l.chain_attention(b, stream);
    const bool last = i + 1 == (int)m.layers.size();
    half *qkv = last ? nullptr : chained ? m.stack_buffers(i + 1).qkv : b.qkv;
    run_local(m, i, chained ? 0 : i, b.z, nullptr, x, nullptr, to, qkv, stream);
    if (to != out) copy_rows(m, out, to, stream);
}

void run_layers_local(et_model_s &m, half *out, half *in, stream_t stream) {
    const int n = (int)m.layers.size();
    const et::LayerBuffers first = m.stack_buffers(0), end = m.stack_buffers(n - 1);
    m.layers[0]->chain_qkv_first(first, in, stream);
    half *x = local_input(m, first, in, stream), *to = local_result(end, out);
    for (int i = 0; i < n; i++) {
        ILayer &l = *m.layers[(size_t)i];
        const et::LayerBuffers b = m.stack_buffers(i);
        const bool last = i == n - 1;
        l.chain_attention(b, stream);
        run_local(m, i, 0, b.z, i ? m.local_x[(i - 1) & 1]->get() : nullptr, i ? nullptr : x, last ? nullptr : m.local_x[i & 1]->get(),
                  last ? to : nullptr, last ? nullptr : m.stack_buffers(i + 1).qkv, stream);
    }
    if (to != out) copy_rows(m, out, to, stream);
}

void run_layers_split(et_model_s &m, half *out, half *in, stream_t stream) {
    if (m.chain) return run_layers_chain(m, out, in, stream);
    const int n = (int)m.layers.size();
    // the first layer adds the binary16 input as its residual: no widened copy
    et::SplitSum carry;
    for (int i = 0; i < n; i++)
        carry = m.layers[(size_t)i]->forward_split(m.stack_buffers(i), i ? &carry : nullptr, nullptr, in, stream);
    m.layers[(size_t)n - 1]->finish_split(nullptr, out, carry, stream);
}

void run_layers_mixed(et_model_s &m, half *out, half *in, stream_t stream) {
    if (m.split) return run_layers_split(m, out, in, stream);
    const int n = (int)m.layers.size();
    const std::size_t elems = (std::size_t)m.rows() * m.desc.emdim;
    constexpr int R = et_model_s::kRing;
    etChk(et_f16_to_f32(m.pp32[R - 1]->get(), et::f16(in), elems, stream));
    const float *src32 = m.pp32[R - 1]->get();
    half *src16 = in;
    for (int i = 0; i < n; i++) {
        const bool last = i == n - 1;
        float *dst32 = last ? nullptr : m.pp32[i % R]->get();
        half *dst16 = last ? out : m.pp[i % R]->get();
        m.layers[(size_t)i]->forward_mixed(m.stack_buffers(i), dst32, dst16, src32, src16, stream);
        src32 = dst32;
        src16 = dst16;
    }
}

void run_layers(et_model_s &m, half *out, half *in, stream_t stream) {
    if (m.desc.mixed) return m.local.empty() ? run_layers_mixed(m, out, in, stream) : run_layers_local(m, out, in, stream);
    const int n = (int)m.layers.size();
    half *src = in;
    for (int i = 0; i < n; i++) {
        half *dst = (i == n - 1) ? out : m.pp[i % et_model_s::kRing]->get();
        run_layer_f16(m, i, dst, src, true, stream);
        src = dst;
    }
}

std::vector<half> to_half(const float *src, size_t n) {
    std::vector<half> v(n);
    for (size_t i = 0; i < n; i++) v[i] = static_cast<half>(src[i]);
    return v;
}
std::vector<half> to_half(const et_f16 *src, size_t n) {
    std::vector<half> v(n);
    if (n) std::memcpy(v.data(), src, n * sizeof(half));  // an empty vector's data() may be null
    return v;
}

template <typename T>
int set_bsr16(et_model m, int layer, int which, const int32_t *row_ptr, const int32_t *column, const T *data,
              int ntile, const T *bias) {
    return guarded([&]() -> int {
        check_layer_index(m, layer);
        et::require(!m->finalized, "et_model: weights cannot change after et_model_finalize");
        et::require(which >= ET_W_QKV && which <= ET_W_FF2, "et_model_set_bsr16: bad matrix selector");
        et::require(row_ptr && ntile >= 0 && (ntile == 0 || (column && data)), "et_model_set_bsr16: NULL pointer");
        const Dims d = m->dims(which);
        et::require(d.out % 16 == 0 && d.in % 16 == 0, "et_model_set_bsr16: model widths must be multiples of 16");
        HostMatrix &w = m->host[(size_t)layer].w[(size_t)which];
        w.kind = HostMatrix::Bsr16;
        w.row_ptr.assign(row_ptr, row_ptr + d.out / 16 + 1);
        w.column.assign(column, column + ntile);
        w.data = to_half(data, (size_t)ntile * 256);
        w.bias = bias ? to_half(bias, (size_t)d.out) : std::vector<half>((size_t)d.out, half_zero);
        et::fmt::validate_bsr16(w.row_ptr, w.column, (size_t)ntile, d.in / 16);
        return ET_OK;
    });
}

template <typename T>
int set_dense(et_model m, int layer, int which, const T *W, const T *bias) {
    return guarded([&]() -> int {
        check_layer_index(m, layer);
        et::require(!m->finalized, "et_model: weights cannot change after et_model_finalize");
        et::require(which >= ET_W_QKV && which <= ET_W_FF2, "et_model_set_dense: bad matrix selector");
        et::require(W != nullptr, "et_model_set_dense: NULL pointer");
        const Dims d = m->dims(which);
        HostMatrix &w = m->host[(size_t)layer].w[(size_t)which];
        w.kind = HostMatrix::Dense;
        w.data = to_half(W, (size_t)d.out * d.in);
        w.bias = bias ? to_half(bias, (size_t)d.out) : std::vector<half>((size_t)d.out, half_zero);
        return ET_OK;
    });
}

template <typename T> int set_norm(et_model m, int layer, int which, const T *gamma, const T *beta) {
    return guarded([&]() -> int {
        check_layer_index(m, layer);
        et::require(!m->finalized, "et_model: weights cannot change after et_model_finalize");
        et::require((which == 0 || which == 1) && gamma && beta, "et_model_set_norm: bad arguments");
        m->host[(size_t)layer].gamma[(size_t)which] = to_half(gamma, (size_t)m->desc.emdim);
        m->host[(size_t)layer].beta[(size_t)which] = to_half(beta, (size_t)m->desc.emdim);
        return ET_OK;
    });
}

}  // namespace

extern "C" {

int et_model_create(const et_model_desc *desc, et_model *out) {
    return guarded([&]() -> int {
        et::require(desc && out, "et_model_create: NULL argument");
        *out = nullptr;
        const et_model_desc &d = *desc;
        et::require(d.kdim > 0 && d.vdim > 0 && d.seq_len > 0 && d.nhead > 0 && d.dimFF > 0 && d.emdim > 0 &&
                        d.nlayer > 0 && d.batch > 0,
                    "et_model_create: every dimension must be positive");
        et::require(d.kdim == d.vdim && d.kdim % d.nhead == 0, "et_model_create: kdim must equal vdim and divide by nhead");
        et::require(d.act == ET_ACT_RELU || d.act == ET_ACT_GELU, "et_model_create: act must be ET_ACT_RELU or ET_ACT_GELU");
        auto m = std::make_unique<et_model_s>();
        m->desc = d;
        if (m->desc.eps <= 0.0f) m->desc.eps = 1e-5f;
        m->model = std::make_shared<Model_t>(Model_t{d.kdim, d.vdim, d.seq_len, d.nhead, d.dimFF, d.emdim, d.nlayer});
        m->host.resize((size_t)d.nlayer);
        *out = m.release();
        return ET_OK;
    });
}

int et_model_set_bsr16(et_model m, int layer, int which, const int32_t *row_ptr, const int32_t *column,
                       const float *data, int ntile, const float *bias) {
    return set_bsr16<float>(m, layer, which, row_ptr, column, data, ntile, bias);
}

int et_model_set_bsr16_f16(et_model m, int layer, int which, const int32_t *row_ptr, const int32_t *column,
                           const et_f16 *data, int ntile, const et_f16 *bias) {
    return set_bsr16<et_f16>(m, layer, which, row_ptr, column, data, ntile, bias);
}

int et_model_set_dense(et_model m, int layer, int which, const float *W, const float *bias) {
    return set_dense<float>(m, layer, which, W, bias);
}

int et_model_set_dense_f16(et_model m, int layer, int which, const et_f16 *W, const et_f16 *bias) {
    return set_dense<et_f16>(m, layer, which, W, bias);
}

int et_model_set_norm(et_model m, int layer, int which, const float *gamma, const float *beta) {
    return set_norm<float>(m, layer, which, gamma, beta);
}

int et_model_set_norm_f16(et_model m, int layer, int which, const et_f16 *gamma, const et_f16 *beta) {
    return set_norm<et_f16>(m, layer, which, gamma, beta);
}

int et_model_set_lens(et_model m, const int32_t *lens_host) {
    return guarded([&]() -> int {
        et::require(m != nullptr, "et_model_set_lens: NULL handle");
        if (lens_host) m->lens.assign(lens_host, lens_host + m->desc.batch);
        else m->lens.clear();
        if (m->finalized) {
            etChk(et_device_sync());  // a replay in flight may still read the old lengths
            apply_attention_state(*m);
            m->drop_graph();          // the graph holds the old device pointers
        }
        return ET_OK;
    });
}

int et_model_set_mask(et_model m, const et_f16 *mask_host) {
    return guarded([&]() -> int {
        et::require(m != nullptr, "et_model_set_mask: NULL handle");
        const size_t n = (size_t)m->desc.seq_len * m->desc.seq_len;
        if (mask_host) m->mask = to_half(mask_host, n);
        else m->mask.clear();
        if (m->finalized) {
            etChk(et_device_sync());
            apply_attention_state(*m);
            m->drop_graph();
        }
        return ET_OK;
    });
}

int et_model_finalize(et_model m) {
    return guarded([&]() -> int {
        et::require(m != nullptr, "et_model_finalize: NULL handle");
        et::require(!m->finalized, "et_model_finalize: already finalized");
        // every device buffer of the model comes from slabs of the model's own, at fixed places in them
        struct PoolScope {
            PoolScope() { etChk(et_pool_private_begin(0)); }
            ~PoolScope() { (void)et_pool_private_end(); }
        } pool_scope;
        for (int i = 0; i < m->desc.nlayer; i++) {
            const HostLayer &h = m->host[(size_t)i];
            const HostMatrix::Kind kind = h.w[0].kind;
            for (const HostMatrix &w : h.w) {
                et::require(w.kind != HostMatrix::None, "et_model_finalize: a weight matrix was never set");
                et::require(w.kind == kind, "et_model_finalize: one layer mixes dense and BSR weights");
            }
            for (int k = 0; k < 2; k++)
                et::require(!h.gamma[(size_t)k].empty(), "et_model_finalize: a LayerNorm was never set");
            if (kind == HostMatrix::Bsr16) m->layers.push_back(build_layer_act<tile_mat, tile_attn_cfg>(*m, h));
            else m->layers.push_back(build_layer_act<base_mat, dense_attn_cfg>(*m, h));
        }
        const size_t act_elems = (size_t)m->rows() * m->desc.emdim;
        for (auto &b : m->pp) b = std::make_unique<et::DeviceBuffer<half>>(act_elems);
        m->warm = std::make_unique<et::DeviceBuffer<half>>(act_elems);
        // The QKV projection inside the attention kernel: asked for (mixed == 4), or where it measured faster than
        // the two launches it replaces — one workgroup per (sequence, head) that reads and normalises its whole
        // sequence: 12-layer 768-wide stacks at 80 / 90 / 95 % sparsity ran 0.89 - 0.99 of the five-launch time
        // with 96 to 384 such workgroups (sequences of 32 to 128 tokens) — 96 of them on sequences of 96 or 128
        // tokens 0.99 - 1.01 —, 1.04 - 1.05 at 72 and below, 1.09 - 1.11 at 768.
        const et_model_desc &d = m->desc;
        const long heads = (long)d.batch * d.nhead;
        const bool want_fused = (d.mixed == 4 || (d.mixed == 1 && heads >= 96 && heads <= 400)) && m->layers.size() > 1;
        const bool fused_ok = want_fused && et_norm_qkv_mha_f32in_supported(d.batch, d.seq_len, d.emdim, d.nhead, d.kdim / d.nhead) == 1;
        if (d.mixed == 0 || d.mixed == 1 || (d.mixed == 4 && !fused_ok)) build_local(*m);
        if (m->desc.mixed) {
            for (auto &b : m->pp32) b = std::make_unique<et::DeviceBuffer<float>>(act_elems);
            for (auto &l : m->layers) l->enable_mixed();
            // mixed == 1: the engine folds SkipLayerNorm into the projections where every layer can
            m->split = (m->desc.mixed == 1 || m->desc.mixed == 3 || m->desc.mixed == 4 || m->desc.mixed == 5) && !m->layers.empty();
            for (auto &l : m->layers) m->split = m->split && l->split_ok();
            if (m->split && m->local.empty()) {
                for (auto &l : m->layers) l->enable_split();
                m->chain = m->desc.mixed == 3 && build_chain(*m);
                if (want_fused) {
                    m->fused_qkv = true;
                    // (the affine part of the normalisation a layer is handed — the second one of the layer before —
                    // goes into its projection's pack)
                    for (size_t i = 1; i < m->layers.size(); i++)
                        m->fused_qkv = m->layers[i]->enable_fused_qkv(m->layers[i - 1]->norm2_gamma(), m->layers[i - 1]->norm2_beta()) &&
                                       m->fused_qkv;
                }
            }
        }
        plan_ahead(*m);
        etChk(et_stream_create(&m->own_stream));
        apply_attention_state(*m);
        m->host.clear();
        m->host.shrink_to_fit();
        m->finalized = true;
        return ET_OK;
    });
}

int et_model_forward_layer(et_model m, int layer, et_f16 *out, const et_f16 *in, et_stream stream) {
    return guarded([&]() -> int {
        check_layer_index(m, layer);
        et::require(m->finalized, "et_model_forward_layer: call et_model_finalize first");
        et::require(out && in, "et_model_forward_layer: NULL pointer");
        half *o = reinterpret_cast<half *>(out);
        half *i = reinterpret_cast<half *>(const_cast<et_f16 *>(in));
        if (m->desc.mixed) {  // one layer between binary16 buffers: the residual starts from the binary16 input
            etChk(et_f16_to_f32(m->pp32[0]->get(), in, (std::size_t)m->rows() * m->desc.emdim, stream));
            m->layers[(size_t)layer]->forward_mixed(m->layers[(size_t)layer]->buffers(), nullptr, o, m->pp32[0]->get(), i, stream);
        } else {
            run_layer_f16(*m, layer, o, i, false, stream);
        }
        return ET_OK;
    });
}

int et_model_forward(et_model m, et_f16 *out, const et_f16 *in, et_stream stream) {
    return guarded([&]() -> int {
        et::require(m != nullptr && m->finalized, "et_model_forward: call et_model_finalize first");
        et::require(out && in, "et_model_forward: NULL pointer");
        half *o = reinterpret_cast<half *>(out);
        half *i = reinterpret_cast<half *>(const_cast<et_f16 *>(in));
        stream_t s = stream ? stream : m->own_stream;
        if (!m->desc.use_graph) {
            run_layers(*m, o, i, s);
            return ET_OK;
        }
        if (!m->graph || m->graph_in != in || m->graph_out != out) {
            // (Re)capture for this pair of buffers.  An eager pass first runs every kernel once
            // outside capture (lazy one-time kernel setup); its result goes to a buffer of the
            // model's own, so that a caller who normalises in place (out == in) still has the
            // untouched input when the graph runs.
            m->drop_graph();
            run_layers(*m, m->warm->get(), i, s);
            etChk(et_stream_sync(s));
            std::string why;
            if (m->chain && !chain_ran_clean(*m, why)) {
                // a workgroup gave up at a barrier or ran on another XCD than its id says: separate
                // launches from here on (the eager pass is repeated so that its result is valid too)
                m->chain = false;
                et_set_last_error(("et_model_forward: the one-launch chain did not run as it must (" + why +
                                   "); using separate launches").c_str());
                run_layers(*m, m->warm->get(), i, s);
                etChk(et_stream_sync(s));
            }
            etChk(et_graph_begin_capture(s));
            try {
                run_layers(*m, o, i, s);
            } catch (...) {
                et_graph dead = nullptr;
                (void)et_graph_end_capture(s, &dead);
                (void)et_graph_destroy(dead);
                throw;
            }
            etChk(et_graph_end_capture(s, &m->graph));
            m->graph_in = in;
            m->graph_out = out;
        }
        etChk(et_graph_launch(m->graph, s));
        return ET_OK;
    });
}

int et_model_sync(et_model m) {
    return guarded([&]() -> int {
        et::require(m != nullptr, "et_model_sync: NULL handle");
        if (m->own_stream) etChk(et_stream_sync(m->own_stream));
        return ET_OK;
    });
}

int et_model_launches_per_layer(et_model m, int *launches) {
    return guarded([&]() -> int {
        et::require(m != nullptr && launches != nullptr, "et_model_launches_per_layer: NULL argument");
        if (!m->finalized) *launches = 0;
        else if (!m->local.empty()) *launches = m->local_shares.empty() || !m->local_join.empty() ? 2 : 3;
        else *launches = m->chain ? 2 : m->fused_qkv ? 4 : m->split ? 5 : 7;
        return ET_OK;
    });
}

int et_model_load(const char *weights_txt, const char *dir, const et_model_desc *desc, et_model *out) {
    return guarded([&]() -> int {
        et::require(weights_txt && dir && desc && out, "et_model_load: NULL argument");
        int s = et_model_create(desc, out);
        if (s != ET_OK) return s;
        std::unique_ptr<et_model_s> guard(*out);
        *out = nullptr;
        Weights weights(weights_txt, dir);
        // archive names of the exporter (example/npy2pt.py:141-174, example/main.cu:46-90)
        static const char *const mats[4] = {"self_attn.in_proj_.npz", "self_attn.out_proj..npz", "linear1..npz",
                                            "linear2..npz"};
        static const char *const norms[2] = {"norm1..npz", "norm2..npz"};
        for (int l = 0; l < desc->nlayer; l++) {
            const std::string prefix = "transformer_encoder.layers." + std::to_string(l) + ".";
            for (int w = 0; w < 4; w++) {
                const std::string f = prefix + mats[w];
                auto row_ptr = weights.load_mat<int>("row_ptr", f);
                auto column = weights.load_mat<int>("column", f);
                auto data = weights.load_mat<float>("data", f);
                auto bias = weights.load_mat<float>("B", f);
                const Dims d = guard->dims(w);
                et::require((int)row_ptr.size() == d.out / 16 + 1 && (int)bias.size() == d.out &&
                                data.size() == column.size() * 256,
                            "et_model_load: an archive does not match the model dimensions");
                etChk(et_model_set_bsr16(guard.get(), l, w, row_ptr.data(), column.data(), data.data(),
                                         (int)column.size(), bias.data()));
            }
            for (int k = 0; k < 2; k++) {
                const std::string f = prefix + norms[k];
                auto g = weights.load_mat<float>("W", f);
                auto b = weights.load_mat<float>("B", f);
                et::require((int)g.size() == desc->emdim && (int)b.size() == desc->emdim,
                            "et_model_load: a LayerNorm archive does not match emdim");
                etChk(et_model_set_norm(guard.get(), l, k, g.data(), b.data()));
            }
        }
        etChk(et_model_finalize(guard.get()));
        *out = guard.release();
        return ET_OK;
    });
}

int et_model_destroy(et_model m) {
    return guarded([&]() -> int {
        if (m) {
            (void)et_device_sync();
            delete m;
        }
        return ET_OK;
    });
}

}  // extern "C"
