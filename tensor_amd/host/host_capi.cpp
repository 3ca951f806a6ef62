// extern "C" facade over the C++ host layer, for hosts that cannot include otter_hip.hpp (the python tests and the
// benchmark drive the Net through it). Options are "key=value;key=value" strings with the reference's own keys.
#include <algorithm>
#include <chrono>
#include <cstring>
#include <memory>
#include <optional>
#include <string>

#include "../../include/otter_hip_int8.h"
#include "otter_file.hpp"
#include "otter_hip.hpp"

using namespace otter;

namespace {
thread_local std::string g_err;
int fail(const std::string& s) {
    g_err = s;
    return -1;
}
LayerOption parse_options(const char* opts) {
    LayerOption lo;
    std::string s(opts ? opts : "");
    size_t pos = 0;
    while (pos < s.size()) {
        size_t e = s.find(';', pos);
        if (e == std::string::npos) e = s.size();
        const std::string kv = s.substr(pos, e - pos);
        const size_t eq = kv.find('=');
        if (eq != std::string::npos) lo[kv.substr(0, eq)] = kv.substr(eq + 1);
        pos = e + 1;
    }
    return lo;
}
// a pass's result, unpacked: what it is, and its values in host memory where the caller has room for them. `unpacked` (or
// null) receives the blob itself first.
void fetched(const Tensor& top, void* out, size_t capacity, int* dtype, int64_t* shape4, Tensor* unpacked = nullptr) {
    const Tensor f = top.dim() == 4 && top.elempack() != 1 ? top.packing(1) : top;
    if (unpacked) *unpacked = f;
    const ScalarType b = base_of(f.scalar_type());
    if (dtype) *dtype = b == ScalarType::Float ? 0 : (b == ScalarType::Byte ? 1 : 2);
    if (shape4)
        for (int i = 0; i < 4; ++i) shape4[i] = i < f.dim() ? f.size(i) : 1;
    if (out) {
        OTTER_CHECK(f.nbytes() <= capacity, "output buffer too small");
        f.download(out);
    }
}
Tensor f32_vec(const float* p, int n) { return Tensor::from_blob(p, {n}, ScalarType::Float); }
}  // namespace

extern "C" {

const char* otter_host_last_error(void) { return g_err.c_str(); }

void* otter_host_net_create(int use_packing_layout, int lightmode) {
    try {
        if (otter_hip_init(0)) {
            g_err = otter_hip_last_error();
            return nullptr;
        }
        Net* n = new Net();
        n->option.use_packing_layout = use_packing_layout != 0;
        n->option.lightmode = lightmode != 0;
        return n;
    } catch (const std::exception& e) {
        g_err = e.what();
        return nullptr;
    }
}

void otter_host_net_destroy(void* net) { delete static_cast<Net*>(net); }

int otter_host_net_add_layer(void* net, const char* options) {
    try {
        static_cast<Net*>(net)->addLayer(parse_options(options));
        return 0;
    } catch (const std::exception& e) {
        return fail(e.what());
    }
}

// initial != 0: CompileMode::Initial (random model + pipelines); else the weights are injected afterwards
int otter_host_net_compile(void* net, int initial) {
    try {
        static_cast<Net*>(net)->compile(initial ? CompileMode::Initial : CompileMode::Inference);
        return 0;
    } catch (const std::exception& e) {
        return fail(e.what());
    }
}

// fills the public members of a ConvolutionLayer exactly as load_model would (Tensor/ConvolutionLayer.cpp:245-296:
// depthwise layers get their blob scales replicated per group) and builds its pipeline
int otter_host_net_set_conv(void* net, const char* layer_name, const int8_t* weight, const float* bias,
                            const float* weight_scales, int n_weight_scales, float in_scale, float top_scale) {
    try {
        Net* n = static_cast<Net*>(net);
        auto* L = dynamic_cast<ConvolutionLayer*>(n->layer_by_name(layer_name));
        if (!L) return fail(std::string("no Convolution layer named ") + layer_name);
        n->invalidate_plan();
        const int K = L->out_channels, C = L->in_channels, g = L->groups;
        L->weight_data = Tensor::from_blob(weight, {K, C / g, L->kernel_height, L->kernel_width}, ScalarType::Byte);
        if (L->bias_term && bias) L->bias_data = f32_vec(bias, K);
        std::vector<float> ws(K);
        for (int i = 0; i < K; ++i) ws[i] = n_weight_scales == 1 ? weight_scales[0] : weight_scales[i];
        L->weight_data_int8_scales = f32_vec(ws.data(), K);
        const bool dw = C == g && g == K;
        std::vector<float> bs(dw ? g : 1, in_scale), ts(dw ? g : 1, top_scale);
        L->bottom_blob_int8_scales = f32_vec(bs.data(), (int)bs.size());
        if (L->int8_scale_term > 100) L->top_blob_int8_scales = f32_vec(ts.data(), (int)ts.size());
        const int rc = L->create_pipeline(n->option);
        if (rc) return fail(std::string("create_pipeline: ") + otter_hip_last_error());
        return 0;
    } catch (const std::exception& e) {
        return fail(e.what());
    }
}

// Calibration aid: while `on`, an int8-output convolution (int8_scale_term > 100) runs as its fp32-output twin
// (int8_scale_term - 100: same weights and input scale, dequantize + activation instead of requantize), so that a
// calibrator can look at the values its output scale has to cover. `on` = 0 restores the layer.
int otter_host_net_conv_fp32_probe(void* net, const char* layer_name, int on) {
    try {
        Net* n = static_cast<Net*>(net);
        auto* L = dynamic_cast<ConvolutionLayer*>(n->layer_by_name(layer_name));
        if (!L) return fail(std::string("no Convolution layer named ") + layer_name);
        if (on && L->int8_scale_term > 100) L->int8_scale_term -= 100;
        else if (!on && L->int8_scale_term > 0 && L->int8_scale_term < 100 && L->top_blob_int8_scales.defined()) L->int8_scale_term += 100;
        else return 0;
        n->changed();
        const int rc = L->create_pipeline(n->option);
        if (rc) return fail(std::string("create_pipeline: ") + otter_hip_last_error());
        return 0;
    } catch (const std::exception& e) {
        return fail(e.what());
    }
}

int otter_host_net_get_scale_in(void* net, const char* layer_name, float* out) {
    auto* L = dynamic_cast<ConvolutionLayer*>(static_cast<Net*>(net)->layer_by_name(layer_name));
    if (!L || !L->scale_in_data.defined()) return fail("no such layer / pipeline not built");
    std::memcpy(out, L->scale_in_data.data_ptr<float>(), sizeof(float) * L->out_channels);
    return 0;
}

int otter_host_net_set_inner_product(void* net, const char* layer_name, const float* weight, const float* bias) {
    try {
        Net* n = static_cast<Net*>(net);
        auto* L = dynamic_cast<InnerProductLayer*>(n->layer_by_name(layer_name));
        if (!L) return fail(std::string("no InnerProduct layer named ") + layer_name);
        n->changed();
        L->weight_data = Tensor::from_blob(weight, {L->out_features, L->in_features}, ScalarType::Float);
        if (L->bias_term && bias) L->bias_data = f32_vec(bias, L->out_features);
        if (L->create_pipeline(n->option)) return fail(std::string("create_pipeline: ") + otter_hip_last_error());
        return 0;
    } catch (const std::exception& e) {
        return fail(e.what());
    }
}

// One pass: input NCHW (fp32 or int8) on the host -> extract(out_name, type 0) -> unpacked host result.
// out_dtype: 0 fp32, 1 int8, 2 int32. repeat > 1 re-runs the pass with the input resident on the device and returns
// the mean seconds per pass in *seconds (device-synchronised around the timed region).
int otter_host_net_run(void* net, const char* in_name, const void* x, int x_is_int8, int n, int c, int h, int w,
                       const char* out_name, void* out, size_t out_capacity_bytes, int* out_dtype, int64_t* out_shape4,
                       int repeat, double* seconds) {
    try {
        Net* N = static_cast<Net*>(net);
        // resident before the timed region
        const Tensor in = Tensor::from_host(x, {n, c, h, w}, x_is_int8 ? ScalarType::Byte : ScalarType::Float);
        Tensor feat;
        auto pass = [&]() -> int {
            Extractor ex = N->create_extractor();
            if (ex.input(in_name, in)) return -1;
            return ex.extract(out_name, feat, 1);
        };
        int rc = pass();
        if (rc) return fail("forward failed with code " + std::to_string(rc) + ": " + otter_hip_last_error());
        if (repeat > 1) {
            otter_hip_stream_synchronize(nullptr);
            const auto t0 = std::chrono::steady_clock::now();
            for (int i = 0; i < repeat; ++i)
                if ((rc = pass())) return fail("forward failed with code " + std::to_string(rc));
            otter_hip_stream_synchronize(nullptr);
            if (seconds) *seconds = std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count() / repeat;
        }
        fetched(feat, out, out_capacity_bytes, out_dtype, out_shape4);
        return 0;
    } catch (const std::exception& e) {
        return fail(e.what());
    }
}

// A session keeps the input resident on the device and runs passes without synchronising, so that a caller can time
// a stream of passes with its own events. out_name may list several blobs separated by commas (the heads of a
// detection network): a pass extracts every one of them from the same Extractor, the fetch returns the last.
struct otter_host_session {
    Net* net;
    std::string in_name;
    std::vector<std::string> out_names;
    Tensor in, out;
    RecordedPasses recorded;
};

void* otter_host_session_create(void* net, const char* in_name, const void* x, int x_is_int8, int n, int c, int h, int w,
                                const char* out_name) {
    try {
        auto* s = new otter_host_session();
        s->net = static_cast<Net*>(net);
        s->in_name = in_name;
        std::string names(out_name);
        for (size_t at = 0, e; at <= names.size(); at = e + 1) {
            e = std::min(names.find(',', at), names.size());
            s->out_names.push_back(names.substr(at, e - at));
        }
        s->in = Tensor::from_host(x, {n, c, h, w}, x_is_int8 ? ScalarType::Byte : ScalarType::Float);
        return s;
    } catch (const std::exception& e) {
        g_err = e.what();
        return nullptr;
    }
}

int otter_host_session_pass(void* session) {
    try {
        auto* s = static_cast<otter_host_session*>(session);
        auto pass = [&](const std::vector<Tensor>&) {
            Extractor ex = s->net->create_extractor();
            Tensor out;
            OTTER_CHECK(!ex.input(s->in_name, s->in), "no such input blob");
            ex.only(s->out_names);
            for (const std::string& name : s->out_names) {
                const int rc = ex.extract(name, out, 1);
                OTTER_CHECK(!rc, "forward failed with code " + std::to_string(rc) + ": " + otter_hip_last_error());
            }
            return out;
        };
        const auto lease = s->recorded.lease(*s->net, "", false, [] { return std::vector<Tensor>(); }, pass);
        if (const Tensor* out = lease.result()) {
            lease.replay();
            s->out = *out;
        } else {
            s->out = pass({});
        }
        return 0;
    } catch (const std::exception& e) {
        return fail(e.what());
    }
}

// copies the last pass's result (unpacked) to the host; returns the number of bytes, or -1
long otter_host_session_fetch(void* session, void* out, size_t capacity) {
    try {
        auto* s = static_cast<otter_host_session*>(session);
        if (!s->out.defined()) return fail("no pass has run");
        fetched(s->out, out, capacity, nullptr, nullptr);
        return (long)s->out.nbytes();
    } catch (const std::exception& e) {
        return fail(e.what());
    }
}

void otter_host_session_destroy(void* session) { delete static_cast<otter_host_session*>(session); }

// function-level mirror checks: quantize_to_int8 -> convolution -> requantize / dequantize on packed host tensors
int otter_host_functional_chain(const float* x, int n, int c, int h, int w, float in_scale, const int8_t* weight, int k,
                                int kh, int kw, int stride, int pad, int groups, const float* scale_in, const float* bias,
                                int int8_out, float top_scale, int act, int32_t* acc_out, void* out) {
    try {
        if (otter_hip_init(0)) return fail(otter_hip_last_error());
        Tensor xin = Tensor::from_blob(x, {n, c, h, w}, ScalarType::Float);
        if (c % 8 == 0) xin = xin.packing(8);
        else if (c % 4 == 0) xin = xin.packing(4);
        Tensor xq = quantize_to_int8(xin, f32_vec(&in_scale, 1), true);
        Tensor wt = Tensor::from_blob(weight, {k, c / groups, kh, kw}, ScalarType::Byte);
        Tensor acc = convolution(xq, wt, Tensor(), Tensor(), {stride, stride}, {pad, pad}, {1, 1}, false, {0, 0}, groups, true);
        Tensor si = f32_vec(scale_in, k), bi = bias ? f32_vec(bias, k) : Tensor();
        Tensor y = int8_out ? requantize_from_int32_to_int8(acc, si, f32_vec(&top_scale, 1), bi, act, Tensor(), true)
                            : dequantize_from_int32(acc, si, bi, true);
        Tensor a1 = acc.elempack() != 1 ? acc.packing(1) : acc;
        if (acc_out) std::memcpy(acc_out, a1.data_ptr(), a1.nbytes());
        Tensor y1 = y.elempack() != 1 ? y.packing(1) : y;
        std::memcpy(out, y1.data_ptr(), y1.nbytes());
        return 0;
    } catch (const std::exception& e) {
        return fail(e.what());
    }
}

// ---------------------------------------------------------------------------------------------------
// model files
// ---------------------------------------------------------------------------------------------------

// Net::load_otter (Tensor/Net.cpp:518-536)
int otter_host_net_load_otter(void* net, const char* path, int initial) {
    try {
        if (static_cast<Net*>(net)->load_otter(path, initial ? CompileMode::Initial : CompileMode::Inference))
            return fail(std::string("cannot read ") + path);
        return 0;
    } catch (const std::exception& e) {
        return fail(e.what());
    }
}

// Net::load_weight (Tensor/Net.cpp:538-586); ncnn != 0: ncnn `.bin`, else Otter's fp32 stream
int otter_host_net_load_weight(void* net, const char* path, int ncnn) {
    try {
        const int rc = static_cast<Net*>(net)->load_weight(path, ncnn ? Net::WeightType::Ncnn : Net::WeightType::Otter);
        return rc ? fail("load_weight returned " + std::to_string(rc) + ": " + otter_hip_last_error()) : 0;
    } catch (const std::exception& e) {
        return fail(e.what());
    }
}

// One line per layer, "type name bottoms tops N C H W" (the logical shape of its first top blob) and for a convolution
// its weights as load_model will ask for them: "... K C groups kh kw bias_term int8_scale_term".
// how many runs of convolution layers went through the chain entry point as one launch, in this process
long otter_host_chain_forward_count(void) { return ConvolutionLayer::chain_forward_count(); }
long otter_host_block_forward_count(void) { return ConvolutionLayer::block_forward_count(); }
// of this process so far: passes recorded, replays, passes that turned out not to be recordable
void otter_host_recording_counts(long counts[3]) {
    const RecordedPasses::Counts c = RecordedPasses::counts();
    counts[0] = c.recorded, counts[1] = c.replayed, counts[2] = c.refused;
}

long otter_host_net_describe(void* net, char* buf, size_t capacity) {
    try {
        const std::string out = static_cast<Net*>(net)->describe();
        if (out.size() + 1 > capacity) return fail("description larger than the buffer");
        std::memcpy(buf, out.c_str(), out.size() + 1);
        return (long)out.size();
    } catch (const std::exception& e) {
        return fail(e.what());
    }
}

// One pass with any number of blobs set beforehand (Extractor::input on each), e.g. a layer's bottoms when a test
// drives a single layer: inputs are NCHW fp32 / int8 on the host, shapes4 holds 4 entries per input. out_dtype and
// out_shape4 are known even where out holds too little (status -1) or is null; the result is then still to be had, once, from
// otter_host_net_eval_fetch on the same thread.
static thread_local Tensor t_eval_result;

int otter_host_net_eval(void* net, int n_inputs, const char* const* in_names, const void* const* in_ptrs,
                        const int* in_is_int8, const int64_t* shapes4, const char* out_name, void* out,
                        size_t out_capacity_bytes, int* out_dtype, int64_t* out_shape4) {
    try {
        Net* N = static_cast<Net*>(net);
        t_eval_result = Tensor();
        std::vector<std::unique_ptr<HostInput>> ins;
        auto sizes = [&](int i) { return std::vector<int64_t>(shapes4 + 4 * i, shapes4 + 4 * i + 4); };
        auto dtype = [&](int i) { return in_is_int8[i] ? ScalarType::Byte : ScalarType::Float; };
        auto pass = [&](const std::vector<Tensor>& blobs, bool light) {
            Extractor ex = N->create_extractor();
            ex.set_lightmode(light);
            for (int i = 0; i < n_inputs; ++i) OTTER_CHECK(!ex.input(in_names[i], blobs[i]), std::string("unknown blob ") + in_names[i]);
            ex.only({out_name});
            Tensor feat;
            const int rc = ex.extract(out_name, feat, 0);
            OTTER_CHECK(!rc, "forward failed with code " + std::to_string(rc) + ": " + otter_hip_last_error());
            return feat;
        };
        // a result that is left to be fetched later has to outlive the next pass: such a pass is not a recorded one
        std::optional<RecordedPasses::Lease> lease;
        if (out) {
            std::string key(out_name);
            for (int i = 0; i < n_inputs; ++i) {
                key += std::string(";") + in_names[i] + (in_is_int8[i] ? ":b" : ":f");
                for (int k = 0; k < 4; ++k) key += "," + std::to_string(shapes4[4 * i + k]);
            }
            lease.emplace(N->recorded().lease(
                *N, key, true,
                [&] {
                    std::vector<Tensor> blobs;
                    for (int i = 0; i < n_inputs; ++i) blobs.push_back(Tensor::empty_device(sizes(i), dtype(i)));
                    return blobs;
                },
                [&](const std::vector<Tensor>& blobs) {
                    const Tensor f = pass(blobs, true);
                    return f.dim() == 4 && f.elempack() != 1 ? f.packing(1) : f;
                }));
        }
        const Tensor* const recorded = lease ? lease->result() : nullptr;
        const bool replay = recorded && recorded->nbytes() <= out_capacity_bytes;
        std::vector<Tensor> blobs;
        for (int i = 0; i < n_inputs; ++i) {
            ins.push_back(replay ? std::make_unique<HostInput>(in_ptrs[i], lease->inputs()[i])
                                 : std::make_unique<HostInput>(in_ptrs[i], sizes(i), dtype(i)));
            blobs.push_back(ins.back()->blob);
        }
        if (replay) lease->replay();
        const Tensor feat = replay ? *recorded : pass(blobs, false);
        fetched(feat, out, out_capacity_bytes, out_dtype, out_shape4, &t_eval_result);
        if (out) {  // the download has waited for the pass
            t_eval_result = Tensor();
            for (auto& in : ins) in->pass_done();
        }
        return 0;
    } catch (const std::exception& e) {
        return fail(e.what());
    }
}

// the result that the last otter_host_net_eval of this thread had no room for
int otter_host_net_eval_fetch(void* out, size_t capacity) {
    try {
        if (!t_eval_result.defined()) return fail("no result is waiting");
        OTTER_CHECK(out && t_eval_result.nbytes() <= capacity, "output buffer too small");
        t_eval_result.download(out);
        t_eval_result = Tensor();
        return 0;
    } catch (const std::exception& e) {
        return fail(e.what());
    }
}

// What OtterLeader::readProject makes of a file, as text: "N <project name>", "G key=value" per file-level
// parameter, then per block "T <name>" and "P key=value" for every option Net::load_otter passes to the layer.
long otter_host_otter_dump(const char* path, char* buf, size_t capacity) {
    try {
        core::OtterLeader leader;
        if (!leader.readProject(path)) return fail("readProject failed");
        std::string out = "N " + leader.getProjectName() + "\n";
        for (const core::Param& p : leader.getParams()) out += "G " + p.type + "=" + p.info + "\n";
        for (size_t i = 0; i < leader.teams_size(); ++i) {
            out += "T " + leader.getTeamName((int)i) + "\n";
            for (const core::Param& p : leader.getTeamParams((int)i)) out += "P " + p.type + "=" + p.info + "\n";
        }
        if (out.size() + 1 > capacity) return fail("dump larger than the buffer");
        std::memcpy(buf, out.c_str(), out.size() + 1);
        return (long)out.size();
    } catch (const std::exception& e) {
        return fail(e.what());
    }
}

// InitializerNcnnFromDataReader over a file: reads `n` tensors of the given shapes (4 entries each, unused trailing
// entries 0) and kinds (0 weight with tag, 1 plain fp32), appends their bytes to `out`, records 0 (fp32) / 1 (int8) /
// -1 (undefined) per tensor in `dtypes`, and reports the bytes left in the file.
long otter_host_ncnn_read(const char* path, int n, const long long* shapes, const int* kinds, int* dtypes,
                          unsigned char* out, size_t capacity, long long* remain) {
    FILE* f = std::fopen(path, "rb");
    if (!f) return fail("cannot open file");
    size_t used = 0;
    try {
        DataReaderFromStdio dr(f);
        InitializerNcnnFromDataReader init(dr);
        for (int i = 0; i < n; ++i) {
            std::vector<int64_t> shape;
            for (int d = 0; d < 4 && shapes[i * 4 + d] > 0; ++d) shape.push_back(shapes[i * 4 + d]);
            Tensor t = init.load(shape, kinds[i]);
            if (!t.defined()) {
                dtypes[i] = -1;
                continue;
            }
            dtypes[i] = t.scalar_type() == ScalarType::Byte ? 1 : 0;
            if (used + t.nbytes() > capacity) {
                std::fclose(f);
                return fail("tensors larger than the buffer");
            }
            std::memcpy(out + used, t.data_ptr(), t.nbytes());
            used += t.nbytes();
        }
        *remain = (long long)dr.remain();
    } catch (const std::exception& e) {
        std::fclose(f);
        return fail(e.what());
    }
    std::fclose(f);
    return (long)used;
}

}  // extern "C"
