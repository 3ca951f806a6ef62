// A stand-in for the C ABI that the C++ Net runs on, for tests of the Net without a GPU: every blob holds the number of an expression that
// says what it was computed from ("c3(q(shuffle(c1(x),y))[1])"), so that two ways through a net can be compared, whatever launches
// they take. Launches on a recording's stream are kept and made when it is launched; a convolution that has been destroyed may not be
// launched again. Loaded in front of the library that the host layer names.
#include <algorithm>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <map>
#include <string>
#include <vector>

#include "../include/otter_hip_int8.h"

struct otter_hip_conv {
    otter_hip_conv_desc d;
    std::string name;  // of its weights: their first value
    bool alive = true;
};
struct otter_hip_recording {
    std::vector<std::function<void()>> work;
};

namespace {
std::vector<std::string> g_expr;
std::map<std::string, long> g_number;
std::map<std::string, int> g_set;  // what the test asks for: fake_set
std::map<std::string, long> g_count;
otter_hip_recording* g_open = nullptr;
int g_stream = 0;

long number(const std::string& e) {
    auto it = g_number.find(e);
    if (it != g_number.end()) return it->second;
    g_expr.push_back(e);
    return g_number[e] = (long)g_expr.size() - 1;
}
void put(void* blob, const std::string& e) {
    if (!blob) return;
    const long n = number(e);
    std::memcpy(blob, &n, sizeof n);
}
std::string at(const void* blob) {
    long n;
    std::memcpy(&n, blob, sizeof n);
    return n >= 0 && n < (long)g_expr.size() ? g_expr[n] : "?";
}
int launched(const char* what, void* stream, std::function<void()> f) {
    ++g_count[what];
    if (stream && stream == &g_stream && g_open) g_open->work.push_back(std::move(f));
    else f();
    return 0;
}
// the value of an fp32 blob that an int8 one was quantized from (a convolution does that itself where it is given the fp32 blob)
std::string values(const std::string& e) { return e.compare(0, 2, "q(") == 0 ? e.substr(2, e.size() - 3) : e; }
std::string q(const std::string& e) { return "q(" + e + ")"; }
std::string conv(const otter_hip_conv* c, const std::string& in) {
    ++g_count[c->alive ? c->name : "dead"];
    return c->name + "(" + values(in) + ")";
}
std::string sum(std::string a, std::string b) {
    if (b < a) a.swap(b);
    return "sum(" + a + "," + b + ")";
}
std::string half(const std::string& e, int k) { return "half" + std::to_string(k) + "(" + e + ")"; }
std::string shuffle(const std::string& cat) { return "shuffle(" + cat + ")"; }
std::string cat2(const std::string& a, const std::string& b) { return "cat(" + a + "," + b + ")"; }
// a blob that is written slice by slice: it holds the concatenation once every channel is there
void slice(void* blob, int total, int first, int channels, const std::string& e) {
    static std::map<void*, std::map<int, std::pair<int, std::string>>> open;
    auto& parts = open[blob];
    parts[first] = {channels, e};
    int at = 0;
    std::string all;
    for (const auto& p : parts) {
        if (p.first != at) return;
        at += p.second.first, all += (all.empty() ? "cat(" : ",") + p.second.second;
    }
    if (at == total) put(blob, q(all + ")")), open.erase(blob);
}
int form() { return g_set.count("form") ? g_set["form"] : 3; }
bool on(const char* what) { return !g_set.count(what) || g_set[what]; }
void out_hw(const otter_hip_conv_desc& d, int h, int w, int* oh, int* ow) {
    *oh = (h + 2 * d.pad_h - d.dilation_h * (d.kernel_h - 1) - 1) / d.stride_h + 1;
    *ow = (w + 2 * d.pad_w - d.dilation_w * (d.kernel_w - 1) - 1) / d.stride_w + 1;
}
}  // namespace

extern "C" {
long fake_number(const char* e) { return number(e); }
const char* fake_expr(long n) { return n >= 0 && n < (long)g_expr.size() ? g_expr[n].c_str() : "?"; }
void fake_set(const char* what, int v) { g_set[what] = v; }
long fake_count(const char* what) { return g_count[what]; }

int otter_hip_init(int) { return 0; }
const char* otter_hip_last_error(void) { return "refused"; }
int otter_hip_malloc(void** p, size_t n) { return (g_set["no_memory"] && n > 64) ? *p = nullptr, -2 : (*p = std::calloc(1, n < 8 ? 8 : n), ++g_count["malloc"], 0); }
int otter_hip_free(void* p) { return std::free(p), 0; }
int otter_hip_host_malloc(void** p, size_t n) { return *p = std::malloc(n), 0; }
int otter_hip_host_free(void* p) { return std::free(p), 0; }
int otter_hip_upload(void* d, const void* s, size_t n, void*) { return std::memcpy(d, s, n), 0; }
int otter_hip_download(void* d, const void* s, size_t n, void*) { return std::memcpy(d, s, n), 0; }
int otter_hip_copy(void* d, const void* s, size_t n, void* stream) {
    return launched("copy", stream, [=] { std::memcpy(d, s, n); });
}
int otter_hip_stream_synchronize(void*) { return 0; }

int otter_hip_record_begin(void** stream) {
    if (g_set["no_recording"]) return -3;
    ++g_count["record"];
    g_open = new otter_hip_recording();
    return *stream = &g_stream, 0;
}
int otter_hip_record_end(void*, otter_hip_recording_t** r) {
    if (r) *r = g_open;
    else delete g_open;
    return g_open = nullptr, 0;
}
int otter_hip_record_launch(otter_hip_recording_t* r, void*) {
    ++g_count["replay"];
    for (auto& f : r->work) f();
    return 0;
}
int otter_hip_record_destroy(otter_hip_recording_t* r) { return delete r, 0; }

int otter_hip_conv_create(const otter_hip_conv_desc* d, const int8_t* w, const float*, const float*, float, const float*, int,
                          otter_hip_conv_t** h) {
    if (g_set["no_conv"]) return -2;
    return *h = new otter_hip_conv{*d, "c" + std::to_string((int)w[0])}, 0;
}
int otter_hip_conv_destroy(otter_hip_conv_t* h) { return h->alive = false, 0; }  // (kept: what still names it is to be seen)
int otter_hip_conv_output_shape(const otter_hip_conv_t* h, int ih, int iw, int* oh, int* ow) { return out_hw(h->d, ih, iw, oh, ow), 0; }
int otter_hip_conv_default_out_layout(const otter_hip_conv_t* h) {
    const int k = h->d.out_channels;
    return h->d.out_kind == OTTER_HIP_OUT_F32 ? k % 4 ? OTTER_HIP_F32 : OTTER_HIP_F32_P4 : k % 8 ? OTTER_HIP_I8 : OTTER_HIP_I8_P8;
}
size_t otter_hip_conv_workspace_bytes(const otter_hip_conv_t*, int, int, int, int) { return 0; }
int otter_hip_conv_forward(const otter_hip_conv_t* h, const void* in, int, int, int, int, void* out, int, void*, size_t, void* s) {
    return launched("conv", s, [=] { put(out, conv(h, at(in))); });
}
int otter_hip_conv_forward_twin(const otter_hip_conv_t* h, const void* in, int, int, int, int, void* out, int, void* oq, float, int, void*,
                                size_t, void* s) {
    return launched("twin", s, [=] { const std::string r = conv(h, at(in)); put(out, r), put(oq, q(r)); });
}
int otter_hip_conv_forward_residual(const otter_hip_conv_t* h, const void* in, int, int, int, int, const float* res, void* out, int, void* oq,
                                    float, int, void*, size_t, void* s) {
    return launched("residual", s, [=] { const std::string r = sum(conv(h, at(in)), at(res)); put(out, r), put(oq, q(r)); });
}
int otter_hip_conv_join_launches(const otter_hip_conv_t*, int, int, int, int) { return on("join") ? 1 : 2; }
int otter_hip_conv_forward_shuffle(const otter_hip_conv_t* h, const void* in, int, int, int, int, const float* other, int, int other_odd,
                                   float* first, float* second, int8_t* q0, int8_t* q1, int joined, float, int, void* s) {
    return launched("shuffle", s, [=] {
        const std::string r = conv(h, at(in)), o = at(other), sh = shuffle(other_odd ? cat2(r, o) : cat2(o, r));
        if (joined) put(first, sh), put(q0, q(sh));
        else put(first, half(sh, 0)), put(q0, q(half(sh, 0))), put(second, half(sh, 1)), put(q1, q(half(sh, 1)));
    });
}
int otter_hip_conv_forward_residual_concat(const otter_hip_conv_t* h, const void* in, int, int, int, int, const float* p0, int, int,
                                           const float* p1, int, float* out, int8_t* oq, float, int, void* s) {
    return launched("residual_concat", s, [=] { const std::string r = sum(conv(h, at(in)), cat2(at(p0), at(p1))); put(out, r), put(oq, q(r)); });
}
int otter_hip_conv_pair_launches(const otter_hip_conv_t*, const otter_hip_conv_t*, int, int, int, const otter_hip_conv_tail*, int) { return on("pair") ? 1 : 2; }
int otter_hip_conv_pair_forward(const otter_hip_conv_t* a, const otter_hip_conv_t* b, const void* in, int, int, int, const otter_hip_conv_tail* t,
                                void* out, int, void* s) {
    const otter_hip_conv_tail tail = *t;
    return launched("pair", s, [=] {
        std::string r = conv(a, at(in));
        if (tail.other) {
            const std::string o = at(tail.other), sh = shuffle(tail.other_odd ? cat2(r, o) : cat2(o, r));
            put(tail.first_half, half(sh, 0));
            r = half(sh, 1);
        }
        put(out, conv(b, r));
    });
}
int otter_hip_conv_dwpw_launches(const otter_hip_conv_t*, const otter_hip_conv_t*, int, int, int, const otter_hip_conv_end* e, int) {
    return on(e->next ? "dwpw_next" : "dwpw") ? 1 : 2;
}
int otter_hip_conv_dwpw_forward(const otter_hip_conv_t* d, const otter_hip_conv_t* p, const void* in, int, int, int, const otter_hip_conv_end* e, void* out,
                                int, void* s) {
    const otter_hip_conv_end end = *e;
    return launched(end.next ? "dwpw_next" : "dwpw", s, [=] {
        std::string r = conv(p, conv(d, at(in)));
        if (end.residual) r = sum(r, end.residual1 ? cat2(at(end.residual), at(end.residual1)) : at(end.residual));
        if (end.other) {
            const std::string o = at(end.other), sh = shuffle(end.other_odd ? cat2(r, o) : cat2(o, r));
            if (end.joined) put(end.first_half, sh), put(end.first_half_q, q(sh));
            else put(end.first_half, half(sh, 0)), put(end.second_half, half(sh, 1)), put(end.second_half_q, q(half(sh, 1)));
            r = half(sh, 1);
        } else if (end.next) {
            put(end.sum, r);
        } else {
            put(out, r), put(end.out_q, q(r));
        }
        if (end.next) put(out, conv(end.next, r));
    });
}
int otter_hip_conv_maxpool_launches(const otter_hip_conv_t*, int, int, int, int) { return on("stem_pool") ? 1 : 2; }
int otter_hip_conv_forward_maxpool(const otter_hip_conv_t* h, const void* in, int, int, int, int, float, float* out, int8_t* oq, float, int, void* s) {
    return launched("stem_pool", s, [=] { const std::string r = "maxpool(" + conv(h, at(in)) + ")"; put(out, r), put(oq, q(r)); });
}
int otter_hip_conv_slice_launches(const otter_hip_conv_t*, int, int, int, int, int, int) { return on("slice") ? 1 : 2; }
int otter_hip_conv_forward_slice(const otter_hip_conv_t* h, const void* in, int, int, int, int, int8_t* twin, float, int, int8_t* blob, int total, int first,
                                 float, int, void* s) {
    return launched("slice", s, [=] { const std::string r = conv(h, at(in)); put(twin, q(r)), slice(blob, total, first, h->d.out_channels, r); });
}
int otter_hip_upsample2d(const float* src, int, int, int, int, int, int, int, int, int, float* dst, int, void* s) {
    return launched("upsample", s, [=] { put(dst, "up(" + at(src) + ")"); });
}
int otter_hip_upsample2d_slice_launches(int, int, int, int, int, int, int, int, int) { return on("slice") ? 1 : 2; }
int otter_hip_upsample2d_slice(const float* src, int, int, int c, int, int, int, int, int, int, int8_t* blob, int total, int first, float, int, void* s) {
    return launched("slice", s, [=] { slice(blob, total, first, c, "up(" + at(src) + ")"); });
}
int otter_hip_conv_avgpool_launches(const otter_hip_conv_t*, int, int, int, int) { return on("avgpool") ? 1 : 2; }
int otter_hip_conv_forward_avgpool(const otter_hip_conv_t* h, const void* in, int, int, int, int, float* out, void*, size_t, void* s) {
    return launched("avgpool", s, [=] { put(out, "mean(" + conv(h, at(in)) + ")"); });
}
int otter_hip_conv_chain_launches(const otter_hip_conv_t* const*, int n, int, int, int) { return on("chain") ? 1 : n; }
size_t otter_hip_conv_chain_workspace_bytes(const otter_hip_conv_t* const*, int, int, int, int) { return 0; }
int otter_hip_conv_chain_forward(const otter_hip_conv_t* const* hs, int n, const void* in, int, int, int, void* out, void*, size_t, void* s) {
    const std::vector<const otter_hip_conv_t*> all(hs, hs + n);
    return launched("chain", s, [=] {
        std::string r = at(in);
        for (const auto* h : all) r = conv(h, r);
        put(out, r);
    });
}
int otter_hip_conv_chain_status(int* gave_up) { return *gave_up = 0, 0; }
int otter_hip_conv_chain_set_min_tiles(int) { return 96; }
int otter_hip_conv_block_set_always(int) { return 0; }
int otter_hip_conv_block_set_pair(int) { return 0; }
int otter_hip_conv_block_fastest(const otter_hip_conv_t*, const otter_hip_conv_t*, const otter_hip_conv_t*, int, int, int) { return form(); }
size_t otter_hip_conv_block_form_workspace_bytes(const otter_hip_conv_t*, const otter_hip_conv_t*, const otter_hip_conv_t*, int, int, int, int) {
    return (size_t)g_set["block_workspace"];
}
int otter_hip_conv_block_forward_form(const otter_hip_conv_t* e, const otter_hip_conv_t* d, const otter_hip_conv_t* p, int, const void* in, int,
                                      int, int, const float* res, void* out, int, void* oq, float, int, void*, size_t, void* s) {
    return launched("block", s, [=] {
        std::string r = conv(p, conv(d, conv(e, at(in))));
        if (res) r = sum(r, at(res));
        put(out, r), put(oq, q(r));
    });
}
int otter_hip_repack(const void* src, int, int, int, int, int, void* dst, int, void* s) {
    return launched("repack", s, [=] { put(dst, at(src)); });
}
int otter_hip_eltwise_add(const float* a, const float* b, float* out, size_t, void* s) {
    return launched("add", s, [=] { put(out, sum(at(a), at(b))); });
}
int otter_hip_eltwise_add_quantize(const float* a, const float* b, int, int, int, int, int, float, int, float* out, int8_t* oq, void* s) {
    return launched("add", s, [=] { const std::string r = sum(at(a), at(b)); put(out, r), put(oq, q(r)); });
}
int otter_hip_activation(float* x, size_t, int act, float, void* s) {
    return launched("activation", s, [=] { put(x, "act" + std::to_string(act) + "(" + at(x) + ")"); });
}
int otter_hip_global_avgpool(const float* x, int, int, int, int, int, float* out, void* s) {
    return launched("mean", s, [=] { put(out, "mean(" + at(x) + ")"); });
}
int otter_hip_inner_product(const float* x, int, int, const float* w, const float*, int, float* y, void* s) {
    return launched("inner_product", s, [=] { put(y, "fc" + std::to_string((int)w[0]) + "(" + at(x) + ")"); });
}
int otter_hip_concat_channels(const float* const* src, const int*, const int*, int n, float* dst, int, int, int, int, int8_t* oq, float, int, void* s) {
    const std::vector<const float*> all(src, src + n);
    return launched("concat", s, [=] {
        std::string r;
        for (const float* b : all) r += (r.empty() ? "cat(" : ",") + at(b);
        put(dst, r + ")"), put(oq, q(r + ")"));
    });
}
int otter_hip_channel_shuffle(const float* x, int, float* out, int, int, int, int, int, int, void* s) {
    return launched("channel_shuffle", s, [=] { put(out, shuffle(at(x))); });
}
int otter_hip_channel_shuffle_quantize(const float* x, int, float* out, int, int, int, int, int, int, int8_t* oq, float, int, void* s) {
    return launched("channel_shuffle", s, [=] { put(out, shuffle(at(x))), put(oq, q(shuffle(at(x)))); });
}
int otter_hip_shuffle2_split(const float* a, int, const float* b, int, int, int, int, int, float* lo, float* hi, int8_t* oq, float, int, void* s) {
    return launched("split", s, [=] {
        const std::string sh = shuffle(cat2(at(a), at(b)));
        put(lo, half(sh, 0)), put(hi, half(sh, 1)), put(oq, q(half(sh, 1)));
    });
}
int otter_hip_maxpool2d(const float* src, int, int, int, int, int, int, int, int, int, int, int, int, int, int, int, float, float* dst, int, void* s) {
    return launched("maxpool", s, [=] { put(dst, "maxpool(" + at(src) + ")"); });
}
// (the Crop layers of the tests take one half of their input)
int otter_hip_copy_channels(const float* src, int, int, int c0, float* dst, int, int, int, int, int, int, int, void* s) {
    return launched("crop", s, [=] { put(dst, half(at(src), c0 ? 1 : 0)); });
}
}
