// What a C++ program does with the Net, for the tests that drive it over fake_capi.cpp.
#include "../include/otter_hip_int8.h"
#include "../tensor_amd/host/otter_hip.hpp"

using namespace otter;

namespace {
// Layers of the program's own: they launch on the null stream, as the library's documentation says of its passes.
class Doubled : public Layer {
public:
    Doubled() { one_blob_only = support_packing = true; }
    int compute_output_shape(ParamDict&) override { return top_shapes = {bottom_shapes[0]}, 0; }
    int forward(const Tensor& b, Tensor& top, const NetOption&) const override {
        top = Tensor::empty_device(b.sizes(), b.scalar_type());
        if (otter_hip_eltwise_add((const float*)b.device_ptr(), (const float*)b.device_ptr(), (float*)top.device_ptr(),
                                  (size_t)b.numel() * b.elempack(), nullptr))
            return -1;
        return top.mark_device_written(), 0;
    }
    std::string type() const override { return "Doubled"; }
};
class OwnConvolution : public ConvolutionLayer {  // (in the place of the library's)
public:
    int forward(const Tensor& b, Tensor& top, const NetOption& opt) const override {
        Tensor once;
        const int rc = ConvolutionLayer::forward(b, once, opt);
        return rc ? rc : Doubled().forward(once, top, opt);
    }
};
}  // namespace

extern "C" {
void program_register(int own_convolution) {
    register_hip_layers();
    LayerRegistry::AddCreator("Doubled", []() -> Layer* { return new Doubled(); });
    if (own_convolution) LayerRegistry::AddCreator("Convolution", []() -> Layer* { return new OwnConvolution(); });
}
// a pass that is to give `only` alone (lightmode as the net has it), asked for `name`: the number of the expression that it holds, or a
// negative status
long program_extract(void* net, const char* in, const void* x, int c, int h, int w, const char* only, const char* name) {
    Extractor ex = static_cast<Net*>(net)->create_extractor();
    if (ex.input(in, Tensor::from_host(x, {1, c, h, w}, ScalarType::Float))) return -10;
    ex.only({only});
    Tensor t;
    const int rc = ex.extract(name, t, 1);
    if (rc) return rc;
    return t.defined() ? *static_cast<const long*>(t.data_ptr()) : -11;
}
// a layer's pipeline built anew by the program itself
int program_rebuild(void* net, const char* layer) {
    Net* n = static_cast<Net*>(net);
    return n->layer_by_name(layer)->create_pipeline(n->option);
}
}
