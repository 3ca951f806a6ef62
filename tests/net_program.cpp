// What a C++ program does with the Net, for the tests that drive it over fake_capi.cpp.
#include "../include/otter_hip_int8.h"
#include "../tensor_amd/host/otter_hip.hpp"

using namespace otter;

extern "C" {
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
