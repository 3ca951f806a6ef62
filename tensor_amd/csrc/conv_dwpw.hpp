// A depthwise layer with one or two pointwise layers behind it as one launch (conv_dwpw.hip).
#pragma once

#include "common.hpp"

namespace ohip {

size_t dwpw_weight_bytes(int C, int ks);
void dwpw_pack_weights(const int8_t* w, int C, int ks, int8_t* dst);

// gd, ed: the depthwise layer (int8 result); g0, e0: the pointwise layer behind it, with what is to become of its result; g1, e1: the
// pointwise layer that reads its int8 result, the second half of its shuffle or the quantization (twin_scale) of its fp32 one, or null
bool conv_dwpw_applicable(const ConvGeom& gd, const Epilogue& ed, const ConvGeom& g0, const Epilogue& e0, const ConvGeom* g1, const Epilogue* e1);
// whether the launch is faster than the layers by themselves (the pointwise ones as a pair where that is a launch)
bool conv_dwpw_faster(const ConvGeom& gd, const ConvGeom& g0, const Epilogue& e0, const ConvGeom* g1);
// w, so: packed weights and the output scale of every channel of the pointwise layers; sum: the first one's fp32 result in front of a
// second layer, or null; force: 0 = automatic, else groups of 16 pixels of a workgroup (1, 2, 4, 8), + 16 with four waves to it,
// + 32 with staged pixels
hipError_t run_conv_dwpw(const int8_t* x, const int8_t* dw_w, float dw_so, const ConvGeom& gd, const Epilogue& ed, const int8_t* const w[2],
                         const float so[2], void* out, float* sum, const ConvGeom& g0, const Epilogue& e0, const ConvGeom* g1, const Epilogue* e1,
                         int force, hipStream_t stream);

}  // namespace ohip
