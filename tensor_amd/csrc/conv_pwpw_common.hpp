// What the launches of two pointwise layers (conv_pwpw.hip) and of a depthwise layer with the pointwise ones behind it (conv_dwpw.hip)
// share: a pointwise layer as the kernels read it, and its epilogues.
#pragma once

#include "conv_igemm.hpp"
#include "conv_pw_common.hpp"

namespace ohip {

namespace {

enum { PP_I8, PP_NONNEG, PP_F32 };  // an int8 result, one behind ReLU / clip, an fp32 one

// one of the two layers, as PwRegArgs has it
struct PwPwLayer {
    const int8_t* w;
    const float *scale_in, *bias;
    float p0, scale, half;
    unsigned qh;
    int K, mt, steps, kind, lrelu;  // (whole words: shorter fields of kernel arguments may come by vector loads)
};

// Eight channels of a pixel as bytes (PP_I8, PP_NONNEG); four as values (PP_F32). (The clamp is open for LeakyReLU.)
// CLAMP: as epi_clamp says (2: PwPwLayer::scale is doubled)
template <int CLAMP>
__device__ __forceinline__ v2i pp_bytes(const Epilogue& ep, const PwPwLayer& l, const float (&si)[8], const float (&bi)[8], const v4i& c0, const v4i& c1) {
    Epi8 prm;
#pragma unroll
    for (int e = 0; e < 8; ++e) prm.si[e] = si[e], prm.bi[e] = bi[e], prm.so[e] = l.scale;
#pragma unroll
    for (int e = 0; e < 4; ++e) prm.qh[e] = l.qh;
    const int a8[8] = {c0[0], c0[1], c0[2], c0[3], c1[0], c1[1], c1[2], c1[3]};
    return epi8_quant_i8p8<CLAMP>(ep, prm, a8);
}
__device__ __forceinline__ v4i pp_values(const Epilogue& ep, const float* si, const float* bi, const v4i& c) {
    v4i r;
#pragma unroll
    for (int e = 0; e < 4; ++e)
        r[e] = __float_as_int(lrelu_or_not(ep, __builtin_amdgcn_fmed3f(__fmaf_rn((float)c[e], si[e], bi[e]), ep.act_lo, ep.act_hi)));
    return r;
}
__device__ __forceinline__ Epilogue pp_epilogue(const PwPwLayer& l) {
    Epilogue ep{};
    ep.act_p0 = l.p0, ep.lrelu = l.lrelu;
    if (l.kind == PP_F32) ep.act_lo = l.scale, ep.act_hi = l.half;
    else ep.round_half = l.half;
    return ep;
}

inline bool pwpw_pointwise(const ConvGeom& g) {
    return g.groups == 1 && g.kh == 1 && g.kw == 1 && g.sh == 1 && g.sw == 1 && g.ph == 0 && g.pw == 0 && g.C % 8 == 0;
}
inline int pwpw_kind(const Epilogue& ep, int K) {
    switch (pick_epilogue(ep, K)) {
    case EPI_I8_P8: return PP_I8;
    case EPI_I8_P8_NONNEG: return PP_NONNEG;
    case EPI_F32_P4: return PP_F32;
    }
    return -1;
}
// g, ep: the layer; w: its packed weights; so: the output scale of every channel
inline PwPwLayer pwpw_layer(const ConvGeom& g, const Epilogue& ep, const int8_t* w, float so) {
    PwPwLayer l{};
    l.w = w, l.scale_in = ep.scale_in, l.bias = ep.bias, l.p0 = ep.act_p0, l.lrelu = ep.lrelu, l.K = g.K;
    l.mt = igemm_padded_rows(g.K) / 16, l.steps = igemm_channel_groups(g.C), l.kind = pwpw_kind(ep, g.K);
    l.scale = l.kind == PP_F32 ? ep.act_lo : so, l.half = l.kind == PP_F32 ? ep.act_hi : ep.round_half;
    const float both[2] = {so, so};
    if (l.kind == PP_NONNEG) conv_pw_stream_clamps(ep.act_hi, ep.round_half, both, 2, &l.qh);
    return l;
}

}  // namespace

}  // namespace ohip
