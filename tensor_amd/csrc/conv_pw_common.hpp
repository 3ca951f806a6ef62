// What the pointwise kernels with their operands in registers (conv_pw_reg.hip) and the launch of two pointwise layers (conv_pwpw.hip)
// share: buffer loads and stores, the arguments of the epilogues that carry other layers' work.
#pragma once

#include "conv_dw_common.hpp"

namespace ohip {

namespace {

constexpr unsigned PR_OOB = 0x80000000u;  // past any buffer here: a load returns zero, a store is dropped

// the rest of an epilogue that needs more
struct PwFused {
    const float* residual;
    int8_t* twin;
    float twin_scale, twin_half;
    static PwFused of(const Epilogue& ep) { return {ep.residual, ep.twin, ep.twin_scale, ep.twin_half}; }
};
struct PwParts : PwFused {  // JoinArgs::residual1 and the like
    const float* residual1;
    int split;
    short pack0, pack1;
    static PwParts of(const Epilogue& ep) {
        return {PwFused::of(ep), ep.join->residual1, ep.join->res_split, (short)ep.join->res_pack0, (short)ep.join->res_pack1};
    }
    __device__ JoinArgs join() const {
        JoinArgs ja{};
        ja.residual1 = residual1, ja.res_split = split, ja.res_pack0 = pack0, ja.res_pack1 = pack1;
        return ja;
    }
};
struct PwShuffle {  // JoinArgs::other and the like
    const float* other;
    float *sh_out0, *sh_out1;
    int8_t *sh_q0, *sh_q1;
    float twin_scale, twin_half;
    unsigned sh_image;
    short other_pack, other_odd;
    static PwShuffle of(const Epilogue& ep) {
        const JoinArgs& j = *ep.join;
        return {j.other, j.sh_out0, j.sh_out1, j.sh_q0, j.sh_q1, ep.twin_scale, ep.twin_half, (unsigned)j.sh_image, (short)j.other_pack, (short)j.other_odd};
    }
};
// A result that is only ever read quantized, in a Concat and by another layer, is written that way in both places: 2 bytes a value where
// fp32, its quantization and the Concat's pass over it move 10. 64 -> 64 @52x52 b16 with the depthwise layer behind it and their Concat
// 10.4 + 5.5 + 8.6 us, now 6.7 + 4.6; @13x13, where it is launches that count, 3.5 + 3.2 + 3.4 and 3.5 + 3.5.
struct PwSlice {  // JoinArgs::slice and the like
    int8_t *twin, *slice;
    float twin_scale, twin_half, slice_scale, slice_half;
    unsigned octets;
    static PwSlice of(const Epilogue& ep) {
        const JoinArgs& j = *ep.join;
        return {ep.twin, j.slice, ep.twin_scale, ep.twin_half, j.slice_scale, j.slice_half, (unsigned)j.slice_octets};
    }
};
template <int EPI>
struct PwAddOf {
    using Type = NoJoin;
};
template <>
struct PwAddOf<EPI_F32_P4_FUSED> {
    using Type = PwFused;
};
template <>
struct PwAddOf<EPI_F32_SHUFFLE> {
    using Type = PwShuffle;
};
template <>
struct PwAddOf<EPI_F32_SLICE> {
    using Type = PwSlice;
};
template <>
struct PwAddOf<EPI_F32_P4_PARTS> {
    using Type = PwParts;
};
template <int EPI>
using PwAdd = typename PwAddOf<EPI>::Type;

__device__ __forceinline__ __amdgpu_buffer_rsrc_t rsrc(const void* p, unsigned bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, (int)bytes, 0x00020000);
}
__device__ __forceinline__ v4i load16(__amdgpu_buffer_rsrc_t r, unsigned v, unsigned s) {
    return __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(r, (int)v, (int)s, 0));
}
__device__ __forceinline__ v2i load8(__amdgpu_buffer_rsrc_t r, unsigned v, unsigned s) {
    return __builtin_bit_cast(v2i, __builtin_amdgcn_raw_buffer_load_b64(r, (int)v, (int)s, 0));
}
__device__ __forceinline__ void store16(__amdgpu_buffer_rsrc_t r, v4i d, unsigned v, unsigned s) { store_b128_row(d, r, v, s); }
__device__ __forceinline__ void store8(__amdgpu_buffer_rsrc_t r, v2i d, unsigned v, unsigned s) {
    __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(v2u_store, d), r, (int)v, (int)s, 0);
}

}  // namespace

}  // namespace ohip
