// Shared device/host helpers of the gfx950 int8 convolution library.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>
#include <utility>

#include "../../include/otter_hip_int8.h"

namespace ohip {

// The stream of this thread's last launch, unless it has waited for that stream in a call of the library since (otter_hip_download chooses by
// it how it copies).
struct LaunchedOn {
    bool any = false;
    hipStream_t stream = nullptr;
    void set(hipStream_t s) { any = true, stream = s; }
    void waited_for(hipStream_t s) { any = any && stream != s; }
    bool is(hipStream_t s) const { return any && stream == s; }
};
inline thread_local LaunchedOn t_launched;

// A launch without the call configuration that the <<<>>> form pushes and pops: 0.05 to 0.2 us of the host's time less (112 bytes of arguments,
// 4000 in a row: 2.48 -> 2.43 us in one process, 3.90 -> 3.73 in another). The error, if any, is there for hipGetLastError; launched
// returns it.
template <typename... P, typename... A>
inline hipError_t launched(void (*kernel)(P...), dim3 grid, dim3 block, size_t lds, hipStream_t stream, A&&... args) {
    static_assert(sizeof...(P) == sizeof...(A), "one argument for each parameter");
    return [&](P... p) {
        void* ptrs[] = {const_cast<void*>(static_cast<const void*>(&p))...};
        t_launched.set(stream);
        return hipLaunchKernel(reinterpret_cast<const void*>(kernel), grid, block, ptrs, lds, stream);
    }(std::forward<A>(args)...);
}
template <typename... P, typename... A>
inline void launch(void (*kernel)(P...), dim3 grid, dim3 block, size_t lds, hipStream_t stream, A&&... args) {
    (void)launched(kernel, grid, block, lds, stream, std::forward<A>(args)...);
}

// ---------------------------------------------------------------------------------------------------
// layouts
// ---------------------------------------------------------------------------------------------------
__host__ __device__ inline int layout_pack(int layout) {
    switch (layout) {
    case OTTER_HIP_F32_P4:
    case OTTER_HIP_I32_P4:
        return 4;
    case OTTER_HIP_F32_P8:
    case OTTER_HIP_I8_P8:
    case OTTER_HIP_I32_P8:
        return 8;
    default:
        return 1;
    }
}

// 0 = f32, 1 = i8, 2 = i32
__host__ __device__ inline int layout_elem(int layout) {
    if (layout <= OTTER_HIP_F32_P8) return 0;
    if (layout <= OTTER_HIP_I8_P8) return 1;
    return 2;
}

__host__ __device__ inline int layout_elem_bytes(int layout) { return layout_elem(layout) == 1 ? 1 : 4; }

// element offset of (n, c, pix) in a tensor [N, C/p, HW, p]
__host__ __device__ inline size_t elem_offset(int p, int n, int c, int pix, int C, int HW) {
    return (((size_t)n * (C / p) + (c / p)) * HW + pix) * p + (c % p);
}

// ---------------------------------------------------------------------------------------------------
// epilogue arithmetic: bit-for-bit what the reference's x86 build evaluates
// ---------------------------------------------------------------------------------------------------

// float2int8_sse (Tensor/VecIntrinsic.hpp:71-95): trunc(v + copysign(0.5f, v)), saturate to [-127,127].
// float2int8 (Tensor/QuantizeX86.cpp:18-23): (int)round(v). Adding the largest float below 0.5 before
// truncating rounds half away from zero exactly for every finite float, so the two primitives differ only
// in the constant.
template <int ROUND>
__device__ __forceinline__ int float2int8(float v) {
    const float half = (ROUND == OTTER_HIP_ROUND_SSE) ? 0.5f : 0.49999997f;
    float adj = __fadd_rn(v, __builtin_copysignf(half, v));
    int i = (int)adj;  // v_cvt_i32_f32: toward zero, saturating
    return min(max(i, -127), 127);
}

__device__ __forceinline__ int float2int8_rt(float v, int round_mode) {
    const float half = (round_mode == OTTER_HIP_ROUND_SSE) ? 0.5f : 0.49999997f;
    float adj = __fadd_rn(v, __builtin_copysignf(half, v));
    int i = (int)adj;
    return min(max(i, -127), 127);
}

// activation_sse (Tensor/QuantizeX86.hpp:72-106) and the Relu / LRelu / Relu6 / Sigmoid layers that follow
// dequantize on the fp32 path (Tensor/ConvolutionLayer.cpp:838-843)
__device__ __forceinline__ float activate(float v, int act, float p0) {
    switch (act) {
    case 1:
        return fmaxf(v, 0.f);
    case 2:
        return v > 0.f ? v : __fmul_rn(v, p0);
    case 3:
        return fminf(fmaxf(v, 0.f), 6.f);
    case 4:
        return 1.f / (1.f + __expf(-v));
    case 5:  // mish: reachable through the standalone requantize only (no option string of the layer selects it)
        return __fmul_rn(v, tanhf(logf(__expf(v) + 1.f)));
    default:
        return v;
    }
}

// v = acc*scale_in (+bias, single rounding: the reference build contracts it to vfmadd)
template <bool BIAS>
__device__ __forceinline__ float dequant(int acc, float si, float b) {
    return BIAS ? __fmaf_rn((float)acc, si, b) : __fmul_rn((float)acc, si);
}

__device__ __forceinline__ float dequant_rt(int acc, float si, float b, bool has_bias) {
    return has_bias ? __fmaf_rn((float)acc, si, b) : __fmul_rn((float)acc, si);
}

__device__ __forceinline__ int requant_rt(int acc, float si, float b, bool has_bias, int act, float p0, float so,
                                          int round_mode) {
    float v = dequant_rt(acc, si, b, has_bias);
    v = activate(v, act, p0);
    v = __fmul_rn(v, so);
    return float2int8_rt(v, round_mode);
}

// ---------------------------------------------------------------------------------------------------
// epilogue parameters shared by every convolution kernel
// ---------------------------------------------------------------------------------------------------
struct Epilogue {
    const float* scale_in;   // [Kpad]
    const float* bias;       // [Kpad] or nullptr
    const float* scale_out;  // [Kpad] (broadcast on the host when one value was given)
    int act;
    float act_p0;
    int round_mode;
    int out_kind;    // otter_hip_out_kind
    int out_layout;  // otter_hip_layout
    // fast epilogues (activation none / ReLU / clip[0,6] as one clamp, rounding mode as one constant)
    float act_lo, act_hi;  // v = min(max(v, act_lo), act_hi)
    float round_half;      // 0.5f (ROUND_SSE) or 0.49999997f (ROUND_EXACT)
    bool so_positive;      // every output scale is finite and > 0 (lets the int8 epilogue clamp after rounding)
    bool lrelu;            // LeakyReLU with a slope in [0, 1]: v = max(v, v * act_p0), applied by the fast epilogues
    bool so_full = false;  // so_positive, and the activation's upper end is no tighter than int8's: every upper clamp is 127
    float so_one = 0.f;    // the output scale of every channel, 0 where they differ (host side; with so_full in what was padding)
    // fp32 output only: also write the Byte8 quantization of the result, q = float2int8(v * twin_scale), for an int8
    // convolution that reads this blob next (null: no twin). Honoured by the implicit-GEMM Float4 epilogue.
    int8_t* twin = nullptr;
    float twin_scale = 0.f, twin_half = 0.5f;
    // fp32 output only: a blob in the output's layout that is added to the activated result (the Eltwise sum of a
    // residual block; null: none). The twin, if any, is the quantization of the sum. Float4 epilogue only.
    const float* residual = nullptr;
    // host side only: what the EPI_F32_SHUFFLE and EPI_F32_P4_PARTS instances take beside this struct (null: neither)
    const struct JoinArgs* join = nullptr;
    bool fused() const { return twin != nullptr || residual != nullptr || join != nullptr; }
};

// Other layers' work in the epilogue of a Float4 layer (K % 8 == 0). An argument of its own: with it inside Epilogue every launch
// of the library carried 100 to 300 bytes more of arguments, 0.1 us each.
struct JoinArgs {
    // The addend is a concatenation that nobody else reads: channels below res_split come from Epilogue::residual, the rest from
    // residual1, each Float4 or Float8; res_split is a multiple of 8.
    const float* residual1 = nullptr;
    int res_split = 0, res_pack0 = 4, res_pack1 = 4;
    // The layer is one half of Concat -> ChannelShuffle(2) and writes the shuffled blob, its channels alternating with those of
    // `other` (K channels too, Float4 or Float8: other_pack; null: no shuffle). The 2 K channels are two halves of K, each an fp32
    // blob sh_out and a Byte8 blob sh_q (quantized with twin_scale), null where not wanted; sh_image: elements from one image to
    // the next in all four.
    int other_pack = 0;
    const float* other = nullptr;
    bool other_odd = false;  // `other` takes the odd channels of the shuffled blob, else the even ones
    float *sh_out0 = nullptr, *sh_out1 = nullptr;
    int8_t *sh_q0 = nullptr, *sh_q1 = nullptr;
    size_t sh_image = 0;
    // The result is a slice of a Byte8 blob of slice_octets octets, quantized with slice_scale (null: none); Epilogue::twin then is a blob of
    // its own with the same result quantized with twin_scale, or null, and there is no fp32 blob
    int8_t* slice = nullptr;
    int slice_octets = 0;
    float slice_scale = 0.f, slice_half = 0.f;
    int sh_pack0 = 8;  // channels of an element of sh_out0: 8, or 4 (the launch behind a depthwise layer only)
};

// which epilogue code a kernel instance carries
enum {
    EPI_GENERIC = 0,
    EPI_I8_P8 = 1,
    EPI_F32_P4 = 2,
    EPI_I8_P8_NONNEG = 3,
    EPI_F32_P8 = 4,       // depthwise only
    EPI_F32_P4_FUSED = 5,  // implicit GEMM only: EPI_F32_P4 plus the residual addend and / or the int8 twin
    EPI_F32_SHUFFLE = 6,   // the same kernels: the channels interleaved with another blob's (JoinArgs::other)
    EPI_F32_P4_PARTS = 7,  // EPI_F32_P4_FUSED with the addend in two parts (JoinArgs::residual1)
    EPI_F32_SLICE = 8,     // the pointwise register kernels and the depthwise matrix-core kernel: the quantized result in a slice of a blob (JoinArgs::slice)
    EPI_I8_P8_FULL = 9     // EPI_I8_P8_NONNEG with every upper clamp at 127 (Epilogue::so_full), see quant4_full; its instances take doubled output scales
};
constexpr bool epi_is_i8(int epi) { return epi == EPI_I8_P8 || epi == EPI_I8_P8_NONNEG || epi == EPI_I8_P8_FULL; }
// how an int8 epilogue ends: 0 = the int8 range alone, 1 = clamped to [0, its channel's upper clamp], 2 = to [0, 127]
constexpr int epi_clamp(int epi) { return epi == EPI_I8_P8_FULL ? 2 : epi == EPI_I8_P8_NONNEG ? 1 : 0; }

// the argument that an instance takes for them
struct NoJoin {
    static NoJoin of(const Epilogue&) { return {}; }
};
struct WithJoin : JoinArgs {
    static WithJoin of(const Epilogue& ep) { return {*ep.join}; }
};
template <int EPI>
struct JoinOf {
    using Type = NoJoin;
};
template <>
struct JoinOf<EPI_F32_SHUFFLE> {
    using Type = WithJoin;
};
template <>
struct JoinOf<EPI_F32_P4_PARTS> {
    using Type = WithJoin;
};
template <int EPI>
using JoinParam = typename JoinOf<EPI>::Type;

// What a kernel instance reads of Epilogue, as its argument: 32 to 56 bytes instead of 112. A launch costs the host 0.1 us more for
// every 32 bytes of arguments.
// (A kernel's parameter type names an instance by its template argument, not by an expression of the EPI_ constants: their enum has no
// name, and the host's and the device's symbols would number it differently.)
struct EpiBase {
    const float *scale_in, *bias;
    float act_p0, act_lo, act_hi;
    int lrelu;
};
struct EpiI8 : EpiBase {
    const float* scale_out;
    float round_half;
};
struct EpiTwin : EpiBase {
    float twin_scale, twin_half;
};
struct EpiFused : EpiTwin {
    const float* residual;
    int8_t* twin;
};
template <int EPI>
struct EpiArgs {
    static constexpr bool I8 = epi_is_i8(EPI), FUSED = EPI == EPI_F32_P4_FUSED || EPI == EPI_F32_P4_PARTS;
    std::conditional_t<I8, EpiI8, std::conditional_t<FUSED, EpiFused, std::conditional_t<EPI == EPI_F32_SHUFFLE, EpiTwin, EpiBase>>> a;
    static EpiArgs of(const Epilogue& ep) {
        EpiArgs r{};
        r.a.scale_in = ep.scale_in, r.a.bias = ep.bias, r.a.act_p0 = ep.act_p0, r.a.act_lo = ep.act_lo, r.a.act_hi = ep.act_hi;
        r.a.lrelu = ep.lrelu;
        if constexpr (I8) r.a.scale_out = ep.scale_out, r.a.round_half = ep.round_half;
        if constexpr (FUSED || EPI == EPI_F32_SHUFFLE) r.a.twin_scale = ep.twin_scale, r.a.twin_half = ep.twin_half;
        if constexpr (FUSED) r.a.residual = ep.residual, r.a.twin = ep.twin;
        return r;
    }
    __device__ Epilogue epilogue() const {
        Epilogue ep{};
        ep.scale_in = a.scale_in, ep.bias = a.bias, ep.act_p0 = a.act_p0, ep.act_lo = a.act_lo, ep.act_hi = a.act_hi;
        ep.lrelu = a.lrelu != 0;
        if constexpr (I8) ep.scale_out = a.scale_out, ep.round_half = a.round_half;
        if constexpr (FUSED || EPI == EPI_F32_SHUFFLE) ep.twin_scale = a.twin_scale, ep.twin_half = a.twin_half;
        if constexpr (FUSED) ep.residual = a.residual, ep.twin = a.twin;
        return ep;
    }
};
template <>
struct EpiArgs<EPI_GENERIC> {
    Epilogue ep;
    static EpiArgs of(const Epilogue& ep) { return {ep}; }
    __device__ Epilogue epilogue() const { return ep; }
};

// The fast epilogues need: activation in {none, ReLU, clip, LeakyReLU with a slope in [0, 1]}, and (I8_P8) int8
// output in Byte8 with K % 8 == 0 or (F32_P4) fp32 output in Float4 with K % 4 == 0.
// LeakyReLU there is v = max(v, v * slope): equal to (v > 0 ? v : v * slope) for every v when 0 <= slope <= 1.
__host__ inline int pick_epilogue(const Epilogue& ep, int K) {
    const bool clamp_act = ep.act == 0 || ep.act == 1 || ep.act == 3 || (ep.act == 2 && ep.lrelu);
    if (clamp_act && ep.out_kind == OTTER_HIP_OUT_I8 && ep.out_layout == OTTER_HIP_I8_P8 && K % 8 == 0) {
        if (ep.act == 0 || ep.act == 2) return EPI_I8_P8;  // signed result: no clamp but the int8 range
        // after ReLU / clip the value to round is never negative; the fast path needs positive output scales
        return ep.so_positive ? EPI_I8_P8_NONNEG : EPI_GENERIC;
    }
    if (clamp_act && ep.out_kind == OTTER_HIP_OUT_F32 && ep.out_layout == OTTER_HIP_F32_P4 && K % 4 == 0) return EPI_F32_P4;
    return EPI_GENERIC;
}

// the instance to launch for an epilogue code of pick_epilogue, in kernels that have one for EPI_I8_P8_FULL
__host__ inline int full_epilogue(int epi, const Epilogue& ep) { return epi == EPI_I8_P8_NONNEG && ep.so_full ? (int)EPI_I8_P8_FULL : epi; }

struct ConvGeom {
    int N, C, H, W;        // input
    int K, OH, OW;         // output
    int kh, kw, sh, sw, ph, pw, dh, dw;
    int groups;
    // channels per image of the tensors in memory, when the kernel works on a channel slice of them (one group of a
    // grouped convolution: C, K are the group's, Cs, Ks the tensors'); 0 = the same as C / K
    int Cs = 0, Ks = 0;
    // implicit-GEMM kernel only: kernel taps that share one 64-deep reduction step (2 for at most 32 input channels, 4 for
    // at most 16; the weights are packed to match, igemm_tap_pack); 0 or 1 = a step is one tap x 64 channels
    int tap_pack = 0;
};

// ---------------------------------------------------------------------------------------------------
// Shared tail of the MFMA and depthwise kernels: one lane holds the int32 accumulators of 8 consecutive
// output channels ch0..ch0+7 (ch0 % 8 == 0) of one output pixel; apply the epilogue and store them in the
// requested layout. si/bi/so are the per-channel scale_in / bias / scale_out of those 8 channels.
// ---------------------------------------------------------------------------------------------------
typedef int ohip_v4i __attribute__((ext_vector_type(4)));
typedef int ohip_v2i __attribute__((ext_vector_type(2)));

__device__ __forceinline__ void epilogue_store8(void* __restrict__ out, const Epilogue& ep, int n, int ch0, int pix,
                                                int K, int OHW, const int (&a8)[8], const float (&si)[8],
                                                const float (&bi)[8], const float (&so)[8]) {
    const int out_pack = layout_pack(ep.out_layout);
    const bool has_bias = ep.bias != nullptr;
    if (ep.out_kind == OTTER_HIP_OUT_I8) {
        int q[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            float v = dequant_rt(a8[e], si[e], bi[e], has_bias);
            v = activate(v, ep.act, ep.act_p0);
            q[e] = float2int8_rt(__fmul_rn(v, so[e]), ep.round_mode);
        }
        int8_t* o = (int8_t*)out;
        if (out_pack == 8) {
            ohip_v2i pk;
            pk[0] = (q[0] & 0xff) | ((q[1] & 0xff) << 8) | ((q[2] & 0xff) << 16) | ((q[3] & 0xff) << 24);
            pk[1] = (q[4] & 0xff) | ((q[5] & 0xff) << 8) | ((q[6] & 0xff) << 16) | ((q[7] & 0xff) << 24);
            *reinterpret_cast<ohip_v2i*>(o + elem_offset(8, n, ch0, pix, K, OHW)) = pk;
        } else {
#pragma unroll
            for (int e = 0; e < 8; ++e)
                if (ch0 + e < K) o[elem_offset(1, n, ch0 + e, pix, K, OHW)] = (int8_t)q[e];
        }
    } else {
        int r8[8];
        if (ep.out_kind == OTTER_HIP_OUT_F32) {
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                float v = dequant_rt(a8[e], si[e], bi[e], has_bias);
                r8[e] = __float_as_int(activate(v, ep.act, ep.act_p0));
            }
        } else {
#pragma unroll
            for (int e = 0; e < 8; ++e) r8[e] = a8[e];
        }
        int* o = (int*)out;
        if (out_pack == 8) {
            int* p = o + elem_offset(8, n, ch0, pix, K, OHW);
            *reinterpret_cast<ohip_v4i*>(p) = ohip_v4i{r8[0], r8[1], r8[2], r8[3]};
            *reinterpret_cast<ohip_v4i*>(p + 4) = ohip_v4i{r8[4], r8[5], r8[6], r8[7]};
        } else if (out_pack == 4) {
            *reinterpret_cast<ohip_v4i*>(o + elem_offset(4, n, ch0, pix, K, OHW)) =
                ohip_v4i{r8[0], r8[1], r8[2], r8[3]};
            if (ch0 + 4 < K)
                *reinterpret_cast<ohip_v4i*>(o + elem_offset(4, n, ch0 + 4, pix, K, OHW)) =
                    ohip_v4i{r8[4], r8[5], r8[6], r8[7]};
        } else {
#pragma unroll
            for (int e = 0; e < 8; ++e)
                if (ch0 + e < K) o[elem_offset(1, n, ch0 + e, pix, K, OHW)] = r8[e];
        }
    }
}

// Out-of-line copy of the generic tail: keeps the kernels that carry it small (it is the slow path anyway).
__device__ __noinline__ void epilogue_store8_generic(void* __restrict__ out, const Epilogue* ep, int n, int ch0, int pix,
                                                     int K, int OHW, int a0, int a1, int a2, int a3, int a4, int a5,
                                                     int a6, int a7) {
    const int a8[8] = {a0, a1, a2, a3, a4, a5, a6, a7};
    float si[8], bi[8], so[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        si[e] = ep->scale_in[ch0 + e];
        bi[e] = ep->bias ? ep->bias[ch0 + e] : 0.f;
        so[e] = ep->scale_out ? ep->scale_out[ch0 + e] : 1.f;
    }
    epilogue_store8(out, *ep, n, ch0, pix, K, OHW, a8, si, bi, so);
}

// Per-lane epilogue constants of 8 consecutive channels for the fast paths. `bias` always points at an array
// (filled with -0.0f when the layer has no bias: fma(a, s, -0.0f) == a * s bit for bit, sign of zero included).
struct Epi8 {
    float si[8], bi[8], so[8];
    unsigned qh[4];  // upper clamp of the rounded result per channel, as packed int16 pairs (epi8_clamp_init)
};

__device__ __forceinline__ void epi8_clamp_init(const Epilogue& ep, Epi8& p);

template <int EPI>
__device__ __forceinline__ void epi8_load(Epi8& p, const Epilogue& ep, int ch0) {
    const ohip_v4i* s = reinterpret_cast<const ohip_v4i*>(ep.scale_in + ch0);
    const ohip_v4i* b = reinterpret_cast<const ohip_v4i*>(ep.bias + ch0);
    ohip_v4i s0 = s[0], s1 = s[1], b0 = b[0], b1 = b[1];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        p.si[e] = __int_as_float(s0[e]);
        p.si[4 + e] = __int_as_float(s1[e]);
        p.bi[e] = __int_as_float(b0[e]);
        p.bi[4 + e] = __int_as_float(b1[e]);
    }
    if constexpr (epi_is_i8(EPI)) {
        const ohip_v4i* o = reinterpret_cast<const ohip_v4i*>(ep.scale_out + ch0);
        ohip_v4i o0 = o[0], o1 = o[1];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            p.so[e] = __int_as_float(o0[e]);
            p.so[4 + e] = __int_as_float(o1[e]);
        }
        if constexpr (EPI == EPI_I8_P8_NONNEG) epi8_clamp_init(ep, p);
        if constexpr (EPI == EPI_I8_P8_FULL)
#pragma unroll
            for (int e = 0; e < 8; ++e) p.so[e] += p.so[e];
    }
}

// requantize 8 channels and store one Byte8 element.
// NONNEG (ReLU / clip [0, hi], output scales > 0): the clamp is applied AFTER scaling and rounding, on the packed
// int16 values, instead of on the float before them. x -> trunc(fl(fl(x * so) + half)) is monotone for so > 0, so
// clamping its argument to [0, hi] equals clamping its result to [trunc(0 + half), trunc(fl(fl(hi * so) + half))]
// = [0, qh], bit for bit; qh (capped at the int8 saturation bound 127) is computed once per channel octet by
// epi8_clamp_init. Without an activation (!NONNEG) there is nothing to clamp but the int8 range.
typedef short ohip_v2s __attribute__((ext_vector_type(2)));

// the clamp of one channel pair, as epi8_clamp_init packs it (for kernels that keep the clamps of a row block in LDS)
__device__ __forceinline__ unsigned epi8_clamp_pair(const Epilogue& ep, float so0, float so1) {
    const int q0 = min((int)__fadd_rn(__fmul_rn(ep.act_hi, so0), ep.round_half), 127);
    const int q1 = min((int)__fadd_rn(__fmul_rn(ep.act_hi, so1), ep.round_half), 127);
    return (unsigned)(q0 & 0xffff) | ((unsigned)q1 << 16);
}

__device__ __forceinline__ void epi8_clamp_init(const Epilogue& ep, Epi8& p) {
#pragma unroll
    for (int h = 0; h < 4; ++h) {
        const int q0 = min((int)__fadd_rn(__fmul_rn(ep.act_hi, p.so[2 * h]), ep.round_half), 127);
        const int q1 = min((int)__fadd_rn(__fmul_rn(ep.act_hi, p.so[2 * h + 1]), ep.round_half), 127);
        p.qh[h] = (unsigned)(q0 & 0xffff) | ((unsigned)q1 << 16);
    }
}

// float -> uint32 toward zero, everything below zero (and NaN) to 0, everything above to 2^32 - 1: v_cvt_u32_f32. (As an
// instruction, not as a C++ conversion: that one is undefined for negative values.)
__device__ __forceinline__ unsigned cvt_u32_floor0(float v) {
    unsigned r;
    asm("v_cvt_u32_f32 %0, %1" : "=v"(r) : "v"(v));
    return r;
}

// LeakyReLU decided at run time: max(v, v * slope) with a slope of 1 where there is none, which is v itself. (A choice per value is two
// instructions more, and it is made per value: the compiler turns a uniform branch around three instructions into a select.)
__device__ __forceinline__ float lrelu_or_not(const Epilogue& ep, float v) { return fmaxf(v, __fmul_rn(v, ep.lrelu ? ep.act_p0 : 1.f)); }

// Four values behind ReLU / clip as the bytes min(max((int)fl(t + half), 0), 127), from t2 = 2 t (exact). v_cvt_pk_u8_f32 converts, saturates to
// [0, 255] and packs in one instruction, but rounds to nearest even; with t doubled that is no matter: fl(2 t + half) rounds to 2 q or 2 q + 1
// wherever fl(t + half) truncates to q (a value that lies between two of them is even below, and there the tie goes), and 255 is 127 with a
// bit behind it. For every float t and both rounding constants: tests/test_requant_full.py goes over them. It takes the place of the
// conversion, two packings with saturation, two minima and a permutation: of four requantized values' 96 cycles of vector issue 17.
// Launches that this bounds take 0.92 of the time (16 -> 96 pointwise + depthwise stride 2 @112x112 b64 26.5 -> 24.5 us).
__device__ __forceinline__ unsigned quant4_full(const float (&t2)[4], float half) {
    unsigned w = 0;
#pragma unroll
    for (int e = 0; e < 4; ++e) w = __builtin_amdgcn_cvt_pk_u8_f32(__fadd_rn(t2[e], half), e, w);
    return w >> 1 & 0x7f7f7f7fu;
}

// requantize 4 channels: their bytes
// CLAMP: as epi_clamp says (2: `so` are the doubled output scales)
// LRELU: 0 = no LeakyReLU, 1 = LeakyReLU, -1 = decided by ep.lrelu at run time
template <int CLAMP, int LRELU = -1>
__device__ __forceinline__ int epi4_quant_i8(const Epilogue& ep, const float* si, const float* bi, const float* so, const unsigned* qh,
                                             int a0, int a1, int a2, int a3) {
    constexpr bool NONNEG = CLAMP != 0;
    const int a[4] = {a0, a1, a2, a3};
    if constexpr (CLAMP == 2) {
        float t2[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) t2[e] = __fmul_rn(__fmaf_rn((float)a[e], si[e], bi[e]), so[e]);
        return (int)quant4_full(t2, ep.round_half);
    }
    int q[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        float v = __fmaf_rn((float)a[e], si[e], bi[e]);
        if constexpr (!NONNEG && LRELU == 1) v = fmaxf(v, __fmul_rn(v, ep.act_p0));
        if constexpr (!NONNEG && LRELU == -1) v = lrelu_or_not(ep, v);
        v = __fmul_rn(v, so[e]);
        float adj = NONNEG ? __fadd_rn(v, ep.round_half) : __fadd_rn(v, __builtin_copysignf(ep.round_half, v));
        // toward zero, saturating. NONNEG: to UNSIGNED, which sends everything below zero to zero: the lower clamp of
        // the activation comes with the conversion, and only the upper one is left for the packed values
        if constexpr (NONNEG) q[e] = (int)cvt_u32_floor0(adj);
        else q[e] = (int)adj;
    }
    // two int32 -> two saturated int16 in one dword, clamp both halves at once, then gather the low bytes
    if constexpr (NONNEG) {
        typedef unsigned short ohip_v2us __attribute__((ext_vector_type(2)));
        ohip_v2us lo = __builtin_bit_cast(ohip_v2us, __builtin_amdgcn_cvt_pk_u16((unsigned)q[0], (unsigned)q[1]));
        ohip_v2us hi = __builtin_bit_cast(ohip_v2us, __builtin_amdgcn_cvt_pk_u16((unsigned)q[2], (unsigned)q[3]));
        lo = __builtin_elementwise_min(lo, __builtin_bit_cast(ohip_v2us, qh[0]));
        hi = __builtin_elementwise_min(hi, __builtin_bit_cast(ohip_v2us, qh[1]));
        return (int)__builtin_amdgcn_perm(__builtin_bit_cast(unsigned, hi), __builtin_bit_cast(unsigned, lo), 0x06040200u);
    } else {
        ohip_v2s lo = __builtin_bit_cast(ohip_v2s, __builtin_amdgcn_cvt_pk_i16(q[0], q[1]));
        ohip_v2s hi = __builtin_bit_cast(ohip_v2s, __builtin_amdgcn_cvt_pk_i16(q[2], q[3]));
        const ohip_v2s top = {127, 127}, bot = {-127, -127};
        lo = __builtin_elementwise_max(__builtin_elementwise_min(lo, top), bot);
        hi = __builtin_elementwise_max(__builtin_elementwise_min(hi, top), bot);
        return (int)__builtin_amdgcn_perm(__builtin_bit_cast(unsigned, hi), __builtin_bit_cast(unsigned, lo), 0x06040200u);
    }
}

template <int CLAMP, int LRELU = -1>
__device__ __forceinline__ ohip_v2i epi8_quant_i8p8(const Epilogue& ep, const Epi8& p, const int (&a8)[8]) {
    return ohip_v2i{epi4_quant_i8<CLAMP, LRELU>(ep, p.si, p.bi, p.so, p.qh, a8[0], a8[1], a8[2], a8[3]),
                    epi4_quant_i8<CLAMP, LRELU>(ep, p.si + 4, p.bi + 4, p.so + 4, p.qh + 2, a8[4], a8[5], a8[6], a8[7])};
}

template <int CLAMP>
__device__ __forceinline__ void epi8_store_i8p8(int8_t* __restrict__ out, const Epilogue& ep, const Epi8& p, size_t elem,
                                                const int (&a8)[8]) {
    *reinterpret_cast<ohip_v2i*>(out + elem) = epi8_quant_i8p8<CLAMP>(ep, p, a8);
}

// dequantize 4 channels with the clamp activation (LRELU false) or LeakyReLU (true): the bits of one Float4 element
template <bool LRELU>
__device__ __forceinline__ ohip_v4i epi4_dequant_f32p4(const Epilogue& ep, const float* si, const float* bi, int a0, int a1,
                                                       int a2, int a3) {
    const int a[4] = {a0, a1, a2, a3};
    ohip_v4i r;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        float v = __fmaf_rn((float)a[e], si[e], bi[e]);
        if constexpr (LRELU) v = fmaxf(v, __fmul_rn(v, ep.act_p0));
        else v = fminf(fmaxf(v, ep.act_lo), ep.act_hi);
        r[e] = __float_as_int(v);
    }
    return r;
}

// Channels ch0 .. ch0 + 7 of one pixel into the shuffled blob: with the same channels of JoinArgs::other they are its
// channels 2 ch0 .. 2 ch0 + 15, two packs of 8 that a lane writes whole (32 bytes fp32, 8 bytes int8 each). Bound by the bytes of
// the two fp32 blobs; the layer's own result is neither written nor read back. Layer and shuffle as two launches / as one, in the
// detection network at batch 16: 88 channels @52x52 23 / 14.5 us, 176 @26x26 15.6 / 10.2 us, 352 @13x13 11.8 / 7.5 us.
template <int LRELU>
__device__ __forceinline__ void epi8_store_shuffle(const Epilogue& ep, const JoinArgs& ja, const float* si, const float* bi, const int (&a8)[8], unsigned n,
                                                   unsigned pix, int ch0, int K, int OHW) {
    const size_t plane = (size_t)OHW * ja.other_pack;
    const float* o = ja.other + ((size_t)n * (unsigned)(K / ja.other_pack) + (unsigned)(ch0 / ja.other_pack)) * plane +
                     (size_t)pix * (unsigned)ja.other_pack;
    const ohip_v4i x0 = *reinterpret_cast<const ohip_v4i*>(o);
    const ohip_v4i x1 = *reinterpret_cast<const ohip_v4i*>(o + (ja.other_pack == 8 ? 4 : plane));
    const ohip_v4i v0 = epi4_dequant_f32p4<LRELU>(ep, si, bi, a8[0], a8[1], a8[2], a8[3]);
    const ohip_v4i v1 = epi4_dequant_f32p4<LRELU>(ep, si + 4, bi + 4, a8[4], a8[5], a8[6], a8[7]);
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const ohip_v4i x = h ? x1 : x0, v = h ? v1 : v0;
        const ohip_v4i even = ja.other_odd ? v : x, odd = ja.other_odd ? x : v;  // wave-uniform
        const int f[8] = {even[0], odd[0], even[1], odd[1], even[2], odd[2], even[3], odd[3]};
        const int pack = ch0 / 4 + h, half = K / 8;  // pack of the 2 K channels, packs in each half
        const bool second = pack >= half;
        const size_t e = (size_t)n * ja.sh_image + ((size_t)(unsigned)(second ? pack - half : pack) * (unsigned)OHW + pix) * 8;
        float* out = second ? ja.sh_out1 : ja.sh_out0;
        int8_t* q = second ? ja.sh_q1 : ja.sh_q0;
        if (out != nullptr) {
            const ohip_v4i lo = {f[0], f[1], f[2], f[3]}, hi = {f[4], f[5], f[6], f[7]};
            *reinterpret_cast<ohip_v4i*>(out + e) = lo;
            *reinterpret_cast<ohip_v4i*>(out + e + 4) = hi;
        }
        if (q != nullptr) {
            ohip_v2i pk = {0, 0};
#pragma unroll
            for (int b = 0; b < 8; ++b) {
                const float t = __fmul_rn(__int_as_float(f[b]), ep.twin_scale);
                const int k = (int)__fadd_rn(t, __builtin_copysignf(ep.twin_half, t));
                pk[b / 4] |= (min(max(k, -127), 127) & 0xff) << (8 * (b % 4));
            }
            *reinterpret_cast<ohip_v2i*>(q + e) = pk;
        }
    }
}

// Four channels of one pixel of an addend in two parts (JoinArgs::residual1). Saves the copies that brought the two blobs
// together and into the result's layout, and the pass that added them: 128 channels @52x52, batch 16, concatenation + layer +
// repack + sum 45.6 us as four launches, 14.4 us as one.
__device__ __forceinline__ const float* epi4_residual_at(const Epilogue& ep, const JoinArgs& ja, unsigned n, unsigned pix, int ch, int K, int OHW) {
    const bool second = ch >= ja.res_split;
    const int c = second ? ch - ja.res_split : ch, channels = second ? K - ja.res_split : ja.res_split;
    const int pack = second ? ja.res_pack1 : ja.res_pack0, at = c & (pack - 1);
    return (second ? ja.residual1 : ep.residual) + (size_t)(n * (unsigned)channels + (unsigned)(c - at)) * (unsigned)OHW +
           (size_t)pix * (unsigned)pack + (unsigned)at;
}

// dequantize (+clamp activation) 4 channels and store one Float4 element. FUSED: first add the residual blob's element
// if the epilogue carries one, and return the four bytes of the blob's int8 twin (float2int8(v * twin_scale)) if it
// carries one
// LRELU: 0 = clamp activation only, 1 = LeakyReLU, -1 = decided by ep.lrelu at run time
// res_at: where the residual's element is, if not at `elem` of one blob (epi4_residual_at)
template <bool FUSED = false, int LRELU = -1>
__device__ __forceinline__ unsigned epi4_store_f32p4(float* __restrict__ out, const Epilogue& ep, const float* si,
                                                     const float* bi, size_t elem, int a0, int a1, int a2, int a3,
                                                     const float* res_at = nullptr) {
    const int a[4] = {a0, a1, a2, a3};
    ohip_v4i r;
    unsigned q = 0;
    ohip_v4i res = {0, 0, 0, 0};
    if constexpr (FUSED)
        if (ep.residual != nullptr)  // wave-uniform
            res = *reinterpret_cast<const ohip_v4i*>(res_at != nullptr ? res_at : ep.residual + elem);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        float v = __fmaf_rn((float)a[e], si[e], bi[e]);
        if constexpr (LRELU != 1) v = fminf(fmaxf(v, ep.act_lo), ep.act_hi);  // (open for LeakyReLU)
        if constexpr (LRELU == 1) v = fmaxf(v, __fmul_rn(v, ep.act_p0));
        if constexpr (LRELU == -1) v = lrelu_or_not(ep, v);
        if constexpr (FUSED) {
            if (ep.residual != nullptr) v = __fadd_rn(v, __int_as_float(res[e]));
            if (ep.twin != nullptr) {  // wave-uniform
                const float t = __fmul_rn(v, ep.twin_scale);
                const int k = (int)__fadd_rn(t, __builtin_copysignf(ep.twin_half, t));
                q |= (unsigned)(min(max(k, -127), 127) & 0xff) << (8 * e);
            }
        }
        r[e] = __float_as_int(v);
    }
    if (!FUSED || out != nullptr) *reinterpret_cast<ohip_v4i*>(out + elem) = r;  // (null: the twin alone)
    return q;
}

// float2int8 of four values into the four bytes of a dword (quantize_to_int8)
__device__ __forceinline__ int quantize4(const ohip_v4i& f, float scale, float half) {
    int k[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const float t = __fmul_rn(__int_as_float(f[e]), scale);
        k[e] = (int)__fadd_rn(t, __builtin_copysignf(half, t));  // toward zero, saturating
    }
    const ohip_v2s top = {127, 127}, bot = {-127, -127};
    ohip_v2s a = __builtin_bit_cast(ohip_v2s, __builtin_amdgcn_cvt_pk_i16(k[0], k[1]));
    ohip_v2s b = __builtin_bit_cast(ohip_v2s, __builtin_amdgcn_cvt_pk_i16(k[2], k[3]));
    a = __builtin_elementwise_max(__builtin_elementwise_min(a, top), bot);
    b = __builtin_elementwise_max(__builtin_elementwise_min(b, top), bot);
    return (int)__builtin_amdgcn_perm(__builtin_bit_cast(unsigned, b), __builtin_bit_cast(unsigned, a), 0x06040200u);
}

typedef unsigned ohip_v4u __attribute__((__vector_size__(4 * sizeof(unsigned))));
// A 16-byte buffer store whose row offset sits in a scalar register. The store unit reads the four data registers over
// several cycles, and a vector instruction right behind the store that overwrites one of them can get there first: the
// compiler separates the two behind a store with a constant offset, but takes a scalar-register offset to be safe, which
// on this GPU it is not (seen in the fp32 depthwise epilogue at 16x128x52x52, where the next row's conversion follows the
// store at once: 1 value in 50 000 was the next row's raw accumulator). The data registers are therefore kept live across
// two wait states behind the store.
__device__ __forceinline__ void store_b128_row(ohip_v4i data, __amdgpu_buffer_rsrc_t dst, unsigned v_off, unsigned s_off) {
    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(ohip_v4u, data), dst, (int)v_off, (int)s_off, 0);
    asm volatile("s_nop 1" ::"v"(data) : "memory");
}

// n / d for 0 <= n < 2^31 as a multiplication: with 2^(l-1) < d <= 2^l and m = ceil(2^(31+l) / d) < 2^32 the error m d - 2^(31+l) is
// below 2^l, so that n times it stays below 2^(31+l). (n is doubled, for a product whose upper half begins at bit 31: with m a bit
// longer d = 1 would need a branch, and a kernel's indices are a chain of such divisions.)
struct FastDiv {
    unsigned m, s, d;
};
inline FastDiv fast_div(unsigned d) {
    if (d == 0) d = 1;
    unsigned l = 0;
    while ((1ull << l) < d) ++l;
    return {(unsigned)(((1ull << (31 + l)) + d - 1) / d), l, d};
}
__device__ __forceinline__ unsigned div_by(unsigned n, const FastDiv& f) { return __umulhi(n << 1, f.m) >> f.s; }

}  // namespace ohip
