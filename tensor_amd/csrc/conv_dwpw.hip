// A depthwise k x k layer and the pointwise layer that alone reads its int8 result in one launch, and with them the pointwise layer that
// reads the int8 form of what the first leaves behind, where there is one (conv_pwpw.hip's pair, across a residual sum as well).
//
// What bounds these layers one by one is not bytes and not operations: a launch takes 2 us behind the one in front of it, then a chain of
// memory latencies, and the blob between the layers is written and read back for nothing. Here a workgroup of eight or four waves owns 16 G
// pixels (G = 1, 2, 4, 8 groups of 16, a wave belongs to one) with all their channels:
//  * The depthwise layer goes through the matrix cores, 16 channels x 16 pixels at a time: a B column is one output pixel, its 64
//    reduction bytes are four taps of two channel octets, and the A operand holds each channel's weights at that channel's bytes and
//    zeros elsewhere: 3 instructions for a 3x3 window, 7 for 5x5. (conv_dw_mfma.hip puts eight neighbouring pixels of one octet into a
//    column: half the loads, but runs of four output pixels of a row. Here the pixels are any: no lane idles at the end of a row, and
//    strides, padding and dilation are in the lanes' addresses.) A tap of a pixel is an 8-byte load; one outside the image is out of
//    range and zero. The weights come as one byte per lane and tap and are spread out by v_perm_b32: as whole operands they would be as
//    many bytes as the pixels.
//  * Where the depthwise layer keeps the image's sides, a workgroup may copy the run of pixels that its windows touch into LDS first (plan + 32,
//    DwPwStage), with the weights: a tap is then an LDS read, and the address unit, which takes some 28 cycles for every 8-byte load of
//    scattered pixels, sees a 16-byte copy for two pixels once. What that gives grows with the taps (5x5 128 -> 128 -> 128 @52x52 b16 21.0 -> 18.9
//    us, 88 -> 88 -> 88 @52x52 with a shuffle 15.6 -> 15.3); with wide rows and small tiles the run is several times the tile, and the plan without it stays
//    (32 -> 16 @112x112 b64 52.8, 56.9). The copies go straight to LDS: through registers, with an exposed latency for each batch of them, it was slower.
//  * The bytes go to LDS, a row per pixel, and the pointwise layer's waves take its pairs of 16-row tiles in turn, weights straight
//    from memory in a ring of four reduction steps that is refilled across pairs and layers: the first ones are requested before the
//    depthwise layer begins, as are the elements of a residual or of a shuffle's other blob.
//  * Behind a barrier they do the same for the second pointwise layer.
// Waits are 40, 50 and 57 % of the waves' time, vector issue 53, 34 and 17 % of the kernel's and the address unit 41, 52 and 26 % at 2.3, 2.3 and 1.2
// waves a SIMD (88 channels @52x52 with staged pixels, 176 @26x26 without and 352 @13x13 with, each with a shuffle and a layer behind). In traces of the
// detection model, 16 images, us as two or three launches / as one, with the unit's shuffle and the next unit's first layer: 88 channels @52x52
// 5.1 + 14.3 / 16.4, 176 @26x26 4.1 + 10.0 / 12.4, 352 @13x13 3.7 + 6.1 + 4.9 / 12.1; 5x5 with two pointwise layers, 64 @13x13 3.4 + 4.7 / 6.0.
#include "conv_dwpw.hpp"

#include "conv_pwpw_common.hpp"
#include "dwpw_requests.hpp"

#include <algorithm>

namespace ohip {

namespace {

enum { DP_NONE = 3, DP_FULL = 4 };  // no second pointwise layer, PP_NONNEG with Epilogue::so_full (KIND1, beside PP_I8, PP_NONNEG and PP_F32)

struct DwPwArgs {
    PwPwLayer l[2];
    // the depthwise layer
    const int8_t* dw_w;
    const float *dw_scale_in, *dw_bias;
    float dw_p0, dw_scale, dw_half;
    unsigned dw_qh, in_bytes;
    unsigned hw_m, ow_m, total_pix;  // divisions (FastDiv) by the pixels and the columns of an output image
    int HW, OW, H, W, tiles;         // H, W: of the input
    int sh, sw, ph, pw, dh, dw, C8;
    unsigned hw_s, ow_s;
    int lg, dw_lrelu, dw_nonneg;     // lg: log2 of the pixel groups
    unsigned first_pack;             // channels of an element of a shuffle's first half
    unsigned between;                // bytes of LDS between the first layer's pixels and the constants
};
template <bool STAGED>
using DwPwStaged = std::conditional_t<STAGED, DwPwStage, NoJoin>;  // the pixels that a workgroup stages

// the fp32 blob whose elements an epilogue reads
template <class A>
__device__ __forceinline__ const float* add_blob(const A& ja) {
    if constexpr (std::is_same_v<A, PwShuffle>) return ja.other;
    else if constexpr (std::is_same_v<A, NoJoin>) return nullptr;
    else return ja.residual;
}
// 16 bytes a lane from a buffer to `to` (the same for the wave) and on in LDS, in the lanes' order; out of range: zeros
__device__ __forceinline__ void copy16(__amdgpu_buffer_rsrc_t r, int8_t* to, unsigned v, unsigned s) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void*)to, 16, (int)v, (int)s, 0, 0);
}
template <class A>
__device__ __forceinline__ unsigned sh_image(const A& ja) {
    if constexpr (std::is_same_v<A, PwShuffle>) return ja.sh_image;
    else return 0;
}
template <class A>
__device__ __forceinline__ int ja_pack(const A& ja) {
    if constexpr (std::is_same_v<A, PwShuffle>) return ja.other_pack;
    else return 4;
}

}  // namespace

// A operands of the depthwise layer: [pair of octets][lane 64][4 PK bytes], PK = 2 (3x3) or 4 (5x5) dwords; byte 2 m + e of lane
// (r = lane % 16, g = lane / 16) is channel r's weight of tap 4 m + 2 (g % 2) + e if r is of octet g / 2 of the pair, else zero.
static int dwpw_dwords(int ks) { return ks == 3 ? 2 : 4; }
size_t dwpw_weight_bytes(int C, int ks) { return (size_t)((C / 8 + 1) / 2) * 256 * dwpw_dwords(ks); }
void dwpw_pack_weights(const int8_t* w, int C, int ks, int8_t* dst) {
    const int taps = ks * ks, row = 4 * dwpw_dwords(ks);
    std::fill(dst, dst + dwpw_weight_bytes(C, ks), (int8_t)0);
    for (int op = 0; op < (C / 8 + 1) / 2; ++op)
        for (int lane = 0; lane < 64; ++lane) {
            const int r = lane % 16, g = lane / 16, c = 16 * op + r;
            if (r / 8 != g / 2 || c >= C) continue;
            for (int k = 0; k < (taps + 3) / 4 * 2; ++k) {
                const int tap = 4 * (k / 2) + 2 * (g % 2) + k % 2;
                if (tap < taps) dst[((size_t)op * 64 + lane) * row + k] = w[(size_t)c * taps + tap];
            }
        }
}

// TAPS: 9 or 25. EPI: the first pointwise layer's epilogue: EPI_I8_P8; EPI_F32_P4_FUSED (with or without a residual and a twin; without
// a second layer this is the plain fp32 result as well), EPI_F32_P4_PARTS, EPI_F32_SHUFFLE. KIND1: the second layer's result or DP_NONE.
// DFULL: the depthwise layer ends as EPI_I8_P8_FULL says (else any int8 end). STAGED: the plans that copy the windows' pixels into LDS.
// (An instance of its own: with both ways in one kernel either carried the other's registers, 3x3 102 to 114 of them for 80 to 94, 5x5 154 to
// 166 for 106 to 122, a wave a SIMD less. The plans without staged pixels, the best one of each of 700 drawn layers, half of them with a stride,
// then took up to 1.14 of their time before there were staged ones, 5x5 up to 1.17 and 1.02 on average; now 3x3 0.97, 5x5 0.995, at most 1.04.)
// out: the last layer's result; sum: with a second layer, the first one's fp32 result (null: not wanted).
template <int NW, int TAPS, int EPI, int KIND1, bool DFULL, bool STAGED>
__global__ void __launch_bounds__(64 * NW) conv_dwpw_kernel(const int8_t* __restrict__ x, void* __restrict__ out, float* __restrict__ sum,
                                                                  DwPwArgs pa, PwAdd<EPI> ja, DwPwStaged<STAGED> st) {
    constexpr bool SHUF = EPI == EPI_F32_SHUFFLE, I8 = EPI == EPI_I8_P8, PARTS = EPI == EPI_F32_P4_PARTS, FUSED = EPI == EPI_F32_P4_FUSED || PARTS;
    constexpr bool NEXT = KIND1 != DP_NONE;
    constexpr int KS = TAPS == 9 ? 3 : 5, M = (TAPS + 3) / 4, PK = TAPS == 9 ? 2 : 4;
    constexpr int SC = 4;
    extern __shared__ __attribute__((aligned(16))) int8_t lds[];
    const unsigned tid = threadIdx.x, lane = tid & 63, q = lane >> 4, p = lane & 15;
    const int wave = __builtin_amdgcn_readfirstlane((int)tid >> 6);
    const int xcd = blockIdx.x & 7, tile = (xcd * pa.tiles >> 3) + (int)(blockIdx.x >> 3);  // (grid.x is a multiple of 8)
    if (tile >= (xcd + 1) * pa.tiles >> 3) return;  // (uniform)
    const PwPwLayer &l0 = pa.l[0], &l1 = pa.l[1];
    const unsigned HW = pa.HW, C8 = pa.C8, K0 = l0.K, rb0 = 64u * l0.steps + 16u, rb1 = NEXT ? 64u * l1.steps + 16u : 0u;  // bytes of a pixel's row
    const int pairs0 = (l0.K + 31) / 32, pairs1 = NEXT ? (l1.K + 31) / 32 : 0;
    const int PIX = 16 << pa.lg, group = wave & ((1 << pa.lg) - 1), first = wave >> pa.lg, stride = NW >> pa.lg;
    int8_t *const px0 = lds, *const px1 = lds + PIX * rb0, *const staged = px1;  // (staged: until the depthwise layer ends)
    const unsigned Cd = 16u * ((C8 + 1) / 2);  // channels of the depthwise layer, whole pairs of octets
    float *const constsd = reinterpret_cast<float*>(px1 + pa.between), *const consts0 = constsd + 2 * Cd, *const consts1 = consts0 + 64 * pairs0;

    // ---- the wave's pixels -----------------------------------------------------------------------------------------------------
    const unsigned gp = (unsigned)(tile * PIX + 16 * group) + p;
    const bool ok = gp < pa.total_pix;
    const unsigned n = div_by(gp, FastDiv{pa.hw_m, pa.hw_s, (unsigned)pa.HW}), pix = gp - n * HW;
    const unsigned row0 = (16u * group + p) * rb0, row1 = (16u * group + p) * rb1;
    // byte offset of (image, this lane's channels of a pair, pixel) in a blob of K channels: Byte8, Float4, Float8; a pair is 32 HW
    // (Byte8) or 128 HW (fp32) bytes further
    const unsigned outside = ok ? 0u : PR_OOB;
    auto at_b8 = [&](unsigned K) { return ((n * (K / 8) + q) * HW + pix) * 8u | outside; };
    auto at_f4 = [&](unsigned K) { return ((n * (K / 4) + 2 * q) * HW + pix) * 16u | outside; };
    auto at_f8 = [&](unsigned K) { return ((n * (K / 8) + q) * HW + pix) * 32u | outside; };

    // ---- the pointwise weights: four reduction steps of a pair ----------------------------------------------------------------------
    v4i a[SC][2];
    // (second: of the second layer. Chosen by values and not by branches: behind a branch a wave waits for the loads in front of it)
    auto load_a = [&](bool second, int pr, int step0) {  // (steps that do not exist: at the weights' end, zero)
        const int steps = second ? l1.steps : l0.steps, mt = second ? l1.mt : l0.mt;
        const __amdgpu_buffer_rsrc_t rw = rsrc(second ? l1.w : l0.w, (unsigned)steps * (unsigned)mt * 1024u);
        auto one = [&](int s) {
            const unsigned at = dwpw_weights_at(step0 + s, steps, mt, pr);
#pragma unroll
            for (int h = 0; h < 2; ++h) a[s][h] = load16(rw, lane * 16 + h * 1024, at);
        };
        one(0), one(1);
#pragma unroll
        for (int s = 2; s < SC; s += 2) {
            if (step0 + s < steps) one(s), one(s + 1);  // (uniform)
            else a[s][0] = a[s][1] = a[s + 1][0] = a[s + 1][1] = v4i{0, 0, 0, 0};
        }
    };

    // ---- elements of other blobs ---------------------------------------------------------------------------------------------------
    struct {
        v4i v[2];
    } add;
    const unsigned f_bytes = pa.total_pix * K0 * 4u;  // of an fp32 result or addend; an int8 result may be as many elements as this has bytes
    Epilogue ep0 = pp_epilogue(l0);
    if constexpr (FUSED) ep0.residual = ja.residual, ep0.twin = ja.twin;
    if constexpr (FUSED || SHUF) ep0.twin_scale = ja.twin_scale, ep0.twin_half = ja.twin_half;
    const unsigned add_at = SHUF ? ja_pack(ja) == 8 ? at_f8(K0) : at_f4(K0) : at_f4(K0), add_half = SHUF && ja_pack(ja) == 8 ? 16u : HW * 16u;
    auto load_add = [&](int pr) {
        if constexpr (PARTS) {
            if (pr < pairs0 && 32u * pr + 8 * q < K0 && ok)
#pragma unroll
                for (int h = 0; h < 2; ++h)
                    add.v[h] = *reinterpret_cast<const v4i*>(epi4_residual_at(ep0, ja.join(), n, pix, (int)(32u * pr + 8 * q + 4 * h), (int)K0, (int)HW));
        } else if constexpr (FUSED || SHUF) {
            const DwPwFloats f = dwpw_floats(pr < pairs0 && add_blob(ja) != nullptr, f_bytes, HW, add_half);  // (none: zero, and not used)
            const __amdgpu_buffer_rsrc_t r = rsrc(add_blob(ja), f.bytes);
#pragma unroll
            for (int h = 0; h < 2; ++h) add.v[h] = load16(r, add_at | (32u * pr + 8 * q + 4 * h < K0 ? 0u : PR_OOB), f.at(pr, h));
        }
    };

    // ---- the depthwise layer -----------------------------------------------------------------------------------------------------------
    {
        const unsigned HWi = (unsigned)(pa.H * pa.W), second = q & 1;  // second: of the two pairs of taps in a reduction step
        const unsigned oy = div_by(pix, FastDiv{pa.ow_m, pa.ow_s, (unsigned)pa.OW}), ox = pix - oy * pa.OW;
        const int y0 = (int)oy * pa.sh - pa.ph, x0 = (int)ox * pa.sw - pa.pw;
        // a tap's place in units of 8 bytes: in the blob, or among the staged pixels (one outside the image: the zeros behind them)
        int base, s_first = 0;  // (s_first: where the tile's run begins)
        unsigned none;
        if constexpr (STAGED) {
            const unsigned t_first = (unsigned)(tile * PIX);
            s_first = dwpw_run(st, HW, t_first, div_by(t_first, FastDiv{pa.hw_m, pa.hw_s, HW}));
            base = (int)((q >> 1) * st.pitch) + dwpw_window(st, n, pix) - s_first, none = ((q >> 1) * st.pitch + st.slots) * 8u;
        } else {
            base = (int)((n * C8 + (q >> 1)) * HWi) + y0 * pa.W + x0, none = PR_OOB;
        }
        // the taps inside the image as bits, shifted to the lane's own
        unsigned columns = 0, taps = 0;
#pragma unroll
        for (int d = 0; d < KS; ++d) columns |= (unsigned)(x0 + d * pa.dw) < (unsigned)pa.W ? 1u << d : 0u;
#pragma unroll
        for (int d = 0; d < KS; ++d) taps |= (unsigned)(y0 + d * pa.dh) < (unsigned)pa.H ? columns << KS * d : 0u;
        taps = ok ? second ? taps >> 2 : taps : 0u;
        unsigned v[M][2];
#pragma unroll
        for (int m = 0; m < M; ++m)
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                const int t0 = 4 * m + e, t1 = t0 + 2;
                const int at0 = t0 / KS * pa.dh * pa.W + t0 % KS * pa.dw, at1 = t1 / KS * pa.dh * pa.W + t1 % KS * pa.dw;
                v[m][e] = taps >> t0 & 1 ? (unsigned)(base + (second ? at1 : at0)) * 8u : none;
            }
        // channel r = p's bytes in the operand: dword p / 4 of its octet's two pixels, if the lane's bytes are of that octet
        unsigned sel[2][4];
        {
            // (byte 0x0c of a selector is zero; one byte more of the source is 1 << at further)
            const bool mine = (p >> 3) == (q >> 1), upper = (p >> 2) & 1;
            const unsigned zero = 0x0c0c0c0cu, at = 8u * (p & 3), one = 1u << at;
            const unsigned low = mine && !upper ? one : 0u, high = mine && upper ? one : 0u;
#pragma unroll
            for (unsigned b = 0; b < 4; ++b) sel[0][b] = zero - 12u * low + b * low, sel[1][b] = zero - 12u * high + b * high;
        }
        const int pairs = ((int)C8 + 1) / 2;  // of octets
        const __amdgpu_buffer_rsrc_t rin = rsrc(x, pa.in_bytes), rw = rsrc(pa.dw_w, (unsigned)pairs * 256u * PK);
        v4i b[M];
        int w[PK];
        using Weights = std::conditional_t<PK == 2, v2i, v4i>;
        auto weights = [&](const Weights& t) {
#pragma unroll
            for (int i = 0; i < PK; ++i) w[i] = t[i];
        };
        [[maybe_unused]] int8_t* staged_w = nullptr;
        if constexpr (STAGED) staged_w = staged + st.octets * st.pitch * 8u;
        auto load = [&](int op) {
            const auto pixel = [&](unsigned v) {
                if constexpr (STAGED) return *reinterpret_cast<const v2i*>(staged + (unsigned)op * 16u * st.pitch + v);
                else return load8(rin, v, (unsigned)op * 16u * HWi);
            };
#pragma unroll
            for (int m = 0; m < M; ++m) {
                const v2i lo = pixel(v[m][0]), hi = 4 * m + 1 < TAPS ? pixel(v[m][1]) : v2i{0, 0};
                b[m] = v4i{lo[0], lo[1], hi[0], hi[1]};
            }
            if constexpr (STAGED) weights(*reinterpret_cast<const Weights*>(staged_w + (op * 64 + (int)lane) * 4 * PK));
            else if constexpr (PK == 2) weights(load8(rw, lane * 8, (unsigned)op * 512u));
            else weights(load16(rw, lane * 16, (unsigned)op * 1024u));
        };

        if constexpr (STAGED) {
            // ---- the pixels that the tile's windows touch, octet by octet, and the weights into LDS: two pixels a lane -------------------------
            const unsigned lg = st.lg_lanes, unit = lane & ((1u << lg) - 1), sub = lane >> lg, sets = 64u >> lg;  // sets: octets of a copy
            for (unsigned c = 0; c < st.units; c += 64) {
                const int at = s_first + 2 * (int)(c + unit);
                const unsigned im = div_by((unsigned)at, FastDiv{st.image_m, st.image_s, st.image});
                const bool in = at >= 0 && 2 * (c + unit) < st.slots && im * HW < pa.total_pix;
                const unsigned from = in ? dwpw_copied(st, HW, C8, im, sub, (unsigned)at) : PR_OOB;
                if (c + unit < st.units)
                    for (unsigned o = wave * sets; o < C8; o += NW * sets) copy16(rin, staged + (o * st.pitch + 2 * c) * 8, from, o * HW * 8u);
            }
            for (unsigned i = wave; i < ((unsigned)pairs * PK + 3) / 4; i += NW) copy16(rw, staged_w + i * 1024, lane * 16, i * 1024);
        } else {
            load(min(first, pairs - 1));
        }
        asm volatile("" ::: "memory");  // (in front of the others: the compiler would move them to the loop)

        // ---- constants into LDS: scale_in and bias of each layer (they are padded to whole pairs of tiles and more) ---------------------
        // (an array a wave: six of them. Copied without registers, so that one wait covers them and what was requested before: 88 @52x52 16.6 ->
        // 15.6 us, 5x5 128 @26x26 8.8 -> 8.6)
        for (int w = wave; w < (NEXT ? 6 : 4); w += NW) {
            const unsigned d = w >> 1;  // 0: the depthwise layer, 1, 2: the others
            const float* const si = d == 0 ? pa.dw_scale_in : d == 1 ? l0.scale_in : l1.scale_in;
            const float* const bi = d == 0 ? pa.dw_bias : d == 1 ? l0.bias : l1.bias;
            const unsigned quads = d == 0 ? Cd / 4 : 8u * (d == 1 ? pairs0 : pairs1);
            const __amdgpu_buffer_rsrc_t r = rsrc(w & 1 ? bi : si, quads * 16u);
            int8_t* const to = reinterpret_cast<int8_t*>(d == 0 ? constsd : d == 1 ? consts0 : consts1) + (w & 1 ? quads * 16u : 0u);
            for (unsigned i = 0; i < quads; i += 64)
                if (i + lane < quads) copy16(r, to + i * 16, lane * 16, i * 16);
        }
        __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): this wave's copies have arrived
        __syncthreads();

        // ---- what comes behind the depthwise layer, requested now: weights, elements of another blob --------------------------------------
        const bool begins1 = NEXT && first >= pairs0;  // a wave without a pair of the first layer
        load_a(begins1, min(first, (begins1 ? pairs1 : pairs0) - 1), 0);
        load_add(first);

        // LeakyReLU or none, and the clamp of the rounded result: [0, dw_qh] behind ReLU / clip, else the int8 range
        Epilogue epd{};
        epd.act_p0 = pa.dw_p0, epd.lrelu = pa.dw_lrelu != 0;
        const ohip_v2s top = __builtin_bit_cast(ohip_v2s, pa.dw_qh), bottom = __builtin_bit_cast(ohip_v2s, pa.dw_nonneg ? 0u : 0xff81ff81u);
        if constexpr (STAGED) load(min(first, pairs - 1));
        for (int op = first; op < pairs;) {
            v4i acc = {0, 0, 0, 0};
#pragma unroll
            for (int m = 0; m < M; ++m) {
                constexpr unsigned Z = 0;
                const int e = 2 * (m & 1);
                const v4i A = {(int)__builtin_amdgcn_perm(Z, (unsigned)w[m >> 1], sel[0][e]), (int)__builtin_amdgcn_perm(Z, (unsigned)w[m >> 1], sel[1][e]),
                               (int)__builtin_amdgcn_perm(Z, (unsigned)w[m >> 1], sel[0][e + 1]), (int)__builtin_amdgcn_perm(Z, (unsigned)w[m >> 1], sel[1][e + 1])};
                acc = __builtin_amdgcn_mfma_i32_16x16x64_i8(A, b[m], acc, 0, 0, 0);
            }
            const int now = op;
            op += stride;
            if (op < pairs) load(op);  // (refilled in place: the next pair's bytes arrive under this one's requantization)
            const v4i si = *reinterpret_cast<const v4i*>(constsd + 16 * now + 4 * q), bi = *reinterpret_cast<const v4i*>(constsd + Cd + 16 * now + 4 * q);
            unsigned bytes;
            if constexpr (DFULL) {  // (dw_scale is doubled)
                float t2[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) t2[e] = __fmul_rn(__fmaf_rn((float)acc[e], __int_as_float(si[e]), __int_as_float(bi[e])), pa.dw_scale);
                bytes = quant4_full(t2, pa.dw_half);
            } else {
                int k[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const float t = __fmul_rn(lrelu_or_not(epd, __fmaf_rn((float)acc[e], __int_as_float(si[e]), __int_as_float(bi[e]))), pa.dw_scale);
                    k[e] = (int)__fadd_rn(t, __builtin_copysignf(pa.dw_half, t));
                }
                ohip_v2s lo = __builtin_bit_cast(ohip_v2s, __builtin_amdgcn_cvt_pk_i16(k[0], k[1])), hi = __builtin_bit_cast(ohip_v2s, __builtin_amdgcn_cvt_pk_i16(k[2], k[3]));
                lo = __builtin_elementwise_max(__builtin_elementwise_min(lo, top), bottom);
                hi = __builtin_elementwise_max(__builtin_elementwise_min(hi, top), bottom);
                bytes = __builtin_amdgcn_perm(__builtin_bit_cast(unsigned, hi), __builtin_bit_cast(unsigned, lo), 0x06040200u);
            }
            if (2u * now + (q >> 1) < C8) *reinterpret_cast<unsigned*>(px0 + row0 + 16 * now + 4 * q) = bytes;
        }
    }
    __syncthreads();

    // One pointwise layer: the wave's pairs; finish(pair, sums). Behind the last one the next layer's first weights are requested.
    auto layer = [&](auto second_c, const PwPwLayer& l, int pairs, const int8_t* px, auto finish) {
        constexpr bool SECOND = decltype(second_c)::value;
        for (int pr = first; pr < pairs; pr += stride) {
            v4i c0 = {0, 0, 0, 0}, c1 = {0, 0, 0, 0};
            for (int s0 = 0; s0 < l.steps; s0 += SC) {
                auto step = [&](int s) {  // (one that does not exist: zero weights, and bytes of this workgroup's LDS)
                    const v4i b = *reinterpret_cast<const v4i*>(px + 64 * (s0 + s));
                    c0 = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[s][0], b, c0, 0, 0, 0);
                    c1 = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[s][1], b, c1, 0, 0, 0);
                };
                step(0), step(1);
#pragma unroll
                for (int s = 2; s < SC; s += 2)
                    if (s0 + s < l.steps) step(s), step(s + 1);  // (uniform)
                const bool same = s0 + SC < l.steps, more = same || pr + stride < pairs;
                const bool then = NEXT && !SECOND && !more;
                load_a(SECOND || then, same ? pr : more ? pr + stride : then ? min(first, pairs1 - 1) : pr, same ? s0 + SC : 0);
            }
            finish(pr, c0, c1);
        }
    };
    auto constants = [&](const float* c, int pairs, unsigned ch0, float (&si)[8], float (&bi)[8]) {
#pragma unroll
        for (int e = 0; e < 8; ++e) si[e] = c[ch0 + e], bi[e] = c[32 * pairs + ch0 + e];
    };

    // ---- the first pointwise layer --------------------------------------------------------------------------------------------------
    int8_t* const to1 = px1 + row1;  // this lane's pixel of the second layer's input
    float* const f_out = NEXT ? sum : static_cast<float*>(out);
    const DwPwFloats f0 = dwpw_floats(f_out != nullptr, f_bytes, HW, HW * 16u);
    const __amdgpu_buffer_rsrc_t rout0 = I8 ? rsrc(out, NEXT ? 0u : pa.total_pix * K0) : rsrc(f_out, f0.bytes);
    // elements of a shuffle's blobs. The first half is Float4 or Float8: a store to Float4 touches 8 lines of 128 bytes where it touches 16
    // of Float8's, and the address unit works line by line (88 channels @52x52 b16 16.8 us
    // with Float8 on both sides, 16.4 with Float4; 176 channels on one 26x26 image 6.9 and 6.5)
    const unsigned sh_lane = SHUF ? n * sh_image(ja) + (2u * q * HW + pix) * 8u : 0u;
    const unsigned sh_first = SHUF ? n * sh_image(ja) + 2u * q * HW * 8u + pix * pa.first_pack : 0u, sh_next = pa.first_pack == 4 ? HW * 16u : 16u;
    auto finish0 = [&](int pr, const v4i& c0, const v4i& c1) {
        const unsigned ch0 = 32u * pr + 8 * q;
        float si[8], bi[8];
        constants(consts0, pairs0, ch0, si, bi);
        if constexpr (I8) {
            const v2i b = pp_bytes<0>(ep0, l0, si, bi, c0, c1);
            if constexpr (NEXT) {
                if (ch0 < K0) *reinterpret_cast<v2i*>(to1 + ch0) = b;
            } else {
                store8(rout0, b, ch0 < K0 ? at_b8(K0) : PR_OOB, (unsigned)pr * 32u * HW);
            }
        } else {
            v4i r[2] = {pp_values(ep0, si, bi, c0), pp_values(ep0, si + 4, bi + 4, c1)};
            if constexpr (SHUF) {
                // with the same channels of the other blob these are channels 2 ch0 .. 2 ch0 + 15 of the shuffled one: two packs of 8
                const unsigned half = K0 / 8;  // packs of 8 in each half
#pragma unroll
                for (int w = 0; w < 2; ++w) {
                    float* const f = w ? ja.sh_out1 : ja.sh_out0;
                    int8_t* const b8 = w ? ja.sh_q1 : ja.sh_q0;
                    if (w ? 8u * pr + 8 <= half : 8u * pr >= half) continue;  // (uniform: none of the pair's packs is in this half)
#pragma unroll
                    for (int h = 0; h < 2; ++h) {
                        const v4i o = add.v[h];
                        const v4i even = ja.other_odd ? r[h] : o, odd = ja.other_odd ? o : r[h];  // (uniform)
                        const v4i lo = {even[0], odd[0], even[1], odd[1]}, hi = {even[2], odd[2], even[3], odd[3]};
                        const unsigned pack = ch0 / 4 + h - (w ? half : 0u);  // in this half; beyond it on either side: the other half's
                        const unsigned e = sh_lane + (8u * pr + h - (w ? half : 0u)) * HW * 8u;
                        const bool live = ok && pack < half;  // (a channel past the last one is a pack past the second half)
                        if (NEXT && w) {
                            const v2i b = {quantize4(lo, ja.twin_scale, ja.twin_half), quantize4(hi, ja.twin_scale, ja.twin_half)};
                            if (pack < half) *reinterpret_cast<v2i*>(to1 + 8 * pack) = b;
                            continue;
                        }
                        if (f != nullptr) {
                            const __amdgpu_buffer_rsrc_t rf = rsrc(f, PR_OOB);
                            const unsigned v = live ? (w ? e : sh_first + (8u * pr + h) * HW * 8u) * 4u : PR_OOB;
                            store16(rf, lo, v, 0), store16(rf, hi, v + (w ? 16u : sh_next), 0);
                        }
                        if (b8 != nullptr)
                            store8(rsrc(b8, PR_OOB), v2i{quantize4(lo, ja.twin_scale, ja.twin_half), quantize4(hi, ja.twin_scale, ja.twin_half)},
                                   live ? e : PR_OOB, 0);
                    }
                }
            } else {
                v2i tw;
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    if (PARTS || ep0.residual != nullptr)  // (uniform)
#pragma unroll
                        for (int e = 0; e < 4; ++e) r[h][e] = __float_as_int(__fadd_rn(__int_as_float(r[h][e]), __int_as_float(add.v[h][e])));
                    if (NEXT || ep0.twin != nullptr) tw[h] = quantize4(r[h], ep0.twin_scale, ep0.twin_half);
                    store16(rout0, r[h], ch0 + 4 * h < K0 ? at_f4(K0) : PR_OOB, f0.at(pr, h));
                }
                if constexpr (NEXT) {
                    if (ch0 < K0) *reinterpret_cast<v2i*>(to1 + ch0) = tw;
                } else if (ep0.twin != nullptr) {  // K % 8 == 0 then: the lane's 8 channels are one Byte8 element
                    store8(rsrc(ep0.twin, pa.total_pix * K0), tw, ch0 < K0 ? at_b8(K0) : PR_OOB, (unsigned)pr * 32u * HW);
                }
            }
        }
    };
    auto finish_then_add = [&](int pr, const v4i& c0, const v4i& c1) {
        finish0(pr, c0, c1);
        if ((SHUF || FUSED) && pr + stride < pairs0) load_add(pr + stride);
    };
    if constexpr (!NEXT) {
        layer(std::false_type{}, l0, pairs0, px0 + row0 + 16 * q, finish_then_add);
    } else {
        layer(std::false_type{}, l0, pairs0, px0 + row0 + 16 * q, finish_then_add);
        __syncthreads();

        // ---- the second ------------------------------------------------------------------------------------------------------------
        const unsigned K1 = l1.K;
        const Epilogue ep1 = pp_epilogue(l1);
        const __amdgpu_buffer_rsrc_t rout = rsrc(out, pa.total_pix * K1 * (KIND1 == PP_F32 ? 4u : 1u));
        auto finish1 = [&](int pr, const v4i& c0, const v4i& c1) {
            const unsigned ch0 = 32u * pr + 8 * q;
            float si[8], bi[8];
            constants(consts1, pairs1, ch0, si, bi);
            if constexpr (KIND1 == PP_F32) {
                const v4i r0 = pp_values(ep1, si, bi, c0), r1 = pp_values(ep1, si + 4, bi + 4, c1);
                const unsigned v = at_f4(K1), s = (unsigned)pr * 128u * HW;
                store16(rout, r0, ch0 < K1 ? v : PR_OOB, s), store16(rout, r1, ch0 + 4 < K1 ? v : PR_OOB, s + HW * 16u);
            } else {
                store8(rout, pp_bytes<KIND1 == DP_FULL ? 2 : KIND1 == PP_NONNEG ? 1 : 0>(ep1, l1, si, bi, c0, c1), ch0 < K1 ? at_b8(K1) : PR_OOB, (unsigned)pr * 32u * HW);
            }
        };
        layer(std::true_type{}, l1, pairs1, px1 + row1 + 16 * q, finish1);
    }
}

// ---------------------------------------------------------------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------------------------------------------------------------

// the staged pixels and weights make room for the second layer's pixels
static size_t dwpw_between(const ConvGeom& gd, const ConvGeom* g1, int groups, const DwPwStage& st) {
    const size_t weights = (dwpw_weight_bytes(gd.C, gd.kh) + 1023) / 1024 * 1024;
    return std::max(g1 ? 16 * (size_t)groups * (64 * (size_t)igemm_channel_groups(g1->C) + 16) : 0, st.pitch ? 8 * (size_t)st.octets * st.pitch + weights : 0);
}
static size_t dwpw_lds_bytes(const ConvGeom& gd, const ConvGeom& g0, const ConvGeom* g1, int groups, const DwPwStage& st) {
    return 16 * (size_t)groups * (64 * (size_t)igemm_channel_groups(g0.C) + 16) + dwpw_between(gd, g1, groups, st) +
           256 * (size_t)((g0.K + 31) / 32 + (g1 ? (g1->K + 31) / 32 : 0)) + 128 * (size_t)((g0.C / 8 + 1) / 2);
}
static DwPwStage dwpw_staged(const ConvGeom& gd, int groups) {
    if (gd.sh != 1 || gd.sw != 1 || gd.OH != gd.H || gd.OW != gd.W) return {};
    return dwpw_stage(gd.C, gd.H, gd.W, gd.kh, gd.ph, gd.pw, gd.dh, gd.dw, 16 * groups);  // (without the division by an image)
}

bool dwpw_front_applicable(const ConvGeom& gd, const Epilogue& ed) {
    if (gd.groups != gd.C || gd.K != gd.C || gd.C % 8 || gd.kh != gd.kw || (gd.kh != 3 && gd.kh != 5)) return false;
    for (int v : {gd.sh, gd.sw, gd.ph, gd.pw, gd.dh, gd.dw})
        if (v > 255) return false;
    const int epi = dw_mfma_epilogue(ed, gd.K);
    if (epi != EPI_I8_P8 && epi != EPI_I8_P8_NONNEG) return false;
    const size_t limit = (size_t)1 << 31;
    return (size_t)gd.N * gd.C * gd.H * gd.W < limit && (size_t)gd.C * 64 < limit;
}

bool conv_dwpw_applicable(const ConvGeom& gd, const Epilogue& ed, const ConvGeom& g0, const Epilogue& e0, const ConvGeom* g1, const Epilogue* e1) {
    if (!dwpw_front_applicable(gd, ed) || !pwpw_pointwise(g0) || g0.C != gd.K || g0.N != gd.N || g0.H != gd.OH || g0.W != gd.OW || g0.N < 1) return false;
    if (dwpw_lds_bytes(gd, g0, g1, 1, DwPwStage{}) > 65536) return false;
    const int k0 = pwpw_kind(e0, g0.K);
    const bool shuffle = e0.join && e0.join->other, parts = e0.join && !shuffle;
    if (k0 != PP_I8 && k0 != PP_F32) return false;
    if (k0 == PP_I8 && e0.fused()) return false;
    if ((e0.twin || shuffle || parts || g1) && g0.K % 8) return false;
    if (g1) {
        if (!pwpw_pointwise(*g1) || g1->C != g0.K || g1->N != g0.N || g1->H != g0.H || g1->W != g0.W) return false;
        if (parts || e0.twin || pwpw_kind(*e1, g1->K) < 0) return false;
        if (shuffle && (e0.join->sh_image != (size_t)g0.K * g0.H * g0.W || !e0.join->sh_out0)) return false;  // (two halves)
        if (gd.kh == 5 && k0 != PP_I8) return false;
    } else if (gd.kh == 5 && shuffle) {
        return false;
    }
    const size_t px = (size_t)g0.N * g0.H * g0.W, limit = (size_t)1 << 31;
    if (px * g0.C >= limit || px * g0.K * (k0 == PP_F32 ? 4 : 1) >= limit) return false;
    if (shuffle && px * g0.K * 4 * (g1 ? 1 : 2) >= limit) return false;
    if (g1 && px * g1->K * layout_elem_bytes(e1->out_layout) >= limit) return false;
    for (const ConvGeom* g : {&g0, g1})
        if (g && (size_t)igemm_channel_groups(g->C) * igemm_padded_rows(g->K) * 64 >= limit) return false;  // (the packed weights)
    return true;
}

// Cost models in us, fitted to launches replayed from captured graphs behind a copy that leaves the L2 caches cold, over 11700 drawn layers
// (16 to 720 channels, 5x5 to 112x112 pixels, batches of 1 to 64, every end) and every plan of them: half of the times within 5 %, nine in ten within
// 12 % (13 % over 15700 other layers, where the plan that they choose takes 1.014 of the fastest one's time). The launch:
// a wave walks nd pairs of octets and n0 and n1 pairs of row tiles one behind the other, once if every workgroup is resident, and the more
// often the more waves there are for a compute unit than it holds (the mean of all compute units and the fullest one); with staged pixels it issues
// its share of the copies in front of that.
struct DwPwShape {
    float px, mac, wide;  // output pixels; 10^9 multiply-adds of the pointwise layers; 10^6 values past the 256th channel
    float end, mb;        // bytes that a pointwise end reads and writes beside its input, for a channel of a pixel; 10^6 bytes of the launch
    int octets;
    int pairs_d, pairs[2], steps[2];
    bool k5, f32, adds;
    DwPwShape(const ConvGeom& gd, const ConvGeom& g0, const Epilogue& e0, const ConvGeom* g1)
        : px((float)g0.N * g0.H * g0.W), mac(1e-9f * px * g0.K * (float)(gd.C + (g1 ? g1->K : 0))), wide(1e-6f * px * (float)std::max(0, gd.C - 256)), end(ends(e0, g1)),
          mb(1e-6f * px * ((float)(gd.C * gd.sh * gd.sw) + (float)g0.K * end + (float)(g1 ? g1->K : 0))), octets(gd.C / 8), pairs_d((gd.C / 8 + 1) / 2),
          pairs{(g0.K + 31) / 32, g1 ? (g1->K + 31) / 32 : 0}, steps{igemm_channel_groups(g0.C), g1 ? igemm_channel_groups(g1->C) : 0},
          k5(gd.kh == 5), f32(e0.out_kind == OTTER_HIP_OUT_F32), adds(e0.residual || e0.join) {}
    static float ends(const Epilogue& e0, const ConvGeom* g1) {
        if (e0.out_kind != OTTER_HIP_OUT_F32) return g1 ? 0.f : 1.f;
        if (!e0.join || !e0.join->other) return (e0.residual || e0.join ? 8.f : 4.f) + (e0.twin ? 1.f : 0.f);
        const JoinArgs& j = *e0.join;
        return 4.f + (j.sh_out0 ? 4.f : 0.f) + (j.sh_out1 ? 4.f : 0.f) + (j.sh_q0 ? 1.f : 0.f) + (j.sh_q1 ? 1.f : 0.f);
    }
};
static float dwpw_cost(const DwPwShape& s, int waves, int groups, const DwPwStage& st, size_t lds) {
    static const struct {
        float once[10], more[10], byte, mac, wide;  // for 10^6 bytes, 10^9 multiply-adds of the pointwise layers, 10^6 values past the 256th channel
    } table[4] = {  // four and eight waves, without and with staged pixels
        {{2.85f, 0.386f, 0.711f, 0.381f, 0.0708f, 0.385f, 0.0661f, 0.198f, 0.154f, 0}, {0.572f, 0.252f, 0.78f, 0.19f, 0.0315f, 0.201f, 0.0298f, 0, 0, 0}, 0.0929f, 0.89f, 0.165f},
        {{2.92f, 0.397f, 0.91f, 0.435f, 0.0943f, 0.514f, 0.102f, 0.262f, 0.169f, 0}, {0.62f, 0.287f, 0.738f, 0.169f, 0.0626f, 0.18f, 0.0679f, 0.116f, 0.0493f, 0}, 0.0832f, 0.476f, 0.0247f},
        {{3.45f, 0.132f, 0.341f, 0.367f, 0.0546f, 0.369f, 0.0726f, 0.193f, 0.159f, 0.0592f}, {0.682f, 0.171f, 0.556f, 0.11f, 0.0498f, 0.247f, 0.00552f, 0, 0, 0.0638f}, 0.0926f, 1.13f, 1.65f},
        {{3.24f, 0.25f, 0.561f, 0.432f, 0.0621f, 0.486f, 0.0934f, 0.239f, 0.144f, 0.0525f}, {0.829f, 0.161f, 0.377f, 0.238f, 0, 0.201f, 0.0645f, 0, 0, 0.0838f}, 0.0913f, 0.33f, 0.726f}};
    const int stride = waves / groups, nd = (s.pairs_d + stride - 1) / stride, n0 = (s.pairs[0] + stride - 1) / stride, n1 = (s.pairs[1] + stride - 1) / stride;
    const auto& k = table[(st.pitch ? 2 : 0) + (waves == 8)];
    const float copies = st.pitch ? (float)((st.units + 63) / 64 * ((s.octets + (64 >> st.lg_lanes) - 1) >> (6 - st.lg_lanes))) / (float)waves : 0.f;
    const float f[10] = {1, s.k5 ? 0.f : (float)nd, s.k5 ? (float)nd : 0.f, (float)n0, (float)(n0 * s.steps[0]), (float)n1, (float)(n1 * s.steps[1]), s.f32 ? (float)n0 : 0.f,
                         s.adds ? (float)n0 : 0.f, copies};
    // workgroups for a compute unit, on average and on the fullest one, in rounds of those that run side by side at full speed: eight waves, or what the
    // LDS with staged pixels has room for, which is whole workgroups
    const int per_cu = ((int)((s.px + (float)(16 * groups - 1)) / (float)(16 * groups)) + 255) / 256, room = (int)(163840 / lds);
    const bool few = st.pitch && room * waves <= 8;
    const float held = few ? (float)room : 8.f / (float)waves;
    const float fullest = few ? (float)((per_cu + room - 1) / room) : (float)per_cu / held;
    const float rounds = std::max(0.f, 0.5f * (fullest + s.px / (4096.f * (float)groups * held)) - 1.f);
    float t = k.byte * s.mb + k.mac * s.mac + k.wide * s.wide;
    for (int i = 0; i < 10; ++i) t += f[i] * (k.once[i] + rounds * k.more[i]);
    return t;
}
// the layers by themselves, the pointwise ones as a pair where that is a launch
static float dwpw_cost_apart(const DwPwShape& s, const ConvGeom& gd, const ConvGeom& g0, const ConvGeom* g1) {
    const float mbd = 1e-6f * s.px * gd.C * (gd.sh * gd.sw + 1.f), mb0 = 1e-6f * s.px * (gd.C + g0.K * s.end);
    float t = 4.7f + (0.266f + (s.k5 ? 0.0437f : 0)) * mbd + 0.175f * mb0 + 1.68e-9f * s.px * g0.C * g0.K + 1.35e-3f * gd.C + 0.261e-3f * g0.K;
    if (g1) t += 1.74f + 0.308e-6f * s.px * ((float)g0.K + g1->K) + 1.34e-9f * s.px * g0.K * g1->K + 1.44e-3f * g1->K + (g0.K > 256 ? 0.827f : 0);
    return t;
}

// Groups of 16 pixels for a workgroup, + 16 for one of four waves: those have fewer idle waves where there are many pixels and few
// channels (88 -> 88 -> 88 @52x52 b16 with a shuffle: eight waves and four groups 17.6 us, four and four 15.6), eight a shorter chain;
// + 32 with staged pixels (15.3): not where the input's address is no multiple of their eight bytes.
static int dwpw_plan(const ConvGeom& gd, const ConvGeom& g0, const Epilogue& e0, const ConvGeom* g1, bool aligned, float* cost) {
    const DwPwShape s(gd, g0, e0, g1);
    int best = 0;
    for (int waves = 8; waves >= 4; waves -= 4)
        for (int g = 1; g <= waves; g *= 2)
            for (int staged = 0; staged <= (aligned ? 1 : 0); ++staged) {
                const DwPwStage st = staged ? dwpw_staged(gd, g) : DwPwStage{};
                const size_t lds = dwpw_lds_bytes(gd, g0, g1, g, st);
                if (lds > 65536 || (staged && !st.pitch)) continue;
                const float c = dwpw_cost(s, waves, g, st, lds);
                if (!best || c < *cost) best = g + (waves == 4 ? 16 : 0) + 32 * staged, *cost = c;
            }
    return best;
}
// Over 15684 layers beside the fit the rule takes 58 %, which then take 0.805 of their time apart, and gives 0.886 of the time of all (the faster of both each
// time: 0.869); 69 are over 5 % slower than apart, the worst 1.29. In each band of pixels, windows and layers behind, nine in ten of those that it takes are at
// most level with the layers apart (but for ten 5x5 layers alone on 32768 pixels and more: 1.03). Three kinds stay apart whatever the models say:
//  * 200 MB and more (5x5: 60 MB), which the caches do not hold: both models are a third below the times there, and what 0.92 would take is 1.03 (1.0 to 1.08)
//    of the time, the worst 1.34.
//  * 640 channels and more on 4096 pixels and more: 0.92 would take 27 of 207, up to 1.16.
//  * ten million values and more without a stride: 34 of the 238 that 0.92 would take are over 5 % slower; and apart they find each other's blobs in the caches,
//    which the fits' operands are not in: in 2650 drawn blocks whose depthwise and project layers ran as one launch, the whole block took 0.93 to 0.97 of
//    its time below ten million (stride 2: 0.87 to 0.95 at any size), 1.03 from there, 1.17 from thirty million.
bool conv_dwpw_faster(const ConvGeom& gd, const ConvGeom& g0, const Epilogue& e0, const ConvGeom* g1) {
    const DwPwShape s(gd, g0, e0, g1);
    if (s.mb >= (s.k5 ? 60.f : 200.f) || (gd.C >= 640 && s.px >= 4096) || (gd.sh == 1 && gd.sw == 1 && s.px * gd.C >= 1e7f)) return false;
    float cost = 0;
    dwpw_plan(gd, g0, e0, g1, true, &cost);
    return cost < 0.92f * dwpw_cost_apart(s, gd, g0, g1);
}

template <int NW, int TAPS, int EPI, int KIND1, bool DFULL>
static hipError_t launch_dwpw_waves(const int8_t* x, void* out, float* sum, const DwPwArgs& pa, const DwPwStage& st, const Epilogue& e0, size_t lds, hipStream_t stream) {
    const dim3 grid((pa.tiles + 7) / 8 * 8), block(64 * NW);
    if (st.pitch) launch((conv_dwpw_kernel<NW, TAPS, EPI, KIND1, DFULL, true>), grid, block, lds, stream, x, out, sum, pa, PwAdd<EPI>::of(e0), st);
    else launch((conv_dwpw_kernel<NW, TAPS, EPI, KIND1, DFULL, false>), grid, block, lds, stream, x, out, sum, pa, PwAdd<EPI>::of(e0), NoJoin{});
    return hipGetLastError();
}
template <int TAPS, int EPI, int KIND1>
static hipError_t launch_dwpw(int waves, bool dfull, const int8_t* x, void* out, float* sum, const DwPwArgs& pa, const DwPwStage& st, const Epilogue& e0, size_t lds,
                              hipStream_t stream) {
    if (dfull)
        return waves == 4 ? launch_dwpw_waves<4, TAPS, EPI, KIND1, true>(x, out, sum, pa, st, e0, lds, stream)
                          : launch_dwpw_waves<8, TAPS, EPI, KIND1, true>(x, out, sum, pa, st, e0, lds, stream);
    return waves == 4 ? launch_dwpw_waves<4, TAPS, EPI, KIND1, false>(x, out, sum, pa, st, e0, lds, stream)
                      : launch_dwpw_waves<8, TAPS, EPI, KIND1, false>(x, out, sum, pa, st, e0, lds, stream);
}

hipError_t run_conv_dwpw(const int8_t* x, const int8_t* dw_w, float dw_so, const ConvGeom& gd, const Epilogue& ed, const int8_t* const w[2],
                         const float so[2], void* out, float* sum, const ConvGeom& g0, const Epilogue& e0, const ConvGeom* g1, const Epilogue* e1,
                         int force, hipStream_t stream) {
    if (!conv_dwpw_applicable(gd, ed, g0, e0, g1, e1)) return hipErrorInvalidValue;
    DwPwArgs pa{};
    pa.l[0] = pwpw_layer(g0, e0, w[0], so[0]);
    if (g1) pa.l[1] = pwpw_layer(*g1, *e1, w[1], so[1]);
    pa.dw_w = dw_w, pa.dw_scale_in = ed.scale_in, pa.dw_bias = ed.bias, pa.dw_p0 = ed.act_p0, pa.dw_lrelu = ed.lrelu;
    pa.dw_scale = dw_so, pa.dw_half = ed.round_half, pa.dw_nonneg = dw_mfma_epilogue(ed, gd.K) == EPI_I8_P8_NONNEG;
    const float both[2] = {dw_so, dw_so};
    pa.dw_qh = 0x007f007fu;
    if (pa.dw_nonneg) conv_pw_stream_clamps(ed.act_hi, ed.round_half, both, 2, &pa.dw_qh);
    const FastDiv hw = fast_div((unsigned)(g0.H * g0.W)), ow = fast_div((unsigned)g0.W);
    pa.hw_m = hw.m, pa.hw_s = hw.s, pa.ow_m = ow.m, pa.ow_s = ow.s;
    pa.HW = g0.H * g0.W, pa.OW = g0.W, pa.H = gd.H, pa.W = gd.W, pa.total_pix = (unsigned)g0.N * (unsigned)pa.HW;
    pa.in_bytes = (unsigned)((size_t)gd.N * gd.C * gd.H * gd.W);
    pa.sh = gd.sh, pa.sw = gd.sw, pa.ph = gd.ph, pa.pw = gd.pw, pa.dh = gd.dh, pa.dw = gd.dw, pa.C8 = gd.C / 8;
    float cost = 0;
    const int plan = force ? force : dwpw_plan(gd, g0, e0, g1, (uintptr_t)x % 8 == 0, &cost), groups = plan & 15, waves = plan & 16 ? 4 : 8;
    if (groups > waves) return hipErrorInvalidValue;
    if (groups != 1 && groups != 2 && groups != 4 && groups != 8) return hipErrorInvalidValue;
    DwPwStage st{};
    if (plan & 32) st = dwpw_staged(gd, groups);
    if ((plan & 32) && (!st.pitch || (uintptr_t)x % 8)) return hipErrorInvalidValue;
    const FastDiv image = fast_div(st.image);
    st.image_m = image.m, st.image_s = image.s;
    pa.between = (unsigned)dwpw_between(gd, g1, groups, st);
    const size_t lds = dwpw_lds_bytes(gd, g0, g1, groups, st);
    if (lds > 65536) return hipErrorInvalidValue;
    pa.first_pack = e0.join ? (unsigned)e0.join->sh_pack0 : 8u;
    pa.lg = groups == 1 ? 0 : groups == 2 ? 1 : groups == 4 ? 2 : 3;
    pa.tiles = (int)((pa.total_pix + 16 * groups - 1) / (16 * groups));
    const int next = !g1 ? (int)DP_NONE : pa.l[1].kind == PP_NONNEG && e1->so_full ? (int)DP_FULL : pa.l[1].kind;
    if (next == DP_FULL) pa.l[1].scale += pa.l[1].scale;
    const bool dfull = pa.dw_nonneg && ed.so_full;
    if (dfull) pa.dw_scale += pa.dw_scale;
    const bool shuffle = e0.join && e0.join->other;
#define OHIP_DP(T_, E_, N_) return launch_dwpw<T_, E_, N_>(waves, dfull, x, out, sum, pa, st, e0, lds, stream)
#define OHIP_DPN(T_, E_)                             \
    do {                                             \
        if (next == PP_I8) OHIP_DP(T_, E_, PP_I8);   \
        if (next == PP_NONNEG) OHIP_DP(T_, E_, PP_NONNEG); \
        if (next == DP_FULL) OHIP_DP(T_, E_, DP_FULL); \
        if (next == PP_F32) OHIP_DP(T_, E_, PP_F32); \
    } while (0)
    if (gd.kh == 3) {
        if (shuffle) {
            OHIP_DPN(9, EPI_F32_SHUFFLE);
            OHIP_DP(9, EPI_F32_SHUFFLE, DP_NONE);
        }
        if (e0.join) OHIP_DP(9, EPI_F32_P4_PARTS, DP_NONE);
        if (pa.l[0].kind == PP_F32) {
            OHIP_DPN(9, EPI_F32_P4_FUSED);
            OHIP_DP(9, EPI_F32_P4_FUSED, DP_NONE);
        }
        OHIP_DPN(9, EPI_I8_P8);
        OHIP_DP(9, EPI_I8_P8, DP_NONE);
    }
    if (e0.join) OHIP_DP(25, EPI_F32_P4_PARTS, DP_NONE);
    if (pa.l[0].kind == PP_F32) OHIP_DP(25, EPI_F32_P4_FUSED, DP_NONE);
    OHIP_DPN(25, EPI_I8_P8);
    OHIP_DP(25, EPI_I8_P8, DP_NONE);
#undef OHIP_DPN
#undef OHIP_DP
}

}  // namespace ohip
