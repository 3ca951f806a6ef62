// Pointwise (1x1, stride 1) int8 convolution with every operand in registers and no loop over the reduction. Up to 256 input channels
// (conv_pw_reg_kernel) that is a wave's own work, without LDS or a barrier; up to 1024 (conv_pw_split_kernel) the four waves of a
// workgroup share it, and their sums meet in LDS.
//
// The pointwise layers of a network are short: a wave's whole reduction is CG <= 4 matrix steps, and what their launches cost is
// the instructions around those and the latency of the first loads. On 88 -> 88 @52x52 x16 with LeakyReLU the implicit-GEMM kernel issues
// 1.6 million vector and 1.4 million scalar instructions for 43 000 matrix ones (its tap and column arithmetic, divisions, the way
// through LDS, 64-bit addresses), this one 0.87 and 0.40 million, in 9300 cycles instead of 13700. Here
//  * a wave owns FN groups of 16 consecutive pixels (of the whole batch) and requests all their channels at once: the octets of a
//    reduction step differ by a uniform offset, so a load is one instruction with no address arithmetic;
//  * it walks `per` pairs of 16-row tiles of the output channels. The weights of a pair are refilled in place behind its last
//    multiplication, its constants (and the elements of an addend) are requested one pair ahead;
//  * the pixels of an XCD's workgroups are one contiguous run of the batch, the same for every slice of the output channels, so that
//    a layer finds in its L2 what the layer before it wrote there.
// Epilogues: int8 Byte8 and fp32 Float4 results, the latter with the addend, the int8 twin and the shuffle of the implicit-GEMM
// kernel (common.hpp).
#include "common.hpp"
#include "conv_igemm.hpp"
#include "conv_pw_common.hpp"

#include <algorithm>
#include <cmath>

namespace ohip {

namespace {

// What these kernels read of a layer. Launch arguments are written to device memory one by one: on the host a launch with 32 bytes
// of them takes 3.1 us, with 96 3.35, with 180 (ConvGeom and Epilogue as they are) 3.85, and such a layer's kernel is done in less.
struct PwRegArgs {
    const float *scale_in, *bias;
    unsigned hw_m, total_pix;    // hw_m, hw_s: division by HW (FastDiv)
    int HW, K, tiles, per, mt;   // tiles: workgroups along the pixels; mt: 16-row tiles of the packed weights per step
    unsigned short C8;
    unsigned char hw_s, lrelu;
    float p0;                    // slope of LeakyReLU
    float scale, half;           // int8 result: the output scale of every channel (EPI_I8_P8_FULL: doubled), the rounding constant; fp32: act_lo, act_hi
    unsigned qh;                 // upper clamp of the rounded result, in both halves (EPI_I8_P8_NONNEG)

    __device__ FastDiv hw() const { return {hw_m, hw_s, (unsigned)HW}; }
};
template <int EPI>
__device__ __forceinline__ Epilogue pw_epilogue(const PwRegArgs& pa, const PwAdd<EPI>& ja) {
    constexpr bool I8 = epi_is_i8(EPI);
    Epilogue ep{};
    ep.lrelu = pa.lrelu != 0, ep.act_p0 = pa.p0;
    if (I8) ep.round_half = pa.half;
    else ep.act_lo = pa.scale, ep.act_hi = pa.half;
    if constexpr (!I8 && EPI != EPI_F32_P4) ep.twin_scale = ja.twin_scale, ep.twin_half = ja.twin_half;
    if constexpr (EPI == EPI_F32_P4_FUSED || EPI == EPI_F32_P4_PARTS) ep.residual = ja.residual, ep.twin = ja.twin;
    return ep;
}

}  // namespace

template <int FN, int CG, int EPI>
__global__ void __launch_bounds__(256) conv_pw_reg_kernel(const int8_t* __restrict__ x, const int8_t* __restrict__ wpk, void* __restrict__ out,
                                                          PwRegArgs pa, PwAdd<EPI> ja) {
    constexpr bool I8 = epi_is_i8(EPI), NONNEG = epi_clamp(EPI) != 0;
    constexpr bool SHUF = EPI == EPI_F32_SHUFFLE, PARTS = EPI == EPI_F32_P4_PARTS, FUSED = EPI == EPI_F32_P4_FUSED || PARTS, SLICE = EPI == EPI_F32_SLICE;
    constexpr bool ADD = SHUF || FUSED;  // reads elements of another fp32 blob
    const Epilogue ep = pw_epilogue<EPI>(pa, ja);
    const unsigned lane = threadIdx.x & 63, q = lane >> 4, p = lane & 15;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int xcd = blockIdx.x & 7, first = xcd * pa.tiles >> 3, tile = first + (int)(blockIdx.x >> 3);  // (grid.x is a multiple of 8)
    const unsigned gp0 = (unsigned)(tile * 4 + wave) * (16 * FN);
    if (tile >= (xcd + 1) * pa.tiles >> 3 || gp0 >= pa.total_pix) return;  // (uniform)
    const int pairs = (pa.K + 31) / 32, pr0 = blockIdx.y * pa.per, pr1 = min(pr0 + pa.per, pairs);
    const unsigned HW = pa.HW, K = pa.K, C8 = pa.C8;
    const unsigned kpad = (unsigned)pa.mt * 16u;

    // ---- weights and constants of a channel pair -------------------------------------------------------------------------------
    const __amdgpu_buffer_rsrc_t rw = rsrc(wpk, (unsigned)(CG * pa.mt) * 1024u);
    const __amdgpu_buffer_rsrc_t rsi = rsrc(pa.scale_in, kpad * 4), rbi = rsrc(pa.bias, kpad * 4);
    v4i a[CG][2];
    auto load_a = [&](int pr) {
#pragma unroll
        for (int cg = 0; cg < CG; ++cg)
#pragma unroll
            for (int h = 0; h < 2; ++h) a[cg][h] = load16(rw, lane * 16 + h * 1024, (unsigned)(cg * pa.mt + 2 * pr) * 1024u);
    };
    struct Pair {
        v4i si[2], bi[2];
        v4i add[ADD ? FN : 1][2];
    };

    load_a(pr0);

    // ---- the pixels: every channel of them requested now ---------------------------------------------------------------------------
    const __amdgpu_buffer_rsrc_t rin = rsrc(x, pa.total_pix * C8 * 8u);
    unsigned n[FN], pix[FN];
    bool ok[FN];
    v4i b[FN][CG];
#pragma unroll
    for (int j = 0; j < FN; ++j) {
        const unsigned gp = gp0 + 16 * j + p;
        ok[j] = gp < pa.total_pix;
        n[j] = div_by(gp, pa.hw()), pix[j] = gp - n[j] * HW;
        const unsigned v = ok[j] ? ((n[j] * C8 + 2 * q) * HW + pix[j]) * 8u : PR_OOB;
#pragma unroll
        for (int cg = 0; cg < CG; ++cg) {
            const bool last = cg == CG - 1;  // only the last step may end in octets that do not exist
            const v2i lo = load8(rin, !last || 8 * cg + 2 * q < C8 ? v : PR_OOB, (unsigned)cg * 64u * HW);
            const v2i hi = load8(rin, !last || 8 * cg + 2 * q + 1 < C8 ? v : PR_OOB, ((unsigned)cg * 64u + 8u) * HW);
            b[j][cg] = v4i{lo[0], lo[1], hi[0], hi[1]};
        }
    }

    // byte offset of (image, this lane's channels of a pair, pixel) in a blob of K channels: Byte8, Float4, Float8; a pair is 32 HW
    // (Byte8) or 128 HW (fp32) bytes further
    auto at_b8 = [&](int j) { return ((n[j] * (K / 8) + q) * HW + pix[j]) * 8u; };
    auto at_f4 = [&](int j) { return ((n[j] * (K / 4) + 2 * q) * HW + pix[j]) * 16u; };
    auto at_f8 = [&](int j) { return ((n[j] * (K / 8) + q) * HW + pix[j]) * 32u; };
    const unsigned f_bytes = pa.total_pix * K * 4u;
    unsigned vo[FN];
#pragma unroll
    for (int j = 0; j < FN; ++j) vo[j] = ok[j] ? (I8 ? at_b8(j) : at_f4(j)) : PR_OOB;

    auto load_pair = [&](Pair& k, int pr) {
        const unsigned s = (unsigned)pr * 128u;
#pragma unroll
        for (int h = 0; h < 2; ++h)
            k.si[h] = load16(rsi, q * 32 + h * 16, s), k.bi[h] = load16(rbi, q * 32 + h * 16, s);
        if constexpr (SHUF) {
            const __amdgpu_buffer_rsrc_t r = rsrc(ja.other, f_bytes);
            const bool live = 32u * pr + 8 * q < K;
#pragma unroll
            for (int j = 0; j < FN; ++j) {
                const unsigned v = ok[j] && live ? (ja.other_pack == 8 ? at_f8(j) : at_f4(j)) : PR_OOB;  // (uniform choice)
                k.add[j][0] = load16(r, v, s * HW);
                k.add[j][1] = load16(r, v, s * HW + (ja.other_pack == 8 ? 16u : HW * 16u));
            }
        }
        if constexpr (PARTS) {
#pragma unroll
            for (int j = 0; j < FN; ++j)
                if (ok[j] && 32u * pr + 8 * q < K)
#pragma unroll
                    for (int h = 0; h < 2; ++h)
                        k.add[j][h] = *reinterpret_cast<const v4i*>(epi4_residual_at(ep, ja.join(), n[j], pix[j], (int)(32u * pr + 8 * q + 4 * h), (int)K, (int)HW));
        } else if constexpr (FUSED) {
            if (ep.residual != nullptr) {  // (uniform)
                const __amdgpu_buffer_rsrc_t r = rsrc(ep.residual, f_bytes);
#pragma unroll
                for (int j = 0; j < FN; ++j)
#pragma unroll
                    for (int h = 0; h < 2; ++h) k.add[j][h] = load16(r, 32u * pr + 8 * q + 4 * h < K ? vo[j] : PR_OOB, s * HW + h * HW * 16u);
            }
        }
    };

    const __amdgpu_buffer_rsrc_t rout = rsrc(out, I8 ? pa.total_pix * K : f_bytes);
    auto finish = [&](const Pair& k, int pr, v4i (&c0)[FN], v4i (&c1)[FN], auto lrelu_c) {
        constexpr bool LRELU = decltype(lrelu_c)::value;
        const unsigned ch0 = 32u * pr + 8 * q;
        float si[8], bi[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) si[e] = __int_as_float(k.si[e / 4][e % 4]), bi[e] = __int_as_float(k.bi[e / 4][e % 4]);
        if constexpr (I8) {
            Epi8 prm;
#pragma unroll
            for (int e = 0; e < 8; ++e) prm.si[e] = si[e], prm.bi[e] = bi[e], prm.so[e] = pa.scale;
#pragma unroll
            for (int e = 0; e < 4; ++e) prm.qh[e] = pa.qh;
#pragma unroll
            for (int j = 0; j < FN; ++j) {
                const int a8[8] = {c0[j][0], c0[j][1], c0[j][2], c0[j][3], c1[j][0], c1[j][1], c1[j][2], c1[j][3]};
                store8(rout, epi8_quant_i8p8<epi_clamp(EPI), LRELU ? 1 : 0>(ep, prm, a8), ch0 < K ? vo[j] : PR_OOB, (unsigned)pr * 32u * HW);
            }
        } else {
#pragma unroll
            for (int j = 0; j < FN; ++j) {
                v4i r[2] = {epi4_dequant_f32p4<LRELU>(ep, si, bi, c0[j][0], c0[j][1], c0[j][2], c0[j][3]),
                            epi4_dequant_f32p4<LRELU>(ep, si + 4, bi + 4, c1[j][0], c1[j][1], c1[j][2], c1[j][3])};
                if constexpr (SHUF) {
                    // with the same channels of the other blob these are channels 2 ch0 .. 2 ch0 + 15 of the shuffled one: two packs of 8
                    const unsigned half = K / 8;  // packs of 8 in each half
#pragma unroll
                    for (int w = 0; w < 2; ++w) {
                        float* const f = w ? ja.sh_out1 : ja.sh_out0;
                        int8_t* const b8 = w ? ja.sh_q1 : ja.sh_q0;
                        if (w ? 8u * pr + 8 <= half : 8u * pr >= half) continue;  // (uniform: none of the pair's packs is in this half)
#pragma unroll
                        for (int h = 0; h < 2; ++h) {
                            const v4i o = k.add[j][h];
                            const v4i even = ja.other_odd ? r[h] : o, odd = ja.other_odd ? o : r[h];  // (uniform)
                            const v4i lo = {even[0], odd[0], even[1], odd[1]}, hi = {even[2], odd[2], even[3], odd[3]};
                            const unsigned pack = ch0 / 4 + h - (w ? half : 0u);  // in this half; beyond it on either side: the other half's
                            const unsigned e = n[j] * ja.sh_image + (pack * HW + pix[j]) * 8u;
                            const bool live = ok[j] && pack < half;  // (a channel past the last one is a pack past the second half)
                            if (f != nullptr) {
                                const __amdgpu_buffer_rsrc_t rf = rsrc(f, PR_OOB);
                                store16(rf, lo, live ? e * 4u : PR_OOB, 0), store16(rf, hi, (live ? e * 4u : PR_OOB) + 16u, 0);
                            }
                            if (b8 != nullptr)
                                store8(rsrc(b8, PR_OOB), v2i{quantize4(lo, ep.twin_scale, ep.twin_half), quantize4(hi, ep.twin_scale, ep.twin_half)},
                                       live ? e : PR_OOB, 0);
                        }
                    }
                } else if constexpr (SLICE) {
                    if (ja.twin != nullptr)  // (uniform)
                        store8(rsrc(ja.twin, pa.total_pix * K), v2i{quantize4(r[0], ja.twin_scale, ja.twin_half), quantize4(r[1], ja.twin_scale, ja.twin_half)},
                               ok[j] && ch0 < K ? at_b8(j) : PR_OOB, (unsigned)pr * 32u * HW);
                    store8(rsrc(ja.slice, PR_OOB), v2i{quantize4(r[0], ja.slice_scale, ja.slice_half), quantize4(r[1], ja.slice_scale, ja.slice_half)},
                           ok[j] && ch0 < K ? ((n[j] * ja.octets + q) * HW + pix[j]) * 8u : PR_OOB, (unsigned)pr * 32u * HW);
                } else {
                    v2i tw;
#pragma unroll
                    for (int h = 0; h < 2; ++h) {
                        if constexpr (FUSED) {
                            if (PARTS || ep.residual != nullptr)
#pragma unroll
                                for (int e = 0; e < 4; ++e) r[h][e] = __float_as_int(__fadd_rn(__int_as_float(r[h][e]), __int_as_float(k.add[j][h][e])));
                            if (ep.twin != nullptr) tw[h] = quantize4(r[h], ep.twin_scale, ep.twin_half);
                        }
                        if (!FUSED || out != nullptr) store16(rout, r[h], ch0 + 4 * h < K ? vo[j] : PR_OOB, (unsigned)pr * 128u * HW + h * HW * 16u);
                    }
                    if constexpr (FUSED)
                        if (ep.twin != nullptr)  // K % 8 == 0 then: the lane's 8 channels are one Byte8 element
                            store8(rsrc(ep.twin, pa.total_pix * K), tw, ok[j] && ch0 < K ? at_b8(j) : PR_OOB, (unsigned)pr * 32u * HW);
                }
            }
        }
    };
    auto step = [&](const Pair& k, Pair& next, int pr) {
        if (pr + 1 < pr1) load_pair(next, pr + 1);
        v4i c0[FN], c1[FN];
#pragma unroll
        for (int cg = 0; cg < CG; ++cg)
#pragma unroll
            for (int j = 0; j < FN; ++j) {
                c0[j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[cg][0], b[j][cg], cg ? c0[j] : v4i{0, 0, 0, 0}, 0, 0, 0);
                c1[j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[cg][1], b[j][cg], cg ? c1[j] : v4i{0, 0, 0, 0}, 0, 0, 0);
            }
        if (pr + 1 < pr1) load_a(pr + 1);
        if (!NONNEG && ep.lrelu) finish(k, pr, c0, c1, std::true_type{});  // (uniform)
        else finish(k, pr, c0, c1, std::false_type{});
    };
    Pair k0, k1;
    load_pair(k0, pr0);
    for (int pr = pr0;;) {
        step(k0, k1, pr);
        if (++pr >= pr1) break;
        step(k1, k0, pr);
        if (++pr >= pr1) break;
    }
}

// The same for longer reductions (up to 64 PW_REG_STEPS_SPLIT input channels): the four waves of a workgroup own the same pixels and
// take every fourth reduction step each, NS at most. Per channel pair their partial sums meet in LDS (integers: the same in any
// order), and each wave finishes the half pairs (four channels of a lane's pixel) that are its own. One barrier per pair: the
// sums of consecutive pairs lie in two buffers.
template <int FN, int NS, int EPI>
__global__ void __launch_bounds__(256) conv_pw_split_kernel(const int8_t* __restrict__ x, const int8_t* __restrict__ wpk, void* __restrict__ out,
                                                            PwRegArgs pa, PwAdd<EPI> ja) {
    constexpr bool I8 = epi_is_i8(EPI), NONNEG = epi_clamp(EPI) != 0;
    constexpr bool SHUF = EPI == EPI_F32_SHUFFLE, PARTS = EPI == EPI_F32_P4_PARTS, FUSED = EPI == EPI_F32_P4_FUSED || PARTS, SLICE = EPI == EPI_F32_SLICE;
    constexpr int OWN = FN < 2 ? 1 : FN / 2;  // half pairs that a wave finishes (of 2 FN; with FN == 1 waves 0 and 1 have one each)
    __shared__ v4i red[2][2 * FN][3][64];     // [buffer][half pair][the other waves][lane]
    const Epilogue ep = pw_epilogue<EPI>(pa, ja);
    const unsigned lane = threadIdx.x & 63, q = lane >> 4, p = lane & 15;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int xcd = blockIdx.x & 7, first = xcd * pa.tiles >> 3, tile = first + (int)(blockIdx.x >> 3);  // (grid.x is a multiple of 8)
    if (tile >= (xcd + 1) * pa.tiles >> 3) return;  // (uniform over the workgroup)
    const int pairs = (pa.K + 31) / 32, pr0 = blockIdx.y * pa.per, pr1 = min(pr0 + pa.per, pairs), steps = (pa.C8 + 7) / 8;
    const unsigned HW = pa.HW, K = pa.K, C8 = pa.C8, kpad = (unsigned)pa.mt * 16u, f_bytes = pa.total_pix * K * 4u;

    const __amdgpu_buffer_rsrc_t rw = rsrc(wpk, (unsigned)(steps * pa.mt) * 1024u);
    const __amdgpu_buffer_rsrc_t rsi = rsrc(pa.scale_in, kpad * 4), rbi = rsrc(pa.bias, kpad * 4);
    v4i a[NS][2];
    auto load_a = [&](int pr) {
#pragma unroll
        for (int i = 0; i < NS; ++i) {
            const int s = wave + 4 * i;
            if (i < NS - 1 || s < steps)  // (uniform; only a wave's last step may not exist)
#pragma unroll
                for (int h = 0; h < 2; ++h) a[i][h] = load16(rw, lane * 16 + h * 1024, (unsigned)(s * pa.mt + 2 * pr) * 1024u);
        }
    };
    load_a(pr0);

    const __amdgpu_buffer_rsrc_t rin = rsrc(x, pa.total_pix * C8 * 8u);
    unsigned n[FN], pix[FN];
    bool ok[FN];
    v4i b[FN][NS];
#pragma unroll
    for (int j = 0; j < FN; ++j) {
        const unsigned gp = (unsigned)tile * (16 * FN) + 16 * j + p;
        ok[j] = gp < pa.total_pix;
        n[j] = div_by(gp, pa.hw()), pix[j] = gp - n[j] * HW;
        const unsigned v = ok[j] ? ((n[j] * C8 + 2 * q) * HW + pix[j]) * 8u : PR_OOB;
#pragma unroll
        for (int i = 0; i < NS; ++i) {
            const unsigned s = (unsigned)(wave + 4 * i);
            if (i < NS - 1 || (int)s < steps) {  // (uniform) the last one may end in octets that do not exist
                const v2i lo = load8(rin, 8 * s + 2 * q < C8 ? v : PR_OOB, s * 64u * HW);
                const v2i hi = load8(rin, 8 * s + 2 * q + 1 < C8 ? v : PR_OOB, (s * 64u + 8u) * HW);
                b[j][i] = v4i{lo[0], lo[1], hi[0], hi[1]};
            } else {
                b[j][i] = v4i{0, 0, 0, 0}, a[i][0] = a[i][1] = v4i{0, 0, 0, 0};
            }
        }
    }
    // this wave's half pairs: pixel group jo[o], channels 4 h .. 4 h + 3 of a lane's eight
    const bool finishes = FN > 1 || wave < 2;  // (uniform)
    struct Half {
        v4i si, bi, add[OWN];
    };
    const unsigned h = wave & 1;
    unsigned vo[OWN];  // byte offset of the half pair's element in the result; a pair is 32 HW (Byte8) or 128 HW (fp32) bytes further
    unsigned no[OWN], po[OWN];
    bool oko[OWN];
#pragma unroll
    for (int o = 0; o < OWN; ++o) {
        const int jo = FN == 1 ? 0 : (wave >> 1) + 2 * o;
        // (selected without an index into registers)
        no[o] = n[0], po[o] = pix[0], oko[o] = ok[0];
#pragma unroll
        for (int j = 1; j < FN; ++j)
            if (j == jo) no[o] = n[j], po[o] = pix[j], oko[o] = ok[j];
        vo[o] = !oko[o] ? PR_OOB : I8 ? ((no[o] * (K / 8) + q) * HW + po[o]) * 8u + 4 * h : ((no[o] * (K / 4) + 2 * q + h) * HW + po[o]) * 16u;
    }
    auto load_half = [&](Half& k, int pr) {
        const unsigned s = (unsigned)pr * 128u, ch = 32u * pr + 8 * q + 4 * h;
        k.si = load16(rsi, q * 32 + h * 16, s), k.bi = load16(rbi, q * 32 + h * 16, s);
#pragma unroll
        for (int o = 0; o < OWN; ++o) {
            if constexpr (SHUF) {
                const unsigned v = ja.other_pack == 8 ? ((no[o] * (K / 8) + q) * HW + po[o]) * 32u + 16 * h : vo[o];  // (uniform choice)
                k.add[o] = load16(rsrc(ja.other, f_bytes), oko[o] && ch < K ? v : PR_OOB, s * HW);
            }
            if constexpr (PARTS) {
                if (oko[o] && ch < K) k.add[o] = *reinterpret_cast<const v4i*>(epi4_residual_at(ep, ja.join(), no[o], po[o], (int)ch, (int)K, (int)HW));
            } else if constexpr (FUSED) {
                if (ep.residual != nullptr) k.add[o] = load16(rsrc(ep.residual, f_bytes), ch < K ? vo[o] : PR_OOB, s * HW);  // (uniform)
            }
        }
    };
    const __amdgpu_buffer_rsrc_t rout = rsrc(out, I8 ? pa.total_pix * K : f_bytes);
    auto finish = [&](const Half& k, int pr, const v4i (&c)[OWN], auto lrelu_c) {
        constexpr bool LRELU = decltype(lrelu_c)::value;
        const unsigned ch = 32u * pr + 8 * q + 4 * h;
#pragma unroll
        for (int o = 0; o < OWN; ++o) {
            if constexpr (I8) {
                const v4i so = v4i{1, 1, 1, 1} * __float_as_int(pa.scale);
                const unsigned w = dw_requant4<epi_clamp(EPI), LRELU ? 1 : 0>(ep, c[o], k.si, k.bi, so, pa.qh, pa.qh);
                __builtin_amdgcn_raw_buffer_store_b32(w, rout, (int)(ch < K ? vo[o] : PR_OOB), (int)((unsigned)pr * 32u * HW), 0);
                continue;
            }
            float si[4], bi[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) si[e] = __int_as_float(k.si[e]), bi[e] = __int_as_float(k.bi[e]);
            v4i r = LRELU || ((SHUF || FUSED) && ep.lrelu) ? epi4_dequant_f32p4<true>(ep, si, bi, c[o][0], c[o][1], c[o][2], c[o][3])
                                              : epi4_dequant_f32p4<false>(ep, si, bi, c[o][0], c[o][1], c[o][2], c[o][3]);
            if constexpr (SHUF) {
                // with the same channels of the other blob these are channels 2 ch .. 2 ch + 7 of the shuffled one: a pack of 8
                const v4i even = ja.other_odd ? r : k.add[o], odd = ja.other_odd ? k.add[o] : r;  // (uniform)
                const v4i lo = {even[0], odd[0], even[1], odd[1]}, hi = {even[2], odd[2], even[3], odd[3]};
                const unsigned half = K / 8;  // packs of 8 in each half of the 2 K channels
#pragma unroll
                for (int w = 0; w < 2; ++w) {
                    float* const f = w ? ja.sh_out1 : ja.sh_out0;
                    int8_t* const b8 = w ? ja.sh_q1 : ja.sh_q0;
                    const unsigned pack = ch / 4 - (w ? half : 0u);  // beyond this half on either side: the other half's
                    const unsigned e = no[o] * ja.sh_image + (pack * HW + po[o]) * 8u;
                    const bool live = oko[o] && pack < half;
                    if (f != nullptr) {
                        const __amdgpu_buffer_rsrc_t rf = rsrc(f, PR_OOB);
                        store16(rf, lo, live ? e * 4u : PR_OOB, 0), store16(rf, hi, (live ? e * 4u : PR_OOB) + 16u, 0);
                    }
                    if (b8 != nullptr)
                        store8(rsrc(b8, PR_OOB), v2i{quantize4(lo, ep.twin_scale, ep.twin_half), quantize4(hi, ep.twin_scale, ep.twin_half)},
                               live ? e : PR_OOB, 0);
                }
            } else if constexpr (SLICE) {
                const bool live = oko[o] && ch < K;
                if (ja.twin != nullptr)  // (uniform)
                    __builtin_amdgcn_raw_buffer_store_b32((unsigned)quantize4(r, ja.twin_scale, ja.twin_half), rsrc(ja.twin, pa.total_pix * K),
                                                          (int)(live ? ((no[o] * (K / 8) + q) * HW + po[o]) * 8u + 4 * h : PR_OOB), (int)((unsigned)pr * 32u * HW), 0);
                __builtin_amdgcn_raw_buffer_store_b32((unsigned)quantize4(r, ja.slice_scale, ja.slice_half), rsrc(ja.slice, PR_OOB),
                                                      (int)(live ? ((no[o] * ja.octets + q) * HW + po[o]) * 8u + 4 * h : PR_OOB), (int)((unsigned)pr * 32u * HW), 0);
            } else {
                if constexpr (FUSED)
                    if (PARTS || ep.residual != nullptr)
#pragma unroll
                        for (int e = 0; e < 4; ++e) r[e] = __float_as_int(__fadd_rn(__int_as_float(r[e]), __int_as_float(k.add[o][e])));
                if (!FUSED || out != nullptr) store16(rout, r, ch < K ? vo[o] : PR_OOB, (unsigned)pr * 128u * HW);
                if constexpr (FUSED)
                    if (ep.twin != nullptr)
                        __builtin_amdgcn_raw_buffer_store_b32((unsigned)quantize4(r, ep.twin_scale, ep.twin_half), rsrc(ep.twin, pa.total_pix * K),
                                                              (int)(oko[o] && ch < K ? ((no[o] * (K / 8) + q) * HW + po[o]) * 8u + 4 * h : PR_OOB),
                                                              (int)((unsigned)pr * 32u * HW), 0);
            }
        }
    };
    Half k0, k1;
    if (finishes) load_half(k0, pr0);
    for (int pr = pr0; pr < pr1; ++pr) {
        v4i c[FN][2];
#pragma unroll
        for (int i = 0; i < NS; ++i)
#pragma unroll
            for (int j = 0; j < FN; ++j)
#pragma unroll
                for (int t = 0; t < 2; ++t) c[j][t] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[i][t], b[j][i], i ? c[j][t] : v4i{0, 0, 0, 0}, 0, 0, 0);
        if (pr + 1 < pr1) {
            load_a(pr + 1);
            if (finishes) load_half(k1, pr + 1);
        }
        // half pair u = 2 j + t belongs to wave (j % 2) * 2 + t (FN == 1: wave t)
        v4i own[OWN];
#pragma unroll
        for (int j = 0; j < FN; ++j)
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                const int w = FN == 1 ? t : (j & 1) * 2 + t;
                if (wave == w) own[j >> 1] = c[j][t];
                else red[pr & 1][2 * j + t][wave < w ? wave : wave - 1][lane] = c[j][t];
            }
        __syncthreads();
        if (finishes) {
#pragma unroll
            for (int o = 0; o < OWN; ++o) {
                const int u = FN == 1 ? wave : 2 * ((wave >> 1) + 2 * o) + (wave & 1);
#pragma unroll
                for (int i = 0; i < 3; ++i) own[o] += red[pr & 1][u][i][lane];
            }
            // (uniform. Not where another blob's elements are on their way: they would be waited for in front of the branch, 12.5 -> 14.1 us
            // for 960 -> 160 on 17 25x35 images)
            if (!NONNEG && !SHUF && !FUSED && ep.lrelu) finish(k0, pr, own, std::true_type{});
            else finish(k0, pr, own, std::false_type{});
            k0 = k1;
        }
    }
}

// ---------------------------------------------------------------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------------------------------------------------------------

static int pw_reg_epilogue(const Epilogue& ep, int K) {
    const int epi = pick_epilogue(ep, K);
    if (epi != EPI_F32_P4 || !ep.fused()) return epi;
    if (ep.join != nullptr && ep.join->slice != nullptr) return EPI_F32_SLICE;
    return ep.join == nullptr ? EPI_F32_P4_FUSED : ep.join->other != nullptr ? EPI_F32_SHUFFLE : EPI_F32_P4_PARTS;
}

bool conv_pw_reg_applicable(const ConvGeom& g, const Epilogue& ep) {
    if (g.groups != 1 || g.kh != 1 || g.kw != 1 || g.sh != 1 || g.sw != 1 || g.ph != 0 || g.pw != 0) return false;
    if (g.C % 8 || g.C > 64 * PW_REG_STEPS_SPLIT || g.N < 1) return false;
    const int epi = pw_reg_epilogue(ep, g.K);
    if (epi == EPI_GENERIC || ((ep.twin != nullptr || ep.join != nullptr) && g.K % 8)) return false;
    const size_t px = (size_t)g.N * g.H * g.W;
    if ((size_t)igemm_channel_groups(g.C) * igemm_padded_rows(g.K) * 64 >= ((size_t)1 << 31)) return false;  // (the packed weights)
    // 32-bit byte offsets into every blob; a shuffled result that is one blob has twice the layer's channels
    const size_t joined = epi == EPI_F32_SHUFFLE && ep.join->sh_image > (size_t)g.K * g.H * g.W ? 2 : 1;
    if (epi == EPI_F32_SLICE && (ep.residual || px * ep.join->slice_octets * 8 >= ((size_t)1 << 31))) return false;
    return px * g.C < ((size_t)1 << 31) && px * g.K * joined * layout_elem_bytes(ep.out_layout) < ((size_t)1 << 31);
}

template <int FN, int CG, int EPI>
static hipError_t launch_pw_reg(const int8_t* x, const int8_t* wpk, void* out, const PwRegArgs& pa, const Epilogue& ep, int slices,
                                hipStream_t stream) {
    launch((conv_pw_reg_kernel<FN, CG, EPI>), dim3((pa.tiles + 7) / 8 * 8, slices), dim3(256), 0, stream, x, wpk, out, pa,
                       PwAdd<EPI>::of(ep));
    return hipGetLastError();
}

template <int FN, int CG>
static hipError_t launch_pw_reg_e(int epi, const int8_t* x, const int8_t* wpk, void* out, const PwRegArgs& pa, const Epilogue& ep, int slices,
                                  hipStream_t stream) {
    switch (epi) {
    case EPI_I8_P8: return launch_pw_reg<FN, CG, EPI_I8_P8>(x, wpk, out, pa, ep, slices, stream);
    case EPI_I8_P8_NONNEG: return launch_pw_reg<FN, CG, EPI_I8_P8_NONNEG>(x, wpk, out, pa, ep, slices, stream);
    case EPI_I8_P8_FULL: return launch_pw_reg<FN, CG, EPI_I8_P8_FULL>(x, wpk, out, pa, ep, slices, stream);
    case EPI_F32_P4: return launch_pw_reg<FN, CG, EPI_F32_P4>(x, wpk, out, pa, ep, slices, stream);
    case EPI_F32_P4_FUSED: return launch_pw_reg<FN, CG, EPI_F32_P4_FUSED>(x, wpk, out, pa, ep, slices, stream);
    case EPI_F32_SHUFFLE: return launch_pw_reg<FN, CG, EPI_F32_SHUFFLE>(x, wpk, out, pa, ep, slices, stream);
    case EPI_F32_P4_PARTS: return launch_pw_reg<FN, CG, EPI_F32_P4_PARTS>(x, wpk, out, pa, ep, slices, stream);
    case EPI_F32_SLICE: return launch_pw_reg<FN, CG, EPI_F32_SLICE>(x, wpk, out, pa, ep, slices, stream);
    }
    return hipErrorInvalidValue;
}

template <int CG>
static hipError_t launch_pw_reg_wide(int epi, const int8_t* x, const int8_t* wpk, void* out, const PwRegArgs& pa, const Epilogue& ep, int slices,
                                     hipStream_t stream) {
    switch (epi) {
    case EPI_I8_P8: return launch_pw_reg<4, CG, EPI_I8_P8>(x, wpk, out, pa, ep, slices, stream);
    case EPI_I8_P8_NONNEG: return launch_pw_reg<4, CG, EPI_I8_P8_NONNEG>(x, wpk, out, pa, ep, slices, stream);
    case EPI_I8_P8_FULL: return launch_pw_reg<4, CG, EPI_I8_P8_FULL>(x, wpk, out, pa, ep, slices, stream);
    case EPI_F32_P4: return launch_pw_reg<4, CG, EPI_F32_P4>(x, wpk, out, pa, ep, slices, stream);
    }
    return hipErrorInvalidValue;
}

template <int FN, int NS, int EPI>
static hipError_t launch_pw_split(const int8_t* x, const int8_t* wpk, void* out, const PwRegArgs& pa, const Epilogue& ep, int slices,
                                  hipStream_t stream) {
    launch((conv_pw_split_kernel<FN, NS, EPI>), dim3((pa.tiles + 7) / 8 * 8, slices), dim3(256), 0, stream, x, wpk, out, pa,
                       PwAdd<EPI>::of(ep));
    return hipGetLastError();
}

template <int FN, int NS>
static hipError_t launch_pw_split_e(int epi, const int8_t* x, const int8_t* wpk, void* out, const PwRegArgs& pa, const Epilogue& ep, int slices,
                                    hipStream_t stream) {
    switch (epi) {
    case EPI_I8_P8: return launch_pw_split<FN, NS, EPI_I8_P8>(x, wpk, out, pa, ep, slices, stream);
    case EPI_I8_P8_NONNEG: return launch_pw_split<FN, NS, EPI_I8_P8_NONNEG>(x, wpk, out, pa, ep, slices, stream);
    case EPI_I8_P8_FULL: return launch_pw_split<FN, NS, EPI_I8_P8_FULL>(x, wpk, out, pa, ep, slices, stream);
    case EPI_F32_P4: return launch_pw_split<FN, NS, EPI_F32_P4>(x, wpk, out, pa, ep, slices, stream);
    case EPI_F32_P4_FUSED: return launch_pw_split<FN, NS, EPI_F32_P4_FUSED>(x, wpk, out, pa, ep, slices, stream);
    case EPI_F32_SHUFFLE: return launch_pw_split<FN, NS, EPI_F32_SHUFFLE>(x, wpk, out, pa, ep, slices, stream);
    case EPI_F32_P4_PARTS: return launch_pw_split<FN, NS, EPI_F32_P4_PARTS>(x, wpk, out, pa, ep, slices, stream);
    case EPI_F32_SLICE: return launch_pw_split<FN, NS, EPI_F32_SLICE>(x, wpk, out, pa, ep, slices, stream);
    }
    return hipErrorInvalidValue;
}

// so: the output scale of every channel (int8 results); force: 0 = automatic, else pixel groups | 64 if the reduction is split | pairs per wave << 7
hipError_t run_conv_pw_reg(const int8_t* x, const int8_t* wpk, float so, void* out, const ConvGeom& g, const Epilogue& ep, int force,
                           hipStream_t stream) {
    if (!conv_pw_reg_applicable(g, ep)) return hipErrorInvalidValue;
    const int epi = pw_reg_epilogue(ep, g.K), steps = igemm_channel_groups(g.C), pairs = (g.K + 31) / 32;
    const FastDiv hw = fast_div((unsigned)(g.H * g.W));
    const bool i8 = epi == EPI_I8_P8 || epi == EPI_I8_P8_NONNEG;
    PwRegArgs pa{};
    pa.scale_in = ep.scale_in, pa.bias = ep.bias, pa.hw_m = hw.m, pa.hw_s = (unsigned char)hw.s, pa.HW = g.H * g.W, pa.K = g.K;
    pa.total_pix = (unsigned)g.N * (unsigned)pa.HW, pa.C8 = (unsigned short)(g.C / 8), pa.mt = igemm_padded_rows(g.K) / 16;
    pa.lrelu = ep.lrelu, pa.p0 = ep.act_p0, pa.scale = i8 ? so : ep.act_lo, pa.half = i8 ? ep.round_half : ep.act_hi;
    const float both[2] = {so, so};
    if (epi == EPI_I8_P8_NONNEG) conv_pw_stream_clamps(ep.act_hi, ep.round_half, both, 2, &pa.qh);
    const int instance = full_epilogue(epi, ep);
    if (instance == EPI_I8_P8_FULL) pa.scale = so + so;
    int fn = 1, per = 1;
    const bool split = force ? (force & 64) != 0 : steps > PW_REG_STEPS;
    const bool wide = split || epi == EPI_F32_P4 || epi == EPI_I8_P8 || epi == EPI_I8_P8_NONNEG;  // (registers)
    constexpr long kClampedFrom = 4l << 20;  // results of a layer, see conv_pw_reg_plan_clamped
    if (epi == EPI_I8_P8_NONNEG && !split && (long)pa.total_pix * g.K >= kClampedFrom) conv_pw_reg_plan_clamped(g, &fn, &per);
    else conv_pw_reg_plan(g, split, wide ? 4 : 2, layout_elem_bytes(ep.out_layout) == 4, &fn, &per);
    per = std::max(per, (pairs + 65534) / 65535);  // (slices are grid.y)
    if (force) fn = force & 7, per = force >> 7;
    if ((fn != 1 && fn != 2 && !(fn == 4 && wide)) || per < 1 || (split ? steps < 2 : steps > PW_REG_STEPS)) return hipErrorInvalidValue;
    per = std::min(per, pairs);
    const unsigned wg_pix = (split ? 16u : 64u) * (unsigned)fn;
    pa.per = per, pa.tiles = (int)((pa.total_pix + wg_pix - 1) / wg_pix);
    const int slices = (pairs + per - 1) / per;
    if (slices > 65535) return hipErrorInvalidValue;
    if (split) {
#define OHIP_PWS(NS_)                                                                                             \
    if ((steps + 3) / 4 == NS_) return fn == 1   ? launch_pw_split_e<1, NS_>(instance, x, wpk, out, pa, ep, slices, stream) \
                                       : fn == 2 ? launch_pw_split_e<2, NS_>(instance, x, wpk, out, pa, ep, slices, stream) \
                                                 : launch_pw_split_e<4, NS_>(instance, x, wpk, out, pa, ep, slices, stream);
        OHIP_PWS(1)
        OHIP_PWS(2)
        OHIP_PWS(3)
        OHIP_PWS(4)
#undef OHIP_PWS
        return hipErrorInvalidValue;
    }
#define OHIP_PWR(CG_)                                                                                      \
    if (steps == CG_ && fn == 4) return launch_pw_reg_wide<CG_>(instance, x, wpk, out, pa, ep, slices, stream); \
    if (steps == CG_) return fn == 1 ? launch_pw_reg_e<1, CG_>(instance, x, wpk, out, pa, ep, slices, stream)    \
                                     : launch_pw_reg_e<2, CG_>(instance, x, wpk, out, pa, ep, slices, stream);
    OHIP_PWR(1)
    OHIP_PWR(2)
    OHIP_PWR(3)
    OHIP_PWR(4)
#undef OHIP_PWR
    return hipErrorInvalidValue;
}

// Pixel groups of a wave (1, 2 or 4) and channel pairs that it walks. A pair costs a wave `pair` microseconds of latency whatever
// else runs, a launch the cycles of its waves' loads and stores on the address unit of a compute unit (ta) and of their vector
// instructions (va). More pairs per wave share the loads of the pixels and the prologue (once): with the pairs cut into slices the
// sum is least at the square root below.
// Whole reductions (at most 256 channels): fitted to 150 drawn layers of 16 .. 384 channels, 49 to 800 000 pixels, 2.7 % above the
// best measured split on average, 80 % of the time of the launches before (streamed, implicit GEMM, dealt reduction; the faster
// by their cost models). Split reductions: 138 layers of 257 .. 960 channels, 2.3 % above the best, 85 % of the best of the
// implicit-GEMM kernel and every tile of the dealt reduction. The line between the two is at 256 channels (PW_REG_STEPS): 257 .. 384
// channels, for which whole reductions were built then, are 5 % faster split, 193 .. 256 2 % and up to 192 8 % slower.
void conv_pw_reg_plan(const ConvGeom& g, bool split, int max_groups, bool f32out, int* groups, int* per) {
    const int pairs = (g.K + 31) / 32, cg = igemm_channel_groups(g.C);
    const float px = (float)g.N * (float)g.H * (float)g.W;
    float best = __builtin_inff();
    for (int fn = 1; fn <= max_groups; fn *= 2) {
        const float f = (float)fn, c = (float)cg;
        const float waves = px / (4096.f * f) * (split ? 16.f : 1.f);  // per compute unit (split: workgroups)
        const float pair = split ? 0.11f + 0.203f * f + 0.051f * c : 0.008f + 0.296f * f + 0.017f * c;
        const float once = (split ? 0.27f * f * c + 142.f : 14.9f * f * c + 24.2f) / 2300.f;
        const int want = std::clamp((int)(sqrtf(waves * (float)pairs * once / pair) + 0.5f), 1, pairs);
        const int slices = (pairs + want - 1) / want, p = (pairs + slices - 1) / slices;
        const float ta = 32.f * c + 64.f + f * (f32out ? 32.f : 8.f), va = 20.f + f * (f32out ? 36.f : 64.f);
        const float each = (split ? 0.017f * ta + 6.5f + 1.6f * f : 0.933f * ta + 0.404f * va) / 2300.f;
        const float t = (float)p * pair + (split ? 1.21f * f : 0.f) + waves * (float)slices * (once + (float)p * each);
        if (t < best) best = t, *groups = fn, *per = p;
    }
}

// The same for a whole reduction with a clamped int8 result and many of them. Its requantization is two thirds of the others'
// instructions, so that a wave should walk more pairs of more pixels: by the costs above such layers, which the streamed kernel used to
// take, were up to 1.26 times slower than there (16 -> 96 @112x112 x64 26.4 us, streamed 22.0, now 21.5; 256 -> 512 @28x28 x32 12.4 a
// call, now 10.3). Per pair a wave's latency, per workgroup of a compute unit its share of the loads and instructions; of the last,
// incomplete round about half counts. Fitted to 498 drawn layers of 8 .. 256 channels with all splits (median error 3 %): the split
// named is 1.2 % above the best one, 5.5 % before. Against the streamed kernel over its own range, layers that were not fitted, of 2
// million results or more, or of 200 .. 256 channels and 20 000 pixels: 500 layers take 0.91 of its time, 9 % of them over 3 % more, 11 %
// at worst; 700 by the costs above 0.95, 22 % and 22 %. Below 4 million results the costs above lose to no launch of before; there these
// are level (1.00 of the time over 200 drawn layers, 13 of them over 3 % slower), above 0.98, 0.95 and 0.95 at 4, 8 and 16 million.
void conv_pw_reg_plan_clamped(const ConvGeom& g, int* groups, int* per) {
    const int pairs = (g.K + 31) / 32;
    const float c = (float)igemm_channel_groups(g.C);
    const long px = (long)g.N * g.H * g.W;
    float best = __builtin_inff();
    for (int fn = 1; fn <= 4; fn *= 2) {
        const float f = (float)fn, pair = 0.066f + 0.083f * f + 0.02f * c, once = 0.017f + 0.065f * f * c, each = 0.1f + 0.059f * f + 0.049f * c;
        const long tiles = (px + 64 * fn - 1) / (64 * fn);
        // (slices of the pairs: the real optimum without rounds, and its neighbours)
        const int near = std::clamp((int)(sqrtf(pair * (float)pairs * 256.f / ((float)tiles * once)) + 0.5f), 1, pairs);
        for (int want = std::max(near - 1, 1); want <= std::min(near + 1, pairs); ++want) {
            const int p = (pairs + want - 1) / want, slices = (pairs + p - 1) / p;
            const long groups_all = tiles * slices;
            const float share = (float)groups_all / 256.f, rounds = (float)((groups_all + 255) / 256);
            const float t = (float)p * pair + 0.008f * f * c + (0.51f * share + 0.49f * rounds) * (once + (float)pairs / (float)slices * each);
            if (t < best) best = t, *groups = fn, *per = p;
        }
    }
}

}  // namespace ohip
