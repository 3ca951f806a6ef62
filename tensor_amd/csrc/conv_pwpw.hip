// Two pointwise layers in one launch, the second reading the int8 form of what the first leaves behind: its int8 result, or the
// quantization of the second half of the channels that a ChannelShuffle makes of its fp32 result and another blob (the last layer of
// a ShuffleNetV2 unit and the first of the next).
//
// In a network of small layers a launch of its own costs about 2 us whatever it computes, and the blob between the two layers is
// written and read back for nothing. A pixel of the second layer needs that pixel of the first and nothing else, so a workgroup owns
// 16 FN pixels with all their channels:
//  * it brings the first layer's input and the constants of both layers into LDS, a row per pixel (the pixels' operands are then one
//    16-byte LDS read each for every wave);
//  * its waves take the first layer's pairs of 16-row tiles in turn, weights straight from memory and requested one pair ahead, as in
//    conv_pw_reg.hip, with that kernel's epilogues; the bytes that the second layer reads go to LDS;
//  * behind a barrier they do the same for the second layer.
#include "common.hpp"
#include "conv_pwpw_common.hpp"

#include <algorithm>

namespace ohip {

namespace {

constexpr int PP_WAVES = 4;  // of a workgroup (eight: faster only at 13x13 and below, by 0.1 us)

struct PwPwArgs {
    PwPwLayer l[2];
    unsigned hw_m, total_pix;
    int HW, tiles;
    unsigned short C8;
    unsigned char hw_s;
};

}  // namespace

// EPI: the first layer's epilogue: EPI_I8_P8 or EPI_I8_P8_NONNEG (an int8 result, read by the second layer alone) or EPI_F32_SHUFFLE;
// KIND1: the second layer's result. SC: reduction steps whose weights a wave requests together. (Neither the kinds nor LeakyReLU are
// decided by a branch around the end of a pair: there the wave would wait for the next weights.)
template <int FN, int SC, int EPI, int KIND1>
__global__ void __launch_bounds__(64 * PP_WAVES) conv_pwpw_kernel(const int8_t* __restrict__ x, void* __restrict__ out, PwPwArgs pa, PwAdd<EPI> ja) {
    constexpr bool SHUF = EPI == EPI_F32_SHUFFLE, I8 = !SHUF;
    constexpr int NW = PP_WAVES;
    constexpr int PIX = 16 * FN, THREADS = 64 * NW;
    extern __shared__ __attribute__((aligned(16))) int8_t lds[];
    const unsigned tid = threadIdx.x, lane = tid & 63, q = lane >> 4, p = lane & 15;
    const int wave = __builtin_amdgcn_readfirstlane((int)tid >> 6);
    const int xcd = blockIdx.x & 7, tile = (xcd * pa.tiles >> 3) + (int)(blockIdx.x >> 3);  // (grid.x is a multiple of 8)
    if (tile >= (xcd + 1) * pa.tiles >> 3) return;  // (uniform)
    const PwPwLayer &l0 = pa.l[0], &l1 = pa.l[1];
    const unsigned HW = pa.HW, C8 = pa.C8, K0 = l0.K, rb0 = 64u * l0.steps + 16u, rb1 = 64u * l1.steps + 16u;  // bytes of a pixel's row
    const int pairs0 = (l0.K + 31) / 32, pairs1 = (l1.K + 31) / 32;
    int8_t *const px0 = lds, *const px1 = lds + PIX * rb0;
    float *const consts0 = reinterpret_cast<float*>(px1 + PIX * rb1), *const consts1 = consts0 + 64 * pairs0;
    const FastDiv by_hw{pa.hw_m, pa.hw_s, (unsigned)pa.HW};

    // ---- weights of a pair, shared by the two layers ---------------------------------------------------------------------------
    v4i a[SC][2];
    auto load_a = [&](const PwPwLayer& l, int pr, unsigned cg0) {  // (steps that do not exist: past the weights, zero)
        const __amdgpu_buffer_rsrc_t rw = rsrc(l.w, (unsigned)l.steps * (unsigned)l.mt * 1024u);
#pragma unroll
        for (int s = 0; s < SC; ++s)
#pragma unroll
            for (int h = 0; h < 2; ++h)
                a[s][h] = load16(rw, s == 0 || cg0 + s < l.steps ? lane * 16 + h * 1024 : PR_OOB,
                                 s == 0 || cg0 + s < l.steps ? ((cg0 + s) * (unsigned)l.mt + 2u * pr) * 1024u : 0u);
    };
    load_a(l0, min(wave, pairs0 - 1), 0);

    // ---- the first layer's input and the constants into LDS ----------------------------------------------------------------------
    {
        constexpr int GROUP = THREADS / PIX, U = 8;  // octets that the workgroup's threads move together, that a thread has requested
        const unsigned px = tid % PIX, gp = (unsigned)tile * PIX + px, n = div_by(gp, by_hw), pix = gp - n * HW;
        const __amdgpu_buffer_rsrc_t rin = rsrc(x, pa.total_pix * C8 * 8u);
        const unsigned v = gp < pa.total_pix ? ((n * C8 + tid / PIX) * HW + pix) * 8u : PR_OOB;
        int8_t* const to = px0 + px * rb0 + 8 * (tid / PIX);
        for (unsigned o0 = 0; o0 < C8; o0 += GROUP * U) {
            v2i d[U];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const unsigned o = o0 + GROUP * u;  // (scalar; a thread's octet is o + tid / PIX)
                d[u] = load8(rin, o + tid / PIX < C8 ? v : PR_OOB, o < C8 ? o * HW * 8u : 0u);
            }
            if (o0 == 0) {  // (scale_in and bias are padded to whole pairs and more)
                for (unsigned i = tid; i < 16u * (pairs0 + pairs1); i += THREADS) {
                    const bool second = i >= 16u * pairs0;
                    const PwPwLayer& l = second ? l1 : l0;
                    const unsigned k = second ? i - 16u * pairs0 : i, half = 8u * (second ? pairs1 : pairs0);
                    reinterpret_cast<v4i*>(consts0)[i] = *reinterpret_cast<const v4i*>(k >= half ? l.bias + 4 * (k - half) : l.scale_in + 4 * k);
                }
            }
#pragma unroll
            for (int u = 0; u < U; ++u)
                if (o0 + GROUP * u + tid / PIX < C8) *reinterpret_cast<v2i*>(to + 8 * (o0 + GROUP * u)) = d[u];
        }
    }

    unsigned n[FN], pix[FN];
    bool ok[FN];
#pragma unroll
    for (int j = 0; j < FN; ++j) {
        const unsigned gp = (unsigned)tile * PIX + 16 * j + p;
        ok[j] = gp < pa.total_pix;
        n[j] = div_by(gp, by_hw), pix[j] = gp - n[j] * HW;
    }
    // byte offset of (image, this lane's channels of a pair, pixel) in a blob of K channels: Byte8, Float4, Float8; a pair is 32 HW
    // (Byte8) or 128 HW (fp32) bytes further
    auto at_b8 = [&](int j, unsigned K) { return ok[j] ? ((n[j] * (K / 8) + q) * HW + pix[j]) * 8u : PR_OOB; };
    auto at_f4 = [&](int j, unsigned K) { return ok[j] ? ((n[j] * (K / 4) + 2 * q) * HW + pix[j]) * 16u : PR_OOB; };
    auto at_f8 = [&](int j, unsigned K) { return ok[j] ? ((n[j] * (K / 8) + q) * HW + pix[j]) * 32u : PR_OOB; };

    // One layer: the wave's pairs, weights requested one pair ahead; finish(pair, sums, elements of another blob). `then` requests
    // the next layer's first weights behind the last pair.
    auto layer = [&](const PwPwLayer& l, int pairs, const int8_t* px, unsigned row_bytes, auto& k0, auto& k1, auto load_pair, auto finish, auto then) {
        const int8_t* const b0 = px + p * row_bytes + 16 * q;
        auto step = [&](auto& k, auto& next, int pr) {
            load_pair(next, min(pr + NW, pairs - 1), pr + NW < pairs);
            v4i c0[FN], c1[FN];
#pragma unroll
            for (int j = 0; j < FN; ++j) c0[j] = c1[j] = v4i{0, 0, 0, 0};
            for (unsigned cg0 = 0;;) {
#pragma unroll
                for (int s = 0; s < SC; ++s)
                    if (s == 0 || cg0 + s < l.steps)  // (uniform)
#pragma unroll
                        for (int j = 0; j < FN; ++j) {
                            const v4i b = *reinterpret_cast<const v4i*>(b0 + 16 * j * row_bytes + 64 * (cg0 + s));
                            c0[j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[s][0], b, c0[j], 0, 0, 0);
                            c1[j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[s][1], b, c1[j], 0, 0, 0);
                        }
                if ((cg0 += SC) >= l.steps) break;
                load_a(l, pr, cg0);
            }
            if (pr + NW < pairs) load_a(l, pr + NW, 0);
            else then();
            finish(k, pr, c0, c1);
        };
        for (int pr = wave; pr < pairs;) {
            step(k0, k1, pr);
            if ((pr += NW) >= pairs) break;
            step(k1, k0, pr);
            pr += NW;
        }
        if (wave >= pairs) then();
    };

    // ---- the first layer ---------------------------------------------------------------------------------------------------------
    struct Pair {  // elements of other blobs
        v4i add[I8 ? 1 : FN][2];
    };
    const unsigned f_bytes = pa.total_pix * K0 * 4u;
    auto load_pair = [&](Pair& k, int pr, bool exists) {
        const unsigned s = (unsigned)pr * 128u;
        const bool live = exists && 32u * pr + 8 * q < K0;
        if constexpr (SHUF) {
            const __amdgpu_buffer_rsrc_t r = rsrc(ja.other, f_bytes);
#pragma unroll
            for (int j = 0; j < FN; ++j) {
                const unsigned v = live ? (ja.other_pack == 8 ? at_f8(j, K0) : at_f4(j, K0)) : PR_OOB;  // (uniform choice)
                k.add[j][0] = load16(r, v, s * HW);
                k.add[j][1] = load16(r, v, s * HW + (ja.other_pack == 8 ? 16u : HW * 16u));
            }
        }
    };
    const Epilogue ep0 = pp_epilogue(l0);
    int8_t* const to1 = px1 + p * rb1;  // this lane's pixel of the second layer's input
    auto constants = [&](const float* c, int pairs, unsigned ch0, float (&si)[8], float (&bi)[8]) {
#pragma unroll
        for (int e = 0; e < 8; ++e) si[e] = c[ch0 + e], bi[e] = c[32 * pairs + ch0 + e];
    };
    auto finish0 = [&](const Pair& k, int pr, const v4i (&c0)[FN], const v4i (&c1)[FN]) {
        const unsigned ch0 = 32u * pr + 8 * q;
        float si[8], bi[8];
        constants(consts0, pairs0, ch0, si, bi);
#pragma unroll
        for (int j = 0; j < FN; ++j) {
            int8_t* const to = to1 + 16 * j * rb1;
            if constexpr (I8) {
                const v2i b = pp_bytes<EPI == EPI_I8_P8_NONNEG>(ep0, l0, si, bi, c0[j], c1[j]);
                if (ch0 < K0) *reinterpret_cast<v2i*>(to + ch0) = b;
            } else {
                const v4i r[2] = {pp_values(ep0, si, bi, c0[j]), pp_values(ep0, si + 4, bi + 4, c1[j])};
                {
                    // with the same channels of the other blob these are channels 2 ch0 .. 2 ch0 + 15 of the shuffled one: two packs of 8
                    const unsigned half = K0 / 8;  // packs of 8 in each half
#pragma unroll
                    for (int h = 0; h < 2; ++h) {
                        const v4i o = k.add[j][h];
                        const v4i even = ja.other_odd ? r[h] : o, odd = ja.other_odd ? o : r[h];  // (uniform)
                        const v4i lo = {even[0], odd[0], even[1], odd[1]}, hi = {even[2], odd[2], even[3], odd[3]};
                        const unsigned pack = ch0 / 4 + h;
                        if (8u * pr < half) {  // (uniform: one of the pair's packs is in the first half)
                            const unsigned e = n[j] * ja.sh_image + (pack * HW + pix[j]) * 8u;
                            const bool live = ok[j] && pack < half;
                            const __amdgpu_buffer_rsrc_t rf = rsrc(ja.sh_out0, PR_OOB);
                            store16(rf, lo, live ? e * 4u : PR_OOB, 0), store16(rf, hi, (live ? e * 4u : PR_OOB) + 16u, 0);
                        }
                        if (8u * pr + 8 > half) {  // (uniform: one of them is in the second)
                            const v2i b = {quantize4(lo, ja.twin_scale, ja.twin_half), quantize4(hi, ja.twin_scale, ja.twin_half)};
                            if (pack >= half && pack < 2 * half) *reinterpret_cast<v2i*>(to + 8 * (pack - half)) = b;
                        }
                    }
                }
            }
        }
    };
    Pair k0, k1;
    load_pair(k0, min(wave, pairs0 - 1), wave < pairs0);
    __syncthreads();
    auto weights1 = [&] { load_a(l1, min(wave, pairs1 - 1), 0); };
    layer(l0, pairs0, px0, rb0, k0, k1, load_pair, finish0, weights1);
    __syncthreads();

    // ---- the second layer --------------------------------------------------------------------------------------------------------
    const unsigned K1 = l1.K;
    const Epilogue ep1 = pp_epilogue(l1);
    const __amdgpu_buffer_rsrc_t rout = rsrc(out, pa.total_pix * K1 * (KIND1 == PP_F32 ? 4u : 1u));
    struct None {
    } none;
    auto finish1 = [&](const None&, int pr, const v4i (&c0)[FN], const v4i (&c1)[FN]) {
        const unsigned ch0 = 32u * pr + 8 * q;
        float si[8], bi[8];
        constants(consts1, pairs1, ch0, si, bi);
#pragma unroll
        for (int j = 0; j < FN; ++j) {
            if constexpr (KIND1 == PP_F32) {
                const v4i r0 = pp_values(ep1, si, bi, c0[j]), r1 = pp_values(ep1, si + 4, bi + 4, c1[j]);
                const unsigned v = at_f4(j, K1), s = (unsigned)pr * 128u * HW;
                store16(rout, r0, ch0 < K1 ? v : PR_OOB, s), store16(rout, r1, ch0 + 4 < K1 ? v : PR_OOB, s + HW * 16u);
            } else {
                store8(rout, pp_bytes<KIND1 == PP_NONNEG>(ep1, l1, si, bi, c0[j], c1[j]), ch0 < K1 ? at_b8(j, K1) : PR_OOB, (unsigned)pr * 32u * HW);
            }
        }
    };
    layer(l1, pairs1, px1, rb1, none, none, [](None&, int, bool) {}, finish1, [] {});
}

// ---------------------------------------------------------------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------------------------------------------------------------

static size_t pwpw_lds_bytes(const ConvGeom& g0, const ConvGeom& g1, int fn) {
    const size_t rows = 64 * (size_t)(igemm_channel_groups(g0.C) + igemm_channel_groups(g1.C)) + 32;
    return 16 * (size_t)fn * rows + 256 * (size_t)((g0.K + 31) / 32 + (g1.K + 31) / 32);
}

// e0: the first layer's epilogue with what is to become of its result (twin: a blob for the int8 form, too)
bool conv_pwpw_applicable(const ConvGeom& g0, const Epilogue& e0, const ConvGeom& g1, const Epilogue& e1) {
    if (!pwpw_pointwise(g0) || !pwpw_pointwise(g1) || g1.C != g0.K || g0.K % 8 || g0.N != g1.N || g0.H != g1.H || g0.W != g1.W) return false;
    if (g0.N < 1 || pwpw_lds_bytes(g0, g1, 1) > 65536) return false;
    const int k0 = pwpw_kind(e0, g0.K);
    if (k0 < 0 || pwpw_kind(e1, g1.K) < 0) return false;
    if ((k0 == PP_F32) != (e0.join != nullptr) || e0.residual || e0.twin) return false;
    if (e0.join && (!e0.join->other || e0.join->sh_image != (size_t)g0.K * g0.H * g0.W || !e0.join->sh_out0)) return false;  // (two halves)
    const size_t px = (size_t)g0.N * g0.H * g0.W, limit = (size_t)1 << 31;
    for (const ConvGeom* g : {&g0, &g1})
        if ((size_t)igemm_channel_groups(g->C) * igemm_padded_rows(g->K) * 64 >= limit) return false;  // (the packed weights)
    return px * g0.C < limit && px * g0.K * (k0 == PP_F32 ? 4 : 1) < limit && px * g1.K * layout_elem_bytes(e1.out_layout) < limit;
}

// Whether the launch is faster than the two. It saves a launch and the blob in between, but a workgroup walks through all the channels of
// both layers, a pair of row tiles a wave, where the two launches deal them to workgroups as well: the more pairs, the more workgroups it
// takes before that is made up for. us as two / one: 88 channels @26x26 b16 (6 pairs, 676 tiles) 6.6 / 4.7; 64 -> 128 -> 1280 on one 7x7
// image (44 pairs, 4 tiles) 4.8 / 8.4, on 16 of them 5.9 / 8.1; 176 @26x26 b16 (12 pairs) 8.2 / 6.4, on one 13x13 image 5.0 / 5.1; 352 @26x26
// b16 (22 pairs, 676 tiles) 14.6 / 13.2, @13x13 b16 (169) 8.1 / 8.6. Where the first layer has at most two pairs, two of the four waves
// idle through it: small launches gain all the same, large ones do not (48 channels @26x26 b16 5.4 / 4.4, @52x52 b16 6.6 / 7.0; with a
// shuffle 9.4 / 11.4). Over 11600 drawn pairs of 8 to 512 and 8 to 1280 channels, half of them with a shuffle, the faster of the two is missed
// by 0.5 % on average, by over 5 % for 270 of the 7200 taken and for 210 of the others.
bool conv_pwpw_faster(const ConvGeom& g0, const ConvGeom& g1) {
    const long tiles = ((long)g0.N * g0.H * g0.W + 15) / 16;
    const int first = (g0.K + 31) / 32, pairs = first + (g1.K + 31) / 32;
    if (first <= 2) return pairs <= 10 && tiles < 1536;
    return tiles >= (pairs > 17 ? 640 : pairs > 10 ? 128 : first > 4 ? 8 : 1);
}

template <int FN, int SC, int EPI>
static hipError_t launch_pwpw(const int8_t* x, void* out, const PwPwArgs& pa, const Epilogue& e0, size_t lds, hipStream_t stream) {
    const dim3 grid((pa.tiles + 7) / 8 * 8), block(64 * PP_WAVES);
    if (pa.l[1].kind == PP_NONNEG) launch((conv_pwpw_kernel<FN, SC, EPI, PP_NONNEG>), grid, block, lds, stream, x, out, pa, PwAdd<EPI>::of(e0));
    else if (pa.l[1].kind == PP_I8) launch((conv_pwpw_kernel<FN, SC, EPI, PP_I8>), grid, block, lds, stream, x, out, pa, PwAdd<EPI>::of(e0));
    else launch((conv_pwpw_kernel<FN, SC, EPI, PP_F32>), grid, block, lds, stream, x, out, pa, PwAdd<EPI>::of(e0));
    return hipGetLastError();
}

// w, so: packed weights and the output scale of every channel of each layer; force: 0 = automatic, else pixel groups
hipError_t run_conv_pwpw(const int8_t* x, const int8_t* const w[2], const float so[2], void* out, const ConvGeom& g0,
                         const Epilogue& e0, const ConvGeom& g1, const Epilogue& e1, int force, hipStream_t stream) {
    if (!conv_pwpw_applicable(g0, e0, g1, e1)) return hipErrorInvalidValue;
    PwPwArgs pa{};
    for (int i = 0; i < 2; ++i) pa.l[i] = pwpw_layer(i ? g1 : g0, i ? e1 : e0, w[i], so[i]);
    const FastDiv hw = fast_div((unsigned)(g0.H * g0.W));
    pa.hw_m = hw.m, pa.hw_s = (unsigned char)hw.s, pa.HW = g0.H * g0.W, pa.total_pix = (unsigned)g0.N * (unsigned)pa.HW, pa.C8 = (unsigned short)(g0.C / 8);
    int fn = force ? force : pa.total_pix >= 16384 ? 2 : 1;  // (88 channels @52x52 b16 9.6 us with one group of pixels, 8.3 with two; @26x26 4.8 and 4.7)
    if (fn == 2 && pwpw_lds_bytes(g0, g1, 2) > 65536) fn = 1;
    if (fn != 1 && fn != 2) return hipErrorInvalidValue;
    pa.tiles = (int)((pa.total_pix + 16 * fn - 1) / (16 * fn));
    const size_t lds = pwpw_lds_bytes(g0, g1, fn);
    const bool deep = std::max(pa.l[0].steps, pa.l[1].steps) > 2;
#define OHIP_PP(F_, E_) \
    return fn == F_ && deep ? launch_pwpw<F_, 4, E_>(x, out, pa, e0, lds, stream) : launch_pwpw<F_, 2, E_>(x, out, pa, e0, lds, stream)
#define OHIP_PPE(E_)               \
    do {                           \
        if (fn == 1) OHIP_PP(1, E_); \
        OHIP_PP(2, E_);            \
    } while (0)
    if (e0.join) OHIP_PPE(EPI_F32_SHUFFLE);
    if (pa.l[0].kind == PP_NONNEG) OHIP_PPE(EPI_I8_P8_NONNEG);
    OHIP_PPE(EPI_I8_P8);
#undef OHIP_PPE
#undef OHIP_PP
}

}  // namespace ohip
