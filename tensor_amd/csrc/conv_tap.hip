// Dense and grouped int8 convolution with both matrix operands straight from memory and the reduction dealt to the waves
// of a workgroup: the kernel for launches that do not fill the machine, and for reductions that the 64-channel steps of the
// implicit-GEMM kernel pad heavily.
//
// What bounds those launches is not bandwidth or operations but one chain of dependent latencies per workgroup. The
// implicit-GEMM kernel walks its k-chunks one barrier and one LDS round trip after the other (264 -> 24 5x5 stride 2 on
// twelve 7x7 images: 125 chunks, three workgroups, 46 us); the LDS-halo kernel stages whole rows before its first
// multiplication. Here
//  * WK waves of a workgroup take every WK-th reduction step each, hold their loads DEPTH steps ahead in registers and
//    meet once, in LDS, to add up their int32 accumulators (integers: the same result in any order);
//  * the reduction runs over (tap, channel octet) pairs in that order, eight to a 64-deep matrix step, with no padding but
//    at its end: 8 channels of a 5x5 layer are 4 steps instead of 25, 104 channels of a 3x3 layer 15 instead of 18. A
//    lane's 16-byte operand is two consecutive pairs of its pixel, two 8-byte loads (16 lanes: 128 contiguous bytes each);
//  * the byte offset of a pair and the bit of its tap come from a table in LDS, the taps that fall outside the image from a
//    bit mask per pixel: three vector instructions per load, an invalid one gets an offset beyond the buffer and reads zero.
// The same operands are re-read per tap from L1 / L2, which is why large launches with long reductions stay with the
// kernels that stage them in LDS (conv_tap_cost against conv_family_cost).
//
// Measured, us per launch before / after: 336 -> 184 3x3, one 13x13 image 22.7 / 4.5; 400 -> 216 3x3 stride 2, thirteen 23x23
// 29.1 / 8.1; 160 -> 8 5x5 @184x224 43.0 / 17.7; 16 -> 184 5x5 @168x168 x4 56.4 / 30.9; 720 -> 384 1x1 from fp32, one 13x13
// image 9.2 / 3.7; 64 -> 128 3x3 in 8 groups @32x32 x13 8.8 / 6.2.
// The small launches are bound by what surrounds the loop: 64 -> 64 3x3 on one 56x56 image from fp32 spent 1.8 of 5.1 us before its
// first step, 2.4 in the loop, 0.9 behind it. A window's mask in closed form, a loop whose loads are waited for one by one and tiles
// of one fragment took it to 3.6 (from int8 4.0 / 3.0; 32 -> 64 stride 2 @112x112 x4 from fp32 5.4 / 4.8). 900 drawn k x k layers
// under a million pixels: 0.915 of the time.
//
// INF: the input is a Float8 blob ([N][C/8][H*W][8 floats]); a lane quantizes the pairs it loads (quantize_to_int8,
// Tensor/ConvolutionLayer.cpp:770-775). Every value is quantized once per tap that reads it, which a launch that leaves
// most of the vector ALU idle has room for; it saves the quantize launch and its blob.
#include "common.hpp"
#include "conv_igemm.hpp"

#include <algorithm>
#include <cmath>
#include <utility>

namespace ohip {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v2i __attribute__((ext_vector_type(2)));

namespace {

constexpr int TAP_MAX_TAPS = 31;      // bit 31 of a pixel's mask stands for "past the end of the reduction"
constexpr int TAP_MAX_PAIRS = 2048;   // table entries: 16 KB of LDS

struct TapArgs {  // (a launch costs the host about 0.1 us more for every 32 bytes of arguments)
    int H, W, OW, OHW, K, Ks, Cs8;        // K: one group's channels; Ks, Cs8: the tensors' channels, and octets
    int sh, sw, ph, pw, dh, dw;
    unsigned total_pix, in_bytes, w_bytes;
    unsigned ohw_m, ow_m, c8_m, kw_m;     // divisions (FastDiv): multipliers, and the shifts below
    unsigned char ohw_s, ow_s, c8_s, kw_s;
    unsigned char kh, kw;
    unsigned short C8, steps, pairs;      // one group's octets; reduction steps and (tap, octet) pairs of them
    int m_tiles16;                        // 16-row tiles of one group's packed weights
    int n_pix_tiles;
    unsigned row_ones;                    // bit kw * dy of each kernel row
    float in_half;
    const float* in_scale;
};

}  // namespace

template <int FM, int FN, int WK, int WN, int DEPTH, int EPI, bool INF>
__global__ void __launch_bounds__(64 * WK * WN) conv_tap_kernel(const int8_t* __restrict__ x, const int8_t* __restrict__ wpk,
                                                                void* __restrict__ out, TapArgs ta, EpiArgs<EPI> ea,
                                                                JoinParam<EPI> ja) {
    constexpr int UNITS = FM / 2 * FN;  // (row-tile pair, pixel fragment) accumulators of a wave
    constexpr int OOB = (int)0x80000000;  // beyond any buffer here (below 2 GiB)
    extern __shared__ __attribute__((aligned(16))) int8_t lds[];
    v2i* const table = reinterpret_cast<v2i*>(lds);  // [pairs, rounded up to whole steps]: {byte offset, bit number of the tap}
    v4i* const red = reinterpret_cast<v4i*>(lds + (size_t)ta.steps * 64);  // [wn][wk][unit][half][lane]
    const int tid = threadIdx.x, lane = tid & 63, q = lane >> 4, p = lane & 15;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wk = wave % WK, wn = wave / WK;
    int pt = blockIdx.x;
    {  // a contiguous run of pixel tiles per XCD (workgroups go to the 8 XCDs round-robin)
        const int per = ta.n_pix_tiles / 8;
        if (pt < per * 8) pt = (pt % 8) * per + pt / 8;
    }
    const int mt0 = blockIdx.y * FM;
    const int HW = ta.H * ta.W, OHW = ta.OHW, C8 = ta.C8, steps = ta.steps;
    const int grp = blockIdx.z;
    const FastDiv d_ohw{ta.ohw_m, ta.ohw_s, 0}, d_ow{ta.ow_m, ta.ow_s, 0}, d_c8{ta.c8_m, ta.c8_s, 0}, d_kw{ta.kw_m, ta.kw_s, 0};

    // ---- weights: the first steps are on their way before anything else happens ------------------------------------------
    const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<int8_t*>(wpk + (size_t)grp * ta.w_bytes), 0, (int)ta.w_bytes, 0x00020000);
    v4i a[DEPTH][FM];
    auto load_a = [&](int d, int s) {  // step s (uniform); past the end: zeros
        const int v = s < steps ? lane * 16 : OOB, so = s < steps ? (s * ta.m_tiles16 + mt0) * 1024 : 0;
#pragma unroll
        for (int i = 0; i < FM; ++i) a[d][i] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(rw, v + i * 1024, so, 0));
    };
#pragma unroll
    for (int d = 0; d < DEPTH; ++d) load_a(d, wk + d * WK);

    // ---- the table of pairs ---------------------------------------------------------------------------------------------------
    for (int e = tid; e < steps * 8; e += 64 * WK * WN) {
        const unsigned tap = div_by((unsigned)e, d_c8), oct = (unsigned)e - tap * (unsigned)C8;
        const unsigned dy = div_by(tap, d_kw), dx = tap - dy * (unsigned)ta.kw;
        table[e] = e < ta.pairs ? v2i{(int)(oct * (unsigned)HW + dy * (unsigned)(ta.dh * ta.W) + dx * (unsigned)ta.dw) * 8, (int)tap}
                                : v2i{0, 31};
    }

    // ---- this lane's pixels ---------------------------------------------------------------------------------------------------
    unsigned px_ofs[FN], mask[FN], out_n[FN], out_pix[FN];
    bool px_ok[FN];
    const int kh = ta.kh, kw = ta.kw;
    const bool pointwise = kh == 1 && kw == 1 && ta.sh == 1 && ta.sw == 1 && ta.ph == 0 && ta.pw == 0;
    const bool dilated = ta.dh != 1 || ta.dw != 1;
#pragma unroll
    for (int j = 0; j < FN; ++j) {
        const unsigned gp = ((unsigned)pt * WN + wn) * (16 * FN) + 16 * j + p;
        px_ok[j] = gp < ta.total_pix;
        const unsigned n = div_by(gp, d_ohw), pix = gp - n * (unsigned)OHW;
        out_n[j] = n, out_pix[j] = pix;
        const unsigned img = (n * (unsigned)ta.Cs8 + (unsigned)(grp * C8)) * (unsigned)HW * 8u;
        if (pointwise) {
            px_ofs[j] = img + pix * 8u, mask[j] = 0x80000000u;
        } else {
            const unsigned oy = div_by(pix, d_ow), ox = pix - oy * (unsigned)ta.OW;
            const int iy0 = (int)oy * ta.sh - ta.ph, ix0 = (int)ox * ta.sw - ta.pw;
            px_ofs[j] = img + (unsigned)((iy0 * ta.W + ix0) * 8);  // (modulo 2^32: the pair's offset brings it back)
            if (dilated) {
                unsigned cols = 0, all = (1u << kw) - 1, m = 0x80000000u;
                for (int dx = 0; dx < kw; ++dx) {
                    const int ix = ix0 + dx * ta.dw;
                    cols |= (ix < 0 || ix >= ta.W ? 1u : 0u) << dx;
                }
                for (int dy = 0; dy < kh; ++dy) {
                    const int iy = iy0 + dy * ta.dh;
                    m |= (iy < 0 || iy >= ta.H ? all : cols) << (dy * kw);
                }
                mask[j] = m;
            } else {
                // the taps inside the image are columns x0..x1 of rows y0..y1: the columns' bits, repeated per kernel row, under the
                // rows' bits (the loops above take 100 instructions of a wave that has few others: 0.2 to 0.5 us of a launch)
                const int x1 = min(max(ta.W - ix0, 0), kw), x0 = min(max(-ix0, 0), x1);
                const int y1 = min(max(ta.H - iy0, 0), kh), y0 = min(max(-iy0, 0), y1);
                const unsigned cols = (1u << x1) - (1u << x0), rows = (1u << (y1 * kw)) - (1u << (y0 * kw));
                mask[j] = ~(cols * ta.row_ones & rows);
            }
        }
        if (!px_ok[j]) mask[j] = 0xffffffffu;
    }

    // ---- the reduction --------------------------------------------------------------------------------------------------------
    const __amdgpu_buffer_rsrc_t rin = __builtin_amdgcn_make_buffer_rsrc(const_cast<int8_t*>(x), 0, (int)ta.in_bytes, 0x00020000);
    v2i b[INF ? 1 : DEPTH][FN][2];
    v4i bf[INF ? DEPTH : 1][FN][4];
    float in_scale = 0.f;
    if constexpr (INF) in_scale = ta.in_scale[0];
    __syncthreads();
    auto load_b = [&](int d, int s) {
        // steps past the end keep the bit of the last table row's padding out of reach: they read the table's first step
        // with every pair invalid
        const bool in = s < steps;
        const v4i t = reinterpret_cast<const v4i*>(table)[(in ? s : 0) * 4 + q];
        const int b0 = in ? t[1] : 31, b1 = in ? t[3] : 31;
#pragma unroll
        for (int j = 0; j < FN; ++j) {
            // the tap's invalid bit becomes bit 31 of the offset: beyond the buffer, whatever the rest of it is
            const unsigned i0 = __builtin_amdgcn_ubfe(mask[j], (unsigned)b0, 1) << 31;
            const unsigned i1 = __builtin_amdgcn_ubfe(mask[j], (unsigned)b1, 1) << 31;
            const unsigned o0 = px_ofs[j] + (unsigned)t[0], o1 = px_ofs[j] + (unsigned)t[2];
            if constexpr (INF) {  // (the fp32 element of a pixel's octet lies at four times the int8 element's offset)
                const int f0 = (int)(o0 * 4u | i0), f1 = (int)(o1 * 4u | i1);
                bf[d][j][0] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(rin, f0, 0, 0));
                bf[d][j][1] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(rin, f0 + 16, 0, 0));
                bf[d][j][2] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(rin, f1, 0, 0));
                bf[d][j][3] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(rin, f1 + 16, 0, 0));
            } else {
                b[d][j][0] = __builtin_bit_cast(v2i, __builtin_amdgcn_raw_buffer_load_b64(rin, (int)(o0 | i0), 0, 0));
                b[d][j][1] = __builtin_bit_cast(v2i, __builtin_amdgcn_raw_buffer_load_b64(rin, (int)(o1 | i1), 0, 0));
            }
        }
    };
#pragma unroll
    for (int d = 0; d < DEPTH; ++d) load_b(d, wk + d * WK);
    v4i acc[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) acc[i][j] = v4i{0, 0, 0, 0};
    auto multiply = [&](int d) {
        v4i bb[FN];
#pragma unroll
        for (int j = 0; j < FN; ++j) {
            if constexpr (INF)
                bb[j] = v4i{quantize4(bf[d][j][0], in_scale, ta.in_half), quantize4(bf[d][j][1], in_scale, ta.in_half),
                            quantize4(bf[d][j][2], in_scale, ta.in_half), quantize4(bf[d][j][3], in_scale, ta.in_half)};
            else
                bb[j] = v4i{b[d][j][0][0], b[d][j][0][1], b[d][j][1][0], b[d][j][1][1]};
        }
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
            for (int j = 0; j < FN; ++j) acc[i][j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[d][i], bb[j], acc[i][j], 0, 0, 0);
    };
    // No load of the loop is conditional: behind a conditional one the compiler waits for every load in flight (which made the
    // stages ahead worthless). The last trip's 1 to DEPTH - 1 loads are code of their own (EXACT); where that takes too
    // many registers (from fp32, the widest tile) they go beyond the buffer where a step is missing.
    constexpr bool EXACT = !INF && FM * FN < 16;
    constexpr int WHOLE = EXACT ? 2 * DEPTH : DEPTH + 1;
    int s = wk, left = (steps - wk + WK - 1) / WK;  // this wave's next step, and how many it has from there on
    for (; left >= WHOLE; left -= DEPTH) {
#pragma unroll
        for (int d = 0; d < DEPTH; ++d, s += WK) {
            multiply(d);
            load_a(d, s + DEPTH * WK);
            load_b(d, s + DEPTH * WK);
        }
    }
    bool done = false;
    if constexpr (EXACT) {
#pragma unroll
        for (int r = 1; r < DEPTH; ++r)
            if (left == DEPTH + r) {
#pragma unroll
                for (int d = 0; d < r; ++d, s += WK) {
                    multiply(d);
                    load_a(d, s + DEPTH * WK);
                    load_b(d, s + DEPTH * WK);
                }
#pragma unroll
                for (int d = r; d < DEPTH + r; ++d) multiply(d % DEPTH);
                done = true;
            }
    }
    if (!done) {
#pragma unroll
        for (int d = 0; d < DEPTH; ++d)
            if (d < left) multiply(d);
    }

    // ---- the waves' sums meet: unit u of a pixel group is finished by its wave u % WK ---------------------------------------------
    if constexpr (WK > 1) {
        v4i* const mine = red + (size_t)((wn * WK + wk) * UNITS) * 128 + lane;
#pragma unroll
        for (int u = 0; u < UNITS; ++u) {
            if (u % WK == wk) continue;
            mine[u * 128] = acc[2 * (u / FN)][u % FN];
            mine[u * 128 + 64] = acc[2 * (u / FN) + 1][u % FN];
        }
        __syncthreads();
    }
    const int K = ta.K, Ks = ta.Ks;
    const size_t ch_base = (size_t)grp * K;
    Epilogue ep = ea.epilogue();
    ep.scale_in += ch_base, ep.bias += ch_base;
    if (ep.scale_out) ep.scale_out += ch_base;
#pragma unroll
    for (int u = 0; u < UNITS; ++u) {
        if (WK > 1 && u % WK != wk) continue;  // (uniform)
        const int pair = u / FN, j = u % FN;
        v4i lo = acc[2 * pair][j], hi = acc[2 * pair + 1][j];
        if constexpr (WK > 1) {
            const v4i* const r = red + (size_t)(wn * WK * UNITS + u) * 128 + lane;
#pragma unroll
            for (int k = 0; k < WK; ++k) {
                if (k == u % WK) continue;
                lo += r[k * UNITS * 128];
                hi += r[k * UNITS * 128 + 64];
            }
        }
        const int ch0 = 16 * mt0 + 32 * pair + 8 * q;  // this lane's 8 consecutive output channels of the group
        if (!px_ok[j] || ch0 >= K) continue;
        const int a8[8] = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
        const unsigned n = out_n[j], pix = out_pix[j];
        if constexpr (EPI == EPI_GENERIC) {
            epilogue_store8_generic(out, &ep, (int)n, ch0, (int)pix, K, OHW, a8[0], a8[1], a8[2], a8[3], a8[4], a8[5], a8[6], a8[7]);
        } else {
            Epi8 prm;
            epi8_load<EPI>(prm, ep, ch0);
            const unsigned ch = (unsigned)ch_base + (unsigned)ch0;  // in the tensor
            if constexpr (epi_is_i8(EPI)) {
                const size_t o = ((size_t)(n * (unsigned)(Ks / 8) + ch / 8) * (unsigned)OHW + pix) * 8;
                epi8_store_i8p8<epi_clamp(EPI)>((int8_t*)out, ep, prm, o, a8);
            } else if constexpr (EPI == EPI_F32_SHUFFLE) {
                if (ep.lrelu) epi8_store_shuffle<1>(ep, ja, prm.si, prm.bi, a8, n, pix, ch0, K, OHW);
                else epi8_store_shuffle<0>(ep, ja, prm.si, prm.bi, a8, n, pix, ch0, K, OHW);
            } else {
                constexpr bool FUSED = EPI == EPI_F32_P4_FUSED || EPI == EPI_F32_P4_PARTS;
                const size_t e = ((size_t)(n * (unsigned)(Ks / 4) + ch / 4) * (unsigned)OHW + pix) * 4;
                const float *r0 = nullptr, *r1 = nullptr;
                if constexpr (EPI == EPI_F32_P4_PARTS) {  // (one group)
                    r0 = epi4_residual_at(ep, ja, n, pix, ch0, K, OHW);
                    r1 = epi4_residual_at(ep, ja, n, pix, ch0 + 4, K, OHW);
                }
                ohip_v2i tw = {0, 0};
                tw[0] = (int)epi4_store_f32p4<FUSED>((float*)out, ep, prm.si, prm.bi, e, a8[0], a8[1], a8[2], a8[3], r0);
                if (ch0 + 4 < K)
                    tw[1] = (int)epi4_store_f32p4<FUSED>((float*)out, ep, prm.si + 4, prm.bi + 4, e + (size_t)OHW * 4, a8[4], a8[5],
                                                         a8[6], a8[7], r1);
                if constexpr (FUSED)
                    if (ep.twin != nullptr)  // K % 8 == 0 then: the lane's 8 channels are one Byte8 element
                        *reinterpret_cast<ohip_v2i*>(ep.twin + ((size_t)(n * (unsigned)(Ks / 8) + ch / 8) * (unsigned)OHW + pix) * 8) = tw;
            }
        }
    }
}

// ---------------------------------------------------------------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------------------------------------------------------------

static int tap_pairs(int C, int kh, int kw) { return kh * kw * (C / 8); }
static int tap_steps(int C, int kh, int kw) { return (tap_pairs(C, kh, kw) + 7) / 8; }

// whether the implicit-GEMM packing of these weights already is this kernel's: a step is then whole taps, or one tap's part
bool tap_weights_are_igemm(int C, int kh, int kw, int tap_pack) {
    if (kh * kw == 1 || C % 64 == 0) return true;
    return tap_pack > 1 && C * tap_pack == 64;
}

size_t tap_packed_weight_bytes(int K, int C, int kh, int kw) {
    return (size_t)tap_steps(C, kh, kw) * (igemm_padded_rows(K) / 16) * 1024;
}

// weight [K, C, kh, kw] int8 -> [step][16-row tile][lane][16 bytes]: bytes 0-7 / 8-15 of lane (r, q) are the octets of pairs
// 8 step + 2 q and + 1, pair e = (tap e / (C/8), octet e % (C/8))
void tap_pack_weights(const int8_t* w, int K, int C, int kh, int kw, int8_t* dst) {
    const int mt16 = igemm_padded_rows(K) / 16, taps = kh * kw, C8 = C / 8, pairs = tap_pairs(C, kh, kw);
    size_t o = 0;
    for (int s = 0; s < tap_steps(C, kh, kw); ++s)
        for (int mt = 0; mt < mt16; ++mt)
            for (int lane = 0; lane < 64; ++lane) {
                const int ch = igemm_row_channel(mt * 16 + (lane & 15));
                for (int h = 0; h < 2; ++h) {
                    const int e = 8 * s + 2 * (lane >> 4) + h, tap = e / C8, c0 = e % C8 * 8;
                    for (int b = 0; b < 8; ++b, ++o)
                        dst[o] = ch < K && e < pairs ? w[((size_t)ch * C + c0 + b) * taps + tap] : 0;
                }
            }
}

size_t tap_grouped_weight_bytes(int K, int C, int groups, int kh, int kw) {
    return (size_t)groups * tap_packed_weight_bytes(K / groups, C / groups, kh, kw);
}
void tap_pack_weights_grouped(const int8_t* w, int K, int C, int groups, int kh, int kw, int8_t* dst) {
    const int kg = K / groups, cg = C / groups;
    const size_t per = tap_packed_weight_bytes(kg, cg, kh, kw);
    for (int grp = 0; grp < groups; ++grp)
        tap_pack_weights(w + (size_t)grp * kg * cg * kh * kw, kg, cg, kh, kw, dst + grp * per);
}

bool conv_tap_supported(const ConvGeom& g, const Epilogue& ep, bool f32in) {
    if (g.OH < 1 || g.OW < 1 || g.C % g.groups || g.K % g.groups) return false;
    const int cg = g.C / g.groups, kg = g.K / g.groups;
    if (cg % 8 || g.kh * g.kw > TAP_MAX_TAPS || tap_pairs(cg, g.kh, g.kw) > TAP_MAX_PAIRS || g.groups > 65535) return false;
    const int epi = pick_epilogue(ep, kg);
    if (g.groups > 1 && (epi == EPI_GENERIC || ep.fused())) return false;
    if (ep.fused() && epi != EPI_F32_P4) return false;
    if (f32in && (epi == EPI_GENERIC || ep.join != nullptr)) return false;
    return (size_t)g.N * g.C * g.H * g.W * (f32in ? 4 : 1) < ((size_t)1 << 31);  // 32-bit byte offsets
}

namespace {
// A tile is 16 fm output channels x 16 fn wn pixels, `resident` workgroups of it a compute unit's registers hold. The cost of a
// launch in microseconds (measured inside a graph of launches, warm) is start + chain * S + c * (waves * S * step + group, with
// `quant` more where the result is int8) + round for every time the compute unit fills up again + in_mb and out_mb per megabyte,
// with S the reduction steps of one wave and c the workgroups of the busiest compute unit. Chain and step grow by `strided` where the
// stride is not 1, a load then using every second 8 bytes of its lines, and by up to `far` where the pixels of the workgroups side by
// side on a compute unit are more than its share of an XCD's L2 (128 KB: 4 MB over 32) holds from one tap, or one row block, to the
// next: from the whole share (fp32 blobs, the widest tile) or half of it on, fully at twice that, and only as far as the blob is over
// 4 MB, fully at 16. Fitted to 2900 layers drawn over 8..800 channels, 1x1 to 5x5, 50 to 2.5 million pixels, errors below the
// measurement counted 1.6 times; the median error is 3 to 5 %. (The widest tile keeps an older fit: this one called strided layers of
// 300 channels and more on it 2 times too fast.) The tile that the costs name is 1.1 % slower than the fastest one on average.
// Tiles of one pixel fragment per wave (the last two) are the fastest for 45 % of the layers from fp32 and 30 % of those from int8:
// they fill the machine with half the pixels. 64 -> 64 3x3 on one 56x56 image from fp32 3.6 us, 4.0 to 5.0 with the others.
struct TapCost {
    float start, chain, step, group, out_mb, strided, far, in_mb, quant, round;
};
struct TapConfig {
    int fm, fn, wk, wn, resident, resident_f32;
    TapCost i8, f32;
};
constexpr TapConfig kTapConfigs[] = {
    {2, 1, 8, 1, 3, 3, {2.53f, 0.005f, 0.024f, 0.52f, 0.3f, 0.139f, 4.f, 0.f, 0.064f, 0.581f},
                       {2.497f, 0.043f, 0.049f, 0.222f, 0.3f, 0.295f, 0.875f, 0.051f, 0.097f, 0.626f}},
    {2, 2, 4, 1, 5, 4, {2.717f, 0.028f, 0.034f, 0.251f, 0.207f, 0.132f, 0.666f, 0.f, 0.07f, 1.082f},
                       {2.833f, 0.122f, 0.082f, 0.159f, 0.191f, 0.195f, 0.955f, 0.06f, 0.076f, 0.919f}},
    {4, 2, 4, 1, 4, 3, {2.745f, 0.031f, 0.052f, 0.082f, 0.158f, 0.16f, 0.497f, 0.f, 0.074f, 0.696f},
                       {2.929f, 0.177f, 0.097f, 0.05f, 0.178f, 0.187f, 0.906f, 0.051f, 0.087f, 1.476f}},
    {4, 2, 2, 2, 4, 3, {2.787f, 0.043f, 0.05f, 0.058f, 0.166f, 0.126f, 0.472f, 0.005f, 0.168f, 0.718f},
                       {3.026f, 0.145f, 0.098f, 0.05f, 0.193f, 0.223f, 0.84f, 0.062f, 0.17f, 1.221f}},
    {4, 4, 1, 4, 3, 0, {3.568f, 0.036f, 0.084f, 1.238f, 0.096f, 0.101f, 0.8f, 0.f, 0.f, 0.f}, {}},  // (no fp32 input: registers)
    {4, 1, 4, 1, 6, 5, {2.611f, 0.016f, 0.041f, 0.081f, 0.188f, 0.082f, 0.501f, 0.f, 0.04f, 0.355f},
                       {2.604f, 0.078f, 0.055f, 0.093f, 0.267f, 0.197f, 1.033f, 0.046f, 0.08f, 0.642f}},
    {4, 1, 8, 1, 3, 2, {2.537f, 0.012f, 0.04f, 0.244f, 0.262f, 0.125f, 4.f, 0.001f, 0.143f, 0.447f},
                       {2.666f, 0.018f, 0.06f, 0.12f, 0.3f, 0.323f, 2.149f, 0.056f, 0.136f, 0.957f}},
};
constexpr int kTapConfigCount = (int)(sizeof(kTapConfigs) / sizeof(kTapConfigs[0]));

template <int FM, int FN, int WK, int WN, int DEPTH, int EPI, bool INF>
hipError_t launch_tap(const void* x, const int8_t* wpk, void* out, const TapArgs& ta, const Epilogue& ep, int groups, hipStream_t stream) {
    const size_t lds = (size_t)ta.steps * 64 + (WK > 1 ? (size_t)WN * WK * (FM / 2) * FN * 2048 : 0);
    const dim3 grid((unsigned)ta.n_pix_tiles, (unsigned)((ta.K + 16 * FM - 1) / (16 * FM)), (unsigned)groups);
    launch((conv_tap_kernel<FM, FN, WK, WN, DEPTH, EPI, INF>), grid, dim3(64 * WK * WN), lds, stream, (const int8_t*)x,
                       wpk, out, ta, EpiArgs<EPI>::of(ep), JoinParam<EPI>::of(ep));
    return hipGetLastError();
}
}  // namespace

namespace {
struct TapLayer {  // what the costs of the tiles have in common
    int K, steps, groups, pack;  // pack: bytes of a pixel's channels, times the stride
    long px;
    float in_mb, out_mb, beyond_mb;
    bool f32in, i8out, strided, k1;
};
// (a tile's sizes are powers of two known to the compiler: the loop over the table took 0.17 us of divisions, this takes 0.04)
template <int I>
void tap_tile_cost(const TapLayer& l, float* best, int* config) {
    constexpr TapConfig c = kTapConfigs[I];
    const TapCost& k = l.f32in ? kTapConfigs[I].f32 : kTapConfigs[I].i8;
    if (k.step == 0.f) return;
    auto clamp01 = [](float v) { return fminf(fmaxf(v, 0.f), 1.f); };
    const int blocks = (l.K + 16 * c.fm - 1) / (16 * c.fm), resident = l.f32in ? c.resident_f32 : c.resident;
    const long groups = (l.px + 16 * c.fn * c.wn - 1) / (16 * c.fn * c.wn) * blocks * l.groups;
    const int cus = (int)std::min((groups + 255) / 256, 1l << 24);
    const float s = (float)((l.steps + c.wk - 1) / c.wk), cu = (float)cus, w = (float)(c.wk * c.wn) * s;
    const float side = fminf(cu, (float)resident) * (float)(16 * c.fn * c.wn) * (float)l.pack;
    const float beyond = clamp01(side * (l.f32in || c.fn == 4 ? 1.f / 131072.f : 1.f / 65536.f) - 1.f) * l.beyond_mb;
    const bool again = !l.k1 || blocks > 1;  // the pixels are read more than once
    const float slow = (l.strided ? 1.f + k.strided : 1.f) * (again ? 1.f + k.far * beyond : 1.f);
    float rounds = 0.f;  // behind the first
    if (cus > c.resident || cus > c.resident_f32) rounds = (float)(l.f32in ? (cus - 1) / std::max(c.resident_f32, 1) : (cus - 1) / c.resident);
    const float t = k.start + k.chain * s * slow + cu * (w * k.step * slow + k.group + (l.i8out ? k.quant : 0.f)) + rounds * k.round +
                    k.in_mb * l.in_mb + k.out_mb * l.out_mb;
    if (t < *best) *best = t, *config = I;
}
template <int... I>
float tap_costs(const TapLayer& l, int* config, std::integer_sequence<int, I...>) {
    float best = __builtin_inff();
    (tap_tile_cost<I>(l, &best, config), ...);
    return best;
}
}  // namespace

float conv_tap_cost(const ConvGeom& g, bool f32in, int out_bytes, int* config) {
    const float in_mb = (float)g.N * g.C * g.H * g.W * (f32in ? 4e-6f : 1e-6f);
    const int C = g.C / g.groups;
    TapLayer l;
    l.K = g.K / g.groups, l.steps = tap_steps(C, g.kh, g.kw), l.groups = g.groups, l.pack = C * g.sw * (f32in ? 4 : 1);
    l.px = (long)g.N * g.OH * g.OW;
    l.in_mb = in_mb * fminf(1.f, (float)g.kh / (float)g.sh);  // (the rows that are read)
    l.out_mb = (float)l.px * (float)g.K * 1e-6f * (float)out_bytes;
    l.beyond_mb = fminf(fmaxf((in_mb - 4.f) / 12.f, 0.f), 1.f);
    l.f32in = f32in, l.i8out = out_bytes == 1, l.strided = g.sw > 1, l.k1 = g.kh * g.kw == 1;
    *config = -1;
    return tap_costs(l, config, std::make_integer_sequence<int, kTapConfigCount>{});
}

// The same for the launches that the kernel above competes with (families of otter_hip_conv_kernel_kind): the
// implicit-GEMM kernel (1; with fp32 input for pointwise layers), the LDS-halo kernel (3), the fp32 pointwise kernel (6).
// Start + chain * chunks + matrix work + epilogue + bytes in + bytes out, fitted to drawn layers; median error 4 to 11 % (k x k layers of
// the implicit-GEMM kernel 6 %, 13 % on the slow side before its index divisions became multiplications). The fp32
// pointwise kernel walks all output channels per workgroup of 64 pixels, so that its chain grows with them (128 -> 1280 on one
// 29x29 image: 15.6 us, where the kernel above takes 5.8). other: what it is compared with (conv3x3_halo_cost).
float conv_family_cost(const ConvGeom& g, int family, bool f32in, int out_bytes, float other) {
    const int C = g.C / g.groups, K = g.K / g.groups, taps = g.kh * g.kw, tp = g.groups > 1 ? igemm_tap_pack(C, g.kh, g.kw) : 1;
    const float chunks = tp > 1 ? (float)((taps + tp - 1) / tp) : (float)(taps * igemm_channel_groups(C));
    const float px = (float)g.N * g.OH * g.OW * g.groups, rows = K <= 32 ? 32.f : (float)((K + 63) / 64 * 64);
    const float in_mb = (float)g.N * g.C * g.H * g.W * 1e-6f, out_mb = (float)g.N * g.OH * g.OW * g.K * out_bytes * 1e-6f;
    const float mac = px * rows * chunks * 1e-9f, epi = px * rows * 1e-8f;
    if (family == 6) {
        const float cu = ceilf((float)g.N * (float)((g.H * g.W + 63) / 64) / 256), k = 0.01f * (float)K;
        return 2.18f + 0.5f * cu + 0.2f * chunks + k * (0.336f + 0.333f * cu + chunks * (0.063f + 0.096f * cu)) + 0.39f * in_mb + 0.048f * out_mb;
    }
    if (family == 3) return conv3x3_halo_cost(g, out_mb, other);
    if (taps > 1) return 2.93f + 0.308f * chunks + 59.7f * mac + 30.2f * epi + px * (3.43e-6f + 1.121e-6f * chunks) + 0.095f * in_mb + 0.065f * out_mb;
    if (f32in) return 2.37f + 0.50f * chunks + 201.f * mac + 18.f * epi + 0.33f * in_mb + 0.09f * out_mb;
    return 2.46f + 0.34f * chunks + 94.f * mac + 26.f * epi + 0.03f * in_mb + 0.07f * out_mb;
}

hipError_t run_conv_tap(const void* x, bool f32in, const int8_t* wpk, void* out, const ConvGeom& g, const Epilogue& ep, int config,
                        const float* in_scale, int in_round_mode, hipStream_t stream) {
    if (!conv_tap_supported(g, ep, f32in) || config < 0 || config >= kTapConfigCount) return hipErrorInvalidValue;
    const int C = g.C / g.groups, K = g.K / g.groups;
    const FastDiv ohw = fast_div((unsigned)(g.OH * g.OW)), ow = fast_div((unsigned)g.OW), c8 = fast_div((unsigned)(C / 8)),
                  kw = fast_div((unsigned)g.kw);
    TapArgs ta;
    ta.H = g.H, ta.W = g.W, ta.OW = g.OW, ta.OHW = g.OH * g.OW, ta.K = K, ta.Ks = g.K, ta.Cs8 = g.C / 8;
    ta.sh = g.sh, ta.sw = g.sw, ta.ph = g.ph, ta.pw = g.pw, ta.dh = g.dh, ta.dw = g.dw;
    ta.total_pix = (unsigned)g.N * (unsigned)ta.OHW;
    ta.ohw_m = ohw.m, ta.ow_m = ow.m, ta.c8_m = c8.m, ta.kw_m = kw.m;
    ta.ohw_s = (unsigned char)ohw.s, ta.ow_s = (unsigned char)ow.s, ta.c8_s = (unsigned char)c8.s, ta.kw_s = (unsigned char)kw.s;
    ta.kh = (unsigned char)g.kh, ta.kw = (unsigned char)g.kw, ta.C8 = (unsigned short)(C / 8);  // (conv_tap_supported bounds them)
    ta.steps = (unsigned short)tap_steps(C, g.kh, g.kw), ta.pairs = (unsigned short)tap_pairs(C, g.kh, g.kw);
    ta.m_tiles16 = igemm_padded_rows(K) / 16;
    ta.in_bytes = (unsigned)((size_t)g.N * g.C * g.H * g.W * (f32in ? 4 : 1));
    ta.w_bytes = (unsigned)tap_packed_weight_bytes(K, C, g.kh, g.kw);
    ta.row_ones = 0;
    for (int dy = 0; dy < g.kh; ++dy) ta.row_ones |= 1u << (dy * g.kw);
    ta.in_scale = in_scale;
    ta.in_half = in_round_mode == OTTER_HIP_ROUND_SSE ? 0.5f : 0.49999997f;
    const TapConfig c = kTapConfigs[config];
    const long px = (long)g.N * g.OH * g.OW, per = 16l * c.fn * c.wn;
    ta.n_pix_tiles = (int)((px + per - 1) / per);
    int epi = full_epilogue(pick_epilogue(ep, K), ep);
    if (epi == EPI_F32_P4 && ep.fused()) epi = ep.join == nullptr ? EPI_F32_P4_FUSED : ep.join->other != nullptr ? EPI_F32_SHUFFLE : EPI_F32_P4_PARTS;
#define OHIP_TAP2(I_, FM_, FN_, WK_, WN_, D_, E_)                                                                           \
    if (config == I_ && epi == E_) {                                                                                        \
        if (!f32in) return launch_tap<FM_, FN_, WK_, WN_, D_, E_, false>(x, wpk, out, ta, ep, g.groups, stream);         \
        if constexpr (E_ != EPI_GENERIC && (E_ < EPI_F32_SHUFFLE || E_ == EPI_I8_P8_FULL) && FN_ < 4) return launch_tap<FM_, FN_, WK_, WN_, D_ < 4 ? D_ : 2, E_, true>(x, wpk, out, ta, ep, g.groups, stream); \
    }
#define OHIP_TAP(I_, FM_, FN_, WK_, WN_, D_)                 \
    OHIP_TAP2(I_, FM_, FN_, WK_, WN_, D_, EPI_I8_P8)         \
    OHIP_TAP2(I_, FM_, FN_, WK_, WN_, D_, EPI_I8_P8_NONNEG)  \
    OHIP_TAP2(I_, FM_, FN_, WK_, WN_, D_, EPI_I8_P8_FULL)    \
    OHIP_TAP2(I_, FM_, FN_, WK_, WN_, D_, EPI_F32_P4)        \
    OHIP_TAP2(I_, FM_, FN_, WK_, WN_, D_, EPI_F32_P4_FUSED)  \
    OHIP_TAP2(I_, FM_, FN_, WK_, WN_, D_, EPI_F32_SHUFFLE)   \
    OHIP_TAP2(I_, FM_, FN_, WK_, WN_, D_, EPI_F32_P4_PARTS)  \
    OHIP_TAP2(I_, FM_, FN_, WK_, WN_, D_, EPI_GENERIC)
    OHIP_TAP(0, 2, 1, 8, 1, 4)
    OHIP_TAP(1, 2, 2, 4, 1, 4)
    OHIP_TAP(2, 4, 2, 4, 1, 2)
    OHIP_TAP(3, 4, 2, 2, 2, 2)
    OHIP_TAP(4, 4, 4, 1, 4, 2)
    OHIP_TAP(5, 4, 1, 4, 1, 2)
    OHIP_TAP(6, 4, 1, 8, 1, 2)
#undef OHIP_TAP
#undef OHIP_TAP2
    return hipErrorInvalidValue;
}

}  // namespace ohip
