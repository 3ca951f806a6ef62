// Depthwise 3x3 int8 convolution (stride 1 or 2, dilation 1, pad <= 1) on the reference's Byte8 layout, with the
// multiply-accumulate on the matrix cores.
//
// Why matrix cores for a layer with no channel reduction: with dot4 on the vector ALU the layer costs ~20 vector
// instructions per output value (9 dot4 + requantize) and is bound by the vector ALU at ~2x the time HBM needs.
// v_mfma_i32_16x16x64_i8 computes D[16][16] += A[16][64] * B[64][16]. Here a B column n is a run of 4 output pixels
// (stride 1; 2 for stride 2) of one channel octet, and its 64 reduction bytes are the 8 input pixels 4n-2 .. 4n+5 of
// one input row x 8 channels: lane (n, g = lane / 16) supplies pixels 4n-2+2g and +1, i.e. ONE aligned 16-byte load.
// A D row m is (output pixel phase p, channel c) and A is zero except A[(p, c)][(pixel e, channel c)] = w[c][dy][dx]
// for the dx that connects input pixel e to output phase p. One instruction does one kernel ROW for 16 x 16 (phase,
// channel, column) outputs, three do the 3x3 window, and the vector ALU is left with the requantize epilogue only.
// Most multiplies are by zero; the matrix pipe has the room (it runs beside the vector ALU).
//
// Stride 1: two A sets (channels 0-3 and 4-7 of the octet) share the B fragment; a lane ends up with all 8 channels
// of output pixel 4n + lane/16 and stores one Byte8 element. Stride 2: one A set, rows = 2 phases x 8 channels; a
// lane ends up with 4 channels of output pixel 2n + lane/32.
// A lane's fragment of input row y serves kernel row 2 of output row y-2, row 1 of y-1 and row 0 of y (stride 1),
// so a wave walks down a strip of output rows with the input rows in a ring of registers, each loaded once.
// Image borders cost no instructions: loads and stores go through buffer descriptors, a lane that falls outside
// the image carries an out-of-range offset, reads zero and writes nothing.
#include <algorithm>
#include <cmath>

#include "common.hpp"
#include "conv_dw_common.hpp"
#include "conv_igemm.hpp"
#include "dw_strips.hpp"

namespace ohip {

// weight [C, 1, ks, ks] int8 (ks = 3 or 5) -> A operands [C/8 octets][kernel row ks][set T][lane 64][16 bytes], T = 2 for stride 1
// (set t = channels 4t..4t+3) and 1 for stride 2. Lane (r = lane % 16, g = lane / 16) holds A[row r][16g .. 16g+15];
// reduction byte 16g + 8e + j is (input pixel 4n-2+2g+e, channel j).
static int dw_mfma_sets(int stride) { return stride == 1 ? 2 : 1; }
size_t dw_mfma_weight_bytes(int C, int stride, int ks) { return (size_t)(C / 8) * ks * dw_mfma_sets(stride) * 64 * 16; }

// The 8 input pixels 4n-2 .. 4n+5 of a column must cover the windows of its 4 (stride 1) or 2 (stride 2) outputs:
// with pad_w columns of padding the window of output phase p starts at pixel slot 2 + stride*p - pad_w.
bool dw_mfma_window_fits(int ks, int stride, int pad_w) {
    const int phases = 4 / stride;
    return 2 - pad_w >= 0 && (ks - 1) + 2 + stride * (phases - 1) - pad_w <= 7;
}

void dw_mfma_pack_weights(const int8_t* w, int C, int stride, int pad_w, int ks, int8_t* dst) {
    const int T = dw_mfma_sets(stride);
    std::fill(dst, dst + dw_mfma_weight_bytes(C, stride, ks), (int8_t)0);
    for (int o = 0; o < C / 8; ++o)
        for (int dy = 0; dy < ks; ++dy)
            for (int t = 0; t < T; ++t)
                for (int lane = 0; lane < 64; ++lane) {
                    const int r = lane % 16, g = lane / 16;
                    // D row r -> (output pixel phase p, channel c of the octet)
                    const int p = stride == 1 ? r / 4 : r / 8;
                    const int c = stride == 1 ? 4 * t + r % 4 : r % 8;
                    for (int e = 0; e < 2; ++e) {
                        // input pixel 4n - 2 + 2g + e feeds output pixel (4/stride) n + p through tap dx
                        const int dx = 2 * g + e - 2 - stride * p + pad_w;
                        if (dx < 0 || dx >= ks) continue;
                        dst[((((size_t)o * ks + dy) * T + t) * 64 + lane) * 16 + 8 * e + c] =
                            w[(size_t)(8 * o + c) * ks * ks + dy * ks + dx];
                    }
                }
}

// LRELU as in dw_requant4 (its layers have an open clamp)
template <int LRELU = -1>
__device__ __forceinline__ v4i dw_dequant4(const Epilogue& ep, const v4i& acc, const v4i& si, const v4i& bi) {
    v4i res;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        float v = __fmaf_rn((float)acc[e], __int_as_float(si[e]), __int_as_float(bi[e]));
        if constexpr (LRELU != 1) v = fminf(fmaxf(v, ep.act_lo), ep.act_hi);
        if constexpr (LRELU == 1) v = fmaxf(v, __fmul_rn(v, ep.act_p0));
        if constexpr (LRELU == -1) v = lrelu_or_not(ep, v);
        res[e] = __float_as_int(v);
    }
    return res;
}

// What the kernel reads of a layer and what its launch is cut into, with the divisions of its indices (a division by a kernel
// argument is some 40 scalar instructions, and a short strip's wave issues few others). 152 bytes, where ConvGeom and Epilogue
// made 268: the host writes launch arguments to device memory one by one (3.85 us a launch with 180 bytes, 3.35 with 96).
struct DwArgs {
    const float *scale_in, *bias, *scale_out;
    unsigned gx_m, gx, c8_m, chunks_m, chunks;  // divisions (FastDiv) by the workgroups along x, the octets, the column chunks of a row
    int N, H, W, OH, OW, rps;           // rps: output rows of a strip
    unsigned total, in_bytes, out_bytes;
    float p0, lo, hi, half;             // LeakyReLU slope, clamp of an fp32 result, rounding constant (EPI_F32_SLICE: of its quantization)
    unsigned short c8, lpi_m;           // octets; 1 / lane columns of an image, for lanes below 16 (16.8 fixed point)
    unsigned char gx_s, c8_s, chunks_s, lpi, ipw, ph, lrelu;  // ipw: images of a wave
    // EPI_F32_SLICE: octets of an image of the blob that the result is a slice of. (In what was padding: with 12 bytes more every launch was
    // 0.03 us longer. In a union with the words above they became an array in LDS and the launch three times as long.)
    unsigned octets;
    // and the scale of its quantization, in the clamp's or the slope's place, whichever the instance does not read
    template <bool LR>
    __device__ float q_scale() const { return LR ? lo : p0; }

    __device__ Epilogue epilogue() const {
        Epilogue ep{};
        ep.scale_in = scale_in, ep.bias = bias, ep.scale_out = scale_out;
        ep.act_p0 = p0, ep.act_lo = lo, ep.act_hi = hi, ep.round_half = half, ep.lrelu = lrelu != 0;
        return ep;
    }
};

// A wave owns one channel octet x 16 lane columns (64 output pixels of a row at stride 1, 32 at stride 2) and walks
// down `rps` output rows. The input rows live in a ring of 8 register fragments: a step computes 8/S output rows
// from the ring and refills every slot as soon as its last reader has issued, so the loads run 5 input rows ahead of
// the matrix instructions for the whole walk. Narrow images sit side by side in the wave (`lpi` lane columns each).
// LR: the layer has LeakyReLU. Decided per value it made a signed result 12 vector instructions where it is 8 without.
template <int S, int EPI, bool ODDW, int KS, bool LR>
__global__ void __launch_bounds__(64) conv_dw3x3_mfma_kernel(const int8_t* __restrict__ x, const int8_t* __restrict__ wa,
                                                              void* __restrict__ out, DwArgs g) {
    constexpr int RING = 8, U = RING / S;  // U output rows per step
    constexpr int PH = 4 / S;              // output pixels per lane column
    constexpr int T = S == 1 ? 2 : 1;      // A sets
    const Epilogue ep = g.epilogue();
    const int C8 = g.c8, ipw = g.ipw, rps = g.rps;
    // Workgroups go to the 8 XCDs round-robin in launch order. Work items that share input cache lines - the column
    // chunks of a row (a 128-byte line straddles the chunk border), the strip groups of a plane (halo rows), the
    // octets of an image - get consecutive indices on ONE XCD, so that a shared line comes from memory once.
    unsigned w = blockIdx.y * g.gx + blockIdx.x;
    const unsigned per = g.total / 8;
    if (w < per * 8) w = (w % 8) * per + w / 8;
    const unsigned by = div_by(w, FastDiv{g.gx_m, g.gx_s, g.gx}), bx = w - by * g.gx;
    const unsigned img = div_by(by, FastDiv{g.c8_m, g.c8_s, g.c8}), sg = div_by(bx, FastDiv{g.chunks_m, g.chunks_s, g.chunks});
    const int o = (int)(by - img * (unsigned)C8), n0 = (int)img * ipw, chunk = (int)(bx - sg * g.chunks);
    const int strip = (int)sg;
    const int lane = threadIdx.x, n = lane & 15, q = lane >> 4;
    int di = 0, nl = chunk * 16 + n;  // image within the wave, lane column within the image
    if (ipw > 1) {
        di = n * g.lpi_m >> 8;
        nl = n - di * g.lpi;
    }
    const bool lane_ok = di < ipw && n0 + di < g.N;

    v4i a[KS][T];
    {
        const v4i* ap = reinterpret_cast<const v4i*>(wa) + (size_t)o * KS * T * 64 + lane;
#pragma unroll
        for (int dy = 0; dy < KS; ++dy)
#pragma unroll
            for (int t = 0; t < T; ++t) a[dy][t] = ap[(dy * T + t) * 64];
    }

    // ---- input: one 16-byte load per lane and row; per-lane byte offset fixed for the walk + per-row scalar offset --
    const unsigned HW8 = (unsigned)(g.H * g.W * 8);
    const int ic = 4 * nl - 2 + 2 * q;  // first input pixel of this lane's pair
    const bool in_ok = lane_ok && ic >= 0 && ic < g.W;
    const unsigned v_in = in_ok ? (unsigned)di * (unsigned)C8 * HW8 + (unsigned)ic * 8u : DW_OOB;
    const unsigned v_in2 = (in_ok && ic + 1 < g.W) ? v_in + 8u : DW_OOB;  // second pixel of the pair (odd widths only)
    const unsigned s_in = (unsigned)(n0 * C8 + o) * HW8;
    const int oy0 = strip * rps;
    const int iy0 = oy0 * S - g.ph;
    const int rows_needed = (min(rps, g.OH - oy0) - 1) * S + KS;  // input rows this strip really reads
    const unsigned row_end = (unsigned)min(g.H, iy0 + rows_needed);
    // j: input row relative to iy0; rows outside the image or the strip read zero, through a descriptor of no bytes
    auto load_row = [&](int j) -> v4i {
        const int iy = iy0 + j;
        const bool ok = (unsigned)iy < row_end;  // wave-uniform
        const __amdgpu_buffer_rsrc_t r = dw_rsrc(x, ok ? g.in_bytes : 0u);
        const unsigned s_row = ok ? s_in + (unsigned)(iy * g.W * 8) : 0u;
        if constexpr (ODDW) {  // odd width: a row ends on half a pair, which is loaded as 8 bytes + zero
            const v2i lo = __builtin_bit_cast(v2i, __builtin_amdgcn_raw_buffer_load_b64(r, (int)v_in, (int)s_row, 0));
            const v2i hi = __builtin_bit_cast(v2i, __builtin_amdgcn_raw_buffer_load_b64(r, (int)v_in2, (int)s_row, 0));
            return v4i{lo[0], lo[1], hi[0], hi[1]};
        }
        return __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(r, (int)v_in, (int)s_row, 0));
    };
    v4i frag[RING];
#pragma unroll
    for (int j = 0; j < RING; ++j) frag[j] = load_row(j);

    // ---- epilogue constants: stride 1 -> the octet's 8 channels (same for every lane); stride 2 -> this lane's 4 ----
    const int ch = 8 * o + (S == 1 ? 0 : 4 * (q & 1));
    v4i si[T], bi[T], so[T];
#pragma unroll
    for (int t = 0; t < T; ++t) {
        si[t] = *reinterpret_cast<const v4i*>(ep.scale_in + ch + 4 * t);
        bi[t] = *reinterpret_cast<const v4i*>(ep.bias + ch + 4 * t);
        so[t] = v4i{0, 0, 0, 0};
        if constexpr (EPI != EPI_F32_P4 && EPI != EPI_F32_P8 && EPI != EPI_F32_SLICE) so[t] = *reinterpret_cast<const v4i*>(ep.scale_out + ch + 4 * t);
        // the bias is the fma's vector operand in every row: keep it resident (the compiler would otherwise re-copy
        // it from scalar registers row after row)
#pragma unroll
        for (int e = 0; e < 4; ++e) asm volatile("" : "+v"(bi[t][e]));
    }
    if constexpr (EPI == EPI_I8_P8_FULL)
#pragma unroll
        for (int t = 0; t < T; ++t) so[t] = dw_doubled(so[t]);
    unsigned qh[T][2] = {};
    if constexpr (EPI == EPI_I8_P8_NONNEG) {
#pragma unroll
        for (int t = 0; t < T; ++t) {
            qh[t][0] = dw_clamp_pair(ep, so[t][0], so[t][1]);
            qh[t][1] = dw_clamp_pair(ep, so[t][2], so[t][3]);
        }
    }

    // ---- output: this lane's pixel of the row, same addressing scheme ----------------------------------------------
    const unsigned OHW = (unsigned)(g.OH * g.OW);
    const int ox = PH * nl + (S == 1 ? q : (q >> 1));
    const bool st_ok = lane_ok && ox < g.OW;
    unsigned v_out, s_out, row_bytes;
    if constexpr (EPI == EPI_F32_P4) {  // Float4: [N][C/4][OH*OW][4 floats]; packs 2o and 2o+1
        v_out = st_ok ? ((unsigned)di * (unsigned)(2 * C8) + (S == 1 ? 0u : (unsigned)(q & 1))) * OHW * 16u + (unsigned)ox * 16u
                      : DW_OOB;
        s_out = (unsigned)(n0 * (2 * C8) + 2 * o) * OHW * 16u;
        row_bytes = (unsigned)g.OW * 16u;
    } else if constexpr (EPI == EPI_F32_P8) {  // Float8: [N][C/8][OH*OW][8 floats]; a lane's sets are the pixel's halves
        v_out = st_ok ? (unsigned)di * (unsigned)C8 * OHW * 32u + (unsigned)ox * 32u + (S == 1 ? 0u : (unsigned)(q & 1) * 16u)
                      : DW_OOB;
        s_out = (unsigned)(n0 * C8 + o) * OHW * 32u;
        row_bytes = (unsigned)g.OW * 32u;
    } else {  // Byte8: [N][C/8][OH*OW][8 bytes], or (EPI_F32_SLICE) a slice of such a blob: the quantized result where a Concat would put it
        const unsigned octets = EPI == EPI_F32_SLICE ? g.octets : (unsigned)C8;
        v_out = st_ok ? (unsigned)di * octets * OHW * 8u + (unsigned)ox * 8u + (S == 1 ? 0u : (unsigned)(q & 1) * 4u)
                      : DW_OOB;
        s_out = ((unsigned)n0 * octets + (unsigned)o) * OHW * 8u;
        row_bytes = (unsigned)g.OW * 8u;
    }
    const __amdgpu_buffer_rsrc_t rout = dw_rsrc(out, g.out_bytes);

    // Software pipeline, one output row deep: a step issues the matrix instructions of row r+1, refills the ring slots
    // they free, and then runs the epilogue of row r while those instructions execute. The scheduling barriers keep
    // the compiler from batching all matrix instructions at the top of the loop (which exposes the load latency).
    auto row_mfma = [&](int u, v4i (&acc)[T]) {  // u: output row within the step (ring phase)
#pragma unroll
        for (int t = 0; t < T; ++t) {
            acc[t] = v4i{0, 0, 0, 0};
#pragma unroll
            for (int dy = 0; dy < KS; ++dy)
                acc[t] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[dy][t], frag[(u * S + dy) % RING], acc[t], 0, 0, 0);
        }
    };
    v4i cur[T], nxt[T];
    row_mfma(0, cur);

    auto epilogue_store = [&](unsigned v_o, unsigned s_row, bool row_ok) {
        if constexpr (EPI == EPI_F32_P4 || EPI == EPI_F32_P8) {
#pragma unroll
            for (int t = 0; t < T; ++t) {
                const v4i res = dw_dequant4<LR ? 1 : 0>(ep, cur[t], si[t], bi[t]);
                // the second set's channels 4..7: the next Float4 pack is one plane further, in Float8 they follow
                const unsigned vo_t = (t == 0 || !row_ok) ? v_o : v_o + (EPI == EPI_F32_P4 ? OHW * 16u : 16u);
                store_b128_row(res, rout, vo_t, s_row);
            }
        } else if constexpr (EPI == EPI_F32_SLICE) {  // (stride 1)
            v2i w2;
#pragma unroll
            for (int t = 0; t < 2; ++t) w2[t] = quantize4(dw_dequant4<LR ? 1 : 0>(ep, cur[t % T], si[t % T], bi[t % T]), g.q_scale<LR>(), g.half);
            __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(v2u_store, w2), rout, (int)v_o, (int)s_row, 0);
        } else {
            constexpr int CLAMP = epi_clamp(EPI);
            if constexpr (S == 1) {
                v2i w2;
                w2[0] = (int)dw_requant4<CLAMP, LR ? 1 : 0>(ep, cur[0], si[0], bi[0], so[0], qh[0][0], qh[0][1]);
                w2[1] = (int)dw_requant4<CLAMP, LR ? 1 : 0>(ep, cur[T - 1], si[T - 1], bi[T - 1], so[T - 1], qh[T - 1][0], qh[T - 1][1]);
                __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(v2u_store, w2), rout, (int)v_o, (int)s_row, 0);
            } else {
                const unsigned w1 = dw_requant4<CLAMP, LR ? 1 : 0>(ep, cur[0], si[0], bi[0], so[0], qh[0][0], qh[0][1]);
                __builtin_amdgcn_raw_buffer_store_b32(w1, rout, (int)v_o, (int)s_row, 0);
            }
        }
    };

    const int nrows = min(rps, g.OH - oy0);
    unsigned s_st = s_out + (unsigned)oy0 * row_bytes;
    if (rows_needed <= RING) {  // (wave-uniform) a short strip: every input row is in the ring already
#pragma unroll
        for (int u = 0; u < (RING - KS) / S + 1; ++u) {
            if (u + 1 < nrows) row_mfma(u + 1, nxt);
            epilogue_store(v_out, s_st, true);
            if (u + 1 >= nrows) return;
            s_st += row_bytes;
#pragma unroll
            for (int t = 0; t < T; ++t) cur[t] = nxt[t];
        }
        return;
    }
#pragma unroll
    for (int k = 0; k < S; ++k) frag[k % RING] = load_row(k + RING);
    __builtin_amdgcn_sched_barrier(0);
    // A step of U rows is "interior" when every row it stores lies inside the strip and every row it loads inside
    // the image: then the per-row scalar offsets just advance and nothing is predicated. The step at the end of a strip takes the
    // checked path (a strip need not be a whole number of steps). There, too, every load is in the main flow, only sent to nowhere:
    // behind a return between the rows the compiler moves the loads down to their first use, a row's latency each.
    // loads of rows [RING, in_rows_ok) stay inside the image (iy0 + RING > 0); the few an interior step fetches past
    // the strip's own last row are rows the next strip reads anyway
    const __amdgpu_buffer_rsrc_t rin = dw_rsrc(x, g.in_bytes);
    const int in_rows_ok = g.H - iy0;
    const unsigned in_row_bytes = (unsigned)(g.W * 8);
    // (two loops and not one with two paths: a ring slot that either path may refill is refilled elsewhere and copied at the end of a
    // step, which waits for every load in flight)
    int rb = 0;
    for (; rb + U <= nrows && (rb + U) * S + S - 1 + RING < in_rows_ok; rb += U) {
        unsigned s_ld = s_in + (unsigned)(iy0 + (rb + 1) * S + RING) * in_row_bytes;
#pragma unroll
        for (int u = 0; u < U; ++u) {
            row_mfma((u + 1) % U, nxt);
#pragma unroll
            for (int k = 0; k < S; ++k) {
                v4i& f = frag[((u + 1) * S + k) % RING];
                if constexpr (ODDW) {
                    const v2i lo = __builtin_bit_cast(v2i, __builtin_amdgcn_raw_buffer_load_b64(rin, (int)v_in, (int)s_ld, 0));
                    const v2i hi = __builtin_bit_cast(v2i, __builtin_amdgcn_raw_buffer_load_b64(rin, (int)v_in2, (int)s_ld, 0));
                    f = v4i{lo[0], lo[1], hi[0], hi[1]};
                } else {
                    f = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(rin, (int)v_in, (int)s_ld, 0));
                }
                s_ld += in_row_bytes;
            }
            epilogue_store(v_out, s_st, true);
            s_st += row_bytes;
#pragma unroll
            for (int t = 0; t < T; ++t) cur[t] = nxt[t];
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    for (; rb < nrows; rb += U) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int r = rb + u;  // output row of the strip whose epilogue runs now
            if (r < nrows) {       // wave-uniform
                // row r+1: its input rows start (r+1)*S rows into the strip; the ring phase repeats every U rows
                row_mfma((u + 1) % U, nxt);
                epilogue_store(v_out, s_st, true);
            }
#pragma unroll
            for (int k = 0; k < S; ++k) frag[((u + 1) * S + k) % RING] = load_row((r + 1) * S + k + RING);
            s_st += row_bytes;
#pragma unroll
            for (int t = 0; t < T; ++t) cur[t] = nxt[t];
            __builtin_amdgcn_sched_barrier(0);
        }
    }
}

constexpr int dwf_lines(int ks) { return ks == 3 ? 4 : 8; }  // a wave's ring of LDS lines
constexpr int dwf_line_bytes(int loads) { return (64 * ((loads + 1) / 2) + 8) * 8; }  // (of loads of 32 pixels each)

// ---------------------------------------------------------------------------------------------------------------------
// The same layer (3x3 or 5x5) straight from an fp32 blob: quantize_to_int8 (Tensor/ConvolutionLayer.cpp:770-775,
// Tensor/QuantizeX86.cpp:402-490) and the depthwise convolution in ONE launch, for a Float8 input ([N][C/8][H*W][8
// floats]) of at most 128 columns. As two launches the int8 copy of the blob is written and read back (c1: 103 MB in +
// 26 MB out + 26 MB back in + 26 MB out); here every fp32 value is read once and nothing but the result is written.
//
// A wave owns one channel octet x the full width x a strip of output rows and walks along the input rows. A row of the
// blob is W x 32 contiguous bytes; lane l of load k takes bytes 16 (64 k + l) .. + 15 of it -- half a pixel, four
// channels -- so that one load instruction reads 1 KB of whole cache lines (NL = 1..4 loads per row for up to 128
// columns). Loading a whole pixel per lane instead (two 16-byte loads 32 bytes apart) touches every cache line twice,
// and the texture addresser, which works per cache line touched, then bounds the kernel: measured 30 us against 24 us.
// The lane quantizes its four values with the layer's input scale and rounding primitive -- every value once -- and
// writes the four bytes into the wave's own ring of four (5x5: eight) LDS lines [pixel + 2][8 B] (pixels -2, -1 and the ones past
// the row's end are zero: the padding columns). The matrix operand of lane (n, g) for column chunk c -- pixels 64c + 4n -
// 2 + 2g and + 1 -- is then one aligned 16-byte LDS read per kernel row. LDS instructions of one wave execute in order, so
// the wave needs no barrier between its lanes' writes and reads. The loads run four input rows ahead of the
// quantization in a ring of registers; the matrix instructions of a row run under the quantization of the next one, its
// epilogue follows that. Rows outside the image or past the strip read zero through the buffer descriptor.
template <int S, int EPI, int NL, int KS>
__global__ void __launch_bounds__(256, 3) conv_dw3x3_f32in_kernel(const float* __restrict__ x, const int8_t* __restrict__ wa,
                                                               void* __restrict__ out, ConvGeom g, Epilogue ep,
                                                               const float* __restrict__ in_scale_p, float in_half, DwGrid dg,
                                                               int n_strips, int rps, unsigned in_bytes, unsigned out_bytes) {
    constexpr int RL = dwf_lines(KS), PF = 4;  // LDS lines / register stages per wave
    constexpr int NCH = (NL + 1) / 2;  // column chunks of 64 pixels (a matrix operand covers 4 x 16 of them)
    const float in_scale = in_scale_p[0];
    constexpr int T = S == 1 ? 2 : 1;  // A sets
    constexpr int PH = 4 / S;          // output pixels per lane column
    constexpr int LINE = dwf_line_bytes(NL);
    extern __shared__ __attribute__((aligned(16))) int8_t dwf_lds[];  // [waves][RL][LINE]
    const int C8 = g.C / 8;
    unsigned bx, o_u, img_u;
    dg.locate(&bx, &o_u, &img_u);
    const int o = (int)o_u, img = (int)img_u;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int strip = __builtin_amdgcn_readfirstlane(bx * dg.wpb + wave);
    if (strip >= n_strips) return;  // whole wave
    const int lane = threadIdx.x & 63, n = lane & 15, q = lane >> 4;
    int8_t* const lds = dwf_lds + wave * (RL * LINE);
    // where this lane writes and reads in a line (as offsets: worked out from the pointer, one instance has a register too many)
    const unsigned to = (unsigned)wave * (unsigned)(RL * LINE) + 16u + 4u * lane, from = (unsigned)wave * (unsigned)(RL * LINE) + (4u * n + 2u * q) * 8u;

    // the padding slots of every line: pixels -2, -1 and 32 NL .. 64 NCH + 5 (the row's own pixels from W on are written
    // as zeros with every row)
    for (int i = lane; i < (2 + 64 * NCH + 6 - 32 * NL) * RL; i += 64) {
        constexpr int PADS = 2 + 64 * NCH + 6 - 32 * NL;
        const int line = i / PADS, k = i % PADS;
        const int slot = k < 2 ? k : 32 * NL + k;
        *reinterpret_cast<v2i*>(lds + line * LINE + slot * 8) = v2i{0, 0};
    }

    // ---- input: this lane's 16 bytes of the row in every load ---------------------------------------------------------
    const unsigned HW32 = (unsigned)(g.H * g.W) * 32u;
    const unsigned s_in = (unsigned)(img * C8 + o) * HW32;
    unsigned v_in[NL];
#pragma unroll
    for (int k = 0; k < NL; ++k) v_in[k] = 64 * k + lane < 2 * g.W ? (unsigned)(64 * k + lane) * 16u : DW_OOB;
    const __amdgpu_buffer_rsrc_t rin = dw_rsrc(x, in_bytes);
    const int oy0 = strip * rps;
    const int nrows = min(rps, g.OH - oy0);
    const int iy0 = oy0 * S - g.ph;
    const int nq = (nrows - 1) * S + KS;  // input rows this strip reads
    // Odd strips walk UP: a strip and its neighbour below then read the rows they share at the same end of their walks
    // (both last, or both first), i.e. at about the same time, and the second reader finds them in the XCD's L2 instead
    // of fetching them from memory again (the strips of a plane run side by side on one XCD). Walking up only mirrors
    // the row indices: input row j of the walk is row iy0 + nq - 1 - j, output row r of the walk is the strip's row
    // nrows - 1 - r, and kernel row dy meets the line that holds walk row KS - 1 - dy (the weights are loaded mirrored).
    const bool up = (strip & 1) != 0;  // wave-uniform
    auto issue = [&](int j, v4i (&dst)[NL]) {  // j: input row of the walk
        const int iy = up ? iy0 + nq - 1 - j : iy0 + j;
        const bool ok = iy >= 0 && iy < g.H && j < nq;  // wave-uniform
        // (said to the compiler in so many words: it otherwise loops over the lanes' "different" scalar offsets)
        const unsigned s_row = (unsigned)__builtin_amdgcn_readfirstlane((int)(ok ? s_in + (unsigned)(iy * g.W) * 32u : 0u));
#pragma unroll
        for (int k = 0; k < NL; ++k)
            dst[k] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(rin, (int)(ok ? v_in[k] : DW_OOB), (int)s_row, 0));
    };
    // float2int8 of four values into four bytes (the arithmetic of otter_hip_quantize)
    auto quant4 = [&](const v4i& f) -> int {
        int k[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const float t = __fmul_rn(__int_as_float(f[e]), in_scale);
            k[e] = (int)__fadd_rn(t, __builtin_copysignf(in_half, t));  // toward zero, saturating
        }
        const ohip_v2s top = {127, 127}, bot = {-127, -127};
        ohip_v2s a = __builtin_bit_cast(ohip_v2s, __builtin_amdgcn_cvt_pk_i16(k[0], k[1]));
        ohip_v2s b = __builtin_bit_cast(ohip_v2s, __builtin_amdgcn_cvt_pk_i16(k[2], k[3]));
        a = __builtin_elementwise_max(__builtin_elementwise_min(a, top), bot);
        b = __builtin_elementwise_max(__builtin_elementwise_min(b, top), bot);
        return (int)__builtin_amdgcn_perm(__builtin_bit_cast(unsigned, b), __builtin_bit_cast(unsigned, a), 0x06040200u);
    };
    // lane l of load k holds pixel 32 k + l / 2, channels 4 (l & 1) ..: byte (pixel + 2) * 8 + 4 (l & 1) = 16 + 256 k + 4 l
    auto quant_write = [&](int line, const v4i (&src)[NL]) {
#pragma unroll
        for (int k = 0; k < NL; ++k) *reinterpret_cast<int*>(dwf_lds + to + line * LINE + 256 * k) = quant4(src[k]);
    };

    v4i a[KS][T];  // a[k]: the kernel row that meets the k-th of an output row's lines
    {
        const v4i* ap = reinterpret_cast<const v4i*>(wa) + (size_t)o * KS * T * 64 + lane;
#pragma unroll
        for (int k = 0; k < KS; ++k)
#pragma unroll
            for (int t = 0; t < T; ++t) a[k][t] = ap[((up ? KS - 1 - k : k) * T + t) * 64];
    }
    // (requested before any input row: loads return in order, so the wait for these in front of the first matrix
    // instruction -- which sits inside the loop and is executed on every pass -- then never reaches past a row's loads)
    __builtin_amdgcn_sched_barrier(0);

    v4i ld[PF][NL];
#pragma unroll
    for (int j = 0; j < PF; ++j) issue(j, ld[j]);

    // ---- epilogue constants (as in conv_dw3x3_mfma_kernel) -----------------------------------------------------------
    const int ch = 8 * o + (S == 1 ? 0 : 4 * (q & 1));
    v4i si[T], bi[T], so[T];
#pragma unroll
    for (int t = 0; t < T; ++t) {
        si[t] = *reinterpret_cast<const v4i*>(ep.scale_in + ch + 4 * t);
        bi[t] = *reinterpret_cast<const v4i*>(ep.bias + ch + 4 * t);
        so[t] = v4i{0, 0, 0, 0};
        if constexpr (EPI != EPI_F32_P4 && EPI != EPI_F32_P8) so[t] = *reinterpret_cast<const v4i*>(ep.scale_out + ch + 4 * t);
    }
    if constexpr (EPI == EPI_I8_P8_FULL)
#pragma unroll
        for (int t = 0; t < T; ++t) so[t] = dw_doubled(so[t]);
    unsigned qh[T][2] = {};
    if constexpr (EPI == EPI_I8_P8_NONNEG) {
#pragma unroll
        for (int t = 0; t < T; ++t) {
            qh[t][0] = dw_clamp_pair(ep, so[t][0], so[t][1]);
            qh[t][1] = dw_clamp_pair(ep, so[t][2], so[t][3]);
        }
    }
    // ---- output: this lane's pixel of the row in every column chunk --------------------------------------------------
    const unsigned OHW = (unsigned)(g.OH * g.OW);
    unsigned v_out[NCH], s_out, row_bytes;
#pragma unroll
    for (int c = 0; c < NCH; ++c) {
        const int ox = PH * (16 * c + n) + (S == 1 ? q : (q >> 1));
        const bool st_ok = ox < g.OW;
        if constexpr (EPI == EPI_F32_P4)
            v_out[c] = st_ok ? (S == 1 ? 0u : (unsigned)(q & 1)) * OHW * 16u + (unsigned)ox * 16u : DW_OOB;
        else if constexpr (EPI == EPI_F32_P8)
            v_out[c] = st_ok ? (unsigned)ox * 32u + (S == 1 ? 0u : (unsigned)(q & 1) * 16u) : DW_OOB;
        else
            v_out[c] = st_ok ? (unsigned)ox * 8u + (S == 1 ? 0u : (unsigned)(q & 1) * 4u) : DW_OOB;
    }
    if constexpr (EPI == EPI_F32_P4) s_out = (unsigned)(img * (g.C / 4) + 2 * o) * OHW * 16u, row_bytes = (unsigned)g.OW * 16u;
    else if constexpr (EPI == EPI_F32_P8) s_out = (unsigned)(img * C8 + o) * OHW * 32u, row_bytes = (unsigned)g.OW * 32u;
    else s_out = (unsigned)(img * C8 + o) * OHW * 8u, row_bytes = (unsigned)g.OW * 8u;
    const __amdgpu_buffer_rsrc_t rout = dw_rsrc(out, out_bytes);

    v4i cur[NCH][T];
    auto epilogue_store = [&](int r) {  // output row r of the walk, from cur
        const unsigned s_row =
            (unsigned)__builtin_amdgcn_readfirstlane((int)(s_out + (unsigned)(oy0 + (up ? nrows - 1 - r : r)) * row_bytes));
#pragma unroll
        for (int c = 0; c < NCH; ++c) {
            if constexpr (EPI == EPI_F32_P4 || EPI == EPI_F32_P8) {
#pragma unroll
                for (int t = 0; t < T; ++t) {
                    const v4i res = dw_dequant4(ep, cur[c][t], si[t], bi[t]);
                    const unsigned vo_t = (t == 0 || v_out[c] == DW_OOB) ? v_out[c] : v_out[c] + (EPI == EPI_F32_P4 ? OHW * 16u : 16u);
                    store_b128_row(res, rout, vo_t, s_row);
                }
            } else {
                constexpr int CLAMP = epi_clamp(EPI);
                if constexpr (S == 1) {
                    v2i w2;
                    w2[0] = (int)dw_requant4<CLAMP>(ep, cur[c][0], si[0], bi[0], so[0], qh[0][0], qh[0][1]);
                    w2[1] = (int)dw_requant4<CLAMP>(ep, cur[c][T - 1], si[T - 1], bi[T - 1], so[T - 1], qh[T - 1][0], qh[T - 1][1]);
                    __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(v2u_store, w2), rout, (int)v_out[c], (int)s_row, 0);
                } else {
                    const unsigned w1 = dw_requant4<CLAMP>(ep, cur[c][0], si[0], bi[0], so[0], qh[0][0], qh[0][1]);
                    __builtin_amdgcn_raw_buffer_store_b32(w1, rout, (int)v_out[c], (int)s_row, 0);
                }
            }
        }
    };
    auto row_mfma = [&](int line0) {  // the input rows of an output row sit in lines line0, +1, .. (mod RL)
#pragma unroll
        for (int c = 0; c < NCH; ++c) {
            v4i b[KS];
#pragma unroll
            for (int dy = 0; dy < KS; ++dy)
                b[dy] = *reinterpret_cast<const v4i*>(dwf_lds + from + ((line0 + dy) % RL) * LINE + 512 * c);
#pragma unroll
            for (int t = 0; t < T; ++t) {
                cur[c][t] = v4i{0, 0, 0, 0};
#pragma unroll
                for (int dy = 0; dy < KS; ++dy) cur[c][t] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[dy][t], b[dy], cur[c][t], 0, 0, 0);
            }
        }
    };

    // Input row j of the walk sits in line j % RL and register stage j % 4 and completes output row (j - KS + 1) / S when that is
    // whole. Rows 0..KS - 1 (everything up to the first output row) run in front of the loop, so that every pass of the loop
    // issues the same loads and stores on every path: the waits for a row's loads are counted back from the youngest
    // request, and a path with fewer requests would pull them (and with them the loads in flight) closer.
    // (where the rows in front of the loop have no output row to store yet they issue stores that go nowhere -- an
    // out-of-range offset -- so that the count of requests behind a row's loads is the loop's own from the first pass on)
    auto no_store = [&](int i) {  // (a different nowhere each time, or the compiler drops all but the last as dead stores)
#pragma unroll
        for (int c = 0; c < NCH; ++c) {
            const int nowhere = (int)(DW_OOB + 256u * (unsigned)i + 64u * (unsigned)c);
            if constexpr (EPI == EPI_F32_P4 || EPI == EPI_F32_P8) {
#pragma unroll
                for (int t = 0; t < T; ++t)
                    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(v4u_store, v4i{0, 0, 0, 0}), rout, nowhere + 16 * t, 0, 0);
            } else if constexpr (S == 1) {
                __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(v2u_store, v2i{0, 0}), rout, nowhere, 0, 0);
            } else {
                __builtin_amdgcn_raw_buffer_store_b32(0u, rout, nowhere, 0, 0);
            }
        }
    };
    auto input_row = [&](int j, int jj, bool store_prev) {  // jj = j modulo 8; both a compile-time constant at every call
        quant_write(jj % RL, ld[jj % PF]);
        issue(j + PF, ld[jj % PF]);
        if ((jj - (KS - 1) + 8) % S == 0) {
            if (store_prev) epilogue_store((j - (KS - 1)) / S - 1);
            else no_store(j);
            row_mfma((jj - (KS - 1) + 8) % RL);
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    no_store(KS);
#pragma unroll
    for (int i = 0; i < KS; ++i) input_row(i, i, false);
    // (eight rows per pass: the waits the compiler places in the first rows of a pass reach a row or two further back
    // than the ring needs, so the passes are long)
    constexpr int UNR = 8;
    const int steps = (nq - KS) / UNR;
    int jb = KS;
    for (int st = 0; st < steps; ++st, jb += UNR) {
#pragma unroll
        for (int i = 0; i < UNR; ++i) input_row(jb + i, KS + i, true);
    }
#pragma unroll
    for (int i = 0; i < UNR - 1; ++i)
        if (jb + i < nq) input_row(jb + i, KS + i, true);  // wave-uniform
    epilogue_store(nrows - 1);
}

// true when the fused fp32 -> depthwise launch takes this layer and blob (Float8 input; the caller has checked
// dw_mfma_applicable)
bool dw_f32in_applicable(const ConvGeom& g, int in_layout) {
    if (in_layout != OTTER_HIP_F32_P8) return false;
    if (g.W > 128 || g.C % 8 != 0) return false;
    if ((size_t)g.N * g.C * g.H * g.W * 4 >= ((size_t)1 << 31)) return false;  // 32-bit buffer offsets
    return (long)g.N * (g.C / 8) <= 65535;
}

// strips of equal height, about two waves per SIMD over the chip (as in run_conv_dw_mfma)
static int dw_f32in_rows(const ConvGeom& g) {
    const long planes = (long)g.N * (g.C / 8);
    int ns = 1;
    while (ns < g.OH && ns * planes < 2048) ++ns;
    return (g.OH + ns - 1) / ns;
}

// Whether this launch is faster than a quantize pass and the int8 kernel: 3x3 on 17 columns and more, wherever it can run (0.80 of the time over 2800
// drawn layers); narrower images, of whose rows a wave fills a part of its lanes, and 5x5, which reads four rows more for a strip, by models of the
// two (us, launches replayed from graphs; fitted to 3670 drawn layers while every workgroup had four waves' LDS lines, half within 6 and 3 %, nine in ten within
// 16 and 8 %). Of 31780 drawn layers that the rule takes one launch needs 0.80 of the time of two, the faster of both each time 0.80; 234 are over 5 % slower, the worst 1.19. Of
// calls one by one, which the host bounds: 0.67. 360 channels 5x5 @22x22 b2 6.0 us as two; 120 3x3 @13x13 b10 5.0.
bool dw_f32in_faster(const ConvGeom& g, int out_bytes) {
    if (g.kh == 3 && g.W >= 17) return true;
    const int rps = dw_f32in_rows(g), NL = (g.W + 31) / 32, T = g.sh == 1 ? 2 : 1;
    const float planes = (float)g.N * (g.C / 8), in = planes * (float)(g.H * g.W) * 8e-6f, res = planes * (float)(g.OH * g.OW) * 8e-6f;
    const float m = std::max(planes * (float)((g.OH + rps - 1) / rps) / 1024.f, 1.f), rows = (float)((rps - 1) * g.sh + g.kh);
    const float one = 4.63f + m * (0.0235f * rows * NL + (float)(rps * ((NL + 1) / 2) * T) * (g.kh == 5 ? 0.1506f : 0.087f)) + 0.415f * in + 0.0193f * res * out_bytes;
    const float two = 5.99f + 0.858f * in + (g.kh == 5 ? 0.143f * res : 0.f) + 0.4f * planes * (float)(g.OH * ((g.OW + 3) / 4 * 4)) * 8e-6f + 2.5e-5f * std::max(0.f, planes - 2048.f);
    return one < two;
}

hipError_t run_conv_dw_f32in(const float* x, const int8_t* wa, void* out, const ConvGeom& g, const Epilogue& ep, int epi,
                             const float* in_scale, int in_round_mode, int strip_rows, hipStream_t stream) {
    if (g.N == 0 || g.OH * g.OW == 0) return hipSuccess;
    const int C8 = g.C / 8;
    const long planes = (long)g.N * C8;
    if (planes > 65535) return hipErrorInvalidValue;
    const int rps = strip_rows > 0 ? std::min(strip_rows, g.OH) : dw_f32in_rows(g);
    const int n_strips = (g.OH + rps - 1) / rps;
    const int wpb = n_strips % 4 == 0 ? 4 : (n_strips % 2 == 0 ? 2 : 1);
    const dim3 grid((unsigned)(n_strips / wpb), (unsigned)planes), block(64 * wpb);
    const float in_half = in_round_mode == OTTER_HIP_ROUND_SSE ? 0.5f : 0.49999997f;
    // A grid of a few workgroups per CU is resident all at once, and the dispatcher is free to give one CU three of them
    // and another one: the kernel then lasts as long as the fullest CU. Reserving a share of the CU's 160 KB of LDS per
    // workgroup (beyond its waves' lines) caps the workgroups per CU at the even share.
    // (The lines are those of the waves that there are: with four waves' for every workgroup, 35 KB with a 5x5 window, a CU held four of the one-wave
    // workgroups of an odd number of strips, and more than 1024 of them were two rounds: 120 channels 5x5 @80x80 b4 11.4 -> 8.5 us, as two launches 9.6)
    const long wgs = (long)grid.x * grid.y, per_cu = (wgs + 255) / 256;
    unsigned lds = (unsigned)(wpb * dwf_lines(g.kh) * dwf_line_bytes((g.W + 31) / 32));
    if (wpb == 4 && per_cu >= 2 && per_cu <= 3) lds = std::max(lds, std::min(63u * 1024, (unsigned)(160 * 1024 / per_cu - 1024) / 1024 * 1024));  // (within the default 64 KB limit)
    const unsigned in_bytes = (unsigned)((size_t)g.N * g.C * g.H * g.W * 4);
    const unsigned out_bytes = (unsigned)((size_t)g.N * g.K * g.OH * g.OW * (epi == EPI_F32_P4 || epi == EPI_F32_P8 ? 4 : 1));
#define OHIP_DWF_L(S_, E_, L_)                                                                                           \
    do {                                                                                                                 \
        if (g.kh == 3)                                                                                                   \
            launch((conv_dw3x3_f32in_kernel<S_, E_, L_, 3>), grid, block, lds, stream, x, wa, out, g, ep, in_scale, in_half, \
                   DwGrid::of(grid.x, grid.y, (unsigned)C8, wpb), n_strips, rps, in_bytes, out_bytes);                   \
        else                                                                                                             \
            launch((conv_dw3x3_f32in_kernel<S_, E_, L_, 5>), grid, block, lds, stream, x, wa, out, g, ep, in_scale, in_half, \
                   DwGrid::of(grid.x, grid.y, (unsigned)C8, wpb), n_strips, rps, in_bytes, out_bytes);                   \
    } while (0)
#define OHIP_DWF_N(S_, E_)                       \
    do {                                         \
        switch ((g.W + 31) / 32) {               \
        case 1: OHIP_DWF_L(S_, E_, 1); break;    \
        case 2: OHIP_DWF_L(S_, E_, 2); break;    \
        case 3: OHIP_DWF_L(S_, E_, 3); break;    \
        default: OHIP_DWF_L(S_, E_, 4); break;   \
        }                                        \
    } while (0)
#define OHIP_DWF_E(S_)                                                  \
    do {                                                                \
        const int e = full_epilogue(epi, ep);                           \
        if (e == EPI_I8_P8_FULL) OHIP_DWF_N(S_, EPI_I8_P8_FULL);        \
        else if (epi == EPI_I8_P8_NONNEG) OHIP_DWF_N(S_, EPI_I8_P8_NONNEG); \
        else if (epi == EPI_I8_P8) OHIP_DWF_N(S_, EPI_I8_P8);           \
        else if (epi == EPI_F32_P8) OHIP_DWF_N(S_, EPI_F32_P8);         \
        else OHIP_DWF_N(S_, EPI_F32_P4);                                \
    } while (0)
    if (g.sh == 1) OHIP_DWF_E(1);
    else OHIP_DWF_E(2);
#undef OHIP_DWF_E
#undef OHIP_DWF_N
#undef OHIP_DWF_L
    return hipGetLastError();
}

// the epilogue code of a depthwise layer: the common rule, plus fp32 output in the depthwise default layout Float8
int dw_mfma_epilogue(const Epilogue& ep, int K) {
    const int epi = pick_epilogue(ep, K);
    const bool clamp_act = ep.act == 0 || ep.act == 1 || ep.act == 3 || (ep.act == 2 && ep.lrelu);
    if (epi == EPI_GENERIC && clamp_act && ep.out_kind == OTTER_HIP_OUT_F32 && ep.out_layout == OTTER_HIP_F32_P8 && K % 8 == 0)
        return EPI_F32_P8;
    return epi;
}

// true when this layer / batch can take the matrix-core kernel (the caller falls back to the vector kernels otherwise)
bool dw_mfma_applicable(const ConvGeom& g, const Epilogue& ep, int epi, bool scale_out_positive) {
    if (epi == EPI_I8_P8_NONNEG && !scale_out_positive) return false;  // the clamp is moved past the output scale
    if (!(g.kh == g.kw && (g.kh == 3 || g.kh == 5) && g.dh == 1 && g.dw == 1 && g.sh == g.sw && (g.sh == 1 || g.sh == 2))) return false;
    if (g.ph > g.kh / 2 || !dw_mfma_window_fits(g.kh, g.sh, g.pw) || g.C % 8 != 0 || g.C != g.K) return false;
    if (epi != EPI_I8_P8 && epi != EPI_I8_P8_NONNEG && epi != EPI_F32_P4 && epi != EPI_F32_P8) return false;
    const size_t in_bytes = (size_t)g.N * g.C * g.H * g.W;
    const size_t out_bytes = (size_t)g.N * g.K * g.OH * g.OW * (epi == EPI_F32_P4 || epi == EPI_F32_P8 ? 4 : 1);
    return in_bytes < ((size_t)1 << 31) && out_bytes < ((size_t)1 << 31);  // 32-bit buffer offsets
}

// strip_blocks: 0 = automatic, > 0: steps of 8 / stride output rows of a strip, < 0: rows of it
hipError_t run_conv_dw_mfma(const int8_t* x, const int8_t* wa, void* out, const ConvGeom& g, const Epilogue& ep, int epi,
                            int strip_blocks, hipStream_t stream) {
    const JoinArgs* const slice = epi == EPI_F32_SLICE ? ep.join : nullptr;
    if (slice != nullptr && g.sh != 1) return hipErrorInvalidValue;
    if (g.N == 0 || g.OH * g.OW == 0) return hipSuccess;
    const int C8 = g.C / 8;
    const int PH = 4 / g.sh;  // output pixels per lane column
    // lane columns an image row needs
    const int cols = (g.OW + PH - 1) / PH;
    int lpi = 16, ipw = 1, col_chunks = (cols + 15) / 16;
    if (cols <= 8) {  // narrow images side by side in one wave
        lpi = cols;
        ipw = std::min(16 / lpi, g.N);
        col_chunks = 1;
    }
    const long groups = (long)((g.N + ipw - 1) / ipw) * C8;
    if (groups > 65535) return hipErrorInvalidValue;  // grid.y limit; the caller splits the batch
    const int U = 8 / g.sh;
    const int rps = strip_blocks > 0   ? std::min(strip_blocks, (g.OH + U - 1) / U) * U
                    : strip_blocks < 0 ? std::min(-strip_blocks, g.OH)
                                       : DwStrips(g.OH, g.sh, g.kh, epi == EPI_I8_P8_NONNEG ? 1 : epi == EPI_I8_P8 || slice ? 0 : 2,
                                                  (float)(col_chunks * groups)).choose();
    const int n_strips = (g.OH + rps - 1) / rps;
    // a workgroup is one strip: with two and four strips a workgroup, and shares of LDS reserved to even them out over the compute
    // units, 140 drawn layers were 2 % and 5 % slower at their best strip height
    const dim3 grid((unsigned)(col_chunks * n_strips), (unsigned)groups), block(64);
    const unsigned in_bytes = (unsigned)((size_t)g.N * g.C * g.H * g.W);
    const unsigned out_bytes = (unsigned)((size_t)g.N * g.K * g.OH * g.OW * (epi == EPI_F32_P4 || epi == EPI_F32_P8 ? 4 : 1));
    const size_t slice_bytes = slice ? ((size_t)(g.N - 1) * slice->slice_octets + C8) * g.OH * g.OW * 8 : 0;
    const FastDiv gx = fast_div(grid.x), c8 = fast_div((unsigned)C8), ch = fast_div((unsigned)col_chunks);
    DwArgs pl{};
    pl.scale_in = ep.scale_in, pl.bias = ep.bias, pl.scale_out = ep.scale_out;
    pl.gx_m = gx.m, pl.gx_s = (unsigned char)gx.s, pl.gx = grid.x, pl.c8_m = c8.m, pl.c8_s = (unsigned char)c8.s, pl.c8 = (unsigned short)C8;
    pl.chunks_m = ch.m, pl.chunks_s = (unsigned char)ch.s, pl.chunks = (unsigned)col_chunks;
    pl.lpi = (unsigned char)lpi, pl.lpi_m = (unsigned short)(256 / lpi + 1), pl.ipw = (unsigned char)ipw;
    pl.N = g.N, pl.H = g.H, pl.W = g.W, pl.OH = g.OH, pl.OW = g.OW, pl.ph = (unsigned char)g.ph, pl.rps = rps;
    pl.total = grid.x * grid.y, pl.in_bytes = in_bytes, pl.out_bytes = slice ? (unsigned)slice_bytes : out_bytes;
    pl.p0 = ep.act_p0, pl.lo = ep.act_lo, pl.hi = ep.act_hi, pl.half = ep.round_half, pl.lrelu = ep.lrelu;
    if (slice) pl.octets = (unsigned)slice->slice_octets, pl.half = slice->slice_half, (ep.lrelu ? pl.lo : pl.p0) = slice->slice_scale;
    static_assert(sizeof(DwArgs) == 112);
#define OHIP_DWM_L(S_, E_, O_, K_)                                                                                        \
    do {                                                                                                                   \
        if (epi_clamp(E_) == 0 && ep.lrelu)                                                                                \
            launch((conv_dw3x3_mfma_kernel<S_, E_, O_, K_, epi_clamp(E_) == 0>), grid, block, 0, stream, x, wa, out, pl);  \
        else                                                                                                               \
            launch((conv_dw3x3_mfma_kernel<S_, E_, O_, K_, false>), grid, block, 0, stream, x, wa, out, pl);    \
    } while (0)
#define OHIP_DWM_K(S_, E_, O_)                  \
    do {                                        \
        if (g.kh == 3) OHIP_DWM_L(S_, E_, O_, 3); \
        else OHIP_DWM_L(S_, E_, O_, 5);         \
    } while (0)
#define OHIP_DWM(S_, E_) \
    do {                                                                                                               \
        if (g.W & 1)                                                                                                   \
            OHIP_DWM_K(S_, E_, true);                                                                                  \
        else                                                                                                           \
            OHIP_DWM_K(S_, E_, false);                                                                                 \
    } while (0)
#define OHIP_DWM_E(S_)                                                \
    do {                                                              \
        const int e = full_epilogue(epi, ep);                         \
        if (e == EPI_I8_P8_FULL) OHIP_DWM(S_, EPI_I8_P8_FULL);        \
        else if (epi == EPI_I8_P8_NONNEG) OHIP_DWM(S_, EPI_I8_P8_NONNEG); \
        else if (epi == EPI_I8_P8) OHIP_DWM(S_, EPI_I8_P8);           \
        else if (epi == EPI_F32_P8) OHIP_DWM(S_, EPI_F32_P8);         \
        else OHIP_DWM(S_, EPI_F32_P4);                                \
    } while (0)
    if (slice != nullptr) OHIP_DWM(1, EPI_F32_SLICE);
    else if (g.sh == 1) OHIP_DWM_E(1);
    else OHIP_DWM_E(2);
#undef OHIP_DWM_E
#undef OHIP_DWM_K
#undef OHIP_DWM_L
#undef OHIP_DWM
    return hipGetLastError();
}

}  // namespace ohip
