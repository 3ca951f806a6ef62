// 3x3 convolution of an image with very few channels (an RGB stem: 3 -> 24 / 32 channels, stride 2), straight from the
// unpacked blob -- fp32 quantized on the way (Tensor/QuantizeX86.cpp:617-641) or int8 -- with no channel-padded copy
// in between. Replaces the reference's pack1to4 path (conv2d_3x3s2_int8_pack1to4_x86 / sgemm pack1to4,
// Tensor/ConvolutionMM2DInt8X86Pack.cpp:148-841) for these shapes.
//
// The reduction is only C*9 <= 45 long, so one v_mfma_i32_16x16x64_i8 holds all of it: B column n is an output pixel,
// its 64 reduction bytes are split over the four lanes (n, kg): lane kg < 3 supplies kernel ROW kg -- the 3 x C input
// values of that row under the window -- and lane kg = 3 supplies bytes that meet zero weights. A rows are 16 output
// channels with the same byte order (zero where there is no tap). A wave owns 16 consecutive pixels of an output row;
// per row it issues one MFMA per 16 output channels and stores 4 channels of its pixel per MFMA (one Float4 element,
// or half a Byte8 element).
//
// Up to 4 channels (conv_stem3x3_lds_kernel): a workgroup first quantizes the input rows of a strip of output rows into
// LDS, every value once, with 16-byte loads, as int8 lines [input row][channel][pixel]; a lane's operand is then, per
// channel, the dword that starts at its window's first pixel (two LDS dwords and one v_alignbit): byte 4*c + v, the
// fourth byte of each channel (the next pixel) meeting a zero weight. 5 channels (conv_stem3x3_kernel, byte 3*c + v):
// every lane gathers and quantizes its 3*C values itself.
#include <algorithm>
#include <cstdint>
#include <type_traits>

#include "common.hpp"
#include "conv_igemm.hpp"

namespace ohip {

typedef int v4i __attribute__((ext_vector_type(4)));

constexpr int STEM_MAX_C = 5;         // 3*C bytes must fit a lane's 16
constexpr int STEM_LDS_MAX_C = 4;     // 4*C bytes must fit a lane's 16: the kernel that stages the input in LDS
constexpr int STEM_MAX_TILES = 4;     // K <= 64
constexpr int STEM_ROWS_PER_WAVE = 8;

size_t stem_packed_weight_bytes(int K) { return (size_t)((K + 15) / 16) * 64 * 16; }

// w [K][C][3][3] -> [tile][lane = 16*kg + r][byte j] = w[16*tile + r][c][kg][v], j = 4*c + v for up to 4 channels
// (byte 4*c + 3 stays zero), j = 3*c + v for 5
void stem_pack_weights(const int8_t* w, int K, int C, int8_t* dst) {
    const int tiles = (K + 15) / 16;
    const int per = C <= STEM_LDS_MAX_C ? 4 : 3;
    for (int m = 0; m < tiles; ++m)
        for (int lane = 0; lane < 64; ++lane) {
            const int r = lane & 15, kg = lane >> 4, k = 16 * m + r;
            for (int j = 0; j < 16; ++j) {
                const int c = j / per, v = j % per;
                int8_t val = 0;
                if (kg < 3 && v < 3 && c < C && k < K) val = w[(((size_t)k * C + c) * 3 + kg) * 3 + v];
                dst[((size_t)m * 64 + lane) * 16 + j] = val;
            }
        }
}

// (absent channels are loaded from a clamped address and dropped)
template <int MT, bool F32_OUT, bool IN_F32>
__global__ void __launch_bounds__(256) conv_stem3x3_kernel(const void* __restrict__ x_, const int8_t* __restrict__ wpk,
                                                           void* __restrict__ out, ConvGeom g, Epilogue ep,
                                                           const float* __restrict__ in_scale, int in_round,
                                                           int col_groups, int strips, int total_waves) {
    const int wave = __builtin_amdgcn_readfirstlane((int)(blockIdx.x * 4 + (threadIdx.x >> 6)));
    if (wave >= total_waves) return;
    const int lane = threadIdx.x & 63, n = lane & 15, kg = lane >> 4;
    const int cg = wave % col_groups;
    const int strip = (wave / col_groups) % strips;
    const int img = wave / (col_groups * strips);
    const int ox = cg * 16 + n;
    const int S = g.sh;

    v4i a[MT];
#pragma unroll
    for (int m = 0; m < MT; ++m) a[m] = reinterpret_cast<const v4i*>(wpk)[m * 64 + lane];

    // epilogue constants of this lane's channels 16*m + 4*kg + i
    float si[MT][4], bi[MT][4], so[MT][4];
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int ch = 16 * m + 4 * kg + i;
            si[m][i] = ep.scale_in[ch];
            bi[m][i] = ep.bias[ch];
            so[m][i] = F32_OUT ? 0.f : ep.scale_out[ch];
        }
    const float qs = IN_F32 ? in_scale[0] : 0.f;
    const float half = in_round == OTTER_HIP_ROUND_SSE ? 0.5f : 0.49999997f;

    const int ix0 = ox * S - g.pw;
    const bool col_ok = ox < g.OW;
    const size_t plane = (size_t)g.H * g.W;
    const size_t img_in = (size_t)img * g.C * plane;
    const int OHW = g.OH * g.OW;
    const int oy_end = min((strip + 1) * STEM_ROWS_PER_WAVE, g.OH);

    constexpr int NC = STEM_MAX_C;
    const int C = g.C;
    const unsigned plane_u = (unsigned)plane;
    for (int oy = strip * STEM_ROWS_PER_WAVE; oy < oy_end; ++oy) {
        // ---- this lane's 16 reduction bytes: kernel row kg, byte 3*c + v. Every lane loads all of its 3*NC values
        // from clamped (always valid) addresses first, so that the loads are in flight together; what lies outside
        // the image, the channel count or the kernel is zeroed afterwards.
        const int iy = oy * S - g.ph + kg;
        const bool row_ok = kg < 3 && iy >= 0 && iy < g.H && col_ok;
        const unsigned row_off = (unsigned)min(max(iy, 0), g.H - 1) * (unsigned)g.W;
        unsigned col_off[3];
        bool ok[3];
#pragma unroll
        for (int v = 0; v < 3; ++v) {
            const int ix = ix0 + v;
            ok[v] = row_ok && ix >= 0 && ix < g.W;
            col_off[v] = (unsigned)min(max(ix, 0), g.W - 1);
        }
        float fv[3 * NC];
        int q[15];
#pragma unroll
        for (int j = 0; j < 15; ++j) q[j] = 0;
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            const unsigned ch_off = (unsigned)min(c, C - 1) * plane_u + row_off;
#pragma unroll
            for (int v = 0; v < 3; ++v) {
                if constexpr (IN_F32) fv[3 * c + v] = static_cast<const float*>(x_)[img_in + ch_off + col_off[v]];
                else q[3 * c + v] = static_cast<const int8_t*>(x_)[img_in + ch_off + col_off[v]];
            }
        }
#pragma unroll
        for (int c = 0; c < NC; ++c)
#pragma unroll
            for (int v = 0; v < 3; ++v) {
                if constexpr (IN_F32) {
                    const float t = __fmul_rn(fv[3 * c + v], qs);
                    const int r = (int)__fadd_rn(t, __builtin_copysignf(half, t));
                    q[3 * c + v] = min(max(r, -127), 127);
                }
                if (!(ok[v] && c < C)) q[3 * c + v] = 0;
            }
        v4i b;
        b[0] = (q[0] & 0xff) | ((q[1] & 0xff) << 8) | ((q[2] & 0xff) << 16) | (q[3] << 24);
        b[1] = (q[4] & 0xff) | ((q[5] & 0xff) << 8) | ((q[6] & 0xff) << 16) | (q[7] << 24);
        b[2] = (q[8] & 0xff) | ((q[9] & 0xff) << 8) | ((q[10] & 0xff) << 16) | (q[11] << 24);
        b[3] = (q[12] & 0xff) | ((q[13] & 0xff) << 8) | ((q[14] & 0xff) << 16);

        const int pix = oy * g.OW + ox;
#pragma unroll
        for (int m = 0; m < MT; ++m) {
            const v4i acc = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[m], b, v4i{0, 0, 0, 0}, 0, 0, 0);
            const int ch0 = 16 * m + 4 * kg;  // D rows 4*kg .. 4*kg+3 of column n
            if (!col_ok || ch0 >= g.K) continue;
            float v[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                float t = __fmaf_rn((float)acc[i], si[m][i], bi[m][i]);
                t = fminf(fmaxf(t, ep.act_lo), ep.act_hi);
                if (ep.lrelu) t = fmaxf(t, __fmul_rn(t, ep.act_p0));
                v[i] = t;
            }
            if constexpr (F32_OUT) {  // Float4: [N][K/4][OH*OW][4]
                float4* o = reinterpret_cast<float4*>(out) + ((size_t)img * (g.K / 4) + ch0 / 4) * OHW + pix;
                *o = make_float4(v[0], v[1], v[2], v[3]);
            } else {  // Byte8: [N][K/8][OH*OW][8]; these 4 channels are one half of an element
                unsigned pk = 0;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const float t = __fmul_rn(v[i], so[m][i]);
                    const int r = (int)__fadd_rn(t, __builtin_copysignf(ep.round_half, t));
                    pk |= (unsigned)(min(max(r, -127), 127) & 0xff) << (8 * i);
                }
                unsigned* o = reinterpret_cast<unsigned*>(out) + (((size_t)img * (g.K / 8) + ch0 / 8) * OHW + pix) * 2 + (ch0 / 4 & 1);
                *o = pk;
            }
        }
    }
}

// ---------------------------------------------------------------------------------------------------------------------
// Up to 4 channels: the strip's input rows quantized into LDS once, operands from LDS
// ---------------------------------------------------------------------------------------------------------------------

// A workgroup (4 waves) owns R output rows of one image. LDS: [input row r < RIN][channel][pitch_dw dwords] of int8;
// dword d of a line holds pixels 4*(d-1) .. 4*(d-1)+3 (dword 0 and everything past the row's end are zeros: the
// padding columns), rows outside the image are zeros.
enum { STEM_VALUES, STEM_UNITS, STEM_LINES };  // how the strip is loaded
struct StemPlan {
    int R, strips, cgs, RIN, pitch_dw, fill;
    FastDiv by_strips, by_cgs;
    float inv_pitch, inv_c;
};

constexpr int STEM_UN = 8;        // 4-pixel units a thread has in flight while the strip is loaded
constexpr int STEM_POOL_ROWS = 4;  // pooled rows per workgroup with the pooling behind it (2, 4 level from 16 images on, 8 slower below 64)
constexpr int STEM_LDS_ROWS = 4;  // output rows per workgroup (measured: 2, 4, 8 within 5 % of each other at 224 x 224, 16 slower)

// Input rows iy0 .. iy0 + RIN - 1 of an image, quantized, into the LDS lines of a strip, in one of three ways (stem_fill_rule). Those that load
// units of four pixels take fp32 rows of four pixels and more (a 16-byte load at any pixel; the last unit of a row of no whole units is loaded
// where it ends with the row and moved down) and int8 rows of whole, aligned units.

// STEM_LINES: a wave takes lines, 64 units of one at a time. Row and channel of a line are scalar and go on by additions (worked out anew for each
// they were 25 scalar instructions and a branch in front of every load), what is outside the image lies outside a descriptor and is zero, and a unit
// costs its quantization and little else.
template <bool IN_F32, int CT>
__device__ __forceinline__ void stem_fill_lines(unsigned* stem_lds, const void* __restrict__ x_, const ConvGeom& g, const StemPlan& p, size_t img_in, int iy0,
                                                float qs, float half) {
    constexpr unsigned E = IN_F32 ? 4 : 1, OUT = 0x80000000u;
    const unsigned lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int C = CT ? CT : g.C, lines = p.RIN * C;
    const unsigned row = (unsigned)g.W * E, plane = (unsigned)g.H * row, bytes = (unsigned)C * plane;
    const char* const image = static_cast<const char*>(x_) + img_in * E;
    // the wave's first line, and four lines further
    const int r0 = C == 1 ? wave : C == 2 ? wave >> 1 : C == 3 && wave == 3 ? 1 : 0, c0 = wave - r0 * C;
    const int dr = C == 1 ? 4 : C == 2 ? 2 : 1, dc = C == 3 ? 1 : 0;
    for (int d0 = 0; d0 < p.pitch_dw; d0 += 64) {
        const int d = d0 + (int)lane, ix = 4 * (d - 1);
        const int over = max(ix + 4 - g.W, 0);  // pixels of the unit past the row's end
        const unsigned v = ix >= 0 && ix < g.W ? (unsigned)(ix - over) * E : OUT, down = 8u * (unsigned)(over & 3);
        int iy = iy0 + r0, c = c0;
        unsigned at = (unsigned)iy * row + (unsigned)c * plane;
        unsigned* to = stem_lds + wave * p.pitch_dw + d;
        for (int left = lines - wave; left > 0; left -= 4 * STEM_UN) {
            v4i raw[STEM_UN];
#pragma unroll
            for (int j = 0; j < STEM_UN; ++j) {
                const bool in = left > 4 * j && (unsigned)iy < (unsigned)g.H;  // (uniform; a line that does not exist: a descriptor of no bytes)
                const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(image), 0, in ? (int)bytes : 0, 0x00020000);
                if constexpr (IN_F32) raw[j] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(rs, (int)v, in ? (int)at : 0, 0));
                else raw[j][0] = (int)__builtin_amdgcn_raw_buffer_load_b32(rs, (int)v, in ? (int)at : 0, 0);
                iy += dr, c += dc, at += (unsigned)dr * row + (unsigned)dc * plane;
                const bool next = dc != 0 && c >= C;
                iy += next ? 1 : 0, c -= next ? C : 0, at += next ? row - bytes : 0u;
            }
#pragma unroll
            for (int j = 0; j < STEM_UN; ++j) {
                if (left <= 4 * j) break;  // (uniform)
                const unsigned pk = IN_F32 ? (unsigned)quantize4(raw[j], qs, half) >> down : (unsigned)raw[j][0];
                if (d < p.pitch_dw) to[4 * j * p.pitch_dw] = pk;
            }
            to += 4 * STEM_UN * p.pitch_dw;
        }
    }
}

// STEM_UNITS: the units of all lines dealt to the threads. Row, channel and column of a unit are worked out by each (28 vector instructions, as many
// as its quantization), but nothing else stands in front of its load.
typedef v4i v4i_any __attribute__((aligned(4)));  // (four floats of rows of any width)
template <bool IN_F32, int CT>
__device__ __forceinline__ void stem_fill_units(unsigned* stem_lds, const void* __restrict__ x_, const ConvGeom& g, const StemPlan& p, size_t img_in, int iy0,
                                                float qs, float half) {
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int C = CT ? CT : g.C, total = p.RIN * C * p.pitch_dw;
    const unsigned plane = (unsigned)(g.H * g.W);
    for (int base = 0; base < total; base += 256 * STEM_UN) {
        v4i raw[STEM_UN];
        unsigned keep[STEM_UN], down[STEM_UN];
#pragma unroll
        for (int j = 0; j < STEM_UN; ++j) {
            if (base + 256 * j + 64 * wave >= total) continue;  // (none of this wave's units exists)
            // unit idx = dword idx of the LDS image: line = idx / pitch, row = line / C (exact: the quotients' fractional
            // parts stay 0.5 / divisor away from an integer, far more than the rounding of these products)
            const int idx = min(base + 256 * j + tid, total - 1);
            const int line = (int)(((float)idx + 0.5f) * p.inv_pitch);
            const int d = idx - line * p.pitch_dw;
            const int r = (int)(((float)line + 0.5f) * p.inv_c);
            const int c = line - r * C;
            const int iy = iy0 + r, ix = 4 * (d - 1);
            // every load from a clamped (always valid) address, so that all are in flight together; what lies outside
            // the image is zeroed afterwards
            const unsigned off = (unsigned)c * plane + (unsigned)min(max(iy, 0), g.H - 1) * (unsigned)g.W + (unsigned)min(max(ix, 0), g.W - 4);
            if constexpr (IN_F32) raw[j] = *reinterpret_cast<const v4i_any*>(static_cast<const float*>(x_) + img_in + off);
            else raw[j][0] = *reinterpret_cast<const int*>(static_cast<const int8_t*>(x_) + img_in + off);
            keep[j] = iy >= 0 && iy < g.H && ix >= 0 && ix < g.W ? 0xffffffffu : 0u;
            if constexpr (IN_F32) down[j] = 8u * (unsigned)(max(ix + 4 - g.W, 0) & 3);
        }
#pragma unroll
        for (int j = 0; j < STEM_UN; ++j) {
            if (base + 256 * j + 64 * wave >= total) continue;
            const unsigned pk = IN_F32 ? (unsigned)quantize4(raw[j], qs, half) >> down[j] : (unsigned)raw[j][0];
            const int idx = base + 256 * j + tid;
            if (idx < total) stem_lds[idx] = pk & keep[j];
        }
    }
}

// STEM_VALUES: any rows, a value at a time
template <bool IN_F32>
__device__ __forceinline__ void stem_fill_values(unsigned* stem_lds, const void* __restrict__ x_, const ConvGeom& g, const StemPlan& p, int C, size_t img_in,
                                              int iy0, float qs, float half) {
    const int tid = threadIdx.x;
    const int total = p.RIN * C * p.pitch_dw;
    const unsigned plane = (unsigned)(g.H * g.W);
    for (int idx = tid; idx < total; idx += 256) {
        // dword idx of the LDS image: line = idx / pitch, row = line / C (exact: the quotients' fractional
        // parts stay 0.5 / divisor away from an integer, far more than the rounding of these products)
        const int line = (int)(((float)idx + 0.5f) * p.inv_pitch);
        const int d = idx - line * p.pitch_dw;
        const int r = (int)(((float)line + 0.5f) * p.inv_c);
        const int c = line - r * C;
        const int iy = iy0 + r, ix = 4 * (d - 1);
        const bool row_ok = iy >= 0 && iy < g.H;
        const unsigned off0 = (unsigned)c * plane + (unsigned)min(max(iy, 0), g.H - 1) * (unsigned)g.W;
        // every load from a clamped (always valid) address, so that all are in flight together; what lies outside
        // the image is zeroed afterwards
        v4i raw;
        unsigned keep = 0;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int ixe = ix + e;
            const unsigned off = off0 + (unsigned)min(max(ixe, 0), g.W - 1);
            if constexpr (IN_F32) raw[e] = __float_as_int(static_cast<const float*>(x_)[img_in + off]);
            else raw[e] = static_cast<const int8_t*>(x_)[img_in + off];
            if (row_ok && ixe >= 0 && ixe < g.W) keep |= 0xffu << (8 * e);
        }
        unsigned pk;
        if constexpr (IN_F32) pk = (unsigned)quantize4(raw, qs, half);
        else pk = (unsigned)(raw[0] & 0xff) | (unsigned)(raw[1] & 0xff) << 8 | (unsigned)(raw[2] & 0xff) << 16 | (unsigned)raw[3] << 24;
        stem_lds[idx] = pk & keep;
    }
}

// EPI: 0 = fp32 Float4 result, 1 = int8 Byte8, 2 = int8 Byte8 of a layer that clamps at zero with positive output
// scales (the clamp applied to the rounded values, see epi8_quant_i8p8)
template <int MT, int EPI, bool IN_F32, int CT>
__global__ void __launch_bounds__(256) conv_stem3x3_lds_kernel(const void* __restrict__ x_, const int8_t* __restrict__ wpk,
                                                               void* __restrict__ out, ConvGeom g, Epilogue ep,
                                                               const float* __restrict__ in_scale, int in_round, StemPlan p) {
    extern __shared__ unsigned stem_lds[];
    const int tid = threadIdx.x, lane = tid & 63, n = lane & 15, kg = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int img = (int)div_by(blockIdx.x, p.by_strips), strip = (int)blockIdx.x - img * p.strips;
    const int S = g.sh, C = CT ? CT : g.C;
    constexpr int NC = CT ? CT : STEM_LDS_MAX_C;

    // ---- the strip's input rows -> int8 lines in LDS
    const int oy0 = strip * p.R, iy0 = oy0 * S - g.ph;
    const size_t img_in = (size_t)img * g.C * (unsigned)(g.H * g.W);
    const float qs = IN_F32 ? in_scale[0] : 0.f;
    const float half = in_round == OTTER_HIP_ROUND_SSE ? 0.5f : 0.49999997f;
    if (p.fill == STEM_LINES) stem_fill_lines<IN_F32, CT>(stem_lds, x_, g, p, img_in, iy0, qs, half);
    else if (p.fill == STEM_UNITS) stem_fill_units<IN_F32, CT>(stem_lds, x_, g, p, img_in, iy0, qs, half);
    else stem_fill_values<IN_F32>(stem_lds, x_, g, p, C, img_in, iy0, qs, half);

    // ---- this lane's weights and the constants of its channels 16*m + 4*kg + i (requested once the strip's loads have
    // been consumed, so that their registers are not held across them; they arrive while the workgroup meets at the barrier)
    v4i a[MT];
    float si[MT][4], bi[MT][4], so[MT][4];
#pragma unroll
    for (int m = 0; m < MT; ++m) {
        a[m] = reinterpret_cast<const v4i*>(wpk)[m * 64 + lane];
        const int ch = 16 * m + 4 * kg;
        const v4i s4 = *reinterpret_cast<const v4i*>(ep.scale_in + ch), b4 = *reinterpret_cast<const v4i*>(ep.bias + ch);
        v4i o4 = {0, 0, 0, 0};
        if constexpr (EPI != 0) o4 = *reinterpret_cast<const v4i*>(ep.scale_out + ch);
#pragma unroll
        for (int i = 0; i < 4; ++i) si[m][i] = __int_as_float(s4[i]), bi[m][i] = __int_as_float(b4[i]), so[m][i] = __int_as_float(o4[i]);
    }

    unsigned qh[MT][2];
    if constexpr (EPI == 2) {
#pragma unroll
        for (int m = 0; m < MT; ++m) {
            qh[m][0] = epi8_clamp_pair(ep, so[m][0], so[m][1]);
            qh[m][1] = epi8_clamp_pair(ep, so[m][2], so[m][3]);
        }
    }
    __syncthreads();

    // ---- the output rows of the strip: item = (row, group of 16 pixels)
    const int rows = min(p.R, g.OH - oy0);
    const int items = rows * p.cgs;
    const int lc0 = S * n - g.pw + 4;  // this lane's window starts at this byte of a line (plus 16*S per pixel group)
    const unsigned shift = 8u * (unsigned)(lc0 & 3);
    const int OHW = g.OH * g.OW;
    for (int it = wave; it < items; it += 4) {
        const int orow = (int)div_by((unsigned)it, p.by_cgs), cg = it - orow * p.cgs;
        const int r = min(S * orow + kg, p.RIN - 1);  // (kernel row 3 does not exist: its bytes meet zero weights)
        const unsigned* line = stem_lds + r * C * p.pitch_dw + (lc0 >> 2) + 4 * S * cg;
        v4i b = {0, 0, 0, 0};
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            const unsigned* l = line + (CT ? c : min(c, C - 1)) * p.pitch_dw;  // (absent channels meet zero weights too)
            b[c] = (int)__builtin_amdgcn_alignbit(l[1], l[0], shift);
        }
        const int ox = 16 * cg + n;
        const bool col_ok = ox < g.OW;
        const int pix = (oy0 + orow) * g.OW + ox;
#pragma unroll
        for (int m = 0; m < MT; ++m) {
            const v4i acc = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[m], b, v4i{0, 0, 0, 0}, 0, 0, 0);
            const int ch0 = 16 * m + 4 * kg;  // D rows 4*kg .. 4*kg+3 of column n
            if (!col_ok || ch0 >= g.K) continue;
            if constexpr (EPI == 2) {
                int q[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const float t = __fmul_rn(__fmaf_rn((float)acc[i], si[m][i], bi[m][i]), so[m][i]);
                    q[i] = (int)cvt_u32_floor0(__fadd_rn(t, ep.round_half));  // (to unsigned: the clamp at zero comes with it)
                }
                typedef unsigned short ohip_v2us __attribute__((ext_vector_type(2)));
                ohip_v2us lo = __builtin_bit_cast(ohip_v2us, __builtin_amdgcn_cvt_pk_u16((unsigned)q[0], (unsigned)q[1]));
                ohip_v2us hi = __builtin_bit_cast(ohip_v2us, __builtin_amdgcn_cvt_pk_u16((unsigned)q[2], (unsigned)q[3]));
                lo = __builtin_elementwise_min(lo, __builtin_bit_cast(ohip_v2us, qh[m][0]));
                hi = __builtin_elementwise_min(hi, __builtin_bit_cast(ohip_v2us, qh[m][1]));
                unsigned* o = reinterpret_cast<unsigned*>(out) + (((size_t)img * (g.K / 8) + ch0 / 8) * OHW + pix) * 2 + (ch0 / 4 & 1);
                *o = __builtin_amdgcn_perm(__builtin_bit_cast(unsigned, hi), __builtin_bit_cast(unsigned, lo), 0x06040200u);
            } else {
                float v[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    float t = __fmaf_rn((float)acc[i], si[m][i], bi[m][i]);
                    t = fminf(fmaxf(t, ep.act_lo), ep.act_hi);
                    if (ep.lrelu) t = fmaxf(t, __fmul_rn(t, ep.act_p0));
                    v[i] = t;
                }
                if constexpr (EPI == 0) {  // Float4: [N][K/4][OH*OW][4]
                    float4* o = reinterpret_cast<float4*>(out) + ((size_t)img * (g.K / 4) + ch0 / 4) * OHW + pix;
                    *o = make_float4(v[0], v[1], v[2], v[3]);
                } else {  // Byte8: [N][K/8][OH*OW][8]; these 4 channels are one half of an element
                    unsigned pk = 0;
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const float t = __fmul_rn(v[i], so[m][i]);
                        const int rr = (int)__fadd_rn(t, __builtin_copysignf(ep.round_half, t));
                        pk |= (unsigned)(min(max(rr, -127), 127) & 0xff) << (8 * i);
                    }
                    unsigned* o = reinterpret_cast<unsigned*>(out) + (((size_t)img * (g.K / 8) + ch0 / 8) * OHW + pix) * 2 + (ch0 / 4 & 1);
                    *o = pk;
                }
            }
        }
    }
}

// ---------------------------------------------------------------------------------------------------------------------
// A stride-2 layer and the 3x3 stride-2 max pooling that alone reads its fp32 result
// ---------------------------------------------------------------------------------------------------------------------

// What the two cost as launches is the blob between them: the layer's result is four times the pooled one and fp32 (24 channels, 416x416
// -> 208x208 -> 104x104, 16 images: 66 MB written and read, 19.8 + 20.0 us, 25 + 19.5 in the detection model; its quantization for the layers behind
// 4.2 us more). As one launch 19.4 us with both results, 17.1 with the int8 one alone, 18.0 in the model; for one image 6.0 (14.5 as three). The bytes it
// cannot do without take 8, the rest is the chain of a strip: rows in, barrier, windows. Dequantization, clamp and LeakyReLU are monotone where
// scale_in >= 0, rounding included: the largest of nine results is the result of the largest sum, and a pooled value costs nine integer comparisons
// and one epilogue.
//
// A workgroup owns R pooled rows. A lane's pixel is a pooled one, and its three columns of the layer come from the same three LDS dwords
// of a line (windows 2 pixels apart); a column or row outside the layer's result repeats the one beside it, and the window then also
// counts pad_value. What is computed twice, the rows and columns that neighbouring windows share, is matrix work: 9 instructions of 16
// cycles for 16 pixels x 16 channels.
template <int MT, bool IN_F32, int CT>
__global__ void __launch_bounds__(256) conv_stem_pool_kernel(const void* __restrict__ x_, const int8_t* __restrict__ wpk, float* __restrict__ out,
                                                             int8_t* __restrict__ out_q, ConvGeom g, Epilogue ep, const float* __restrict__ in_scale,
                                                             int in_round, StemPlan p, int POH, int POW, float pad_value) {
    extern __shared__ unsigned stem_lds[];
    const int tid = threadIdx.x, lane = tid & 63, n = lane & 15, kg = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int img = (int)div_by(blockIdx.x, p.by_strips), strip = (int)blockIdx.x - img * p.strips;
    const int C = CT ? CT : g.C;
    constexpr int NC = CT ? CT : STEM_LDS_MAX_C;
    const int py0 = strip * p.R, r0 = 2 * py0 - 1;  // first pooled row; first row of the layer
    {
        const size_t img_in = (size_t)img * g.C * (unsigned)(g.H * g.W);
        const float qs = IN_F32 ? in_scale[0] : 0.f;
        const float half = in_round == OTTER_HIP_ROUND_SSE ? 0.5f : 0.49999997f;
        if (p.fill == STEM_LINES) stem_fill_lines<IN_F32, CT>(stem_lds, x_, g, p, img_in, 2 * r0 - g.ph, qs, half);
        else stem_fill_values<IN_F32>(stem_lds, x_, g, p, C, img_in, 2 * r0 - g.ph, qs, half);
    }
    v4i a[MT];
    float si[MT][4], bi[MT][4];
#pragma unroll
    for (int m = 0; m < MT; ++m) {
        a[m] = reinterpret_cast<const v4i*>(wpk)[m * 64 + lane];
        const int ch = 16 * m + 4 * kg;
        const v4i s4 = *reinterpret_cast<const v4i*>(ep.scale_in + ch), b4 = *reinterpret_cast<const v4i*>(ep.bias + ch);
#pragma unroll
        for (int i = 0; i < 4; ++i) si[m][i] = __int_as_float(s4[i]), bi[m][i] = __int_as_float(b4[i]);
    }
    __syncthreads();

    // a wave walks down a group of 16 columns, or a part of it where the groups are fewer than the waves: the layer's row that two windows
    // share is computed once
    const int rows = min(p.R, POH - py0);
    const int parts = p.cgs >= 4 ? 1 : p.cgs >= 2 ? 2 : 4, per = (rows + parts - 1) / parts;
    // the window of the layer's column 2 x - 1 + j starts at byte 4 x + 2 + 2 j - pw of a line
    const unsigned shift[3] = {8u * ((2u - g.pw) & 3u), 8u * ((4u - g.pw) & 3u), 8u * ((6u - g.pw) & 3u)};
    const bool first_aligned = g.pw == 0;  // the middle window: at dword x + 1, else at the end of dword x
    const int POHW = POH * POW;
    for (int it = wave; it < p.cgs * parts; it += 4) {
        const int cg = it >> (parts >> 1), part = it - cg * parts, x = 16 * cg + n;  // (parts: 1, 2, 4)
        const bool left = x == 0, right = 2 * x + 1 >= g.OW;
        // the largest sums of the three columns of the layer's row r0 + row
        auto across = [&](int row, v4i (&most)[MT]) {
            const int r = min(2 * row + kg, p.RIN - 1);  // (kernel row 3 does not exist: its bytes meet zero weights)
            const unsigned* line = stem_lds + r * C * p.pitch_dw + x;
            v4i b[3] = {v4i{0, 0, 0, 0}, v4i{0, 0, 0, 0}, v4i{0, 0, 0, 0}};
#pragma unroll
            for (int c = 0; c < NC; ++c) {
                const unsigned* l = line + (CT ? c : min(c, C - 1)) * p.pitch_dw;  // (absent channels meet zero weights too)
                const unsigned d0 = l[0], d1 = l[1], d2 = l[2];
                const int mid = (int)(first_aligned ? d1 : __builtin_amdgcn_alignbit(d1, d0, shift[1]));
                b[1][c] = mid;
                b[0][c] = left ? mid : (int)__builtin_amdgcn_alignbit(d1, d0, shift[0]);
                b[2][c] = right ? mid : (int)__builtin_amdgcn_alignbit(d2, d1, shift[2]);
            }
#pragma unroll
            for (int m = 0; m < MT; ++m) {
                v4i acc[3];
#pragma unroll
                for (int j = 0; j < 3; ++j) acc[j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[m], b[j], v4i{0, 0, 0, 0}, 0, 0, 0);
#pragma unroll
                for (int e = 0; e < 4; ++e) most[m][e] = max(max(acc[0][e], acc[1][e]), acc[2][e]);
            }
        };
        v4i above[MT];
        const int first = part * per, last = min(first + per, rows);
        for (int orow = first; orow < last; ++orow) {
            const int py = py0 + orow;
            const bool top = py == 0, bottom = 2 * py + 1 >= g.OH;  // (uniform)
            v4i middle[MT], below[MT], best[MT];
            across(2 * orow + 1, middle);
            across(bottom ? 2 * orow + 1 : 2 * orow + 2, below);
            if (orow == first) across(top ? 2 * orow + 1 : 2 * orow, above);  // (uniform)
#pragma unroll
            for (int m = 0; m < MT; ++m)
#pragma unroll
                for (int e = 0; e < 4; ++e) best[m][e] = max(max(above[m][e], middle[m][e]), below[m][e]), above[m][e] = below[m][e];
            const float pad = left || right || top || bottom ? pad_value : -__builtin_inff();
            const unsigned pix = (unsigned)(py * POW + x);
#pragma unroll
            for (int m = 0; m < MT; ++m) {
                const int ch0 = 16 * m + 4 * kg;  // D rows 4*kg .. 4*kg+3 of column n
                v4i v;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    float t = __fmaf_rn((float)best[m][e], si[m][e], bi[m][e]);
                    t = lrelu_or_not(ep, fminf(fmaxf(t, ep.act_lo), ep.act_hi));
                    v[e] = __float_as_int(fmaxf(t, pad));
                }
                if (x >= POW || ch0 >= g.K) continue;
                const size_t at = (((size_t)img * (g.K / 8) + ch0 / 8) * (size_t)POHW + pix) * 8 + (ch0 & 4);
                if (out != nullptr) *reinterpret_cast<v4i*>(out + at) = v;
                if (out_q != nullptr) *reinterpret_cast<int*>(out_q + at) = quantize4(v, ep.twin_scale, ep.twin_half);
            }
        }
    }
}

// whether the rows can be loaded in units (offsets inside an image are of 32 bits)
static bool stem_units(const void* x, bool in_f32, const ConvGeom& g) {
    if ((size_t)g.C * g.H * g.W * (in_f32 ? 4 : 1) >= ((size_t)1 << 31)) return false;
    return in_f32 ? g.W >= 4 && ((uintptr_t)x & 3) == 0 : g.W % 4 == 0 && ((uintptr_t)x & 3) == 0;
}
// How a strip of the layer alone is loaded. Lines where they keep five lanes of eight busy (six where the channels are not the three that the line's
// figures are compiled for) and every wave has three of them: 3 -> 32 stride 2 @224x224 on one image 5.4 us (units 5.9), 64 images 16.6 (18.5),
// 3 -> 24 @416x416, 16 images, 19.7 (20.8), 3 -> 40 @334x334, 14 images, 14.8 (16.0); with more lanes idle or fewer lines they lose: 2 -> 48
// @199x244, two images, 7.3 (6.5). Rows below 64 pixels value by value, the least code in front of the loads: 3 -> 16 stride 2 @32x32, 64 images, 3.3
// (units 3.4, lines 3.9), 1 -> 8 @28x28, 64 images, 3.4 (3.6, 4.2). Between them units: 3 -> 32 @96x96, one image, 4.1 (lines 4.4). Over drawn
// layers 0.97 of the time with units of whole rows and values for the others, with lines alone 1.08.
static int stem_fill_rule(const void* x, bool in_f32, const ConvGeom& g, const StemPlan& p) {
    if (!stem_units(x, in_f32, g)) return STEM_VALUES;
    const int busy = g.C == 3 ? 5 : 6;  // lanes of eight
    if (8 * p.pitch_dw >= busy * 64 * ((p.pitch_dw + 63) / 64) && p.RIN * g.C >= 12) return STEM_LINES;
    return g.W < 64 ? STEM_VALUES : STEM_UNITS;
}
// rows per workgroup and the LDS image of a strip; false where even one output row's input does not fit 64 KB
static bool stem_lds_plan(const ConvGeom& g, StemPlan* p, size_t* lds_bytes) {
    const int S = g.sh, cgs = (g.OW + 15) / 16;
    const int pitch_dw = std::max(((S * (16 * cgs - 1) - g.pw + 4) >> 2) + 2, (g.W + 3) / 4 + 1);
    for (int R = std::min(STEM_LDS_ROWS, g.OH); R >= 1; --R) {
        const int RIN = S * (R - 1) + 3;
        const size_t bytes = (size_t)RIN * g.C * pitch_dw * 4;
        if (bytes > 64 * 1024) continue;
        p->R = R, p->strips = (g.OH + R - 1) / R, p->cgs = cgs, p->RIN = RIN, p->pitch_dw = pitch_dw, p->fill = STEM_VALUES;
        p->by_strips = fast_div((unsigned)p->strips), p->by_cgs = fast_div((unsigned)cgs);
        p->inv_pitch = 1.0f / (float)pitch_dw, p->inv_c = 1.0f / (float)g.C;
        *lds_bytes = bytes;
        return true;
    }
    return false;
}

// shapes and epilogues this kernel takes; everything else goes through the channel-padded copy and the generic kernel
bool conv_stem_applicable(const ConvGeom& g, const Epilogue& ep, int in_layout) {
    if (g.groups != 1 || g.kh != 3 || g.kw != 3 || g.dh != 1 || g.dw != 1 || g.sh != g.sw || g.sh < 1 || g.sh > 2) return false;
    if (g.ph > 1 || g.pw > 1 || g.C > STEM_MAX_C || g.K > 16 * STEM_MAX_TILES) return false;
    if (in_layout != OTTER_HIP_F32 && in_layout != OTTER_HIP_I8) return false;
    if (g.C <= STEM_LDS_MAX_C) {  // (the weights are packed for the kernel that stages the input in LDS)
        StemPlan p;
        size_t lds = 0;
        if ((long)g.C * g.H * g.W >= (1l << 31) || !stem_lds_plan(g, &p, &lds)) return false;
    }
    const bool clamp_act = ep.act == 0 || ep.act == 1 || ep.act == 3 || (ep.act == 2 && ep.lrelu);
    if (!clamp_act) return false;
    if (ep.out_kind == OTTER_HIP_OUT_F32) return ep.out_layout == OTTER_HIP_F32_P4 && g.K % 4 == 0;
    if (ep.out_kind == OTTER_HIP_OUT_I8) return ep.out_layout == OTTER_HIP_I8_P8 && g.K % 8 == 0;
    return false;
}

// the strip of R pooled rows; false where it does not fit 64 KB
static bool stem_pool_plan(const ConvGeom& g, int R, int POH, int POW, StemPlan* p, size_t* lds_bytes) {
    p->R = R, p->strips = (POH + R - 1) / R, p->cgs = (POW + 15) / 16, p->RIN = 4 * R + 3, p->fill = STEM_VALUES;
    p->pitch_dw = std::max(16 * p->cgs + 2, (g.W + 3) / 4 + 1);
    p->by_strips = fast_div((unsigned)p->strips), p->by_cgs = fast_div((unsigned)p->cgs);
    p->inv_pitch = 1.0f / (float)p->pitch_dw, p->inv_c = 1.0f / (float)g.C;
    *lds_bytes = (size_t)p->RIN * g.C * p->pitch_dw * 4;
    return *lds_bytes <= 64 * 1024;
}
static int stem_pooled(int size) { return (size - 1) / 2 + 1; }  // (3x3, stride 2, padding 1)

// (scale_in >= 0 and finite constants are the caller's to check: they are on the device)
bool conv_stem_pool_applicable(const ConvGeom& g, const Epilogue& ep, int in_layout) {
    if (!conv_stem_applicable(g, ep, in_layout) || g.C > STEM_LDS_MAX_C || g.sh != 2 || g.K % 8 || ep.out_kind != OTTER_HIP_OUT_F32) return false;
    if (g.OH < 1 || g.OW < 1 || (size_t)g.N * g.K * g.OH * g.OW >= ((size_t)1 << 31)) return false;
    StemPlan p;
    size_t lds;
    return stem_pool_plan(g, 1, stem_pooled(g.OH), stem_pooled(g.OW), &p, &lds);
}

template <int MT>
static hipError_t launch_stem_pool(const void* x, bool in_f32, const int8_t* wpk, float* out, int8_t* out_q, const ConvGeom& g, const Epilogue& ep,
                                   const float* in_scale, int in_round, float pad_value, const StemPlan& p, size_t lds, hipStream_t stream) {
    const int POH = stem_pooled(g.OH), POW = stem_pooled(g.OW);
    const dim3 grid((unsigned)((long)g.N * p.strips)), block(256);
#define OHIP_STEM_P(FI_, CT_) \
    launch((conv_stem_pool_kernel<MT, FI_, CT_>), grid, block, lds, stream, x, wpk, out, out_q, g, ep, in_scale, in_round, p, POH, POW, pad_value)
    if (in_f32 && g.C == 3) OHIP_STEM_P(true, 3);
    else if (in_f32) OHIP_STEM_P(true, 0);
    else if (g.C == 3) OHIP_STEM_P(false, 3);
    else OHIP_STEM_P(false, 0);
#undef OHIP_STEM_P
    return hipGetLastError();
}

// out (Float8), out_q (Byte8, quantized with ep.twin_scale): either may be null. force: pooled rows of a workgroup, 0 = automatic
hipError_t run_conv_stem_pool(const void* x, bool in_f32, const int8_t* wpk, float* out, int8_t* out_q, const ConvGeom& g, const Epilogue& ep,
                              const float* in_scale, int in_round, float pad_value, int force, hipStream_t stream) {
    if (g.N == 0) return hipSuccess;
    StemPlan p;
    size_t lds = 0;
    const int POH = stem_pooled(g.OH), POW = stem_pooled(g.OW);
    int R = force ? force : STEM_POOL_ROWS;
    // fewer rows where the workgroups would not fill the compute units: a row more is read for every strip
    while (!force && R > 1 && (long)g.N * ((POH + R - 1) / R) < 512) R /= 2;
    while (R > 1 && !stem_pool_plan(g, R, POH, POW, &p, &lds)) R /= 2;
    if (!stem_pool_plan(g, R, POH, POW, &p, &lds) || (long)g.N * p.strips >= (1l << 31)) return hipErrorInvalidValue;
    p.fill = stem_units(x, in_f32, g) ? STEM_LINES : STEM_VALUES;
    switch ((g.K + 15) / 16) {
    case 1: return launch_stem_pool<1>(x, in_f32, wpk, out, out_q, g, ep, in_scale, in_round, pad_value, p, lds, stream);
    case 2: return launch_stem_pool<2>(x, in_f32, wpk, out, out_q, g, ep, in_scale, in_round, pad_value, p, lds, stream);
    case 3: return launch_stem_pool<3>(x, in_f32, wpk, out, out_q, g, ep, in_scale, in_round, pad_value, p, lds, stream);
    case 4: return launch_stem_pool<4>(x, in_f32, wpk, out, out_q, g, ep, in_scale, in_round, pad_value, p, lds, stream);
    default: return hipErrorInvalidValue;
    }
}

template <int MT>
static hipError_t launch_stem_lds(const void* x, bool in_f32, const int8_t* wpk, void* out, const ConvGeom& g, const Epilogue& ep,
                                  const float* in_scale, int in_round, hipStream_t stream) {
    StemPlan p;
    size_t lds = 0;
    if (!stem_lds_plan(g, &p, &lds)) return hipErrorInvalidValue;
    const long wgs = (long)g.N * p.strips;
    if (wgs >= (1l << 31)) return hipErrorInvalidValue;
    p.fill = stem_fill_rule(x, in_f32, g, p);
    const int epi = ep.out_kind == OTTER_HIP_OUT_F32 ? 0 : pick_epilogue(ep, g.K) == EPI_I8_P8_NONNEG ? 2 : 1;
    const dim3 grid((unsigned)wgs), block(256);
#define OHIP_STEM_L(EPI_, FI_)                                                                                          \
    do {                                                                                                                \
        if (g.C == 3)                                                                                                   \
            launch((conv_stem3x3_lds_kernel<MT, EPI_, FI_, 3>), grid, block, lds, stream, x, wpk, out, g, ep, \
                               in_scale, in_round, p);                                                                  \
        else                                                                                                            \
            launch((conv_stem3x3_lds_kernel<MT, EPI_, FI_, 0>), grid, block, lds, stream, x, wpk, out, g, ep, \
                               in_scale, in_round, p);                                                                  \
    } while (0)
    if (in_f32) {
        if (epi == 0) OHIP_STEM_L(0, true);
        else if (epi == 1) OHIP_STEM_L(1, true);
        else OHIP_STEM_L(2, true);
    } else {
        if (epi == 0) OHIP_STEM_L(0, false);
        else if (epi == 1) OHIP_STEM_L(1, false);
        else OHIP_STEM_L(2, false);
    }
#undef OHIP_STEM_L
    return hipGetLastError();
}

hipError_t run_conv_stem(const void* x, bool in_f32, const int8_t* wpk, void* out, const ConvGeom& g, const Epilogue& ep,
                         const float* in_scale, int in_round, hipStream_t stream) {
    if (g.N == 0 || g.OH * g.OW == 0) return hipSuccess;
    const int mt = (g.K + 15) / 16;
    if (g.C <= STEM_LDS_MAX_C) {
        switch (mt) {
        case 1: return launch_stem_lds<1>(x, in_f32, wpk, out, g, ep, in_scale, in_round, stream);
        case 2: return launch_stem_lds<2>(x, in_f32, wpk, out, g, ep, in_scale, in_round, stream);
        case 3: return launch_stem_lds<3>(x, in_f32, wpk, out, g, ep, in_scale, in_round, stream);
        case 4: return launch_stem_lds<4>(x, in_f32, wpk, out, g, ep, in_scale, in_round, stream);
        default: return hipErrorInvalidValue;
        }
    }
    const int col_groups = (g.OW + 15) / 16;
    const int strips = (g.OH + STEM_ROWS_PER_WAVE - 1) / STEM_ROWS_PER_WAVE;
    const long total = (long)g.N * strips * col_groups;
    if (total >= (1l << 31)) return hipErrorInvalidValue;
    const dim3 grid((unsigned)((total + 3) / 4)), block(256);
    const bool f32_out = ep.out_kind == OTTER_HIP_OUT_F32;
#define OHIP_STEM(MT_, FO_, FI_)                                                                                   \
    launch((conv_stem3x3_kernel<MT_, FO_, FI_>), grid, block, 0, stream, x, wpk, out, g, ep, in_scale,    \
                       in_round, col_groups, strips, (int)total)
#define OHIP_STEM_IO(MT_)                                  \
    do {                                                   \
        if (f32_out && in_f32) OHIP_STEM(MT_, true, true); \
        else if (f32_out) OHIP_STEM(MT_, true, false);     \
        else if (in_f32) OHIP_STEM(MT_, false, true);      \
        else OHIP_STEM(MT_, false, false);                 \
    } while (0)
    switch (mt) {
    case 1: OHIP_STEM_IO(1); break;
    case 2: OHIP_STEM_IO(2); break;
    case 3: OHIP_STEM_IO(3); break;
    case 4: OHIP_STEM_IO(4); break;
    default: return hipErrorInvalidValue;
    }
#undef OHIP_STEM_IO
#undef OHIP_STEM
    return hipGetLastError();
}

}  // namespace ohip
