// Dense and grouped k x k int8 convolution (k up to 5, any stride and dilation) on input rows staged in LDS: the kernel for
// large launches that conv3x3_halo_kernel does not take or pads heavily -- 5x5 windows, groups, few input or output channels --
// and for k x k layers on an fp32 blob, which is quantized once per value on its way into LDS.
//
// What bounds the implicit-GEMM kernel on these layers is vector issue: addresses, bounds checks and 8-byte loads are paid per
// tap (256 -> 256 3x3 in 8 groups @28x28 b64: 10.1 M vector instructions, 0.36 M of them memory reads, beside 0.25 M matrix
// ones; issuing them takes 80 % of the 22.6 us). Here a tile pays them once per staged row and a step reads LDS: 3.3 M vector
// instructions, 0.09 M memory reads, 51 % of the time in vector issue, 22 % in the LDS pipe, 16 % in the matrix cores.
//
// A workgroup of four waves owns PT = 64 FN consecutive output pixels and FM 16-row tiles of output channels (all of them, one
// block after the other, where the input channels fit one stage). Wide images are cut into column strips first, and a strip
// then counts as an image of its own: pixels are numbered (image, strip, row, column in strip), so that a tile may run over
// the end of a small image into the next and no lane is idle but in the last tile. The rows of such a sequence of images lie
// in LDS one after the other with their padding rows and columns as zeros: virtual row v of the tile is row v % VH - pad of
// image v / VH, VH the padded height. A reduction step is eight (tap, channel octet) pairs of the stage; a lane's two pairs are
// byte offsets added to its pixel's address. The channel octets come in stages of at most 8; octet planes are 64 bytes off a
// multiple of 128, which puts the pairs of neighbouring lane quarters into different halves of the banks.
//
// Measured, us per launch before / after: 256 -> 256 3x3 in 8 groups @28x28 b64 22.6 / 13.2; 384 -> 64 5x5 in 4 groups
// @67x67 b9 73 / 20; 272 -> 24 3x3 @157x157 b16 129 / 60; 24 -> 32 5x5 @162x162 b13 51.5 / 16.8; 16 -> 16 3x3 dilated
// @204x204 b55 107 / 56; 8 -> 344 5x5 @113x113 b24 96 / 62; from fp32 128 -> 64 5x5 in 8 groups @75x89 b32 48.6 / 28.9.
// The octets of a stage are requested together and the weights of a step ahead without a condition: with a branch on the parity of
// the width at each load the compiler waited for every octet before the next. 256 -> 256 in 8 groups @28x28 b64 15.0 -> 14.2 per call.
// What is left above the floor is the chain of a tile (rows in, barrier, steps, stores), which the workgroups of a compute unit hide
// from each other: registers are held to what six (two row tiles, two pixel tiles), five (two, four), four and three of them leave, and the set-up
// and the end of a tile to what they need. Pixels are walked, not divided out, the stage's dividers come with the arguments, the epilogue's
// constants come through LDS and for four channels at a time (for eight from memory: 28 registers, and the wave waits for them at the end of its chain). us per
// launch in a graph, over 26 layers 0.92 of the time: 256 -> 256 in 8 groups @28x28 b64 15.4 -> 13.6; 384 -> 352 in 4 groups
// @147x147 b4 65.7 -> 53.7; 16 -> 48 @167x167 b47 60.3 -> 51.5; 40 -> 168 from fp32 @53x53 b14 14.5 -> 13.0.
#include "common.hpp"
#include "conv_igemm.hpp"
#include "rows_stage.hpp"

#include <algorithm>
#include <cmath>

namespace ohip {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef int v2i __attribute__((ext_vector_type(2)));

namespace {

constexpr int ROWS_OCTETS = 8;             // channel octets of a stage
constexpr int ROWS_LDS = 64 * 1024;        // what a workgroup may use: two to a compute unit

struct RowsArgs {
    ConvGeom g;                            // one group's channels; g.Cs / g.Ks the tensors'
    FastDiv img, tw, vh, vw, ntx, kw;      // dividers: pixels of a strip, its width, VH, VW2, strips per image, kernel width
    FastDiv count, count1;                 // octets of a stage: the first `more` ones have one more
    int base, more;
    int strips, strip_w, VH, VW2;          // column strips per image, output columns of one, padded height, pixel pairs of a row
    int rows_max, pitch, plane;            // LDS rows of an octet plane, bytes of a row and of a plane
    int stages, blocks_per_wg;             // stages of the channels; row blocks that a workgroup walks
    int m_tiles16, n_tiles;
    unsigned total_pix;                    // numbered as above, ragged strips included
    unsigned in_bytes, w_bytes;
    const float* in_scale;
    float in_half;
    int warm_steps;                        // steps of a row block whose weights are requested ahead
    int consts;                            // LDS bytes in front of the epilogue constants
};

// octets [first, first + count) of stage c: the C/8 octets dealt to the stages as evenly as whole octets allow
inline void rows_stage(int C8, int stages, int c, int* first, int* count) {
    const int base = C8 / stages, more = C8 % stages;
    *first = c * base + (c < more ? c : more);
    *count = base + (c < more ? 1 : 0);
}

}  // namespace

static int rows_stages(int C) { return (C / 8 + ROWS_OCTETS - 1) / ROWS_OCTETS; }
static int rows_steps(int C, int taps) {
    int steps = 0;
    for (int c = 0, n = rows_stages(C); c < n; ++c) {
        int first, count;
        rows_stage(C / 8, n, c, &first, &count);
        steps += (taps * count + 7) / 8;
    }
    return steps;
}

template <int FM, int FN, int EPI, bool INF>
__global__ void __launch_bounds__(256, EPI == EPI_GENERIC ? 2 : FM == 2 && !INF ? (FN == 4 ? 5 : 6) : FM == 4 && FN == 2 ? 4 : 2)
    conv_rows_kernel(const int8_t* __restrict__ x, const int8_t* __restrict__ wpk, void* __restrict__ out, RowsArgs ra, EpiArgs<EPI> ea) {
    constexpr int OOB = (int)0x80000000;  // beyond any buffer here (below 2 GiB)
    extern __shared__ __attribute__((aligned(16))) int8_t lds[];
    const ConvGeom& g = ra.g;
    Epilogue ep = ea.epilogue();
    const int tid = threadIdx.x, lane = tid & 63, q = lane >> 4, p = lane & 15;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    int pt = blockIdx.x;
    {  // a contiguous run of tiles per XCD: neighbours share input rows and weights
        const int per = ra.n_tiles / 8;
        if (pt < per * 8) pt = (pt % 8) * per + pt / 8;
    }
    const int grp = blockIdx.z;
    const int HW = g.H * g.W, OHW = g.OH * g.OW, C8 = g.C / 8, Cs8 = g.Cs / 8;
    const int taps = g.kh * g.kw;
    v2i* const table = reinterpret_cast<v2i*>(lds);            // [pair / 2]: the byte offsets of two pairs
    v2i* const row_tab = table + (taps * ROWS_OCTETS + 7) / 8 * 4;  // [row]: {byte offset of its column 0, first | last + 1 << 16 valid}
    int8_t* const data = reinterpret_cast<int8_t*>(row_tab + (ra.rows_max + 1) / 2 * 2);

    // ---- the tile: its first pixel (uniform), its virtual rows ---------------------------------------------------------------------
    const unsigned t0 = (unsigned)pt * (64 * FN), t1 = min(t0 + 64 * FN, ra.total_pix) - 1;
    const unsigned m0 = div_by(t0, ra.img), m1 = div_by(t1, ra.img);
    const unsigned r0 = div_by(t0 - m0 * ra.img.d, ra.tw), r1 = div_by(t1 - m1 * ra.img.d, ra.tw);
    const int v0 = (int)r0 * g.sh;
    const int rows = (int)(m1 - m0) * ra.VH + (int)r1 * g.sh + (g.kh - 1) * g.dh + 1 - v0;  // at most rows_max

    // The constants of the workgroup's channels come through LDS: a channel per thread, requested in front of everything else. (Where the
    // lanes that finish eight channels each load them, every request brings 16 bytes to each lane, and the wave waits for them at the
    // end of its chain.)
    constexpr int CN = 16 * FM;
    const int block0 = blockIdx.y * ra.blocks_per_wg, nc = ra.blocks_per_wg * CN;  // at most 512
    float* const consts = reinterpret_cast<float*>(lds + ra.consts);
    float c_si = 0.f, c_bi = 0.f, c_so = 0.f;
    if (EPI != EPI_GENERIC && tid < nc && block0 * CN + tid < g.K) {
        const int ch = grp * g.K + block0 * CN + tid;
        c_si = ep.scale_in[ch], c_bi = ep.bias[ch];
        if constexpr (EPI != EPI_F32_P4) c_so = ep.scale_out[ch];
    }

    // ---- this lane's pixels: LDS address of tap (0, 0), place in the output -----------------------------------------------------------
    int px[FN];
    unsigned out_n[FN], out_pix[FN], out_at[FN];  // (the first two for the generic epilogue only)
    bool px_ok[FN];
    constexpr unsigned OUT_E = EPI == EPI_F32_P4 ? 4u : 8u;
    if (EPI != EPI_GENERIC && ra.strips == 1 && ra.tw.d >= 16) {
        // One place by division, the next 16 pixels on from it: at most one row's end and one image's are passed on the way. (Three
        // divisions are eight 32-bit multiplications, 16 cycles each; for four places they took as long as requantizing the wave's
        // 2048 results.)
        unsigned t = t0 + wave * FN * 16 + p;
        const unsigned n = div_by(t, ra.img);
        unsigned in = t - n * ra.img.d;
        const unsigned oy = div_by(in, ra.tw);
        unsigned ox = in - oy * ra.tw.d;
        int at = ((int)(n - m0) * ra.VH + (int)oy * g.sh - v0) * ra.pitch + ((int)ox * g.sw + (g.pw & 1)) * 8;
        unsigned o = n * (unsigned)(g.Ks * OHW) + in * OUT_E;
        const int row_on = g.sh * ra.pitch - (int)ra.tw.d * g.sw * 8, image_on = (ra.VH - g.OH * g.sh) * ra.pitch;
        const unsigned o_on = (unsigned)(g.Ks * OHW) - (unsigned)OHW * OUT_E;
#pragma unroll
        for (int j = 0; j < FN; ++j) {
            px_ok[j] = t < ra.total_pix;
            px[j] = px_ok[j] ? at : 0;
            out_at[j] = o;
            t += 16, ox += 16, in += 16, at += 128 * g.sw, o += 16 * OUT_E;
            const bool row = ox >= ra.tw.d, image = in >= ra.img.d;
            ox -= row ? ra.tw.d : 0, in -= image ? ra.img.d : 0;
            at += (row ? row_on : 0) + (image ? image_on : 0), o += image ? o_on : 0;
        }
    } else {
#pragma unroll
        for (int j = 0; j < FN; ++j) {
            const unsigned t = t0 + (wave * FN + j) * 16 + p;
            const unsigned m = div_by(t, ra.img), in = t - m * ra.img.d, oy = div_by(in, ra.tw), oxs = in - oy * ra.tw.d;
            const unsigned n = div_by(m, ra.ntx), ox = (m - n * ra.ntx.d) * (unsigned)ra.strip_w + oxs;
            px_ok[j] = t < ra.total_pix && ox < (unsigned)g.OW;
            px[j] = t < ra.total_pix ? ((int)(m - m0) * ra.VH + (int)oy * g.sh - v0) * ra.pitch +
                                           ((int)oxs * g.sw + (((int)(m - n * ra.ntx.d) * ra.strip_w * g.sw - g.pw) & 1)) * 8
                                     : 0;
            out_n[j] = n, out_pix[j] = oy * (unsigned)g.OW + ox;
            out_at[j] = n * (unsigned)(g.Ks * OHW) + out_pix[j] * OUT_E;
        }
    }

    const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<int8_t*>(wpk + (size_t)grp * ra.w_bytes), 0, (int)ra.w_bytes, 0x00020000);
    const __amdgpu_buffer_rsrc_t rin = __builtin_amdgcn_make_buffer_rsrc(const_cast<int8_t*>(x), 0, (int)ra.in_bytes, 0x00020000);
    float in_scale = 0.f;
    if constexpr (INF) in_scale = ra.in_scale[0];

    // Long reductions: the weights of the workgroup's first row block, lines of 128 bytes, into the L2 of this die. A launch finds it empty, and the loop
    // below asks for one step at a time; the tiles that a die has of the block take a share each. (448 -> 168 k 5 on one 99x99 image, 175
    // steps: 60 -> 54 us; 456 -> 256 k 3 @150x150, 66 steps: 39.3 -> 37.0. At 9 steps the requests cost 1 to 4 % and bring nothing.)
    constexpr int LINES = FM * 8, WARM = 4;  // lines of a step; requests of a thread
    int warm[WARM] = {};
    if (ra.warm_steps) {
        const unsigned per = max(ra.n_tiles / 8, 1), share = (unsigned)pt % per, total = (unsigned)ra.warm_steps * LINES;
#pragma unroll
        for (int u = 0; u < WARM; ++u) {
            const unsigned l = (u * per + share) * 256 + tid;
            warm[u] = __builtin_amdgcn_raw_buffer_load_b32(rw, l < total ? (int)(l / LINES * (unsigned)ra.m_tiles16 * 1024 + l % LINES * 128) : OOB,
                                                           block0 * FM * 1024, 0);
        }
    }

    // the rows: a strip's columns start at an even one (the one before its first where that is odd), so that a pixel pair never
    // lies across the left edge of the image
    for (int r = tid; r < rows; r += 256) {
        const unsigned v = (unsigned)(r + v0), im = div_by(v, ra.vh), m = m0 + im, n = div_by(m, ra.ntx);
        const int iy = (int)(v - im * (unsigned)ra.VH) - g.ph;
        const int c0 = ((int)(m - n * ra.ntx.d) * ra.strip_w * g.sw - g.pw) & ~1;
        const bool in = iy >= 0 && iy < g.H && n < (unsigned)g.N;
        const int first = c0 < 0 ? -c0 : 0, last = g.W - c0 < 2 * ra.VW2 ? g.W - c0 : 2 * ra.VW2;
        row_tab[r] = v2i{(int)(((n * (unsigned)Cs8 + (unsigned)(grp * C8)) * (unsigned)HW + (unsigned)(iy * g.W + c0)) * 8u),
                         in && last > first ? first | last << 16 : 0};
    }

    auto put = [&](int c, float si, float bi, float so) {
        consts[c] = si, consts[nc + c] = bi;
        if constexpr (EPI != EPI_F32_P4) consts[2 * nc + c] = EPI == EPI_I8_P8_FULL ? so + so : so;
        if constexpr (EPI == EPI_I8_P8_NONNEG)
            reinterpret_cast<unsigned short*>(consts + 3 * nc)[c] = (unsigned short)min((int)__fadd_rn(__fmul_rn(ep.act_hi, so), ep.round_half), 127);
    };
    if (EPI != EPI_GENERIC && tid < nc) {
        put(tid, c_si, c_bi, c_so);
        // (a workgroup of more channels than threads walks many row blocks: what it waits for here is little of its time)
        if (const int c = tid + 256; c < nc) {
            const bool ok = block0 * CN + c < g.K;
            const int ch = grp * g.K + (ok ? block0 * CN + c : 0);
            const float si = ep.scale_in[ch], bi = ep.bias[ch];
            float so = 0.f;
            if constexpr (EPI != EPI_F32_P4) so = ep.scale_out[ch];
            put(c, ok ? si : 0.f, ok ? bi : 0.f, ok ? so : 0.f);
        }
    }

#pragma unroll
    for (int u = 0; u < WARM; ++u) asm volatile("" ::"v"(warm[u]));

    const int HW8 = HW * 8;
    const bool even = (g.W & 1) == 0;    // then no pair lies across the right edge either
    constexpr int UN = INF ? 2 : 4;      // octets in flight per thread
    constexpr int D = 2;    // weight steps in flight
    constexpr int INS = INF ? 4 : 1;     // bytes of an input value

    v4i acc[FM][FN];
    int block = block0;
    const int block_end = min(block + ra.blocks_per_wg, (g.K + 16 * FM - 1) / (16 * FM));
    auto load_a = [&](v4i (&a)[FM], int step) {
#pragma unroll
        for (int i = 0; i < FM; ++i)
            a[i] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(rw, lane * 16 + i * 1024,
                                                                                (step * ra.m_tiles16 + block * FM) * 1024, 0));
    };

    for (int c = 0, step0 = 0; c < ra.stages; ++c) {
        const int first = c * ra.base + min(c, ra.more), count = ra.base + (c < ra.more ? 1 : 0);
        const FastDiv by_count = c < ra.more ? ra.count1 : ra.count;
        const int steps = (taps * count + 7) / 8;
        v4i a[D][FM];
#pragma unroll
        for (int d = 0; d + 1 < D; ++d)
            if (d < steps) load_a(a[d], step0 + d);
        __syncthreads();  // the row table stands / everyone has read the stage before
        // the table of this stage's pairs e = (tap e / count, octet e % count); pairs past the end meet zero weights
        for (int e = tid; e < steps * 8; e += 256) {
            const unsigned tap = div_by((unsigned)e, by_count), oct = (unsigned)e - tap * (unsigned)count;
            const unsigned dy = div_by(tap, ra.kw), dx = tap - dy * (unsigned)g.kw;
            reinterpret_cast<int*>(table)[e] =
                e < taps * count ? (int)oct * ra.plane + (int)dy * g.dh * ra.pitch + (int)dx * g.dw * 8 : 0;
        }
        // the stage's rows, zeros outside the image, as pixel pairs. A thread keeps one place of the octet planes and walks the
        // octets, so that an octet costs it a load and a write and no address arithmetic
        const int pairs = rows * ra.VW2, sub_shift = rows_parts_shift(pairs), sub = 1 << sub_shift;
        const int oct0 = tid >> (8 - sub_shift);
        // (two walks, not a choice per load: behind loads on two branches the compiler waited for each octet before it requested the
        // next, four memory latencies in a row)
        auto stage_rows = [&](auto even_c) {
            constexpr bool EVEN = decltype(even_c)::value;
            for (int pos = tid & ((256 >> sub_shift) - 1); pos < pairs; pos += 256) {
                const int row = (int)div_by((unsigned)pos, ra.vw), c0 = 2 * (pos - row * ra.VW2);
                const v2i rt = row_tab[row];
                const int lo = rt[1] & 0xffff, hi = rt[1] >> 16;
                const bool in0 = c0 >= lo && c0 < hi, in1 = c0 + 1 >= lo && c0 + 1 < hi;
                const int o = rt[0] + c0 * 8 + oct0 * HW8;
                const int o0 = in0 ? o * INS : OOB, o1 = in1 ? (o + 8) * INS : OOB;
                int8_t* at = data + oct0 * ra.plane + pos * 16;  // (rows are VW2 pairs long)
                RowsWalk walk = rows_walk((unsigned)(HW8 * INS), first, count, sub);
                for (int oct = oct0; oct < count; oct += UN * sub) {
                    v4i v[UN];
                    v4i f[INF ? UN : 1][4];
#pragma unroll
                    for (int u = 0; u < UN; ++u) {
                        const bool there = u == 0 || oct + u * sub < count;
                        const int a0 = there ? o0 : OOB, a1 = there ? o1 : OOB, so = (int)walk.next();
                        if constexpr (INF) {
                            f[u][0] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(rin, a0, so, 0));
                            f[u][1] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(rin, a0 + 16, so, 0));
                            f[u][2] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(rin, a1, so, 0));
                            f[u][3] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(rin, a1 + 16, so, 0));
                        } else if constexpr (EVEN) {
                            v[u] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(rin, a0, so, 0));
                        } else {
                            const v2i l = __builtin_bit_cast(v2i, __builtin_amdgcn_raw_buffer_load_b64(rin, a0, so, 0));
                            const v2i h = __builtin_bit_cast(v2i, __builtin_amdgcn_raw_buffer_load_b64(rin, a1, so, 0));
                            v[u] = v4i{l[0], l[1], h[0], h[1]};
                        }
                    }
                    // (all of them are requested here: the compiler would move the last one behind the condition of its write)
#pragma unroll
                    for (int u = 0; u < UN; ++u) {
                        if constexpr (INF) asm volatile("" : "+v"(f[u][0]), "+v"(f[u][1]), "+v"(f[u][2]), "+v"(f[u][3]));
                        else asm volatile("" : "+v"(v[u]));
                    }
#pragma unroll
                    for (int u = 0; u < UN; ++u) {
                        if constexpr (INF)
                            v[u] = v4i{quantize4(f[u][0], in_scale, ra.in_half), quantize4(f[u][1], in_scale, ra.in_half),
                                       quantize4(f[u][2], in_scale, ra.in_half), quantize4(f[u][3], in_scale, ra.in_half)};
                        if (u == 0 || oct + u * sub < count) *reinterpret_cast<v4i*>(at + u * sub * ra.plane) = v[u];
                    }
                    at += UN * sub * ra.plane;
                }
            }
        };
        if constexpr (INF) stage_rows(std::true_type{});  // (reads values, not pixel pairs)
        else if (even) stage_rows(std::true_type{});
        else stage_rows(std::false_type{});
        __syncthreads();
        // one block of output channels per pass over the stage; several only when there is one stage
        for (;;) {
            if (c == 0) {
#pragma unroll
                for (int i = 0; i < FM; ++i)
#pragma unroll
                    for (int j = 0; j < FN; ++j) acc[i][j] = v4i{0, 0, 0, 0};
            }
            auto multiply = [&](int s, const v4i (&aa)[FM]) {
                const v2i t = table[s * 4 + q];
                v4i b[FN];
#pragma unroll
                for (int j = 0; j < FN; ++j) {
                    const v2i lo = *reinterpret_cast<const v2i*>(data + px[j] + t[0]);
                    const v2i hi = *reinterpret_cast<const v2i*>(data + px[j] + t[1]);
                    b[j] = v4i{lo[0], lo[1], hi[0], hi[1]};
                }
#pragma unroll
                for (int i = 0; i < FM; ++i)
#pragma unroll
                    for (int j = 0; j < FN; ++j) acc[i][j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(aa[i], b[j], acc[i][j], 0, 0, 0);
            };
            // No request is conditional where there are registers for it: behind one every load is waited for. The last step's weights
            // are requested once more then. (Four row tiles: 0 to 3 % slower that way.)
            if constexpr (FM == 2) {
                int s = 0;
                for (; s + D <= steps; s += D) {
#pragma unroll
                    for (int d = 0; d < D; ++d) {
                        load_a(a[(d + D - 1) % D], step0 + min(s + d + D - 1, steps - 1));
                        multiply(s + d, a[d]);
                    }
                }
#pragma unroll
                for (int d = 0; d + 1 < D; ++d)
                    if (s + d < steps) multiply(s + d, a[d]);
            } else {
                for (int s = 0; s < steps; s += D) {
#pragma unroll
                    for (int d = 0; d < D; ++d)
                        if (s + d < steps) {
                            if (s + d + D - 1 < steps) load_a(a[(d + D - 1) % D], step0 + s + d + D - 1);
                            multiply(s + d, a[d]);
                        }
                }
            }
            if (c + 1 < ra.stages) break;
            // ---- epilogue of the block -------------------------------------------------------------------------------------------
            const int mt0 = block * FM, c0 = (block - block0) * CN;
            ++block;
            if (block < block_end)
#pragma unroll
                for (int d = 0; d + 1 < D; ++d)
                    if (d < steps) load_a(a[d], d);  // (one stage: step0 == 0)
#pragma unroll
            for (int pair = 0; pair < FM / 2; ++pair) {
                const int ch0 = 16 * mt0 + 32 * pair + 8 * q;  // this lane's 8 consecutive output channels of the group
                if (ch0 >= g.K) continue;
                if constexpr (EPI == EPI_GENERIC) {
#pragma unroll
                    for (int j = 0; j < FN; ++j) {
                        const v4i lo = acc[2 * pair][j], hi = acc[2 * pair + 1][j];
                        if (px_ok[j])
                            epilogue_store8_generic(out, &ep, (int)out_n[j], ch0, (int)out_pix[j], g.K, OHW, lo[0], lo[1], lo[2], lo[3], hi[0],
                                                    hi[1], hi[2], hi[3]);
                    }
                } else {
                    const unsigned ch_at = (unsigned)(grp * g.K + ch0) * (unsigned)OHW;
                    int bytes[FN];
#pragma unroll
                    for (int h = 0; h < 2; ++h) {  // (four channels at a time: the constants of eight are 28 registers)
                        if (EPI == EPI_F32_P4 && ch0 + 4 * h >= g.K) continue;
                        const float* const at = consts + c0 + 32 * pair + 8 * q + 4 * h;
                        const v4f si4 = *reinterpret_cast<const v4f*>(at), bi4 = *reinterpret_cast<const v4f*>(at + nc);
                        v4f so4 = {};
                        if constexpr (EPI != EPI_F32_P4) so4 = *reinterpret_cast<const v4f*>(at + 2 * nc);
                        const float si[4] = {si4[0], si4[1], si4[2], si4[3]}, bi[4] = {bi4[0], bi4[1], bi4[2], bi4[3]};
                        const float so[4] = {so4[0], so4[1], so4[2], so4[3]};
                        unsigned qh[2] = {};
                        if constexpr (EPI == EPI_I8_P8_NONNEG) {
                            const v2i t = *reinterpret_cast<const v2i*>(reinterpret_cast<const unsigned short*>(consts + 3 * nc) + (at - consts));
                            qh[0] = (unsigned)t[0], qh[1] = (unsigned)t[1];
                        }
#pragma unroll
                        for (int j = 0; j < FN; ++j) {
                            const v4i v = acc[2 * pair + h][j];
                            if constexpr (EPI == EPI_F32_P4) {
                                if (px_ok[j])
                                    epi4_store_f32p4<false>((float*)out, ep, si, bi, (size_t)(out_at[j] + ch_at + (unsigned)h * (unsigned)OHW * 4), v[0], v[1], v[2], v[3]);
                            } else {
                                const int b4 = epi4_quant_i8<epi_clamp(EPI)>(ep, si, bi, so, qh, v[0], v[1], v[2], v[3]);
                                if (h == 0) {
                                    bytes[j] = b4;
                                    asm volatile("" : "+v"(bytes[j]));  // (packed here, not behind the condition of the store)
                                }
                                if (h == 1 && px_ok[j]) *reinterpret_cast<v2i*>((int8_t*)out + (out_at[j] + ch_at)) = v2i{bytes[j], b4};
                            }
                        }
                    }
                }
            }
            if (block >= block_end) break;
        }
        step0 += steps;
    }
}

// ---------------------------------------------------------------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------------------------------------------------------------

static size_t rows_packed_weight_bytes(int K, int C, int taps) { return (size_t)rows_steps(C, taps) * (igemm_padded_rows(K) / 16) * 1024; }
size_t rows_grouped_weight_bytes(int K, int C, int groups, int kh, int kw) {
    return (size_t)groups * rows_packed_weight_bytes(K / groups, C / groups, kh * kw);
}

// weight [K, C / groups, kh, kw] int8 -> per group [stage][step][16-row tile][lane][16 bytes]: bytes 0-7 / 8-15 of lane (r, q) are
// the octets of the stage's pairs 8 step + 2 q and + 1
void rows_pack_weights_grouped(const int8_t* w, int K, int C, int groups, int kh, int kw, int8_t* dst) {
    const int kg = K / groups, cg = C / groups, taps = kh * kw, mt16 = igemm_padded_rows(kg) / 16, stages = rows_stages(cg);
    size_t o = 0;
    for (int grp = 0; grp < groups; ++grp)
        for (int c = 0; c < stages; ++c) {
            int first, count;
            rows_stage(cg / 8, stages, c, &first, &count);
            for (int s = 0; s < (taps * count + 7) / 8; ++s)
                for (int mt = 0; mt < mt16; ++mt)
                    for (int lane = 0; lane < 64; ++lane) {
                        const int ch = igemm_row_channel(mt * 16 + (lane & 15));
                        for (int h = 0; h < 2; ++h) {
                            const int e = 8 * s + 2 * (lane >> 4) + h, tap = e / count, c0 = (first + e % count) * 8;
                            for (int b = 0; b < 8; ++b, ++o)
                                dst[o] = ch < kg && e < taps * count ? w[(((size_t)grp * kg + ch) * cg + c0 + b) * taps + tap] : 0;
                        }
                    }
        }
}

static bool rows_plan(const ConvGeom& g_in, int fn, RowsArgs* ra, size_t* lds) {
    ra->g = g_in;
    ra->g.Cs = g_in.C, ra->g.Ks = g_in.K;
    ra->g.C = g_in.C / g_in.groups, ra->g.K = g_in.K / g_in.groups;
    const ConvGeom& g = ra->g;
    const int pt = 64 * fn, taps = g.kh * g.kw;
    // the number of strips that makes a tile stage the fewest bytes: wide strips read padding rows, narrow ones padding columns.
    // (Rows and columns in 64 bits: with dilations in the thousands their product passes 2^32.)
    const long vh = (long)(g.OH - 1) * g.sh + (long)(g.kh - 1) * g.dh + 1, max_px = (1l << 31) - pt;
    long best = 0, best_rows = 0, best_vw2 = 0;
    for (int strips = (g.OW + 79) / 80; strips <= (g.OW + 15) / 16; ++strips) {
        const int w = (g.OW + strips - 1) / strips;
        const long vw2 = ((long)(w - 1) * g.sw + (long)(g.kw - 1) * g.dw + 1 + 2) / 2;  // (one column more in front)
        const long total = (long)g.N * g.OH * strips * w, strip_px = (long)g.OH * w;
        if (total >= max_px || strip_px >= max_px) break;
        const int tiles = (int)((unsigned)(total + pt - 1) / (unsigned)pt);
        // rows of a tile: the output rows it can touch, and the padding rows between the images it can run over
        const long out_rows = (pt - 1) / w + 2, crossings = (pt - 1) / (int)strip_px + 1;
        const long between = vh - (long)g.OH * g.sh;  // virtual rows an image has more than its output rows' share (may be negative)
        const long rows = (out_rows - 1) * g.sh + (between > 0 ? crossings * between : 0) + (long)(g.kh - 1) * g.dh + 1;
        const long cost = (long)tiles * (rows * vw2 + 64);
        if (best == 0 || cost < best) {
            best = cost, best_rows = rows, best_vw2 = vw2;
            ra->strips = strips, ra->strip_w = w, ra->total_pix = (unsigned)total, ra->n_tiles = tiles;
        }
    }
    if (best == 0 || best_rows * best_vw2 * 16 > ROWS_LDS) return false;  // (one octet plane alone)
    ra->VH = (int)vh, ra->rows_max = (int)best_rows, ra->VW2 = (int)best_vw2;
    ra->pitch = ra->VW2 * 16;
    ra->plane = (ra->rows_max * ra->pitch + 63) / 128 * 128 + 64;
    ra->stages = rows_stages(g.C);
    const int oct = (g.C / 8 + ra->stages - 1) / ra->stages;
    *lds = (size_t)(taps * ROWS_OCTETS + 7) / 8 * 32 + (size_t)(ra->rows_max + 1) / 2 * 16 + (size_t)oct * ra->plane;
    ra->m_tiles16 = igemm_padded_rows(g.K) / 16;
    ra->w_bytes = (unsigned)rows_packed_weight_bytes(g.K, g.C, taps);
    return *lds <= (size_t)ROWS_LDS;
}

bool conv_rows_plan(const ConvGeom& g, int pixels, int plan[6]) {
    RowsArgs ra;
    size_t lds;
    if (g.OH < 1 || g.OW < 1 || !rows_plan(g, pixels / 64, &ra, &lds)) return false;
    plan[0] = ra.strips, plan[1] = ra.strip_w, plan[2] = ra.rows_max, plan[3] = ra.VW2, plan[4] = ra.plane, plan[5] = (int)lds;
    return true;
}

bool conv_rows_supported(const ConvGeom& g, const Epilogue& ep, bool f32in) {
    if (g.OH < 1 || g.OW < 1 || g.C % g.groups || g.K % g.groups || g.kh * g.kw < 2 || g.kh * g.kw > 25 || g.groups > 65535) return false;
    if ((g.C / g.groups) % 8 || ep.fused()) return false;
    const int epi = pick_epilogue(ep, g.K / g.groups);
    if (epi == EPI_GENERIC && (g.groups > 1 || f32in)) return false;
    return (size_t)g.N * g.C * g.H * g.W * (f32in ? 4 : 1) < ((size_t)1 << 31) && (size_t)g.N * g.K * g.OH * g.OW < ((size_t)1 << 31);
}

// one stage: a workgroup walks row blocks over its staged pixels, as many as leave two workgroups per compute unit, and at most 512
// channels (a thread brings the constants of two), dealt evenly: every further workgroup stages the rows again. With at most 256 channels,
// the first workgroups filled: 64 -> 272 3x3 @216x216 b4 in four and one blocks 51.2 us, in one workgroup 47.4; 24 -> 344 @185x224 b7 48.3
// (62.4 with the constants from memory, on the tile chosen then).
static int rows_blocks_per_workgroup(const RowsArgs& ra, int blocks, int fm) {
    if (ra.stages > 1) return 1;
    const long tiles = (long)ra.n_tiles * ra.g.groups;
    const int want = (int)((512 + tiles - 1) / tiles), least = (blocks * fm + 31) / 32;
    const int slices = want > blocks ? blocks : want > least ? want : least;
    return (blocks + slices - 1) / slices;
}

// LDS of a workgroup: what the plan takes, and the epilogue constants behind it
static size_t rows_lds(size_t plan, int blocks_per_wg, int fm) { return (plan + 15) / 16 * 16 + (size_t)(blocks_per_wg * 16 * fm * 14); }

namespace {
// A tile, the workgroups of it that the register file holds per compute unit, and the coefficients of its duration in us (inside
// a graph of launches, warm) for int8 and fp32 input. A workgroup's chain is step * steps + stage * stages, and a compute unit
// runs as many of them one after the other as its workgroups do not fit side by side; per workgroup of the busiest compute unit
// comes what they share: steps, staged places (pixel pairs of a thread) and row blocks; per launch the megabytes in and out. With
// a stride the lanes of a pixel read lie on every other 8 bytes, and a step costs 1 + strided of what it does else. Fitted to drawn layers (k 3
// and 5, 8..512 channels, up to 2.5 million pixels), from int8 4700 of them: median error 4 to 5 %, 9 in 10 below 11 to 13 %; from fp32 2600:
// 6 %, 9 in 10 below 18 to 24 % without a stride, 8 % and 34 to 40 % with one. The tile it chooses takes 0.6 % (0.5 %) more than the
// fastest of the four on average, one in seventy 10 % or more.
struct RowsCoef {
    float start, step, stage, cu_step, cu_place, cu_block, strided, in_mb, out_mb;
};
struct RowsCost {
    int resident;
    RowsCoef at;
};
struct RowsConfig {
    int fm, fn;
    RowsCost i8, f32;
};
constexpr RowsConfig kRowsConfigs[] = {
    {2, 2, {6, {3.02f, 0.062f, 0.813f, 0.05f, 0.033f, 0.186f, 0.397f, 0.057f, 0.113f}}, {5, {2.42f, 0.099f, 1.33f, 0.041f, 0.108f, 0.123f, 0.964f, 0.067f, 0.102f}}},
    {2, 4, {5, {3.21f, 0.106f, 0.818f, 0.055f, 0.045f, 0.38f, 0.504f, 0.057f, 0.12f}}, {4, {2.75f, 0.176f, 1.19f, 0.038f, 0.141f, 0.287f, 0.708f, 0.073f, 0.111f}}},
    {4, 2, {4, {3.09f, 0.067f, 0.811f, 0.094f, 0.034f, 0.271f, 0.279f, 0.032f, 0.138f}}, {4, {2.61f, 0.114f, 1.28f, 0.079f, 0.106f, 0.124f, 0.768f, 0.058f, 0.143f}}},
    {4, 4, {3, {3.39f, 0.145f, 0.806f, 0.085f, 0.048f, 0.573f, 0.346f, 0.054f, 0.154f}}, {3, {2.85f, 0.246f, 1.39f, 0.056f, 0.145f, 0.335f, 0.637f, 0.065f, 0.154f}}},
};
constexpr int kRowsConfigCount = (int)(sizeof(kRowsConfigs) / sizeof(kRowsConfigs[0]));
}  // namespace

float conv_rows_cost(const ConvGeom& g_in, bool f32in, int out_bytes, int* config) {
    float best = __builtin_inff();
    *config = -1;
    RowsArgs ra;
    size_t lds;
    bool fits = false;
    const int steps = rows_steps(g_in.C / g_in.groups, g_in.kh * g_in.kw);
    // 2 % (four row tiles 4 %) per MB of weights beyond the first: every die fetches them all. (5 to 8 % is what layers of over 2 MB took
    // more than the fit; 504 -> 264 k 5 on one 80x92 image 57 us with two row tiles, 65 with four.)
    const float more_mb = std::max(0.f, (float)g_in.groups * rows_packed_weight_bytes(g_in.K / g_in.groups, g_in.C / g_in.groups, g_in.kh * g_in.kw) * 1e-6f - 1.f);
    const float in_mb = (float)g_in.N * g_in.C * g_in.H * g_in.W * (f32in ? 4e-6f : 1e-6f);
    const float out_mb = (float)g_in.N * g_in.K * g_in.OH * g_in.OW * 1e-6f * out_bytes;
    for (const int i : {0, 2, 1, 3}) {  // by pixels of a tile: one plan for two
        const RowsConfig& c = kRowsConfigs[i];
        if (i == 0 || i == 1) fits = rows_plan(g_in, c.fn, &ra, &lds);
        if (!fits) continue;
        const int blocks = (ra.g.K + 16 * c.fm - 1) / (16 * c.fm), bpw = rows_blocks_per_workgroup(ra, blocks, c.fm);
        const int pairs = ra.rows_max * ra.VW2, oct = (ra.g.C / 8 + ra.stages - 1) / ra.stages;
        const int shift = rows_parts_shift(pairs);
        const float places = (float)(ra.stages * oct * ((pairs + (256 >> shift) - 1) >> (8 - shift))) * (shift == 0 ? 1.f : shift == 1 ? 0.5f : shift == 2 ? 0.25f : 0.125f);
        const int slices = (blocks + bpw - 1) / bpw;
        const int wgs = (int)std::min(((long)ra.n_tiles * slices * ra.g.groups + 255) / 256, 1l << 24);
        const RowsCost& cost = f32in ? c.f32 : c.i8;
        const int side = std::min(cost.resident, (int)(160 * 1024 / rows_lds(lds, bpw, c.fm)));
        const float cu = (float)wgs, rounds = (float)((wgs + side - 1) / side);
        const RowsCoef& k = cost.at;
        const float s = (float)steps * (g_in.sw > 1 ? 1.f + k.strided : 1.f), walked = (float)blocks / (float)slices;  // (of one workgroup, on average)
        float t = k.start + rounds * (k.step * s * (float)bpw + k.stage * (float)ra.stages) +
                        cu * (walked * (k.cu_step * s + k.cu_block) + k.cu_place * places) + k.in_mb * in_mb + k.out_mb * out_mb;
        t *= 1.f + 0.01f * (float)c.fm * more_mb;
        if (t < best) best = t, *config = i;
    }
    return best;
}

hipError_t run_conv_rows(const void* x, bool f32in, const int8_t* wpk, void* out, const ConvGeom& g_in, const Epilogue& ep, int config,
                         const float* in_scale, int in_round_mode, hipStream_t stream) {
    if (!conv_rows_supported(g_in, ep, f32in) || config < 0 || config >= kRowsConfigCount) return hipErrorInvalidValue;
    const RowsConfig c = kRowsConfigs[config];
    RowsArgs ra;
    size_t lds;
    if (!rows_plan(g_in, c.fn, &ra, &lds)) return hipErrorInvalidValue;
    ra.img = fast_div((unsigned)(ra.g.OH * ra.strip_w)), ra.tw = fast_div((unsigned)ra.strip_w), ra.vh = fast_div((unsigned)ra.VH);
    ra.vw = fast_div((unsigned)ra.VW2), ra.ntx = fast_div((unsigned)ra.strips), ra.kw = fast_div((unsigned)ra.g.kw);
    ra.in_bytes = (unsigned)((size_t)ra.g.N * ra.g.Cs * ra.g.H * ra.g.W * (f32in ? 4 : 1));
    ra.base = ra.g.C / 8 / ra.stages, ra.more = ra.g.C / 8 % ra.stages;
    ra.count = fast_div((unsigned)ra.base), ra.count1 = fast_div((unsigned)ra.base + 1);
    ra.in_scale = in_scale;
    ra.in_half = in_round_mode == OTTER_HIP_ROUND_SSE ? 0.5f : 0.49999997f;
    const int blocks = (ra.g.K + 16 * c.fm - 1) / (16 * c.fm);
    ra.blocks_per_wg = rows_blocks_per_workgroup(ra, blocks, c.fm);
    const int steps = rows_steps(ra.g.C, ra.g.kh * ra.g.kw);
    ra.warm_steps = steps >= 24 ? steps : 0;
    ra.consts = (int)((lds + 15) / 16 * 16);
    lds = rows_lds(lds, ra.blocks_per_wg, c.fm);
    const dim3 grid((unsigned)ra.n_tiles, (unsigned)((blocks + ra.blocks_per_wg - 1) / ra.blocks_per_wg), (unsigned)g_in.groups);
    const int epi = full_epilogue(pick_epilogue(ep, ra.g.K), ep);
    auto go = [&](auto kernel, auto ea) {
        if (lds > 64 * 1024) {  // (rows that fill the tile's share: the constants lie beyond it)
            const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, 72 * 1024);
            if (e != hipSuccess) return e;
        }
        launch(kernel, grid, dim3(256), lds, stream, (const int8_t*)x, wpk, out, ra, ea);
        return hipGetLastError();
    };
#define OHIP_ROWS2(I_, FM_, FN_, E_)                                                                     \
    if (config == I_ && epi == E_) {                                                                     \
        if (!f32in) return go(conv_rows_kernel<FM_, FN_, E_, false>, EpiArgs<E_>::of(ep));               \
        if constexpr (E_ != EPI_GENERIC) return go(conv_rows_kernel<FM_, FN_, E_, true>, EpiArgs<E_>::of(ep)); \
    }
#define OHIP_ROWS(I_, FM_, FN_) \
    OHIP_ROWS2(I_, FM_, FN_, EPI_I8_P8) OHIP_ROWS2(I_, FM_, FN_, EPI_I8_P8_NONNEG) OHIP_ROWS2(I_, FM_, FN_, EPI_I8_P8_FULL) OHIP_ROWS2(I_, FM_, FN_, EPI_F32_P4) OHIP_ROWS2(I_, FM_, FN_, EPI_GENERIC)
    OHIP_ROWS(0, 2, 2)
    OHIP_ROWS(1, 2, 4)
    OHIP_ROWS(2, 4, 2)
    OHIP_ROWS(3, 4, 4)
#undef OHIP_ROWS
#undef OHIP_ROWS2
    return hipErrorInvalidValue;
}

}  // namespace ohip
