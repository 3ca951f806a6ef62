"""CPU: the scalar offsets with which the launch of a depthwise layer and the pointwise layers behind it (dwpw_requests.hpp) reads weights and
reads and writes fp32 blobs. None is beyond the descriptor's bytes, where the difference that the hardware compares a lane's offset with
would wrap: reduction steps that do not exist, addends and sums that nobody has or wants, channels past the last whole pair of tiles. Every
step and element that exists is at its place."""
import os
import subprocess

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "tensor_amd", "csrc")

SOURCE = r"""
#include <cstdio>
#include <initializer_list>
#include "dwpw_requests.hpp"
using namespace ohip;
typedef unsigned long long u64;
static int fail(const char* what, int a, int b, int c, int d) { return std::printf("%s: %d %d %d %d\n", what, a, b, c, d), 1; }
int main() {
    for (int steps = 1; steps <= 20; ++steps)
        for (int K : {8, 32, 40, 88, 128, 264, 1280}) {
            const int mt = (K + 127) / 128 * 8, pairs = (K + 31) / 32;
            const u64 bytes = (u64)steps * mt * 1024;
            for (int step = 0; step < (steps + 3) / 4 * 4; ++step)  // (asked for in fours, the odd ones by twos)
                for (int pair = 0; pair < pairs; ++pair) {
                    const u64 at = dwpw_weights_at(step, steps, mt, pair);
                    if (at > bytes) return fail("weights: beyond them", step, steps, K, pair);
                    if (step >= steps && at != bytes) return fail("weights: a step that does not exist", step, steps, K, pair);  // (every lane is out of range there)
                    if (step < steps && at != ((u64)step * mt + 2 * pair) * 1024) return fail("weights: another step", step, steps, K, pair);
                }
        }
    // elements of 4 channels (a pixel's are HW * 16 bytes apart) and of 8 (two quarters of 16 bytes each)
    for (int pack : {4, 8})
        for (int K : {4, 8, 12, 24, 32, 36, 40, 88, 264, 1280})
            for (u64 HW : {1ull, 49ull, 2704ull, 1ull << 20})
                for (u64 n : {1ull, 2ull, 17ull}) {
                    const u64 bytes = n * HW * (u64)K * 4;
                    if (K % pack || bytes >= 1ull << 31) continue;
                    for (bool there : {true, false}) {
                        const DwPwFloats f = dwpw_floats(there, (unsigned)bytes, (unsigned)HW, pack == 8 ? 16u : (unsigned)HW * 16u);
                        if (f.bytes != (there ? bytes : 0)) return fail("floats: bytes", pack, K, (int)HW, there);
                        for (int pr = 0; pr < (K + 31) / 32; ++pr)
                            for (int h = 0; h < 2; ++h) {
                                if (f.at(pr, h) > f.bytes) return fail("floats: beyond the blob", pack, K, (int)HW, there);
                                for (int q = 0; q < 4 && there; ++q) {
                                    const u64 ch = 32u * pr + 8 * q + 4 * h;
                                    if (ch >= (u64)K) continue;
                                    const u64 lane = pack == 8 ? q * HW * 32 : 2 * q * HW * 16;  // of the first pixel
                                    const u64 want = pack == 8 ? ch / 8 * HW * 32 + ch % 8 * 4 : ch / 4 * HW * 16;
                                    if (lane + f.at(pr, h) != want) return fail("floats: another element", pack, K, (int)HW, (int)ch);
                                }
                            }
                    }
                }
    return 0;
}
"""


def test_requests_stay_inside_what_they_name(tmp_path):
    src, exe = tmp_path / "dwpw_requests.cpp", str(tmp_path / "dwpw_requests")
    src.write_text(SOURCE)
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-I", CSRC, str(src), "-o", exe])
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout


STAGED = r"""
#include <cstdio>
#include <initializer_list>
#include <vector>
#include "dwpw_requests.hpp"
using namespace ohip;
// N images of C channels (octets of 8 bytes), copied into places as the launch copies them; a place holds the number of the blob's element plus one
int main() {
    struct Case { int ks, pad, dil, C, N, H, W; };
    for (const Case& c : {Case{3, 1, 1, 88, 3, 13, 13}, {3, 1, 1, 16, 5, 7, 7}, {5, 2, 1, 24, 2, 9, 26}, {3, 1, 1, 8, 9, 1, 1}, {3, 2, 2, 40, 2, 12, 9}, {5, 2, 1, 128, 2, 52, 52},
                          {3, 1, 1, 72, 4, 3, 5}, {3, 1, 1, 32, 2, 4, 112}, {5, 4, 2, 8, 3, 6, 3}, {3, 1, 1, 136, 1, 14, 14}})
        for (int pixels : {16, 32, 64, 128}) {
            const DwPwStage st = dwpw_stage(c.C, c.H, c.W, c.ks, c.pad, c.pad, c.dil, c.dil, pixels);
            const unsigned HW = c.H * c.W, C8 = c.C / 8, total = c.N * HW, sets = 64u >> st.lg_lanes;
            const size_t elements = (size_t)total * C8, places = (size_t)st.octets * st.pitch;
            if (st.octets < (C8 + 1) / 2 * 2 || st.slots + 2 > st.pitch) return std::printf("room\n"), 1;
            for (unsigned first = 0; first < total; first += pixels) {
                const unsigned n_first = first / HW;
                const int begin = dwpw_run(st, HW, first, n_first);
                std::vector<size_t> lds(places, ~(size_t)0);
                for (unsigned from = 0; from < st.units; from += 64)
                    for (unsigned o = 0; o < C8; o += sets)
                        for (unsigned lane = 0; lane < 64; ++lane) {
                            const unsigned unit = lane & ((1u << st.lg_lanes) - 1), sub = lane >> st.lg_lanes;
                            if (from + unit >= st.units) continue;
                            const int at = begin + 2 * (int)(from + unit);
                            const unsigned im = (unsigned)at / st.image;
                            const bool in = at >= 0 && 2 * (from + unit) < st.slots && im * HW < total;
                            const size_t place = (size_t)o * st.pitch + 2 * from + 2 * lane;
                            if (place + 2 > places) return std::printf("a copy beyond its room\n"), 1;
                            for (int e = 0; e < 2; ++e) {
                                const size_t element = in ? ((size_t)dwpw_copied(st, HW, C8, im, sub, (unsigned)at) + (size_t)o * HW * 8) / 8 + e : elements;
                                lds[place + e] = element < elements ? element + 1 : 0;
                            }
                        }
                for (unsigned p = 0; p < (unsigned)pixels && first + p < total; ++p) {
                    const unsigned n = (first + p) / HW, pix = first + p - n * HW;
                    const int y = pix / c.W, x = pix % c.W, window = dwpw_window(st, n, pix) - begin;
                    for (unsigned o = 0; o < C8; ++o) {
                        if (lds[(size_t)o * st.pitch + st.slots] != 0) return std::printf("no zeros behind the pixels\n"), 1;
                        for (int dy = 0; dy < c.ks; ++dy)
                            for (int dx = 0; dx < c.ks; ++dx) {
                                const int iy = y - c.pad + dy * c.dil, ix = x - c.pad + dx * c.dil;
                                if (iy < 0 || iy >= c.H || ix < 0 || ix >= c.W) continue;
                                const int slot = window + dy * c.dil * c.W + dx * c.dil;
                                if (slot < 0 || slot >= (int)st.slots) return std::printf("a tap beyond the run\n"), 1;
                                if (lds[(size_t)o * st.pitch + slot] != ((size_t)n * C8 + o) * HW + iy * c.W + ix + 1)
                                    return std::printf("another pixel: %dx%d k%d, %d pixels, octet %u\n", c.H, c.W, c.ks, pixels, o), 1;
                            }
                    }
                }
            }
        }
    return 0;
}
"""


def test_staged_pixels_are_those_of_the_windows(tmp_path):
    """Every tap inside the image finds its pixel among the places that a tile's copies fill (image sides whose product is odd and even, images of
    one pixel, tiles over several images, dilation), one outside it zeros, and no copy leaves its room."""
    src, exe = tmp_path / "dwpw_stage.cpp", str(tmp_path / "dwpw_stage")
    src.write_text(STAGED)
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-I", CSRC, str(src), "-o", exe])
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout
