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
