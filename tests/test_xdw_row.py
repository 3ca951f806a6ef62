"""CPU: the descriptor and the scalar offsets with which the pointwise + depthwise launch requests an input row (xdw_row.hpp). No scalar
offset is beyond the descriptor's bytes, where the difference that the hardware compares a lane's offset with would wrap; every byte
that a lane asks for lies in the blob; an absent row asks for nothing."""
import os
import subprocess

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "tensor_amd", "csrc")

SOURCE = r"""
#include <cstdio>
#include <initializer_list>
#include "xdw_row.hpp"
using namespace ohip;
static const char* check(int N, int octets, int H, int W, int img, int iy) {
    const unsigned plane = (unsigned)(H * W) * 8u, bytes = (unsigned)(N * octets) * plane;
    const bool there = iy >= 0 && iy < H;
    const unsigned first = (unsigned)(img * octets) * plane + (unsigned)(iy * W) * 8u;
    const XdwRow r = xdw_row(there, bytes, first, xdw_octets(plane, octets));
    const unsigned at[4] = {r.at, r.at1, r.at8, r.at9};
    const int step[4] = {0, 1, 8, 9};
    if (r.bytes != (there ? bytes : 0u)) return "bytes";
    for (int i = 0; i < 4; ++i) {
        if (at[i] > r.bytes) return "an offset beyond the descriptor";
        if (!there || step[i] >= octets) continue;
        if (at[i] != first + (unsigned)step[i] * plane) return "another octet";
        for (int q = 0; 2 * q + step[i] < octets && q < 4; ++q)  // lane group q starts at octet 2 q, its last pixel is W - 1
            if (at[i] + (unsigned)(2 * q) * plane + (unsigned)(W - 1) * 8u + 8u > bytes) return "a byte beyond the blob";
    }
    return nullptr;
}
int main() {
    const int sides[][2] = {{1, 1}, {1, 64}, {7, 7}, {14, 13}, {56, 3}, {112, 112}};
    for (int N : {1, 3})
        for (int octets = 1; octets <= 16; ++octets)
            for (auto& s : sides)
                for (int img = 0; img < N; ++img)
                    for (int iy = -2; iy < s[0] + 10; ++iy)
                        if (const char* e = check(N, octets, s[0], s[1], img, iy)) {
                            std::printf("%s: N %d octets %d %dx%d image %d row %d\n", e, N, octets, s[0], s[1], img, iy);
                            return 1;
                        }
    return 0;
}
"""


def test_requests_stay_inside_their_descriptor(tmp_path):
    src, exe = tmp_path / "xdw_row.cpp", str(tmp_path / "xdw_row")
    src.write_text(SOURCE)
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-I", CSRC, str(src), "-o", exe])
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout
