"""CPU: the scalar offsets with which the launch on staged rows requests the octets of a stage (rows_stage.hpp). None is beyond the blob's bytes,
where the difference that the hardware compares a lane's offset with would wrap, and every octet that the stage has is asked for at
its place: layers of few octets on one image, of several stages, of blobs of up to 2 GB. The parts that the threads are dealt in hold
the places of a plane."""
import os
import subprocess

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "tensor_amd", "csrc")

SOURCE = r"""
#include <cstdio>
#include <initializer_list>
#include "rows_stage.hpp"
using namespace ohip;
typedef unsigned long long u64;
// a blob of `octets` planes of one image; octets [first, first + count) of it are the stage
static const char* check(u64 plane, int octets, int first, int count, int sub, int together) {
    const u64 bytes = plane * (u64)octets;
    for (int part = 0; part < sub; ++part) {
        RowsWalk w = rows_walk((unsigned)plane, first, count, sub);
        for (int oct = part; oct < count; oct += together * sub)
            for (int u = 0; u < together; ++u) {
                const unsigned at = w.next();
                if (at > bytes) return "a scalar offset beyond the blob";
                if (oct + u * sub < count && at + part * plane != (u64)(first + oct + u * sub) * plane) return "another octet";
            }
    }
    return nullptr;
}
int main() {
    for (int places = 1; places <= 4096; ++places) {
        const int shift = rows_parts_shift(places), part = 256 >> shift;
        // a part holds the plane where there are several, and is no larger than it has to be
        if (shift < 0 || shift > 3 || (shift > 0 && places > part) || (shift < 3 && places <= part / 2)) {
            std::printf("%d places in parts of %d threads\n", places, part);
            return 1;
        }
    }
    for (int octets = 1; octets <= 40; ++octets)
        for (u64 plane : {8ull, 32ull, 392ull, 40000ull, 1ull << 26, (1ull << 31) / (u64)octets / 8 * 8})
            if (plane * (u64)octets < (1ull << 31))
                for (int count = 1; count <= 8 && count <= octets; ++count)
                    for (int first = 0; first + count <= octets; ++first)
                        for (int sub : {1, 2, 4, 8})
                            for (int together : {2, 4})
                                if (const char* e = check(plane, octets, first, count, sub, together)) {
                                    std::printf("%s: plane %llu, octets %d, stage %d + %d, %d parts, %d together\n", e, plane, octets, first, count, sub, together);
                                    return 1;
                                }
    return 0;
}
"""


def test_requests_stay_inside_the_blob(tmp_path):
    src, exe = tmp_path / "rows_stage.cpp", str(tmp_path / "rows_stage")
    src.write_text(SOURCE)
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-I", CSRC, str(src), "-o", exe])
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout
