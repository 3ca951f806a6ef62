"""The requantization behind ReLU / clip whose upper clamps are all 127 (quant4_full in common.hpp): bytes from doubled values, rounded to nearest
even by the conversion, instead of values that are truncated, clamped and packed. On the CPU the rule over every float; on the GPU the kernels
that have it, at scales where every second result is a tie, against the oracle."""
import subprocess

import numpy as np
import pytest

from gpu_util import run_conv
from tensor_amd import capi

SOURCE = r"""
#include <math.h>
#include <stdint.h>
#include <stdio.h>
#include <string.h>
int main(void) {
    const float halves[2] = {0.5f, 0.49999997f};
    long bad = 0;
    for (int h = 0; h < 2; ++h) {
        const float half = halves[h];
#pragma omp parallel for reduction(+ : bad)
        for (uint32_t b = 0; b <= 0x7f800000u; ++b)  /* zero to infinity, and their negatives */
            for (int neg = 0; neg < 2; ++neg) {
                float t;
                memcpy(&t, &b, 4);
                if (neg) t = -t;
                volatile float y = t + half, t2 = t + t, z = t2 + half;
                const int want = y >= 127.f ? 127 : y <= 0.f ? 0 : (int)y;
                /* v_cvt_pk_u8_f32: to nearest even, saturated to a byte */
                const int byte = z >= 255.f ? 255 : z <= 0.f ? 0 : (int)nearbyintf(z);
                bad += byte >> 1 != want;
            }
    }
    printf("%ld\n", bad);
    return bad != 0;
}
"""


def test_the_rule_for_every_float(tmp_path):
    src, exe = tmp_path / "full.c", str(tmp_path / "full")
    src.write_text(SOURCE)
    subprocess.check_call(["gcc", "-O2", "-fopenmp", str(src), "-o", exe, "-lm"])
    assert subprocess.run([exe], capture_output=True, text=True).stdout.strip() == "0"


@pytest.mark.gpu
@pytest.mark.parametrize("half,out_round", [(0.5, capi.ROUND_SSE), (0.49999997, capi.ROUND_EXACT)])
def test_the_rule_on_the_gpu(hip, half, out_round):
    """The conversion itself: every quarter step from -1 to 129 and the three floats on either side, as the biases of a layer without weights."""
    values = [np.arange(-4, 517, dtype=np.float32) / np.float32(4)]
    for way in (-np.inf, np.inf):
        beside = values[0]
        for _ in range(3):
            beside = np.nextafter(beside, np.float32(way))
            values.append(beside)
    bias = np.concatenate(values + [np.zeros(1, np.float32)])
    K, C, s = bias.size, 64, 4
    assert K % 8 == 0
    conv = hip.conv(wq=np.zeros((K, C, 1, 1), np.int8), scale_in=np.ones(K, np.float32), bias=bias, in_scale=1.0, out_scale=[1.0], out_kind=capi.OUT_I8, act=1,
                    out_round=out_round)
    x = hip.to_device(np.ones(C * s * s, np.int8))
    got = capi.unpack_np(conv.forward(x, capi.I8_P8, 1, s, s, capi.I8_P8).cpu().numpy(), 8, (1, K, s, s))
    want = np.clip((bias + np.float32(half)).astype(np.int32), 0, 127).astype(np.int8)
    np.testing.assert_array_equal(got, np.broadcast_to(want[None, :, None, None], got.shape))


LAYERS = [
    # C, K, kernel, stride, groups, N, H, W, fp32 input
    (64, 128, 3, 1, 1, 8, 28, 28, False),   # LDS-halo kernel
    (88, 176, 3, 2, 1, 2, 21, 19, False),   # operands straight from memory
    (256, 256, 3, 1, 8, 8, 28, 28, False),  # staged rows
    (96, 576, 1, 1, 1, 4, 14, 14, False),   # pointwise, whole reduction
    (576, 96, 1, 1, 1, 2, 14, 14, False),   # pointwise, split reduction
    (64, 40, 1, 1, 1, 1, 9, 7, True),
    (32, 32, 3, 1, 32, 2, 30, 30, False),
    (32, 32, 3, 2, 32, 2, 31, 29, False),
    (24, 24, 5, 1, 24, 2, 17, 20, False),
    (32, 32, 3, 1, 32, 2, 30, 30, True),
]


@pytest.mark.gpu
@pytest.mark.parametrize("scale", [1.0, 21.25, 21.0])  # clip: 6 * 21.25 is beyond 127, 6 * 21 is 126
@pytest.mark.parametrize("act", [1, 3])
@pytest.mark.parametrize("C,K,k,stride,groups,N,H,W,f32", LAYERS)
def test_ties_and_clamps(hip, oracle, C, K, k, stride, groups, N, H, W, f32, act, scale):
    rng = np.random.default_rng(C * K + k)
    x = rng.integers(-60, 61, (N, C, H, W)).astype(np.float32 if f32 else np.int8)
    cg = C // groups
    wq = np.zeros((K, cg * k * k), np.int8)
    for row in wq:  # sums that cover a few hundred steps, whatever the reduction
        row[rng.choice(cg * k * k, 5, replace=False)] = rng.integers(-3, 4, 5)
    wq = wq.reshape(K, cg, k, k)
    # results of half a step: sums times 1 / 2 at scale 1, so that every odd one is a tie; sums times 1 / 32 behind the others
    ws = np.full(K, 2.0 if scale == 1.0 else 32.0, np.float32)
    bias = rng.integers(-4, 5, K).astype(np.float32) * np.float32(0.5)
    got, _ = run_conv(hip, oracle, x, wq, ws, 1.0, stride=stride, pad=k // 2, groups=groups, bias=bias, top_scale=scale, out_kind=capi.OUT_I8, act=act)
    want = oracle.conv_layer_forward(x, wq, ws, 1.0, stride=(stride, stride), pad=(k // 2,) * 2, groups=groups, bias=bias, top_scale=scale,
                                     int8_out=True, act_type=act)
    assert got.max() >= (6 if act == 3 and scale == 1.0 else 100)
    np.testing.assert_array_equal(got, want)


@pytest.mark.gpu
@pytest.mark.parametrize("scale", [21.25, 21.0])  # upper clamps of 127 and 126
@pytest.mark.parametrize("act", [1, 3])
@pytest.mark.parametrize("C,K,k,stride,groups,N,H,W,f32", LAYERS)
def test_results_beyond_the_range(hip, oracle, C, K, k, stride, groups, N, H, W, f32, act, scale):
    """Biases that are infinite, beyond every scale or not a number: the clamps, and zero, whichever way the bytes are made."""
    rng = np.random.default_rng(C + K + k)
    x = rng.integers(-60, 61, (N, C, H, W)).astype(np.float32 if f32 else np.int8)
    wq = rng.integers(-3, 4, (K, C // groups, k, k)).astype(np.int8)
    bias = np.resize(np.array([np.inf, -np.inf, np.nan, 3e38, -3e38, 0.5, 1e30], np.float32), K)
    got, _ = run_conv(hip, oracle, x, wq, np.full(K, 32.0, np.float32), 1.0, stride=stride, pad=k // 2, groups=groups, bias=bias, top_scale=scale,
                      out_kind=capi.OUT_I8, act=act)
    top = int(6 * scale) if act == 3 and scale == 21.0 else 127
    for first, want in ((0, top), (1, 0), (2, 0), (3, top), (4, 0), (6, top)):
        assert (got[:, first::7] == want).all(), first
    zero = np.where(np.isfinite(bias), bias, np.float32(0))
    want = oracle.conv_layer_forward(x, wq, np.full(K, 32.0, np.float32), 1.0, stride=(stride, stride), pad=(k // 2,) * 2, groups=groups, bias=zero,
                                     top_scale=scale, int8_out=True, act_type=act)
    np.testing.assert_array_equal(got[:, 5::7], want[:, 5::7])
