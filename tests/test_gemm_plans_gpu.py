"""The GEMM's launch plan over the ranges of its rules: the kernel that a call takes, by its profiled name, and
sampled rows of its output against the oracle, at the tolerance of the sweep (f32 sums in another order)."""

import functools

import numpy as np
import pytest

import oracle as ox
import wavo_amd as wa
from wavo_amd import gguf

pytestmark = pytest.mark.gpu

KW32, KW3264, KW64 = "32x32_w1x1_n2_p3_k8", "32x64_w1x1_n2_p3_k8", "64x64_w1x1_n2_p3_k4"
NAMES = {wa.Q8_0: "q8_0", wa.Q4_0: "q4_0", wa.F16: "f16"}


@functools.lru_cache(maxsize=2)
def weights(n, k, wtype):
    w = np.random.default_rng(n * 7 + k).standard_normal(n * k, dtype=np.float32) * np.float32(0.02)
    return gguf.encode(w, wtype), np.random.default_rng(n).standard_normal(n, dtype=np.float32)


def check(gpu, m, n, k, wtype, plan, out16=False):
    raw, bias = weights(n, k, wtype)
    l = gpu.linear([(raw, wtype, k, n)], bias)
    a = np.random.default_rng(m + k).standard_normal((m, k), dtype=np.float32)
    ah = gpu.upload(a.astype(np.float16))
    cb = gpu.buffer(m * l.width)
    gpu.profile(1)
    try:
        gpu.gemm_h(ah, l, cb, m, wa.BIAS, 0.0, out16=out16)
        names = [x["kernel"].split(" ")[0] for x in gpu.profile_read()]
    finally:
        gpu.profile(0)
    assert names[0] == f"gemm_{NAMES[wtype]}_{plan}", f"{m}x{n}x{k} {NAMES[wtype]}: {names}"
    rng = np.random.default_rng(m)
    rows = np.unique(np.concatenate([[0, m - 1], rng.choice(m, min(m, 24), replace=False)]))
    dtype = np.float16 if out16 else np.float32
    size = np.dtype(dtype).itemsize
    got = np.stack([gpu.read(cb, (l.width,), dtype, offset_bytes=size * int(r) * l.width) for r in rows])[:, :n].astype(np.float32)
    want = ox.gemm(a[rows], ox.Linear(wtype, k, [(raw, n)], bias), len(rows), ox.BIAS)
    top = max(1.0, float(np.abs(want).max()))
    tol = (2e-5 + (2.0 ** -11 if out16 else 0.0)) * top  # (f16 outputs: rounded once)
    assert np.abs(got - want).max() <= tol, f"{m}x{n}x{k} {NAMES[wtype]} {plan}"


# Wavefronts that split k: not over one k step (of 64), on 32x64 tiles not over two, from there on yes.
@pytest.mark.parametrize("m,n,k,wtype,plan", [
    (28, 832, 64, wa.Q8_0, "64x64_w2x2_n3"), (3, 4800, 64, wa.F16, "64x64_w2x2_n3"), (260, 1408, 64, wa.Q4_0, "64x64_w2x2_n3"),
    (2020, 160, 128, wa.Q4_0, "64x64_w2x2_n4_k2"), (44, 576, 128, wa.Q4_0, KW32), (11, 128, 128, wa.F16, KW32),
    (1133, 288, 192, wa.Q8_0, KW3264), (465, 800, 512, wa.Q4_0, KW3264), (60, 1024, 4096, wa.F16, KW32)])
def test_k_wavefronts_need_k_to_split(gpu, m, n, k, wtype, plan):
    check(gpu, m, n, k, wtype, plan)


# One to two 64x64 tiles per CU: 96x64 tiles in two k groups where k has pairs of steps, else 64x64 tiles; few rows
# whose 96x64 tiles do not run at once by k wavefronts with quantized weights, on 64x64 tiles with F16 ones.
@pytest.mark.parametrize("m,n,k,wtype,plan", [
    (750, 2048, 1024, wa.Q8_0, "96x64_w1x2_n2_k2"), (750, 2048, 1024, wa.F16, "96x64_w1x2_n2_k2"),
    (765, 1408, 512, wa.F16, "96x64_w1x2_n2_k2"), (513, 2176, 896, wa.Q4_0, "96x64_w1x2_n2_k2"),
    (500, 3072, 1024, wa.Q8_0, KW64), (500, 3072, 1024, wa.F16, "64x64_w2x2_n3"), (623, 2688, 1536, wa.F16, "96x64_w1x2_n2_k2"),
    (392, 3520, 1728, wa.Q4_0, KW64), (339, 3392, 1088, wa.Q8_0, KW64), (918, 1472, 1984, wa.F16, "64x64_w2x2_n3"),
    (1393, 1344, 2880, wa.Q4_0, "64x64_w2x2_n3"), (1286, 1024, 2496, wa.Q8_0, "64x64_w2x2_n3")])
@pytest.mark.parametrize("out16", [False, True])
def test_one_to_two_tiles_per_cu(gpu, m, n, k, wtype, plan, out16):
    check(gpu, m, n, k, wtype, plan, out16)


# A long k: split over few tiles, whole in two k groups from there on, on the widest of the 64x64, 96x64 and 96x128
# tiles that still gives every CU one.  k of pairs of steps that no split into four divides (4224, 4992) as well.
@pytest.mark.parametrize("m,n,k,wtype,plan", [
    (750, 1024, 4096, wa.Q8_0, "96x64_w1x2_n2_s4_k2"), (166, 2752, 4224, wa.Q8_0, "64x64_w2x2_n4_k2"),
    (400, 1408, 4992, wa.Q4_0, "64x64_w2x2_n4_k2"), (1024, 1024, 4224, wa.F16, "64x64_w2x2_n4_k2"),
    (549, 1664, 4608, wa.F16, "64x64_w2x2_n4_k2"), (750, 1792, 4096, wa.Q4_0, "96x64_w1x2_n2_k2"), (670, 1664, 4224, wa.Q4_0, "96x64_w1x2_n2_k2"),
    (300, 4288, 4224, wa.Q4_0, "96x128_w1x4_n3_k2"), (1500, 1280, 5120, wa.Q8_0, "96x128_w1x4_n3_k2"),
    (757, 1792, 4096, wa.F16, "128x128_w2x2_n2_s4")])
def test_long_k(gpu, m, n, k, wtype, plan):
    check(gpu, m, n, k, wtype, plan)


# About a tile per CU and more: each tile of the choice by rounds, for quantized and F16 weights, over rows and columns
# that end inside a tile, a k without pairs of steps (960) and short ones (256); and where the choice begins.
@pytest.mark.parametrize("m,n,k,wtype,plan", [
    (2970, 900, 256, wa.Q8_0, "96x128_w1x4_n3_k2"),
    (2970, 900, 256, wa.F16, "96x128_w1x4_n3_k2"),
    (3220, 516, 960, wa.Q8_0, "96x128_w1x4_n3"),
    (3220, 516, 960, wa.F16, "96x128_w1x4_n3"),
    (3503, 772, 256, wa.Q4_0, "128x128_w2x4_n3"),
    (3503, 772, 256, wa.F16, "128x128_w2x4_n3"),
    (3680, 3204, 960, wa.Q8_0, "128x128_w2x2_n2"),
    (2309, 2489, 256, wa.F16, "128x128_w2x2_n2"),
    (3000, 4096, 1024, wa.Q8_0, "192x128_w2x4_n2"),
    (2947, 1284, 256, wa.Q4_0, "192x128_w2x4_n2"),
    (2947, 1284, 256, wa.F16, "192x128_w2x4_n2"),
    (2502, 2336, 2048, wa.Q8_0, "256x128_w2x4_n3"),
    (2502, 2336, 2048, wa.F16, "256x128_w2x4_n3"),
    (22384, 288, 1984, wa.F16, "192x256_w2x4_n2"),
    (3894, 3097, 768, wa.Q4_0, "256x256_w2x4_n2"),
    (9477, 1280, 5120, wa.Q8_0, "192x256_w2x4_n2"),
    (3894, 3097, 768, wa.F16, "256x256_w2x4_n2"),
    (750, 4096, 1024, wa.Q8_0, "96x128_w1x4_n3_k2"),
    (30020, 256, 256, wa.Q8_0, "128x128_w2x4_n3"),
    (4633, 480, 512, wa.Q8_0, "96x128_w1x4_n3_k2"),
    (5163, 512, 192, wa.Q4_0, "64x64_w2x2_n3"), (5735, 512, 192, wa.F16, "64x64_w2x2_n3"),
    (500, 4096, 512, wa.F16, "96x128_w1x4_n3_k2"), (491, 4544, 256, wa.F16, "96x128_w1x4_n3_k2"),
    (500, 4096, 512, wa.Q8_0, KW64)])
def test_choice_by_rounds(gpu, m, n, k, wtype, plan):
    check(gpu, m, n, k, wtype, plan)
