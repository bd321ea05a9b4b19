"""How often a layer's weights are held on the device: a loaded model holds each once, in the form its readers
take; a layer of wh_linear_new holds its GGUF bytes and, for the GEMMs, tiles of as many bytes, which it does
without where the caller says so, the GEMM then reading the GGUF bytes."""

import ctypes
import os
import re

import numpy as np
import pytest

import oracle as ox
import wavo_amd as wa
from wavo_amd import gguf, synth

pytestmark = pytest.mark.gpu

MODELS = os.environ.get("WAVO_MODELS", "/tmp/wavo_models")


def free_bytes(gpu):
    """Device memory not allocated (hipMemGetInfo of the runtime the library is linked to)."""
    gpu.sync()
    path = next(p for line in open("/proc/self/maps") for p in re.findall(r"/\S*libamdhip64\S*", line))
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert ctypes.CDLL(path).hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


# Models of a few hundred MB, most of it weights: beside them the device holds biases, norms and tables, each in
# an allocation of whole 2 MiB pages, 0.15 to 0.5 of the file.  Each weight twice would be 2.05 and more.
@pytest.mark.parametrize("name,cut,wtype", [("gigaam", {}, gguf.Q8_0), ("gigaam", dict(layers=6), gguf.F16), ("parakeet", {}, gguf.Q8_0),
                                            ("whisper", dict(layers=1), gguf.Q8_0)])
def test_a_model_holds_each_weight_once(gpu, tmp_path, name, cut, wtype):
    if cut:
        path = synth.write_model(str(tmp_path / "m.gguf"), dict(synth.CONFIGS[name], **cut), 0, wtype)
    else:
        path = synth.model_path(name, wtype=wtype, directory=MODELS)
    size = os.path.getsize(path)
    wa.Model(gpu, path).free()  # the upload's own buffers are there from here on
    before = free_bytes(gpu)
    m = wa.Model(gpu, path)
    held = before - free_bytes(gpu)
    m.free()
    left = before - free_bytes(gpu)
    assert held < 1.75 * size, f"{held / 1e6:.1f} MB held for a file of {size / 1e6:.1f} MB"
    assert left < size / 4, f"{left / 1e6:.1f} MB kept after the model was freed"


@pytest.mark.parametrize("wtype", [wa.Q8_0, wa.Q4_0, wa.F16])
def test_a_layer_without_tiles(gpu, wtype):
    """The GEMMs of a layer that holds its GGUF bytes alone, at the tolerances of one that has tiles, over the
    entry points and epilogues; its GEMV and memory."""
    m, n, k, d = 70, 16385, 1024, 64
    w = np.random.default_rng(1).normal(0, 0.02, (n, k)).astype(np.float32)
    raw, bias = ox.quantize(w, wtype), np.random.default_rng(2).standard_normal(n + d).astype(np.float32)
    a = np.random.default_rng(3).standard_normal((m, k)).astype(np.float32)
    both = [gpu.linear([(raw, wtype, k, n)], bias)]
    at = free_bytes(gpu)
    both.append(gpu.linear([(raw, wtype, k, n)], bias))
    two = at - free_bytes(gpu)
    gpu.tune("weight_tiles", "0")
    try:
        at = free_bytes(gpu)
        l = gpu.linear([(raw, wtype, k, n)], bias)
        one = at - free_bytes(gpu)
    finally:
        gpu.tune("weight_tiles", "1")
    size = len(raw)
    assert one < size + (6 << 20) < 2 * size <= two, (one, two, size)  # rows and bias in whole 2 MiB pages
    ol = ox.Linear(wtype, k, [(raw, n)], bias[:n])
    c0 = np.random.default_rng(4).standard_normal((m, l.width)).astype(np.float32)
    ab, ah = gpu.upload(a), gpu.upload(a.astype(np.float16))
    gpu.profile(1)
    try:
        for e, alpha in ((wa.BIAS, 0.0), (wa.RESIDUAL, 0.5), (wa.SILU, 0.0), (wa.GELU, 0.0)):
            cb = gpu.upload(c0)
            gpu.gemm(ab, l, cb, m, e, alpha)
            got = gpu.read(cb, c0.shape)
            want = ox.gemm_wide(a, ol, m, e, alpha, c=c0, bias2=bias[n:], dual=d)
            tol = 2e-5 * max(1.0, float(np.abs(want).max()))  # f32 sums in another order
            assert np.abs(got - want).max() <= tol, f"type {wtype} epilogue {e}"
            if e in (wa.BIAS, wa.SILU):
                hb = gpu.buffer((c0.size + 1) // 2)
                gpu.gemm_h(ah, l, hb, m, e, 0.0, out16=True)
                got = gpu.read(hb, c0.shape, np.float16).astype(np.float32)
                assert np.abs(got - want).max() <= tol + 2.0 ** -11 * float(np.abs(want).max()), f"f16, epilogue {e}"
        names = [x["kernel"] for x in gpu.profile_read()]
    finally:
        gpu.profile(0)
    assert any(x.startswith("gemm_reg_") for x in names) and not any("to_half" in x for x in names), names
    y, z = gpu.buffer(l.width), gpu.buffer(l.width)
    gpu.gemv(ab, l, y, wa.BIAS)
    gpu.gemv(ab, both[0], z, wa.BIAS)
    assert np.array_equal(gpu.read(y, (n,)), gpu.read(z, (n,)))
