"""The LDS-DMA ring at the sizes where its tilings, tails and trimmed rings can go wrong, against the
oracle: K tails (a multiple of 8 that is not one of 64; fp32: of 4), N that no group of 4 divides, single
rows, reductions of one slice up to more than the ring's stages, every tiling the estimate can pick
(named one by one: test_every_tiling), 1x1 convs as dense products, and the fp32 tiles (ring and split K).

Tolerances: 16-bit outputs are one rounding of an fp32 sum (2^-11 / 2^-8 relative to the element, whose
magnitude is at most the maximum). The fp32 sums of K terms, of unit variance in all, differ in order only: each of
K roundings is at most 2^-24 of a partial sum, sqrt(K) 2^-24 of the largest result as a random walk, and four times
that bounds the largest of 10^6 such errors; 2e-6 for the activations' approximations. (A sum over 16-bit operands
would be 1e-4 off.) The oracle's convs sum directly: its Winograd transforms round at a multiple of that."""
import os
import re

import numpy as np
import pytest

import oracle as O
from conftest import max_rel
from oracle.interp import _bf16
from simdonnx_amd import synth
from simdonnx_amd.backend import HipInferenceSession
from simdonnx_amd.plan import NHWC, PlanBuilder

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _on_the_ring(monkeypatch):
    # ragged rows and short reductions too, where the implicit GEMM is the faster kernel
    monkeypatch.setenv("SIMDONNX_HIP_RING", "1")


def stored(a, storage):
    a = np.asarray(a, np.float32)
    return a if storage == "f32" else _bf16(a) if storage == "bf16" else a.astype(np.float16).astype(np.float32)


def tol(storage, k):
    return {"f32": 2e-6 + 4 * k**0.5 * 2.0**-24, "f16": 1e-3, "bf16": 8e-3}[storage]


def run(hip, plan, ins, storage):
    g = hip.graph(plan, storage)
    kernels = g.kernels
    with HipInferenceSession(g) as s:
        for i, x in enumerate(ins):
            s.set_input(x, i)
        return s.run().copy(), kernels


GEMMS = [(1, 8, 1), (1, 64, 64), (3, 16, 5), (64, 24, 64), (47, 40, 88), (65, 72, 97), (33, 120, 6), (130, 200, 200),
         (256, 1000, 96), (200, 520, 190), (40, 192, 768), (63, 768, 192), (786, 760, 760), (900, 16, 300), (2000, 24, 96),
         (6000, 320, 640), (6016, 328, 1288), (3000, 136, 1000), (4096, 264, 768), (12300, 40, 192), (16640, 200, 384),
         (33000, 16, 7), (65537, 72, 24), (66000, 64, 32), (40001, 128, 17)]


@pytest.mark.parametrize("storage", ["f16", "bf16", "f32"])
@pytest.mark.parametrize("case", GEMMS, ids=lambda c: "x".join(map(str, c)))
def test_gemm_tails_and_tilings(hip, storage, case):
    m, k, n = case
    x = stored(synth.normal(141, 1, (m, k), 1.0), storage)
    w = stored(synth.normal(141, 2, (k, n), k**-0.5), storage)
    b = synth.uniform(141, 3, (n,), -0.5, 0.5)
    r = stored(synth.normal(141, 4, (m, n), 1.0), storage)
    for act, bias, residual in (("gelu", True, False), ("none", False, True)):
        pb = PlanBuilder()
        xv, rv = pb.input((m, k), None, "x"), pb.input((m, n), None, "r")
        y = pb.gemm(xv, w, b if bias else None, act=act, name="gemm")
        y = pb.add(rv, y, name="res") if residual else y
        got, kernels = run(hip, pb.build(y), [x, r], storage)
        print(f"[gpu] {storage} {case} {kernels[0]}", flush=True)
        assert len(kernels) == 1 and "igemm" not in kernels[0], kernels
        want = O.gemm(x, w, b if bias else None, act=act)
        assert max_rel(got, want + r if residual else want) < tol(storage, k), kernels


def test_default_tilings_of_products(hip):
    """The tilings that the shapes above and some wide products take (every tiling by name: test_every_tiling)."""
    kernels = set()
    for storage in ("f16", "f32"):
        for m, k, n in GEMMS + [(8192, 768, 3072), (4096, 1024, 2000), (4096, 1024, 1000), (8192, 760, 3000),
                                (1024, 1536, 1024), (8192, 512, 512), (512, 384, 8192), (8192, 1016, 8192), (8192, 512, 1024)]:
            pb = PlanBuilder()
            y = pb.gemm(pb.input((m, k), None, "x"), np.zeros((k, n), np.float32), None, name="gemm")
            g = hip.graph(pb.build(y), storage)
            kernels.update(g.kernels)
            g.release()
    want = ["gemm_f16_256x192_w8k64s2", "gemm_f16_256x128_w8k64s2", "gemm_f16_128x64_k64s2e", "gemm_f16_64x64_k64s2",
            "gemm_kt_f16_256x128_w8k64s2", "gemm_kt_f16_64x64_k64s2",
            "gemm_kt_f16_128x96_k32s2", "gemm_f16_128x32_k64s2", "gemm_kt_f16_128x32_k32s2",
            "gemm_kt_f16_64x64_k32s2", "gemm_f32_64x64_k32s2", "conv_f32_split"]
    missing = [w for w in want if "sox_" + w not in kernels]
    assert not missing, (missing, sorted(kernels))


# (n, h, w, ic, oc, k, stride, act, residual, pad_mode)
CONVS = [(1, 7, 9, 8, 8, 1, 1, "relu", False, 0), (2, 33, 31, 24, 88, 1, 1, "none", True, 0),
         (1, 30, 41, 16, 72, 1, 1, "hardswish", False, 0), (2, 60, 60, 40, 240, 1, 1, "relu", False, 0),
         (1, 20, 20, 576, 96, 1, 1, "none", True, 0), (1, 9, 11, 40, 80, 3, 1, "relu", False, 0),
         (2, 47, 63, 96, 168, 3, 1, "hardswish", True, 0), (1, 15, 17, 72, 100, 3, 2, "none", False, 0),
         (1, 40, 40, 64, 24, 5, 1, "relu", False, 0), (2, 40, 40, 128, 256, 3, 1, "gelu", False, 0),
         (1, 31, 33, 96, 96, 3, 1, "relu", False, 1), (8, 50, 30, 48, 56, 5, 1, "none", False, 0),
         (4, 64, 64, 40, 80, 3, 1, "relu", False, 0), (8, 64, 64, 128, 128, 3, 1, "relu", False, 0),
         (1, 1, 5, 8, 9, 3, 1, "none", False, 0), (1, 12, 160, 64, 192, 1, 1, "none", False, 0),
         (1, 301, 299, 24, 32, 3, 2, "relu", False, 0), (1, 250, 203, 16, 20, 3, 1, "none", True, 0),
         (2, 160, 240, 40, 7, 5, 1, "relu", False, 1)]


@pytest.mark.parametrize("storage", ["f16", "bf16", "f32"])
@pytest.mark.parametrize("case", CONVS, ids=lambda c: "x".join(map(str, c)))
def test_conv_tails_and_tilings(hip, storage, case, monkeypatch):
    n, h, w, ic, oc, k, st, act, res, mode = case
    monkeypatch.setenv("SIMDONNX_HIP_NOHALO", "1")  # every 3x3 through the ring
    p = k // 2
    oh, ow = (h + 2 * p - k) // st + 1, (w + 2 * p - k) // st + 1
    x = stored(synth.normal(142, 1, (n, h, w, ic), 1.0), storage)
    wt = stored(synth.normal(142, 2, (oc, ic, k, k), (k * k * ic)**-0.5), storage)
    b = synth.uniform(142, 3, (oc,), -0.5, 0.5)
    r = stored(synth.normal(142, 4, (n, oh, ow, oc), 1.0), storage) if res else None
    pb = PlanBuilder()
    ins = [pb.input((n, ic, h, w), NHWC, "x")] + ([pb.input((n, oc, oh, ow), NHWC, "r")] if res else [])
    y = pb.conv(ins[0], wt, b, stride=st, pad=p, act=act, add=ins[1] if res else None, pad_mode=mode, name="conv")
    got, kernels = run(hip, pb.build(y), [x] + ([r] if res else []), storage)
    print(f"[gpu] {storage} {case} {kernels[0]}", flush=True)
    assert len(kernels) == 1 and "igemm" not in kernels[0], kernels
    want = O.conv(x, wt, b, r, stride=(st, st), pads=(p, p, p, p), act=act, pad_mode=mode, algo=1)
    assert max_rel(got, want) < tol(storage, k * k * ic), kernels


@pytest.mark.parametrize("storage", ["f16", "bf16"])
@pytest.mark.parametrize("t", [1, 16, 47, 63])
def test_fused_block_below_64_rows(hip, storage, t, monkeypatch):
    """A mixer block of one short line: attention and MLP run fused (the LayerNorms folded for them), within
    the 16-bit contract of the oracle and of the unfused dispatches."""
    from oracle.interp import run_plan
    from test_gpu_workloads import _attention_block_plan
    plan, x = _attention_block_plan(1, t, seed=143, mlp=True)
    g = hip.graph(plan, storage)
    assert [d[0] for d in g.dispatches] == ["qkv_attn", "mlp", "mlp_sum"]
    g.release()
    got, _ = run(hip, plan, [x], storage)
    monkeypatch.setenv("SIMDONNX_HIP_NO_LN_FOLD", "1")
    unfused, kernels = run(hip, plan, [x], storage)
    assert len(kernels) > 5
    want = run_plan(plan, [x], f16_storage="bf16" if storage == "bf16" else True)
    bound = 5e-3 if storage == "f16" else 2e-2
    assert max_rel(got, want) < bound and max_rel(got, unfused) < bound


def tilings():
    """Every tiling that the estimates choose from, as (storage, name): the tables' entries with cost constants."""
    src = open(os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "simdonnx_amd", "csrc", "host",
                            "backend.cpp")).read()
    names = re.findall(r'\{"(sox_(?:gemm|conv)_\w+)", \d+, \d+, \d+, \d+, [\d.]+f', src)
    assert len(names) >= 27 and len(set(names)) == len(names), names
    return [(st, n) for n in names for st in (("f32",) if "_f32_" in n else ("f16", "bf16"))] + [
        ("f32", "sox_conv_f32_split"), ("f32", "sox_conv_f32_split gemm")]


@pytest.mark.parametrize("storage,name", tilings(), ids=lambda v: v.replace("sox_", ""))
def test_every_tiling(hip, storage, name, monkeypatch):
    """Each tiling, forced, over ragged rows and columns, a K tail, a residual and more tiles than resident workgroups
    (a workgroup's ring crosses tile borders)."""
    monkeypatch.setenv("SIMDONNX_HIP_NOHALO", "1")
    kernel = name.split()[0]
    gemm = "gemm" in name
    monkeypatch.setenv("SIMDONNX_HIP_GEMM" if gemm else "SIMDONNX_HIP_CONV", kernel)
    k0 = 200 if "_kt_" in name else 100 if storage == "f32" else 128  # a slice tail where the tiling takes one
    # (rows, k, n, residual), or (batch, h, w, channels, oc, kernel, stride, residual)
    cases = [(130, k0, 200, False), (65, k0 // 2 // 4 * 4 if storage == "f32" else 72 if "_kt_" in name else 64, 97, True),
             (140001, 36 if storage == "f32" else 40 if "_kt_" in name else 64, 20, False)] if gemm else [
             (2, 47, 63, 40, 104, 3, 1, True), (1, 33, 31, 72, 77, 3, 2, False), (8, 130, 131, 8, 20, 3, 1, False)]
    for i, c in enumerate(cases):
        pb = PlanBuilder()
        if gemm:
            m, k, n, res = c
            red, xs, ys = k, (m, k), (m, n)
            x = pb.input(xs, None, "x")
            w = stored(synth.normal(147, 3 * i, (k, n), red**-0.5), storage)
        else:
            b_, h, wd, ic, n, kk, st, res = c
            p = kk // 2
            red, xs = kk * kk * ic, (b_, h, wd, ic)
            ys = (b_, (h + 2 * p - kk) // st + 1, (wd + 2 * p - kk) // st + 1, n)
            x = pb.input((b_, ic, h, wd), NHWC, "x")
            w = stored(synth.normal(147, 3 * i, (n, ic, kk, kk), red**-0.5), storage)
        xin = stored(synth.normal(147, 3 * i + 1, xs, 1.0), storage)
        r = stored(synth.normal(147, 3 * i + 2, ys, 1.0), storage) if res else None
        bias = synth.uniform(148, i, (n,), -0.5, 0.5)
        ins = [xin] + ([r] if res else [])
        if gemm:
            y = pb.gemm(x, w, bias, act="none" if res else "gelu", name="y")
            if res: y = pb.add(y, pb.input(ys, None, "r"), name="add")
            want = O.gemm(xin, w, bias, act="none" if res else "gelu")
            want = want + r if res else want
        else:
            rv = pb.input((ys[0], ys[3], ys[1], ys[2]), NHWC, "r") if res else None
            y = pb.conv(x, w, bias, stride=st, pad=p, act="hardswish", add=rv, name="y")
            want = O.conv(xin, w, bias, r, stride=(st, st), pads=(p, p, p, p), act="hardswish", algo=1)
        got, kernels = run(hip, pb.build(y), ins, storage)
        err = max_rel(got, want)
        print(f"[gpu] {storage} {name} {c} {err:.2e} of {tol(storage, red):.2e}", flush=True)
        assert kernels == [kernel.replace("_f16_", f"_{storage}_")], (c, kernels)
        assert err < tol(storage, red), c


# (batch, h, w, ic, oc, act, residual, concat): both register kernels and the LDS one, tile edges, a last channel
# block of 8 .. 32 channels, one and two blocks of output channels, fewer tiles than XCDs, several tiles a workgroup
HALOS = [(1, 8, 16, 8, 8, "relu", False, False), (1, 9, 17, 32, 40, "hardswish", True, False), (3, 50, 70, 24, 64, "gelu", False, True),
         (1, 1, 1, 16, 16, "none", True, False), (2, 300, 310, 16, 24, "none", True, False), (1, 200, 333, 32, 64, "none", False, False),
         (1, 260, 270, 40, 64, "relu", True, False), (2, 250, 200, 64, 32, "hardswish", False, False),
         (1, 320, 330, 56, 24, "none", False, True), (1, 40, 40, 64, 32, "relu", False, False), (1, 21, 33, 32, 12, "none", False, False)]


@pytest.mark.parametrize("storage", ["f16", "bf16"])
@pytest.mark.parametrize("case", HALOS, ids=lambda c: "x".join(str(v) for v in c))
def test_halo_filter_in_registers(hip, storage, case):
    n, h, w, ic, oc, act, res, cat = case
    x = stored(synth.normal(144, 1, (n, h, w, ic), 1.0), storage)
    wt = stored(synth.normal(144, 2, (oc, ic, 3, 3), (9 * ic)**-0.5), storage)
    b = synth.uniform(144, 3, (oc,), -0.5, 0.5)
    r = stored(synth.normal(144, 4, (n, h, w, oc), 1.0), storage)
    pb = PlanBuilder()
    ins = [pb.input((n, ic, h, w), NHWC, "x")] + ([pb.input((n, oc, h, w), NHWC, "r")] if res else [])
    y = pb.conv(ins[0], wt, b, stride=1, pad=1, act=act, add=ins[1] if res else None, name="conv")
    if cat:  # the second half of a concat
        y = pb.concat_channels([pb.conv(ins[0], wt, b, stride=1, pad=1, name="first"), y])
    got, kernels = run(hip, pb.build(y), [x] + ([r] if res else []), storage)
    tiles = n * -(-h // 8) * -(-w // 16) * -(-oc // 32)
    want_k = "3x3s1" if oc % 8 or (ic > 32 and tiles < 768) else "3x3s1_c32" if ic <= 32 else "3x3s1_c64"
    assert kernels[-1] == f"sox_conv_halo_{storage}_{want_k}", kernels
    want = O.conv(x, wt, b, r if res else None, stride=(1, 1), pads=(1, 1, 1, 1), act=act)
    if cat: want = np.concatenate([O.conv(x, wt, b, None, stride=(1, 1), pads=(1, 1, 1, 1), act="none"), want], axis=-1)
    assert max_rel(got, want) < tol(storage, 9 * ic), kernels


ODD_GEMMS = [(1, 9, 1), (5, 17, 3), (64, 65, 64), (33, 33, 130), (130, 1001, 97), (700, 255, 255), (2000, 30, 90), (3000, 127, 20)]


@pytest.mark.parametrize("storage", ["f16", "bf16", "f32"])
@pytest.mark.parametrize("case", ODD_GEMMS, ids=lambda c: "x".join(map(str, c)))
def test_gemm_rows_padded_to_chunks(hip, storage, case):
    """K that is no whole 16-byte chunk: the rows are padded into scratch first, from `short` on."""
    m, k, n = case
    x = stored(synth.normal(145, 1, (m, k), 1.0), storage)
    w = stored(synth.normal(145, 2, (k, n), k**-0.5), storage)
    b = synth.uniform(145, 3, (n,), -0.5, 0.5)
    pb = PlanBuilder()
    got, kernels = run(hip, pb.build(pb.gemm(pb.input((m, k), None, "x"), w, b, act="gelu", name="gemm")), [x], storage)
    short, ld = (32, 4) if storage == "f32" else (16, 8)
    assert ("padc" in kernels[0]) == (k >= short and k % ld != 0), kernels
    assert max_rel(got, O.gemm(x, w, b, act="gelu")) < tol(storage, k), kernels


ODD_CONVS = [(1, 7, 9, 9, 5, 3, 1, "relu", False, 0), (2, 16, 16, 17, 17, 3, 1, "none", True, 0), (1, 40, 30, 33, 64, 3, 2, "gelu", False, 0),
             (1, 25, 31, 129, 60, 1, 1, "relu", True, 0), (2, 50, 40, 31, 45, 5, 1, "hardswish", False, 1),
             (1, 20, 20, 250, 250, 3, 1, "none", False, 0), (1, 60, 60, 11, 3, 3, 1, "relu", False, 0), (1, 30, 30, 7, 20, 3, 1, "none", False, 0),
             (1, 33, 20, 50, 41, 1, 2, "none", False, 0), (1, 20, 20, 63, 64, 3, 1, "relu", False, 0), (2, 10, 13, 15, 16, 3, 1, "none", True, 0)]


@pytest.mark.parametrize("storage", ["f16", "bf16", "f32"])
@pytest.mark.parametrize("case", ODD_CONVS, ids=lambda c: "x".join(map(str, c)))
def test_conv_channels_padded_to_chunks(hip, storage, case):
    n, h, w, ic, oc, k, st, act, res, mode = case
    p = k // 2
    oh, ow = (h + 2 * p - k) // st + 1, (w + 2 * p - k) // st + 1
    x = stored(synth.normal(146, 1, (n, h, w, ic), 1.0), storage)
    wt = stored(synth.normal(146, 2, (oc, ic, k, k), (k * k * ic)**-0.5), storage)
    b = synth.uniform(146, 3, (oc,), -0.5, 0.5)
    r = stored(synth.normal(146, 4, (n, oh, ow, oc), 1.0), storage) if res else None
    pb = PlanBuilder()
    ins = [pb.input((n, ic, h, w), NHWC, "x")] + ([pb.input((n, oc, oh, ow), NHWC, "r")] if res else [])
    y = pb.conv(ins[0], wt, b, stride=st, pad=p, act=act, add=ins[1] if res else None, pad_mode=mode, name="conv")
    got, kernels = run(hip, pb.build(y), [x] + ([r] if res else []), storage)
    ld = 4 if storage == "f32" else 8
    assert ("padc" in kernels[0]) == (ic % ld != 0 and ic >= 9), kernels
    want = O.conv(x, wt, b, r, stride=(st, st), pads=(p, p, p, p), act=act, pad_mode=mode, algo=1)
    assert max_rel(got, want) < tol(storage, k * k * ic), kernels


@pytest.mark.parametrize("storage", ["f16", "bf16", "f32"])
@pytest.mark.parametrize("case", [(8001, 24, 301, "gelu", False), (20000, 16, 61, "none", True), (1500, 40, 1142, "relu", True)],
                         ids=lambda c: "x".join(map(str, c[:3])))
def test_ragged_products_on_the_implicit_gemm(hip, storage, case, monkeypatch):
    """Products that the rule takes off the ring for their ragged rows, with and without a residual and a bias."""
    monkeypatch.delenv("SIMDONNX_HIP_RING")
    m, k, n, act, res = case
    x, w = stored(synth.normal(149, 1, (m, k), 1.0), storage), stored(synth.normal(149, 2, (k, n), k**-0.5), storage)
    b, r = None if res else synth.uniform(149, 3, (n,), -0.5, 0.5), stored(synth.normal(149, 4, (m, n), 1.0), storage)
    pb = PlanBuilder()
    xv, rv = pb.input((m, k), None, "x"), pb.input((m, n), None, "r")
    y = pb.gemm(xv, w, b, act="none" if res else act, name="gemm")
    got, kernels = run(hip, pb.build(pb.add(y, rv, act=act, name="add") if res else y), [x, r], storage)
    assert len(kernels) == 1 and "igemm" in kernels[0], kernels
    want = O.gemm(x, w, b, act="none" if res else act)
    if res: want = np.maximum(want + r, 0) if act == "relu" else want + r
    assert max_rel(got, want) < tol(storage, k), kernels


# (n, h, w, ic, oc, k, stride, act, residual, pad_mode, concat): few channels, ragged rows, a concat's pitch
@pytest.mark.parametrize("case", [(1, 20, 20, 4, 8, 3, 1, "relu", False, 0, False), (1, 64, 139, 4, 62, 5, 1, "gelu", True, 1, False),
                                  (2, 39, 79, 8, 262, 3, 1, "hardswish", True, 0, False), (3, 77, 101, 4, 40, 3, 2, "none", False, 1, False),
                                  (1, 128, 150, 4, 64, 3, 1, "relu", False, 0, True)], ids=lambda c: "x".join(map(str, c)))
def test_fp32_convs_on_the_implicit_gemm(hip, case, monkeypatch):
    """fp32 convs that the rule takes off the ring."""
    monkeypatch.delenv("SIMDONNX_HIP_RING")
    n, h, w, ic, oc, k, st, act, res, mode, cat = case
    p = k // 2
    oh, ow = (h + 2 * p - k) // st + 1, (w + 2 * p - k) // st + 1
    x, wt = synth.normal(150, 1, (n, h, w, ic), 1.0), synth.normal(150, 2, (oc, ic, k, k), (k * k * ic)**-0.5)
    b, r = synth.uniform(150, 3, (oc,), -0.5, 0.5), synth.normal(150, 4, (n, oh, ow, oc), 1.0) if res else None
    pb = PlanBuilder()
    ins = [pb.input((n, ic, h, w), NHWC, "x")] + ([pb.input((n, oc, oh, ow), NHWC, "r")] if res else [])
    y = pb.conv(ins[0], wt, b, stride=st, pad=p, act=act, add=ins[1] if res else None, pad_mode=mode, name="conv")
    if cat: y = pb.concat_channels([pb.conv(ins[0], wt[:8], b[:8], stride=st, pad=p, name="first"), y])
    got, kernels = run(hip, pb.build(y), [x] + ([r] if res else []), "f32")
    assert "igemm" in kernels[-1], kernels
    want = O.conv(x, wt, b, r, stride=(st, st), pads=(p, p, p, p), act=act, pad_mode=mode, algo=1)
    if cat: want = np.concatenate([O.conv(x, wt[:8], b[:8], stride=(1, 1), pads=(1, 1, 1, 1), act="none", algo=1), want], axis=-1)
    assert max_rel(got, want) < tol("f32", k * k * ic), kernels


NAN_GEMMS = [(5, 8, 24), (33, 40, 104), (7, 96, 219), (951, 248, 93), (300, 128, 200), (4, 39, 154), (4100, 192, 776), (16400, 64, 24)]


@pytest.mark.parametrize("storage", ["f16", "bf16", "f32"])
def test_gelu_keeps_nan(hip, storage, monkeypatch):
    """A NaN reaches the outputs that depend on it, and only those, through every kernel's GELU: dense products, convs
    (ring, halo) and the MLP of few and many rows."""
    for m, k, n in NAN_GEMMS:
        x = stored(synth.normal(151, 1, (m, k), 1.0), storage)
        x[m // 2, k // 3] = np.nan
        pb = PlanBuilder()
        y = pb.gemm(pb.input((m, k), None, "x"), synth.normal(151, 2, (k, n), k**-0.5), None, act="gelu", name="gemm")
        got, kernels = run(hip, pb.build(y), [x], storage)
        nan = np.isnan(got.reshape(m, n))
        assert nan[m // 2].all() and nan.sum() == n, (m, k, n, kernels)
    for h, w, ic, oc, k in ((19, 33, 24, 40, 3), (40, 50, 96, 100, 3), (30, 30, 64, 256, 3), (21, 20, 16, 72, 1), (20, 20, 16, 24, 5)):
        x = synth.normal(151, 3, (1, h, w, ic), 1.0)
        x[0, 9, 11, ic // 2] = np.nan
        wt = synth.normal(151, 4, (oc, ic, k, k), (k * k * ic)**-0.5)
        for nohalo in (False, True):
            monkeypatch.setenv("SIMDONNX_HIP_NOHALO", "1") if nohalo else monkeypatch.delenv("SIMDONNX_HIP_NOHALO", raising=False)
            pb = PlanBuilder()
            y = pb.conv(pb.input((1, ic, h, w), NHWC, "x"), wt, None, pad=k // 2, act="gelu", name="conv")
            got, kernels = run(hip, pb.build(y), [x], storage)
            assert np.array_equal(np.isnan(got), np.isnan(O.conv(x, wt, None, pads=(k // 2,) * 4, act="gelu", algo=1))), kernels
    for rows in (3, 63, 200):
        x = synth.normal(151, 5, (1, rows, 192), 1.0)
        x[0, rows // 2, 7] = np.nan
        pb = PlanBuilder()
        h = pb.layer_norm(pb.input((1, rows, 192), None, "x"), np.ones(192, np.float32), np.zeros(192, np.float32), 1e-6, name="ln")
        h = pb.gemm(h, synth.normal(151, 6, (192, 768), 0.05), np.zeros(768, np.float32), act="gelu", name="fc1")
        got, kernels = run(hip, pb.build(pb.gemm(h, synth.normal(151, 7, (768, 192), 0.05), np.zeros(192, np.float32), name="fc2")), [x], storage)
        nan = np.isnan(got.reshape(rows, 192))
        assert nan[rows // 2].all() and nan.sum() == 192, (rows, kernels)
