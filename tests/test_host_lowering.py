"""The host lowering on the CPU, with no device: every workload plan goes through graph creation on a
backend built by sox_backend_create_offline (the graph-creation rewrites, the arena moves, const
packing, the kernel choice against the embedded code objects' symbol tables), and the result is
checked for what can be checked without running it:
  - every dispatch's kernel exists in the embedded code objects, and every arena / const binding lies
    inside the slab / the const store;
  - a rewritten output moved to a buffer of its own takes its zero-copy views along (Engine/ExecPlan.cs:
    207, 211; Backends/Vulkan/VkGraph.cs:365-367), and the node reading the view binds the new place.
The same file then runs again in a child process against the host-sanitizer build of the library
(AddressSanitizer + UndefinedBehaviorSanitizer, simdonnx_amd.build.build_sanitized_backend), the HIP
counterpart of the reference's validation-layer mode (Backends/Vulkan/VkDevice.cs:176).
"""
import functools
import os
import subprocess
import sys

import pytest

from simdonnx_amd import graphs
from simdonnx_amd import native as N
from simdonnx_amd.backend import HipBackend
from tests import relocation_cases as RC

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
STORAGES = ["f32", "f16", "bf16"]


@functools.lru_cache(maxsize=None)
def _workload(name):
    return {
        "conv3x3": graphs.conv3x3_bias_relu,
        "matmul_gelu": graphs.matmul_bias_gelu,
        "mobilenetv3": graphs.mobilenetv3_small,
        "dbnet": graphs.dbnet,
        "svtr": graphs.svtr,
        "svtr_features": lambda: graphs.svtr(head="features")[:2],
    }[name]()[0]


@pytest.fixture(scope="module")
def offline():
    b = HipBackend.offline()
    yield b
    b.close()


def _check_binds(g):
    arena, consts, sync = g.arena_bytes, g.const_bytes, g.sync_bytes
    for i in range(len(g.dispatches)):
        for slot, off, size in g.binds(i):
            if slot == N.SLOT_ARENA:
                assert off + size <= arena, (i, g.kernels[i], off, size, arena)
            elif slot == N.SLOT_CONSTS:
                assert off + size <= consts, (i, g.kernels[i], off, size, consts)
            elif slot == N.SLOT_SYNC:
                assert off + size <= sync, (i, g.kernels[i], off, size, sync)
            else:
                assert slot == N.SLOT_DUMMY, (i, g.kernels[i], slot)


def test_sanitizer_build_is_the_one_loaded_when_asked():
    """Under SIMDONNX_HIP_BACKEND_LIB (the child run below) the sanitizer build and its runtime are
    the ones mapped into the process."""
    want = os.environ.get("SIMDONNX_HIP_BACKEND_LIB")
    if not want:
        pytest.skip("runs in the sanitizer child process")
    N.backend()
    maps = open("/proc/self/maps").read()
    assert os.path.realpath(want) in maps
    assert "libclang_rt.asan" in maps


@pytest.mark.parametrize("storage", STORAGES)
@pytest.mark.parametrize("name", ["conv3x3", "matmul_gelu", "mobilenetv3", "dbnet", "svtr", "svtr_features"])
def test_workload_lowers_without_device(offline, name, storage):
    g = offline.graph(_workload(name), storage)
    try:
        kernels = g.kernels
        assert kernels and all(k.startswith("sox_") for k in kernels)
        _check_binds(g)
    finally:
        g.release()


@pytest.mark.parametrize("storage", STORAGES)
@pytest.mark.parametrize("name", ["mobilenetv3", "dbnet"])
def test_se_in_depthwise_lowers_without_device(offline, name, storage, monkeypatch):
    """Under SIMDONNX_HIP_SE_IN_DW every SE gate of the convnets runs in its depthwise conv's launch:
    nine depthwise_se dispatches, no gap_part / se_gate, each with its own counters in the session's
    counter block (33 dispatches for MobileNetV3-small, 44 for the fp16 / bf16 detector)."""
    monkeypatch.setenv("SIMDONNX_HIP_SE_IN_DW", "1")
    g = offline.graph(_workload(name), storage)
    try:
        labels = [d[0] for d in g.dispatches]
        assert labels.count("depthwise_se") == 9 and "se_gate" not in labels and "gap_part" not in labels, labels
        if storage != "f32":
            assert len(labels) == {"mobilenetv3": 33, "dbnet": 43}[name], labels
        _check_binds(g)
        syncs = [(off, size) for i in range(len(labels)) for slot, off, size in g.binds(i) if slot == N.SLOT_SYNC]
        assert len(syncs) == 9 and len({off for off, _ in syncs}) == 9
        assert sum(size for _, size in syncs) <= g.sync_bytes
    finally:
        g.release()


def test_offline_backend_refuses_device_work(offline):
    from simdonnx_amd.backend import HipInferenceSession
    g = offline.graph(_workload("conv3x3"), "f16")
    try:
        with pytest.raises(N.NotSupportedError):
            HipInferenceSession(g)
        with pytest.raises(N.NotSupportedError):
            offline.create_buffer_pool()
    finally:
        g.release()


@pytest.mark.parametrize("storage", STORAGES)
@pytest.mark.parametrize("case", list(RC.CASES))
def test_relocated_output_keeps_its_views(offline, case, storage, monkeypatch):
    c = RC.CASES[case]()
    if storage not in c.storages:
        pytest.skip(f"the rewrite is not taken on {storage} graphs")
    p = RC.forced(c)
    assert RC.overlaps(p, c.moved, c.over) and not RC.conflicts(p)
    es = 4 if storage == "f32" else 2
    g = offline.graph(p, storage)
    monkeypatch.setenv(c.switch, "1")
    g_off = offline.graph(p, storage)
    try:
        labels, labels_off = [d[0] for d in g.dispatches], [d[0] for d in g_off.dispatches]
        assert len(labels) < len(labels_off) or (c.fused_label in labels and c.fused_label not in labels_off), \
            f"the rewrite was not taken: {labels} / {labels_off}"
        _check_binds(g)
        place = g.value_place(c.moved)
        assert g.value_place(c.view)[0] == place[0], "the view stayed behind"
        assert place[0] != p.buf_offset[p.values[c.moved].buf] * es, "the output was not moved"
        assert place[0] >= p.arena_floats * es, "the new place is past the planned activations"
        # the unfused graph keeps the planned place
        assert g_off.value_place(c.moved)[0] == p.buf_offset[p.values[c.moved].buf] * es
        reader = next(k for k, n in enumerate(p.nodes) if c.view in n.ins)
        binds = [b for i, d in enumerate(g.dispatches) if d[2] == reader for b in g.binds(i)]
        assert (N.SLOT_ARENA, place[0]) in [(s, o) for s, o, _ in binds], binds
    finally:
        g.release()
        g_off.release()


def test_host_lowering_under_sanitizers():
    """This file's other tests again, in a child process that loads the ASan + UBSan build of the
    backend library; any sanitizer report fails the child."""
    if os.environ.get("SIMDONNX_HIP_BACKEND_LIB"):
        pytest.skip("already the sanitizer child")
    from simdonnx_amd import build as B
    rt = B.sanitizer_runtime()
    if not rt:
        pytest.skip("the host compiler has no shared AddressSanitizer runtime")
    src = os.path.join(B.HDIR, "backend.cpp")
    if not os.path.exists(B.SAN_BACKEND) or os.path.getmtime(B.SAN_BACKEND) < os.path.getmtime(src):
        B.build_sanitized_backend()
    env = dict(os.environ)
    env["LD_PRELOAD"] = rt + (":" + env["LD_PRELOAD"] if env.get("LD_PRELOAD") else "")
    env["ASAN_OPTIONS"] = "detect_leaks=0:halt_on_error=1"
    env["UBSAN_OPTIONS"] = "halt_on_error=1:print_stacktrace=1"
    env["SIMDONNX_HIP_BACKEND_LIB"] = B.SAN_BACKEND
    r = subprocess.run([sys.executable, "-m", "pytest", "-q", "-x", "-p", "no:cacheprovider", os.path.abspath(__file__),
                        "-k", "not under_sanitizers"], cwd=ROOT, env=env, capture_output=True, text=True, timeout=1200)
    out = r.stdout + r.stderr
    assert r.returncode == 0, out[-6000:]
    for marker in ("AddressSanitizer", "runtime error:", "LeakSanitizer"):
        assert marker not in out, out[-6000:]


@pytest.mark.parametrize("storage", ["f16", "bf16"])
def test_upsample_add_input_survives_fused_writes(offline, storage):
    """plan_upsample_add runs the lateral conv at the Add's place, so its input must survive what the
    dispatches in between write, including outputs written by a fused dispatch for a folded node (the
    transformer MLP writes fc2's output from fc1's place): an fc2 output planned over the conv's input
    moves to a buffer of its own (tests/relocation_cases.py: upsample_add_after_fused_write)."""
    plan, ins, xi, f2, up = RC.upsample_add_after_fused_write()
    p = RC.place_over(plan, f2, xi)
    assert RC.overlaps(p, f2, xi) and not RC.conflicts(p)
    g = offline.graph(p, storage)
    try:
        labels = [d[0] for d in g.dispatches]
        assert "mlp" in labels and "nearest" not in labels and labels[-1] == "conv", labels
        _check_binds(g)
        (xo, xb), (fo, fb) = g.value_place(xi), g.value_place(f2)
        assert fo + fb <= xo or xo + xb <= fo, "the fused MLP writes over the lateral conv's input"
        conv = len(labels) - 1
        assert (N.SLOT_ARENA, xo) in [(s, o) for s, o, _ in g.binds(conv)]
    finally:
        g.release()


def _conv3x3_256(n, h, w, stride=1):
    import numpy as np
    from simdonnx_amd.plan import NHWC, PlanBuilder
    pb = PlanBuilder()
    x = pb.input((n, 256, h, w), NHWC, "x")
    y = pb.conv(x, np.zeros((256, 256, 3, 3), np.float32), np.zeros(256, np.float32), stride=stride, pad=1, act="relu",
                name="c")
    return pb.build(y)


def test_large_conv_takes_the_halo_tile(offline, monkeypatch):
    """A large 3x3 stride-1 conv over 256 channels takes the halo tile (sox_conv_*_h256), also with a
    partial last tile per row (264 = 8.25 tiles of 32 pixels), and the ring under SIMDONNX_HIP_NO_H256;
    forcing the halo tile onto a conv it does not take (stride 2) is refused at graph creation."""
    for storage in ("f16", "bf16"):
        for w in (256, 264):
            g = offline.graph(_conv3x3_256(2, 256, w), storage)
            assert g.kernels == [f"sox_conv_{storage}_h256"], g.kernels
            g.release()
    monkeypatch.setenv("SIMDONNX_HIP_NO_H256", "1")
    g = offline.graph(_conv3x3_256(2, 256, 256), "f16")
    assert g.kernels == ["sox_conv_f16_256x256_w8k64s2"], g.kernels
    g.release()
    monkeypatch.delenv("SIMDONNX_HIP_NO_H256")
    monkeypatch.setenv("SIMDONNX_HIP_CONV", "sox_conv_f16_h256")
    with pytest.raises(N.NotSupportedError):
        offline.graph(_conv3x3_256(2, 256, 256, stride=2), "f16")


def test_large_conv_tile_takes_inputs_under_2_pow_31_elements(offline, monkeypatch):
    """The 256x256 conv tile keeps one 32-bit offset into the whole input per DMA row: a large conv takes
    it below 2^31 input elements and the 256x128 tile (64-bit image bases) from there; forcing the
    256x256 tile onto a larger input is refused at graph creation, not run."""
    monkeypatch.setenv("SIMDONNX_HIP_NO_H256", "1")  # the ring's choice
    g = offline.graph(_conv3x3_256(2, 256, 256), "f16")
    assert g.kernels == ["sox_conv_f16_256x256_w8k64s2"], g.kernels
    g.release()
    big = _conv3x3_256(1, 1024, 8448)  # 2^31 + 2^26 input elements
    g = offline.graph(big, "f16")
    assert g.kernels == ["sox_conv_f16_256x128_w8k64s2"], g.kernels
    g.release()
    monkeypatch.setenv("SIMDONNX_HIP_CONV", "sox_conv_f16_256x256_w8k64s2")
    with pytest.raises(N.NotSupportedError):
        offline.graph(big, "f16")


def test_gemm_pp_takes_16_bit_graphs_only(offline, monkeypatch):
    """SIMDONNX_HIP_GEMMPP opts 16-bit Gemms of whole 256x128 tiles with K = 768 into sox_gemmpp_*, whose kernels
    read 16-bit operands: the same fp32 Gemm stays on the fp32 kernels."""
    import numpy as np
    from simdonnx_amd.plan import PlanBuilder
    monkeypatch.setenv("SIMDONNX_HIP_GEMMPP", "1")
    pb = PlanBuilder()
    y = pb.gemm(pb.input((8192, 768), None, "a"), np.zeros((768, 1024), np.float32), None, act="gelu", name="gemm")
    plan = pb.build(y)
    for storage in STORAGES:
        g = offline.graph(plan, storage)
        kernels = g.kernels
        g.release()
        if storage == "f32":
            assert all("gemmpp" not in k and "f32" in k for k in kernels), kernels
        else:
            assert kernels == [f"sox_gemmpp_{storage}_256x128_k768_gelu"], kernels


@pytest.mark.parametrize("storage", ["f16", "bf16"])
@pytest.mark.parametrize("rows", [16, 128])
@pytest.mark.parametrize("gamma", [1.0, 1e-2, 3e-3, 1e-3, 4e6])
def test_layernorm_folds_where_its_weights_keep_their_precision(offline, gamma, rows, storage):
    """LayerNorm -> fc1 + GELU -> fc2 folds the gamma into fc1's weights. With weights of 0.02, gamma 3e-3 or 1e-3 takes
    most of them below fp16's normal range and 4e6 past its largest value: such a LayerNorm stays a node of its own
    (bf16 has fp32's range and folds)."""
    import numpy as np
    from simdonnx_amd import synth
    from simdonnx_amd.plan import PlanBuilder
    pb = PlanBuilder()
    x = pb.input((1, rows, 192), None, "x")
    h = pb.layer_norm(x, np.full(192, gamma, np.float32), np.zeros(192, np.float32), 1e-6, name="ln")
    h = pb.gemm(h, synth.normal(5, 1, (192, 768), 0.02), np.zeros(768, np.float32), act="gelu", name="fc1")
    y = pb.gemm(h, synth.normal(5, 2, (768, 192), 0.02), np.zeros(192, np.float32), name="fc2")
    g = offline.graph(pb.build(y), storage)
    labels = [d[0] for d in g.dispatches]
    g.release()
    folds = storage == "bf16" or gamma in (1.0, 1e-2)
    assert labels[0] == ("mlp" if folds else "layernorm"), labels


@pytest.mark.parametrize("storage", STORAGES)
def test_padded_rows_can_be_refused(offline, storage, monkeypatch):
    """Rows of odd channel counts are copied to padded ones in the arena; SIMDONNX_HIP_NO_PAD_ROWS keeps the arena
    to the plan's activations and leaves the other kernels as they are."""
    import numpy as np
    from simdonnx_amd.plan import NHWC, PlanBuilder
    pb = PlanBuilder()
    x = pb.input((1, 65, 128, 128), NHWC, "x")
    h = pb.conv(x, np.zeros((129, 65, 3, 3), np.float32), np.zeros(129, np.float32), pad=1, name="odd")
    y = pb.conv(h, np.zeros((64, 129, 1, 1), np.float32), np.zeros(64, np.float32), name="odd1")
    y = pb.conv(y, np.zeros((64, 64, 1, 1), np.float32), np.zeros(64, np.float32), name="even")
    plan = pb.build(y)
    g = offline.graph(plan, storage)
    kernels, arena = g.kernels, g.arena_bytes
    _check_binds(g)
    g.release()
    monkeypatch.setenv("SIMDONNX_HIP_NO_PAD_ROWS", "1")
    g = offline.graph(plan, storage)
    plain, plain_arena = g.kernels, g.arena_bytes
    _check_binds(g)
    g.release()
    assert sum("padc" in k for k in kernels) == 2 and not any("padc" in k for k in plain)
    assert plain[-1] == kernels[-1] and ["igemm" in k for k in plain] == [True, True, False], plain
    es = 4 if storage == "f32" else 2
    assert plain_arena <= (plan.arena_floats * es + 255) // 256 * 256 < arena


def _conv_kernel(offline, storage, n, h, w, ic, oc, k, stride):
    import numpy as np
    from simdonnx_amd.plan import NHWC, PlanBuilder
    pb = PlanBuilder()
    x = pb.input((n, ic, h, w), NHWC, "x")
    y = pb.conv(x, np.zeros((oc, ic, k, k), np.float32), np.zeros(oc, np.float32), stride=stride, pad=k // 2, name="c")
    g = offline.graph(pb.build(y), storage)
    kernels = g.kernels
    g.release()
    assert len(kernels) == 1, kernels
    return kernels[0]


@pytest.mark.parametrize("storage", ["f16", "bf16"])
def test_many_taps_of_few_channels_take_the_wide_shallow_tile(offline, storage):
    """5x5 convs over at most 32 channels of large maps: 128x128 tiles with 32-deep slices, 40 us where the 64x64 tile
    takes 55; few channels on small maps stay on the small tiles."""
    for ic in (8, 24, 32):
        assert _conv_kernel(offline, storage, 8, 93, 91, ic, 112, 5, 1) == f"sox_conv_{storage}_128x128_k32s4"
        assert _conv_kernel(offline, storage, 1, 20, 20, ic, 112, 5, 1) == f"sox_conv_{storage}_64x64_k32s4"


def _gemm_kernel(offline, storage, m, k, n):
    import numpy as np
    from simdonnx_amd.plan import PlanBuilder
    pb = PlanBuilder()
    g = offline.graph(pb.build(pb.gemm(pb.input((m, k), None, "a"), np.zeros((k, n), np.float32), None, name="gemm")), storage)
    kernels = g.kernels
    g.release()
    assert len(kernels) == 1, kernels
    return kernels[0]


@pytest.mark.parametrize("storage", STORAGES)
def test_ragged_rows_take_the_implicit_gemm_where_it_is_faster(offline, storage, monkeypatch):
    """Products whose rows are not whole 4-element groups: many outputs over a short reduction go to the implicit GEMM
    (the ring stores them as single elements), few outputs, long reductions and whole groups to the ring."""
    for shape in ((20000, 16, 1142), (8000, 24, 301), (1500, 40, 5058)):
        assert "igemm" in _gemm_kernel(offline, storage, *shape), shape
    for shape in ((20000, 16, 1144), (512, 320, 301), (20000, 768, 301), (4096, 768, 3072), (130, 200, 200)):
        assert "igemm" not in _gemm_kernel(offline, storage, *shape), shape
    monkeypatch.setenv("SIMDONNX_HIP_RING", "1")
    assert "igemm" not in _gemm_kernel(offline, storage, 20000, 16, 1142)


def test_fp32_convs_of_few_channels_take_the_implicit_gemm(offline):
    """fp32 convs over 4 or 8 channels: the implicit GEMM packs their taps where the ring's slices are mostly zeros;
    from 64 channels on the ring, as do few output tiles from 8 channels on."""
    for shape in ((1, 128, 277, 4, 366, 5, 1), (1, 20, 20, 4, 8, 3, 1), (4, 250, 16, 8, 344, 3, 1), (1, 223, 150, 8, 408, 2, 1)):
        assert "igemm" in _conv_kernel(offline, "f32", *shape), shape
    for shape in ((1, 20, 20, 8, 64, 3, 1), (1, 40, 40, 40, 64, 3, 1), (4, 64, 64, 128, 128, 3, 1), (1, 160, 160, 96, 24, 3, 1)):
        assert "igemm" not in _conv_kernel(offline, "f32", *shape), shape


@pytest.mark.parametrize("storage", ["f16", "bf16"])
def test_narrow_tile_is_for_many_rows(offline, storage):
    """The 128x32 tile takes products of at most 32 columns over many rows; few rows take 64x64, which costs less."""
    for k, kt in ((24, f"sox_gemm_kt_{storage}_128x32_k32s2"), (128, f"sox_gemm_{storage}_128x32_k64s2")):
        for n in (8, 24, 32):
            assert _gemm_kernel(offline, storage, 66000, k, n) == kt
            for m in (1, 8, 47):
                assert "_64x64_" in _gemm_kernel(offline, storage, m, k, n), (m, k, n)


# a shape that takes each tiling by the estimate, at 256 CUs: (rows, k, n), or (batch, h, w, channels, oc, kernel, stride)
TILING_SHAPES = {
    "sox_gemm_f16_256x192_w8k64s2": (8192, 768, 3072), "sox_gemm_f16_256x128_w8k64s2": (21124, 64, 280),
    "sox_gemm_f16_128x128_k64s2": (19893, 3072, 1352), "sox_gemm_f16_128x64_k64s2e": (25612, 64, 68),
    "sox_gemm_f16_64x64_k64s2": (1, 64, 15), "sox_gemm_f16_128x32_k64s2": (18889, 128, 10),
    "sox_gemm_kt_f16_256x128_w8k64s2": (3769, 8, 1988), "sox_gemm_kt_f16_128x128_k64s2": (1264, 408, 3042),
    "sox_gemm_kt_f16_128x64_k64s2": (19563, 136, 296), "sox_gemm_kt_f16_64x64_k64s2": (2, 232, 9),
    "sox_gemm_kt_f16_128x96_k32s2": (6202, 8, 908), "sox_gemm_kt_f16_64x64_k32s2": (1, 8, 8),
    "sox_gemm_kt_f16_128x32_k32s2": (23362, 8, 12), "sox_gemm_f32_128x64_k32s2": (8192, 512, 1024),
    "sox_gemm_f32_64x64_k32s2": (786, 760, 760), "sox_gemm_f32_128x32_k32s2": (12300, 40, 192),
    "sox_conv_f32_split": (40, 192, 768), "sox_conv_f16_128x128_k64s2": (8, 64, 64, 128, 256, 3, 1),
    "sox_conv_f16_128x128_k32s4": (8, 93, 91, 24, 112, 5, 1), "sox_conv_f16_128x96_k64s2": (2, 160, 160, 40, 80, 3, 1),
    "sox_conv_f16_128x96_k32s2": (2, 95, 127, 96, 168, 3, 1), "sox_conv_f16_128x64_k64s2": (1, 184, 190, 40, 35, 3, 1),
    "sox_conv_f16_64x64_k64s4": (1, 6, 4, 48, 15, 3, 2), "sox_conv_f16_64x64_k32s4": (1, 5, 5, 8, 15, 3, 1),
    "sox_conv_f16_128x32_k32s2": (4, 47, 137, 8, 9, 3, 1), "sox_conv_f32_128x64_k32s2": (8, 35, 54, 56, 223, 3, 1),
    "sox_conv_f32_64x64_k32s4": (4, 6, 100, 24, 268, 3, 1), "sox_conv_f32_128x32_k32s2": (2, 147, 96, 32, 9, 3, 1)}


def test_every_tiling_of_the_estimate_is_taken_by_some_shape(offline, monkeypatch):
    """No table entry is out of the estimate's reach, and the numeric tests' list of tilings (test_gpu_ring.tilings, read
    from the tables) is the list of these shapes."""
    from tests.test_gpu_ring import tilings
    assert {n.split()[0] for _, n in tilings()} == set(TILING_SHAPES)
    monkeypatch.setenv("SIMDONNX_HIP_NOHALO", "1")
    for name, shape in TILING_SHAPES.items():
        for storage in ("f32",) if "_f32_" in name else ("f16", "bf16"):
            got = _gemm_kernel(offline, storage, *shape) if len(shape) == 3 else _conv_kernel(offline, storage, *shape)
            assert got == name.replace("_f16_", f"_{storage}_"), (name, shape, got)
