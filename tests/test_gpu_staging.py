"""The staging kernels (staging.hip): a session's fp32 windows read and written in place, through a plan
that only copies. Counts at the edges of a vector, of a workgroup's pass and of the grid, arena offsets
that are not aligned to a vector, and an output large enough for the copy engine. The result is the
input rounded to the storage type to nearest even, exactly."""
import numpy as np
import pytest

from oracle.interp import _bf16
from simdonnx_amd.backend import HipInferenceSession, HipUnitRunner
from simdonnx_amd.plan import PlanBuilder

pytestmark = pytest.mark.gpu

COUNTS = [1, 3, 4, 5, 2047, 2049, 64 * 2048 - 1, 64 * 2048 + 2053, 256 * 4096 + 4099]


def copy_plan(count, shift=0):
    pb = PlanBuilder()
    y = pb.unary("Copy", pb.input((count,), None, "x"), name="copy")
    plan = pb.build(y)
    if shift:  # both activations off the planner's 32-element alignment, still apart
        plan.buf_offset = [o + shift * (i + 1) for i, o in enumerate(plan.buf_offset)]
        plan.arena_floats += 2 * shift + 32
    return plan


def stored(x, storage):
    """x as the storage type holds it, in fp32."""
    with np.errstate(over="ignore"):
        return {"f32": lambda: x, "f16": lambda: x.astype(np.float16).astype(np.float32), "bf16": lambda: _bf16(x)}[storage]()


def data(count):
    x = np.random.default_rng(count).standard_normal(count).astype(np.float32)
    special = np.array([np.inf, -np.inf, 65504.0, 65520.0, 1e-8, -0.0, 3.4e38], np.float32)
    x[: min(count, 7)] = special[: min(count, 7)]
    return x


@pytest.mark.parametrize("storage", ["f32", "f16", "bf16"])
@pytest.mark.parametrize("shift", [0, 1, 2])
def test_session_staging(hip, storage, shift):
    for count in COUNTS:
        print(f"[gpu] staging {storage} {count} shift {shift}", flush=True)
        x = data(count)
        with HipInferenceSession(hip.graph(copy_plan(count, shift), storage)) as s:
            s.set_input(x)
            got = s.run().copy()
        want = stored(x, storage)
        assert got.tobytes() == want.tobytes(), (count, np.flatnonzero(got != want)[:4])


@pytest.mark.parametrize("storage", ["f32", "f16"])
def test_large_output_by_the_copy_engine(hip, storage):
    count = (8 << 20) + 5  # one element above 32 MiB of fp32 and a ragged tail
    x = data(count)
    want = stored(x, storage)
    with HipInferenceSession(hip.graph(copy_plan(count), storage)) as s:
        s.set_input(x)
        for replay in (False, True):
            s.set_replay(replay)
            s.output[:] = 0
            assert s.run().tobytes() == want.tobytes(), replay


def test_runner_mixes_large_and_small_outputs(hip):
    counts = [5, (8 << 20) + 1, 4099]
    r = HipUnitRunner(hip, streams=2)
    for c in counts:
        r.add(hip.graph(copy_plan(c), "f16"))
    xs = [data(c) for c in counts]
    for i, x in enumerate(xs):
        r.input(i)[:] = x
    for _ in range(2):
        r.submit()
        r.wait()
        for i, x in enumerate(xs):
            assert r.output(i).tobytes() == stored(x, "f16").tobytes(), i
    r.close()
