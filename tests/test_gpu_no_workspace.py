"""FP32 frame plans launched without a workspace, as before the split-BF16 forms took
them over: the kernels with FP32 products, on several streams at once, with an
epilogue, and from a request table."""
import numpy as np
import pytest

import cogconv._lib as L
import oracle as O
from gpuhelp import desc_pair

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def device():
    L.init(0)
    yield
    L.synchronize()


N, K, H, W = 32, 40, 96, 100
SHAPES = [("unit", O.CLAMP, O.NONE, 1, 5), ("up", O.ZERO, O.UP, 2, 7), ("down", O.CLAMP, O.DOWN, 2, 5),
          ("down9", O.CLAMP, O.DOWN, 2, 9)]


def plans(border, sampling, step, F):
    xs, ws = (N, H, W), (K * N, F, F)
    _, cd = desc_pair(O.PF_BRS, border, O.XCORR, sampling, step, 1, xs, ws)
    split = [v for v in range(L.variant_count(cd)) if L.Plan(cd, v).description.split()[0].endswith("x3")]
    plan = L.Plan(cd, split[0])
    assert plan.workspace_bytes
    plain = None
    if F < 9:
        _, hint = desc_pair(O.PF_BRS, border, O.XCORR, sampling, step, 1, xs, ws, algo=L.ALGO_IMPLICIT_GEMM)
        plain = L.Plan(hint)
    else:  # the direct kernel
        plain = L.Plan(cd, [v for v in range(L.variant_count(cd)) if L.Plan(cd, v).description.startswith("direct")][0])
    return plan, plain


def result(plan, bx, bw, ws=None, **kw):
    out = L.DeviceBuffer(4 * int(np.prod(plan.out_shape)))
    plan.launch(bx, bw, out, ws, **kw)
    L.synchronize()
    got = out.download(plan.out_shape)
    out.close()
    return got


@pytest.mark.parametrize("name,border,sampling,step,F", SHAPES)
def test_plain_kernel_without_a_workspace(name, border, sampling, step, F):
    rng = np.random.default_rng(F)
    plan, plain = plans(border, sampling, step, F)
    print("CASE no workspace", name, plan.description, "|", plain.description, flush=True)
    bx = L.DeviceBuffer.from_array(rng.uniform(-1, 1, (N, H, W)).astype(np.float32))
    bw = L.DeviceBuffer.from_array(rng.uniform(-1, 1, (K * N, F, F)).astype(np.float32))
    want = result(plain, bx, bw)
    assert np.array_equal(result(plan, bx, bw), want)
    epi = L.make_epilogue([(L.EPI_MUL_CONST, 3.0, 0), (L.EPI_MAX_CONST, 0.5, 0)])
    plan.set_epilogue(epi)
    assert np.array_equal(result(plan, bx, bw), np.maximum(want * np.float32(3.0), np.float32(0.5)))
    if name in ("unit", "down"):
        assert plan.table_supported()
        plan.set_epilogue(None)
        out, tab = L.DeviceBuffer(4 * want.size), L.DeviceBuffer(16)
        plan.launch_table([(bx, out)], tab, in1=bw)
        L.synchronize()
        assert np.array_equal(out.download(want.shape), want)
        out.close()
        tab.close()
    for b in (bx, bw):
        b.close()
    plan.close()
    plain.close()


def test_one_plan_on_two_streams():
    rng = np.random.default_rng(3)
    plan, plain = plans(O.CLAMP, O.NONE, 1, 5)
    print("CASE two streams", plan.description, flush=True)
    bx = L.DeviceBuffer.from_array(rng.uniform(-1, 1, (N, H, W)).astype(np.float32))
    banks = [L.DeviceBuffer.from_array(rng.uniform(-1, 1, (K * N, 5, 5)).astype(np.float32)) for _ in range(2)]
    want = [result(plain, bx, bw) for bw in banks]
    streams = [L.Stream(), L.Stream()]
    outs = [[L.DeviceBuffer(4 * want[0].size) for _ in range(4)] for _ in range(2)]
    for i in range(4):
        for s in range(2):
            plan.launch(bx, banks[s], outs[s][i], None, stream=streams[s])
    L.synchronize()
    for s in range(2):
        for o in outs[s]:
            assert np.array_equal(o.download(want[s].shape), want[s])
            o.close()
    for b in banks + [bx]:
        b.close()
    for s in streams:
        s.close()
    plan.close()
    plain.close()
