"""The FP32 plans that run as split-BF16 products (igemm_f32x3, igemm_f32_up2x3 and
fa_igemm_f32x3) on operands outside the split's range: subnormal ones, whose BF16
terms all vanish, in every sampling the split forms take, and the time a field
full of non-finite samples takes, and their epilogues."""
import time

import numpy as np
import pytest

import cogconv._lib as L
import oracle as O
from gpuhelp import desc_pair, oracle_ref, run_gpu

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def device():
    L.init(0)
    yield
    L.synchronize()


# (mode, border, sampling, step, filter): batch 1, 18 -> 34 planes, 20x40
FORMS = {
    "unit": (O.PF_BRS, O.CLAMP, O.NONE, 1, 5),
    "up": (O.PF_BRS, O.ZERO, O.UP, 2, 5),
    "down": (O.PF_BRS, O.CLAMP, O.DOWN, 2, 5),
    "weight_grad": (O.FA_BRS, O.VALID, O.NONE, 1, 3),
}
N, K, H, W = 18, 34, 20, 40


def split_plans(form):
    """Descriptors, operand shapes and the split variants of a form."""
    mode, border, sampling, step, F = FORMS[form]
    xs = (N, H, W)
    ws = (K, H - F + 1, W - F + 1) if mode == O.FA_BRS else (K * N, F, F)
    od, cd = desc_pair(mode, border, O.XCORR, sampling, step, 1, xs, ws)
    split = []
    for v in range(L.variant_count(cd)):
        p = L.Plan(cd, v)
        if p.description.split()[0].endswith("x3"):
            split.append((v, p.description))
        p.close()
    assert split
    return od, cd, xs, ws, split


@pytest.mark.parametrize("form", FORMS)
@pytest.mark.parametrize("sx,sw", [(1e-41, 1e30), (1e30, 1e-41), (1e-44, 1e36)])
def test_operands_that_vanish_in_the_split(form, sx, sw):
    """Operands under 2^-134 round to 0 as BF16, and so do their remainders: the
    results, far from 0, are FP32 sums of them all the same."""
    rng = np.random.default_rng(11)
    od, cd, xs, ws, split = split_plans(form)
    x = (rng.uniform(0.5, 1, xs) * sx).astype(np.float32)
    w = (rng.uniform(0.5, 1, ws) * sw).astype(np.float32)
    ref, mag = oracle_ref(od, x, w)
    for v, name in split:
        print("CASE vanishing", form, sx, sw, name, flush=True)
        assert np.all(np.abs(run_gpu(cd, x, w, variant=v) - ref) <= 1e-5 * mag), name


@pytest.mark.parametrize("form", FORMS)
def test_vanishing_operands_beside_others(form):
    """A field of zeros with subnormal samples in some columns and ordinary ones in
    others: every output that only subnormal samples reach is their sum."""
    rng = np.random.default_rng(12)
    od, cd, xs, ws, split = split_plans(form)
    x = np.zeros(xs, np.float32)
    x[:, :, 3::16] = rng.uniform(0.5, 1, x[:, :, 3::16].shape) * 1e-41
    x[:, 10:, 11::16] = rng.uniform(0.5, 1, x[:, 10:, 11::16].shape)
    w = (rng.uniform(0.5, 1, ws) * 1e30).astype(np.float32)
    ref, mag = oracle_ref(od, x, w)
    for v, name in split:
        print("CASE vanishing beside others", form, name, flush=True)
        assert np.all(np.abs(run_gpu(cd, x, w, variant=v) - ref) <= 1e-5 * mag), name


@pytest.mark.parametrize("mode,B,N,K,H,W,F", [
    (O.PF_BRS, 1, 32, 32, 128, 128, 9),
    (O.FA_BRS, 16, 22, 2, 100, 256, 3),
])
@pytest.mark.parametrize("value", (np.nan, -np.inf, np.finfo(np.float32).min))
def test_masked_fields_keep_their_speed(mode, B, N, K, H, W, F, value):
    """A tenth of the samples NaN, infinite or the lowest float: every output is
    computed a second time, by the matrix cores as well (it took 117 and 20 times as
    long when each lane summed its outputs by itself, and takes 3 now)."""
    rng = np.random.default_rng(13)
    x = rng.uniform(-1, 1, (B * N, H, W)).astype(np.float32)
    ws = (B * K, H - F + 1, W - F + 1) if mode == O.FA_BRS else (K * N, F, F)
    w = rng.uniform(-1, 1, ws).astype(np.float32)
    _, cd = desc_pair(mode, O.VALID if mode == O.FA_BRS else O.CLAMP, O.XCORR, O.NONE, 1, B, x.shape, ws)
    plan = L.Plan(cd)
    assert plan.description.split()[0].endswith("x3")
    print("CASE masked field", value, plan.description, flush=True)
    bw, bo = L.DeviceBuffer.from_array(w), L.DeviceBuffer(4 * int(np.prod(plan.out_shape)))
    wk = L.DeviceBuffer(plan.workspace_bytes)
    best = []
    for a in (x, np.where(rng.random(x.shape) < 0.1, np.float32(value), x)):
        ba = L.DeviceBuffer.from_array(a)
        times = []
        for _ in range(8):
            L.synchronize()
            start = time.perf_counter()
            plan.launch(ba, bw, bo, wk)
            L.synchronize()
            times.append(time.perf_counter() - start)
        best.append(min(times))
        ba.close()
    for b in (bw, bo, wk):
        b.close()
    plan.close()
    assert best[1] <= 8 * best[0]


@pytest.mark.parametrize("form,F", [("unit", 5), ("unit", 9), ("up", 7), ("down", 3), ("weight_grad", 3)])
@pytest.mark.parametrize("inf", (False, True))
def test_epilogue_equals_its_own_pass(form, F, inf):
    """Constants and every kind of field operand, on plain outputs and on ones that
    are computed a second time."""
    rng = np.random.default_rng(14)
    mode, border, sampling, step, _ = FORMS[form]
    xs = (N, H, W)
    ws = (K, H - F + 1, W - F + 1) if mode == O.FA_BRS else (K * N, F, F)
    _, cd = desc_pair(mode, border, O.XCORR, sampling, step, 1, xs, ws)
    x = rng.uniform(-1, 1, xs).astype(np.float32)
    if inf:
        x[3, 7, 11] = np.inf
    bx = L.DeviceBuffer.from_array(x)
    bw = L.DeviceBuffer.from_array(rng.uniform(-1, 1, ws).astype(np.float32))
    plans = [L.Plan(cd, v) for v in range(L.variant_count(cd))]
    split = [p for p in plans if p.description.split()[0].endswith("x3")]
    assert split
    planes, rows, cols = split[0].out_shape
    n = planes * rows * cols
    fields = [(2, rows, cols, planes, 1), (2, rows, cols, 1, 0), (0, 1, 1, planes, 1), (0, 1, 1, 1, 0)]
    operands = [L.DeviceBuffer.from_array(rng.uniform(0.5, 2, (t[3], t[1], t[2])).astype(np.float32)) for t in fields]
    epi = L.make_epilogue([(L.EPI_MUL_FIELD, 0, 0), (L.EPI_SUB_FIELD, 0, 1), (L.EPI_ADD_FIELD, 0, 2),
                           (L.EPI_DIV_FIELD, 0, 3), (L.EPI_TANH, 0, 0), (L.EPI_MAX_CONST, -0.25, 0)],
                          [L.field_type(*t) for t in fields])
    out, want, got = (L.DeviceBuffer(4 * n) for _ in range(3))
    for plan in split:
        print("CASE split epilogue", form, inf, plan.description, flush=True)
        wk = L.DeviceBuffer(plan.workspace_bytes)
        plan.launch(bx, bw, out, wk)
        L.elementwise(out, want, (2, rows, cols, planes, 1), epi, operands)
        plan.set_epilogue(epi)
        plan.launch_epilogue(bx, bw, got, wk, operands)
        L.synchronize()
        a, b = got.download(plan.out_shape), want.download(plan.out_shape)
        assert np.array_equal(a, b, equal_nan=True), plan.description
        wk.close()
    for p in plans:
        p.close()
    for b in operands + [bx, bw, out, want, got]:
        b.close()
