"""The epilogue of a frame or PlaneByPlane plan, applied several output elements
of a thread at a time, gives bit for bit what the same ops give as their own
pass (cogconv_elementwise) over the plan's plain output: every op and operand
kind, at sizes with partial tiles, partial output-plane blocks and unaligned rows."""
import numpy as np
import pytest

import cogconv._lib as L

pytestmark = pytest.mark.gpu

PF, PBP = L.PROJECT_FRAME_BLOCK_REDUCE_SUM, L.PLANE_BY_PLANE


@pytest.fixture(scope="module", autouse=True)
def device():
    L.init(0)
    yield
    L.synchronize()


def op_lists(planes, rows, cols):
    """Epilogues covering every op (at most eight ops and four operands each)."""
    own, scalar, vector, zero = (2, rows, cols, planes, 1), (2, rows, cols, 1, 0), (0, 1, 1, planes, 1), (0, 1, 1, 1, 0)
    if planes == 1:
        own, vector = scalar, zero
    fields = [own, scalar, vector, zero]
    yield [(L.EPI_ADD_FIELD, 0, 2), (L.EPI_MAX_CONST, 0.0, 0)], fields
    yield [(L.EPI_MUL_FIELD, 0, 0), (L.EPI_SUB_FIELD, 0, 1), (L.EPI_RSUB_FIELD, 0, 2), (L.EPI_DIV_FIELD, 0, 3),
           (L.EPI_MIN_FIELD, 0, 0), (L.EPI_MAX_FIELD, 0, 1), (L.EPI_RDIV_FIELD, 0, 2), (L.EPI_TANH, 0, 0)], fields
    yield [(L.EPI_SQ, 0, 0), (L.EPI_ADD_CONST, 0.5, 0), (L.EPI_SQRT, 0, 0), (L.EPI_LOG, 0, 0), (L.EPI_EXP, 0, 0),
           (L.EPI_RDIV_CONST, 2.0, 0), (L.EPI_DIV_CONST, 3.0, 0), (L.EPI_SUB_CONST, 0.25, 0)], []
    yield [(L.EPI_NEG, 0, 0), (L.EPI_RSUB_CONST, 0.1, 0), (L.EPI_MUL_CONST, 1.5, 0), (L.EPI_MIN_CONST, 0.7, 0),
           (L.EPI_SIGNUM, 0, 0), (L.EPI_ABS, 0, 0)], []


@pytest.mark.parametrize("mode,precision,step,B,N,K,H,W,F", [
    (PF, L.FP32, 1, 2, 3, 8, 9, 35, 3),    # one output block, rows of odd length
    (PF, L.FP32, 1, 1, 5, 33, 17, 36, 5),  # aligned rows, a partial output block
    (PF, L.FP32, 1, 2, 4, 49, 8, 32, 1),
    (PF, L.FP32, 2, 1, 3, 17, 11, 13, 3),  # 2x up-sampled input
    (PF, L.BF16, 1, 2, 3, 8, 9, 35, 1),    # the smallest LDS footprint
    (PF, L.BF16, 1, 1, 33, 50, 13, 36, 3),
    (PF, L.FP16, 1, 1, 6, 20, 16, 64, 7),
    (PF, L.SPLIT_BF16, 1, 1, 4, 5, 10, 31, 3),
    (PF, L.BF16, 2, 1, 3, 17, 11, 13, 5),
    (PBP, L.FP32, 1, 1, 2, 1, 33, 131, 7),
])
def test_epilogue_equals_its_own_pass(mode, precision, step, B, N, K, H, W, F):
    rng = np.random.default_rng(H * W + F)
    x = rng.uniform(-1, 1, (B * N, H, W)).astype(np.float32)
    w = rng.uniform(-1, 1, (1 if mode == PBP else K * N, F, F)).astype(np.float32)
    desc = L.make_desc(mode, L.BORDER_ZERO, L.CROSS_CORRELATION, L.UPSAMPLE_INPUT if step > 1 else L.NO_SAMPLING, step,
                       B, (2, H, W, B * N), (2, F, F, w.shape[0]), precision)
    plain = L.Plan(desc)
    planes, rows, cols = plain.out_shape
    bx, bw = L.DeviceBuffer.from_array(x), L.DeviceBuffer.from_array(w)
    n = planes * rows * cols
    out, want, got = (L.DeviceBuffer(4 * n) for _ in range(3))
    ws = L.DeviceBuffer(max(4, plain.workspace_bytes))
    print("CASE epilogue", mode, precision, step, B, N, K, H, W, F, plain.description, flush=True)
    plain.launch(bx, bw, out, ws)
    L.synchronize()
    for ops, fields in op_lists(planes, rows, cols):
        operands = [L.DeviceBuffer.from_array(rng.uniform(0.5, 2, (t[3], t[1], t[2])).astype(np.float32))
                    for t in fields]
        epi = L.make_epilogue(ops, [L.field_type(*t) for t in fields])
        L.elementwise(out, want, (2, rows, cols, planes, 0 if planes == 1 else 1), epi, operands)
        plan = L.Plan(desc)
        plan.set_epilogue(epi)
        plan.launch_epilogue(bx, bw, got, ws, operands)
        L.synchronize()
        a, b = got.download(plain.out_shape), want.download(plain.out_shape)
        assert np.array_equal(a, b, equal_nan=True), ops
        plan.close()
        for o in operands:
            o.close()
    for buf in (bx, bw, out, want, got, ws):
        buf.close()
    plain.close()
