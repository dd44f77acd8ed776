"""The row-walking frame kernel: the split-BF16 form of the FP32 frame modes
(igemm_f32x3 plans) and its BF16, FP16 and split-BF16 forms.  Parity with the FP64
oracle at the edges of its tiles, every candidate bit for bit alike, operands
outside the split's range, unaligned buffers and request tables."""
import numpy as np
import pytest

import cogconv._lib as L
import oracle as O
from gpuhelp import assert_parity, desc_pair, oracle_ref

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def device():
    L.init(0)
    yield
    L.synchronize()


def candidates(cd):
    """(igemm_f32x3 plans, the FP32 MFMA plan) of a descriptor."""
    plans = [L.Plan(cd, v) for v in range(L.variant_count(cd))]
    rows = [p for p in plans if p.description.startswith("igemm_f32x3")]
    mfma = [p for p in plans if p.description.startswith("igemm_f32 ")]
    return rows, mfma[0] if mfma else None


def launch(plan, a, k, off=0):
    """The plan's result, with operands and output `off` floats past an aligned address."""
    n = int(np.prod(plan.out_shape))
    ba, bk, bo = L.DeviceBuffer(4 * (a.size + off)), L.DeviceBuffer.from_array(k), L.DeviceBuffer(4 * (n + off))
    ba.upload(np.concatenate([np.zeros(off, np.float32), a.ravel()]))
    bo.upload(np.full(n + off, 7.0, np.float32))
    ws = L.DeviceBuffer(plan.workspace_bytes) if plan.workspace_bytes else None
    plan.launch(ba.ptr + 4 * off, bk, bo.ptr + 4 * off, ws)
    L.synchronize()
    out = bo.download((n + off,))
    assert np.all(out[:off] == 7.0)
    for b in (ba, bk, bo, ws):
        if b is not None:
            b.close()
    return out[off:].reshape(plan.out_shape)


@pytest.mark.parametrize("mode", (O.PF_BRS, O.BPF_BRS))
@pytest.mark.parametrize("border,B,N,K,H,W,F", [
    (O.ZERO, 1, 1, 1, 5, 7, 3),       # smaller than one tile in every dimension
    (O.CLAMP, 2, 15, 31, 8, 32, 3),   # whole tile, partial chunk and output block
    (O.CYCLIC, 1, 16, 32, 9, 33, 5),  # one row and column past the tile
    (O.VALID, 1, 17, 33, 37, 45, 5),  # one plane past the chunk and the output block
    (O.FULL, 2, 33, 5, 11, 30, 7),
    (O.CLAMP, 1, 40, 9, 31, 64, 7),
    (O.ZERO, 1, 20, 65, 33, 35, 9),
    (O.CYCLIC, 1, 5, 3, 4, 5, 9),     # the filter larger than the field
])
def test_every_candidate(mode, border, B, N, K, H, W, F):
    rng = np.random.default_rng(F * 100 + H)
    a = rng.uniform(-1, 1, (B * N, H, W)).astype(np.float32)
    k = rng.uniform(-1, 1, (K * N, F, F)).astype(np.float32)
    orient = O.CONV if mode == O.BPF_BRS else O.XCORR
    od, cd = desc_pair(mode, border, orient, O.NONE, 1, B, a.shape, k.shape)
    rows, _ = candidates(cd)
    assert rows
    ref, mag = oracle_ref(od, a, k)
    first = None
    for i, p in enumerate(rows):
        print("CASE rows", mode, border, p.description, flush=True)
        got = launch(p, a, k, off=i)
        assert_parity(got, ref, mag, what=p.description)
        first = got if first is None else first
        assert np.array_equal(got, first), p.description
        p.close()


@pytest.mark.parametrize("border,B,N,K,H,W,F,orient", [
    (O.ZERO, 1, 1, 1, 2, 3, 3, O.XCORR),        # one sample of some phases
    (O.CYCLIC, 2, 16, 32, 8, 32, 3, O.CONV),    # whole tiles at every row count
    (O.FULL, 1, 17, 33, 9, 33, 5, O.XCORR),     # odd output sizes, one row, column, plane, output past the tiles
    (O.VALID, 1, 7, 5, 12, 40, 5, O.XCORR),
    (O.ZERO, 2, 20, 9, 7, 31, 7, O.XCORR),      # odd halo
    (O.FULL, 1, 33, 40, 5, 18, 7, O.CONV),      # even halo
    (O.CYCLIC, 1, 5, 3, 3, 4, 9, O.XCORR),      # the filter larger than the stored field
    (O.VALID, 1, 18, 20, 17, 35, 9, O.XCORR),
])
def test_upsampled_every_candidate(border, B, N, K, H, W, F, orient):
    """2x up-sampled input (igemm_f32_up2x3): parity, every candidate alike, an
    epilogue applied as afterwards, and non-finite samples reaching exactly the
    outputs they reach in the FP32 MFMA kernel (no inserted zero multiplies them)."""
    rng = np.random.default_rng(F * 100 + H + W)
    mode = O.BPF_BRS if orient == O.CONV else O.PF_BRS
    a = rng.uniform(-1, 1, (B * N, H, W)).astype(np.float32)
    k = rng.uniform(-1, 1, (K * N, F, F)).astype(np.float32)
    od, cd = desc_pair(mode, border, orient, O.UP, 2, B, a.shape, k.shape)
    plans = [L.Plan(cd, v) for v in range(L.variant_count(cd))]
    rows = [p for p in plans if p.description.startswith("igemm_f32_up2x3")]
    mfma = [p for p in plans if "fused" in p.description]
    assert len(rows) == 2
    ref, mag = oracle_ref(od, a, k)
    b = a.copy()
    b[0, H // 2, W // 2], b[N - 1, 0, W - 1] = np.inf, np.nan
    first = None
    for i, p in enumerate(rows):
        print("CASE up rows", border, p.description, flush=True)
        got = launch(p, a, k, off=i)
        assert_parity(got, ref, mag, what=p.description)
        first = got if first is None else first
        assert np.array_equal(got, first), p.description
        if mfma:
            want = launch(mfma[0], b, k)
            bad = launch(p, b, k)
            assert np.array_equal(np.isnan(bad), np.isnan(want)) and np.array_equal(np.isinf(bad), np.isinf(want))
        p.set_epilogue(L.make_epilogue([(L.EPI_MUL_CONST, 3.0, 0), (L.EPI_MAX_CONST, 0.5, 0)]))
        assert np.array_equal(launch(p, a, k), np.maximum(got * np.float32(3.0), np.float32(0.5)))
    for p in plans:
        p.close()


@pytest.mark.parametrize("border,B,N,K,H,W,F", [
    (O.CLAMP, 1, 1, 1, 2, 4, 3),       # one output row and two columns
    (O.CYCLIC, 2, 16, 32, 16, 128, 3), # whole tiles
    (O.ZERO, 1, 17, 33, 18, 66, 5),    # one output row, column, plane and block past the tiles
    (O.VALID, 1, 40, 9, 30, 40, 7),
    (O.ZERO, 2, 9, 20, 22, 26, 9),
    (O.CYCLIC, 1, 5, 3, 4, 6, 9),      # the filter larger than the field
])
def test_output_step_every_candidate(border, B, N, K, H, W, F):
    """Every second output: parity, and non-finite samples reaching exactly the
    outputs they reach in the FP32 MFMA kernel."""
    rng = np.random.default_rng(F * 100 + H + W)
    a = rng.uniform(-1, 1, (B * N, H, W)).astype(np.float32)
    k = rng.uniform(-1, 1, (K * N, F, F)).astype(np.float32)
    od, cd = desc_pair(O.PF_BRS, border, O.XCORR, O.DOWN, 2, B, a.shape, k.shape)
    rows, _ = candidates(cd)
    other = [L.Plan(cd, v) for v in range(L.variant_count(cd))]
    other = [p for p in other if p.description.startswith(("igemm_f32 ", "direct"))]
    assert rows
    ref, mag = oracle_ref(od, a, k)
    b = a.copy()
    b[0, H // 2, W // 2], b[N - 1, 0, W - 1] = np.inf, np.nan
    want = launch(other[0], b, k)
    for i, p in enumerate(rows):
        print("CASE down rows", border, p.description, flush=True)
        assert_parity(launch(p, a, k, off=i + 1), ref, mag, what=p.description)
        bad = launch(p, b, k)
        assert np.array_equal(np.isnan(bad), np.isnan(want)) and np.array_equal(np.isinf(bad), np.isinf(want))


@pytest.mark.parametrize("scale", (1e-36, 1e-30, 1e30))
def test_magnitudes_beyond_the_split(scale):
    """Operands whose low BF16 terms underflow, and large ones: as exact as near 1."""
    rng = np.random.default_rng(5)
    a = (rng.uniform(0.5, 1, (18, 20, 40)) * np.float64(scale)).astype(np.float32)
    k = rng.uniform(0.5, 1, (34 * 18, 5, 5)).astype(np.float32)
    od, cd = desc_pair(O.PF_BRS, O.CLAMP, O.XCORR, O.NONE, 1, 1, a.shape, k.shape)
    rows, _ = candidates(cd)
    ref, mag = oracle_ref(od, a, k)
    for p in rows:
        print("CASE magnitude", scale, p.description, flush=True)
        # all terms positive: the oracle's magnitude sum is the result itself
        assert np.abs(launch(p, a, k) - ref).max() <= 1e-5 * ref.max()
        assert np.all(np.abs(launch(p, a, k) - ref) <= 1e-5 * mag)


@pytest.mark.parametrize("xs,ws", [(1e-36, 1e8), (1e10, 1e-37), (1e-33, 1e30)])
def test_small_operands_with_large_ones(xs, ws):
    """One operand too small for its low BF16 terms, the other large enough that
    the results are not small: still FP32 accuracy."""
    rng = np.random.default_rng(8)
    a = (rng.uniform(0.5, 1, (18, 20, 40)) * xs).astype(np.float32)
    k = (rng.uniform(0.5, 1, (34 * 18, 5, 5)) * ws).astype(np.float32)
    od, cd = desc_pair(O.PF_BRS, O.CLAMP, O.XCORR, O.NONE, 1, 1, a.shape, k.shape)
    rows, _ = candidates(cd)
    ref, mag = oracle_ref(od, a, k)
    for p in rows:
        print("CASE small and large", xs, ws, p.description, flush=True)
        assert np.all(np.abs(launch(p, a, k) - ref) <= 1e-5 * mag)


def rounded(a, precision):
    if precision == L.FP16:
        return a.astype(np.float16).astype(np.float32)
    bits = a.view(np.uint32).astype(np.uint64)
    return ((bits + 0x7FFF + ((bits >> 16) & 1)) & 0xFFFF0000).astype(np.uint32).view(np.float32)


@pytest.mark.parametrize("precision", (L.BF16, L.FP16, L.SPLIT_BF16))
@pytest.mark.parametrize("mode,border,B,N,K,H,W,F", [
    (O.PF_BRS, O.CLAMP, 1, 3, 2, 5, 4, 3),       # one column group a row, clamped on both sides
    (O.BPF_BRS, O.CLAMP, 2, 17, 33, 9, 36, 5),   # a group past the tile, one plane and output past their blocks
    (O.PF_BRS, O.CYCLIC, 1, 40, 9, 17, 8, 9),    # wrapped by more than a group on both sides
    (O.PF_BRS, O.ZERO, 2, 16, 32, 16, 64, 7),    # whole tiles
    (O.BPF_BRS, O.FULL, 1, 33, 5, 7, 28, 9),
    (O.PF_BRS, O.VALID, 3, 8, 20, 18, 44, 3),
    (O.PF_BRS, O.ZERO, 1, 20, 12, 8, 33, 3),     # rows of an odd width: no 16-byte loads
    (O.BPF_BRS, O.CYCLIC, 1, 50, 7, 5, 6, 7),    # the filter larger than the field
    (O.PF_BRS, O.CLAMP, 1, 24, 70, 33, 64, 3),   # three output blocks in workgroups of two, whole-line rows
    (O.BPF_BRS, O.ZERO, 1, 35, 33, 10, 12, 3),   # filters packed in the kernel: partial chunk and block, both
    (O.BPF_BRS, O.ZERO, 2, 19, 3, 9, 31, 5),     # orientations
])
def test_low_precision_every_candidate(precision, mode, border, B, N, K, H, W, F):
    """BF16 and FP16: FP32 summation error only, against the oracle on the rounded
    operands.  Split-BF16 drops the product of the low terms, 2^-16 of a product
    at most.  Aligned and unaligned fields give the same bits (16-byte and 4-byte
    staging), and so does the packed launch."""
    if precision == L.SPLIT_BF16 and F > 5:
        return
    rng = np.random.default_rng(F * 1000 + H * 10 + precision)
    a = rng.uniform(-1, 1, (B * N, H, W)).astype(np.float32)
    k = rng.uniform(-1, 1, (K * N, F, F)).astype(np.float32)
    orient = O.CONV if mode == O.BPF_BRS else O.XCORR
    od, cd = desc_pair(mode, border, orient, O.NONE, 1, B, a.shape, k.shape, precision=precision)
    if precision == L.SPLIT_BF16:
        ref, mag = oracle_ref(od, a, k)
        tol = 2.0 ** -16 + 2e-6
    else:
        ref, mag = oracle_ref(od, rounded(a, precision), rounded(k, precision))
        tol = 2e-6
    first, inline = None, 0
    for v in range(L.variant_count(cd)):
        p = L.Plan(cd, v)
        inline += "inline" in p.description
        print("CASE low precision", mode, border, p.description, flush=True)
        assert "x1" in p.description or "x2" in p.description
        for off in (0, 1):
            got = launch(p, a, k, off=off)
            assert np.all(np.abs(got - ref) <= tol * mag), (p.description, off)
            first = got if first is None else first
            assert np.array_equal(got, first), (p.description, off)
        ba, bk, ws = L.DeviceBuffer.from_array(a), L.DeviceBuffer.from_array(k), L.DeviceBuffer(p.workspace_bytes)
        bo = L.DeviceBuffer(4 * int(np.prod(p.out_shape)))
        assert p.pack_operand(bk, ws)
        p.launch_packed(ba, bo, ws)
        L.synchronize()
        assert np.array_equal(bo.download(p.out_shape), first)
        for x in (ba, bk, ws, bo):
            x.close()
        p.close()
    assert inline == (2 if F == 3 else int(F == 5 and precision != L.SPLIT_BF16))


def test_non_finite_operands():
    """Infinities, NaNs and the largest floats reach exactly the outputs they reach in
    the FP32 MFMA kernel, and leave the others as they are."""
    rng = np.random.default_rng(6)
    a = rng.integers(-3, 4, (17, 24, 70)).astype(np.float32)
    k = rng.integers(1, 4, (33 * 17, 3, 3)).astype(np.float32)
    a[0, 0, 0], a[3, 10, 40], a[16, 23, 69], a[5, 20, 20] = np.inf, np.nan, -np.inf, 3.4028235e38
    k[2 * 17 + 4, 1, 1], k[30 * 17, 0, 2] = np.inf, np.nan
    for border in (O.ZERO, O.CLAMP):
        _, cd = desc_pair(O.PF_BRS, border, O.XCORR, O.NONE, 1, 1, a.shape, k.shape)
        rows, mfma = candidates(cd)
        want = launch(mfma, a, k)
        for p in rows:
            print("CASE non-finite", border, p.description, flush=True)
            got = launch(p, a, k)
            assert np.array_equal(np.isnan(got), np.isnan(want)), p.description
            assert np.array_equal(got, want, equal_nan=True), p.description  # small integers: every sum is exact


def test_table_launch_equals_plain():
    rng = np.random.default_rng(7)
    B, N, K, H, W, F = 3, 18, 20, 26, 50, 5
    a = rng.uniform(-1, 1, (B * N, H, W)).astype(np.float32)
    k = rng.uniform(-1, 1, (K * N, F, F)).astype(np.float32)
    _, cd = desc_pair(O.PF_BRS, O.ZERO, O.XCORR, O.NONE, 1, B, a.shape, k.shape)
    rows, _ = candidates(cd)
    for p in rows:
        print("CASE table", p.description, flush=True)
        want = launch(p, a, k)
        assert p.table_supported()
        order = [2, 0, 1]  # images at unrelated addresses, in another order
        ins = [L.DeviceBuffer.from_array(a[b * N:(b + 1) * N]) for b in range(B)]
        outs = [L.DeviceBuffer(4 * K * H * W) for _ in range(B)]
        bk, tab, ws = L.DeviceBuffer.from_array(k), L.DeviceBuffer(16 * B), L.DeviceBuffer(p.workspace_bytes)
        p.launch_table([(ins[b], outs[b]) for b in order], tab, in1=bk, workspace=ws)
        L.synchronize()
        for b in range(B):
            assert np.array_equal(outs[b].download((K, H, W)), want[b * K:(b + 1) * K])
        for x in ins + outs + [bk, tab, ws]:
            x.close()
