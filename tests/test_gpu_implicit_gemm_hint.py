"""COGCONV_ALGO_IMPLICIT_GEMM on the frame modes: the tiled low-precision kernel
(whole filters, tap-row groups and the one-row ring, every output block) at 3x3 to
9x9 with and without an epilogue, and FP32 products for FP32."""
import numpy as np
import pytest

import cogconv._lib as L
import oracle as O
from gpuhelp import desc_pair, run_gpu

pytestmark = pytest.mark.gpu

NAMES = {L.BF16: "igemm_bf16 ", L.FP16: "igemm_fp16 ", L.SPLIT_BF16: "igemm_split_bf16 "}


@pytest.fixture(scope="module", autouse=True)
def device():
    L.init(0)
    yield
    L.synchronize()


def rounded(a, precision):
    """`a` as the MFMA reads it: rounded to nearest even."""
    if precision == L.FP16:
        return a.astype(np.float16).astype(np.float32)
    bits = a.view(np.uint32).astype(np.uint64)
    return ((bits + 0x7FFF + ((bits >> 16) & 1)) & 0xFFFF0000).astype(np.uint32).view(np.float32)


def candidates(cd):
    names = []
    for v in range(L.variant_count(cd)):
        p = L.Plan(cd, v)
        names.append(p.description)
        p.close()
    return names


@pytest.mark.parametrize("precision", (L.BF16, L.FP16, L.SPLIT_BF16))
@pytest.mark.parametrize("mode,border,B,N,K,H,W,F", [
    (O.PF_BRS, O.CLAMP, 2, 36, 20, 23, 68, 3),   # 16-byte staging with a halo pass, a partial 16-plane block
    (O.BPF_BRS, O.CYCLIC, 1, 33, 50, 21, 37, 5), # one plane past the chunk, four output blocks, unaligned rows
    (O.PF_BRS, O.ZERO, 1, 20, 64, 16, 64, 7),    # whole tiles
    (O.BPF_BRS, O.FULL, 1, 9, 16, 9, 30, 9),
])
def test_low_precision_every_candidate(precision, mode, border, B, N, K, H, W, F):
    """FP32 summation error only against the oracle on rounded operands (split-BF16:
    and the dropped product of the low terms, 2^-16 of a product), all candidates bit
    for bit alike, and an epilogue as its own pass over the result."""
    rng = np.random.default_rng(F * 1000 + H + precision)
    a = rng.uniform(-1, 1, (B * N, H, W)).astype(np.float32)
    k = rng.uniform(-1, 1, (K * N, F, F)).astype(np.float32)
    orient = O.CONV if mode == O.BPF_BRS else O.XCORR
    od, cd = desc_pair(mode, border, orient, O.NONE, 1, B, a.shape, k.shape, precision, L.ALGO_IMPLICIT_GEMM)
    names = candidates(cd)
    assert all(n.startswith(NAMES[precision]) for n in names), names
    if precision != L.SPLIT_BF16:
        assert any(" ring" in n for n in names) and any(" ring" not in n for n in names), names
    if precision == L.SPLIT_BF16:
        ra, rk, tol = a, k, 2.0 ** -16 + 2e-6
    else:
        ra, rk, tol = rounded(a, precision), rounded(k, precision), 2e-6
    ref, mag = O.conv(od, ra, rk), O.conv(od, np.abs(ra), np.abs(rk))
    planes, rows, cols = ref.shape
    fields = [(2, rows, cols, planes, 1), (0, 1, 1, planes, 1)]
    ops = [(L.EPI_MUL_FIELD, 0, 0), (L.EPI_ADD_FIELD, 0, 1), (L.EPI_MAX_CONST, 0.25, 0)]
    operands = [L.DeviceBuffer.from_array(rng.uniform(0.5, 2, (t[3], t[1], t[2])).astype(np.float32)) for t in fields]
    epi = L.make_epilogue(ops, [L.field_type(*t) for t in fields])
    ba, bk = L.DeviceBuffer.from_array(a), L.DeviceBuffer.from_array(k)
    plain, want, got = (L.DeviceBuffer(4 * ref.size) for _ in range(3))
    first = None
    for v, name in enumerate(names):
        print("CASE hinted candidate", mode, border, name, flush=True)
        plan = L.Plan(cd, v)
        ws = L.DeviceBuffer(plan.workspace_bytes)
        plan.launch(ba, bk, plain, ws)
        L.elementwise(plain, want, (2, rows, cols, planes, 1), epi, operands)
        plan.set_epilogue(epi)
        plan.launch_epilogue(ba, bk, got, ws, operands)
        L.synchronize()
        out = plain.download(ref.shape)
        assert np.all(np.abs(out - ref) <= tol * mag), name
        first = out if first is None else first
        assert np.array_equal(out, first), (name, names[0])
        assert np.array_equal(got.download(ref.shape), want.download(ref.shape)), name
        ws.close()
        plan.close()
    for b in operands + [ba, bk, plain, want, got]:
        b.close()


@pytest.mark.parametrize("sampling,step,border", [(O.NONE, 1, O.CLAMP), (O.UP, 2, O.ZERO), (O.DOWN, 2, O.CLAMP)])
def test_fp32_products_round_once(sampling, step, border):
    """A bank of one tap an output scales planes: the hinted FP32 plan rounds each
    product once."""
    rng = np.random.default_rng(21)
    N, K, H, W, F = 18, 34, 40, 64, 3
    x = rng.uniform(1, 2, (N, H, W)).astype(np.float32)
    w = np.zeros((K, N, F, F), np.float32)
    for k in range(K):
        w[k, k % N, 1, 1] = rng.uniform(1, 2)
    w = w.reshape(K * N, F, F)
    od, cd = desc_pair(O.PF_BRS, border, O.XCORR, sampling, step, 1, x.shape, w.shape, algo=L.ALGO_IMPLICIT_GEMM)
    want = O.conv(od, x, w).astype(np.float32)  # exact in 64 bits
    for v, name in enumerate(candidates(cd)):
        if name.startswith("igemm_f32"):
            print("CASE hinted FP32", name, flush=True)
            assert not name.split()[0].endswith("x3")
            assert np.array_equal(run_gpu(cd, x, w, variant=v), want), name


@pytest.mark.parametrize("sampling,step,border,F", [(O.NONE, 1, O.CLAMP, 9), (O.NONE, 1, O.ZERO, 3), (O.UP, 2, O.ZERO, 5),
                                                    (O.DOWN, 2, O.CYCLIC, 5)])
def test_fp32_bits_do_not_depend_on_the_batch(sampling, step, border, F):
    """One image's result under the hint is the same at every batch size."""
    rng = np.random.default_rng(22)
    N, K, H, W = 20, 36, 50, 64
    x = rng.uniform(-1, 1, (16 * N, H, W)).astype(np.float32)
    w = rng.uniform(-1, 1, (K * N, F, F)).astype(np.float32)
    first = None
    for B in (1, 3, 16):
        a = np.ascontiguousarray(x[:B * N])
        _, cd = desc_pair(O.PF_BRS, border, O.XCORR, sampling, step, B, a.shape, w.shape, algo=L.ALGO_IMPLICIT_GEMM)
        print("CASE batch", B, sampling, F, flush=True)
        got = run_gpu(cd, a, w)[:K]
        first = got if first is None else first
        assert np.array_equal(got, first)
