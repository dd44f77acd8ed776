"""FP32 FilterAdjoint as split-BF16 products (fa_igemm_f32x3 plans): parity with the
FP64 oracle at the edges of its tiles, operands outside the split's range, and
non-finite operands."""
import numpy as np
import pytest

import cogconv._lib as L
import oracle as O
from gpuhelp import assert_parity, desc_pair, oracle_ref, run_gpu

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def device():
    L.init(0)
    yield
    L.synchronize()


def case(B, N, K, H, W, F):
    xs, ds = (B * N, H, W), (B * K, H - F + 1, W - F + 1)
    od, cd = desc_pair(O.FA_BRS, O.VALID, O.XCORR, O.NONE, 1, B, xs, ds)
    names = []
    for v in range(L.variant_count(cd)):
        p = L.Plan(cd, v)
        names.append(p.description)
        p.close()
    rows = [v for v, n in enumerate(names) if n.startswith("fa_igemm_f32x3")]
    assert rows
    return od, cd, xs, ds, rows, names


@pytest.mark.parametrize("B,N,K,H,W,F", [
    (1, 1, 1, 3, 3, 3),      # one dy pixel
    (2, 16, 32, 18, 34, 3),  # whole tiles, one 32-pixel chunk
    (1, 17, 33, 20, 35, 3),  # one plane and one pixel past
    (3, 5, 7, 9, 67, 1),
    (1, 65, 20, 12, 30, 1),
])
def test_every_candidate(B, N, K, H, W, F):
    rng = np.random.default_rng(H * 100 + W)
    od, cd, xs, ds, rows, names = case(B, N, K, H, W, F)
    x = rng.uniform(-1, 1, xs).astype(np.float32)
    dy = rng.uniform(-1, 1, ds).astype(np.float32)
    ref, mag = oracle_ref(od, x, dy)
    for v in rows:
        print("CASE fa rows f32", names[v], flush=True)
        assert_parity(run_gpu(cd, x, dy, variant=v), ref, mag, what=names[v])


@pytest.mark.parametrize("xs_,ds_", [(1e-36, 1e8), (1e10, 1e-37), (1e-36, 1.0), (1e30, 1.0)])
def test_magnitudes(xs_, ds_):
    rng = np.random.default_rng(3)
    od, cd, xs, ds, rows, names = case(1, 6, 9, 14, 40, 3)
    x = (rng.uniform(0.5, 1, xs) * xs_).astype(np.float32)
    dy = (rng.uniform(0.5, 1, ds) * ds_).astype(np.float32)
    ref, mag = oracle_ref(od, x, dy)
    for v in rows:
        print("CASE fa rows magnitude", xs_, ds_, names[v], flush=True)
        assert np.all(np.abs(run_gpu(cd, x, dy, variant=v) - ref) <= 1e-5 * mag)


def test_non_finite():
    """Infinities and NaNs reach exactly the outputs whose sums hold them (the FP32
    MFMA kernel adds some: its padded tap columns multiply them by 0)."""
    rng = np.random.default_rng(4)
    od, cd, xs, ds, rows, names = case(2, 18, 35, 12, 41, 3)
    x = rng.integers(1, 4, xs).astype(np.float32)
    dy = rng.integers(1, 4, ds).astype(np.float32)
    x[3, 5, 20], x[20, 11, 40], dy[7, 2, 3], dy[40, 9, 38] = np.inf, np.nan, -np.inf, 3.4028235e38
    with np.errstate(all="ignore"):
        want = O.conv(od, x, dy).astype(np.float32)
    for v in rows:
        print("CASE fa rows non-finite", names[v], flush=True)
        got = run_gpu(cd, x, dy, variant=v)
        assert np.array_equal(np.isnan(got), np.isnan(want)) and np.array_equal(np.isinf(got), np.isinf(want))
        ok = np.isfinite(want) & (np.abs(want) < 1e30)
        assert np.array_equal(got[ok], want[ok])  # small integers: every sum is exact
