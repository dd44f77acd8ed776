"""The autotuner's results reach the serving loop's FP32 plans also where the fastest
candidate is a split-BF16 form, which serving does not offer; and its times are those
of operands with every bit in use."""
import time

import numpy as np
import pytest

import cogconv._lib as L
import oracle as O
from gpuhelp import desc_pair
from test_plain_plans_host import serving_plan

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def device():
    L.init(0)
    L.tune_cache_clear()
    yield
    L.tune_cache_clear()
    L.synchronize()


def test_serving_takes_the_best_plain_candidate(tmp_path):
    _, cd = desc_pair(O.PF_BRS, O.CLAMP, O.XCORR, O.NONE, 1, 1, (32, 128, 128), (32 * 32, 9, 9))
    r = L.autotune(cd, warmup_steps=1, run_steps=2, flush_bytes=16 << 20)
    print("CASE tuned", r["description"], flush=True)
    assert r["description"].split()[0].endswith("x3")  # 49 us against 68 us for the FP32 MFMA kernel
    path = tmp_path / "tune.txt"
    L.tune_cache_save(str(path))
    samples = {ln.split("\t")[1]: ln.split("\t") for ln in path.read_text().splitlines() if not ln.startswith("#")}
    plain = [f for k, f in samples.items() if k.endswith(" plain")]
    assert len(samples) == 2 and len(plain) == 1
    assert serving_plan(cd)[0] == plain[0][7]
    assert L.autotune(cd, warmup_steps=1, run_steps=2, flush_bytes=16 << 20)["from_cache"]

    # Any plain sample is the one that serving runs, whatever its index in the list.
    names = []
    for v in range(L.variant_count(cd)):
        p = L.Plan(cd, v)
        names.append(p.description)
        p.close()
    other = [n for n in names if not n.split()[0].endswith("x3") and n != plain[0][7]][-1]
    lines = []
    for f in samples.values():
        if f in plain:
            f = f[:2] + ["0"] + f[3:7] + [other]
        lines.append("\t".join(f))
    L.tune_cache_clear()
    path.write_text("\n".join(lines) + "\n")
    L.tune_cache_load(str(path))
    assert serving_plan(cd)[0] == other
    plan = L.Plan(cd)
    assert plan.description == r["description"]
    plan.close()

    # A file without the plain sample (an older library's) is timed again.
    L.tune_cache_clear()
    path.write_text("\n".join(ln for ln in lines if " plain\t" not in ln) + "\n")
    L.tune_cache_load(str(path))
    assert not L.autotune(cd, warmup_steps=1, run_steps=2, flush_bytes=16 << 20)["from_cache"]


def test_sample_keeps_its_meaning_at_another_index(tmp_path):
    """A sample whose index is of another list names its candidate all the same."""
    _, cd = desc_pair(O.PF_BRS, O.VALID, O.XCORR, O.NONE, 1, 2, (2 * 8, 40, 44), (16 * 8, 3, 3))
    r = L.autotune(cd, warmup_steps=0, run_steps=1, flush_bytes=0)
    path = tmp_path / "tune.txt"
    L.tune_cache_save(str(path))
    n = L.variant_count(cd)
    last = L.Plan(cd, n - 1)
    lines = []
    for ln in path.read_text().splitlines():
        f = ln.split("\t")
        if len(f) == 8 and not f[1].endswith(" plain"):
            f[2], f[7] = "0", last.description
        lines.append("\t".join(f))
    path.write_text("\n".join(lines) + "\n")
    L.tune_cache_clear()
    L.tune_cache_load(str(path))
    plan = L.Plan(cd)
    print("CASE renumbered sample", r["description"], plan.description, flush=True)
    assert plan.description == last.description and plan.variant == n - 1
    plan.close()
    last.close()


def test_tuned_times_are_those_of_varied_operands():
    """The FP32 split forms are bound by the matrix cores' power, and operands whose
    low BF16 terms are all zero ran in 0.81 of the time."""
    B, N, K, H, F = 8, 32, 32, 256, 9
    _, cd = desc_pair(O.PF_BRS, O.CLAMP, O.XCORR, O.NONE, 1, B, (B * N, H, H), (K * N, F, F))
    r = L.autotune(cd, warmup_steps=2, run_steps=6)
    plan = L.Plan(cd)
    print("CASE tuned times", r["avg_us"], plan.description, flush=True)
    assert plan.variant == r["variant"]
    rng = np.random.default_rng(1)
    bx = L.DeviceBuffer.from_array(rng.uniform(-1, 1, (B * N, H, H)).astype(np.float32))
    bw = L.DeviceBuffer.from_array(rng.uniform(-1, 1, (K * N, F, F)).astype(np.float32))
    bo, ws = L.DeviceBuffer(4 * int(np.prod(plan.out_shape))), L.DeviceBuffer(plan.workspace_bytes)
    times = []
    for _ in range(4):
        L.synchronize()
        start = time.perf_counter()
        for _ in range(20):
            plan.launch(bx, bw, bo, ws)
        L.synchronize()
        times.append((time.perf_counter() - start) / 20 * 1e6)
    for b in (bx, bw, bo, ws):
        b.close()
    plan.close()
    assert r["avg_us"] >= 0.92 * min(times)
