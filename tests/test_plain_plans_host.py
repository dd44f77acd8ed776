"""The plans that leave the split-BF16 forms of FP32 out (no GPU): the serving loop's,
which has no workspace for a packed operand 2, and those under the implicit-GEMM
hint, which asks for FP32 products."""
import ctypes

import pytest

import cogconv._lib as L
import oracle as O
from gpuhelp import desc_pair

CREATE = "_ZN7cogconv19plan_create_servingEPK12cogconv_descPP14cogconv_plan_s"


def serving_plan(cd):
    """(description, workspace bytes) of the serving loop's plan."""
    lib = L.lib()
    create = getattr(lib, CREATE)
    create.restype = ctypes.c_int
    handle = ctypes.c_void_p()
    L.check(create(ctypes.byref(cd), ctypes.byref(handle)))
    text, size = ctypes.create_string_buffer(256), ctypes.c_size_t()
    L.check(lib.cogconv_plan_describe(handle, text, len(text)))
    L.check(lib.cogconv_plan_workspace_bytes(handle, ctypes.byref(size)))
    L.check(lib.cogconv_plan_destroy(handle))
    return text.value.decode(), size.value


@pytest.mark.parametrize("mode,border,sampling,step,N,K,side,F,prefix", [
    (O.PF_BRS, O.ZERO, O.UP, 2, 32, 32, 256, 7, "igemm_f32_up2 "),
    (O.PF_BRS, O.CYCLIC, O.UP, 2, 64, 32, 32, 7, "igemm_f32_up2 "),
    (O.BPF_BRS, O.FULL, O.UP, 2, 48, 16, 90, 5, "igemm_f32_up2 "),
    (O.PF_BRS, O.VALID, O.UP, 2, 16, 64, 128, 3, "igemm_f32_up2 "),
    (O.PF_BRS, O.ZERO, O.NONE, 1, 64, 64, 96, 3, "igemm_f32 "),
    (O.PF_BRS, O.CLAMP, O.DOWN, 2, 24, 40, 150, 5, "igemm_f32 "),
    (O.PF_BRS, O.CLAMP, O.DOWN, 2, 22, 16, 128, 9, "direct "),  # the MFMA kernel takes no 9x9 with an output step
    (O.FA_BRS, O.VALID, O.NONE, 1, 22, 2, 250, 3, "fa_igemm_f32 "),
])
def test_fp32_requests_run_the_plain_kernels(mode, border, sampling, step, N, K, side, F, prefix):
    orient = O.CONV if mode == O.BPF_BRS else O.XCORR
    planes = K if mode == O.BPF_BRS else N
    ws = (K, side - F + 1, side - F + 1) if mode == O.FA_BRS else (K * N, F, F)
    _, cd = desc_pair(mode, border, orient, sampling, step, 1, (planes, side, side), ws)
    name, workspace = serving_plan(cd)
    assert name.startswith(prefix), name
    if mode != O.FA_BRS:
        assert workspace == 0


def test_low_precision_requests_run_the_default_plan():
    _, cd = desc_pair(O.PF_BRS, O.ZERO, O.XCORR, O.NONE, 1, 1, (32, 64, 64), (48 * 32, 3, 3), precision=L.BF16)
    plan = L.Plan(cd)
    assert serving_plan(cd) == (plan.description, plan.workspace_bytes)
    plan.close()


@pytest.mark.parametrize("mode,border,sampling,step,N,K,side,F,prefix", [
    (O.PF_BRS, O.ZERO, O.UP, 2, 32, 32, 256, 7, "igemm_f32_up2 "),
    (O.PF_BRS, O.ZERO, O.NONE, 1, 64, 64, 96, 3, "igemm_f32 "),
    (O.PF_BRS, O.CLAMP, O.DOWN, 2, 24, 40, 150, 5, "igemm_f32 "),
    (O.FA_BRS, O.VALID, O.NONE, 1, 22, 2, 250, 3, "fa_igemm_f32 "),
])
def test_implicit_gemm_hint_keeps_fp32_products(mode, border, sampling, step, N, K, side, F, prefix):
    ws = (K, side - F + 1, side - F + 1) if mode == O.FA_BRS else (K * N, F, F)
    _, cd = desc_pair(mode, border, O.XCORR, sampling, step, 1, (N, side, side), ws, algo=L.ALGO_IMPLICIT_GEMM)
    plan = L.Plan(cd)
    assert plan.description.startswith(prefix), plan.description
    plan.close()


def test_implicit_gemm_hint_refuses_what_it_has_no_kernel_for():
    _, cd = desc_pair(O.PF_BRS, O.CLAMP, O.XCORR, O.DOWN, 2, 1, (22, 128, 128), (16 * 22, 9, 9),
                      algo=L.ALGO_IMPLICIT_GEMM)
    with pytest.raises(L.CogconvError) as e:
        L.Plan(cd)
    assert e.value.status == L.ERR_UNSUPPORTED


def test_register_ring_is_named_where_there_is_one():
    _, cd = desc_pair(O.PF_BRS, O.ZERO, O.XCORR, O.NONE, 1, 1, (16, 64, 64), (32 * 16, 3, 3), precision=L.BF16)
    names = []
    for v in range(L.variant_count(cd)):
        plan = L.Plan(cd, v)
        names.append(plan.description)
        plan.close()
    assert all((" ring" in n) != (" inline" in n) for n in names) and any(" inline" in n for n in names)
