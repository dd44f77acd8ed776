"""Default plans of calls where the kernel estimated fastest had not been the fastest
measured on an MI355X (no GPU needed): the times in us are those measured."""
import pytest

import cogconv._lib as L

PF, BPF = L.PROJECT_FRAME_BLOCK_REDUCE_SUM, L.BACK_PROJECT_FRAME_BLOCK_REDUCE_SUM
FA = L.FILTER_ADJOINT_BLOCK_REDUCE_SUM
CLAMP, CYCLIC, ZERO, FULL, VALID = L.BORDER_CLAMP, L.BORDER_CYCLIC, L.BORDER_ZERO, L.BORDER_FULL, L.BORDER_VALID
NONE, UP, DOWN = L.NO_SAMPLING, L.UPSAMPLE_INPUT, L.DOWNSAMPLE_OUTPUT


@pytest.mark.parametrize("mode,border,sampling,precision,B,N,K,H,W,F,kernel", [
    # FP32 MFMA kernels against the split-BF16 forms
    (BPF, CLAMP, NONE, L.FP32, 2, 16, 24, 146, 116, 9, "igemm_f32 "),       # 41.0, 53.7 split
    (PF, CYCLIC, DOWN, L.FP32, 16, 23, 25, 134, 162, 3, "igemm_f32 "),      # 32.3, 36.0
    (PF, CYCLIC, UP, L.FP32, 2, 32, 39, 141, 126, 3, "igemm_f32_up2 "),     # 20.6, 25.2
    (PF, ZERO, UP, L.FP32, 3, 7, 33, 48, 64, 9, "igemm_f32_up2 "),          # 16.9, 20.4
    (FA, VALID, NONE, L.FP32, 24, 51, 38, 56, 82, 3, "fa_igemm_f32 "),      # 85.9, 106.1
    (FA, VALID, NONE, L.FP32, 5, 17, 16, 181, 221, 3, "fa_igemm_f32 "),     # 40.7, 50.2
    # the split-BF16 forms where they are faster
    (PF, CLAMP, NONE, L.FP32, 8, 32, 32, 256, 256, 9, "igemm_f32x3 "),      # 341, 726 FP32 MFMA
    (PF, ZERO, UP, L.FP32, 8, 32, 32, 256, 256, 7, "igemm_f32_up2x3 "),     # 265, 484
    (BPF, FULL, NONE, L.FP32, 19, 7, 10, 68, 108, 7, "rows=2 "),            # 46.2, 47.9 FP32 MFMA, 56.9 one row a wave
    (PF, ZERO, NONE, L.FP32, 11, 34, 10, 28, 39, 3, "igemm_f32x3 "),        # 13.9, 17.5
    (PF, ZERO, UP, L.FP32, 5, 12, 49, 49, 51, 3, "igemm_f32_up2x3 "),       # 11.8, 24.8
    # rows a wave of the low-precision forms
    (PF, ZERO, NONE, L.BF16, 3, 25, 9, 180, 222, 5, "rows=2 "),             # 15.4, 18.1 with four (15.9 tiled)
    (BPF, FULL, NONE, L.SPLIT_BF16, 13, 12, 31, 94, 61, 5, "rows=2 "),      # 21.1, 31.5 with four (27.9 tiled)
    (BPF, ZERO, NONE, L.BF16, 15, 26, 31, 41, 34, 5, "rows=1 ring "),       # 13.9, 15.7 packing in the kernel
    (PF, ZERO, NONE, L.BF16, 32, 64, 64, 128, 128, 3, "rows=4 ring threads=512"),  # 84, 95 tiled
])
def test_default_plan(mode, border, sampling, precision, B, N, K, H, W, F, kernel):
    planes = K if mode == BPF else N
    f = (2, H - F + 1, W - F + 1, B * K) if mode == FA else (2, F, F, K * N)
    orient = L.CONVOLUTION if mode == BPF else L.CROSS_CORRELATION
    d = L.make_desc(mode, border, orient, sampling, 1 if sampling == NONE else 2, B, (2, H, W, B * planes), f, precision)
    plan = L.Plan(d)
    assert kernel in plan.description, plan.description
    plan.close()
