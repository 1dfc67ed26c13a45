"""MXFP4 with few rows of x1 (qmm_mxfp4_rows.hip) through the two-phase entry point, against the oracle."""
import numpy as np
import pytest

import cases
import oracle_api as orc
from test_gpu_other_modes import check_close
from test_gpu_routes import route

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _reset(gpu):
    gpu.lib().opsnnSetForcePlain(0)
    yield
    gpu.lib().opsnnSetForcePlain(0)


@pytest.mark.parametrize("M,K,N,tB,batch,out", [
    # every row-block count and its edges, 16 and 32 columns per workgroup (wide N), columns that end inside a block of 16 and that
    # are no multiple of four
    (1, 1024, 256, True, 1, "f32"), (15, 1152, 257, True, 1, "bf16"), (16, 2048, 8200, True, 1, "f16"), (5, 1024, 9001, True, 1, "f32"),
    (17, 1024, 300, True, 1, "f32"), (32, 1152, 4100, True, 1, "bf16"), (33, 1024, 271, True, 1, "f32"), (48, 1024, 2100, True, 1, "f32"),
    (49, 1152, 300, True, 1, "bf16"), (64, 1024, 2104, True, 1, "f32"), (65, 1024, 600, True, 1, "f32"), (128, 1152, 2200, True, 1, "f32"),
    # K tails: one MX block past a whole step, a unit of two and of four steps less or more, less than one unit, fewer units than waves
    (3, 128, 256, True, 1, "f32"), (16, 160, 272, True, 1, "f32"), (7, 224, 4112, True, 1, "f32"), (16, 480, 4112, True, 1, "f32"),
    (16, 512, 8192, True, 1, "f32"), (16, 544, 8192, True, 1, "f32"), (20, 288, 256, True, 1, "f32"), (40, 352, 4112, True, 1, "f32"),
    (2, 4448, 264, True, 1, "f32"), (60, 3008, 300, True, 1, "bf16"),
    # batches, and the weight in [K, N] storage (re-laid out in front of the kernel)
    (12, 1984, 264, True, 3, "f32"), (33, 1088, 270, True, 2, "f32"), (4, 1056, 256, False, 1, "f32"), (18, 1024, 300, False, 2, "bf16"),
])
def test_few_rows(gpu, M, K, N, tB, batch, out):
    """fp4 products and their scaling are exact; the sums are fp32, in the waves' order: fp32 outputs within 2^-18 of the sum of
    magnitudes (K <= 4448 terms in at most 36 dependent steps), 16-bit ones at the stated bar."""
    m = gpu
    print(f"case mxfp4 few rows M={M} K={K} N={N} tB={tB} batch={batch} out={out}", flush=True)
    dt = {"bf16": m.ACL_BF16, "f16": m.ACL_FLOAT16, "f32": m.ACL_FLOAT}[out]
    inp = cases.make_mx_inputs(m, M, K, N, K + N + M, tB, True, batch=batch, exp_range=1 if out == "f16" else 4)   # (fp16 ends at 65504)
    bias = np.random.default_rng(1).normal(0, 1, N).astype(np.float32) if M % 2 == 0 else None
    want = cases.oracle_mx(m, inp, M, K, N, tB, dt, bias)
    got = cases.run_mx_aclnn(m, inp, M, K, N, tB, dt, bias)
    assert route(m)[0] == "mxfp4_rows", route(m)
    if out == "f32":
        pos = dict(inp, x1=inp["x1"] & 0x77, x2=inp["x2"] & 0x77)
        abs_sum = cases.oracle_mx(m, pos, M, K, N, tB, dt).astype(np.float64) + (np.abs(bias) if bias is not None else 0.0)
        err = np.abs(got.astype(np.float64) - want.astype(np.float64))
        assert (err <= 2.0 ** -18 * abs_sum + 1e-30).all(), f"worst error / sum of magnitudes: {float((err / (abs_sum + 1e-30)).max()):.3e}"
    else:
        check_close(got, want, orc.BF16 if out == "bf16" else orc.F16, "mxfp4 few rows")


def test_one_row_against_many_equal_rows(gpu):
    """A row of x1 does not depend on the rows beside it."""
    m = gpu
    K, N = 1184, 8200
    inp = cases.make_mx_inputs(m, 16, K, N, 3, True, True)
    all_rows = cases.run_mx_aclnn(m, inp, 16, K, N, True, m.ACL_FLOAT, None)
    one = dict(inp, x1=np.ascontiguousarray(inp["x1"][:, 5:6]), s1=np.ascontiguousarray(inp["s1"][:, 5:6]))
    row = cases.run_mx_aclnn(m, one, 1, K, N, True, m.ACL_FLOAT, None)
    assert np.array_equal(all_rows.reshape(16, N)[5], row.reshape(N))
