"""Weight-only calls on the kernel whose workgroups stage 128 columns of the weight and the rows of x together (wq_wide.hip): the edges
of its row blocks (16, 32, 64, 128) and of several slabs, a last K tile of 32, 64 and 96, a ragged last strip of columns, groups of 32
to K with a short last one, more groups than one round of its table holds, one scale for the whole weight; both storages of the
weight.  The bar is the sweep's: one rounding of the output beside the sum of K products in fp32."""
import pytest

import cases
import oracle_api as orc
from test_gpu_shape_sweep import _b16_bar

pytestmark = pytest.mark.gpu

KINDS = [("i4", "f16", True), ("i4", "bf16", False), ("i4", "bf16", True), ("i8", "f16", False), ("i8", "bf16", True)]


def _check(m, M, K, N, group, nk, w_dt, x_dt, off):
    xd = m.ACL_FLOAT16 if x_dt == "f16" else m.ACL_BF16
    inp = cases.make_wq_inputs(m, M, K, N, M + K, xd, m.ACL_INT4 if w_dt == "i4" else m.ACL_INT8, group, nk, off, xd if M % 2 else None)
    print(f"case {'nk' if nk else 'kn'} M={M} K={K} N={N} g={group} {w_dt} {x_dt} off={off}", flush=True)
    _b16_bar(cases.run_wq_aclnn(m, inp, M, K, N), cases.oracle_wq(m, inp, M, K, N), orc.F16 if x_dt == "f16" else orc.BF16, "wide", K)


@pytest.mark.parametrize("M,K,N,group", [
    (1, 1056, 1024, 32), (16, 16416, 1056, 128), (17, 2080, 4128, 64), (33, 8192, 1056, 128), (64, 4160, 2080, 0),
    (65, 1344, 1664, 64), (128, 1120, 1920, 256), (130, 2336, 1056, 128), (200, 1536, 1568, 0), (300, 4096, 544, 32),
])
@pytest.mark.parametrize("w_dt,x_dt,off", KINDS)
def test_rows_of_k(gpu, M, K, N, group, w_dt, x_dt, off):
    _check(gpu, M, K, N, group, False, w_dt, x_dt, off)


@pytest.mark.parametrize("M,K,N,group", [
    (9, 17280, 1873, 64), (20, 13568, 1730, 128), (40, 12544, 1793, 64), (64, 12928, 802, 32), (67, 14976, 1111, 128),
    (130, 8832, 1026, 0), (257, 7040, 1090, 128),
])
@pytest.mark.parametrize("w_dt,x_dt,off", KINDS)
def test_rows_of_n(gpu, M, K, N, group, w_dt, x_dt, off):
    _check(gpu, M, K, N, group, True, w_dt, x_dt, off)


def test_one_scale(gpu):
    m = gpu
    inp = cases.make_wq_inputs(m, 70, 2080, 1056, 3, m.ACL_FLOAT16, m.ACL_INT8, 0, False, True, None, per_tensor=True)
    _b16_bar(cases.run_wq_aclnn(m, inp, 70, 2080, 1056), cases.oracle_wq(m, inp, 70, 2080, 1056), orc.F16, "wide, one scale", 2080)
