"""Weight-only calls with up to 64 rows against a weight in [N, K] storage of any shape (wq_nk.hip): the edges of its row blocks,
the last 128 columns of an N of every alignment, K with a partly filled last chunk, K in segments, groups of 32 and 64, groups
that are no power of two, short last groups."""
import pytest

import cases
import oracle_api as orc
from test_gpu_shape_sweep import _b16_bar

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,K,N,group", [
    (1, 288, 256, 64), (16, 4160, 257, 128), (17, 5632, 1453, 64), (32, 1088, 520, 128), (33, 2080, 385, 32), (64, 4160, 301, 64),
    (7, 16448, 640, 128), (3, 1024, 1026, 64), (48, 3008, 4099, 96), (15, 11040, 770, 352),
])
@pytest.mark.parametrize("w_dt,x_dt,off", [("i4", "f16", True), ("i4", "bf16", False), ("i8", "f16", False), ("i8", "bf16", True)])
def test_nk_stream(gpu, M, K, N, group, w_dt, x_dt, off):
    m = gpu
    xd = m.ACL_FLOAT16 if x_dt == "f16" else m.ACL_BF16
    inp = cases.make_wq_inputs(m, M, K, N, M + K, xd, m.ACL_INT4 if w_dt == "i4" else m.ACL_INT8, group, True, off, xd if M % 2 else None)
    print(f"case nk M={M} K={K} N={N} g={group} {w_dt} {x_dt}", flush=True)
    _b16_bar(cases.run_wq_aclnn(m, inp, M, K, N), cases.oracle_wq(m, inp, M, K, N), orc.F16 if x_dt == "f16" else orc.BF16, "nk stream", K)
