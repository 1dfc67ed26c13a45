"""Weight-only calls with many rows: the weight dequantised once into the workspace, then a dense 16-bit product (wq_dense.hip,
gemm16.hip).  The shapes sit at the edges of that route: [K, N] storage with a ragged last block of columns, N of every
alignment, K of one and of several 64-element tiles, groups of 64 and a short last group, the 128 x 128 tiles with and without
a K split and the four-wave kernel."""
import pytest

import cases
import oracle_api as orc
from test_gpu_shape_sweep import _b16_bar

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,K,N,group,tW", [
    (65, 64, 129, 0, False), (70, 192, 1001, 0, True), (130, 320, 1002, 64, False), (129, 704, 257, 64, True),
    (257, 1088, 520, 128, False), (300, 4160, 300, 128, True), (200, 6208, 136, 64, False), (77, 448, 2056, 128, False),
    (513, 4096, 7944, 128, True), (1030, 1024, 2827, 64, True),
])
@pytest.mark.parametrize("w_dt,x_dt,off", [("i4", "f16", True), ("i4", "bf16", False), ("i8", "f16", False), ("i8", "bf16", True)])
def test_dense_route(gpu, M, K, N, group, tW, w_dt, x_dt, off):
    m = gpu
    if w_dt == "i4" and not tW and N % 2:
        N += 1
    xd = m.ACL_FLOAT16 if x_dt == "f16" else m.ACL_BF16
    inp = cases.make_wq_inputs(m, M, K, N, M + K + N, xd, m.ACL_INT4 if w_dt == "i4" else m.ACL_INT8, group if group < K else 0, tW, off,
                               xd if M % 2 else None)
    print(f"case dense M={M} K={K} N={N} g={group} tW={tW} {w_dt} {x_dt}", flush=True)
    got = cases.run_wq_aclnn(m, inp, M, K, N)
    _b16_bar(got, cases.oracle_wq(m, inp, M, K, N), orc.F16 if x_dt == "f16" else orc.BF16, "dense route", K)


def test_more_columns_than_a_grid_dimension_holds(gpu):
    """262152 columns: the pass over the weight has them on grid.x (four per workgroup on grid.y would be 65538)."""
    m = gpu
    M, K, N = 65, 64, 262152
    inp = cases.make_wq_inputs(m, M, K, N, 9, m.ACL_FLOAT16, m.ACL_INT4, 0, True, False, None)
    print(f"case dense M={M} K={K} N={N}", flush=True)
    _b16_bar(cases.run_wq_aclnn(m, inp, M, K, N), cases.oracle_wq(m, inp, M, K, N), orc.F16, "dense, wide", K)
