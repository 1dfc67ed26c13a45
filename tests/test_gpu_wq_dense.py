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


@pytest.mark.parametrize("M,K,N,w_dt,x_dt,group,tW,off,bias", [(66, 16384, 33000, "i8", "bf16", 0, False, True, True), (300, 16384, 33003, "i4", "f16", 128, True, True, False),
                                                               (520, 16384, 34000, "i4", "bf16", 64, False, False, True)])
def test_column_strips(gpu, M, K, N, w_dt, x_dt, group, tW, off, bias):
    """A weight of more than 1 GiB in 16 bits goes in strips of whole 256 columns: the columns at both ends and on both sides of every
    place where a strip can end."""
    import numpy as np
    m = gpu
    xd, od = (m.ACL_FLOAT16, orc.F16) if x_dt == "f16" else (m.ACL_BF16, orc.BF16)
    inp = cases.make_wq_inputs(m, M, K, N, M, xd, m.ACL_INT4 if w_dt == "i4" else m.ACL_INT8, group, tW, off, xd if bias else None)
    print(f"case strips M={M} K={K} N={N} {w_dt} {x_dt} tW={tW}", flush=True)
    got = cases.run_wq_aclnn(m, inp, M, K, N)
    at = np.unique(np.concatenate([np.arange(0, 24), (np.arange(256, N - 1, 256)[:, None] + np.arange(-2, 2)).ravel(), np.arange(N - 25, N)]))
    at = np.unique(np.concatenate([at & ~1, at | 1]))   # whole pairs of columns
    at = at[at < N - N % 2]
    G = -(-K // group) if group else 1
    sub = dict(inp)
    if tW:
        sub["w"] = np.ascontiguousarray(inp["w"].reshape(N, -1)[at])
    elif w_dt == "i4":
        sub["w"] = np.ascontiguousarray(inp["w"].reshape(K, N // 2)[:, at[::2] // 2])
    else:
        sub["w"] = np.ascontiguousarray(inp["w"].reshape(K, N)[:, at])
    for k in ("scale", "offset"):
        if inp[k] is not None:
            v = inp[k].reshape((N, G) if tW else (G, N))
            sub[k] = np.ascontiguousarray(v[at] if tW else v[:, at])
    if bias:
        sub["bias"] = np.ascontiguousarray(inp["bias"][at])
    rows = np.linspace(0, M - 1, 40).astype(int)
    want = cases.oracle_wq(m, sub, M, K, len(at), rows=rows)
    _b16_bar(np.ascontiguousarray(got[rows][:, at]), want, od, "strips", K)


@pytest.mark.parametrize("M,K,N,w_dt,x_dt,group,tW,off,bias,segments", [
    (1158, 1728, 18043, "i4", "bf16", 64, True, False, True, 6), (1939, 2432, 11623, "i8", "f16", 0, True, False, False, 1),
    (2106, 2368, 10144, "i4", "f16", 128, False, True, True, 1), (1793, 1344, 11330, "i4", "bf16", 64, True, True, True, 1)])
def test_product_in_two_launches(gpu, M, K, N, w_dt, x_dt, group, tW, off, bias, segments):
    """The product's whole rounds of the chip and the rest apart: the first 17952 columns (the rest with K split) and 11264, the first 2048 rows
    and 1792 (the rest one row).  Two are estimated at 0.83 to 0.93 of the time of one, and taken below 0.95."""
    import numpy as np
    from test_gpu_routes import route
    m = gpu
    xd, od = (m.ACL_FLOAT16, orc.F16) if x_dt == "f16" else (m.ACL_BF16, orc.BF16)
    inp = cases.make_wq_inputs(m, M, K, N, M, xd, m.ACL_INT4 if w_dt == "i4" else m.ACL_INT8, group, tW, off, xd if bias else None)
    print(f"case two launches M={M} K={K} N={N} {w_dt} {x_dt} tW={tW}", flush=True)
    got = cases.run_wq_aclnn(m, inp, M, K, N)
    assert route(m) == ("wq_dense_two", segments), route(m)
    rows = np.unique(np.concatenate([np.linspace(0, M - 1, 24).astype(int), np.arange(256, M, 256) - 1, np.arange(256, M, 256), [M - 1]]))
    _b16_bar(np.ascontiguousarray(got[rows]), cases.oracle_wq(m, inp, M, K, N, rows=rows), od, "two launches", K)
