"""Weight-only calls with up to 64 rows against a weight in [K, N] storage, streamed as it lies (wq_kn.hip): the edges of its
row blocks (16, 32, 64), a ragged last strip of columns at every alignment, K of a few steps, K in segments, short last
groups, groups of 32 to K, one scale for the whole weight."""
import pytest

import cases
import oracle_api as orc
from test_gpu_shape_sweep import _b16_bar

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,K,N,group", [
    (1, 256, 256, 0), (16, 288, 258, 128), (17, 1024, 520, 64), (32, 4096, 1002, 128), (33, 2080, 384, 32), (64, 8192, 300, 128),
    (7, 4160, 2048, 128), (3, 18432, 1026, 0), (48, 3008, 4098, 64), (15, 11008, 770, 352), (9, 8192, 2064, 0),
])
@pytest.mark.parametrize("w_dt,x_dt,off", [("i4", "f16", True), ("i4", "bf16", False), ("i8", "f16", False), ("i8", "bf16", True)])
def test_kn_stream(gpu, M, K, N, group, w_dt, x_dt, off):
    m = gpu
    xd = m.ACL_FLOAT16 if x_dt == "f16" else m.ACL_BF16
    n = N + (1 if w_dt == "i8" and N % 16 == 2 else 0)   # (odd N with 8-bit weights)
    inp = cases.make_wq_inputs(m, M, K, n, M + K, xd, m.ACL_INT4 if w_dt == "i4" else m.ACL_INT8, group, False, off, xd if M % 2 else None)
    print(f"case kn M={M} K={K} N={n} g={group} {w_dt} {x_dt}", flush=True)
    _b16_bar(cases.run_wq_aclnn(m, inp, M, K, n), cases.oracle_wq(m, inp, M, K, n), orc.F16 if x_dt == "f16" else orc.BF16, "kn stream", K)


def test_kn_one_scale(gpu):
    m = gpu
    inp = cases.make_wq_inputs(m, 9, 512, 272, 3, m.ACL_FLOAT16, m.ACL_INT8, 0, False, True, None, per_tensor=True)
    _b16_bar(cases.run_wq_aclnn(m, inp, 9, 512, 272), cases.oracle_wq(m, inp, 9, 512, 272), orc.F16, "kn one scale", 512)


@pytest.mark.parametrize("M,K,N,w_dt", [(16, 1024, 512, "i4"), (1, 4096, 512, "i8"), (16, 4096, 1024, "i8")])
def test_small_weights_give_the_bits_of_their_k_contiguous_form(gpu, M, K, N, w_dt):
    import numpy as np
    m = gpu
    wd = m.ACL_INT4 if w_dt == "i4" else m.ACL_INT8
    inp = cases.make_wq_inputs(m, M, K, N, 5, m.ACL_BF16, wd, 0, False, False, None)
    w = inp["w"].reshape(K, -1)
    if w_dt == "i4":
        n = orc.unpack_nibbles(inp["w"]).reshape(K, N).T
        w = ((n[:, 0::2] & 15) | (n[:, 1::2] << 4)).astype(np.uint8)
    else:
        w = w.T
    other = dict(inp, w=np.ascontiguousarray(w), tW=True)
    assert np.array_equal(cases.run_wq_aclnn(m, inp, M, K, N), cases.run_wq_aclnn(m, other, M, K, N))


# groups of 32 against a wave's 13 steps: the table of scales is laid down again while the loop runs
@pytest.mark.parametrize("w_dt,x_dt,off", [("i4", "f16", True), ("i4", "bf16", False)])
def test_table_of_scales_in_several_windows(gpu, w_dt, x_dt, off):
    m = gpu
    M, K, N = 5, 16384, 12290
    xd = m.ACL_FLOAT16 if x_dt == "f16" else m.ACL_BF16
    inp = cases.make_wq_inputs(m, M, K, N, 11, xd, m.ACL_INT4, 32, False, off, None)
    print(f"case kn windows M={M} K={K} N={N} {x_dt}", flush=True)
    got = cases.run_wq_aclnn(m, inp, M, K, N)
    assert m.lib().opsnnDebugLastRoute(None) == b"wq_kn_table_w8"
    _b16_bar(got, cases.oracle_wq(m, inp, M, K, N), orc.F16 if x_dt == "f16" else orc.BF16, "kn windows", K)


@pytest.mark.parametrize("w_dt,x_dt,off", [("i4", "f16", True), ("i4", "bf16", False), ("i8", "bf16", True)])
@pytest.mark.parametrize("M,K,N,group", [(16, 6176, 28674, 128), (5, 6432, 28416, 0)])
def test_eight_waves(gpu, M, K, N, group, w_dt, x_dt, off):
    """An even count of segments with the table of scales: two segments a workgroup of eight waves; steps that are no multiple of the waves', a
    ragged last strip of columns."""
    from test_gpu_routes import route
    m = gpu
    xd = m.ACL_FLOAT16 if x_dt == "f16" else m.ACL_BF16
    inp = cases.make_wq_inputs(m, M, K, N, M + K, xd, m.ACL_INT4 if w_dt == "i4" else m.ACL_INT8, group, False, off, xd if M % 2 else None)
    print(f"case kn eight waves M={M} K={K} N={N} g={group} {w_dt} {x_dt}", flush=True)
    got = cases.run_wq_aclnn(m, inp, M, K, N)
    assert route(m) == ("wq_kn_table_w8", 2), route(m)
    _b16_bar(got, cases.oracle_wq(m, inp, M, K, N), orc.F16 if x_dt == "f16" else orc.BF16, "kn eight waves", K)


@pytest.mark.parametrize("M,x_dt,off,bias", [(16, "f16", True, True), (5, "bf16", False, True), (9, "bf16", True, False)])
def test_eight_waves_in_one_segment(gpu, M, x_dt, off, bias):
    """A plan of two segments is one workgroup of eight waves, which rounds and adds the bias itself; a ragged last strip of columns."""
    import numpy as np
    from test_gpu_routes import route
    m = gpu
    K, N = 3072, 44680
    xd = m.ACL_FLOAT16 if x_dt == "f16" else m.ACL_BF16
    inp = cases.make_wq_inputs(m, M, K, N, M, xd, m.ACL_INT4, 128, False, off, xd if bias else None)
    print(f"case kn eight waves, one segment M={M} K={K} N={N} {x_dt}", flush=True)
    got = cases.run_wq_aclnn(m, inp, M, K, N)
    assert route(m) == ("wq_kn_table_w8", 1), route(m)
    rows = np.array([0, M // 2, M - 1])
    _b16_bar(np.ascontiguousarray(got[rows]), cases.oracle_wq(m, inp, M, K, N, rows=rows), orc.F16 if x_dt == "f16" else orc.BF16, "kn eight waves, one segment", K)
