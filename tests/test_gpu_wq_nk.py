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


@pytest.mark.parametrize("M,K,N,group,w_dt", [(7, 4160, 300, 64, "i4"), (20, 4160, 257, 64, "i4"), (40, 1056, 520, 32, "i4"), (5, 288, 256, 0, "i8"), (50, 2080, 300, 32, "i8")])
@pytest.mark.parametrize("x_dt", ["f16", "bf16"])
def test_infinite_weights_in_the_last_piece(gpu, M, K, N, group, w_dt, x_dt):
    """A K that ends inside a chunk: the lanes past its end repeat the last piece and must add nothing, also where its
    dequantised weights are infinite (an infinite scale; in fp16 also a product past 65504)."""
    import numpy as np
    m = gpu
    xd, od = (m.ACL_FLOAT16, orc.F16) if x_dt == "f16" else (m.ACL_BF16, orc.BF16)
    inp = cases.make_wq_inputs(m, M, K, N, M + K, xd, m.ACL_INT4 if w_dt == "i4" else m.ACL_INT8, group, True, False, None)
    last, hot = K - (group or K), [3, 17, N - 1]          # the last group of three columns: codes 1, x positive, so the sum is +inf
    xf = orc.b16_to_f32(inp["x"], od)
    inp["x"] = orc.f32_to_b16(np.where(np.arange(K) >= last, np.abs(xf) + 0.25, xf).astype(np.float32), xd)
    if w_dt == "i4":
        inp["w"].reshape(N, K // 2)[hot, last // 2:] = 0x11
    else:
        inp["w"].reshape(N, K)[hot, last:] = 1
    sc = orc.b16_to_f32(inp["scale"], od).reshape(N, -1)
    sc[hot, -1] = [np.inf, 60000.0, np.inf]
    if w_dt == "i4":
        inp["w"].reshape(N, K // 2)[17, last // 2:] = 0x77   # 7 * 60000: infinite in fp16
    else:
        inp["w"].reshape(N, K)[17, last:] = 100
    inp["scale"] = orc.f32_to_b16(sc.astype(np.float32), xd).reshape(inp["scale"].shape)
    print(f"case nk infinite M={M} K={K} N={N} g={group} {w_dt} {x_dt}", flush=True)
    got = orc.b16_to_f32(cases.run_wq_aclnn(m, inp, M, K, N), od)
    want = orc.b16_to_f32(cases.oracle_wq(m, inp, M, K, N), od)
    assert np.isinf(want[:, [3, N - 1]]).all()
    assert np.array_equal(np.isnan(got), np.isnan(want)) and np.array_equal(np.isinf(got), np.isinf(want))
    keep = np.isfinite(want)
    assert np.mean(np.abs(got[keep] - want[keep])) <= 2.0 ** -8 * np.mean(np.abs(want[keep]))
