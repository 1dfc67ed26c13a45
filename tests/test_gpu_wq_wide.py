"""Weight-only calls on the kernel whose workgroups stage 128 columns of the weight and the rows of x together (wq_wide.hip): the edges
of its row blocks (16, 32, 64, 128) and of several slabs, a last K tile of 32, 64 and 96, a ragged last strip of columns, groups of 32
to K with a short last one, more groups than one round of its table holds, one scale for the whole weight; both storages of the
weight.  The bar is the sweep's: one rounding of the output beside the sum of K products in fp32."""
import numpy as np
import pytest

import cases
import oracle_api as orc
from test_gpu_routes import route
from test_gpu_shape_sweep import _b16_bar

pytestmark = pytest.mark.gpu

KINDS = [("i4", "f16", True), ("i4", "bf16", False), ("i4", "bf16", True), ("i8", "f16", False), ("i8", "bf16", True)]
# what the estimates send to another kernel
ELSEWHERE = {(17, 2080, 4128) + k: "wq_kn" for k in KINDS}
ELSEWHERE.update({(17, 2080, 16416) + k: "wq_kn" for k in KINDS if k[1] == "bf16"})
ELSEWHERE.update({(1, 1056, 16416) + k: "wq_kn" for k in KINDS if k[1:] == ("bf16", True)})
ELSEWHERE.update({(1, 1056, 1024) + k: "wq_general" for k in KINDS if k[0] == "i8"})
ELSEWHERE.update({shape + k: "wq_general" for shape in [(1, 4128, 1064), (16, 4128, 1080)] for k in KINDS if k[0] == "i8"})
ELSEWHERE[(33, 8192, 1048, "i4", "bf16", False)] = "wq_kn"


def _check(m, M, K, N, group, nk, w_dt, x_dt, off):
    xd = m.ACL_FLOAT16 if x_dt == "f16" else m.ACL_BF16
    inp = cases.make_wq_inputs(m, M, K, N, M + K, xd, m.ACL_INT4 if w_dt == "i4" else m.ACL_INT8, group, nk, off, xd if M % 2 else None)
    print(f"case {'nk' if nk else 'kn'} M={M} K={K} N={N} g={group} {w_dt} {x_dt} off={off}", flush=True)
    got = cases.run_wq_aclnn(m, inp, M, K, N)
    assert route(m)[0] == ELSEWHERE.get((M, K, N, w_dt, x_dt, off), "wq_wide"), route(m)
    _b16_bar(got, cases.oracle_wq(m, inp, M, K, N), orc.F16 if x_dt == "f16" else orc.BF16, "wide", K)


@pytest.mark.parametrize("M,K,N,group", [
    (1, 1056, 1024, 32), (16, 16416, 1056, 128), (17, 2080, 4128, 64), (33, 8192, 1056, 128), (64, 4160, 2080, 0),
    (65, 1344, 1664, 64), (128, 1120, 1920, 256), (130, 2336, 1056, 128), (200, 1536, 1568, 0), (300, 4096, 544, 32), (900, 1056, 2080, 128),
    (1, 1056, 16416, 32), (17, 2080, 16416, 64), (40, 8192, 1056, 128),
])
@pytest.mark.parametrize("w_dt,x_dt,off", KINDS)
def test_rows_of_k(gpu, M, K, N, group, w_dt, x_dt, off):
    _check(gpu, M, K, N, group, False, w_dt, x_dt, off)


@pytest.mark.parametrize("M,K,N,group", [
    (1, 4128, 1064, 32), (16, 4128, 1080, 64), (33, 8192, 1048, 128), (64, 4160, 2088, 0), (65, 1344, 1672, 64), (96, 2080, 2124, 0),
    (130, 2336, 1068, 0), (300, 4096, 552, 32), (400, 2080, 4104, 128),
])
@pytest.mark.parametrize("w_dt,x_dt,off", KINDS)
def test_rows_of_k_in_whole_dwords(gpu, M, K, N, group, w_dt, x_dt, off):
    if w_dt == "i4" and N % 8 != 0:
        N += 4
    _check(gpu, M, K, N, group, False, w_dt, x_dt, off)


@pytest.mark.parametrize("M,K,N,group", [
    (9, 17280, 1873, 64), (20, 13568, 1730, 128), (40, 12544, 1793, 64), (64, 12928, 802, 32), (67, 14976, 1111, 128),
    (130, 8832, 1026, 0), (257, 7040, 1090, 128), (257, 3104, 1090, 128), (641, 1440, 5231, 32),
])
@pytest.mark.parametrize("w_dt,x_dt,off", KINDS)
def test_rows_of_n(gpu, M, K, N, group, w_dt, x_dt, off):
    _check(gpu, M, K, N, group, True, w_dt, x_dt, off)


def test_one_scale(gpu):
    m = gpu
    inp = cases.make_wq_inputs(m, 70, 2080, 1056, 3, m.ACL_FLOAT16, m.ACL_INT8, 0, False, True, None, per_tensor=True)
    got = cases.run_wq_aclnn(m, inp, 70, 2080, 1056)
    assert route(m)[0] == "wq_wide", route(m)
    _b16_bar(got, cases.oracle_wq(m, inp, 70, 2080, 1056), orc.F16, "wide, one scale", 2080)


def _tensors(m, inp, M, K, N, d, d_w_ptr, d_y):
    G = -(-K // inp["group"])
    st = (1, G) if inp["tW"] else None
    return (m.Tensor((M, K), inp["x_dt"], d["x"]), m.Tensor((K, N), inp["w_dt"], d_w_ptr, strides=(1, K) if inp["tW"] else None),
            m.Tensor((G, N), inp["x_dt"], d["scale"], strides=st), m.Tensor((G, N), inp["x_dt"], d["offset"], strides=st), m.Tensor((M, N), inp["x_dt"], d_y))


@pytest.mark.parametrize("M,K,N", [(40, 8192, 2048), (130, 4096, 1024)])
def test_cached_copy_of_the_other_storage(gpu, M, K, N):
    """[K, N] storage with the weight cache on: the call runs here on the K-contiguous copy, with that form's bits."""
    m = gpu
    print(f"case wide, cached copy M={M} K={K} N={N}", flush=True)
    inp = cases.make_wq_inputs(m, M, K, N, 3, m.ACL_FLOAT16, m.ACL_INT4, 128, False, True, None)
    w = orc.unpack_nibbles(inp["w"]).reshape(K, N).T & 15
    packed = dict(inp, w=np.ascontiguousarray((w[:, 0::2] | (w[:, 1::2] << 4)).astype(np.uint8)), tW=True,
                  scale=np.ascontiguousarray(inp["scale"].T), offset=np.ascontiguousarray(inp["offset"].T))
    want = cases.run_wq_aclnn(m, packed, M, K, N)
    assert route(m)[0] == "wq_wide"
    m.lib().opsnnSetWeightCache(256 << 20)
    try:
        d = {k: m.DeviceBuffer(host=v) for k, v in inp.items() if isinstance(v, np.ndarray)}
        d_y = m.DeviceBuffer(M * N * 2)
        for _ in range(2):   # (laid out, then found)
            d_y.fill(0xEE)
            x, tw, sc, off, y = _tensors(m, inp, M, K, N, d, d["w"], d_y)
            keep = m.weight_quant_batch_matmul(x, tw, sc, y, offset=off, group_size=128)
            m.check(m.lib().aclrtSynchronizeDevice(), "sync")
            assert route(m)[0] == "wq_wide"
            assert np.array_equal(d_y.to_host(np.uint16, (M, N)), want)
            del keep
    finally:
        m.lib().opsnnSetWeightCache(0)


@pytest.mark.parametrize("M,K,N", [(40, 8192, 1056), (130, 4096, 1056)])
@pytest.mark.parametrize("nk", [True, False])
def test_unaligned_weight_runs_elsewhere(gpu, M, K, N, nk):
    """Phase 1 does not look at the address: a weight that is not 16-byte aligned goes to the kernels behind this one, in the workspace
    that the plan asked for."""
    m = gpu
    print(f"case wide, unaligned weight M={M} K={K} N={N} nk={nk}", flush=True)
    inp = cases.make_wq_inputs(m, M, K, N, 3, m.ACL_FLOAT16, m.ACL_INT4, 128, nk, True, None)
    cases.run_wq_aclnn(m, inp, M, K, N)
    assert route(m)[0] == "wq_wide"
    d = {k: m.DeviceBuffer(host=v) for k, v in inp.items() if isinstance(v, np.ndarray) and k != "w"}
    d_w = m.DeviceBuffer(host=np.concatenate([np.zeros(8, np.uint8), inp["w"].reshape(-1).view(np.uint8)]))
    d_y = m.DeviceBuffer(M * N * 2)
    x, tw, sc, off, y = _tensors(m, inp, M, K, N, d, d_w.ptr + 8, d_y)
    rc, ws, ex = m.weight_quant_batch_matmul_get_workspace(x, tw, sc, y, offset=off, group_size=128)
    assert rc == 0, m.err_msg()
    guard = 1 << 22
    buf = m.DeviceBuffer(ws + guard)
    buf.fill(0xA5)
    m.check(m.lib().aclnnWeightQuantBatchMatmulV2(buf.ptr, ws, ex, None), "aclnnWeightQuantBatchMatmulV2")
    m.check(m.lib().aclrtSynchronizeDevice(), "sync")
    assert route(m)[0] != "wq_wide"
    assert (buf.to_host(np.uint8, (ws + guard,))[ws:] == 0xA5).all()
    _b16_bar(d_y.to_host(np.uint16, (M, N)), cases.oracle_wq(m, inp, M, K, N), orc.F16, "unaligned weight", K)


@pytest.mark.parametrize("M,K,N,group,nk", [(40, 8192, 1056, 128, False), (1, 1056, 1024, 32, False), (40, 12544, 1793, 64, True), (130, 8832, 1026, 0, True)])
def test_scales_at_the_end_of_the_range(gpu, M, K, N, group, nk):
    """bf16 x int4 without offsets converts by way of w + 8, which is exact while eight scales are a number: an infinite, a NaN and a
    scale of 2^126 in one column each, and in a workgroup without them nothing changes."""
    m = gpu
    print(f"case wide, large scales M={M} K={K} N={N} nk={nk}", flush=True)
    inp = cases.make_wq_inputs(m, M, K, N, 5, m.ACL_BF16, m.ACL_INT4, group, nk, False, None)
    inp["x"] = orc.f32_to_b16(np.abs(orc.b16_to_f32(inp["x"], orc.BF16)) * np.float32(2.0 ** -20), orc.BF16)
    codes = orc.unpack_nibbles(inp["w"]).reshape((N, K) if nk else (K, N)) & 15
    scale = inp["scale"].reshape((N, -1) if nk else (-1, N))
    for col, s in ((3, np.inf), (N // 2, np.nan), (N - 2, 2.0 ** 126), (N - 1, -np.inf)):
        c = np.random.default_rng(col).integers(1, 4, K).astype(codes.dtype)
        (codes[col] if nk else codes[:, col])[...] = c
        (scale[col] if nk else scale[:, col])[...] = orc.f32_to_b16(np.array([s], np.float32), orc.BF16)[0]
    inp["w"], inp["scale"] = orc.pack_nibbles(codes.astype(np.uint8)), np.ascontiguousarray(scale.reshape(inp["scale"].shape))
    got, want = cases.run_wq_aclnn(m, inp, M, K, N), cases.oracle_wq(m, inp, M, K, N)
    assert route(m)[0] == "wq_wide", route(m)
    g, w = orc.b16_to_f32(got, orc.BF16), orc.b16_to_f32(want, orc.BF16)
    assert np.array_equal(np.isnan(g), np.isnan(w)) and np.array_equal(np.isinf(g), np.isinf(w)) and np.isinf(w[:, 3]).all() and np.isnan(w[:, N // 2]).all()
    assert np.array_equal(np.sign(g[np.isinf(w)]), np.sign(w[np.isinf(w)])) and np.isfinite(w[:, N - 2]).all()
    rest = np.isfinite(w).all(axis=0)
    rest[N - 2] = False
    _b16_bar(np.ascontiguousarray(got[:, rest]), np.ascontiguousarray(want[:, rest]), orc.BF16, "wide, other columns", K)
    assert np.abs(g[:, N - 2] / w[:, N - 2] - 1).max() <= 2.0 ** -7


@pytest.mark.parametrize("x_dt,off", [("bf16", False), ("f16", True)])
def test_table_of_scales_as_large_as_the_lds_has_room_for(gpu, x_dt, off):
    """79 groups of 128 and one that a segment could begin in: the table of 80 fills the LDS beside the ring, K in one piece."""
    m = gpu
    M, K, N = 212, 10112, 12096
    xd = m.ACL_FLOAT16 if x_dt == "f16" else m.ACL_BF16
    inp = cases.make_wq_inputs(m, M, K, N, 7, xd, m.ACL_INT4, 128, False, off, None)
    print(f"case wide, full table M={M} K={K} N={N} {x_dt} off={off}", flush=True)
    got = cases.run_wq_aclnn(m, inp, M, K, N)
    assert route(m) == ("wq_wide", 1), route(m)
    rows = np.array([0, 63, 64, 127, 128, 211])
    _b16_bar(np.ascontiguousarray(got[rows]), cases.oracle_wq(m, inp, M, K, N, rows=rows), orc.F16 if x_dt == "f16" else orc.BF16, "full table", K)
