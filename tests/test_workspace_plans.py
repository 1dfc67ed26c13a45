"""The workspace that phase 1 reports against what phase 2 plans with: where a call's operand lies at another address in phase 2
(a FRACTAL_NZ weight is laid out in the workspace first), both phases have to come to the same plan.  Host only: phase 1 and
the workspace query look at addresses, never at data."""
import ctypes as C
import random

import pytest

import opsnn as m

ALIGNED, ODD = 1 << 20, (1 << 20) + 4


def _wq_args(M, N, K, group, wbits, x_dt, w_ptr, nk=True, ws=None):
    a = m.OpsnnWqmmArgs()
    a.M, a.N, a.K = M, N, K
    a.x, a.x_dtype = ALIGNED, x_dt
    a.w.ptr = w_ptr
    a.w.row_stride, a.w.col_stride = (1, K) if nk else (N, 1)
    a.w_dtype = m.ACL_INT4 if wbits == 4 else m.ACL_INT8
    G = -(-K // group) if group else 1
    a.scale.ptr, a.scale_dtype, a.scale_n = ALIGNED, x_dt, N
    a.scale.row_stride, a.scale.col_stride = ((1, G) if nk else (N, 1)) if G > 1 else (0, 1)
    a.group, a.y = group, ALIGNED
    return a


def _wq_shapes(n):
    rng = random.Random(5)
    yield 8, 4096, 10240, 64, 4   # 3 slices planned for one address, 10 for the other
    for _ in range(n):
        K = rng.randrange(8, 700) * 32
        yield rng.choice([1, 3, 16, 17, 40, 64, 65, 300]), rng.randrange(64, 9000), K, rng.choice([g for g in (0, 32, 64, 96, 128) if g < K]), rng.choice([4, 8])


@pytest.mark.parametrize("nk", [True, False])
def test_weight_only_plan_does_not_depend_on_the_weights_address(nk):
    for M, N, K, group, wbits in _wq_shapes(600):
        N += N % 2
        for x_dt in (m.ACL_FLOAT16, m.ACL_BF16):
            want = m.lib().opsnnWqmmWorkspace(C.byref(_wq_args(M, N, K, group, wbits, x_dt, ALIGNED, nk)))
            for ptr in (ODD, ALIGNED + 8, ALIGNED + 1):
                assert m.lib().opsnnWqmmWorkspace(C.byref(_wq_args(M, N, K, group, wbits, x_dt, ptr, nk))) == want, (M, N, K, group, wbits, ptr)


def _nz_workspace(x_dt, M, N, K, group, wbits, w_ptr):
    G = -(-K // group) if group else 1
    w_dt, c0e = (m.ACL_INT4, 16) if wbits == 4 else (m.ACL_INT8, 32)
    x, y = m.Tensor((M, K), x_dt, ALIGNED), m.Tensor((M, N), x_dt, ALIGNED)
    w = m.Tensor((K, N), w_dt, w_ptr, strides=(1, K), fmt=m.ACL_FORMAT_FRACTAL_NZ, storage_shape=(-(-K // c0e), -(-N // 16), 16, c0e))
    sc = m.Tensor((G, N), x_dt, ALIGNED, strides=(1, G)) if group else m.Tensor((N,), x_dt, ALIGNED)
    rc, ws, ex = m.weight_quant_batch_matmul_get_workspace(x, w, sc, y, group_size=group, weight_nz=True)
    assert rc == 0, m.err_msg()
    m.lib().aclDestroyAclOpExecutor(ex)
    return ws


def test_nz_weight_reserves_what_its_nd_copy_needs():
    """The ND copy sits at the front of the workspace, 16-byte aligned: phase 1 has to reserve at least what the ND call at such
    an address plans, wherever the NZ weight itself lies."""
    for M, N, K, group, wbits in _wq_shapes(200):
        nd = m.lib().opsnnWqmmWorkspace(C.byref(_wq_args(M, N, K, group, wbits, m.ACL_FLOAT16, ALIGNED)))
        front = -(-(N * K * wbits // 8) // 256) * 256
        for ptr in (ALIGNED, ODD):
            assert _nz_workspace(m.ACL_FLOAT16, M, N, K, group, wbits, ptr) >= front + nd, (M, N, K, group, wbits, ptr)


@pytest.mark.gpu
@pytest.mark.parametrize("M,K,N,group", [(8, 10240, 512, 64), (16, 4160, 257, 128), (33, 1088, 520, 128)])
def test_nz_weight_at_an_unaligned_address_stays_inside_the_workspace(gpu, M, K, N, group):
    import numpy as np

    import cases
    from test_nz_entry_points import nd_to_nz
    inp = cases.make_wq_inputs(m, M, K, N, 3, m.ACL_FLOAT16, m.ACL_INT4, group, True, False, None)
    want = cases.run_wq_aclnn(m, inp, M, K, N)
    nz = nd_to_nz(inp["w"].reshape(N, -1).view(np.uint8), 8)
    d = {k: m.DeviceBuffer(host=v) for k, v in inp.items() if isinstance(v, np.ndarray) and k != "w"}
    d_w = m.DeviceBuffer(host=np.concatenate([np.zeros(4, np.uint8), nz.reshape(-1)]))
    G, d_y = -(-K // group), m.DeviceBuffer(M * N * 2)
    w = m.Tensor((K, N), m.ACL_INT4, d_w.ptr + 4, strides=(1, K), fmt=m.ACL_FORMAT_FRACTAL_NZ, storage_shape=nz.shape[:2] + (16, 16))
    rc, ws, ex = m.weight_quant_batch_matmul_get_workspace(m.Tensor((M, K), m.ACL_FLOAT16, d["x"]), w,
                                                           m.Tensor((G, N), m.ACL_FLOAT16, d["scale"], strides=(1, G)),
                                                           m.Tensor((M, N), m.ACL_FLOAT16, d_y), group_size=group, weight_nz=True)
    assert rc == 0, m.err_msg()
    guard = 1 << 22   # (more than the second plan's slices would take)
    buf = m.DeviceBuffer(ws + guard)
    buf.fill(0xA5)
    print(f"case nz unaligned M={M} K={K} N={N} g={group}", flush=True)
    m.check(m.lib().aclnnWeightQuantBatchMatmulNz(buf.ptr, ws, ex, None), "aclnnWeightQuantBatchMatmulNz")
    m.check(m.lib().aclrtSynchronizeDevice(), "sync")
    assert np.array_equal(d_y.to_host(np.uint16, (M, N)), want)
    assert (buf.to_host(np.uint8, (ws + guard,))[ws:] == 0xA5).all()


def _v5_nz_call(mode, M, N, K, x2_ptr, nk):
    """Phase 1 of aclnnQuantMatmulWeightNz: (status, workspace)."""
    four = mode in ("mxfp4", "a8w4")
    x1_dt, x2_dt = {"int8": (m.ACL_INT8, m.ACL_INT8), "mxfp4": (m.ACL_FLOAT4_E2M1,) * 2,
                    "a8w4": (m.ACL_FLOAT8_E4M3FN, m.ACL_FLOAT4_E2M1)}.get(mode, (m.ACL_FLOAT8_E4M3FN,) * 2)
    c0e, cols, rows = 32, K if nk else N, N if nk else K
    x1 = m.Tensor((M, K), x1_dt, ALIGNED)
    x2 = m.Tensor((K, N), x2_dt, x2_ptr, strides=(1, K) if nk else None, fmt=m.ACL_FORMAT_FRACTAL_NZ,
                  storage_shape=(-(-cols // c0e), -(-rows // 16), 16, c0e))
    out = m.Tensor((M, N), m.ACL_BF16, ALIGNED)
    kw = {}
    if mode in ("int8", "fp8_token"):
        s1, s2 = m.Tensor((M,), m.ACL_FLOAT, ALIGNED), m.Tensor((N,), m.ACL_FLOAT, ALIGNED)
    elif mode == "fp8_block":
        KB, NB = -(-K // 128), -(-N // 128)
        s1, s2 = m.Tensor((M, KB), m.ACL_FLOAT, ALIGNED), m.Tensor((KB, NB), m.ACL_FLOAT, ALIGNED, strides=(1, KB) if nk else None)
        kw["group_size"] = (1 << 32) | (128 << 16) | 128
    else:
        KS = -(-K // 64)
        s1 = m.Tensor((M, KS, 2), m.ACL_FLOAT8_E8M0, ALIGNED)
        s2 = m.Tensor((KS, N, 2), m.ACL_FLOAT8_E8M0, ALIGNED, strides=(2, KS * 2, 1) if nk else None)
        kw["group_size"] = (1 << 32) | (1 << 16) | 32
    rc, ws, ex = m.quant_matmul_v5_get_workspace(x1, x2, s1, s2, out, weight_nz=True, **kw)
    if ex:
        m.lib().aclDestroyAclOpExecutor(ex)
    return rc, ws


@pytest.mark.parametrize("mode", ["int8", "fp8_token", "fp8_block", "mxfp4", "mxfp8", "a8w4"])
def test_quant_matmul_nz_plan_does_not_depend_on_the_nz_address(mode):
    """(MXFP4 with K % 128 == 64 and a K split: the padded copies were planned only for an aligned NZ address, and written in
    phase 2, where the ND copy is aligned, all the same.)"""
    rng = random.Random(9)
    taken = 0
    for i in range(300):
        M, N, K = rng.choice([1, 16, 20, 33, 64, 128, 300]), rng.randrange(16, 600) * 16, rng.randrange(8, 160) * 64
        if i == 0:
            M, N, K = 64, 1024, 8256
        nk = rng.random() < 0.7
        rc, want = _v5_nz_call(mode, M, N, K, ALIGNED, nk)
        if rc != 0:
            continue
        taken += 1
        for ptr in (ODD, ALIGNED + 8):
            assert _v5_nz_call(mode, M, N, K, ptr, nk) == (0, want), (M, N, K, nk, ptr)
    assert taken > 50, m.err_msg()


@pytest.mark.gpu
@pytest.mark.parametrize("mode,M,K,N", [("mxfp4", 64, 8256, 1024), ("int8", 64, 8192, 512), ("int8", 64, 8192, 500)])
@pytest.mark.parametrize("x2_off,ws_off", [(4, 0), (0, 4), (8, 8)])
def test_quant_matmul_nz_stays_inside_the_workspace(gpu, mode, M, K, N, x2_off, ws_off):
    """NZ operands and workspaces at addresses that are not 16-byte aligned."""
    import numpy as np

    import cases
    import oracle_api as orc
    from test_gpu_shape_sweep import _b16_bar
    from test_nz_entry_points import nd_to_nz
    if mode == "int8":
        inp = cases.make_qmm_int8_inputs(m, M, K, N, 3, m.ACL_BF16, True)
        want, dt, c0 = cases.run_qmm_int8_aclnn(m, inp, M, K, N, True, m.ACL_BF16)[0], m.ACL_INT8, 32
        nz = nd_to_nz(inp["x2"][0].view(np.uint8), c0)
    else:
        inp = cases.make_mx_inputs(m, M, K, N, 3, True, True)
        want, dt, c0 = cases.run_mx_aclnn(m, inp, M, K, N, True, m.ACL_BF16)[0], m.ACL_FLOAT4_E2M1, 16
        nz = nd_to_nz(inp["x2"][0].view(np.uint8).reshape(N, K // 2), c0)
    d = {k: m.DeviceBuffer(host=v) for k, v in inp.items() if isinstance(v, np.ndarray) and k != "x2"}
    d_x2 = m.DeviceBuffer(host=np.concatenate([np.zeros(x2_off, np.uint8), nz.reshape(-1)]))
    d_out = m.DeviceBuffer(M * N * 2)
    x1 = m.Tensor((M, K), dt, d["x1"])
    x2 = m.Tensor((N, K), dt, d_x2.ptr + x2_off, fmt=m.ACL_FORMAT_FRACTAL_NZ, storage_shape=nz.shape[:2] + (16, 32))
    kw = {}
    if mode == "int8":
        s1, s2 = m.Tensor((M,), m.ACL_FLOAT, d["s1"]), m.Tensor((N,), m.ACL_FLOAT, d["s2"])
        kw["bias"] = m.Tensor((N,), m.ACL_BF16, d["bias"])
    else:
        s1, s2 = m.Tensor(inp["s1"].shape[1:], m.ACL_FLOAT8_E8M0, d["s1"]), m.Tensor(inp["s2"].shape[1:], m.ACL_FLOAT8_E8M0, d["s2"])
        kw["group_size"] = (1 << 32) | (1 << 16) | 32
    rc, ws, ex = m.quant_matmul_v5_get_workspace(x1, x2, s1, s2, m.Tensor((M, N), m.ACL_BF16, d_out), transpose_x2=True, weight_nz=True, **kw)
    assert rc == 0, m.err_msg()
    guard = (M + N) * K + 4096   # (more than padded copies of both operands would take)
    buf = m.DeviceBuffer(ws_off + ws + guard)
    buf.fill(0xA5)
    print(f"case nz {mode} M={M} K={K} N={N} x2 +{x2_off} workspace +{ws_off}", flush=True)
    m.check(m.lib().aclnnQuantMatmulWeightNz(buf.ptr + ws_off, ws, ex, None), "aclnnQuantMatmulWeightNz")
    m.check(m.lib().aclrtSynchronizeDevice(), "sync")
    got = d_out.to_host(np.uint16, (M, N))
    if mode == "int8":
        assert np.array_equal(got, want)
    else:
        _b16_bar(got, want, orc.BF16, "mxfp4 nz", K)
    after = buf.to_host(np.uint8, (ws_off + ws + guard,))
    assert (after[:ws_off] == 0xA5).all() and (after[ws_off + ws:] == 0xA5).all()


def test_kn_storage_leaves_room_for_the_cached_copys_k_split():
    """[K, N] storage with more than 64 rows: whether the weight cache serves the call is only known in phase 2, so the workspace
    holds what the K-contiguous form asks for as well."""
    for M, N, K, group, wbits in _wq_shapes(400):
        M, N = M + 64, N + N % 2
        nk = m.lib().opsnnWqmmWorkspace(C.byref(_wq_args(M, N, K, group, wbits, m.ACL_FLOAT16, ALIGNED, True)))
        assert m.lib().opsnnWqmmWorkspace(C.byref(_wq_args(M, N, K, group, wbits, m.ACL_FLOAT16, ALIGNED, False))) >= nk, (M, N, K, group, wbits)


@pytest.mark.parametrize("nk", [True, False])
def test_dequantised_weight_is_bounded(nk):
    """The 16-bit weight that many rows are multiplied with takes 1 GiB of workspace at most (beside a K split's partial sums)."""
    for M, N, K in ((600, 152064, 8192), (2048, 57344, 8192), (300, 70000, 8192), (65, 1 << 20, 1024)):
        ws = m.lib().opsnnWqmmWorkspace(C.byref(_wq_args(M, N, K, 64, 4, m.ACL_BF16, ALIGNED, nk)))
        assert 0 < ws <= (1 << 30) + 256 * K * 2 + 16 * 4 * M * min(N, (1 << 30) // (2 * K) + 256), (M, N, K, ws)
