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
