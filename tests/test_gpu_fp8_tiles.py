"""The tiles of the exact fp8 kernel (fp8x_plan): each, pinned, gives the bits of the 256 x 128 one -- a row more and less than a
tile, ragged N with one and with two scale blocks in the last tile, fewer K tiles than stages -- and that one is held to the
oracle by the mode's own tests; shapes that the plan cuts along K against the oracle."""
import ctypes as C

import numpy as np
import pytest

import cases
import oracle_api as orc
from test_gpu_shape_sweep import _b16_bar

pytestmark = pytest.mark.gpu

TILES = (32, 33, 34)   # OPSNN_VARIANT_FP8X_256x128, _128x256, _128x128


@pytest.mark.parametrize("M,K,N", [(129, 128, 257), (300, 256, 390), (257, 384, 128), (128, 1152, 1001), (511, 640, 520), (140, 896, 384)])
@pytest.mark.parametrize("mode", ["rowcol", "block", "mx"])
def test_each_tile_gives_the_same_bits(gpu, mode, M, K, N):
    m = gpu
    print(f"case fp8 tiles {mode} M={M} K={K} N={N}", flush=True)
    rng = np.random.default_rng(M + K + N)
    x1, x2 = cases.gen_fp8(rng, (M, K)), cases.gen_fp8(rng, (N, K))
    NB, KB = (N + 127) // 128, K // 128
    a = m.OpsnnQmmArgs()
    a.M, a.N, a.K, a.batch = M, N, K, 1
    if mode == "rowcol":
        s1, s2 = rng.uniform(0.5, 2, M).astype(np.float32), rng.uniform(0.5, 2, N).astype(np.float32)
    elif mode == "block":
        s1, s2 = rng.uniform(0.5, 2, (M, KB)).astype(np.float32), rng.uniform(0.5, 2, (NB, KB)).astype(np.float32)
    else:
        s1, s2 = rng.integers(120, 130, (M, K // 32)).astype(np.uint8), rng.integers(120, 130, (N, K // 32)).astype(np.uint8)
    d1, d2, ds1, ds2 = (m.DeviceBuffer(host=v) for v in (x1, x2, s1, s2))
    a.x1, a.x2 = m.OpsnnMat(d1.ptr, K, 1, 0), m.OpsnnMat(d2.ptr, 1, K, 0)
    a.x1_dtype = a.x2_dtype = m.ACL_FLOAT8_E4M3FN
    if mode == "rowcol":
        a.x1_scale, a.x1_scale_len, a.x2_scale, a.x2_scale_dtype, a.x2_scale_len = ds1.ptr, M, ds2.ptr, m.ACL_FLOAT, N
    elif mode == "block":
        a.gsM, a.gsN, a.gsK = 1, 128, 128
        a.x1_scale_mat, a.x2_scale_mat = m.OpsnnMat(ds1.ptr, KB, 1, 0), m.OpsnnMat(ds2.ptr, 1, KB, 0)
    else:
        a.gsM, a.gsN, a.gsK = 1, 1, 32
        a.x1_scale_mat, a.x2_scale_mat = m.OpsnnMat(ds1.ptr, K // 32, 2, 0), m.OpsnnMat(ds2.ptr, K // 32, 2, 0)
    call = {"rowcol": m.lib().opsnnQmmTc, "block": m.lib().opsnnQmmBlockScale, "mx": m.lib().opsnnQmmMx}[mode]
    outs = []
    for tile in TILES:
        d_out = cases.guarded_out(m, M * N * 2)
        a.out, a.out_dtype, a.force_variant = d_out.ptr, m.ACL_BF16, tile
        assert call(C.byref(a), None) == 0
        m.check(m.lib().aclrtSynchronizeDevice(), "sync")
        outs.append(d_out.to_host(np.uint16, (M, N)))
    assert np.array_equal(outs[1], outs[0]) and np.array_equal(outs[2], outs[0])


@pytest.mark.parametrize("M,K,N", [(200, 7168, 520), (333, 4096, 1030), (130, 16384, 256)])
def test_planned_block_scale_shapes(gpu, M, K, N):
    m = gpu
    print(f"case fp8 block planned M={M} K={K} N={N}", flush=True)
    inp = cases.make_blockscale_inputs(m, M, K, N, M + N, True)
    _b16_bar(cases.run_blockscale_aclnn(m, inp, M, K, N, True, m.ACL_BF16), cases.oracle_blockscale(m, inp, M, K, N, True, m.ACL_BF16), orc.BF16, "planned tiles", K)


@pytest.mark.parametrize("M,K,N", [(193, 384, 257), (191, 128, 390), (383, 1152, 1001), (65, 256, 129), (449, 640, 520)])
@pytest.mark.parametrize("mode", ["rowcol", "block", "mx"])
def test_tiles_of_192_and_64_rows(gpu, monkeypatch, mode, M, K, N):
    """OPSNN_VARIANT_FP8X_192x128 and _64x256, as above."""
    monkeypatch.setitem(globals(), "TILES", (32, 35, 36))
    test_each_tile_gives_the_same_bits(gpu, mode, M, K, N)


@pytest.mark.parametrize("N,shift", [(264, 2), (263, 0), (261, 6)])
def test_rows_of_the_output_at_any_address(gpu, N, shift):
    """The output at an address that is no multiple of 16, in whole and in ragged rows: the bits of the aligned, whole-row call, and nothing
    beside them."""
    m = gpu
    M, K = 131, 256
    rng = np.random.default_rng(N)
    x1, x2 = cases.gen_fp8(rng, (M, K)), cases.gen_fp8(rng, (264, K))
    s1, s2 = rng.uniform(0.5, 2, M).astype(np.float32), rng.uniform(0.5, 2, 264).astype(np.float32)
    d1, d2, ds1, ds2 = (m.DeviceBuffer(host=v) for v in (x1, x2, s1, s2))
    outs = []
    for n, off in ((264, 0), (N, shift)):
        a = m.OpsnnQmmArgs()
        a.M, a.N, a.K, a.batch = M, n, K, 1
        a.x1, a.x2 = m.OpsnnMat(d1.ptr, K, 1, 0), m.OpsnnMat(d2.ptr, 1, K, 0)
        a.x1_dtype = a.x2_dtype = m.ACL_FLOAT8_E4M3FN
        a.x1_scale, a.x1_scale_len, a.x2_scale, a.x2_scale_dtype, a.x2_scale_len = ds1.ptr, M, ds2.ptr, m.ACL_FLOAT, n
        host = np.full(M * n + 64, 0x5a5a, np.uint16)
        d_out = m.DeviceBuffer(host=host)
        a.out, a.out_dtype, a.force_variant = d_out.ptr + 32 + off, m.ACL_BF16, 32
        print(f"case fp8 out N={n} shift={off}", flush=True)
        assert m.lib().opsnnQmmTc(C.byref(a), None) == 0
        m.check(m.lib().aclrtSynchronizeDevice(), "sync")
        got = d_out.to_host(np.uint16, (M * n + 64,))
        at = 16 + off // 2
        assert (got[:at] == 0x5a5a).all() and (got[at + M * n:] == 0x5a5a).all()
        outs.append(got[at:at + M * n].reshape(M, n))
    assert np.array_equal(outs[1], outs[0][:, :N])
