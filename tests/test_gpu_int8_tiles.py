"""int8 per-token x per-channel calls whose 256 x 256 tiles do not fill the chip (tile_plan): each of their tiles, pinned, at
its edges -- one row, a row more and less than a tile, ragged N, fewer K tiles than stages, a K that ends inside a tile -- and
shapes that the plan cuts along K.  Integer sums: bit-identical to the oracle."""
import ctypes as C

import numpy as np
import pytest

import cases
import oracle_api as orc
from test_gpu_routes import route

pytestmark = pytest.mark.gpu

TILES = {"32x64": 12, "64x64": 13, "128x128": 14, "128x256": 15, "192x256": 18}   # OPSNN_VARIANT_I8_T*


@pytest.mark.parametrize("M,K,N", [(1, 256, 4100), (33, 128, 257), (31, 400, 264), (65, 896, 1001), (129, 1040, 520), (193, 640, 261), (300, 144, 770)])
@pytest.mark.parametrize("tile", sorted(TILES))
def test_each_tile_is_bit_identical(gpu, tile, M, K, N):
    m = gpu
    print(f"case int8 tile {tile} M={M} K={K} N={N}", flush=True)
    bias_dt = m.ACL_INT32 if M % 2 else m.ACL_BF16
    out_dt = m.ACL_FLOAT16 if N % 2 else m.ACL_BF16
    inp = cases.make_qmm_int8_inputs(m, M, K, N, M + K, bias_dt, True)
    want, _ = cases.oracle_qmm_int8(m, inp, M, K, N, True, out_dt)
    d = {k: m.DeviceBuffer(host=inp[k]) for k in ("x1", "x2", "s1", "s2", "bias")}
    d_out = cases.guarded_out(m, M * N * 2)
    a = cases.qmm_args_int8(m, d, M, K, N, 1, True, d_out.ptr, out_dt, m.ACL_FLOAT, N, bias_dt, variant=TILES[tile])
    assert m.lib().opsnnQmmInt8(C.byref(a), None) == 0
    m.check(m.lib().aclrtSynchronizeDevice(), "sync")
    assert np.array_equal(d_out.to_host(want.dtype, want.shape), want)


@pytest.mark.parametrize("M,K,N", [(1, 8192, 1024), (5, 16384, 260), (50, 7168, 2050), (64, 8192, 1032), (200, 14336, 513), (129, 2048, 1500), (150, 1152, 7001)])
def test_planned_shapes_are_bit_identical(gpu, M, K, N):
    m = gpu
    print(f"case int8 planned M={M} K={K} N={N}", flush=True)
    got, want, _ = cases.run_qmm_int8_case(m, orc, M, K, N, seed=M + N, out_dtype=m.ACL_BF16, bias_dtype=m.ACL_FLOAT if M % 2 else None, transpose_x2=True)
    assert np.array_equal(got, want)


# fewer than 64 x 64 outputs: on the tiles from 256 columns and K = 128 on
@pytest.mark.parametrize("transpose_x2", [True, False])
@pytest.mark.parametrize("M,K,N,tiles", [(1, 128, 256, True), (1, 112, 256, False), (1, 1536, 255, False), (15, 144, 273, True), (1, 1024, 4095, True), (3, 1536, 1365, True), (1, 2048, 2040, True)])
def test_few_outputs_are_bit_identical(gpu, M, K, N, tiles, transpose_x2):
    m = gpu
    print(f"case int8 few outputs M={M} K={K} N={N} transpose_x2={transpose_x2}", flush=True)
    got, want, _ = cases.run_qmm_int8_case(m, orc, M, K, N, seed=M + N, out_dtype=m.ACL_BF16, bias_dtype=m.ACL_FLOAT if M % 2 else None, transpose_x2=transpose_x2)
    assert np.array_equal(got, want)
    assert route(m)[0] == ("int8_tiles" if tiles else "plain"), route(m)
