"""Which kernel a call goes to (opsnnDebugLastRoute), at the edges of the rules that choose one by estimates."""
import ctypes as C

import numpy as np
import pytest

import cases

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _reset(gpu):
    gpu.lib().opsnnSetForcePlain(0)
    gpu.lib().opsnnSetFp8Fast(0)
    yield
    gpu.lib().opsnnSetForcePlain(0)
    gpu.lib().opsnnSetFp8Fast(0)


def route(m):
    segments = C.c_int(0)
    return m.lib().opsnnDebugLastRoute(C.byref(segments)).decode(), segments.value


def block_route(m, M, K, N):
    cases.run_blockscale_aclnn(m, cases.make_blockscale_inputs(m, M, K, N, M + N + K, True), M, K, N, True, m.ACL_BF16)
    return route(m)


def test_names(gpu):
    m = gpu
    assert block_route(m, 40, 1024, 512)[0] in ("fp8_stream", "fp8_wide")
    m.lib().opsnnSetForcePlain(1)
    assert block_route(m, 4, 256, 300) == ("plain", 1)


def mx_route(m, M, K, N, fp4=True, batch=1, out=None, bias=None, tB=True):
    cases.run_mx_aclnn(m, cases.make_mx_inputs(m, M, K, N, M + N + K, tB, fp4, batch=batch), M, K, N, tB, m.ACL_BF16 if out is None else out, bias)
    return route(m)


# K % 128 == 64: what the plan cuts along K is launched cut, and large tiles in one piece are never few
@pytest.mark.parametrize("M,K,N", [(514, 2624, 13504), (505, 6208, 17472), (594, 16320, 5312), (2642, 12736, 1088), (200, 9024, 390), (130, 6208, 260)])
def test_mxfp4_tail_is_launched_as_planned(gpu, M, K, N):
    name, segments = mx_route(gpu, M, K, N)
    tiles = -(-M // 256) * -(-N // 256)
    assert name == "mxfp4_tiles_128" or (name == "mxfp4_tiles_256" and (segments > 1 or tiles > 128)), (name, segments)


# (some rows of large tiles in segments, all of small ones)
@pytest.mark.parametrize("M,K,N,rows", [(594, 16320, 5312, [0, 1, 255, 256, 511, 512, 593]), (200, 9024, 390, None), (130, 6208, 260, None)])
def test_mxfp4_tail_in_segments(gpu, M, K, N, rows):
    import oracle_api as orc
    from test_gpu_other_modes import check_close
    m = gpu
    print(f"case mxfp4 tail segments M={M} K={K} N={N}", flush=True)
    inp = cases.make_mx_inputs(m, M, K, N, K + N, True, True)
    got = cases.run_mx_aclnn(m, inp, M, K, N, True, m.ACL_BF16, None)
    assert route(m)[1] > 1
    check_close(got if rows is None else np.ascontiguousarray(got[:, rows]), cases.oracle_mx(m, inp, M, K, N, True, m.ACL_BF16, rows=rows), orc.BF16, "mxfp4 tail in segments")


# 17 to 128 rows of MXFP4: short K and many columns on the few-rows kernel, long K against few columns on tiles that cut it, whatever
# K's tail
@pytest.mark.parametrize("M,K,N,batch,want", [
    (50, 18176, 1088, 1, "mxfp4_tiles_128"), (62, 11264, 1472, 1, "mxfp4_tiles_128"), (79, 15104, 1408, 1, "mxfp4_tiles_128"),
    (44, 11200, 2504, 1, "mxfp4_rows"), (84, 2752, 4096, 1, "mxfp4_rows"), (24, 4480, 4096, 1, "mxfp4_rows"), (64, 4480, 1280, 1, "mxfp4_rows"),
    (36, 5952, 2064, 2, "mxfp4_rows"), (64, 4096, 28672, 1, "mxfp4_tiles_128"), (16, 18176, 1088, 1, "mxfp4_rows")])
def test_mxfp4_rows_or_tiles(gpu, M, K, N, batch, want):
    assert mx_route(gpu, M, K, N, batch=batch)[0] == want


# fp8 block scales with whole scale blocks of columns: few workgroups against a long K run in segments, as with a ragged last block
@pytest.mark.parametrize("M,K,N", [(128, 7168, 2048), (128, 8192, 1024), (72, 12288, 2560), (40, 16384, 1024)])
def test_block_scales_are_cut_for_any_columns(gpu, M, K, N):
    for n in (N, N - 28):
        assert block_route(gpu, M, K, n)[1] > 1, n


# up to 16 rows of fp8: shapes that were measured on both kernels, the weight from memory and from the last-level cache
@pytest.mark.parametrize("mode,M,K,N,want", [
    ("mx", 8, 3200, 1920, "fp8_stream"), ("mx", 3, 6272, 19456, "fp8_decode"), ("mx", 1, 1792, 8192, "fp8_decode"),
    ("block", 1, 1792, 4096, "fp8_decode"),
    ("mx", 1, 12800, 4096, "fp8_wide"), ("block", 1, 12800, 4096, "fp8_wide"),
    # (x1's load into the registers: 15.3 us there and 10.5 here, x2 resident, 13.0 and 8.9, 12.7 and 9.1)
    ("mx", 16, 15872, 1344, "fp8_wide"), ("mx", 16, 7680, 1920, "fp8_wide"), ("block", 12, 12288, 1728, "fp8_wide")])
def test_up_to_16_rows_of_fp8(gpu, mode, M, K, N, want):
    got = mx_route(gpu, M, K, N, False) if mode == "mx" else block_route(gpu, M, K, N)
    assert got[0] == want, got


# from 65 rows: small products on the stream kernels, the others on the exact tiles, by measured shapes
@pytest.mark.parametrize("mode,M,K,N,want", [
    ("mx", 65, 2048, 2304, "fp8_wide fp8_stream"), ("mx", 128, 1664, 1472, "fp8_wide fp8_stream"), ("mx", 128, 13568, 4096, "fp8_exact"),
    ("mx", 70, 13440, 4096, "fp8_exact"), ("mx", 64, 13440, 4096, "fp8_wide"), ("block", 100, 2048, 2304, "fp8_wide fp8_stream"),
    ("block", 405, 1664, 3848, "fp8_wide"), ("block", 512, 4096, 8192, "fp8_exact"), ("mx", 300, 1280, 1152, "fp8_wide fp8_stream"), ("mx", 512, 8192, 4096, "fp8_exact")])
def test_from_65_rows_of_fp8(gpu, mode, M, K, N, want):
    got = mx_route(gpu, M, K, N, False) if mode == "mx" else block_route(gpu, M, K, N)
    assert got[0] in want.split(), got


def rowcol_route(m, M, K, N):
    d1, d2, ds = (m.DeviceBuffer(host=np.zeros(n, t)) for n, t in ((M * K, np.uint8), (N * K, np.uint8), (max(M, N), np.float32)))
    out = m.DeviceBuffer(M * N * 2)
    fp8 = m.ACL_FLOAT8_E4M3FN
    t = [m.Tensor((M, K), fp8, d1), m.Tensor((N, K), fp8, d2), m.Tensor((M,), m.ACL_FLOAT, ds), m.Tensor((N,), m.ACL_FLOAT, ds), m.Tensor((M, N), m.ACL_BF16, out)]
    workspace = m.quant_matmul_v5(*t, transpose_x2=True)
    m.check(m.lib().aclrtSynchronizeDevice(), "sync")
    del workspace
    return route(m)


# calls that the corrections of the tiles' former plan sent to the tiles: us here and there
@pytest.mark.parametrize("mode,M,K,N", [
    ("rowcol", 109, 16640, 15253),   # 91 and 106
    ("rowcol", 204, 2688, 5018),     # 18.5 and 21.1
    ("rowcol", 171, 8704, 2388),     # 19.8 and 21.1
    ("block", 194, 6144, 1472),      # 16.9 and 18.8
    ("block", 184, 10240, 1399),     # 19.1 and 20.1
    ("block", 147, 12416, 1792),     # 20.8 and 22.0
    ("mx", 114, 2944, 4757),         # 18.2 and 19.5
    ("mx", 160, 3840, 1450)])        # 14.1 and 15.6
def test_from_65_rows_of_fp8_on_the_stream_kernel(gpu, mode, M, K, N):
    got = rowcol_route(gpu, M, K, N) if mode == "rowcol" else mx_route(gpu, M, K, N, False) if mode == "mx" else block_route(gpu, M, K, N)
    assert got[0] in ("fp8_wide", "fp8_stream"), got


# with the 8-bit instruction asked for, MXFP8 with few rows keeps its kernels, also below 64 x 64 outputs
@pytest.mark.parametrize("M,K,N", [(1, 2176, 256), (1, 3968, 3968), (1, 10624, 3968), (2, 2112, 1088), (16, 3200, 1920), (24, 1536, 512), (100, 1664, 1472)])
def test_mxfp8_few_rows_with_the_8_bit_instruction(gpu, M, K, N):
    m = gpu
    print(f"case mxfp8 fast few rows M={M} K={K} N={N}", flush=True)
    inp = cases.make_mx_inputs(m, M, K, N, M + N + K, True, False)
    exact, exact_route = cases.run_mx_aclnn(m, inp, M, K, N, True, m.ACL_FLOAT), route(m)
    m.lib().opsnnSetFp8Fast(1)
    fast, fast_route = cases.run_mx_aclnn(m, inp, M, K, N, True, m.ACL_FLOAT), route(m)
    assert fast_route == exact_route and exact_route[0] in ("fp8_stream", "fp8_wide", "fp8_decode", "mxfp8_few_outputs"), (exact_route, fast_route)
    assert np.array_equal(fast, exact)


# fp32 outputs have no 8-bit form: with the switch on they go where they go without it
@pytest.mark.parametrize("M,K,N", [(200, 4096, 1024), (300, 3072, 771), (512, 8192, 4096)])
def test_fp32_outputs_with_the_8_bit_instruction(gpu, M, K, N):
    m = gpu
    inp = cases.make_blockscale_inputs(m, M, K, N, M + N + K, True)
    exact, exact_route = cases.run_blockscale_aclnn(m, inp, M, K, N, True, m.ACL_FLOAT), route(m)
    m.lib().opsnnSetFp8Fast(1)
    fast, fast_route = cases.run_blockscale_aclnn(m, inp, M, K, N, True, m.ACL_FLOAT), route(m)
    assert fast_route == exact_route, (exact_route, fast_route)
    assert np.array_equal(fast, exact)


# weight-only: shapes that were timed on both sides, the weight from memory and in the last-level cache
@pytest.mark.parametrize("M,K,N,group,w,x,nk,off,want", [
    (491, 8448, 2112, 32, "i8", "f16", False, True, "wq_dense"), (27, 17920, 2112, 64, "i4", "bf16", False, False, "wq_wide"),
    (30, 15360, 12288, 64, "i4", "bf16", False, True, "wq_kn"), (32, 2304, 2176, 128, "i4", "f16", False, True, "wq_kn"),
    (110, 11008, 4096, 128, "i4", "f16", False, True, "wq_wide"), (9, 17280, 1888, 64, "i4", "f16", False, True, "wq_wide"),
    (3, 1536, 13184, 0, "i4", "bf16", True, True, "wq_resx"), (9, 1536, 6144, 0, "i8", "f16", True, False, "wq_resx"),
    (18, 3328, 1152, 0, "i8", "bf16", True, True, "wq_nk"), (57, 9856, 4352, 128, "i4", "f16", True, True, "wq_wide"),
    (16, 8192, 28672, 128, "i4", "f16", False, True, "wq_kn_table_w8"), (55, 2432, 1024, 128, "i4", "f16", True, False, "wq_nk"), (4, 3072, 3136, 128, "i4", "f16", True, False, "wq_resx")])
def test_weight_only(gpu, M, K, N, group, w, x, nk, off, want):
    m = gpu
    xd = m.ACL_FLOAT16 if x == "f16" else m.ACL_BF16
    cases.run_wq_aclnn(m, cases.make_wq_inputs(m, M, K, N, 1, xd, m.ACL_INT4 if w == "i4" else m.ACL_INT8, group, nk, off, None), M, K, N)
    assert route(m)[0] == want, route(m)


# the same from 65 rows: pass, wide kernel or many-rows kernel.  us on the one taken and on the next
@pytest.mark.parametrize("M,K,N,group,w,x,nk,off,want", [
    (558, 1728, 27136, 0, "i8", "bf16", True, False, "wq_dense"),     # 84, tile kernel 111
    (827, 12288, 6976, 128, "i4", "bf16", True, False, "wq_dense"),   # 187, tile kernel 700: the many-rows kernel's table does not fit
    (257, 8192, 13312, 0, "i8", "f16", True, False, "wq_rows"),       # 84, wide kernel 118
    (257, 7040, 1090, 128, "i4", "bf16", True, True, "wq_wide")])     # 23.3, pass 25.9
def test_weight_only_from_65_rows(gpu, M, K, N, group, w, x, nk, off, want):
    test_weight_only(gpu, M, K, N, group, w, x, nk, off, want)
