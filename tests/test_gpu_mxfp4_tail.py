"""MXFP4 on 256 x 256 tiles with a K that is no whole pair of 256-element K tiles: the tiles end in zeros, the last scale words by
word, and a K inside a word behind scale rows that are copied (the data is read as it lies)."""
import numpy as np
import pytest

import cases
import oracle_api as orc
from test_gpu_other_modes import check_close
from test_gpu_routes import route

pytestmark = pytest.mark.gpu


# 65 batches of one tile: more than the 64 tiles below which 128 x 128 ones take over.  One K tile and less, an odd and an even count,
# a last tile of a quarter, a half and three quarters, and (32, 96, 160 mod 128) a last scale word that is not full
@pytest.mark.parametrize("K", [32, 96, 128, 160, 256, 384, 544, 640, 768, 992, 1088, 1152, 1408])
@pytest.mark.parametrize("tB", [True, False])
def test_k_tail_on_whole_tiles(gpu, K, tB):
    m = gpu
    B, M, N = 65, 131, 140
    print(f"case mxfp4 tail B={B} M={M} K={K} N={N} tB={tB}", flush=True)
    m.lib().opsnnSetForcePlain(0)
    inp = cases.make_mx_inputs(m, M, K, N, K, tB, True, batch=B)
    if K % 64:   # the byte behind the last block scales nothing: a NaN code there must not reach any sum
        inp["s1"][..., -1, 1] = 0xFF
        if tB:
            inp["s2"][..., -1, 1] = 0xFF
        else:
            inp["s2"][:, -1, :, 1] = 0xFF
    bias = np.random.default_rng(1).normal(0, 1, N).astype(np.float32)
    want = cases.oracle_mx(m, inp, M, K, N, tB, m.ACL_BF16, bias)
    got = cases.run_mx_aclnn(m, inp, M, K, N, tB, m.ACL_BF16, bias)
    assert route(m) == ("mxfp4_tiles_256", 1), route(m)
    check_close(got, want, orc.BF16, "mxfp4 tail")


def test_neighbours_with_infinite_scales_stay_out(gpu):
    """Rows whose scales are NaN codes reach their own outputs only: nothing of a row is read for the tail of the row in front of it."""
    m = gpu
    B, M, N, K = 65, 131, 140, 640
    m.lib().opsnnSetForcePlain(0)
    inp = cases.make_mx_inputs(m, M, K, N, 7, True, True, batch=B)
    inp["s1"][:, 1::2] = 0xFF
    inp["s2"][:, 1::2] = 0xFF
    got = orc.b16_to_f32(cases.run_mx_aclnn(m, inp, M, K, N, True, m.ACL_BF16, None), orc.BF16).reshape(B, M, N)
    want = orc.b16_to_f32(cases.oracle_mx(m, inp, M, K, N, True, m.ACL_BF16, None), orc.BF16).reshape(B, M, N)
    assert np.isnan(got[:, 1::2]).all() and np.isnan(got[:, :, 1::2]).all()
    assert np.isfinite(got[:, ::2, ::2]).all() and np.allclose(got[:, ::2, ::2], want[:, ::2, ::2], rtol=1e-2, atol=1e-2)


# few tiles of either size against a long K: K in segments of whole tiles of 128 elements, an odd count of them and a shorter last segment
@pytest.mark.parametrize("M,K,N", [(130, 6272, 260), (200, 4480, 390), (65, 8320, 520), (2100, 6272, 2090)])
def test_segments_of_odd_tiles(gpu, M, K, N):
    m = gpu
    print(f"case mxfp4 segments M={M} K={K} N={N}", flush=True)
    inp = cases.make_mx_inputs(m, M, K, N, K + N, True, True)
    got = cases.run_mx_aclnn(m, inp, M, K, N, True, m.ACL_BF16, None)
    assert route(m)[1] > 1, route(m)
    check_close(got, cases.oracle_mx(m, inp, M, K, N, True, m.ACL_BF16, None), orc.BF16, "mxfp4 in segments")


# on small tiles the operands are copied as well; large ones copy the scale rows alone
@pytest.mark.parametrize("M,K,N,want", [(260, 32, 262000, "mxfp4_tiles_128"), (512, 736, 262000, "mxfp4_tiles_256")])
def test_scale_rows_of_both_operands_beyond_the_grids_second_axis(gpu, M, K, N, want):
    """M + N rows of scales are copied by one launch, four a workgroup: more workgroups than the second and third axis of a grid hold."""
    m = gpu
    print(f"case mxfp4 tail M={M} K={K} N={N}", flush=True)
    inp = cases.make_mx_inputs(m, M, K, N, 5, True, True)
    got = cases.run_mx_aclnn(m, inp, M, K, N, True, m.ACL_BF16, None)
    assert route(m) == (want, 1), route(m)
    rows = None if K == 32 else [0, 1, 130, 255, 256, M - 1]   # (of the larger case some rows)
    check_close(got if rows is None else np.ascontiguousarray(got[:, rows]), cases.oracle_mx(m, inp, M, K, N, True, m.ACL_BF16, rows=rows), orc.BF16,
                "mxfp4 tail, many scale rows")


@pytest.mark.parametrize("M,K,N", [(40, 256, 65536), (97, 384, 65500)])
def test_eight_waves_and_four_give_the_same_bits(gpu, M, K, N):
    """128 x 128 tiles on either side of the line between eight and four waves, 512 workgroups: the same columns by themselves and with 128 more."""
    m = gpu
    inp = cases.make_mx_inputs(m, M, K, N + 128, N, True, True)
    few = dict(inp)
    few["x2"], few["s2"] = (np.ascontiguousarray(inp[k][:, :N]) for k in ("x2", "s2"))
    print(f"case mxfp4 eight and four waves M={M} K={K} N={N}", flush=True)
    got = []
    for i, n, want in ((few, N, "mxfp4_tiles_128_w8"), (inp, N + 128, "mxfp4_tiles_128")):
        got.append(cases.run_mx_aclnn(m, i, M, K, n, True, m.ACL_BF16, None).reshape(M, n)[:, :N])
        assert route(m) == (want, 1), route(m)
    assert np.array_equal(got[0], got[1])
    rows = [0, 31, 32, M - 1]
    check_close(np.ascontiguousarray(got[0][rows]).reshape(1, 4, N), cases.oracle_mx(m, few, M, K, N, True, m.ACL_BF16, rows=rows), orc.BF16, "mxfp4 eight waves")


@pytest.mark.parametrize("M,K,N", [(107, 16896, 1536), (74, 9216, 3840)])
def test_segments_of_small_tiles_are_four_waves(gpu, M, K, N):
    m = gpu
    print(f"case mxfp4 segments of small tiles M={M} K={K} N={N}", flush=True)
    inp = cases.make_mx_inputs(m, M, K, N, M, True, True)
    got = cases.run_mx_aclnn(m, inp, M, K, N, True, m.ACL_BF16, None)
    name, segments = route(m)
    assert name == "mxfp4_tiles_128" and segments > 1 and K <= 18 * 128 * segments, (name, segments)
    check_close(got, cases.oracle_mx(m, inp, M, K, N, True, m.ACL_BF16, None), orc.BF16, "mxfp4 segments of small tiles")
