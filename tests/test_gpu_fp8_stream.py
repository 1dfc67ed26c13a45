"""fp8 with up to 128 rows of x1, or small products of up to 512 rows, on the stream kernels (qmm_fp8_stream.hip) through the two-phase entry point, against the oracle."""
import numpy as np
import pytest

import cases
import oracle_api as orc
from test_gpu_other_modes import check_close
from test_gpu_routes import route

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _reset(gpu):
    gpu.lib().opsnnSetForcePlain(0)
    gpu.lib().opsnnSetFp8Fast(0)


# rows on either side of each row-block count and slab; columns that end inside a block of 16, of a wave and of a workgroup, and odd
# counts; K of one block, fewer blocks than waves or stages, a wave with one block less than the others, segments with partial sums
SHAPES = [(1, 128, 256), (15, 256, 257), (16, 1152, 300), (17, 384, 271), (32, 640, 1033), (33, 1280, 260), (48, 512, 2050), (64, 2176, 515),
          (65, 1024, 258), (100, 640, 1100), (128, 1408, 530), (5, 2048, 4361), (40, 896, 8200), (64, 4608, 1030), (16, 13440, 258), (24, 8320, 390), (128, 7040, 280),
          (129, 1024, 520), (193, 1152, 1030), (300, 3072, 771), (512, 1024, 257)]


@pytest.mark.parametrize("M,K,N", SHAPES)
@pytest.mark.parametrize("gsM,out", [(1, "bf16"), (128, "f32")])
def test_block_scales(gpu, M, K, N, gsM, out):
    m = gpu
    print(f"case fp8 stream block M={M} K={K} N={N} gsM={gsM} out={out}", flush=True)
    dt = {"bf16": m.ACL_BF16, "f32": m.ACL_FLOAT}[out]
    inp = cases.make_blockscale_inputs(m, M, K, N, M + N + K, True, gsM)
    want = cases.oracle_blockscale(m, inp, M, K, N, True, dt)
    got = cases.run_blockscale_aclnn(m, inp, M, K, N, True, dt)
    assert route(m)[0] in STREAM, route(m)
    if out == "f32":
        assert np.isfinite(got).all()
        mx, mean = orc.rel_err_stats(got, want)
        assert mean <= 2.0 ** -16 and orc.isclose_fraction(got, want) == 0.0, f"max rel {mx:.3e} mean rel {mean:.3e}"
    else:
        check_close(got, want, orc.BF16, "fp8 stream, block scales")


STREAM = ("fp8_stream", "fp8_wide")
ELSEWHERE = {("mx", 5, 2048, 4361): "fp8_decode", ("mx", 3, 192, 256): "mxfp8_few_outputs", ("mx", 3, 2112, 1088): "mxfp8_few_outputs", ("mx", 2, 1088, 260): "mxfp8_few_outputs"}


# (K % 128 == 64 as well: the narrow kernel, with four column blocks where N is wide)
@pytest.mark.parametrize("M,K,N", SHAPES + [(3, 192, 256), (16, 320, 300), (33, 1088, 4500), (70, 1984, 1030), (12, 704, 9001), (32, 4160, 17000), (161, 2496, 300),
                                            (3, 2112, 1088), (2, 1088, 260)])   # (the last two: fewer than 64 x 64 outputs)
@pytest.mark.parametrize("form", ["rowcol", "mx"])
def test_row_column_and_mx_scales(gpu, form, M, K, N):
    """fp32 outputs: exact products, fp32 sums of at most 8 terms a step inside the instruction and K / 128 steps beyond, so within
    2^-18 of the sum of magnitudes."""
    m = gpu
    print(f"case fp8 stream {form} M={M} K={K} N={N}", flush=True)
    rng = np.random.default_rng(M + K + N)
    x1, x2 = cases.gen_fp8(rng, (M, K)), cases.gen_fp8(rng, (N, K))
    bias = rng.normal(0, 1, N).astype(np.float32) if M % 2 else None
    if form == "rowcol":
        s1, s2 = rng.uniform(0.5, 2, M).astype(np.float32), rng.uniform(0.5, 2, N).astype(np.float32)
        r1, r2 = s1[:, None].astype(np.float64), s2[:, None].astype(np.float64)
    else:
        KS = -(-K // 64)
        s1, s2 = (rng.integers(122, 133, (r, KS, 2)).astype(np.uint8) for r in (M, N))
        if K % 64:
            s1[:, -1, 1] = s2[:, -1, 1] = 0xFF
        r1, r2 = (np.repeat(np.exp2(s.reshape(len(s), -1)[:, :K // 32].astype(np.float64) - 127), 32, 1) for s in (s1, s2))
    code = _codes()
    a, b = code[x1] * r1, code[x2] * r2
    want, terms = a @ b.T, np.abs(a) @ np.abs(b).T
    if bias is not None:
        want, terms = want + bias, terms + np.abs(bias)
    d = {k: m.DeviceBuffer(host=v) for k, v in dict(x1=x1, x2=x2, s1=s1, s2=s2).items()}
    d_out = m.DeviceBuffer(M * N * 4 + 64)
    d_out.fill(0xEE)
    acl = m.ACL_FLOAT8_E4M3FN
    kw = dict(transpose_x2=True)
    if bias is not None:
        d["bias"] = m.DeviceBuffer(host=bias)
        kw["bias"] = m.Tensor((N,), m.ACL_FLOAT, d["bias"])
    if form == "mx":
        kw["group_size"] = (1 << 32) | (1 << 16) | 32
    st = m.ACL_FLOAT if form == "rowcol" else m.ACL_FLOAT8_E8M0
    keep = m.quant_matmul_v5(m.Tensor((M, K), acl, d["x1"]), m.Tensor((N, K), acl, d["x2"]), m.Tensor(s1.shape, st, d["s1"]), m.Tensor(s2.shape, st, d["s2"]),
                             m.Tensor((M, N), m.ACL_FLOAT, d_out), **kw)
    m.check(m.lib().aclrtSynchronizeDevice(), "sync")
    assert route(m)[0] in ([ELSEWHERE[form, M, K, N]] if (form, M, K, N) in ELSEWHERE else STREAM), route(m)
    raw = d_out.to_host(np.uint8, (M * N * 4 + 64,))
    assert (raw[M * N * 4:] == 0xEE).all(), "wrote past the output"
    got = raw[:M * N * 4].view(np.float32).reshape(M, N).astype(np.float64)
    err = np.abs(got - want)
    assert (err <= 2.0 ** -18 * terms + 1e-30).all(), f"worst error / sum of magnitudes {float((err / (terms + 1e-30)).max()):.3e}"
    del keep


# a weight from 100 MB on: every second of the wide kernel's copies goes past the last-level cache, from 150 MB on three of four; a last strip of
# one column, segments
@pytest.mark.parametrize("form,M,K,N", [("block", 17, 12288, 8193), ("rowcol", 33, 13568, 7400), ("mx", 20, 18432, 5440),
                                        ("block", 18, 16384, 9217), ("rowcol", 20, 18432, 8200), ("mx", 33, 12800, 11800)])
def test_weights_from_100_mb_on(gpu, form, M, K, N):
    assert N * K > 100_000_000
    if form == "block":
        test_block_scales(gpu, M, K, N, 1, "bf16")
    else:
        test_row_column_and_mx_scales(gpu, form, M, K, N)
    assert route(gpu)[0] == "fp8_wide", route(gpu)


# rows of x1 so far apart that the last ones lie 2^32 bytes and more behind the first: the stream kernels' lane offsets have 32 bits
# (a K tail runs on padded copies, whose rows lie close together)
@pytest.mark.parametrize("M,K,N,want", [(300, 1024, 256, "fp8_exact"), (300, 1088, 260, "fp8_stream")])
def test_rows_far_apart(gpu, M, K, N, want):
    m = gpu
    stride = (1 << 24) - 128
    print(f"case fp8 stream rowcol, rows {stride} apart M={M} K={K} N={N}", flush=True)
    rng = np.random.default_rng(M + K)
    x1, x2 = cases.gen_fp8(rng, (M, K)), cases.gen_fp8(rng, (N, K))
    s1, s2 = rng.uniform(0.5, 2, M).astype(np.float32), rng.uniform(0.5, 2, N).astype(np.float32)
    d = {k: m.DeviceBuffer(host=v) for k, v in dict(x2=x2, s1=s1, s2=s2).items()}
    d["x1"] = m.DeviceBuffer((M - 1) * stride + K)
    for r in range(M):
        m.check(m.lib().aclrtMemcpy(d["x1"].ptr + r * stride, K, x1[r].ctypes.data, K, m.binding.H2D), "aclrtMemcpy H2D")
    d_out = m.DeviceBuffer(M * N * 4)
    acl = m.ACL_FLOAT8_E4M3FN
    keep = m.quant_matmul_v5(m.Tensor((M, K), acl, d["x1"], strides=(stride, 1), storage_shape=((M - 1) * stride + K,)), m.Tensor((N, K), acl, d["x2"]),
                             m.Tensor((M,), m.ACL_FLOAT, d["s1"]), m.Tensor((N,), m.ACL_FLOAT, d["s2"]), m.Tensor((M, N), m.ACL_FLOAT, d_out), transpose_x2=True)
    m.check(m.lib().aclrtSynchronizeDevice(), "sync")
    assert route(m)[0] == want, route(m)
    got = d_out.to_host(np.float32, (M, N)).astype(np.float64)
    code = _codes()
    a, b = code[x1] * s1[:, None].astype(np.float64), code[x2] * s2[:, None].astype(np.float64)
    err = np.abs(got - a @ b.T)
    assert (err <= 2.0 ** -18 * (np.abs(a) @ np.abs(b).T) + 1e-30).all(), f"worst {err.max():.3e}"
    del keep


def _codes():
    c = np.arange(256)
    e, f, s = (c >> 3) & 15, c & 7, np.where(c & 128, -1.0, 1.0)
    return np.where((e == 15) & (f == 7), np.nan, s * np.where(e == 0, f * 2.0 ** -9, (8 + f) * 2.0 ** (e - 10.0)))
