"""MXFP8 on the kernels that widen both operands to bf16 with their block scales: rows with some scales up to 60 binades below the
others, a NaN scale, a K split, the second kernel of a split at every alignment of N, and the whole e8m0 range on single products."""
import numpy as np
import pytest

import cases
import oracle_api as orc
from test_gpu_shape_sweep import _b16_bar

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,K,N", [(300, 128, 100), (257, 256, 513), (300, 4096, 302), (512, 2048, 515), (700, 1024, 1001), (260, 8192, 384)])
@pytest.mark.parametrize("spread", [4, 60])
def test_mxfp8_tiles(gpu, M, K, N, spread):
    m = gpu
    inp = cases.make_mx_inputs(m, M, K, N, M + N, True, False, exp_range=4)
    if spread > 4:   # some rows with scales far below the others'
        rng = np.random.default_rng(1)
        for s in (inp["s1"], inp["s2"]):
            low = rng.random(s.shape) < 0.3
            s[low] = (s[low].astype(np.int32) - rng.integers(20, spread, size=int(low.sum()))).astype(np.uint8)
    print(f"case mxfp8 tiles M={M} K={K} N={N} spread={spread}", flush=True)
    got = cases.run_mx_aclnn(m, inp, M, K, N, True, m.ACL_BF16)
    _b16_bar(got, cases.oracle_mx(m, inp, M, K, N, True, m.ACL_BF16), orc.BF16, "mxfp8 tiles", K)


@pytest.mark.parametrize("M,K,N", [(129, 992, 1024), (129, 1024, 1024), (129, 1024, 2080), (192, 1152, 515), (256, 2048, 6976)])
@pytest.mark.parametrize("out", ["f32", "bf16"])
def test_mxfp8_short_k_split(gpu, M, K, N, out):
    """Around the K of eight tiles of 128 from which the exact kernel's plan may cut it.  Two fp32 sums of the same exact products differ by
    at most K roundings each, relative to the sum of the terms' magnitudes; the stated bar holds for bf16."""
    m = gpu
    inp = cases.make_mx_inputs(m, M, K, N, M + N, True, False, exp_range=4)
    dt = m.ACL_FLOAT if out == "f32" else m.ACL_BF16
    print(f"case mxfp8 short K M={M} K={K} N={N} {out}", flush=True)
    got, want = cases.run_mx_aclnn(m, inp, M, K, N, True, dt), cases.oracle_mx(m, inp, M, K, N, True, dt)
    if out == "bf16":
        _b16_bar(got, want, orc.BF16, "mxfp8 short K", K)
    else:
        vals = np.abs(_e4m3_values())

        def wide(x, s):
            e = s.reshape(x.shape[1], -1)[:, : K // 32, None].astype(np.int64) - 127
            return np.ldexp(vals[x[0] & 127].reshape(x.shape[1], K // 32, 32), e).reshape(x.shape[1], K)
        terms = wide(inp["x1"], inp["s1"]) @ wide(inp["x2"], inp["s2"]).T
        assert (np.abs(got.reshape(M, N).astype(np.float64) - want.reshape(M, N)) <= 2 * K * 2.0 ** -24 * terms).all()


@pytest.mark.parametrize("M,K,N", [(300, 512, 260), (300, 4096, 256)])
def test_mxfp8_nan_scale_stays_in_its_row(gpu, M, K, N):
    m = gpu
    inp = cases.make_mx_inputs(m, M, K, N, 7, True, False)
    clean = cases.oracle_mx(m, inp, M, K, N, True, m.ACL_BF16)
    inp["s1"][0, 5, 1, 0] = 255
    inp["s2"][0, 9, 2, 1] = 255
    print(f"case mxfp8 nan scale M={M} K={K} N={N}", flush=True)
    got = orc.b16_to_f32(cases.run_mx_aclnn(m, inp, M, K, N, True, m.ACL_BF16), orc.BF16).reshape(M, N)
    want = orc.b16_to_f32(clean, orc.BF16).reshape(M, N)
    assert np.isnan(got[5]).all() and np.isnan(got[:, 9]).all()
    keep = np.ones((M, N), bool)
    keep[5], keep[:, 9] = False, False
    assert np.isfinite(got[keep]).all()
    assert np.mean(np.abs(got[keep] - want[keep])) <= 1e-3 * np.mean(np.abs(want[keep]))


def _e4m3_values():
    b = np.arange(256)
    e, m = (b >> 3) & 15, b & 7
    v = np.where(e == 0, m * 2.0 ** -9, (8 + m) * 2.0 ** (e - 10.0))
    return np.where(b & 128, -v, v)   # (0x7f and 0xff are NaN and not drawn)


@pytest.mark.parametrize("M", [16, 64, 300])
@pytest.mark.parametrize("out", ["f32", "bf16"])
@pytest.mark.parametrize("lo1,hi1,lo2,hi2", [(0, 2, 200, 245), (3, 12, 100, 245), (0, 245, 0, 245), (236, 245, 0, 2)])
def test_mxfp8_single_products_over_the_e8m0_range(gpu, M, out, lo1, hi1, lo2, hi2):
    """One element of x1 per row is not zero, so every output is one product, which has to be exact.  Both operands are widened to
    bf16: exact from scale byte 3 on; for the bytes 0 to 2 the smallest codes lie between bf16's subnormal values (multiples of
    2^-133) and are rounded to the nearest.  (Bytes up to 245: no value beyond fp32.  Products below fp32's normal range aside.)"""
    m = gpu
    K, N = 256, 320
    rng = np.random.default_rng(M + lo1)
    vals = _e4m3_values()
    codes = np.array([b for b in range(256) if b & 127 != 127], np.uint8)
    x2 = rng.choice(codes, (1, N, K)).astype(np.uint8)
    s1 = rng.integers(lo1, hi1 + 1, (1, M, K // 64, 2)).astype(np.uint8)
    s2 = rng.integers(lo2, hi2 + 1, (1, N, K // 64, 2)).astype(np.uint8)
    k, c = rng.integers(0, K, M), rng.choice(codes, M)
    x1 = np.zeros((1, M, K), np.uint8)
    x1[0, np.arange(M), k] = c

    def widened(code, byte):
        return np.round(np.ldexp(vals[code], byte.astype(np.int64) - 127 + 133)) * 2.0 ** -133   # (round: to even, as the conversion)
    a = widened(c, s1.reshape(M, K // 32)[np.arange(M), k // 32])
    b = widened(x2[0][:, k], s2.reshape(N, K // 32)[:, k // 32])          # [N, M]
    want = (a[None, :] * b).T
    with np.errstate(over="ignore"):
        want32 = want.astype(np.float32)
    print(f"case mxfp8 range M={M} {out} s1 {lo1}..{hi1} s2 {lo2}..{hi2}", flush=True)
    got = cases.run_mx_aclnn(m, dict(x1=x1, x2=x2, s1=s1, s2=s2, fp4=False), M, K, N, True, m.ACL_FLOAT if out == "f32" else m.ACL_BF16)[0]
    normal = np.abs(want) >= 2.0 ** -126
    assert normal.mean() > 0.3
    if out == "f32":
        assert np.array_equal(got[normal], want32[normal])
    else:
        assert np.array_equal(got[normal], orc.f32_to_b16(want32, m.ACL_BF16)[normal])


# fewer than 64 x 64 outputs, K % 128 == 64: the operands stay in 32 bits, also where x1's scale bytes are 0 to 2 (2^-127 .. 2^-125), which
# bf16 holds only in part.  fp32 sums of exact products in chains of at most K / 4096 + 8 steps of 16: within 2^-18 of the sum of magnitudes
@pytest.mark.parametrize("M,K,N", [(1, 192, 256), (1, 2112, 4000), (2, 1088, 1500), (3, 704, 1300), (4, 64, 700), (7, 4160, 513), (8, 1984, 300), (15, 320, 257)])
@pytest.mark.parametrize("tB", [True, False])
def test_few_outputs_keep_32_bit_operands(gpu, M, K, N, tB):
    m = gpu
    m.lib().opsnnSetForcePlain(0)
    print(f"case mxfp8 few outputs M={M} K={K} N={N} tB={tB}", flush=True)
    inp = cases.make_mx_inputs(m, M, K, N, M + N + K, tB, False)
    rng = np.random.default_rng(M)
    inp["s1"] = rng.integers(0, 4, inp["s1"].shape).astype(np.uint8)
    inp["s2"] = rng.integers(232, 238, inp["s2"].shape).astype(np.uint8)
    bias = rng.normal(0, 2.0 ** -12, N).astype(np.float32) if M % 2 else None
    c = np.arange(256)
    e, f, s = (c >> 3) & 15, c & 7, np.where(c & 128, -1.0, 1.0)
    code = np.where((e == 15) & (f == 7), np.nan, s * np.where(e == 0, f * 2.0 ** -9, (8 + f) * 2.0 ** (e - 10.0)))
    s1 = np.exp2(inp["s1"][0].reshape(M, -1).astype(np.float64) - 127)
    s2 = np.exp2((inp["s2"][0] if tB else np.moveaxis(inp["s2"][0], 1, 0)).reshape(N, -1).astype(np.float64) - 127)
    a = code[inp["x1"][0]] * np.repeat(s1, 32, 1)[:, :K]
    b = code[inp["x2"][0] if tB else inp["x2"][0].T] * np.repeat(s2, 32, 1)[:, :K]
    want, terms = a @ b.T, np.abs(a) @ np.abs(b).T
    if bias is not None:
        want, terms = want + bias, terms + np.abs(bias)
    got = cases.run_mx_aclnn(m, inp, M, K, N, tB, m.ACL_FLOAT, bias).reshape(M, N).astype(np.float64)
    assert m.lib().opsnnDebugLastRoute(None) == b"mxfp8_few_outputs"
    err = np.abs(got - want)
    assert (err <= 2.0 ** -18 * terms).all(), f"worst error / sum of magnitudes {float((err / terms).max()):.3e}"
