"""MXFP8 on the tile kernel that widens both operands to bf16 with their block scales: the ends of the e8m0 range, rows whose
scales spread over the whole fp32 range, a NaN scale, a K split, and the second kernel of a split at every alignment of N."""
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
