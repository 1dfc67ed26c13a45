"""Outputs at any address that holds whole elements: kernels store several columns at a time, and rows of any length begin anywhere.  The
bits are those of the call whose output lies on 256 bytes, and nothing beside the output changes.  One shape per kernel, with rows that are no
whole number of the columns of a store."""
import numpy as np
import pytest

import cases
from test_gpu_routes import route

pytestmark = pytest.mark.gpu


def _run(m, call, M, N, size, want):
    """call(address): the call with its output there."""
    outs = []
    for shift in (0, size, 3 * size):
        guard = 256
        buf = m.DeviceBuffer(M * N * size + 2 * guard)
        buf.fill(0x5A)
        keep = call(buf.ptr + guard + shift)
        m.check(m.lib().aclrtSynchronizeDevice(), "sync")
        del keep
        assert route(m)[0] == want, route(m)
        raw = buf.to_host(np.uint8, (M * N * size + 2 * guard,))
        at = guard + shift
        assert (raw[:at] == 0x5A).all() and (raw[at + M * N * size:] == 0x5A).all(), shift
        outs.append(raw[at:at + M * N * size])
    assert np.array_equal(outs[0], outs[1]) and np.array_equal(outs[0], outs[2])


@pytest.mark.parametrize("form,M,K,N,out,want", [
    ("int8", 131, 256, 263, "bf16", "int8_tiles"), ("int8", 1027, 256, 4099, "bf16", "int8_tiles"), ("int8", 1027, 256, 4099, "f16", "int8_tiles"),
    ("rowcol", 517, 256, 1031, "bf16", "fp8_exact"), ("rowcol", 517, 256, 1031, "f32", "fp8_exact"), ("rowcol", 9, 1024, 1031, "f32", "fp8_stream"),
    ("rowcol", 40, 8192, 1031, "bf16", "fp8_wide"), ("mx", 517, 256, 1031, "f32", "fp8_exact"), ("mx", 1, 1792, 8195, "bf16", "fp8_decode"),
    ("mx4", 235, 1536, 2055, "bf16", "mxfp4_tiles_128_w8"), ("mx4", 1030, 512, 4103, "bf16", "mxfp4_tiles_256"), ("mx4", 1030, 512, 4103, "f32", "mxfp4_tiles_256"),
    ("mx4", 24, 4480, 4099, "bf16", "mxfp4_rows"), ("mx4", 24, 4480, 4099, "f32", "mxfp4_rows")])
def test_both_operands_quantized(gpu, form, M, K, N, out, want):
    m = gpu
    rng = np.random.default_rng(M + N)
    bits = 4 if form == "mx4" else 8
    x1, x2 = (rng.integers(0, 256, (n, K * bits // 8), np.uint8) & (0xFF if form in ("int8", "mx4") else 0xB7) for n in (M, N))   # (fp8: no NaN)
    if form.startswith("mx"):
        s1, s2 = (rng.integers(120, 130, (n, K // 64, 2)).astype(np.uint8) for n in (M, N))
        shapes, st, kw = [(M, K // 64, 2), (N, K // 64, 2)], m.ACL_FLOAT8_E8M0, {"group_size": (1 << 32) | (1 << 16) | 32}
    else:
        s1, s2 = (rng.uniform(0.5, 2, n).astype(np.float32) for n in (M, N))
        shapes, st, kw = [(M,), (N,)], m.ACL_FLOAT, {}
    dt = {"int8": m.ACL_INT8, "mx4": m.ACL_FLOAT4_E2M1}.get(form, m.ACL_FLOAT8_E4M3FN)
    d = [m.DeviceBuffer(host=v) for v in (x1, x2, s1, s2)]
    t = [m.Tensor((M, K), dt, d[0]), m.Tensor((N, K), dt, d[1]), m.Tensor(shapes[0], st, d[2]), m.Tensor(shapes[1], st, d[3])]
    print(f"case output address {form} M={M} K={K} N={N} {out}", flush=True)
    acl, size = {"bf16": (m.ACL_BF16, 2), "f16": (m.ACL_FLOAT16, 2), "f32": (m.ACL_FLOAT, 4)}[out]
    _run(m, lambda p: m.quant_matmul_v5(*t, m.Tensor((M, N), acl, p), transpose_x2=True, **kw), M, N, size, want)


@pytest.mark.parametrize("M,K,N,group,w,x,nk,off,want", [
    (40, 4096, 1091, 128, "i4", "bf16", True, False, "wq_wide"), (140, 4096, 1096, 128, "i4", "f16", False, True, "wq_wide"), (140, 4096, 1090, 128, "i4", "f16", False, True, "wq_dense"),
    (32, 2304, 2178, 128, "i4", "f16", False, True, "wq_kn"), (55, 2432, 1026, 128, "i4", "f16", True, False, "wq_nk"),
    (9, 1536, 6147, 0, "i8", "f16", True, False, "wq_resx"), (16, 4096, 4099, 0, "i8", "bf16", True, False, "wq_xreg"),
    (1100, 1024, 4099, 128, "i4", "bf16", True, False, "wq_dense")])
def test_weight_only(gpu, M, K, N, group, w, x, nk, off, want):
    m = gpu
    xd = m.ACL_FLOAT16 if x == "f16" else m.ACL_BF16
    wd = m.ACL_INT4 if w == "i4" else m.ACL_INT8
    inp = cases.make_wq_inputs(m, M, K, N, 1, xd, wd, group, nk, off, None)
    d = {k: m.DeviceBuffer(host=v) for k, v in inp.items() if isinstance(v, np.ndarray)}
    G = -(-K // group) if group else 1
    shape, st = ((G, N), (1, G) if nk else None) if group else ((N,), None)
    t = [m.Tensor((M, K), xd, d["x"]), m.Tensor((K, N), wd, d["w"], strides=(1, K) if nk else None), m.Tensor(shape, xd, d["scale"], strides=st)]
    offset = m.Tensor(shape, xd, d["offset"], strides=st) if off else None
    print(f"case output address weight-only M={M} K={K} N={N} {w} {x}", flush=True)
    _run(m, lambda p: m.weight_quant_batch_matmul(*t, m.Tensor((M, N), xd, p), offset=offset, group_size=group), M, N, 2, want)
