"""The calls that the library is timed on: the linear layers of a quantized language model, as a serving program makes them.

A pass is one layer on one batch of tokens, through the two-phase entry points: phase 1, then phase 2 into buffers that
the program keeps (workspace, output).  Two families:

  * weight-only: aclnnWeightQuantBatchMatmulV2, 16-bit activations against int8 (per channel) or int4 (per group) weights;
  * both operands quantized: aclnnQuantMatmulV5 with int8 per-token x per-channel scales, fp8 e4m3 per-token x per-channel
    scales, fp8 e4m3 block scales, MXFP8 or MXFP4.  With "quantize" the activation arrives in bf16 and the pass starts with
    the quantizer that makes the left operand (aclnnDynamicQuant, aclnnDynamicBlockQuant, aclnnDynamicMxQuant); without it
    the operand is already there, as behind a fused normalisation.

Sizes are those of bench.py's configurations and of the projection shapes in the tests; `draw` spreads over the same
ranges: 1 to 4096 tokens, 1024 to 18432 input features, 1024 to 28672 output features.
"""
import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "ops-nn_amd"))
if os.path.isdir("ops-nn_amd"):   # the tree that is the working folder comes first
    sys.path.insert(0, os.path.abspath("ops-nn_amd"))

import opsnn  # noqa: E402

TORCH = {"fp16": torch.float16, "bf16": torch.bfloat16}
ACL = {"fp16": opsnn.ACL_FLOAT16, "bf16": opsnn.ACL_BF16}


def _wq(name, w, x, M, K, N, group=0, offset=False, layout="nk", bias=False):
    return {"name": name, "op": "weight_only", "w": w, "x": x, "M": M, "K": K, "N": N, "group": group, "offset": offset, "layout": layout,
            "bias": bias}


def _qmm(name, op, M, K, N, quantize, B=1, bias=False):
    return {"name": name, "op": op, "B": B, "M": M, "K": K, "N": N, "quantize": quantize, "bias": bias}


def listed():
    return [
        # one attention projection in a small decode batch: the smallest call of a step, where launch and host time count
        _wq("w8a16_decode_16", "int8", "bf16", 16, 4096, 4096),
        # the widest projection of a large model, one sequence: the weight stream is everything
        _wq("w4a16_decode_1", "int4", "fp16", 1, 8192, 28672, group=128, offset=True),
        # the same with a full decode batch
        _wq("w4a16_decode_64", "int4", "fp16", 64, 8192, 28672, group=128, offset=True),
        # the same operator with the weight in its literal [K, N] storage, as checkpoints often hold it
        _wq("w4a16_kn_decode_16", "int4", "fp16", 16, 8192, 28672, group=128, offset=True, layout="kn"),
        # a prompt of odd length through a weight-only projection (bf16 activations, no zero points)
        _wq("w4a16_prefill_1999", "int4", "bf16", 1999, 4096, 11008, group=128),
        # prefill in int8, activation already quantized, bias
        _qmm("int8_prefill_2048", "int8", 2048, 4096, 11008, False, bias=True),
        # a ragged chunk of tokens through an int8 layer with its activation quantizer
        _qmm("int8_linear_333", "int8", 333, 3584, 18944, True, bias=True),
        # a decode step of an fp8 per-token layer with its quantizer: two small launches
        _qmm("fp8_token_linear_8", "fp8_token", 8, 4096, 4096, True),
        # prefill with fp8 block scales
        _qmm("fp8_block_prefill_4096", "fp8_block", 4096, 7168, 18432, False),
        # the down-projection of the same model in a decode batch, with the 1 x 128 quantizer in front
        _qmm("fp8_block_linear_64", "fp8_block", 64, 18432, 7168, True),
        # a mid-size chunk through an MXFP8 layer with its quantizer
        _qmm("mxfp8_linear_500", "mxfp8", 500, 8192, 8192, True),
        # batched MXFP4: the largest call
        _qmm("mxfp4_batched_8", "mxfp4", 4096, 8192, 8192, False, B=8),
    ]


# 2 * B * M * K * N at most: what keeps a drawn case under the largest listed one, at the rate each kind runs at
MOST_FLOPS = {"weight_only": 4e11, "int8": 1e12, "fp8_token": 6e11, "fp8_block": 1e12, "mxfp8": 6e11, "mxfp4": 4e12}


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def _grain(v, g, lo):
    return max(lo, int(round(v / g)) * g)


def draw(rng):
    op = rng.choice(["weight_only", "weight_only", "weight_only", "int8", "fp8_token", "fp8_block", "mxfp8", "mxfp4"])
    M = max(1, int(round(_log(rng, 1, 4096))))
    # input features come in whole groups of 128, sometimes of 64; output features in multiples of 64, sometimes of 8 or
    # in any count (vocabularies); 4-bit weights in [K, N] storage pair neighbouring columns, so N is even there
    K = _grain(_log(rng, 1024, 18432), 128 if op == "fp8_block" or rng.random() < 0.75 else 64, 1024)
    N = _grain(_log(rng, 1024, 28672), rng.choice([64, 64, 64, 64, 64, 8, 8, 1]), 1024)
    most = MOST_FLOPS[op]
    M = max(1, min(M, int(most / (2.0 * K * N))))
    if op == "weight_only":
        w = rng.choice(["int8", "int4", "int4"])
        layout = "kn" if rng.random() < 0.3 else "nk"
        group = 0 if w == "int8" else rng.choice([128, 128, 128, 64])
        if w == "int4" and layout == "kn":
            N += N % 2
        c = _wq("", w, rng.choice(["fp16", "bf16"]), M, K, N, group=group, offset=group > 0 and rng.random() < 0.5, layout=layout,
                bias=rng.random() < 0.25)
    else:
        B = 1
        if op == "mxfp4" and rng.random() < 0.5:
            B = max(1, min(rng.choice([2, 4, 8]), int(most / (2.0 * M * K * N))))
        c = _qmm("", op, M, K, N, B == 1 and rng.random() < 0.6, B=B, bias=op == "int8" and rng.random() < 0.5)
    del c["name"]
    return c


# ---- inputs ----------------------------------------------------------------------------------------------------------
# Quantized weights and activations are normal values on the format's grid, made by table: a uniform 16-bit number picks
# the code of its normal quantile (an 8-bit code, or two independent 4-bit codes in one byte).

_E2M1 = torch.tensor([0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0])
_tables = {}


def _table(fmt):
    if fmt not in _tables:
        def normal(n):
            u = (torch.arange(n, dtype=torch.float64) + 0.5) / n
            return (torch.erfinv(2 * u - 1) * math.sqrt(2.0)).float()
        if fmt == "int8":
            t = (normal(65536) * 32).round().clamp(-127, 127).to(torch.int8).view(torch.uint8)
        elif fmt == "e4m3":
            t = (normal(65536) * 110).clamp(-448, 448).to(torch.float8_e4m3fn).view(torch.uint8)
        else:
            v = normal(256)
            if fmt == "int4":
                code = (v * 2.7).round().clamp(-8, 7).to(torch.int32) & 15
            else:
                mag = torch.bucketize((v * 2.2).abs(), (_E2M1[1:] + _E2M1[:-1]) / 2).to(torch.int32)
                code = mag + 8 * (v < 0).to(torch.int32)
            t = (code[:, None] + 16 * code[None, :]).reshape(-1).to(torch.uint8)
        _tables[fmt] = t.cuda()
    return _tables[fmt]


def _codes(g, fmt, *shape):
    """Bytes of quantized normal values; the last dim counts bytes."""
    n = math.prod(shape)
    out = torch.empty(n, dtype=torch.uint8, device="cuda")
    for at in range(0, n, 1 << 26):
        m = min(1 << 26, n - at)
        pick = torch.randint(0, 65536, (m,), dtype=torch.int32, device="cuda", generator=g)
        torch.index_select(_table(fmt), 0, pick, out=out[at:at + m])
    return out.view(*shape)


def _uniform(g, lo, hi, *shape, dtype=torch.float32):
    return (torch.rand(*shape, device="cuda", generator=g) * (hi - lo) + lo).to(dtype)


def _activation(g, M, K, dtype):
    """Normal values with channels of different sizes, as behind a normalisation layer."""
    channel = torch.exp(0.5 * torch.randn(K, device="cuda", generator=g))
    return (torch.randn(M, K, device="cuda", generator=g) * channel).to(dtype)


def _e8m0(g, lo, hi, *shape):
    return torch.randint(127 + lo, 127 + hi + 1, shape, device="cuda", generator=g, dtype=torch.int32).to(torch.uint8)


class _State:
    """What a program keeps between calls: tensors with their device memory, and the workspace that phase 1 asked for."""

    def __init__(self):
        self.memory, self.workspace, self.workspace_bytes = [], None, 0

    def tensor(self, data, shape, dtype, strides=None):
        self.memory.append(data)
        return opsnn.Tensor(shape, dtype, data.data_ptr(), strides=strides)

    def plan(self, phase1):
        rc, size, executor = phase1()
        opsnn.check(rc, "phase 1")
        opsnn.lib().aclDestroyAclOpExecutor(executor)
        self.workspace_bytes = size
        if size:
            self.memory.append(torch.empty(size, dtype=torch.uint8, device="cuda"))
            self.workspace = self.memory[-1].data_ptr()


def prepare(case, seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    s = _State()
    (_prepare_weight_only if case["op"] == "weight_only" else _prepare_quantized)(s, case, g)
    return s


def _prepare_weight_only(s, c, g):
    M, K, N, group, nk = c["M"], c["K"], c["N"], c["group"], c["layout"] == "nk"
    dt, adt = TORCH[c["x"]], ACL[c["x"]]
    s.x = s.tensor(_activation(g, M, K, dt), (M, K), adt)
    four = c["w"] == "int4"
    rows, cols = (N, K) if nk else (K, N)
    w = _codes(g, c["w"], rows, cols // 2 if four else cols)
    s.w = s.tensor(w, (K, N), opsnn.ACL_INT4 if four else opsnn.ACL_INT8, strides=(1, K) if nk else None)
    if group:
        G = -(-K // group)
        shape, strides, stored = (G, N), ((1, G) if nk else None), ((N, G) if nk else (G, N))
    else:
        shape, strides, stored = (N,), None, (N,)
    lo, hi = (0.005, 0.02) if four else (2e-4, 1e-3)
    s.scale = s.tensor(_uniform(g, lo, hi, *stored, dtype=dt), shape, adt, strides=strides)
    s.offset = s.tensor(_uniform(g, -1, 1, *stored, dtype=dt), shape, adt, strides=strides) if c["offset"] else None
    s.bias = s.tensor(_uniform(g, -0.3, 0.3, N, dtype=dt), (N,), adt) if c["bias"] else None
    s.out = torch.empty(M, N, dtype=dt, device="cuda")
    s.y = s.tensor(s.out, (M, N), adt)
    s.outputs = s.out

    def phase1():
        return opsnn.weight_quant_batch_matmul_get_workspace(s.x, s.w, s.scale, s.y, offset=s.offset, bias=s.bias, group_size=group)

    s.phase1, s.phase2, s.quantizer = phase1, opsnn.lib().aclnnWeightQuantBatchMatmulV2, None
    s.plan(phase1)


def _prepare_quantized(s, c, g):
    op, B, M, K, N = c["op"], c["B"], c["M"], c["K"], c["N"]
    fmt, acl = {"int8": ("int8", opsnn.ACL_INT8), "mxfp4": ("e2m1", opsnn.ACL_FLOAT4_E2M1)}.get(op, ("e4m3", opsnn.ACL_FLOAT8_E4M3FN))
    kb = K // 2 if op == "mxfp4" else K   # bytes of a row
    batch = (B,) if B > 1 else ()
    quantize = c["quantize"]
    x1 = torch.empty(M, kb, dtype=torch.uint8, device="cuda") if quantize else _codes(g, fmt, B, M, kb)
    x2 = _codes(g, fmt, B, N, kb)
    options = {}
    if op in ("int8", "fp8_token"):
        s1 = torch.empty(M, device="cuda") if quantize else _uniform(g, 0.01, 0.04, M)
        s2 = _uniform(g, 2e-4, 1e-3, N) if op == "int8" else _uniform(g, 5e-5, 3e-4, N)
        t_s1, t_s2 = s.tensor(s1, (M,), opsnn.ACL_FLOAT), s.tensor(s2, (N,), opsnn.ACL_FLOAT)
    elif op == "fp8_block":
        KB, NB = -(-K // 128), -(-N // 128)
        s1 = torch.empty(M, KB, device="cuda") if quantize else _uniform(g, 0.004, 0.012, M, KB)
        s2 = _uniform(g, 5e-5, 3e-4, NB, KB)
        t_s1, t_s2 = s.tensor(s1, (M, KB), opsnn.ACL_FLOAT), s.tensor(s2, (KB, NB), opsnn.ACL_FLOAT, strides=(1, KB))
        options["group_size"] = (1 << 32) | (128 << 16) | 128
    else:
        KS = K // 64
        x_lo, w_lo = (-8, -15) if op == "mxfp8" else (-1, -7)   # the exponents that normal activations and weights get
        s1 = torch.empty(M, KS, 2, dtype=torch.uint8, device="cuda") if quantize else _e8m0(g, x_lo, x_lo + 2, B, M, KS, 2)
        s2 = _e8m0(g, w_lo, w_lo + 2, B, N, KS, 2)
        t_s1 = s.tensor(s1, batch + (M, KS, 2), opsnn.ACL_FLOAT8_E8M0)
        t_s2 = s.tensor(s2, batch + (N, KS, 2), opsnn.ACL_FLOAT8_E8M0)
        options["group_size"] = (1 << 32) | (1 << 16) | 32
    t_x1 = s.tensor(x1, batch + (M, K), acl)
    t_x2 = s.tensor(x2, batch + (N, K), acl)
    if op == "fp8_block":   # its x2 and x2 scales go in as transposed views, the others with the transpose flag
        t_x2 = s.tensor(x2, (K, N), acl, strides=(1, K))
    else:
        options["transpose_x2"] = True
    if c["bias"]:
        options["bias"] = s.tensor(_uniform(g, -0.3, 0.3, N, dtype=torch.bfloat16), (N,), opsnn.ACL_BF16)
    s.out = torch.empty(*batch, M, N, dtype=torch.bfloat16, device="cuda")
    t_out = s.tensor(s.out, batch + (M, N), opsnn.ACL_BF16)
    s.outputs, s.quantizer = s.out, None
    if quantize:
        t_x = s.tensor(_activation(g, M, K, torch.bfloat16), (M, K), opsnn.ACL_BF16)
        s.outputs = {"y": s.out, "x1": x1, "x1_scale": s1}
        if op in ("int8", "fp8_token"):
            s.quantizer = lambda: opsnn.dynamic_quant(t_x, t_x1, t_s1)
        elif op == "fp8_block":
            s.quantizer = lambda: opsnn.dynamic_block_quant(t_x, t_x1, t_s1, row_block=1, col_block=128)
        else:
            s.quantizer = lambda: opsnn.dynamic_mx_quant(t_x, t_x1, t_s1)

    def phase1():
        return opsnn.quant_matmul_v5_get_workspace(t_x1, t_x2, t_s1, t_s2, t_out, **options)

    s.phase1, s.phase2 = phase1, opsnn.lib().aclnnQuantMatmulV5
    s.plan(phase1)


# ---- one pass --------------------------------------------------------------------------------------------------------

def run(s):
    """One layer on the stream that torch works on (the null stream), asynchronously."""
    if s.quantizer is not None:
        s.quantizer()
    rc, _, executor = s.phase1()
    if rc != 0:
        opsnn.check(rc, "phase 1")
    rc = s.phase2(s.workspace, s.workspace_bytes, executor, None)
    if rc != 0:
        opsnn.check(rc, "phase 2")
    return s.outputs


def work(case):
    c = case
    M, K, N = c["M"], c["K"], c["N"]
    if c["op"] == "weight_only":
        four = c["w"] == "int4"
        G = -(-K // c["group"]) if c["group"] else 1
        moved = 2 * M * K + (K * N // 2 if four else K * N) + 2 * G * N * (2 if c["offset"] else 1) + 2 * M * N + (2 * N if c["bias"] else 0)
        return {"bytes": moved, "flops": 2 * M * K * N}
    B, op = c["B"], c["op"]
    kb = K // 2 if op == "mxfp4" else K
    s1, s2 = {"int8": (4 * M, 4 * N), "fp8_token": (4 * M, 4 * N), "fp8_block": (4 * M * -(-K // 128), 4 * -(-K // 128) * -(-N // 128)),
              "mxfp8": (M * K // 32, N * K // 32), "mxfp4": (M * K // 32, N * K // 32)}[op]
    moved = B * (M * kb + N * kb + s1 + s2 + 2 * M * N) + (2 * N if c["bias"] else 0)
    if c["quantize"]:   # the 16-bit activation is read; its quantized form and scales are written (counted above)
        moved += 2 * M * K
    return {"bytes": moved, "flops": 2 * B * M * K * N}


def tolerance(case):
    # the result's own rounding: half an ulp on either side, more where the dequantised weight is rounded to 16 bits too
    # (weight-only).  Codes made by the quantizers are whole values and stay the same.
    if case["op"] == "weight_only" and case["x"] == "fp16":
        return {"rel": 1e-3, "max": 1e-2}
    return {"rel": 5e-3, "max": 3e-2}
