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
