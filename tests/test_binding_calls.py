"""The binding's extension (csrc/python/calls.cpp) against the same entry points called through ctypes: statuses, workspace sizes and
whether an executor comes back, for calls that are accepted and for calls that are refused; and views of up to eight dims."""
import ctypes as C
import os
import subprocess
import sys
import sysconfig
import threading

import pytest

import opsnn as m

PTR = 1 << 20


def _ctypes(name, *args):
    fn = C.CDLL(m.LIB_PATH)[name]   # (a function object of its own)
    fn.restype, fn.argtypes = m.binding._SIGS[name]
    ws, ex = C.c_uint64(0), C.c_void_p()
    rc = fn(*args, C.byref(ws), C.byref(ex))
    return rc, ws.value, ex.value


def _same(got, want):
    for ex in (got[2], want[2]):
        if ex:
            m.check(m.lib().aclDestroyAclOpExecutor(ex))
    assert got[:2] == want[:2] and (got[2] is None) == (want[2] is None), (got, want, m.err_msg())


def _t(shape, dtype, **kw):
    return m.Tensor(shape, dtype, PTR, **kw)


def _h(t):
    return t.handle if t is not None else None


@pytest.mark.parametrize("M,K,N,wrong", [(8, 4096, 4096, None), (300, 2048, 1536, None), (8, 4096, 4096, "scale"), (8, 4096, 4096, "out"), (0, 4096, 64, None)])
def test_quant_matmul_v5(M, K, N, wrong):
    x1, x2 = _t((M, K), m.ACL_INT8), _t((N, K), m.ACL_INT8)
    s1, s2 = _t((M,), m.ACL_FLOAT), _t((N + (wrong == "scale"),), m.ACL_FLOAT)
    bias, y = _t((N,), m.ACL_BF16), (None if wrong == "out" else _t((M, N), m.ACL_BF16))
    for b in (None, bias):
        _same(m.quant_matmul_v5_get_workspace(x1, x2, s1, s2, y, bias=b, transpose_x2=True),
              _ctypes("aclnnQuantMatmulV5GetWorkspaceSize", x1.handle, x2.handle, s1.handle, s2.handle, None, None, None, None, _h(b), False, True, 0, _h(y)))
    assert m.quant_matmul_v5_get_workspace(x1, x2, s1, s2, y, transpose_x2=True, ws_ptr=False)[0] != 0
    assert m.quant_matmul_v5_get_workspace(x1, x2, s1, s2, y, transpose_x2=True, ex_ptr=False)[0] != 0


@pytest.mark.parametrize("group,off", [(128, True), (64, False), (0, False), (33, False)])
def test_weight_quant(group, off):
    M, K, N = 16, 4096, 1024
    G = max(1, -(-K // group) if group else 1)
    x, w, y = _t((M, K), m.ACL_FLOAT16), _t((K, N), m.ACL_INT4), _t((M, N), m.ACL_FLOAT16)
    s = _t((G, N), m.ACL_FLOAT16)
    o = _t((G, N), m.ACL_FLOAT16) if off else None
    _same(m.weight_quant_batch_matmul_get_workspace(x, w, s, y, offset=o, group_size=group),
          _ctypes("aclnnWeightQuantBatchMatmulV2GetWorkspaceSize", x.handle, w.handle, s.handle, _h(o), None, None, None, group, y.handle))


@pytest.mark.parametrize("rows", [0, 5, 300])
def test_quantizers(rows):
    K = 2048
    x, q8, s = _t((rows, K), m.ACL_BF16), _t((rows, K), m.ACL_INT8), _t((rows,), m.ACL_FLOAT)
    f8, sb, sm = _t((rows, K), m.ACL_FLOAT8_E4M3FN), _t((rows, K // 128), m.ACL_FLOAT), _t((rows, K // 64, 2), m.ACL_FLOAT8_E8M0)
    _same(m.dynamic_quant_get_workspace(x, q8, s), _ctypes("aclnnDynamicQuantGetWorkspaceSize", x.handle, None, q8.handle, s.handle))
    _same(m.dynamic_quant_get_workspace(x, q8, sb), _ctypes("aclnnDynamicQuantGetWorkspaceSize", x.handle, None, q8.handle, sb.handle))
    for mode in (b"rint", b"no such", None, C.c_char_p(b"rint")):
        _same(m.dynamic_block_quant_get_workspace(x, f8, sb, round_mode=mode),
              _ctypes("aclnnDynamicBlockQuantGetWorkspaceSize", x.handle, 0.0, mode, m.ACL_FLOAT8_E4M3FN, 1, 128, f8.handle, sb.handle))
        _same(m.dynamic_mx_quant_get_workspace(x, f8, sm, round_mode=mode),
              _ctypes("aclnnDynamicMxQuantGetWorkspaceSize", x.handle, -1, mode, m.ACL_FLOAT8_E4M3FN, 32, 0, f8.handle, sm.handle))


def test_phase_2_refuses_as_through_ctypes():
    lib = m.lib()
    for name in ("aclnnQuantMatmulV5", "aclnnWeightQuantBatchMatmulV2", "aclnnDynamicQuant", "aclnnDynamicBlockQuant", "aclnnDynamicMxQuant"):
        fn = C.CDLL(m.LIB_PATH)[name]
        fn.restype, fn.argtypes = m.binding._SIGS[name]
        assert getattr(lib, name)(None, 0, None, None) == fn(None, 0, None, None) != 0
        assert getattr(lib, name)(None, 0, 4096, None) == fn(None, 0, 4096, None) != 0       # no live executor
        some = (C.c_char * 16)()
        for args in ((C.c_void_p(), C.c_uint64(0), C.c_void_p(4096), None), (some, 16, 4096, C.c_void_p(64)), (C.byref(some), 2 ** 64 - 1, some, None)):
            assert getattr(lib, name)(*args) == fn(*args) != 0
        with pytest.raises((TypeError, C.ArgumentError)):
            getattr(lib, name)(None, 0, None)
        with pytest.raises((TypeError, C.ArgumentError)):
            getattr(lib, name)(None, 0.5, None, None)


@pytest.mark.parametrize("rank", [2, 3, 7, 8])
def test_an_extent_in_any_place_is_seen(rank):
    shape = [2] * (rank - 2) + [3, 64]
    x, y, s = _t(shape, m.ACL_BF16), _t(shape, m.ACL_INT8), _t(shape[:-1], m.ACL_FLOAT)
    rc, ws, ex = m.dynamic_quant_get_workspace(x, y, s)
    assert rc == 0, m.err_msg()
    m.check(m.lib().aclDestroyAclOpExecutor(ex))
    for at in range(rank):
        other = list(shape)
        other[at] += 1
        assert m.dynamic_quant_get_workspace(x, _t(other, m.ACL_INT8), s)[0] != 0, at
        if at < rank - 1:
            assert m.dynamic_quant_get_workspace(x, y, _t(other[:-1], m.ACL_FLOAT))[0] != 0, at


def test_a_binding_that_failed_leaves_nothing_behind(monkeypatch):
    def fail(library):
        raise OSError("not this one")

    monkeypatch.setattr(m.binding, "_lib", None)
    monkeypatch.setattr(m.binding, "_bind_calls", fail)
    for _ in range(2):
        with pytest.raises(OSError, match="not this one"):
            m.lib()


def test_threads_find_the_library_whole(monkeypatch):
    bind, entered, go, seen = m.binding._bind_calls, threading.Event(), threading.Event(), []

    def slow(library):
        entered.set()
        assert go.wait(30)
        bind(library)

    monkeypatch.setattr(m.binding, "_lib", None)
    monkeypatch.setattr(m.binding, "_bind_calls", slow)
    first = threading.Thread(target=lambda: seen.append(m.lib()))
    first.start()
    assert entered.wait(30)
    second = threading.Thread(target=lambda: seen.append(m.lib()))
    second.start()
    second.join(0.2)
    early = list(seen)
    go.set()
    first.join(30)
    second.join(30)
    assert early == [] and len(seen) == 2 and seen[0] is seen[1]


# Arguments as ctypes takes them: an int of any size counts by its low bits, a ctypes number only as the parameter's own type.
PHASE_1_NUMBERS = [0, 128, True, 2 ** 64 + 128, -1, 2 ** 63, C.c_int64(128), C.c_int(128), C.c_float(128.0), C.c_void_p(128), 128.0, "128", None]


def _outcome(fn, *args):
    try:
        got = fn(*args)
    except Exception as e:
        return "refused", isinstance(e, (TypeError, C.ArgumentError))
    if isinstance(got, tuple):
        if got[2]:
            m.check(m.lib().aclDestroyAclOpExecutor(got[2]))
        got = got[0], got[1], got[2] is None
    return got


@pytest.mark.parametrize("number", PHASE_1_NUMBERS, ids=repr)
def test_phase_1_takes_the_numbers_that_ctypes_takes(number):
    K, N = 4096, 1024
    x, w, y, s = _t((16, K), m.ACL_FLOAT16), _t((K, N), m.ACL_INT4), _t((16, N), m.ACL_FLOAT16), _t((K // 128, N), m.ACL_FLOAT16)
    assert _outcome(lambda: m.weight_quant_batch_matmul_get_workspace(x, w, s, y, group_size=number)) == _outcome(
        lambda: _ctypes("aclnnWeightQuantBatchMatmulV2GetWorkspaceSize", x.handle, w.handle, s.handle, None, None, None, None, number, y.handle))
    x1, x2, s1, s2, out = _t((8, K), m.ACL_INT8), _t((N, K), m.ACL_INT8), _t((8,), m.ACL_FLOAT), _t((N,), m.ACL_FLOAT), _t((8, N), m.ACL_BF16)
    for group, flag in ((number, True), (0, number)):
        assert _outcome(lambda: m.quant_matmul_v5_get_workspace(x1, x2, s1, s2, out, group_size=group, transpose_x2=flag)) == _outcome(
            lambda: _ctypes("aclnnQuantMatmulV5GetWorkspaceSize", x1.handle, x2.handle, s1.handle, s2.handle, None, None, None, None, None, False, flag,
                            group, out.handle))
    q, sb, sm = _t((8, K), m.ACL_FLOAT8_E4M3FN), _t((8, K // 128), m.ACL_FLOAT), _t((8, K // 64, 2), m.ACL_FLOAT8_E8M0)
    xb = _t((8, K), m.ACL_BF16)
    for low, block in ((0.0, number), (number, 128)):
        assert _outcome(lambda: m.dynamic_block_quant_get_workspace(xb, q, sb, min_scale=low, col_block=block)) == _outcome(
            lambda: _ctypes("aclnnDynamicBlockQuantGetWorkspaceSize", xb.handle, low, b"rint", m.ACL_FLOAT8_E4M3FN, 1, block, q.handle, sb.handle))
    for axis, mode in ((number, b"rint"), (-1, number)):
        if isinstance(mode, (int, C.c_void_p)):   # (an address of text for ctypes)
            continue
        assert _outcome(lambda: m.dynamic_mx_quant_get_workspace(xb, q, sm, axis=axis, round_mode=mode)) == _outcome(
            lambda: _ctypes("aclnnDynamicMxQuantGetWorkspaceSize", xb.handle, axis, mode, m.ACL_FLOAT8_E4M3FN, 32, 0, q.handle, sm.handle))


@pytest.mark.parametrize("name", ["aclnnQuantMatmulV5", "aclnnQuantMatmulWeightNz", "aclnnWeightQuantBatchMatmulV2", "aclnnDynamicQuant",
                                  "aclnnDynamicBlockQuant", "aclnnDynamicMxQuant"])
def test_phase_2_takes_the_arguments_that_ctypes_takes(name):
    class Value:
        value = 4096

    fn = C.CDLL(m.LIB_PATH)[name]
    fn.restype, fn.argtypes = m.binding._SIGS[name]
    some = (C.c_char * 16)()
    for odd in (C.c_int(4096), C.c_uint64(4096), C.c_void_p(4096), Value(), 4096.0, "4096", b"4096", some, C.byref(some), -1, 2 ** 64 + 4096):
        for at in range(4):
            if at == 3 and not isinstance(odd, (C.c_int, C.c_uint64, Value, float)):
                continue   # (a stream is used as one)
            args = [None, 0, 4096, None]
            args[at] = odd
            assert _outcome(getattr(m.lib(), name), *args) == _outcome(fn, *args), (odd, at)


def test_an_object_that_is_no_tensor():
    x, y, s = _t((8, 2048), m.ACL_BF16), _t((8, 2048), m.ACL_INT8), _t((8,), m.ACL_FLOAT)
    with pytest.raises(AttributeError):
        m.dynamic_quant_get_workspace(x, 4096, s)
    gone = _t((8,), m.ACL_FLOAT)
    gone.destroy()
    assert m.dynamic_quant_get_workspace(x, y, gone)[0] != 0


def test_without_the_extension(monkeypatch, tmp_path):
    """A tree with the C library alone, or with an extension for another interpreter: the same answers through ctypes."""
    monkeypatch.setattr(m.binding, "CALLS_PATH", str(tmp_path / "none.so"))
    monkeypatch.setattr(m.binding, "_lib", None)
    monkeypatch.setattr(m.binding, "_calls", m.binding._NoCalls())
    test_quant_matmul_v5(8, 4096, 4096, None)
    test_quant_matmul_v5(8, 4096, 4096, "scale")
    test_weight_quant(128, True)
    test_quantizers(5)
    test_phase_2_takes_the_arguments_that_ctypes_takes("aclnnQuantMatmulV5")


def _make(*args):
    csrc = os.path.join(os.path.dirname(m.LIB_PATH), "..", "csrc")
    return subprocess.run(["make", "-n", "-B", "-C", csrc, *args], check=True, capture_output=True, text=True).stdout


def test_the_c_library_is_built_without_python():
    assert "opsnn_calls" + sysconfig.get_config_var("EXT_SUFFIX") in _make(f"PYTHON={sys.executable}")
    rest = _make("PYTHON=/no/python")
    assert "opsnn_calls" not in rest and "Python" not in rest and "libopsnn_amd.so" in rest and "examples/" in rest
