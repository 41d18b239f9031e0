"""The extension behind the ops (csrc/torch_binding.cpp): what it refuses is left to the Python ops, and what it runs
gives the bits the same call gives through ctypes."""
import ctypes
import sys
import warnings

import numpy as np
import pytest
import torch

from helpers import make_inputs_np, to_dev
from tuna_amd import _lib, ops


def test_refused_arguments_are_left_to_the_python_op():
    n = _lib.native()
    x, q = torch.zeros(16, 64, dtype=torch.float16), torch.zeros(8, 8, 32, dtype=torch.uint8)
    s, c, o = torch.zeros(64), torch.zeros(16), torch.zeros(16, 64, dtype=torch.float16)
    assert n.matmul(x, q, s, c, o, 64, 16, 64) is None            # CPU tensors
    assert n.matmul(x, q, s, c, o, 64, 16) is None                # an argument short
    assert n.matmul(None, q, s, c, o, "64", 16, 1 << 40) is None  # no tensor, no int, no 32-bit int
    assert n.matmul_multi([]) is None and n.matmul_multi([(x, q)]) is None and n.matmul_multi(7) is None
    assert n.matmul_grouped(x, q, s, c, o, 64, 1, 64, (0, 16, 16)) is None
    assert n.dequant(q, s, c, o, 64, 64, 48) is None and n.quantize(x, c, None) is None
    with pytest.raises(ValueError):
        n.bind((1, 2))


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k", [(256, 1, 512), (512, 33, 1024)])
def test_ops_through_the_extension_equal_the_ctypes_calls(m, n, k):
    L = _lib.lib()
    q, x, code, absmax = make_inputs_np(m, n, k, seed=m + n)
    q, x, c, s = to_dev(q, x, code, absmax)
    bs = torch.rand(m, k // 64, device="cuda") + 0.5
    res = torch.randn(n, m, device="cuda").half()
    offs = (0, n // 3, n)
    side = torch.cuda.Stream()
    torch.cuda.synchronize()

    def new(*shape):
        return torch.full(shape, float("nan"), dtype=torch.float16, device="cuda")

    def both(shape, op, raw):
        a, b = new(*shape), new(*shape)
        torch.cuda.synchronize()
        with torch.cuda.stream(side):
            op(a)
        assert raw(b.data_ptr(), torch.cuda.current_stream().cuda_stream) == _lib.OK
        torch.cuda.synchronize()
        assert torch.equal(a.view(torch.int16), b.view(torch.int16))

    p = [t.data_ptr() for t in (q, x, c, s)]
    both((n, m), lambda o: ops.matmul(x, q, s, c, o, m, n, k), lambda o, st: L.tuna_matmul(*p, o, m, n, k, st))
    both((n, m), lambda o: ops.matmul_fused(x, q, s, c, o, m, n, k, _lib.EPILOGUE_RESIDUAL, res),
         lambda o, st: L.tuna_matmul_fused(*p, o, m, n, k, None, 1, _lib.EPILOGUE_RESIDUAL, res.data_ptr(), st))
    both((n, m // 2), lambda o: ops.matmul_fused(x, q, s, c, o, m, n, k, _lib.EPILOGUE_SILU_MUL),
         lambda o, st: L.tuna_matmul_fused(*p, o, m, n, k, None, 1, _lib.EPILOGUE_SILU_MUL, None, st))
    both((n, m), lambda o: ops.matmul_blockwise(x, q, bs, c, o, m, n, k, 64),
         lambda o, st: L.tuna_matmul_blockwise(q.data_ptr(), x.data_ptr(), c.data_ptr(), bs.data_ptr(), o, m, n, k, 64, st))
    both((n, m), lambda o: ops.matmul_multi([(x, q, s, c, o, m, n, k)]),
         lambda o, st: L.tuna_matmul_multi((_lib.GemmProblem * 1)(_lib.GemmProblem(*p, o, m, n, k)), 1, st))
    both((n, m // 2), lambda o: ops.matmul_grouped(x, q, s, c, o, m // 2, 2, k, offs),
         lambda o, st: L.tuna_matmul_grouped(*p, o, m // 2, 2, k, (ctypes.c_int * 3)(*offs), None, 1, st))
    both((m, k), lambda o: ops.dequant(q, s, c, o, m, k), lambda o, st: L.tuna_dequant(q.data_ptr(), s.data_ptr(), c.data_ptr(), o, m, k, st))
    both((m, k), lambda o: ops.dequant(q, bs, c, o, m, k, block_size=64),
         lambda o, st: L.tuna_dequant_blockwise(q.data_ptr(), bs.data_ptr(), c.data_ptr(), o, m, k, 64, 2, st))
    w = torch.randn(m, k, device="cuda").half()
    for block in (None, 64):
        a, b = ops.quantize(w, c, block), ops.quantize(w, None, block)  # (no codebook: the Python path)
        q2, s2 = torch.empty_like(a[0]), torch.empty_like(a[1])
        assert L.tuna_quantize_blockwise(w.data_ptr(), c.data_ptr(), q2.data_ptr(), s2.data_ptr(), m, k, block or k,
                                         torch.cuda.current_stream().cuda_stream) == _lib.OK
        torch.cuda.synchronize()
        assert torch.equal(a[0], q2) and torch.equal(a[1], s2) and a[2] is c
        assert b[0].shape == a[0].shape and b[1].shape == a[1].shape


@pytest.fixture
def no_extension(monkeypatch):
    """As where _native.so was not built: its import fails."""
    monkeypatch.setitem(sys.modules, "tuna_amd._native", None)
    monkeypatch.setattr(_lib, "_native", None)


def test_without_the_extension_the_ops_take_the_ctypes_path(no_extension):
    x, q = torch.zeros(16, 64, dtype=torch.float16), torch.zeros(8, 8, 32, dtype=torch.uint8)
    s, c, o = torch.zeros(64), torch.zeros(16), torch.zeros(16, 64, dtype=torch.float16)
    with pytest.warns(RuntimeWarning, match="_native.so"):
        n = _lib.native()
    with warnings.catch_warnings():
        warnings.simplefilter("error")  # (once is enough)
        with _lib.diagnostic_build():
            assert _lib.native() is n
        for call in (lambda: ops.matmul(x, q, s, c, o, 64, 16, 64), lambda: ops.matmul_blockwise(x, q, s, c, o, 64, 16, 64, 64),
                     lambda: ops.matmul_fused(x, q, s, c, o, 64, 16, 64, _lib.EPILOGUE_RESIDUAL, o),
                     lambda: ops.matmul_multi([(x, q, s, c, o, 64, 16, 64)]), lambda: ops.matmul_grouped(x, q, s, c, o, 64, 1, 64, (0, 16)),
                     lambda: ops.dequant(q, s, c, o, 64, 64), lambda: ops.quantize(x, c)):
            with pytest.raises(ValueError, match="HIP device"):  # the Python op's own words for CPU tensors
                call()


@pytest.mark.gpu
def test_without_the_extension_the_ops_give_the_same_bits(no_extension):
    q, x, code, absmax = make_inputs_np(512, 16, 1024, seed=9)
    q, x, c, s = to_dev(q, x, code, absmax)
    o, o2 = (torch.empty(16, 512, dtype=torch.float16, device="cuda") for _ in range(2))
    with pytest.warns(RuntimeWarning):
        ops.matmul(x, q, s, c, o, 512, 16, 1024)
    assert _lib.lib().tuna_matmul(*[t.data_ptr() for t in (q, x, c, s, o2)], 512, 16, 1024, torch.cuda.current_stream().cuda_stream) == _lib.OK
    torch.cuda.synchronize()
    assert torch.equal(o.view(torch.int16), o2.view(torch.int16))


@pytest.mark.gpu
def test_ops_follow_the_active_library():
    q, x, code, absmax = make_inputs_np(256, 16, 512, seed=3)
    q, x, c, s = to_dev(q, x, code, absmax)
    o, o2 = (torch.empty(16, 256, dtype=torch.float16, device="cuda") for _ in range(2))
    ops.matmul(x, q, s, c, o, 256, 16, 512)
    with _lib.diagnostic_build():
        ops.matmul(x, q, s, c, o2, 256, 16, 512)
    torch.cuda.synchronize()
    assert np.array_equal(o.cpu().numpy(), o2.cpu().numpy())
    with pytest.raises(TypeError):
        ops.matmul(x.float(), q, s, c, o, 256, 16, 512)
