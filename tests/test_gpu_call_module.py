"""GPU: the call module (_t2h_pycall) and the ctypes binding of the same
library give the same bits and the same errors, and launches follow torch's
current stream."""
import numpy as np
import pytest
import torch

import oracle as orc
from _parity import to_dev
from t2h import _lib, ops

pytestmark = pytest.mark.gpu


def _args(dev, cols=1536, rows=9, eps=1e-6):
    x = to_dev(orc.randn(1, (rows, cols)), dev)
    sh, sc = (to_dev(orc.randn(i, (1, cols)), dev) for i in (2, 3))
    out = torch.empty_like(x)
    return out, (x.data_ptr(), out.data_ptr(), rows, cols, _lib.F32, eps, _lib.LN_MODULATE, sh.data_ptr(), sc.data_ptr(),
                 cols, None, 1, 0, ops._stream()), (x, sh, sc)


def test_same_bits_and_errors_as_ctypes(dev):
    L = _lib.load()
    fast = _lib._calls["t2h_ln_modulate"]
    assert fast is not L.t2h_ln_modulate
    a, args, keep = _args(dev)
    b = torch.empty_like(a)
    assert fast(*args) == 0
    assert L.t2h_ln_modulate(args[0], b.data_ptr(), *args[2:]) == 0
    assert torch.equal(a, b)
    bad = args[:3] + (-1,) + args[4:]
    assert fast(*bad) == L.t2h_ln_modulate(*bad) == _lib.T2H_EINVAL
    with pytest.raises(ValueError, match="bad shape"):
        _lib.call("t2h_ln_modulate", *bad)
    with pytest.raises(TypeError):
        fast(*args[:-1])
    with pytest.raises(TypeError):
        fast("x", *args[1:])


def test_launches_follow_the_current_stream(dev):
    s = torch.cuda.Stream()
    assert ops._stream() == torch.cuda.current_stream().cuda_stream
    with torch.cuda.stream(s):
        assert ops._stream() == s.cuda_stream == torch.cuda.current_stream().cuda_stream
    x = torch.zeros((64, 1536), device=dev)
    with torch.cuda.stream(s):
        s.wait_stream(torch.cuda.default_stream())
        torch.cuda._sleep(20_000_000)
        x.add_(1.0)
        y = ops.activation(x, ops.ACT_RELU)        # behind the add on s, or it would see zeros
    s.synchronize()
    assert np.array_equal(y.cpu().numpy(), np.ones((64, 1536), np.float32))
