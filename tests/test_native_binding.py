"""The native side of `MiBackend` (ojas_amd/_native): what needs no device."""
import numpy as np
import pytest

from ojas_amd import _native
from ojas_amd.backend import BF16, F32, SHAPE, DeviceTensor, OjasError


@pytest.mark.parametrize("shape, other, numel", [((2, 3, 4), (6, 4), 24), ((5,), (1, 5), 5), ((), (1,), 1), ((0, 7), (7, 0), 0)])
def test_tensor_sizes_and_views(shape, other, numel):
    t = DeviceTensor(None, 4096, shape, BF16, owns=False)
    assert (t.shape, t.numel, t.nbytes, t.dtype) == (shape, numel, 2 * numel, BF16)
    t.compute_bf16 = True
    for view in (t.reshape(other), t.reshape(list(other)), t.reshape(*other)):
        assert view.shape == other and view.ptr == t.ptr and view._base is t and view.compute_bf16 and not view._owns


def test_refusals(monkeypatch):
    with pytest.raises((OjasError, RuntimeError)) as e:
        DeviceTensor(None, 0, (2, 3), F32).reshape(4, 2)
    assert getattr(e.value, "code", SHAPE) == SHAPE
    with pytest.raises(TypeError):
        _native.omx_sync(5)  # not a context
    with pytest.raises(TypeError):
        _native.omx_sync(_native.Context(0), np.zeros(3))  # argument count
