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


def test_native_methods_leave_what_does_not_fit_to_the_python_ones():
    """A call that is not well-formed reaches the checks of the Python method, whatever is wrong with it."""
    from ojas_amd.backend import DTYPE, PLACEMENT, U32, MiBackend

    be = MiBackend.__new__(MiBackend)  # no device: nothing here gets as far as the library
    be._ctx, be._context = None, _native.Context(0)

    def dev(*shape, dtype=BF16):
        return DeviceTensor(be, 4096, shape, dtype, owns=False)

    host = np.zeros((2, 3), np.float32)
    for code, call in [
        (SHAPE, lambda: be.linear_forward(dev(2, 3), dev(4, 5))), (SHAPE, lambda: be.linear_forward(dev(2, 3), dev(3))),
        (SHAPE, lambda: be.linear_forward(dev(0, 3), dev(4, 3))), (DTYPE, lambda: be.linear_forward(dev(2, 3, dtype=U32), dev(4, 3))),
        (PLACEMENT, lambda: be.linear_forward(host, host)), (SHAPE, lambda: be.embedding_forward(dev(4), dev(2, dtype=U32))),
        (DTYPE, lambda: be.embedding_forward(dev(4, 3), dev(2))), (SHAPE, lambda: be.kv_cache_write(dev(1, 4, 2, 8), dev(1, 1, 2, 4, dtype=F32), 0)),
        (DTYPE, lambda: be.kv_cache_write(dev(1, 4, 2, 8), dev(1, 1, 2, 8), 0)),
        (SHAPE, lambda: be.cached_attention_forward(dev(1, 1, 4, 8, dtype=F32), dev(1, 4, 3, 8), dev(1, 4, 3, 8), 1)),
        (SHAPE, lambda: be.cached_attention_forward(dev(1, 1, 4, 8, dtype=F32), dev(1, 4, 2, 8), dev(1, 4, 2, 8), 1, window=0)),
        (DTYPE, lambda: be.cached_attention_forward(dev(1, 1, 4, 8), dev(1, 4, 2, 8), dev(1, 4, 2, 8), 1))]:
        with pytest.raises(OjasError) as e:
            call()
        assert e.value.code == code
    for call in (lambda: be.linear_forward(dev(2, 3), dev(4, 3), nonsense=1), lambda: be.linear_forward(dev(2, 3)),
                 lambda: be.linear_forward(dev(2, 3), dev(4, 3), None, 1), lambda: be.linear_forward(dev(2, 3), dev(4, 3), x=1)):
        with pytest.raises(TypeError):
            call()


@pytest.mark.parametrize("method", ["accumulate_grads", "muon_ns5_step_list", "adamw_step_batched"])
def test_lists_are_checked_as_each_of_their_entries_is(method):
    """A list op refuses what the op on one entry refuses, with its error: shapes (not sizes alone), dtypes, placement."""
    from ojas_amd.backend import DTYPE, PLACEMENT, U32, AdamWConfig, MiBackend, MuonNs5Config

    be = MiBackend.__new__(MiBackend)  # no device: nothing here gets as far as the library
    be._ctx, be._context = None, _native.Context(0)

    def dev(*shape, dtype=F32):
        return DeviceTensor(be, 4096, shape, dtype, owns=False)

    width = {"accumulate_grads": 2, "muon_ns5_step_list": 3, "adamw_step_batched": 4}[method]
    extra = {"accumulate_grads": (), "muon_ns5_step_list": (MuonNs5Config.nanolab_default(),),
             "adamw_step_batched": (0, AdamWConfig.nanolab(1e-3, 0.1))}[method]
    good = lambda: [[dev(4, 6) for _ in range(3)] for _ in range(width)]
    host = np.zeros((4, 6), np.float32)
    for code, bad in [(SHAPE, dev(6, 4)), (SHAPE, dev(24)), (DTYPE, dev(4, 6, dtype=U32)), (DTYPE, dev(4, 6, dtype=BF16)), (PLACEMENT, host)]:
        for which in range(1, width):
            lists = good()
            lists[which][2] = bad
            with pytest.raises(OjasError) as e:
                getattr(be, method)(*lists, *extra)
            assert e.value.code == code, (which, e.value)
    short = good()
    short[-1].pop()
    with pytest.raises(OjasError) as e:
        getattr(be, method)(*short, *extra)
    assert e.value.code == SHAPE
    empty = good()
    for ts in empty:
        ts[1] = dev(0, 6)
    with pytest.raises(OjasError) as e:
        getattr(be, method)(*empty, *extra)
    assert e.value.code == SHAPE


def test_ops_that_know_f32_alone_refuse_other_storage():
    from ojas_amd.backend import DTYPE, MiBackend

    be = MiBackend.__new__(MiBackend)
    be._ctx, be._context = None, _native.Context(0)
    dev = lambda dtype: DeviceTensor(be, 4096, (8,), dtype, owns=False)
    for call in (lambda: be.scale_grad(dev(BF16), 0.5), lambda: be.accumulate_grad(dev(BF16), dev(BF16)),
                 lambda: be.accumulate_grad(dev(F32), dev(BF16))):
        with pytest.raises(OjasError) as e:
            call()
        assert e.value.code == DTYPE


def test_the_package_imports_without_anything_built(tmp_path):
    """Names, constants, configurations and validators need no library; a backend or a tensor says what is missing."""
    import shutil
    import subprocess
    import sys
    from pathlib import Path

    package = Path(_native.__file__).resolve().parent
    (tmp_path / "ojas_amd").mkdir()
    for source in package.glob("*.py"):
        shutil.copy(source, tmp_path / "ojas_amd")
    program = """
import numpy as np
import ojas_amd, ojas_amd.autocast, ojas_amd.lora, ojas_amd.nanolab, ojas_amd.trainer
from ojas_amd import shapes
from ojas_amd.backend import BACKEND, F32, AdamWConfig, DeviceTensor, MiBackend, OjasError
assert shapes.linear_forward_dims(np.zeros((2, 4), np.float32), np.zeros((5, 4), np.float32))[0] == 2
assert AdamWConfig.nanolab(1e-3, 0.1).beta2 == 0.95
for make in (MiBackend, lambda: DeviceTensor(None, 0, (2, 3), F32)):
    try:
        make()
    except OjasError as e:
        assert e.code == BACKEND and "is not built" in e.detail, e
    else:
        raise AssertionError(make)
"""
    done = subprocess.run([sys.executable, "-c", program], cwd=tmp_path, capture_output=True, text=True)
    assert done.returncode == 0, done.stderr


class Named(DeviceTensor):
    def __init__(self, name, *args, **kwargs):
        super().__init__(*args, **kwargs)
        self.name = name


def test_a_tensor_is_an_ordinary_python_object():
    """Attributes, subclasses with an __init__ of their own, weak references, a shape and a dtype that can be set."""
    import gc
    import weakref

    from ojas_amd.backend import MiBackend

    t = DeviceTensor(None, 4096, (2, 3), F32, owns=False)
    t.label, t.me = "weights", t  # a cycle
    assert t.label == "weights" and t.__dict__["me"] is t
    gone = []
    ref = weakref.ref(t, gone.append)
    assert ref() is t
    del t
    gc.collect()
    assert ref() is None and gone == [ref]
    s = Named("q", None, 4096, [4, 6], BF16, owns=False)
    assert isinstance(s, DeviceTensor) and (s.name, s.shape, s.numel, s.nbytes) == ("q", (4, 6), 24, 48)
    assert weakref.ref(s)() is s and s.reshape(24).shape == (24,)
    s.shape, s.dtype = [3, 4], F32
    assert (s.shape, s.numel, s.nbytes) == ((3, 4), 12, 48)
    with pytest.raises(AttributeError):
        s.nothing
    with pytest.raises(TypeError):
        DeviceTensor(None, 0, (2,))
    # Operands of a subclass pass for tensors: what is wrong with this call is its shapes.
    be = MiBackend.__new__(MiBackend)
    be._ctx, be._context = None, _native.Context(0)
    for call in (lambda: be.linear_forward(Named("x", be, 4096, (2, 3), F32, owns=False), Named("w", be, 4096, (4, 5), F32, owns=False)),
                 lambda: be.accumulate_grads([Named("a", be, 4096, (2,), F32, owns=False)], [Named("g", be, 4096, (3,), F32, owns=False)])):
        with pytest.raises(OjasError) as e:
            call()
        assert e.value.code == SHAPE


@pytest.mark.gpu
def test_a_subclass_owns_its_memory_as_a_tensor_does():
    import gc

    from ojas_amd.backend import MiBackend

    be = MiBackend(0)
    live = be.budget()["live"]
    t = be.empty((1024,))
    t._owns = False  # handed over
    s = Named("moved", be, t.ptr, t.shape, t.dtype)
    del t
    assert be.budget()["live"] == live + 4096
    x = np.arange(1024, dtype=np.float32)
    _native.omx_upload(be._context, s, 0, x.ctypes.data, x.nbytes)
    assert np.array_equal(be.download(be.residual_add_forward(s, s)), x + x)
    s.me = s
    del s
    gc.collect()
    assert be.budget()["live"] == live
    be.close()
