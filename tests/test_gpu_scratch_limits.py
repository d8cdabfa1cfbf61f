"""Ops at the limits of their scratch memory: a full device or budget, and inside a captured graph."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def be():
    from ojas_amd.backend import MiBackend

    backend = MiBackend(0)
    yield backend
    backend.close()


def test_a_refused_allocation_leaves_the_next_op_alone(be):
    """More memory than the device has: the refusal is that call's own, and no later launch reports it."""
    from ojas_amd.backend import CAPACITY_EXCEEDED, OjasError

    print("allocation of 64 TiB", flush=True)
    x = be.upload(np.ones((4, 64), np.float32))
    with pytest.raises(OjasError) as e:
        be.empty((1 << 44,))
    assert e.value.code == CAPACITY_EXCEEDED
    assert np.array_equal(be.download(be.residual_add_forward(x, x)), np.full((4, 64), 2.0, np.float32))
