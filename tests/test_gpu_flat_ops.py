"""The sum of a whole array in two launches, and the elementwise forms whose
operands are contiguous or one repeated element: sizes at the edges of a
float4, of a workgroup's pass and of the switch to two launches, aligned and
one float off alignment."""

from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    from ttrl_amd.engine.device import open_device

    return open_device(0)


def _array(dev, x, off):
    """x on the device, starting `off` floats into an allocation."""
    from ttrl_amd.engine.tensor import DeviceArray

    whole = DeviceArray(dev, (x.size + off,))
    view = whole.view(off, x.shape)
    view.upload(x)
    return view


@pytest.mark.parametrize("off", [0, 1])
@pytest.mark.parametrize("n", [1, 3, 255, 1024, 16384, 16385, 16387, 1 << 20, 5308417])
def test_sum_of_a_whole_array(dev, n, off):
    from ttrl_amd.engine.ops import _kernels as K

    x = np.random.default_rng(n).standard_normal(n).astype(np.float32)
    got = float(K.sum_all(_array(dev, x, off)).numpy().reshape(-1)[0])
    # Longest chain of float32 additions: a thread's share of a workgroup's
    # range (four sums where the loads are vectors, one where they are not),
    # the four sums, a wavefront's six folds and its four, and the same again
    # for the parts; each addition rounds by at most 2^-24 of the sum of magnitudes.
    chunk = n if n <= 16384 else max(1024, -(-n // 1024) + 3)
    steps = -(-chunk // 256) + 3 + 2 * (2 + 6 + 4) + 4
    assert abs(got - x.astype(np.float64).sum()) <= steps * 2.0 ** -24 * np.abs(x).astype(np.float64).sum()


@pytest.mark.parametrize("off", [0, 1])
@pytest.mark.parametrize("shapes", [((7,), (7,)), ((1, 1), (3, 5)), ((3, 5), (1, 1)), ((1,), (1,)), ((129, 33), (129, 33)),
                                    ((1, 4, 1), (1, 4, 1)), ((2, 1, 8), (2, 1, 8)), ((5, 4), (1, 4)), ((5, 1), (5, 4))])
@pytest.mark.parametrize("op", ["add", "mul", "sub"])
def test_elementwise_forms(dev, op, shapes, off):
    from ttrl_amd.engine.ops import _kernels as K

    rng = np.random.default_rng(5)
    a, b = (rng.standard_normal(s).astype(np.float32) for s in shapes)
    f = {"add": np.add, "mul": np.multiply, "sub": np.subtract}[op]
    got = K.binary(op, _array(dev, a, off), _array(dev, b, off)).numpy()
    assert np.array_equal(got, f(a, b))


@pytest.mark.parametrize("shape", [(1,), (3,), (4, 5), (1, 1), (257, 9)])
def test_one_element_repeated(dev, shape):
    from ttrl_amd.engine.ops import _kernels as K

    a = np.float32(1.25) * np.ones((1,) * len(shape), np.float32)
    assert np.array_equal(K.repeat_to(_array(dev, a, 1), shape).numpy(), np.broadcast_to(a, shape))
