"""The sine of a zero keeps its sign, as the double-precision function's does."""
import numpy as np

from test_trig import sincos  # noqa: F401  (the fixture)


def test_zeros(sincos):  # noqa: F811
    x = np.float32([0.0, -0.0, 1e-45, -1e-45])
    s, c = sincos(x)
    want = np.sin(x.astype(np.float64)).astype(np.float32)
    assert np.array_equal(s.view(np.int32), want.view(np.int32))
    assert np.array_equal(c, np.ones(4, np.float32))
