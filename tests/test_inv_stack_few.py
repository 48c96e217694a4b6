"""inv_stack inverts one or two matrices one by one and more together: the same bits."""
import numpy as np
import pytest

from jaxrenderer_amd.geometry import inv, inv_stack
from tests.test_host_merge import same_bits

f32 = np.float32


@pytest.mark.parametrize("n", [1, 2, 3])
@pytest.mark.parametrize("kind", ["plain", "moved", "singular", "nan"])
def test_few(n, kind):
    rng = np.random.default_rng(n)
    A = rng.normal(size=(n, 4, 4)).astype(f32)
    if kind == "moved":
        A[:] = np.identity(4)
        A[:, :3, 3] = rng.normal(size=(n, 3))
    elif kind == "singular":
        A[:, 2] = A[:, 1]
    elif kind == "nan":
        A[n - 1, 1, 2] = np.nan
    kept = A.copy()
    got = inv_stack(A)
    with np.errstate(all="ignore"):
        want = np.stack([inv(a) for a in A])
    same_bits(got, want)
    assert np.array_equal(A, kept, equal_nan=True)
    assert inv_stack(A[:0]).shape == (0, 4, 4)
