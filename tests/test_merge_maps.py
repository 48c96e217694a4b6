"""Maps of different numbers of axes are refused, also where numpy would drop an axis."""
import numpy as np
import pytest

from jaxrenderer_amd.model import MergedModel


@pytest.mark.parametrize("shapes", [((2, 2), (1, 1, 1)), ((2, 2), (2, 2, 1)), ((2, 3), (1, 2, 3)),
                                    ((2, 2, 3), (2, 2)), ((4, 4), (4,))], ids=str)
def test_axes_differ(shapes):
    with pytest.raises((ValueError, IndexError)):
        MergedModel.merge_maps([np.ones(s, np.float32) for s in shapes])


def test_padded_and_stacked():
    a, b = np.arange(6, dtype=np.float32).reshape(2, 3) + 1, np.full((3, 1), 9, np.float32)
    merged, single = MergedModel.merge_maps([a, b])
    assert single == (3, 3) and merged.shape == (6, 3) and merged.dtype == np.float32
    assert np.array_equal(merged[:2], a) and not merged[2].any()
    assert np.array_equal(merged[3:, :1], b) and not merged[3:, 1:].any()
