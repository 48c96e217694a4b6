"""The backward with a depth gradient gives a lane two pixels from four triangles a 16x16
tile on, else four.  The same triangles on both sides of that rule (degenerate ones added
to the list, which no pixel shows), upstream gradients on one pixel: every sum then has
one term, so the two agree in every value.  Sums of many terms have the float64 tests of
test_gpu_backward.py, on both sides too."""
import numpy as np
import pytest
import torch

from jaxrenderer_amd.autograd import render_differentiable
from tests.test_gpu_backward import SHADERS, _leaves, _many

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shader", SHADERS, ids=lambda s: s.__name__)
@pytest.mark.parametrize("size", [(48, 40), (51, 39)], ids=str)
def test_two_and_four_pixels_a_lane(shader, size):
    dev = torch.device("cuda")
    cam, faces, extra = _many(shader, 8, *size, 20)
    tiles = -(-size[0] // 16) * -(-size[1] // 16)
    faces = np.asarray(faces)
    assert len(faces) < 4 * tiles
    padded = np.concatenate([faces, np.zeros((4 * tiles, 3), faces.dtype)])
    W, H = size
    sides = []
    for f in (faces, padded):
        L, cam32, extra32 = _leaves(cam, extra, torch.float32, dev)
        zb, cv = render_differentiable(cam32, shader, f, extra32, W, H)
        sides.append((L, zb, cv))
    assert torch.equal(sides[0][1], sides[1][1]) and torch.equal(sides[0][2], sides[1][2])
    # the four corners of a 2x2 block, and a pixel of every eighth of those that are drawn
    drawn = torch.nonzero(sides[0][1] < 1.0)
    picks = [drawn[len(drawn) * k // 8] for k in range(8)]
    i, j = (int(v) & ~1 for v in drawn[len(drawn) // 2])
    picks += [(i + a, j + b) for a in (0, 1) for b in (0, 1)]
    moved = 0
    for i, j in picks:
        grads = []
        for L, zb, cv in sides:
            loss = 1.75 * zb[i, j] + (cv[i, j] * torch.tensor([0.5, -1.25, 2.0], device=dev)).sum()
            grads.append(torch.autograd.grad(loss, list(L.values()), allow_unused=True,
                                             retain_graph=True))
        for name, a, b in zip(sides[0][0], *grads):
            assert (a is None) == (b is None), name
            if a is not None:
                assert torch.equal(a, b), (name, int(i), int(j), float((a - b).abs().max()))
                moved += bool((a != 0).any())
    assert moved > 12
