"""Triangles over many tiles: a wide-list entry's tiles are shared by
ceil(T / 256) wavefronts of a frame of T tiles, so its parts end on, before and
after a frame's last tile; and the tiles' list segments, taken 2,048 tiles at a
time.  Against the oracle, bit for bit."""
import pytest
import torch

from jaxrenderer_amd import _plan
from jaxrenderer_amd.shaders import DepthShader, PhongReflectionShadowTextureShader
from oracle.oracle import run_oracle_plan
from tests import scenes
from tests.parity import assert_parity

pytestmark = pytest.mark.gpu


# 8x8 tiles: T = 256 (one wavefront an entry), 272 and 512 (two), 1056 (five), 2048 (eight,
# one workgroup of segments), 2080 (two workgroups)
@pytest.mark.parametrize("size", [(128, 128), (136, 121), (256, 128), (259, 251), (512, 256),
                                  (517, 255)], ids=str)
@pytest.mark.parametrize("shader", [DepthShader, PhongReflectionShadowTextureShader],
                         ids=lambda s: s.__name__)
def test_wide_triangles(size, shader):
    def calls():
        return scenes.soup_call(shader, 11, *size, 30)

    ref = run_oracle_plan(calls())
    got = _plan.run_plan(calls(), prim_id=True, bary=True)
    torch.cuda.synchronize()
    for tag in ref:
        assert_parity(got[tag], ref[tag], label=f"wide/{size}/{tag}")
