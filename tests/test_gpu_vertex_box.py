"""k_setup's own pixel boxes, and the triangles that it drops for them, against the
oracle bit for bit: the slivers, edge-on, tiny and large triangles of test_vertex_box.py,
each alone in its scene in both windings, behind a degenerate first triangle (a scene's
first triangle is never dropped).  Up to the 8,192 pixels a side for which a box is taken,
and past them."""
import numpy as np
import pytest
import torch

from jaxrenderer_amd import _hip, _plan, _raster
from jaxrenderer_amd._plan import RasterCall
from jaxrenderer_amd.renderer import CameraParameters, Renderer
from oracle.oracle import run_oracle
from tests.parity import assert_parity
from tests.test_vertex_box import triangles

pytestmark = pytest.mark.gpu
f32 = np.float32


def call_of(kind, W, H, n, **kw):
    rng = np.random.default_rng(len(kind) + W)
    pos = triangles(kind, rng, n).astype(f32)
    cam = Renderer.create_camera_from_parameters(CameraParameters(
        viewWidth=W, viewHeight=H, hfov=60.0, vfov=60.0, position=(0.0, -6.0, 2.0)))
    three = np.stack([np.zeros_like(pos), pos, pos[:, ::-1]], 1)  # [n, triangle, corner, 3]
    scenes = [_raster.scene_struct(world_to_clip=cam.world_to_clip, viewport=cam.viewport,
                                   tri_begin=3 * k, tri_end=3 * k + 3) for k in range(n)]
    return RasterCall(shader=_hip.SHADER_DEPTH, width=W, height=H, scenes=scenes,
                      inputs={"positions": three.reshape(-1, 3),
                              "faces": np.arange(9 * n, dtype=np.int32).reshape(-1, 3)},
                      n_slots=9 * n, n_tris=3 * n, want_canvas=False, **kw)


@pytest.mark.parametrize("kind", ["small", "sliver", "edge on", "large"])
@pytest.mark.parametrize("size,n", [((40, 33), 1500), ((7, 96), 1500), ((8192, 3), 600),
                                    ((8193, 3), 600), ((3, 8192), 600)], ids=str)
def test_every_covered_pixel_is_drawn(kind, size, n):
    call = call_of(kind, *size, n)
    ref = run_oracle(call)
    covered = (ref["prim_id"] >= 0).reshape(n, -1).any(1)
    assert covered.sum() > n // 200
    assert_parity(_plan.run(call, prim_id=True, bary=True), ref, label=f"{kind}/{size}")
    # the narrow form: depth keys only
    call = call_of(kind, *size, n, apply_offset=True, depth_offset=0.125)
    got = _plan.run(call)
    torch.cuda.synchronize()
    assert_parity(got, run_oracle(call, prim_id=False, bary=False), label=f"{kind}/{size}/narrow")
