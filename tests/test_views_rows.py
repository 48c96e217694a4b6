"""render_views_differentiable with cameras given as arrays, as tensors and mixed: every
view is drawn with its own camera.

On the CPU the parameter rows that reach RenderFunction; on the GPU pictures and
gradients against render_differentiable view by view, with the bounds of
test_gpu_views.py (depth bit for bit, colours 1e-5, sums of gradients 1e-5 relative:
only the order of the atomic sums differs)."""
import numpy as np
import pytest
import torch

from jaxrenderer_amd import _raster, autograd, workloads
from jaxrenderer_amd.autograd import render_differentiable, render_views_differentiable
from jaxrenderer_amd.renderer import CameraParameters, Renderer
from jaxrenderer_amd.shaders import (DepthExtraInput, DepthShader, GouraudExtraInput, GouraudShader,
                                     GouraudTextureExtraInput, GouraudTextureShader,
                                     PhongTextureExtraInput, PhongTextureShader)
from jaxrenderer_amd.types import LightSource

f32 = np.float32
SHADERS = [DepthShader, GouraudShader, GouraudTextureShader, PhongTextureShader]
N_VIEWS = 4


def scene(shader, size=64):
    cams, faces, v, n, uv, col, texture = workloads.config4(
        seed=5, n_views=N_VIEWS, size=size, tex_size=32, n_lat=12, n_lon=16, perturbed=False)
    light = LightSource(direction=np.array((0.3, -0.5, 0.8), f32), colour=np.ones(3, f32))
    if shader is DepthShader:
        extra = DepthExtraInput(position=v)
    elif shader is GouraudShader:
        extra = GouraudExtraInput(position=v, colour=col, normal=n, light=light)
    elif shader is GouraudTextureShader:
        extra = GouraudTextureExtraInput(position=v, normal=n, uv=uv, light=light, texture=texture)
    else:
        extra = PhongTextureExtraInput(position=v, normal=n, uv=uv, light=light, texture=texture)
    return cams, faces, extra


def as_tensors(nt, dev, grad=False):
    return type(nt)(*(torch.tensor(np.asarray(v, f32), device=dev, requires_grad=grad)
                      for v in nt))


# which of the cameras are tensors, and whether the light is
KINDS = {"arrays": ((), False), "tensors": (range(N_VIEWS), False), "mixed": ((1, 3), False),
         "first a tensor": ((0,), False), "light a tensor": ((), True),
         "all tensors": (range(N_VIEWS), True)}


def given(kind, cams, extra, dev):
    which, light = KINDS[kind]
    cams = [as_tensors(c, dev) if b in which else c for b, c in enumerate(cams)]
    if light and hasattr(extra, "light"):
        extra = extra._replace(light=as_tensors(extra.light, dev))
    return cams, extra


class Stop(Exception):
    pass


@pytest.mark.parametrize("shader", SHADERS, ids=lambda s: s.__name__)
@pytest.mark.parametrize("kind", KINDS)
def test_each_row_holds_its_own_camera(kind, shader, monkeypatch):
    seen = {}

    def apply(call, params, *leaves):
        seen.update(call=call, params=params)
        raise Stop

    cpu = torch.device("cpu")
    monkeypatch.setattr(_raster, "require_device", lambda: cpu)
    monkeypatch.setattr(autograd.RenderFunction, "apply", apply)
    cams, faces, extra = scene(shader)
    given_cams, given_extra = given(kind, cams, extra, cpu)
    with pytest.raises(Stop):
        render_views_differentiable(given_cams, shader, faces, given_extra, 64, 64)
    rows = seen["params"].detach().numpy()
    assert rows.shape == (N_VIEWS, autograd.scene_rows(seen["call"].scenes).shape[1])
    for b, cam in enumerate(cams):
        for name in ("world_to_clip", "viewport", "world_to_eye_norm"):
            at, n = autograd._SLICES[name]
            assert np.array_equal(rows[b, at:at + n], np.asarray(getattr(cam, name)).reshape(-1)), (
                b, name)
    # and what the records hold beside the cameras
    assert np.array_equal(rows, autograd.scene_rows(seen["call"].scenes))


@pytest.mark.gpu
@pytest.mark.parametrize("shader", SHADERS[1:], ids=lambda s: s.__name__)
@pytest.mark.parametrize("kind", KINDS)
def test_views_are_the_single_pictures(kind, shader):
    dev = torch.device("cuda")
    W = H = 64
    cams, faces, extra = scene(shader)
    names = [k for k in ("position", "normal", "texture", "colour") if hasattr(extra, k)]

    def leaves(extra):
        return extra._replace(**{k: torch.tensor(np.asarray(getattr(extra, k), f32), device=dev,
                                                 requires_grad=True) for k in names})

    w = torch.as_tensor(np.random.default_rng(0).normal(size=(N_VIEWS, W, H, 3)),
                        device=dev).float()
    given_cams, given_extra = given(kind, cams, extra, dev)
    ex = leaves(given_extra)
    zb, cv = render_views_differentiable(given_cams, shader, faces, ex, W, H)
    got = torch.autograd.grad((w * cv).sum(), [getattr(ex, k) for k in names])
    total = [torch.zeros_like(g) for g in got]
    for b, cam in enumerate(cams):
        one = leaves(extra)
        zs, cs = render_differentiable(cam, shader, faces, one, W, H)
        assert int((zs < 1.0).sum()) > 100
        assert torch.equal(zs.view(torch.int32), zb[b].view(torch.int32)), b
        assert float((cs - cv[b]).detach().abs().max()) <= 1e-5
        for t, g in zip(total, torch.autograd.grad((w[b] * cs).sum(),
                                                   [getattr(one, k) for k in names])):
            t += g
    for name, a, b in zip(names, got, total):
        assert float((a - b).norm()) <= 1e-5 * max(float(b.norm()), 1e-6), name


@pytest.mark.gpu
def test_known_cameras_of_a_renderer():
    """Cameras as Renderer makes them, only the mesh's colours a leaf: each view's picture
    is the one of its own camera."""
    _, faces, extra = scene(GouraudShader)
    cams = [Renderer.create_camera_from_parameters(CameraParameters(
        viewWidth=48, viewHeight=40, hfov=60.0, vfov=50.0, position=p))
        for p in ((3.0, 0.2, 0.3), (0.1, 3.0, 0.4), (-2.0, -2.0, 1.0))]
    col = torch.tensor(np.asarray(extra.colour, f32), device="cuda", requires_grad=True)
    zb, cv = render_views_differentiable(cams, GouraudShader, faces, extra._replace(colour=col),
                                         48, 40)
    for b, cam in enumerate(cams):
        zs, _ = render_differentiable(cam, GouraudShader, faces, extra, 48, 40)
        assert int((zs < 1.0).sum()) > 100
        assert torch.equal(zs.view(torch.int32), zb[b].view(torch.int32)), b
    assert float(torch.autograd.grad(cv.sum(), col)[0].abs().sum()) > 0
