"""An attribute that a shader reads and that is None is refused, not read as an array of
one element past whose end the vertices' rows lie."""
import numpy as np
import pytest

from jaxrenderer_amd import _hip
from jaxrenderer_amd.autograd import render_differentiable
from jaxrenderer_amd.pipeline import build_call
from jaxrenderer_amd.shaders import BUILTIN
from tests import scenes

FIELDS = {"normal": "normals", "uv": "uvs", "colour": "colours", "texture_index": "tex_index"}


def without():
    for shader in BUILTIN:
        cam, faces, extra, shadow = scenes.soup_inputs(shader, 0)
        if shadow is not None:
            extra = extra._replace(shadow=extra.shadow._replace(
                shadow_map=np.ones((shadow.width, shadow.height), np.float32)))
        for field, name in FIELDS.items():
            if hasattr(extra, field):
                yield pytest.param(shader, cam, faces, extra._replace(**{field: None}), name,
                                   id=f"{shader.__name__}-{field}")


@pytest.mark.parametrize("shader,cam,faces,extra,name", without())
def test_none_stays_none(shader, cam, faces, extra, name):
    assert build_call(cam, shader, faces, extra, 48, 40).inputs[name] is None


@pytest.mark.gpu
@pytest.mark.parametrize("shader,cam,faces,extra,name", without())
def test_none_is_refused(shader, cam, faces, extra, name):
    with pytest.raises(_hip.HipError, match="needs? "):
        render_differentiable(cam, shader, faces, extra, 48, 40)
