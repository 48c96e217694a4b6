"""merge_objects takes every local_scaling that broadcasts against an object's vertices,
bit for bit as Camera.apply_pos of the scaled vertices."""
import numpy as np
import pytest

from jaxrenderer_amd.geometry import Camera, asf32
from jaxrenderer_amd.model import Model, ModelObject, merge_objects
from tests.test_host_merge import same_bits

f32 = np.float32
SHAPES = {"one factor": lambda rng, n: f32(rng.uniform(0.5, 2.0)),
          "[1]": lambda rng, n: rng.uniform(0.5, 2.0, 1),
          "per axis": lambda rng, n: rng.uniform(0.5, 2.0, 3).astype(f32),
          "list": lambda rng, n: [1.0, 2.0, 0.5],
          "[1, 3]": lambda rng, n: rng.uniform(0.5, 2.0, (1, 3)),
          "per vertex": lambda rng, n: rng.uniform(0.5, 2.0, (n, 1)).astype(f32),
          "per vertex and axis": lambda rng, n: rng.uniform(0.5, 2.0, (n, 3)).astype(f32)}


def obj(rng, n, scaling):
    faces = rng.integers(0, n, (5, 3)).astype(np.int32)
    T = rng.normal(size=(4, 4)).astype(f32)
    T[3] = (0, 0, 0, 1)
    return ModelObject(Model(rng.normal(size=(n, 3)).astype(f32),
                             rng.normal(size=(n, 3)).astype(f32), rng.random((n, 2)).astype(f32),
                             faces, faces, faces, rng.random((2, 2, 3)).astype(f32),
                             rng.random((2, 2)).astype(f32)),
                       local_scaling=scaling, transform=T)


@pytest.mark.parametrize("kind", list(SHAPES) + ["all of them"])
def test_local_scaling(kind):
    rng = np.random.default_rng(4)
    kinds = list(SHAPES) if kind == "all of them" else ["per axis", kind]
    objs = []
    for k in kinds:
        n = int(rng.integers(2, 40))
        objs.append(obj(rng, n, SHAPES[k](rng, n)))
    got = merge_objects(objs)
    same_bits(got.verts, np.concatenate([
        Camera.apply_pos((asf32(o.model.verts) * asf32(o.local_scaling)).astype(f32), o.transform)
        for o in objs]))
    at = 0
    for o, part in zip(objs, np.split(got.faces, len(objs))):
        assert np.array_equal(part, o.model.faces + at)
        at += len(o.model.verts)
