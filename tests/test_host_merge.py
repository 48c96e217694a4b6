"""The host side's stacked forms against the ones that they stand for, bit for bit:
inv_stack against inv, merge_objects against Camera.apply_pos and apply_vec of each
object, upload against to_device."""
import numpy as np
import pytest
import torch

from jaxrenderer_amd import _plan
from jaxrenderer_amd.geometry import Camera, asf32, inv, inv_stack
from jaxrenderer_amd.model import Model, ModelObject, merge_objects

f32 = np.float32


def same_bits(a, b):
    a, b = np.asarray(a), np.asarray(b)
    assert a.dtype == b.dtype and a.shape == b.shape
    nan = np.isnan(a)
    assert np.array_equal(nan, np.isnan(b))
    assert np.array_equal(a.view(np.uint32)[~nan], b.view(np.uint32)[~nan])


@pytest.mark.parametrize("kind", ["plain", "zero row", "zero column", "ties", "nan", "inf",
                                  "permutation", "subnormal", "huge"])
def test_inv_stack(kind):
    rng = np.random.default_rng(3)
    A = rng.normal(size=(64, 4, 4)).astype(f32)
    if kind == "zero row":
        A[np.arange(64), rng.integers(0, 4, 64)] = 0
    elif kind == "zero column":
        A[np.arange(64), :, rng.integers(0, 4, 64)] = 0
    elif kind == "ties":
        A = np.round(A)
    elif kind in ("nan", "inf"):
        A[np.arange(64), rng.integers(0, 4, 64), rng.integers(0, 4, 64)] = float(kind)
    elif kind == "permutation":
        A = np.eye(4, dtype=f32)[np.stack([rng.permutation(4) for _ in range(64)])]
    elif kind == "subnormal":
        A = A * f32(1e-39)
    elif kind == "huge":
        A = A * f32(1e30)
    with np.errstate(all="ignore"):
        same_bits(inv_stack(A), np.stack([inv(a) for a in A]))


@pytest.mark.parametrize("seed", range(6))
def test_merge_objects_is_each_object_by_itself(seed):
    rng = np.random.default_rng(seed)
    objs = []
    for k in range(1 + seed):
        v, n = int(rng.integers(1, 40)), int(rng.integers(1, 30))  # 1 normal: summed in order
        T = rng.normal(size=(4, 4)).astype(f32)
        T[3] = [(0, 0, 0, 1), T[3], (0, 0, 0, 0)][k % 3]
        w, h = rng.integers(1, 9, 2)
        faces = rng.integers(0, min(v, n), (4, 3)).astype(np.int32)
        m = Model(rng.normal(size=(v, 3)).astype(f32), rng.normal(size=(n, 3)).astype(f32),
                  rng.random((v, 2)).astype(f32), faces, faces, faces,
                  rng.random((w, h, 3)).astype(f32), rng.random((w, h)).astype(f32))
        objs.append(ModelObject(m, local_scaling=rng.random(3).astype(f32), transform=T))
    with np.errstate(all="ignore"):
        got = merge_objects(objs)
        same_bits(got.verts, np.concatenate([
            Camera.apply_pos(asf32(o.model.verts) * o.local_scaling, o.transform) for o in objs]))
        same_bits(got.norms, np.concatenate([
            Camera.apply_vec(o.model.norms, np.ascontiguousarray(inv(o.transform).T))
            for o in objs]))
    step = got.offset
    for k, o in enumerate(objs):
        w, h = o.model.specular_map.shape
        part = got.specular_map[k * step:(k + 1) * step]
        assert np.array_equal(part[:w, :h], o.model.specular_map)
        assert part.sum() == pytest.approx(o.model.specular_map.sum(), rel=1e-5)


def test_upload():
    rng = np.random.default_rng(0)
    arrays = {"positions": rng.random((7, 3)), "faces": np.arange(9).reshape(3, 3),
              "uvs": np.zeros((0, 2)), "textures": rng.random((300, 300, 3)).astype(f32),
              "normals": torch.ones(5, 3), "clip": None, "tex_index": np.int64(4)}
    dev = torch.device("cpu")
    got = _plan.upload(arrays, dev)
    assert list(got) == list(arrays)
    for k, v in arrays.items():
        want = _plan.to_device(v, dev, k)
        if want is None:
            assert got[k] is None
            continue
        assert got[k].dtype == want.dtype and got[k].shape == want.shape
        assert got[k].is_contiguous() and torch.equal(got[k], want)
