"""The pixel box that k_setup takes from a triangle's projected corners
(vertex_box in jr_forward.hip, restated here in float32) holds every pixel that
the oracle's float32 edge functions cover: one triangle per scene, from ordinary
ones over slivers of any direction to ones of less than a pixel."""
import numpy as np
import pytest

from jaxrenderer_amd import _hip, _raster
from jaxrenderer_amd._plan import RasterCall
from jaxrenderer_amd.renderer import CameraParameters, Renderer
from oracle.oracle import run_oracle_plan

f32 = np.float32


def vertex_box(c, vp, W, H):
    """(known [N], box [N, 4] of i0, i1, j0, j1; empty where i0 > i1 or j0 > j1)
    of clip corners c [N, 3, 4]; each operation rounded to float32."""
    x, y, w = c[..., 0], c[..., 1], c[..., 3]
    wmin, wmax = w.min(1), w.max(1)
    xm = f32(max(abs(vp[0, 3]), abs(W - 1 - vp[0, 3])) / vp[0, 0])
    ym = f32(max(abs(vp[1, 3]), abs(H - 1 - vp[1, 3])) / vp[1, 1])
    m1, m2, xw, yw = np.abs(x).max(1), np.abs(y).max(1), xm * wmax, ym * wmax
    C1, C2 = np.maximum(m1, xw), np.maximum(m2, yw)
    known = (np.minimum(np.minimum(C1, C2), wmin) > 1e-10) & (
        np.maximum(np.maximum(C1, C2), wmax) < 1e12)
    v0 = np.stack([x[:, 0], y[:, 0], w[:, 0]], -1)
    e1 = np.stack([x[:, 1], y[:, 1], w[:, 1]], -1) - v0
    e2 = np.stack([x[:, 2], y[:, 2], w[:, 2]], -1) - v0

    def cross(a, b):
        s, t = [], []
        for p, q in ((1, 2), (2, 0), (0, 1)):
            s.append(a[:, p] * b[:, q])
            t.append(a[:, q] * b[:, p])
        s, t = np.stack(s, -1), np.stack(t, -1)
        return s - t, np.abs(s) + np.abs(t)

    (p, _), (q, _), (n, na) = cross(v0, e1), cross(v0, e2), cross(e1, e2)
    det_lo = np.abs((n * v0).sum(1, dtype=f32)) - f32(6e-7) * (na * np.abs(v0)).sum(1, dtype=f32)
    e = np.stack([8.1 * m1 + 3.1 * xw, 24.1 * m2 + 3.1 * yw, 59.2 * wmax], -1).astype(f32)
    S = f32(2.0**-24) * (e * (np.abs(p) + np.abs(q) + np.abs(q - p + n))).sum(1, dtype=f32)
    known &= det_lo > 0
    with np.errstate(all="ignore"):
        Hs = (S + f32(3e-11) * C1 * C2 * wmax) / det_lo
        rho = wmax / wmin
        KH = Hs * (1 + rho)
        known &= KH <= 0.4
        m = rho * Hs * (f32(1.1) + 4 * KH)
        u, v = x / w * vp[0, 0] + vp[0, 3], y / w * vp[1, 1] + vp[1, 3]
        du = m * (u.max(1) - u.min(1)) + f32(1 / 64)
        dv = m * (v.max(1) - v.min(1)) + f32(1 / 64)
        box = np.stack([np.maximum(np.ceil(u.min(1) - du), 0),
                        np.minimum(np.floor(u.max(1) + du), W - 1),
                        np.maximum(np.ceil(v.min(1) - dv), 0),
                        np.minimum(np.floor(v.max(1) + dv), H - 1)], -1)
    return known, box


def triangles(kind, rng, n):
    if kind == "small":
        a = rng.uniform(-2.5, 2.5, (n, 1, 3))
        return a + rng.normal(size=(n, 3, 3)) * 10.0 ** rng.uniform(-2.5, -0.5, (n, 1, 1))
    if kind == "sliver":  # two corners apart, the third within a hair of their line
        a, b = rng.uniform(-2.5, 2.5, (2, n, 3))
        t = rng.uniform(-0.2, 1.2, (n, 1))
        c = a + t * (b - a) + rng.normal(size=(n, 3)) * 10.0 ** rng.uniform(-5, -1, (n, 1))
        return np.stack([a, b, c], 1)
    if kind == "edge on":  # near a plane through the eye
        eye = np.array((0.0, -6.0, 2.0))
        d = rng.normal(size=(2, n, 3))
        k = rng.uniform(-1.0, 1.0, (2, n, 3))
        flat = eye + np.array((0.0, 6.0, -2.0)) + k[0][..., None] * d[0][:, None] * 0.7 + \
            k[1][..., None] * (eye + d[1])[:, None] * 0.3
        return flat + rng.normal(size=flat.shape) * 10.0 ** rng.uniform(-6, -2, (n, 1, 1))
    return rng.uniform(-4.0, 4.0, (n, 3, 3))  # large: some cross the eye's plane


@pytest.mark.parametrize("kind", ["small", "sliver", "edge on", "large"])
@pytest.mark.parametrize("size", [(40, 33), (7, 96)], ids=str)
def test_box_holds_every_covered_pixel(kind, size):
    W, H = size
    n = 1500
    rng = np.random.default_rng(len(kind) + W)
    pos = triangles(kind, rng, n).astype(f32)
    cam = Renderer.create_camera_from_parameters(CameraParameters(
        viewWidth=W, viewHeight=H, hfov=60.0, vfov=60.0, position=(0.0, -6.0, 2.0)))
    # both windings: whichever faces the eye is drawn
    both = np.concatenate([pos, pos[:, ::-1]])
    scenes = [_raster.scene_struct(world_to_clip=cam.world_to_clip, viewport=cam.viewport,
                                   tri_begin=k, tri_end=k + 1) for k in range(2 * n)]
    call = RasterCall(shader=_hip.SHADER_DEPTH, width=W, height=H, scenes=scenes,
                      inputs={"positions": both.reshape(-1, 3),
                              "faces": np.arange(6 * n, dtype=np.int32).reshape(-1, 3)},
                      n_slots=6 * n, n_tris=2 * n, want_canvas=False)
    seen = run_oracle_plan([call], prim_id=False, bary=False,
                           complexity=True)["main"]["complexity"].reshape(2, n, W, H)
    covered = (seen > 0).any(0)
    M = cam.world_to_clip
    clip = np.zeros((n, 3, 4), f32)
    for r in range(4):
        s = pos[..., 0] * M[r, 0]
        for k in (1, 2):
            s = s + pos[..., k] * M[r, k]
        clip[..., r] = s + M[r, 3]
    known, box = vertex_box(clip, cam.viewport, W, H)
    some = covered.reshape(n, -1).any(1)
    assert some.sum() > 100
    bad = 0
    for k in np.nonzero(known & some)[0]:
        i, j = np.nonzero(covered[k])
        i0, i1, j0, j1 = box[k]
        bad += not (i.min() >= i0 and i.max() <= i1 and j.min() >= j0 and j.max() <= j1)
    assert bad == 0
    # it does bound what a scene is made of, and an empty box is what saves the work
    empty = known & ((box[:, 0] > box[:, 1]) | (box[:, 2] > box[:, 3]))
    assert known.mean() > {"small": 0.9, "sliver": 0.3, "edge on": 0.02, "large": 0.1}[kind]
    assert kind != "small" or empty.sum() > 0.3 * (~some).sum()
