"""What the renderer's speed is measured on: cases over the range that a user's program
puts it to, the inputs of each made from a seed, one pass of it through the public entry
points, and its outputs in 64 bits from a plain restatement of the image formation.

The kinds of cases:

* frame     one scene, one camera, replayed from a captured graph: a viewer or a dataset
            writer that shows one object.  Few triangles; launches and latency count.
* image     Renderer.get_camera_image of a list of objects, the call a program of the
            reference makes for every picture: objects merged, uploaded, rendered.
* batch     many scenes of uneven size in one replay: the camera observations of a vector
            of simulated environments, each environment seen by one or several cameras.
* rollout   the same after the objects have moved (ScenePoser.update, then the replay),
            with the 8-bit display images that a policy or a video takes.
* train     forward, L2 image loss and backward of a batch in one graph: inverse rendering
            of many scenes.  Returns the image and every gradient.
* views     forward and backward of one textured mesh seen by many cameras: texture and
            shape fitting from photographs.
* autograd  render_differentiable and torch.autograd.grad, one picture at a time: the
            renderer inside another program's autograd graph.
"""
import math

import numpy as np
import torch

from jaxrenderer_amd import batch, packing
from jaxrenderer_amd.autograd import build_views_call, render_differentiable
from jaxrenderer_amd.model import Model, ModelObject, merge_objects
from jaxrenderer_amd.pose import ScenePoser
from jaxrenderer_amd.renderer import (CameraParameters, LightParameters, Renderer,
                                      ShadowParameters)
from jaxrenderer_amd.shaders import (GouraudTextureExtraInput, GouraudTextureShader,
                                     PhongTextureDarbouxExtraInput, PhongTextureDarbouxShader,
                                     PhongTextureExtraInput, PhongTextureShader)
from jaxrenderer_amd.types import LightSource

f32 = np.float32


def listed():
    return [
        # one cube, the smallest picture that examples and tests draw
        dict(name="cube frame", kind="frame", mesh="cube", width=320, height=240),
        # one finely tessellated, textured object at a display's size
        dict(name="sphere frame", kind="frame", mesh="sphere", lat=48, tex=256, width=960,
             height=540),
        # one picture of a walker from its objects, with its shadow
        dict(name="camera image", kind="image", width=84, height=84),
        # 200 walkers, 3,276 triangles each, the shadow map as large as the picture
        dict(name="walker batch", kind="batch", scenes="walker", n=200, cameras=1, width=84,
             height=84, shadow=84),
        # 1,024 observations, some 320 to 11,000 triangles each, 256 x 256 shadow maps
        dict(name="coarse batch", kind="batch", scenes="coarse", n=1024, cameras=8, width=84,
             height=84, shadow=256),
        # an ordinary vector of environments, moved and then drawn as 8-bit images
        dict(name="rollout", kind="rollout", scenes="coarse", n=90, cameras=1, width=96,
             height=72, shadow=96),
        # pictures of a recording's size, no shadows: few scenes, many pixels
        dict(name="dense batch", kind="batch", scenes="dense", n=60, cameras=4, width=480,
             height=270, shadow=0),
        # the gradients of 1,024 observations
        dict(name="coarse train", kind="train", scenes="coarse", n=1024, cameras=8, width=84,
             height=84, shadow=256),
        # 512 pictures at 480 x 270 of 1,000 to 20,000 triangles: the largest step
        dict(name="dense train", kind="train", scenes="dense", n=512, cameras=8, width=480,
             height=270, shadow=512),
        # one mesh from 64 cameras, vertex lighting: nearly every pixel has its own texel
        dict(name="gouraud views", kind="views", shader="gouraud_texture", n=64, lat=50, tex=512,
             width=256, height=256),
        # ragged pictures, lighting per pixel, fewer views
        dict(name="phong views", kind="views", shader="phong", n=23, lat=37, tex=300, width=201,
             height=187),
        # a normal-mapped mesh through torch's autograd
        dict(name="normal map autograd", kind="autograd", shader="phong_darboux", lat=40, tex=256,
             width=512, height=512),
    ]


def draw(rng):
    """One more case of the ranges above; no larger than the largest of them."""
    def log(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["frame", "image", "batch", "rollout", "train", "views", "autograd"])
    if kind == "frame":
        if rng.random() < 0.3:
            return dict(kind=kind, mesh="cube", width=log(32, 960), height=log(32, 540))
        return dict(kind=kind, mesh="sphere", lat=log(4, 64), tex=log(8, 256),
                    width=log(64, 960), height=log(48, 540))
    if kind == "image":
        return dict(kind=kind, width=log(32, 320), height=log(32, 240))
    if kind in ("batch", "train"):
        scenes = rng.choice(["walker", "coarse", "dense"])
        dense = scenes == "dense"
        n = log(4, 96) if dense else log(4, 1024)
        return dict(kind=kind, scenes=scenes, n=n, cameras=1 if n < 64 else rng.choice([4, 8]),
                    width=log(200, 480) if dense else log(40, 128),
                    height=log(120, 270) if dense else log(40, 128),
                    shadow=rng.choice([0, log(64, 512 if dense else 256)]))
    if kind == "rollout":
        return dict(kind=kind, scenes=rng.choice(["walker", "coarse"]), n=log(4, 200), cameras=1,
                    width=log(40, 128), height=log(40, 128), shadow=rng.choice([0, log(64, 256)]))
    if kind == "views":
        return dict(kind=kind, shader=rng.choice(["gouraud_texture", "phong"]), n=log(2, 64),
                    lat=log(6, 60), tex=log(16, 512), width=log(48, 256), height=log(48, 256))
    return dict(kind=kind, shader=rng.choice(["phong", "phong_darboux"]), lat=log(6, 60),
                tex=log(16, 512), width=log(48, 512), height=log(48, 512))


# ---- inputs: plain arrays ---------------------------------------------------

def ball(n_lat, n_lon, radius=1.0, half=0.0, radial=None):
    """(vertices, normals, uvs, faces) of a sphere; half > 0 makes it a capsule."""
    th, ph = np.meshgrid(np.linspace(0.0, math.pi, n_lat + 1),
                         np.linspace(0.0, 2.0 * math.pi, n_lon + 1), indexing="ij")
    n = np.stack([np.sin(th) * np.cos(ph), np.sin(th) * np.sin(ph), np.cos(th)], -1)
    v = n * (radius if radial is None else radial[..., None])
    v[..., 2] += half * np.sign(np.round(n[..., 2], 9))
    uv = np.stack([ph / (2 * math.pi), 1.0 - th / math.pi], -1)
    i = np.arange(n.shape[0] * n.shape[1]).reshape(n.shape[:2])
    a, b, c, d = i[:-1, :-1], i[1:, :-1], i[1:, 1:], i[:-1, 1:]
    faces = np.concatenate([np.stack(t, -1).reshape(-1, 3) for t in ((a, b, c), (a, c, d))])
    return (v.reshape(-1, 3).astype(f32), n.reshape(-1, 3).astype(f32),
            uv.reshape(-1, 2).astype(f32), faces.astype(np.int32))


def box(hx, hy, hz, repeat=1.0):
    v, n, uv, faces = [], [], [], []
    for axis in range(3):
        for sign in (1.0, -1.0):
            q, r = np.zeros((3, 3))[:2]
            q[(axis + 1) % 3], r[(axis + 2) % 3] = 1.0, sign
            nrm = np.zeros(3)
            nrm[axis] = sign
            k = len(v)
            for s, t in ((-1, -1), (1, -1), (1, 1), (-1, 1)):
                v.append((nrm + s * q + t * r) * (hx, hy, hz))
                n.append(nrm)
                uv.append((repeat * (s + 1) / 2, repeat * (t + 1) / 2))
            faces += [(k, k + 1, k + 2), (k, k + 2, k + 3)]
    return (np.array(v, f32), np.array(n, f32), np.array(uv, f32), np.array(faces, np.int32))


def bumps(rng, lat, lon):
    """Radii of a smoothly dented sphere."""
    x = rng.normal(size=(lat + 1, lon + 1))
    for _ in range(4):
        x = (x + np.roll(x, 1, 1) + np.roll(x, -1, 1)) / 3.0
        x[1:-1] = (x[1:-1] + x[:-2] + x[2:]) / 3.0
    return 1.0 + 0.05 * x / max(x.std(), 1e-6)


def rotation(rng):
    q = rng.normal(size=4)
    w, x, y, z = q / np.linalg.norm(q)
    return np.array([[1 - 2 * (y * y + z * z), 2 * (x * y - w * z), 2 * (x * z + w * y)],
                     [2 * (x * y + w * z), 1 - 2 * (x * x + z * z), 2 * (y * z - w * x)],
                     [2 * (x * z - w * y), 2 * (y * z + w * x), 1 - 2 * (x * x + y * y)]])


def placed(mesh, tex, spec, at, turn=None):
    """One object: its mesh, its maps and its pose."""
    T = np.identity(4)
    T[:3, :3] = np.identity(3) if turn is None else turn
    T[:3, 3] = at
    return mesh + (tex.astype(f32), spec.astype(f32), T.astype(f32))


def some_pose(rng):
    return rng.uniform(-3.0, 3.0, 3), rotation(rng)


def objects_of(kind, rng, plan):
    """The objects of one scene: a floor and what stands, lies or walks over it.  `plan` picks
    what they are, so that only their sizes, colours and poses differ from seed to seed."""
    spec = np.full((8, 8), 2.0)

    def tex():
        return rng.random((8, 8, 3))

    if kind == "walker":  # 18 objects: a floor and 17 capsules of 192 triangles in a chain
        objs = [placed(box(10.0, 10.0, 0.05, 4.0), tex(), spec, (0.0, 0.0, -0.05))]
        skin, torso = tex(), np.array((0.0, 0.0, 0.75))
        objs.append(placed(ball(8, 12, 0.25), skin, spec, torso))
        for leg in range(4):
            a, at = rng.uniform(0.0, 0.6) + leg * math.pi / 2, torso.copy()
            for part in range(4):
                d = np.array((math.cos(a), math.sin(a), -0.35 * part + rng.uniform(-0.1, 0.1)))
                d /= np.linalg.norm(d)
                s = np.cross(d, (0.31, 0.17, 0.93))
                s /= np.linalg.norm(s)
                objs.append(placed(ball(8, 12, 0.08, 0.09), skin, spec, at + 0.12 * d,
                                   np.stack([s, np.cross(d, s), d], 1)))
                at = at + 0.22 * d
        return objs
    floor = (np.array([[-10, -10, 0], [10, -10, 0], [10, 10, 0], [-10, 10, 0]], f32),
             np.tile(np.array([[0, 0, 1]], f32), (4, 1)),
             np.array([[0, 0], [4, 0], [4, 4], [0, 4]], f32),
             np.array([[0, 1, 2], [0, 2, 3]], np.int32))
    objs = [placed(floor, tex(), spec, (0.0, 0.0, -3.5))]
    if kind == "coarse":
        for _ in range(int(plan.integers(4, 31))):
            k = int(plan.integers(0, 3))
            mesh = (box(*rng.uniform(0.2, 0.6, 3)) if k == 0 else
                    ball(8, 16, rng.uniform(0.1, 0.3), rng.uniform(0.2, 0.5)) if k == 1 else
                    ball(12, 24, rng.uniform(0.2, 0.6)))
            objs.append(placed(mesh, tex(), spec, *some_pose(rng)))
        return objs
    total, want = 2, math.exp(plan.uniform(math.log(1000), math.log(20000)))
    while total < want:
        k, lat = int(plan.integers(0, 3)), int(plan.choice([12, 16, 24, 32]))
        mesh = (box(*rng.uniform(0.2, 0.6, 3)) if k == 0 else
                ball(lat, 2 * lat, rng.uniform(0.15, 0.6), rng.uniform(0.2, 0.5) * (k == 1)))
        objs.append(placed(mesh, tex(), spec, *some_pose(rng)))
        total += len(mesh[3])
    return objs


def camera_of(eye, width, height, fov, target=(0.0, 0.0, 0.0)):
    """A camera's parameters; the angle of view is that of the shorter side."""
    t = math.tan(math.radians(fov) / 2) / min(width, height)
    return dict(eye=tuple(float(e) for e in eye), target=tuple(float(e) for e in target),
                width=width, height=height, hfov=math.degrees(2 * math.atan(t * width)),
                vfov=math.degrees(2 * math.atan(t * height)))


def ring(k, n, radius, z):
    a = 2.0 * math.pi * k / n
    return radius * math.cos(a), radius * math.sin(a), z


LIGHT = dict(direction=(0.57735, -0.57735, 0.57735), colour=(1.0, 1.0, 1.0),
             ambient=(0.8, 0.8, 0.8), diffuse=(0.8, 0.8, 0.8), specular=(0.6, 0.6, 0.6))


def pictures(case, seed):
    """([objects of each distinct scene], [(scene, camera, shadow centre) of each picture])."""
    rng, W, H = np.random.default_rng(seed), case["width"], case["height"]
    if case["kind"] == "frame":
        if case["mesh"] == "cube":
            mesh, t, eye = box(1.0, 1.0, 1.0), 2, (2.0, 4.0, 1.0 + 0.2 * rng.random())
        else:
            lat, t = case["lat"], case["tex"]
            mesh = ball(lat, 2 * lat, radial=bumps(rng, lat, 2 * lat))
            eye = ring(rng.random(), 1, 3.0, 0.5)
        obj = placed(mesh, rng.random((t, t, 3)), rng.uniform(1.0, 4.0, (t, t)), (0.0, 0.0, 0.0))
        return [[obj]], [(0, camera_of(eye, W, H, 60.0), (0.0, 0.0, 0.0))]
    kind = case.get("scenes", "walker")
    n, per = case.get("n", 1), case.get("cameras", 1)
    scenes = [objects_of(kind, rng, np.random.default_rng(k)) for k in range(-(-n // per))]
    out = []
    for k in range(n):
        if kind == "walker":
            centre = (0.0, 0.0, 0.75)
            eye = np.add(ring(rng.random(), 1, 2.5, 1.05), centre)
        else:
            centre, eye = (0.0, 0.0, 0.0), ring(k + rng.random(), n, 8.0, 4.0)
        out.append((k // per, camera_of(eye, W, H, 60.0, centre), centre))
    return scenes, out


def mesh_of(case, seed):
    """The mesh, map and cameras of the views and autograd kinds.  Their shaders take uvs in
    texels."""
    rng, t, lat = np.random.default_rng(seed), case["tex"], case["lat"]
    v, n, uv, faces = ball(lat, lat, radial=bumps(rng, lat, lat))
    nm = np.stack([rng.uniform(-0.3, 0.3, (t, t)), rng.uniform(-0.3, 0.3, (t, t)),
                   np.ones((t, t))], -1)
    m = case.get("n", 1)
    cams = [camera_of(ring(k + rng.random(), m, 3.0, 0.8), case["width"], case["height"], 45.0)
            for k in range(m)]
    return dict(verts=v, norms=n, uvs=(uv * f32(t)).astype(f32), faces=faces,
                tex=rng.random((t, t, 3)).astype(f32),
                normal_map=(nm / np.linalg.norm(nm, axis=-1, keepdims=True)).astype(f32),
                light=((0.3, -0.5, 0.8), (1.0, 1.0, 1.0)), cameras=cams)


def face_of_vertex(faces):
    """The first face that has the vertex as a corner."""
    first = np.zeros(int(faces.max()) + 1, np.int32)
    first[faces[::-1].reshape(-1)] = np.repeat(np.arange(len(faces))[::-1], 3)
    return first


def target_of(shape, seed):
    """The picture that a loss is taken against."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    return torch.rand(shape, generator=g, device="cuda")


# ---- the framework ----------------------------------------------------------

def camera_parameters(c):
    return CameraParameters(viewWidth=c["width"], viewHeight=c["height"], hfov=c["hfov"],
                            vfov=c["vfov"], position=c["eye"], target=c["target"])


def light_parameters():
    return LightParameters(**{k: np.array(v, f32) for k, v in LIGHT.items()})


def model_objects(objs):
    return [ModelObject(model=Model(verts=v, norms=n, uvs=uv, faces=f, faces_norm=f, faces_uv=f,
                                    diffuse_map=tex, specular_map=spec), transform=T)
            for v, n, uv, f, tex, spec, T in objs]


def renderer_of(case, scenes, shots):
    light = light_parameters()
    models = [merge_objects(model_objects(objs)) for objs in scenes]
    plan = [batch.BatchScene(model=models[s], light=light, shadow_centre=centre,
                             camera=Renderer.create_camera_from_parameters(camera_parameters(c)))
            for s, c, centre in shots]
    size = case.get("shadow", 0)
    calls = packing.plan_batch_device(plan, case["width"], case["height"],
                                      batch.ShadowMapSpec(width=size, height=size) if size
                                      else None)
    return renderer(calls, case, display=case["kind"] == "rollout")


def renderer(calls, case, **kw):
    """The launch shapes that the autotuner settles on for such sizes, named here so that
    every run has the same ones."""
    pixels = case["width"] * case["height"]
    if pixels < 30_000:
        br = batch.BatchRenderer(calls, tile=(8, 8), shadow_tile=(16, 16), persistent=False,
                                 shadow_on_demand="auto", **kw)
    else:
        br = batch.BatchRenderer(calls, tile=(16, 16), persistent=False, shadow_on_demand="auto",
                                 **kw)
        if pixels * case.get("n", 1) > 4_000_000:  # four pixels a lane
            br.autotune(candidates=[((16, 16), 1, 4)], reps=1, use_cache=False)
    br.calibrate()
    return br


def shader_of(case, m):
    light = LightSource(direction=np.array(m["light"][0], f32),
                        colour=np.array(m["light"][1], f32))
    both = dict(position=m["verts"], normal=m["norms"], uv=m["uvs"], light=light,
                texture=m["tex"])
    if case["shader"] == "gouraud_texture":
        return GouraudTextureShader, GouraudTextureExtraInput(**both)
    if case["shader"] == "phong":
        return PhongTextureShader, PhongTextureExtraInput(**both)
    return PhongTextureDarbouxShader, PhongTextureDarbouxExtraInput(
        **both, normal_map=m["normal_map"], id_to_face=face_of_vertex(m["faces"]),
        faces_indices=m["faces"])


def prepare(case, seed):
    kind = case["kind"]
    if kind == "image":
        scenes, shots = pictures(case, seed)
        s, c, centre = shots[0]
        return dict(kind=kind, args=(model_objects(scenes[s]), light_parameters(),
                                     camera_parameters(c), case["width"], case["height"]),
                    shadow=ShadowParameters(centre=np.array(centre, f32)))
    if kind == "autograd":
        m = mesh_of(case, seed)
        shader, extra = shader_of(case, m)
        leaves = {k: torch.from_numpy(np.array(getattr(extra, k))).cuda().requires_grad_()
                  for k in LEAVES[case["shader"]]}
        camera = Renderer.create_camera_from_parameters(camera_parameters(m["cameras"][0]))
        W, H = case["width"], case["height"]
        return dict(kind=kind, camera=camera, shader=shader, faces=m["faces"],
                    extra=extra._replace(**leaves), leaves=list(leaves.values()), width=W,
                    height=H, target=target_of((W, H, 3), seed))
    if kind == "views":
        m = mesh_of(case, seed)
        shader, extra = shader_of(case, m)
        cams = [Renderer.create_camera_from_parameters(camera_parameters(c))
                for c in m["cameras"]]
        call = build_views_call(cams, shader, m["faces"], extra, case["width"], case["height"],
                                init_buffers=True)
        br = renderer([call], case)
    else:
        scenes, shots = pictures(case, seed)
        br = renderer_of(case, scenes, shots)
    if kind in ("views", "train"):
        br.enable_backward()
        target = target_of(tuple(br.passes["main"].canvas.shape), seed)
        return dict(kind=kind, renderer=br, target=target, graph=br.capture_train(target))
    br.capture()
    if kind != "rollout":
        return dict(kind=kind, renderer=br)
    poser = ScenePoser([model_objects(objs) for objs in scenes])
    T = torch.from_numpy(np.stack(moved(scenes, seed))).cuda()
    return dict(kind=kind, renderer=br, poser=poser, poses=T)


LEAVES = {"phong": ("position", "normal", "texture"),
          "phong_darboux": ("position", "normal", "texture", "uv", "normal_map")}


def moved(scenes, seed):
    """The pose that each object has moved to."""
    rng, out = np.random.default_rng([seed, 1]), []
    for objs in scenes:
        for o in objs:
            T = o[6].copy()
            if len(o[0]) > 4:  # the floor stays
                T[:3, 3] += rng.uniform(-0.1, 0.1, 3).astype(f32)
            out.append(T)
    return out


def run(state):
    kind = state["kind"]
    if kind == "image":
        return Renderer.get_camera_image(*state["args"], shadow_param=state["shadow"])
    if kind == "autograd":
        _, canvas = render_differentiable(state["camera"], state["shader"], state["faces"],
                                          state["extra"], state["width"], state["height"])
        loss = ((canvas - state["target"]) ** 2).sum()
        return {"canvas": canvas.detach(), "grads": torch.autograd.grad(loss, state["leaves"])}
    br = state["renderer"]
    if kind in ("views", "train"):
        state["graph"].replay()
        main = br.passes["main"]
        return {"canvas": main.canvas, "zbuffer": main.zbuffer, **br.grads}
    if kind == "rollout":
        state["poser"].update(br, state["poses"])
    out = br.replay()
    return {k: out[k] for k in ("canvas", "zbuffer", "display") if k in out}


def work(case):
    """Bytes: positions, normals and uvs, three index triples a triangle, maps, and colour and
    depth of each pixel, once each (twice over for a step with gradients, whose outputs have
    its inputs' sizes).  Operations: 440 a triangle (its corners' transform, determinant,
    inverse), 110 in a shadow pass, 250 a covered pixel; three times that with gradients."""
    n, pixels = case.get("n", 1), case["width"] * case["height"] * case.get("n", 1)
    kind = case["kind"]
    if kind in ("views", "autograd"):
        tris, verts, texels = 2 * case["lat"] ** 2, (case["lat"] + 1) ** 2, case["tex"] ** 2
        ops = n * 440 * tris + 125 * pixels
    else:
        mesh = case.get("mesh")
        tris = (12 if mesh == "cube" else 4 * case["lat"] ** 2 if mesh else
                {"walker": 3276, "coarse": 4900, "dense": 7900}[case.get("scenes", "walker")])
        texels = (4 if mesh == "cube" else case["tex"] ** 2 if mesh else 64 * 18) * n
        tris, verts = tris * n, 0.6 * tris * n
        ops = 440 * tris + 110 * tris * bool(case.get("shadow", kind == "image")) + 165 * pixels
    back = kind in ("views", "train", "autograd")
    return {"bytes": (2 if back else 1) * (32 * verts + 16 * texels + 16 * pixels) + 36 * tris,
            "flops": (3 if back else 1) * ops}


# ---- the same in 64 bits ----------------------------------------------------

def t64(x):
    return torch.as_tensor(np.asarray(x), device="cuda").double()


def unit(v):
    return v / torch.linalg.vector_norm(v, dim=-1, keepdim=True)


def look_at(eye, centre, up=(0.0, 0.0, 1.0)):
    eye, centre, up = (np.asarray(a, np.float64) for a in (eye, centre, up))
    f = (centre - eye) / np.linalg.norm(centre - eye)
    s = np.cross(f, up / np.linalg.norm(up))
    s /= np.linalg.norm(s)
    V = np.identity(4)
    V[0, :3], V[1, :3], V[2, :3] = s, np.cross(s, f), -f
    V[:3, 3] = -V[:3, :3] @ eye
    return V


def viewport(width, height):
    m = np.identity(4)
    m[0, 0] = m[0, 3] = width / 2
    m[1, 1] = m[1, 3] = height / 2
    m[2, 2] = m[2, 3] = 0.5
    return m


def matrices(c):
    """(world to eye, world to clip, viewport) of a camera."""
    ty, tx = (math.tan(math.radians(c[k]) / 2) for k in ("vfov", "hfov"))
    near, far = 0.01, 1000.0
    P = np.zeros((4, 4))
    P[0, 0], P[1, 1], P[3, 2] = 1 / tx, 1 / ty, -1.0
    P[2, 2], P[2, 3] = (far + near) / (near - far), 2 * far * near / (near - far)
    V = look_at(c["eye"], c["target"])
    return V, P @ V, viewport(c["width"], c["height"])


def clip_of(verts, M):
    return verts @ M[:, :3].T + M[:, 3]


def inverse(A):
    """(inverses, determinants) of 3 x 3 matrices, from their rows' cross products."""
    r = A.unbind(-2)
    X = torch.stack([torch.linalg.cross(r[(k + 1) % 3], r[(k + 2) % 3]) for k in range(3)], -1)
    det = (r[0] * X[..., 0]).sum(-1)
    return X / det[..., None, None], det


class Seen:
    """The triangles of a scene that a camera may see, as edge functions."""

    def __init__(self, verts, faces, M, vp):
        c = clip_of(verts, M)[faces]
        A = c[..., [0, 1, 3]]
        X, det = inverse(A)
        self.ids = torch.nonzero(det > 1e-6)[:, 0]
        self.inv, self.z, self.vp = X[self.ids], c[self.ids][..., 2], vp
        # the first triangle is shown, whichever way it faces, where no other is
        self.first = (X[0], c[0, :, 2]) if det[0].abs() > 1e-6 else None
        # the span of each along x in pixels; without a bound where it crosses the eye's plane
        c, far = c[self.ids], torch.tensor(1e9, device="cuda", dtype=torch.float64)
        x = torch.where(c[..., 3] > 1e-6, c[..., 0] / c[..., 3] * vp[0, 0] + vp[0, 3], far)
        behind = (c[..., 3] <= 1e-6).any(-1)
        self.lo = torch.where(behind, -far, x.amin(-1) - 1)
        self.hi = torch.where(behind, far, x.amax(-1) + 1)

    def nearest(self, i, j, step):
        """(triangle or -1, depth) of the samples (i, j), i ascending."""
        xy1 = torch.stack([(i - self.vp[0, 3]) / self.vp[0, 0],
                           (j - self.vp[1, 3]) / self.vp[1, 1], torch.ones_like(i)], -1)
        who = torch.full(i.shape, -1, dtype=torch.int64, device="cuda")
        depth = torch.full(i.shape, math.inf, dtype=torch.float64, device="cuda")
        for a in range(0, len(i), step):
            b = min(a + step, len(i))
            k = torch.nonzero((self.hi >= i[a]) & (self.lo <= i[b - 1]))[:, 0]
            if not len(k):
                continue
            e = (xy1[a:b] @ self.inv[k].permute(1, 0, 2).reshape(3, -1)).view(b - a, -1, 3)
            z = (e * self.z[k]).sum(-1) * self.vp[2, 2] + self.vp[2, 3]
            z = torch.where((e >= 0).all(-1), z, math.inf)
            d, m = z.min(-1)
            depth[a:b], who[a:b] = d, torch.where(d < math.inf, self.ids[k[m]], -1)
        return who, depth


def world(objs):
    """One scene's arrays in world space: maps padded and stacked along their first axis, the
    normals of an object scaled by their common norm, before and after its pose."""
    side = max(o[4].shape[0] for o in objs)
    out = dict(verts=[], norms=[], uvs=[], faces=[], obj=[], tex=[], spec=[])
    base = 0
    for k, (v, n, uv, f, tex, spec, T) in enumerate(objs):
        v, n, T = np.float64(v), np.float64(n), np.float64(T)
        h = (n / np.linalg.norm(n)) @ np.linalg.inv(T)[:3, :3]
        out["verts"].append(v @ T[:3, :3].T + T[:3, 3])
        out["norms"].append(h / np.linalg.norm(h))
        out["uvs"].append(uv)
        out["faces"].append(f + base)
        out["obj"].append(np.full(len(f), k))
        out["tex"].append(np.pad(tex, ((0, side - len(tex)), (0, side - len(tex)), (0, 0))))
        out["spec"].append(np.pad(spec, ((0, side - len(spec)),) * 2))
        base += len(v)
    out = {k: np.concatenate(x) for k, x in out.items()}
    w = {k: t64(out[k]) for k in ("verts", "norms", "uvs", "tex", "spec")}
    w.update({k: torch.as_tensor(out[k], device="cuda").long() for k in ("faces", "obj")})
    w["shape"] = t64([o[4].shape[:2] for o in objs])
    w["side"] = side
    return w


def barycentric(verts, fc, i, j, p):
    """Weights, and depth, of the corners fc at the pixels (i, j)."""
    c = clip_of(verts[fc], p["w2c"])
    vp = p["vp"]
    xy1 = torch.stack([(i - vp[0, 3]) / vp[0, 0], (j - vp[1, 3]) / vp[1, 1],
                       torch.ones_like(i)], -1)
    e = (xy1[:, None, :] @ inverse(c[..., [0, 1, 3]])[0])[:, 0]
    return e / e.sum(-1, keepdim=True), (e * c[..., 2]).sum(-1) * vp[2, 2] + vp[2, 3]


def mixed(b, v):
    return (b[..., None] * v).sum(1)


def eye_normals(n, p):
    return unit(unit(n) @ p["eye"][:3, :3].T)


def wrapped(uv, tex):
    u = torch.floor(uv).long()
    return torch.remainder(u[:, 0], tex.shape[0]), torch.remainder(u[:, 1], tex.shape[1])


def reflection(w, leaf, p, t, i, j, seen):
    """Colour and depth of pixels that show the triangles t, with the light's shadow where
    `seen` is the light's view."""
    fc = w["faces"][t]
    b, z = barycentric(leaf["verts"], fc, i, j, p)
    n = unit(mixed(b, eye_normals(leaf["norms"][fc], p)))
    uv = mixed(b, w["uvs"][fc])
    fr = uv - torch.trunc(uv)
    fr = torch.where(fr < 0, fr + 1, fr)
    obj = w["obj"][t]
    at = fr * w["shape"][obj]
    u = (torch.floor(at[:, 0]).long() + obj * w["side"]).clamp(0, len(w["tex"]) - 1)
    v = torch.floor(at[:, 1]).long().clamp(0, w["side"] - 1)
    tex, power = leaf["tex"][u, v], leaf["spec"][u, v]
    l = unit(p["light_dir_eye"])
    d = (n * l).sum(-1, keepdim=True)
    r = unit(2 * d * n - l)
    k = p["diffuse"] * d.clamp(min=0) + \
        p["specular"] * (r[:, 2].clamp(min=0) ** power)[:, None]
    if seen is not None:
        s = mixed(b, clip_of(leaf["verts"][fc], seen["w2c"])).detach() @ seen["vp"].T
        ij = torch.sign(s[:, :2]) * torch.floor(s[:, :2].abs() + 0.5)
        ij = torch.where(ij < 0, ij + seen["size"], ij)
        inside = ((ij >= 0) & (ij < seen["size"])).all(-1)
        depth = torch.full_like(z, math.inf)
        if inside.any():
            depth[inside] = light_depth(seen, ij[inside])
        k = torch.where((s[:, 2] <= depth)[:, None], 1.0, 1.0 - p["strength"]) * k
    return p["ambient"] * tex + k * tex * p["light_colour"], z


def light_depth(seen, ij):
    """The shadow map's depth at the texels ij; each is looked for once."""
    height = seen["size"][1]
    flat, back = torch.unique(ij[:, 0] * height + ij[:, 1], return_inverse=True)
    i, j = torch.floor(flat / height), torch.remainder(flat, height)
    who, depth = seen["view"].nearest(i, j, 2048)
    if seen["view"].first is not None and (who < 0).any():
        vp = seen["vp"]
        e = torch.stack([(i - vp[0, 3]) / vp[0, 0], (j - vp[1, 3]) / vp[1, 1],
                         torch.ones_like(i)], -1) @ seen["view"].first[0]
        shown = (who < 0) & (e >= 0).all(-1)
        depth = torch.where(shown, e @ seen["view"].first[1] * vp[2, 2] + vp[2, 3], depth)
    return (depth + seen["offset"])[back]


D_SCENE = (("light_direction", 0, 3), ("light_colour", 3, 3), ("light_dir_eye", 6, 3),
           ("ambient", 9, 3), ("diffuse", 12, 3), ("specular", 15, 3), ("w2c", 18, 16),
           ("vp", 34, 16), ("eye", 50, 16), ("strength", 66, 3))


def camera_terms(c, light, strength=(0.6, 0.6, 0.6)):
    V, w2c, vp = matrices(c)
    p = {k: t64(v) for k, v in light.items()}
    p["light_direction"] = t64(f32(light["direction"]))
    p["light_dir_eye"] = t64(V[:3, :3] @ (np.float64(f32(light["direction"]))))
    p["light_dir_eye"] = unit(p["light_dir_eye"])
    p.update(w2c=t64(w2c), vp=t64(vp), eye=t64(np.linalg.inv(V).T), strength=t64(strength))
    return p


def light_terms(w, direction, centre, width, height, offset):
    """The light's orthographic view of the scene, two units wide, ten units away."""
    d = np.float64(f32(direction))
    V = look_at(np.float64(f32(centre)) + 10.0 * d, np.float64(f32(centre)))
    M, vp = t64(np.diag((1.0, 1.0, -1.0, 1.0)) @ V), t64(viewport(width, height))
    return dict(w2c=M, vp=vp, size=t64((width, height)), offset=float(f32(offset)),
                view=Seen(w["verts"], w["faces"], M, vp))


def shown(w, p, W, H):
    """The pixels that show a triangle: (triangle, i, j)."""
    i, j = (g.reshape(-1).double() for g in torch.meshgrid(
        torch.arange(W, device="cuda"), torch.arange(H, device="cuda"), indexing="ij"))
    t, _ = Seen(w["verts"], w["faces"], p["w2c"], p["vp"]).nearest(i, j, 16 * H)
    k = torch.nonzero(t >= 0)[:, 0]
    return t[k], i[k], j[k]


def exact_pictures(case, seed):
    kind, W, H = case["kind"], case["width"], case["height"]
    scenes, shots = pictures(case, seed)
    if kind == "rollout":
        T = iter(moved(scenes, seed))
        scenes = [[o[:6] + (next(T),) for o in objs] for objs in scenes]
    n, size = len(shots), case.get("shadow", 0)
    canvas = torch.ones((n, W, H, 3), dtype=torch.float64, device="cuda")
    zbuffer = torch.ones((n, W, H), dtype=torch.float64, device="cuda")
    target = target_of(canvas.shape, seed).double() if kind == "train" else None
    grads = dict(d_positions=[], d_normals=[], d_textures=[], d_specular_maps=[], d_scene=[])
    for s, (scene, c, centre) in enumerate(shots):
        if not s or scene != shots[s - 1][0]:
            w = world(scenes[scene])
        leaf = {k: w[k].clone().requires_grad_(target is not None)
                for k in ("verts", "norms", "tex", "spec")}
        p = camera_terms(c, dict(LIGHT, light_colour=LIGHT["colour"]))
        seen = light_terms(w, LIGHT["direction"], centre, size, size, 0.05) if size else None
        if kind == "image":
            p["strength"] = t64(1 - f32((0.4, 0.4, 0.4)))
            seen = light_terms(w, LIGHT["direction"], centre, W, H, 0.05)
        if target is not None:
            p = {k: v.requires_grad_() for k, v in p.items()}
        with torch.no_grad():
            t, i, j = shown(w, p, W, H)
        with torch.set_grad_enabled(target is not None):
            col, z = reflection(w, leaf, p, t, i, j, seen)
        at = (torch.full_like(t, s), i.long(), j.long())
        canvas[at], zbuffer[at] = col.detach(), z.detach()
        if target is not None:
            loss = ((col - target[at]) ** 2).sum()
            wrt = list(leaf.values()) + [p[k] for k, _, _ in D_SCENE]
            got = torch.autograd.grad(loss, wrt, allow_unused=True)
            got = [torch.zeros_like(x) if g is None else g for x, g in zip(wrt, got)]
            for key, g in zip(("d_positions", "d_normals", "d_textures", "d_specular_maps"), got):
                grads[key].append(g.reshape(-1))
            grads["d_scene"].append(scene_row(got[4:]))
    if kind == "image":
        return canvas[0]
    out = {"canvas": canvas, "zbuffer": zbuffer}
    if kind == "rollout":
        out["display"] = None  # whole numbers
    if target is not None:
        out.update({k: torch.cat(v) for k, v in grads.items()})
    return out


def scene_row(grads):
    row = torch.zeros(69, dtype=torch.float64, device="cuda")
    for (_, o, m), g in zip(D_SCENE, grads):
        row[o:o + m] = g.reshape(-1)
    return row


def lit(case, m, leaf, p, fc, i, j):
    """Colour and depth of pixels of the views and autograd kinds' shaders."""
    b, z = barycentric(leaf["position"], fc, i, j, p)
    uv = mixed(b, leaf["uv"][fc])
    u, v = wrapped(uv.detach(), leaf["texture"])
    tex, l = leaf["texture"][u, v], unit(p["light_direction"])
    if case["shader"] == "gouraud_texture":
        lam = (unit(leaf["normal"][fc]) * l).sum(-1, keepdim=True)
        return tex * mixed(b, p["light_colour"] * lam), z
    n = unit(mixed(b, eye_normals(leaf["normal"][fc], p)))
    if case["shader"] == "phong_darboux":
        own = m["own"][fc[:, 0]]  # corners of the face of the triangle's first vertex
        c = clip_of(leaf["position"][own], p["w2c"])
        q, st = c[..., :3] / c[..., 3:], leaf["uv"][own]
        A = inverse(torch.stack([q[:, 1] - q[:, 0], q[:, 2] - q[:, 0], n], 1))[0]
        d = torch.stack([st[:, 1] - st[:, 0], st[:, 2] - st[:, 0],
                         torch.zeros_like(st[:, 0])], 1)  # (edge, u or v)
        ij = A @ d
        nm = leaf["normal_map"][u, v]
        n = unit(unit(ij[..., 0]) * nm[:, :1] + unit(ij[..., 1]) * nm[:, 1:2] + n * nm[:, 2:])
    k = p["light_colour"] * (n * l).sum(-1, keepdim=True)
    return torch.where((k >= 0).all(-1, keepdim=True), tex * k, 0.0), z


def exact_mesh(case, seed):
    m, W, H, n = mesh_of(case, seed), case["width"], case["height"], case.get("n", 1)
    faces = torch.as_tensor(m["faces"], device="cuda").long()
    w = dict(verts=t64(m["verts"]), faces=faces)
    src = dict(position="verts", normal="norms", uv="uvs", texture="tex",
               normal_map="normal_map")
    leaf = {k: t64(m[v]).requires_grad_() for k, v in src.items()}
    m = dict(m, own=faces[torch.as_tensor(face_of_vertex(m["faces"]), device="cuda").long()])
    canvas = torch.ones((n, W, H, 3), dtype=torch.float64, device="cuda")
    zbuffer = torch.ones((n, W, H), dtype=torch.float64, device="cuda")
    shape = (W, H, 3) if case["kind"] == "autograd" else tuple(canvas.shape)
    target = target_of(shape, seed).double().view(canvas.shape)
    total, rows = None, []
    light = dict(direction=m["light"][0], light_colour=m["light"][1], ambient=(0,) * 3,
                 diffuse=(0,) * 3, specular=(0,) * 3)
    for s, c in enumerate(m["cameras"]):
        p = {k: v.requires_grad_() for k, v in camera_terms(c, light).items()}
        with torch.no_grad():
            t, i, j = shown(w, p, W, H)
        col, z = lit(case, m, leaf, p, faces[t], i, j)
        if case["shader"] == "gouraud_texture":  # a negative light is not drawn
            kept = (col >= 0).all(-1)
            t, i, j, col, z = t[kept], i[kept], j[kept], col[kept], z[kept]
        at = (torch.full_like(t, s), i.long(), j.long())
        canvas[at], zbuffer[at] = col.detach(), z.detach()
        wrt = list(leaf.values()) + [p[k] for k, _, _ in D_SCENE]
        got = torch.autograd.grad(((col - target[at]) ** 2).sum(), wrt, allow_unused=True)
        got = [torch.zeros_like(x) if g is None else g for x, g in zip(wrt, got)]
        rows.append(scene_row(got[len(leaf):]))
        got = got[:len(leaf)]
        total = got if total is None else [a + b for a, b in zip(total, got)]
    total = dict(zip(leaf, total))
    if case["kind"] == "autograd":
        return {"canvas": canvas[0], "grads": [total[k] for k in LEAVES[case["shader"]]]}
    return {"canvas": canvas, "zbuffer": zbuffer, "d_positions": total["position"],
            "d_normals": total["normal"], "d_textures": total["texture"],
            "d_scene": torch.stack(rows)}


def exact(case, seed):
    """Outputs in 64 bits; None for more pixels than take some ten seconds."""
    if case["kind"] in ("views", "autograd"):
        return exact_mesh(case, seed)
    if case["width"] * case["height"] * case.get("n", 1) > 20_000_000:
        return None
    return exact_pictures(case, seed)
