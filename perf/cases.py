"""Timed workloads of the renderer, each through the package's public entry
points: single frames from thumbnail to 1024^2 in every kind of storage,
transfer-function editing, volume loading, batched views and a served burst.

``listed()`` names the workloads, ``draw(rng)`` gives more of the same
ranges, ``prepare``/``run`` are one program's setup and one pass of its loop,
``work`` is what a pass cannot do without.  Volumes are the seeded
Gaussian-blob fields (and the double sphere) of the benchmark's
configurations, cameras lie around the box, opacity functions leave density 0
transparent.
"""

import math
import random

import numpy as np
import torch

from pyvr_amd.camera import Camera
from pyvr_amd.config import RenderConfig
from pyvr_amd.datasets import create_sample_volume
from pyvr_amd.datasets.synthetic import blob_params
from pyvr_amd.hip_renderer import VolumeRenderer
from pyvr_amd.hip_renderer.batch import BatchRenderer, DeviceBlobVolume
from pyvr_amd.hip_renderer.plain import PlainRenderer
from pyvr_amd.hip_renderer.serve import RenderServer, ServeRequest, estimated_samples
from pyvr_amd.lighting import Light
from pyvr_amd.transferfunctions import ColorTransferFunction, OpacityTransferFunction
from pyvr_amd.volume import Volume

# (scalar storage, normal storage or "none") pairs the library supports
FORMATS = [("f32", "f32x3"), ("f16", "f16x3"), ("f16", "sn8x3"), ("u8", "sn8x3"), ("f32", "sn8x3"),
           ("f16", "f32x3"), ("f32", "none"), ("f16", "none"), ("u8", "none")]


def _case(name, kind, shape, image, preset, formats, **more):
    c = dict(kind=kind, s0=shape[0], s1=shape[1], s2=shape[2], width=image[0], height=image[1], preset=preset,
             scalar=formats[0], normal=formats[1], field="blobs", blobs=8, points=6, tau=0.99, requests=1, volumes=1,
             brick_log2=3)
    c.update(more)
    if name is not None:
        c["name"] = name
    return c


def listed():
    return [
        # a preview thumbnail of a small volume: latency and launches
        _case("thumbnail", "frame", (64, 64, 64), (128, 128), "fast", ("f32", "f32x3")),
        # the plain configuration: double sphere as stored by default
        _case("double_sphere_512", "frame", (128, 128, 128), (512, 512), "balanced", ("f32", "f32x3"),
              field="double_sphere"),
        # the FP32 reference configuration at 1024^2
        _case("f32_256_1024", "frame", (256, 256, 256), (1024, 1024), "high_quality", ("f32", "f32x3"), tau=0.95),
        # an orbit over a large resident FP16 volume, one frame per launch
        _case("f16_512_1024", "plain", (512, 512, 512), (1024, 1024), "high_quality", ("f16", "f16x3"), blobs=32,
              tau=0.95),
        # compact storage, unequal axes, an image of odd size
        _case("u8_ragged", "frame", (96, 160, 224), (767, 433), "balanced", ("u8", "sn8x3")),
        # a scan without normals at the finest preset
        _case("scalar_ultra", "frame", (201, 150, 301), (640, 480), "ultra_quality", ("f32", "none")),
        # a transfer function being edited: a new LUT every frame
        _case("edit_transfer_function", "edit", (256, 256, 256), (800, 600), "balanced", ("f16", "sn8x3")),
        # a time series: every pass loads a volume with its normals and shows it
        _case("load_f32_normals", "load", (192, 192, 192), (512, 512), "balanced", ("f32", "f32x3")),
        # the same with the normals computed on the device, unequal odd axes
        _case("load_f16_device_normals", "load", (255, 193, 160), (512, 512), "balanced", ("f16", "f16x3"),
              normals="device"),
        # a generated volume comes up on first use, renders and leaves
        _case("generate_320", "generate", (320, 320, 320), (512, 512), "balanced", ("f16", "f16x3"), brick_log2=4),
        # 24 views of a large volume in one batch
        _case("batch_24_views", "batch", (512, 512, 512), (1024, 1024), "high_quality", ("f16", "f16x3"), blobs=32,
              tau=0.95, requests=24),
        # a burst of mixed requests to the server: its own volume, image size,
        # preset and LUT each
        _case("serve_burst", "serve", (256, 256, 256), (1024, 1024), "mixed", ("f16", "sn8x3"), requests=32, volumes=4),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["frame", "frame", "frame", "plain", "edit", "load", "generate", "batch", "serve"])
    top = {"load": 224, "generate": 320, "serve": 256, "edit": 288, "frame": 288}.get(kind, 448)
    edge = _log(rng, 40, top)
    shape = tuple(max(16, min(top, int(edge * rng.uniform(0.7, 1.3)))) for _ in range(3))
    side = _log(rng, 64, 640 if kind == "serve" else 1024)
    image = (side + rng.randrange(0, 33), max(48, int(side * rng.uniform(0.55, 1.0))))
    preset = "mixed" if kind == "serve" else rng.choice(["preview", "fast", "balanced", "balanced", "high_quality"])
    resident = kind in ("plain", "batch", "serve", "generate")
    formats = rng.choice([f for f in FORMATS if not (resident and f[1] == "none")])
    return _case(None, kind, shape, image, preset, formats, blobs=rng.choice([4, 8, 16]), points=rng.randrange(4, 9),
                 tau=rng.choice([0.99, 0.95]), requests=rng.randrange(4, 17) if kind in ("batch", "serve") else 1,
                 volumes=rng.randrange(1, 5) if kind == "serve" else 1,
                 normals="device" if kind == "load" and formats[1] != "none" and rng.random() < 0.5 else "host",
                 brick_log2=rng.choice([3, 3, 4]) if resident else 3)


# ---------------------------------------------------------------------------
# inputs

def _rng(seed, what):
    return random.Random("%d/%s" % (seed, what))


def _camera(rng):
    return Camera.from_spherical(target=np.zeros(3, np.float32), azimuth=rng.uniform(0.0, 2.0 * math.pi),
                                 elevation=rng.uniform(-math.pi / 3, math.pi / 3), roll=0.0,
                                 distance=rng.uniform(2.5, 4.0))


def _colors(rng):
    """A 256-entry colour map, one control point per entry, as a named
    colormap gives it."""
    anchors = np.array([[rng.random() for _ in range(3)] for _ in range(5)])
    x = np.linspace(0.0, 1.0, 256)
    rgb = np.stack([np.interp(x, np.linspace(0.0, 1.0, 5), anchors[:, k]) for k in range(3)], axis=-1)
    return ColorTransferFunction([(float(t), tuple(map(float, c))) for t, c in zip(x, rgb)])


def _opacity(case, rng):
    if case["field"] == "double_sphere":
        return OpacityTransferFunction.linear(0.0, 0.1)
    n = case["points"]
    xs = [0.0] + sorted(rng.uniform(0.0, 1.0) for _ in range(n - 2)) + [1.0]
    ys = [0.0] + [rng.uniform(0.0, 0.5) for _ in range(n - 1)]
    return OpacityTransferFunction(list(zip(xs, ys)))


def _light():
    return Light.directional(direction=[1, -1, 0], ambient=0.2, diffuse=0.8)


def _config(preset):
    return getattr(RenderConfig, preset)()


def _volume(case, seed):
    """Host volume: float32 field in [0, 1] and, unless the storage or the
    case says otherwise, its unit gradients."""
    shape = (case["s0"], case["s1"], case["s2"])
    if case["field"] == "double_sphere":
        data = torch.from_numpy(create_sample_volume(shape[0], "double_sphere")).cuda()
    else:
        _, centers, sigmas, amps = blob_params(case["blobs"], seed)
        axes = [torch.linspace(-1.0, 1.0, s, dtype=torch.float64, device="cuda") for s in shape]
        data = torch.zeros(shape, dtype=torch.float32, device="cuda")
        for c, s, a in zip(centers, sigmas, amps):
            f = [torch.exp(-((axes[k] - float(c[k])) ** 2) / (2.0 * float(s) ** 2)).float() for k in range(3)]
            data += float(a) * f[0][:, None, None] * (f[1][:, None] * f[2][None, :])
        g = torch.Generator(device="cuda").manual_seed(seed)
        data += (torch.rand(shape, generator=g, device="cuda") * 2.0 - 1.0) * 1e-3
        data.clamp_(0.0, 1.0)
    normals = None
    if case["normal"] != "none" and case.get("normals", "host") == "host":
        grad = torch.stack(torch.gradient(data), dim=-1)
        normals = (grad / (grad.norm(dim=-1, keepdim=True) + 1e-8)).cpu().numpy()
    one = np.ones(3, np.float32)
    return Volume(data=data.cpu().numpy(), normals=normals, min_bounds=-one, max_bounds=one)


def _blob_volume(case, seed, k=0):
    scale = (1.0, 0.75, 0.5, 0.375)[k]
    shape = tuple(max(16, int(case[s] * scale)) for s in ("s0", "s1", "s2"))
    return DeviceBlobVolume(shape=shape, n_blobs=case["blobs"], seed=4 * seed + k, noise=1e-3)


def prepare(case, seed):
    rng = _rng(seed, "scene")
    kind, w, h = case["kind"], case["width"], case["height"]
    state = dict(case=case, kind=kind)
    if kind in ("frame", "edit", "load"):
        r = VolumeRenderer(width=w, height=h, config=_config(case["preset"]), light=_light(),
                           scalar_format=case["scalar"],
                           normal_format="f32x3" if case["normal"] == "none" else case["normal"])
        volume = _volume(case, seed)
        r.load_volume(volume, device_normals=case.get("normals") == "device")
        r.set_opacity_threshold(case["tau"])
        ctf, otf = _colors(rng), _opacity(case, rng)
        r.set_transfer_functions(ctf, otf)
        camera = _camera(rng)
        r.set_camera(camera)
        state.update(renderer=r, volume=volume, camera=camera, ctf=ctf, otf=otf)
    elif kind == "plain":
        r = PlainRenderer(scalar_format=case["scalar"], normal_format=case["normal"], brick_log2=case["brick_log2"])
        volume, camera = _blob_volume(case, seed), _camera(rng)
        r.prepare(volume, camera, _colors(rng), _opacity(case, rng), w, h, _config(case["preset"]), _light(),
                  case["tau"])
        state.update(renderer=r, volume=volume, camera=camera)
    elif kind in ("batch", "generate"):
        r = BatchRenderer(scalar_format=case["scalar"], normal_format=case["normal"], brick_log2=case["brick_log2"])
        volume = _blob_volume(case, seed)
        if kind == "batch":
            r.upload(volume)
        state.update(renderer=r, volume=volume, cameras=[_camera(rng) for _ in range(case["requests"])],
                     ctf=_colors(rng), otf=_opacity(case, rng), config=_config(case["preset"]), light=_light())
    elif kind == "serve":
        r = RenderServer(scalar_format=case["scalar"], normal_format=case["normal"], brick_log2=case["brick_log2"],
                         memory_budget=16 << 30, max_batch_requests=64, max_batch_pixels=1 << 23)
        for k in range(case["volumes"]):
            r.register(k, _blob_volume(case, seed, k))
        r.preload()
        asks, sizes = [], random.Random(case["requests"])   # the image sizes belong to the case, not to the seed
        for _ in range(case["requests"]):
            s = sizes.uniform(0.5, 1.25)
            asks.append(dict(volume=rng.randrange(case["volumes"]), camera=_camera(rng), ctf=_colors(rng),
                             otf=_opacity(case, rng), width=max(16, int(w * s) // 16 * 16),
                             height=max(16, int(h * s) // 16 * 16),
                             config=_config(rng.choice(["fast", "balanced", "high_quality"])), light=_light(),
                             tau=case["tau"]))
        state.update(server=r, asks=asks)
    else:
        raise ValueError("unknown kind %r" % kind)
    return state


def _pixels(rgba):
    return np.frombuffer(rgba, np.uint8)


class _PinnedPixels(np.ndarray):
    """Pixels in a batch's own pinned memory, which lives as long as the
    renderer: the array keeps it."""


def _pinned(view, renderer):
    a = view.view(_PinnedPixels)
    a.renderer = renderer
    return a


def run(state):
    """One pass: the RGBA8 images, bottom row first."""
    kind, case = state["kind"], state["case"]
    if kind == "frame":
        r = state["renderer"]
        r.set_camera(state["camera"])
        return _pixels(r.render())
    if kind == "edit":
        r = state["renderer"]
        r.set_transfer_functions(state["ctf"], state["otf"])
        return _pixels(r.render())
    if kind == "load":
        r = state["renderer"]
        r.load_volume(state["volume"], device_normals=case.get("normals") == "device")
        return _pixels(r.render())
    if kind == "plain":
        r = state["renderer"]
        r.set_camera(state["camera"])
        return _pixels(r.read())
    if kind == "serve":
        server = state["server"]
        reqs = [server.submit(ServeRequest(**a, tag=k)) for k, a in enumerate(state["asks"])]
        server.drain()
        return [q.rgba for q in reqs]
    # a batch: the volume resident, or generated for this pass alone
    r = state["renderer"]
    r.clear()
    if kind == "generate":
        r.upload(state["volume"])
    for camera in state["cameras"]:
        r.add(state["volume"], camera, state["ctf"], state["otf"], case["width"], case["height"], state["config"],
              state["light"], case["tau"])
    slot = r.submit()
    r.wait(slot)
    images = [_pinned(r.view(k, slot), r) for k in range(len(state["cameras"]))]
    if kind == "generate":
        r.release(state["volume"])
    return images


# ---------------------------------------------------------------------------
# the work a pass cannot do without

_SCALAR_BYTES = {"f32": 4, "f16": 2, "u8": 1}
_NORMAL_BYTES = {"f32x3": 12, "f16x3": 6, "sn8x3": 3, "none": 0}


def work(case):
    """Bytes: every stored voxel read once and every pixel written once; a
    pass that loads also reads the float32 input and writes the stored
    voxels.  Operations: half of the rays' samples (the others lie in
    transparent space or behind the termination alpha) at 100 operations
    each: eight trilinear weights and taps per channel, lookup, light,
    composite."""
    n = case["requests"]
    voxels = case["s0"] * case["s1"] * case["s2"]
    stored = voxels * (_SCALAR_BYTES[case["scalar"]] + _NORMAL_BYTES[case["normal"]])
    pixels = case["width"] * case["height"]
    config = _config("balanced" if case["preset"] == "mixed" else case["preset"])
    camera = _camera(_rng(0, "scene"))
    samples = n * estimated_samples(case["width"], case["height"], camera, config)
    nbytes, flops = stored + 4 * n * pixels, 50.0 * samples
    if case["kind"] == "load":
        host_normals = case["normal"] != "none" and case.get("normals", "host") == "host"
        nbytes += voxels * (16 if host_normals else 4) + stored
        flops += 20.0 * voxels
    elif case["kind"] == "generate":
        nbytes += stored
        flops += voxels * (5.0 * case["blobs"] + 20.0)
    return {"bytes": float(nbytes), "flops": float(flops)}


def exact(case, seed):
    """Every output is a stored RGBA8 byte: compared for equality, so no
    64-bit value stands beside it."""
    return None
