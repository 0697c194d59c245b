"""The work that users of this framework have it do, as measurable cases.

Twelve listed cases: queries of the encodings and of both fields at arrays of
points, the reference network's weight gradients, one training step of each
kind, and renders from a thumbnail to several full views.  Sizes are those of
the repository's benchmark and tests, or generic.  draw() gives further cases
of the same kinds over the same ranges.

The library is called through nerf_amd on device memory that torch allocated;
torch (imported first) and libnerf.so then share one HIP runtime, and the
library's null stream is torch's default stream.
"""
import ctypes as C
import math

import numpy as np
import torch

from nerf_amd import _lib as L, ext

DEV = "cuda"
FIELD_FLOPS = 2 * (32 * 64 + 64 * 16) + 2 * (31 * 64 + 64 * 64 + 64 * 3)
REF_FLOPS = 2 * (64 * 128 + 4 * 128 * 128 + 128 * 16) + 2 * (48 * 128 + 2 * 128 * 128 + 128 * 16)
REF_BACKWARD_FLOPS = 2 * REF_FLOPS + 2 * (16 * 128 + 4 * 128 * 128) + 2 * (16 * 128 + 2 * 128 * 128) + 2 * 15 * 128
BOX = (0.0, 0.0, 0.0, 1.0, 1.0, 1.0)
CENTRE = (0.5, 0.5, 0.5)
RADIUS = 1.32  # the Blender orbit of radius 4 in the frame scaled by 0.33
T_STOP = 1e-4


def listed():
    return [
        # Hash encoding alone on an fp32 table, the smallest call of the benchmark: a
        # host program that runs its own network on the features.
        {"name": "encode_64k", "kind": "encode", "n": 65536, "log2_t": 16, "f32": True},
        # Density and colour at scattered points with directions: baking, mesh
        # extraction or a host's own sampler asking the field.  A ragged count.
        {"name": "field_query", "kind": "field", "n": 300007, "log2_t": 19},
        # Both MLPs on features that a host encoded itself.
        {"name": "field_mlp_4m", "kind": "mlp", "n": 1 << 22},
        # The reference's own network at a ragged number of world points.
        {"name": "ref_field_1m", "kind": "ref_field", "n": 1000003},
        # Its weight gradients for a training batch a host sampled itself.
        {"name": "ref_grad_256k", "kind": "ref_grad", "n": 1 << 18},
        # One training step as the benchmark trains: 2^18-sample batches of long rays.
        {"name": "train_dense", "kind": "train", "ref": False, "width": 800, "height": 800, "rays": 320, "target": 1 << 18, "cap": 1 << 18, "steps": 1024, "log2_t": 19, "interval": 16, "warmup": 16, "cells": 128**3},
        # One step of the reference host program's schedule: 4,096 rays of at most
        # 64 steps, a slice of the occupancy grid refreshed every step.
        {"name": "train_host", "kind": "train", "ref": False, "width": 800, "height": 800, "rays": 4096, "target": 0, "cap": 4096 * 64, "steps": 64, "log2_t": 19, "interval": 1, "warmup": 32, "cells": 65536},
        # The reference's own network trained on 2^18-sample batches.
        {"name": "train_ref", "kind": "train", "ref": True, "width": 800, "height": 800, "rays": 320, "target": 1 << 18, "cap": 1 << 18, "steps": 1024, "log2_t": 19, "interval": 16, "warmup": 16, "cells": 128**3},
        # A thumbnail of an opaque scene while a user turns the camera: launches and
        # latency count.
        {"name": "render_thumb", "kind": "render", "width": 100, "height": 75, "views": 1, "steps": 256, "log2_t": 19, "finest": 0, "res": 128, "cascades": 1, "gaussians": 32, "opaque": True},
        # The headline image: 800x800, thin media, up to 1,024 steps per ray.
        {"name": "render_800", "kind": "render", "width": 800, "height": 800, "views": 1, "steps": 1024, "log2_t": 19, "finest": 0, "res": 128, "cascades": 1, "gaussians": 32, "opaque": False},
        # Views of an unbounded scene in one call: nested cascades, long rays that end
        # early.  The largest case.
        {"name": "render_views", "kind": "render", "width": 1280, "height": 720, "views": 3, "steps": 4096, "log2_t": 21, "finest": 0, "res": 128, "cascades": 5, "gaussians": 512, "opaque": False},
        # The reference host's inference through its own interface: 64 uniform samples
        # per ray of the reference's network, the image returned to host memory.
        {"name": "host_image", "kind": "image", "width": 800, "height": 800, "spp": 64, "ref": True},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["encode", "field", "mlp", "ref_field", "ref_grad", "train", "train_host", "train_ref", "render", "render", "render_cascades", "image"])
    if kind == "encode":
        f32 = rng.random() < 0.5
        return {"kind": kind, "n": _log(rng, 4096, 1 << 22), "log2_t": rng.randint(14, 17 if f32 else 19), "f32": f32}
    if kind == "field":
        return {"kind": kind, "n": _log(rng, 4096, 1 << 21), "log2_t": rng.randint(15, 21)}
    if kind == "mlp":
        return {"kind": kind, "n": _log(rng, 4096, 1 << 22)}
    if kind == "ref_field":
        return {"kind": kind, "n": _log(rng, 4096, 1 << 21)}
    if kind == "ref_grad":
        return {"kind": kind, "n": _log(rng, 4096, 1 << 18)}
    if kind == "train_host":
        rays, steps = _log(rng, 512, 8192), rng.randint(24, 64)
        return {"kind": "train", "ref": False, "width": rng.randint(300, 800), "height": rng.randint(300, 800), "rays": rays, "target": 0, "cap": rays * steps, "steps": steps, "log2_t": rng.randint(17, 19), "interval": 1,
                "warmup": 32, "cells": 65536}
    if kind in ("train", "train_ref"):
        batch, steps = _log(rng, 1 << 14, 1 << 18), rng.randint(256, 1024)
        return {"kind": "train", "ref": kind == "train_ref", "width": rng.randint(300, 800), "height": rng.randint(300, 800), "rays": max(64, batch // 800), "target": batch, "cap": batch, "steps": steps, "log2_t": rng.randint(16, 20),
                "interval": 16, "warmup": 16, "cells": 128**3}
    if kind == "render":
        w = _log(rng, 64, 800)
        return {"kind": kind, "width": w, "height": max(32, int(w * rng.uniform(0.5, 1.0))), "views": 1, "steps": rng.randint(128, 1024), "log2_t": rng.randint(17, 20), "finest": 0, "res": rng.choice([64, 100, 128]), "cascades": 1,
                "gaussians": 32, "opaque": rng.random() < 0.5}
    if kind == "render_cascades":
        w = _log(rng, 160, 1280)
        return {"kind": "render", "width": w, "height": max(90, w * 9 // 16), "views": rng.randint(1, 3), "steps": rng.randint(1024, 4096), "log2_t": rng.randint(18, 21), "finest": rng.choice([0, 4096]), "res": 128,
                "cascades": rng.randint(1, 5), "gaussians": 256, "opaque": rng.random() < 0.3}
    w = _log(rng, 96, 800)
    return {"kind": kind, "width": w, "height": max(64, int(w * rng.uniform(0.5, 1.0))), "spp": rng.randint(16, 64), "ref": rng.random() < 0.6}


# ----------------------------------------------------------------- inputs
class Resident:
    """A torch tensor where nerf_amd takes a device array."""

    def __init__(self, t):
        self.t = t
        self.ptr = t.data_ptr()
        self.dtype = np.dtype({torch.float32: np.float32, torch.float16: np.float16, torch.int32: np.int32, torch.uint8: np.uint8}[t.dtype])


class _Memory:
    """Device memory of the library, for torch to view."""

    def __init__(self, ptr, shape, typestr, owner):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": shape, "typestr": typestr, "data": (int(ptr), False), "version": 2}


def _view(ptr, n, owner):
    return torch.as_tensor(_Memory(ptr, (int(n),), "<f4", owner), device=DEV)


def _gen(seed, salt=0):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed * 1000003 + salt)
    return g


def _uniform(shape, lo, hi, seed, salt):
    return torch.rand(shape, generator=_gen(seed, salt), device=DEV) * (hi - lo) + lo


def _directions(n, seed, salt):
    d = torch.randn((n, 3), generator=_gen(seed, salt), device=DEV)
    return (d / d.norm(dim=1, keepdim=True)).contiguous()


def _grid(case):
    return ext.grid_desc(case["log2_t"], L.NERF_EXT_F32 if case.get("f32") else L.NERF_EXT_F16, finest=case.get("finest", 0))


def _table(case, value_range, seed):
    t = _uniform((16 << case["log2_t"], 2), -value_range, value_range, seed, 1)
    return t if case.get("f32") else t.half()


def _weights(seed, shapes, salt):
    """fp16 matrices of Xavier-uniform weights, one after the other."""
    return torch.cat([_uniform((o * i,), -math.sqrt(6.0 / (o + i)), math.sqrt(6.0 / (o + i)), seed, salt + k) for k, (o, i) in enumerate(shapes)]).half()


DENSITY, COLOR = [(64, 32), (16, 64)], [(64, 32), (64, 64), (16, 64)]
REF_DENSITY, REF_COLOR = [(128, 64)] + [(128, 128)] * 4 + [(16, 128)], [(128, 48)] + [(128, 128)] * 2 + [(16, 128)]


def _field_weights(case, seed):
    wd, wc = _weights(seed, DENSITY, 20), _weights(seed, COLOR, 40)
    if case.get("opaque"):
        wd[2048 : 2048 + 64] = 0.5  # raw density = half the hidden activations' sum
    return wd, wc


def _scene(case, seed):
    """Isotropic Gaussians (centre, sigma, amplitude) as the benchmark's scenes
    draw them: in the unit box, or over radius 16 for nested cascades."""
    r = np.random.default_rng([seed, 7])
    n, wide = case["gaussians"], case["cascades"] > 1
    centre = r.uniform(-16.0, 16.0, (n, 3)) if wide else r.uniform(0.2, 0.8, (n, 3))
    sigma = r.uniform(0.3, 1.5, n) if wide else r.uniform(0.02, 0.1, n)
    return centre, sigma, r.uniform(5.0, 50.0, n)


def _render_box(case):
    return (-1.0, -1.0, -1.0, 1.0, 1.0, 1.0) if case["cascades"] > 1 else BOX


def _occupancy(case, seed):
    """Occupancy bits (density > 0.01 at cell centres, one grid per cascade,
    and a background shell where there are cascades), 32 cells a word."""
    centre, sigma, amplitude = _scene(case, seed)
    res, box, words = case["res"], _render_box(case), []
    for c in range(case["cascades"]):
        half = 0.5 * (box[3] - box[0]) * 2.0**c
        mid = 0.5 * (box[3] + box[0])
        x = (torch.arange(res, device=DEV, dtype=torch.float32) + 0.5) / res * (2 * half) + (mid - half)
        density = torch.zeros((res, res, res), device=DEV)  # z, y, x
        for k in range(len(sigma)):
            e = [torch.exp(-((x - float(centre[k, a])) ** 2) / (2 * float(sigma[k]) ** 2)) for a in range(3)]
            density += float(amplitude[k]) * e[2][:, None, None] * e[1][None, :, None] * e[0][None, None, :]
        on = density > 0.01
        if case["cascades"] > 1:
            r2 = (x**2)[:, None, None] + (x**2)[None, :, None] + (x**2)[None, None, :]
            on |= (r2 >= 144.0) & (r2 <= 240.25)
        bits = torch.zeros(((res**3 + 31) // 32, 32), dtype=torch.int64, device=DEV)
        bits.view(-1)[: res**3] = on.reshape(-1).long()
        word = (bits << torch.arange(32, device=DEV)).sum(1)
        words.append(torch.where(word >= 1 << 31, word - (1 << 32), word).int())
    return torch.cat(words).contiguous()


def _camera(seed, index, width, height, centre=CENTRE, radius=RADIUS):
    """A camera on a sphere about the scene, looking at its centre."""
    r = np.random.default_rng([seed, 11, index])
    back = r.normal(size=3)
    back[1] *= 0.6
    back /= np.linalg.norm(back)
    right = np.cross([0.0, 1.0, 0.0], back)
    right /= np.linalg.norm(right)
    up = np.cross(back, right)
    c2w = np.stack([right, up, back, np.asarray(centre) + radius * back], axis=1).astype(np.float32)
    f = 1111.0 * width / 800.0
    return L.NerfExtCamera((C.c_float * 12)(*c2w.ravel().tolist()), f, f, 0.5 * (width - 1.0), 0.5 * (height - 1.0), width, height)


def _cameras(case, seed):
    wide = case.get("cascades", 1) > 1
    return [_camera(seed, i, case["width"], case["height"], (0.0, 0.0, 0.0) if wide else CENTRE, 4.0 if wide else RADIUS) for i in range(case.get("views", 1))]


VIEWS = 8  # training images


def _images(case, seed):
    """Smooth coloured RGBA8 views with transparent borders."""
    w, h = case["width"], case["height"]
    low = torch.rand((VIEWS, 4, 12, 12), generator=_gen(seed, 3), device=DEV)
    low[:, 3] = (low[:, 3] * 3.0 - 0.5).clamp(0, 1)
    img = torch.nn.functional.interpolate(low, size=(h, w), mode="bilinear", align_corners=True)
    return (img.permute(0, 2, 3, 1) * 255.0).round().to(torch.uint8).cpu().numpy()


class Model:
    """What nerf_amd's renderer takes as a model, on torch's memory."""

    def __init__(self, case, seed):
        self.grid = _grid(case)
        self.table = _table(case, 0.5, seed)
        self.wd, self.wc = _field_weights(case, seed)

    def struct(self):
        return L.NerfExtModel(self.grid, self.table.data_ptr(), self.wd.data_ptr(), self.wc.data_ptr())


class Context:
    """A context of the reference's own interface."""

    def __init__(self, case, seed):
        w, h = case["width"], case["height"]
        cams = [_camera(seed, i, w, h) for i in range(VIEWS)]
        images = np.zeros((VIEWS, h, w), np.uint32)
        mats = np.zeros((VIEWS, 4, 4), np.float32)
        for i, c in enumerate(cams):
            mats[i, :3] = np.array(c.c2w[:], np.float32).reshape(3, 4)
            mats[i, 3, 3] = 1.0
        d = L.NerfCreateDesc(128, 1 << 20, 1 << 16, 256, images.ctypes.data, images.nbytes, mats.ctypes.data, mats.nbytes, VIEWS, w, h, cams[0].fx, cams[0].fy, cams[0].cx, cams[0].cy)
        self.h = C.c_void_p()
        L.call("nerf_create_context", C.byref(d), C.byref(self.h))
        kind = L.NERF_EXT_MODEL_REFERENCE if case["ref"] else L.NERF_EXT_MODEL_HASHGRID
        L.call("nerf_ext_context_configure", self.h, C.byref(L.NerfExtContextOptions(kind, L.NERF_EXT_SAMPLING_UNIFORM)))
        self.image = np.zeros((h, w), np.uint32)
        self.request = L.NerfInferenceRequest(seed % VIEWS, case["spp"], L.NERF_MEMORY_HOST, self.image.ctypes.data, self.image.nbytes)
        self.info = L.NerfInferenceInfo()

    def __del__(self):
        if self.h.value:
            L.call("nerf_destroy_context", self.h)
            self.h = C.c_void_p()


def _hyper(case):
    dense = case["target"] != 0
    if case["ref"] or not dense:  # the reference host's optimiser settings
        return dict(lr=5e-4, beta1=0.9, beta2=0.999, eps=1e-8, clip=1.0, guard=100.0, loss_scale=128.0, lr_decay_ksteps=250)
    return dict(lr=1e-2, beta1=0.9, beta2=0.99, eps=1e-8, clip=1e30, guard=1e30, loss_scale=128.0, lr_decay_ksteps=0)


def _points_case(case, seed):
    n, k = case["n"], case["kind"]
    s = {"n": n}
    if k in ("encode", "field"):
        s["pos"] = Resident(_uniform((n, 3), 0.0, 1.0, seed, 5))
        s["grid"] = _grid(case)
        s["table"] = Resident(_table(case, 0.5, seed))
    if k == "encode":
        s["out"] = Resident(torch.empty((n, 32), device=DEV, dtype=torch.float32 if case["f32"] else torch.float16))
        return s
    s["out"] = torch.empty((n, 4), device=DEV)
    s["dirs"] = _directions(n, seed, 6)
    if k in ("field", "mlp"):
        s["wd"], s["wc"] = _field_weights(case, seed)
        if k == "field":
            s["model"] = L.NerfExtModel(s["grid"], s["table"].ptr, s["wd"].data_ptr(), s["wc"].data_ptr())
        else:
            s["features"] = _uniform((n, 32), -0.5, 0.5, seed, 8).half()
        return s
    s["wd"], s["wc"] = _weights(seed, REF_DENSITY, 60), _weights(seed, REF_COLOR, 80)
    s["pos"] = _uniform((n, 3), 0.0, 1.0, seed, 5)
    if k == "ref_grad":
        s["draw"] = torch.randn((n, 4), generator=_gen(seed, 9), device=DEV) * 1e-2
        s["gd"], s["gc"] = torch.empty(L.NERF_EXT_REF_DENSITY_PARAMS, device=DEV), torch.empty(L.NERF_EXT_REF_COLOR_PARAMS, device=DEV)
    return s


def prepare(case, seed):
    kind = case["kind"]
    if kind == "train":
        img = _images(case, seed)
        cams = [_camera(seed, i, case["width"], case["height"]) for i in range(VIEWS)]
        occ = ext.occupancy_params(decay=0.95, threshold=0.01, cells_per_update=case["cells"], update_interval=case["interval"], warmup_steps=case["warmup"])
        t = ext.Trainer(ext.grid_desc(case["log2_t"], L.NERF_EXT_F16), img, cams, occupancy_res=128, hyper=ext.hyper_params(**_hyper(case)), occupancy=occ, initial_rays=case["rays"],
                        max_rays=max(case["rays"], case["target"]), target_samples=case["target"], sample_capacity=case["cap"], max_steps_per_ray=case["steps"], seed=seed % (1 << 31), table_init_range=0.1,
                        model_kind=L.NERF_EXT_MODEL_REFERENCE if case["ref"] else L.NERF_EXT_MODEL_HASHGRID)
        b = t.buffers()
        n_mlp = L.NERF_EXT_REF_DENSITY_PARAMS + L.NERF_EXT_REF_COLOR_PARAMS if case["ref"] else L.NERF_EXT_DENSITY_PARAMS + L.NERF_EXT_COLOR_PARAMS
        out = {"mlp_grad": _view(b.mlp_grad, n_mlp, t), "mlp": _view(b.mlp_f32, n_mlp, t)}
        if not case["ref"]:
            out["table_grad"], out["table"] = _view(b.table_grad, b.table_elems, t), _view(b.table_f32, b.table_elems, t)
        return {"kind": kind, "trainer": t, "out": out}
    if kind == "render":
        w, h, v = case["width"], case["height"], case["views"]
        bits = Resident(_occupancy(case, seed))
        box = _render_box(case)
        return {"kind": kind, "renderer": ext.Renderer(), "model": Model(case, seed), "bits": bits, "occ": ext.occupancy_struct(bits, case["res"], box[:3], box[3:], case["cascades"]), "cams": _cameras(case, seed),
                "steps": case["steps"], "rgba": Resident(torch.empty((v, h, w, 4), dtype=torch.uint8, device=DEV)), "rgb": Resident(torch.empty((v, h, w, 3), device=DEV)),
                "counts": Resident(torch.empty((v, h, w), dtype=torch.int32, device=DEV))}
    if kind == "image":
        return {"kind": kind, "context": Context(case, seed)}
    return {"kind": kind, **_points_case(case, seed)}


def run(s):
    kind = s["kind"]
    if kind == "encode":
        ext.encode_forward(s["grid"], s["table"], s["pos"], s["n"], s["out"])
        return s["out"].t
    if kind == "field":
        L.call("nerf_ext_field_forward", C.byref(s["model"]), s["pos"].ptr, s["dirs"].data_ptr(), s["n"], s["out"].data_ptr(), None)
        return s["out"]
    if kind == "mlp":
        L.call("nerf_ext_field_mlp", s["wd"].data_ptr(), s["wc"].data_ptr(), s["features"].data_ptr(), s["dirs"].data_ptr(), s["n"], s["out"].data_ptr(), None)
        return s["out"]
    if kind == "ref_field":
        L.call("nerf_ext_ref_field_forward", s["wd"].data_ptr(), s["wc"].data_ptr(), s["pos"].data_ptr(), s["dirs"].data_ptr(), s["n"], s["out"].data_ptr(), None, None)
        return s["out"]
    if kind == "ref_grad":
        L.call("nerf_ext_ref_backward", s["wd"].data_ptr(), s["wc"].data_ptr(), s["pos"].data_ptr(), s["dirs"].data_ptr(), s["draw"].data_ptr(), s["n"], 128.0, s["gd"].data_ptr(), s["gc"].data_ptr(), None)
        return {"density": s["gd"], "color": s["gc"]}
    if kind == "train":
        s["trainer"].step()
        return s["out"]
    if kind == "render":
        s["renderer"].render(s["model"], s["occ"], s["cams"], s["steps"], T_STOP, rgba8=s["rgba"], rgb=s["rgb"], counts=s["counts"])
        return {"rgba8": s["rgba"].t, "rgb": s["rgb"].t, "counts": s["counts"].t}
    c = s["context"]
    L.call("nerf_inference", c.h, C.byref(c.request), C.byref(c.info))
    return c.image.view(np.uint8)


def _samples(case):
    """About how many samples a pass evaluates."""
    k = case["kind"]
    if k == "train":
        return case["target"] or case["rays"] * case["steps"] * 0.9
    if k == "render":  # about a third of the marched steps lie in occupied cells and in front of the stop
        return case["width"] * case["height"] * case["views"] * case["steps"] * (0.1 if case["opaque"] else 0.4)
    if k == "image":
        return case["width"] * case["height"] * case["spp"]
    return case["n"]


def work(case):
    k, n = case["kind"], _samples(case)
    if k in ("ref_field", "ref_grad") or case.get("ref"):
        weights = 2 * (L.NERF_EXT_REF_DENSITY_PARAMS + L.NERF_EXT_REF_COLOR_PARAMS)
        if k == "ref_field":
            return {"bytes": weights + n * (12 + 12 + 16), "flops": n * REF_FLOPS}
        if k == "ref_grad":
            return {"bytes": 3 * weights + n * (12 + 12 + 16), "flops": n * REF_BACKWARD_FLOPS}
        if k == "image":
            return {"bytes": weights + case["width"] * case["height"] * 4, "flops": n * REF_FLOPS}
        return {"bytes": 15 * weights + n * 32, "flops": n * (REF_FLOPS + REF_BACKWARD_FLOPS)}
    table = (32 << case["log2_t"]) * (4 if case.get("f32") else 2) if "log2_t" in case else 32 << 20
    if k == "encode":
        size = 4 if case["f32"] else 2
        return {"bytes": min(table, n * 256 * size) + n * (12 + 32 * size), "flops": n * 16 * 8 * 4}
    if k == "mlp":
        return {"bytes": n * (64 + 12 + 16), "flops": n * FIELD_FLOPS}
    if k == "field":
        return {"bytes": min(table, n * 512) + n * (24 + 16), "flops": n * (FIELD_FLOPS + 512)}
    if k == "train":  # every parameter's master and two moments, read and written, its gradient and its fp16 copy written
        return {"bytes": (32 << case["log2_t"]) * 30 + n * 32, "flops": n * (3 * FIELD_FLOPS + 1024)}
    pixels = case["width"] * case["height"] * case.get("views", 1)
    return {"bytes": min(table, n * 512) + pixels * (20 if k == "render" else 4), "flops": n * (FIELD_FLOPS + 512)}


def tolerance(case):
    """About four times the distance of the path from exact(): the fields and
    renders are 3e-5 and 1e-5 off (fp16 activations), the weight gradients of
    random output gradients 2e-2 (fp16 deltas that cancel; the oracle, which
    rounds at the same points, is within 1e-3), a training step 3e-3 (hash
    grid) and 2e-4 (reference network).  An activation on the other side of a
    ReLU or of an fp16 tie moves single values by more ("max")."""
    k = case["kind"]
    if k == "encode":  # eight products summed in fp32; the cell and its weights have one form
        return {"rel": 1e-6, "max": 1e-5} if case["f32"] else {"rel": 1e-4, "max": 1e-3}
    if k in ("field", "mlp", "ref_field"):
        return {"rel": 2e-4, "max": 1e-2}
    if k == "ref_grad":
        return {"rel": 4e-3, "max": 0.1}
    if k == "train":
        return {"rel": 1e-3, "max": 0.3} if case["ref"] else {"rel": 1e-2, "max": 0.9}
    return {"rel": 5e-5, "max": 5e-3, "differ": 5e-3}  # and bytes that a rounding moves by one


# ----------------------------------------------------------- in 64 bits
PRIMES = (1, 2654435761, 805459861)


def _levels(case):
    if case.get("finest"):
        b = (case["finest"] / 16.0) ** (1.0 / 15.0)
    else:
        b = float(np.float32(1.3819))
    return [int(math.floor(16.0 * b**l + 1e-9)) for l in range(16)]


def _corners(case, p, n_l, level):
    """Entry numbers and trilinear weights of the 8 corners around points p."""
    t = 1 << case["log2_t"]
    q = p.clamp(0, 1) * n_l
    i = q.floor().clamp(max=n_l - 1)
    f, i = q - i, i.long()
    out = []
    for c in range(8):
        o = [(c >> a) & 1 for a in range(3)]
        x = [i[:, a] + o[a] for a in range(3)]
        if (n_l + 1) ** 3 <= t:
            e = x[0] + x[1] * (n_l + 1) + x[2] * (n_l + 1) ** 2
        else:
            e = ((x[0] * PRIMES[0]) ^ (x[1] * PRIMES[1]) ^ (x[2] * PRIMES[2])) & (t - 1)
        w = torch.ones_like(q[:, 0])
        for a in range(3):
            w = w * (f[:, a] if o[a] else 1 - f[:, a])
        out.append((e + level * t, w))
    return out


def _encode(case, table, p):
    out = torch.zeros((p.shape[0], 32), dtype=torch.float64, device=DEV)
    for level, n_l in enumerate(_levels(case)):
        for e, w in _corners(case, p, n_l, level):
            out[:, 2 * level : 2 * level + 2] += w[:, None] * table[e].double()
    return out


def _sh4(d):
    x, y, z = d[:, 0], d[:, 1], d[:, 2]
    x2, y2, z2 = x * x, y * y, z * z
    return torch.stack([
        torch.full_like(x, 0.28209479177387814), -0.48860251190291987 * y, 0.48860251190291987 * z, -0.48860251190291987 * x, 1.0925484305920792 * x * y, -1.0925484305920792 * y * z,
        0.94617469575755997 * z2 - 0.31539156525251999, -1.0925484305920792 * x * z, 0.54627421529603959 * (x2 - y2), 0.59004358992664352 * y * (y2 - 3 * x2), 2.8906114426405538 * x * y * z,
        0.45704579946446572 * y * (1 - 5 * z2), 0.3731763325901154 * z * (5 * z2 - 3), 0.45704579946446572 * x * (1 - 5 * z2), 1.4453057213202769 * z * (x2 - y2), 0.59004358992664352 * x * (3 * y2 - x2)], 1)


def _matrices(flat, shapes):
    out, at = [], 0
    for o, i in shapes:
        out.append(flat[at : at + o * i].view(o, i))
        at += o * i
    return out


def _mlp(x, ms):
    for m in ms[:-1]:
        x = torch.relu(x @ m.T)
    return x @ ms[-1].T


def _hash_raw(features, d, wd, wc):
    """(raw density, raw colour) of the hash-grid model's MLPs."""
    o = _mlp(features, _matrices(wd, DENSITY))
    c = _mlp(torch.cat([o[:, 1:16], _sh4(d), torch.zeros_like(o[:, :1])], 1), _matrices(wc, COLOR))
    return o[:, 0], c[:, :3]


def _freq(v, levels):
    parts = [v]
    for l in range(levels):
        parts += [torch.sin(v * 2.0**l), torch.cos(v * 2.0**l)]
    return torch.cat(parts, 1)


def _ref_raw(p, d, wd, wc):
    """(raw density, raw colour) of the reference's network."""
    pad = lambda x, n: torch.cat([x, torch.zeros((x.shape[0], n - x.shape[1]), dtype=x.dtype, device=DEV)], 1)  # noqa: E731
    o = _mlp(pad(_freq(p, 10), 64), _matrices(wd, REF_DENSITY))
    c = _mlp(pad(torch.cat([o[:, 1:16], _freq(d, 4)], 1), 48), _matrices(wc, REF_COLOR))
    return o[:, 0], c[:, :3]


def _by_chunks(n, chunk, f):
    return torch.cat([f(slice(a, min(n, a + chunk))) for a in range(0, n, chunk)])


def _hash_field(case, table, wd, wc, p, d):
    def part(s):
        sr, cr = _hash_raw(_encode(case, table, p[s].double()), d[s].double(), wd.double(), wc.double())
        return torch.cat([sr.exp()[:, None], torch.sigmoid(cr)], 1)

    return _by_chunks(p.shape[0], 1 << 19, part)


F = np.float32


def _rays(cam, px, py, box):
    """Pixel rays clipped to the box, in 32 bits as they are defined: origin,
    directions, near, far and which hit."""
    m = np.array(cam.c2w[:], F).reshape(3, 4)
    dx, dy, dz = (px - F(cam.cx)) / F(cam.fx), (F(cam.height) - F(1) - py - F(cam.cy)) / F(cam.fy), F(-1)
    d = [m[a, 0] * dx + m[a, 1] * dy + m[a, 2] * dz for a in range(3)]
    inv = F(1) / np.sqrt(d[0] * d[0] + d[1] * d[1] + d[2] * d[2])
    d = np.stack([v * inv for v in d], 1)
    o = m[:, 3]
    with np.errstate(divide="ignore"):
        inv_d = np.where(np.abs(d) > F(1e-8), F(1) / d, np.where(d >= 0, F(1e8), F(-1e8)))
    t0, t1 = (np.array(box[:3], F) - o) * inv_d, (np.array(box[3:], F) - o) * inv_d
    tn, tf = np.minimum(t0, t1).max(1), np.maximum(t0, t1).min(1)
    hit = (tn <= tf) & (tf > 0)
    return o, d.astype(F), np.maximum(tn, F(0)), tf, hit


def _march(cam, rays, box, steps, res, occupied):
    """(ray, t, dt) of the occupied steps of every ray, ray by ray."""
    o, d, tn, tf, hit = rays
    cone = F(0.5) * (F(1) / F(cam.fx) + F(1) / F(cam.fy))
    dt_min = (tf - tn) / F(steps)
    lo, hi = np.array(box[:3], F), np.array(box[3:], F)
    t, got = tn.copy(), []
    for _ in range(steps):
        live = np.nonzero(hit & (t < tf))[0]
        if not live.size:
            break
        dt = np.minimum(np.maximum(dt_min[live], t[live] * cone), tf[live] - t[live])
        tm = t[live] + F(0.5) * dt
        rel = (o + tm[:, None] * d[live] - lo) / (hi - lo)
        inside = ((rel >= 0) & (rel < 1)).all(1)
        cell = np.minimum(res - 1, (rel * F(res)).clip(0).astype(np.int64))
        keep = inside & occupied(cell[:, 0] + cell[:, 1] * res + cell[:, 2] * res * res)
        got.append((live[keep], tm[keep], dt[keep]))
        t[live] = t[live] + dt
    ray, tm, dt = (np.concatenate([g[k] for g in got]) for k in range(3))
    order = np.argsort(ray, kind="stable")
    return ray[order], tm[order], dt[order]


def _tensor(x):
    return torch.from_numpy(np.ascontiguousarray(x)).to(DEV)


def _before(tau, ray, n_rays):
    """Optical depth in front of each sample of its ray, and of whole rays."""
    total = torch.zeros(n_rays, dtype=torch.float64, device=DEV).index_add(0, ray, tau)
    run = torch.cumsum(tau, 0) - tau
    first = torch.cumsum(total, 0) - total
    return run - first[ray], total


def _exact_render(case, seed):
    if case["cascades"] > 1 or case["width"] * case["height"] * case["steps"] > 1 << 23:
        return None
    w, h, box = case["width"], case["height"], _render_box(case)
    m, cam = Model(case, seed), _cameras(case, seed)[0]
    words = _occupancy(case, seed).cpu().numpy().view(np.uint32)
    x, y = np.meshgrid(np.arange(w), np.arange(h))
    rays = _rays(cam, x.ravel().astype(F) + F(0.5), y.ravel().astype(F) + F(0.5), box)
    ray, tm, dt = _march(cam, rays, box, case["steps"], case["res"], lambda i: (words[i >> 5] >> (i & 31).astype(np.uint32)) & 1 == 1)
    rt, d = _tensor(ray), _tensor(rays[1])
    p = _tensor(rays[0]).double() + _tensor(tm).double()[:, None] * d[rt].double()
    f = _hash_field(case, m.table, m.wd, m.wc, p, d[rt])
    tau = f[:, 0] * _tensor(dt).double()
    front, _ = _before(tau, rt, w * h)
    used = torch.exp(-front) >= T_STOP  # the sample that falls below is the last one
    tau = torch.where(used, tau, torch.zeros_like(tau))
    front, total = _before(tau, rt, w * h)
    rgb = torch.zeros((w * h, 3), dtype=torch.float64, device=DEV).index_add(0, rt, (torch.exp(-front) * -torch.expm1(-tau))[:, None] * f[:, 1:])
    return {"rgba8": None, "rgb": (rgb + torch.exp(-total)[:, None]).view(1, h, w, 3), "counts": None}


def _hash32(x):
    x = x.astype(np.uint32)
    with np.errstate(over="ignore"):
        x ^= x >> np.uint32(16)
        x *= np.uint32(0x7FEB352D)
        x ^= x >> np.uint32(15)
        x *= np.uint32(0x846CA68B)
        x ^= x >> np.uint32(16)
    return x


def _splitmix(a, b, n):
    """n 24-bit uniforms in [0, 1) of the splitmix64 stream keyed (a, b)."""
    g, m1, m2 = np.uint64(0x9E3779B97F4A7C15), np.uint64(0xBF58476D1CE4E5B9), np.uint64(0x94D049BB133111EB)
    with np.errstate(over="ignore"):
        z = ((np.uint64(a) + g) ^ (np.uint64(b) * m1)) + np.arange(1, n + 1, dtype=np.uint64) * g
        z = (z ^ (z >> np.uint64(30))) * m1
        z = (z ^ (z >> np.uint64(27))) * m2
        z ^= z >> np.uint64(31)
    return (z >> np.uint64(40)).astype(F) * F(2.0**-24)


def _init(shapes, a, b):
    u, at, out = _splitmix(a, b, sum(o * i for o, i in shapes)), 0, []
    for o, i in shapes:
        out.append((u[at : at + o * i] * F(2) - F(1)) * F(math.sqrt(6.0 / (o + i))))
        at += o * i
    return _tensor(np.concatenate(out))


def _exact_train(case, seed):
    """The first step of a training run, its gradients by autograd."""
    hp, ref, steps = _hyper(case), case["ref"], case["steps"]
    w, h, n_rays = case["width"], case["height"], case["rays"]
    pick = int(_hash32(np.array([2891336453], np.uint32))[0]) % VIEWS
    cam, img = _camera(seed, pick, w, h), _images(case, seed)[pick].astype(F) * F(1.0 / 255.0)
    with np.errstate(over="ignore"):
        key = np.arange(n_rays, dtype=np.uint32) * np.uint32(9781)
    unit = lambda k: (_hash32(key ^ np.uint32(k)) & np.uint32(0xFFFFFF)).astype(F) / F(16777216.0)  # noqa: E731
    px, py = unit(0xA511E9B3) * F(w), unit(0x63D83595) * F(h)
    rays = _rays(cam, px, py, BOX)
    ray, tm, dt = _march(cam, rays, BOX, steps, 128, lambda i: np.ones(i.shape, bool))  # every cell is marked when training begins
    count = np.bincount(ray, minlength=n_rays)
    fits = (count > 0) & (np.cumsum(count) <= case["cap"])
    keep = fits[ray]
    rt, tm, dt = _tensor(ray[keep]), _tensor(tm[keep]).double(), _tensor(dt[keep]).double()
    d = _tensor(rays[1])[rt].double()
    p = _tensor(rays[0]).double() + tm[:, None] * d
    x, y = px.clip(0, w - 1), py.clip(0, h - 1)
    x0, y0 = np.floor(x).astype(int), np.floor(y).astype(int)
    x1, y1 = np.minimum(x0 + 1, w - 1), np.minimum(y0 + 1, h - 1)
    fx, fy = (x - x0)[:, None], (y - y0)[:, None]
    px4 = (img[y0, x0] * (1 - fx) + img[y0, x1] * fx) * (1 - fy) + (img[y1, x0] * (1 - fx) + img[y1, x1] * fx) * fy
    gt, alpha = _tensor(px4[:, :3] * px4[:, 3:] + (1 - px4[:, 3:])).double(), _tensor(px4[:, 3]).double()
    shapes = (REF_DENSITY, REF_COLOR) if ref else (DENSITY, COLOR)
    start = [_init(shapes[0], 0x1234, 0x5678), _init(shapes[1], 0x9ABC, 0xDEF0)]
    wd, wc = (s.half().double().requires_grad_() for s in start)
    if ref:
        sr, cr = _ref_raw(p, d, wd, wc)
        sigma = torch.nn.functional.softplus(sr)
    else:
        table = _tensor((_splitmix(0x7AB1E, seed % (1 << 31), 32 << case["log2_t"]) * F(2) - F(1)) * F(0.1))
        features = _encode(case, table.half().view(-1, 2), p).requires_grad_()
        sr, cr = _hash_raw(features, d, wd, wc)
        sigma = sr.exp()
    tau = sigma * dt.clamp(min=0)
    front, total = _before(tau, rt, n_rays)
    pred = torch.zeros((n_rays, 3), dtype=torch.float64, device=DEV).index_add(0, rt, (torch.exp(-front) * -torch.expm1(-tau))[:, None] * torch.sigmoid(cr)) + torch.exp(-total)[:, None]
    e = (pred - gt)[_tensor(fits)]
    if ref:
        loss = ((0.1 + 0.9 * alpha.clamp(0, 1))[_tensor(fits)][:, None] * e * e).sum()
    else:
        loss = torch.where(e.abs() <= 0.1, 0.5 * e * e, 0.1 * (e.abs() - 0.05)).sum()
    (loss / int(fits.sum()) * hp["loss_scale"]).backward()
    out = {"mlp_grad": torch.cat([wd.grad, wc.grad])}
    weights = {"mlp": torch.cat(start).double()}
    if not ref:
        g = torch.zeros((16 << case["log2_t"], 2), dtype=torch.float64, device=DEV)
        for level, n_l in enumerate(_levels(case)):
            for i, c in _corners(case, p, n_l, level):
                g.index_add_(0, i, c[:, None] * features.grad[:, 2 * level : 2 * level + 2])
        out["table_grad"], weights["table"] = g.view(-1), table.double()
    norm = math.sqrt(sum(float((g * g).sum()) for g in out.values())) / hp["loss_scale"]
    scale = (hp["clip"] / norm if norm > hp["clip"] else 1.0) / hp["loss_scale"]
    lr = hp["lr"] * (0.1 ** (1.0 / (hp["lr_decay_ksteps"] * 1000.0)) if hp["lr_decay_ksteps"] else 1.0)
    for k, v in weights.items():  # the first step's moments, freed of their bias, are the gradient and its square
        g = out[k + "_grad"] * scale
        out[k] = v - lr * g / (g.abs() + hp["eps"])
    return out


def exact(case, seed):
    kind = case["kind"]
    if kind == "render":
        return _exact_render(case, seed)
    if kind == "train":
        return _exact_train(case, seed)
    if kind == "image":  # bytes
        return None
    s = _points_case(case, seed)
    n = case["n"]
    if kind == "encode":
        return _by_chunks(n, 1 << 20, lambda k: _encode(case, s["table"].t, s["pos"].t[k].double()))
    if kind == "field":
        return _hash_field(case, s["table"].t, s["wd"], s["wc"], s["pos"].t, s["dirs"])
    wd, wc = s["wd"].double(), s["wc"].double()
    if kind == "mlp":
        def part(k):
            sr, cr = _hash_raw(s["features"][k].double(), s["dirs"][k].double(), wd, wc)
            return torch.cat([sr.exp()[:, None], torch.sigmoid(cr)], 1)

        return _by_chunks(n, 1 << 20, part)
    if kind == "ref_field":
        def part(k):
            sr, cr = _ref_raw(s["pos"][k].double(), s["dirs"][k].double(), wd, wc)
            return torch.cat([torch.nn.functional.softplus(sr)[:, None], torch.sigmoid(cr)], 1)

        return _by_chunks(n, 1 << 18, part)
    wd.requires_grad_()
    wc.requires_grad_()
    for a in range(0, n, 1 << 17):
        k = slice(a, min(n, a + (1 << 17)))
        sr, cr = _ref_raw(s["pos"][k].double(), s["dirs"][k].double(), wd, wc)
        (128.0 * ((sr * s["draw"][k, 0]).sum() + (cr * s["draw"][k, 1:]).sum())).backward()
    return {"density": wd.grad, "color": wc.grad}
