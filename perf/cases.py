"""The calls whose speed matters to a program that uses splax_amd, over the sizes it calls them at.

Each case is one pass through the public entry points:

- ``view``: ``render`` without gradients (a viewer or an evaluation frame);
- ``fit``: ``render_loss`` and its gradients (fitting a splat to target images);
- ``stages``: ``project`` then ``rasterize``, a loss on the image, and the gradients (programs that
  use the projection's outputs between the two);
- ``objects``: ``render`` with rigidly moved slices of gaussians and the depth map, a loss on both,
  and the gradients, those of the transforms among them (dynamic scenes);
- ``train``: one ``TrainStep`` (antialiased render, L1, Adam, relocation);
- ``adam``: one ``Adam.step`` over the five parameter groups;
- ``mcmc``: ``mcmc.relocate`` then ``mcmc.inject_noise``.

The scenes are those of the benchmark's workloads: a cube of gaussians, or gaussians on 64 random
planes (heavy overlap, early termination), seen by one camera or by cameras on an orbit.
"""

from __future__ import annotations

import math

import numpy as np
import torch

import splax_amd
from splax_amd import mcmc
from splax_amd.optim import Adam
from splax_amd.train import DEFAULT_LRS, SPLAT_KEYS, TrainStep, l1_loss
from splax_amd.utils import look_at

_BASE = {"layout": "planes", "cameras": 1, "pose": False, "antialiased": False, "depth": False,
         "objects": 0, "loss": "mse"}


def _case(name, kind, n, height, width, focal, **more):
    c = {"name": name, "kind": kind, "n": n, "height": height, "width": width,
         "focal": float(focal), **_BASE, **more}
    return c if name else {k: v for k, v in c.items() if k != "name"}


def listed():
    return [
        # a thumbnail or a small preview, drawn once per interaction: latency and launches
        _case("view-256-10k", "view", 10_000, 256, 256, 300, layout="cube1"),
        # the smallest benchmark workload: a unit test's or a toy example's step
        _case("fit-256-10k", "fit", 10_000, 256, 256, 300, layout="cube1"),
        # a Blender-style object at its usual 800 x 800
        _case("fit-800-100k", "fit", 100_000, 800, 800, 1100, layout="cube2"),
        # a full scene at 1080p, the benchmark's headline workload
        _case("fit-1080p-1m", "fit", 1_000_000, 1080, 1920, 1500),
        # the same scene in a viewer: antialiased, with the depth map, no gradients
        _case("view-1080p-1m", "view", 1_000_000, 1080, 1920, 1500, antialiased=True, depth=True),
        # many small cameras in one launch, their poses refined with the splat
        _case("poses-16x512-500k", "fit", 500_000, 512, 512, 600, cameras=16, pose=True),
        # a batch of full-size cameras: image and tile bits leave no room for the packed key
        _case("fit-8x1080p-200k", "fit", 200_000, 1080, 1920, 1500, cameras=8, loss="l1"),
        # odd sizes through the two separate stages
        _case("stages-757x1003-250k", "stages", 250_001, 757, 1003, 1050, loss="l1"),
        # a dynamic scene at VGA: twelve moving objects, colour and depth supervised
        _case("objects-479x637-150k", "objects", 150_001, 479, 637, 620, objects=12, depth=True,
              loss="l1"),
        # the large training step: 3M gaussians, four cameras
        _case("train-4x1600x1060-3m", "train", 3_000_000, 1060, 1600, 1400, cameras=4,
              antialiased=True, loss="l1"),
        # the optimizer by itself, for programs with a step of their own
        _case("adam-1m", "adam", 1_000_000, 0, 0, 0),
        # relocation and noise by themselves, with the share of dead gaussians of early training
        _case("mcmc-1m", "mcmc", 1_000_000, 0, 0, 0),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["view", "view", "fit", "fit", "fit", "fit", "stages", "objects", "train",
                       "adam", "mcmc"])
    if kind in ("adam", "mcmc"):
        return _case("", kind, _log_int(rng, 5_000, 3_000_000), 0, 0, 0)
    layout = rng.choice(["cube1", "cube2", "planes", "planes"])
    n = _log_int(rng, 2_000, 1_500_000 if layout == "planes" else 150_000)
    h, w = _log_int(rng, 97, 1100), _log_int(rng, 97, 1930)
    cameras = 1 if kind in ("stages", "objects") or rng.random() < 0.5 else rng.randint(2, 16)
    while cameras > 1 and (cameras * h * w > 17_000_000 or cameras * n > 12_000_000):
        cameras -= 1
    return _case("", kind, n, h, w, round(max(h, w) * rng.uniform(0.7, 1.2), 1), layout=layout,
                 cameras=cameras, pose=kind == "fit" and rng.random() < 0.3,
                 antialiased=kind == "train" or (kind == "view" and rng.random() < 0.5),
                 depth=kind == "objects" or (kind == "view" and rng.random() < 0.5),
                 objects=rng.randint(1, 24) if kind == "objects" else 0,
                 loss="l1" if kind in ("stages", "objects", "train") else
                 rng.choice(["l1", "mse"]))


# ------------------------------------------------------------------ inputs

_LAYOUTS = {  # half-width of the means, log-scale and opacity-logit (mean, deviation), distance
    "cube1": (1.0, (-4.0, 0.5), (0.0, 1.0), 4.0),
    "cube2": (2.0, (-4.0, 0.5), (0.0, 1.0), 6.0),
    "planes": (3.0, (-5.0, 0.7), (1.0, 1.5), 8.0),
}


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed) * 7919 + 17)


def _normal(g, *shape):
    return torch.randn(shape, generator=g, device="cuda")


def _uniform(g, lo, hi, *shape):
    return torch.rand(shape, generator=g, device="cuda") * (hi - lo) + lo


def _unit(t):
    return t / t.norm(dim=-1, keepdim=True)


def _means(case, g):
    half, n = _LAYOUTS[case["layout"]][0], case["n"]
    if case["layout"] != "planes":
        return _uniform(g, -half, half, n, 3)
    normal = _unit(_normal(g, 64, 3))
    axis = torch.eye(3, device="cuda")[(normal[:, 0].abs() > 0.9).long()]
    e1 = _unit(torch.linalg.cross(normal, axis))
    e2 = torch.linalg.cross(normal, e1)
    offset = _uniform(g, -half, half, 64, 1)
    on = torch.randint(0, 64, (n,), generator=g, device="cuda")
    uv = _uniform(g, -half, half, n, 2)
    return ((offset * normal)[on] + uv[:, :1] * e1[on] + uv[:, 1:] * e2[on]
            + 0.02 * _normal(g, n, 3))


def _splat(case, g):
    """means, log-scales, unit quaternions (wxyz), colours, opacity logits."""
    _, ls, op, _ = _LAYOUTS[case["layout"]]
    n = case["n"]
    return (_means(case, g), ls[0] + ls[1] * _normal(g, n, 3), _unit(_normal(g, n, 4)),
            _uniform(g, 0.0, 1.0, n, 3), op[0] + op[1] * _normal(g, n, 1))


def _viewmats(case):
    b, dist = case["cameras"], _LAYOUTS[case["layout"]][3]
    if b == 1:
        vm = look_at(np.array([[0.0, 0.0, dist]]), np.zeros(3))
    else:
        az, el = 2 * np.pi * np.arange(b) / b, np.radians(20.0)
        eye = (dist - 1.0) * np.stack([np.cos(el) * np.cos(az), np.cos(el) * np.sin(az),
                                       np.full(b, np.sin(el))], 1)
        vm = look_at(eye, np.zeros(3), up=(0, 0, 1))
    return torch.from_numpy(vm).cuda()


def _transforms(k, g):
    """k rigid motions: a turn of up to about 20 degrees and a shift."""
    q = _unit(torch.cat([torch.ones(k, 1, device="cuda"), 0.1 * _normal(g, k, 3)], 1))
    w, x, y, z = q.unbind(1)
    m = torch.zeros(k, 4, 4, device="cuda")
    m[:, 0] = torch.stack([1 - 2 * (y * y + z * z), 2 * (x * y - z * w), 2 * (x * z + y * w),
                           0 * x], 1)
    m[:, 1] = torch.stack([2 * (x * y + z * w), 1 - 2 * (x * x + z * z), 2 * (y * z - x * w),
                           0 * x], 1)
    m[:, 2] = torch.stack([2 * (x * z - y * w), 2 * (y * z + x * w), 1 - 2 * (x * x + y * y),
                           0 * x], 1)
    m[:, :3, 3] = 0.1 * _normal(g, k, 3)
    m[:, 3, 3] = 1.0
    return m


def _slices(n, k):
    """k disjoint runs of gaussians of unequal lengths, with static ones between them."""
    edges = [n * i // k for i in range(k + 1)]
    return [(a, max(a + 1, b - (b - a) * (1 + i % 3) // 8))
            for i, (a, b) in enumerate(zip(edges, edges[1:]))]


def _adam_inputs(case, g):
    n = case["n"]
    widths = dict(zip(SPLAT_KEYS, (3, 3, 4, 3, 1)))
    params = {k: _normal(g, n, w) for k, w in widths.items()}
    grads = {k: 1e-6 * _normal(g, n, w) for k, w in widths.items()}
    mu = {k: 1e-6 * _normal(g, n, w) for k, w in widths.items()}
    nu = {k: (1e-6 * _normal(g, n, w)) ** 2 for k, w in widths.items()}
    return params, grads, mu, nu


_ADAM_COUNT = 100


def prepare(case, seed):
    g, kind, n = _generator(seed), case["kind"], case["n"]
    if kind == "adam":
        params, grads, mu, nu = _adam_inputs(case, g)
        opt = Adam(params, DEFAULT_LRS)
        opt.mu, opt.nu, opt.count = mu, nu, _ADAM_COUNT
        return {"case": case, "opt": opt, "grads": grads}
    if kind == "mcmc":
        means, log_scales, quats, colors, logits = _splat(case, g)
        dead = torch.rand((n, 1), generator=g, device="cuda") < 0.05
        logits = torch.where(dead, -6.0 - logits.abs(), logits)
        colors = torch.logit(colors, eps=1e-4)
        return {"case": case, "params": (means, log_scales, quats, colors, logits),
                "binoms": mcmc.make_binoms(51), "key": int(seed)}
    means, log_scales, quats, colors, logits = _splat(case, g)
    hw, viewmats = (case["height"], case["width"]), _viewmats(case)
    background = torch.ones(3, device="cuda")
    target = _uniform(g, 0.0, 1.0, case["cameras"], *hw, 3)
    camera = {"img_shape": hw, "f": (case["focal"], case["focal"])}
    if kind == "train":
        params = dict(zip(SPLAT_KEYS, (means, log_scales, quats,
                                       torch.logit(colors, eps=1e-4), logits)))
        return {"case": case, "step": TrainStep(
            params, viewmats=viewmats, targets=target, background=background,
            antialiased=case["antialiased"], seed=int(seed) & 0xffff, **camera)}
    if case["cameras"] == 1:
        viewmats, target = viewmats[0], target[0]
    leaves = [means, log_scales.exp(), quats, colors, torch.sigmoid(logits)]
    state = {"case": case, "viewmat": viewmats, "target": target, "background": background,
             "camera": camera, "leaves": leaves}
    if kind != "view":
        if case["pose"]:
            leaves.append(viewmats)
        if kind == "objects":
            state["transforms"] = _transforms(case["objects"], g)
            state["slices"] = _slices(n, case["objects"])
            state["target_depth"] = _uniform(g, 4.0, 12.0, *hw)
            leaves.append(state["transforms"])
        for t in leaves:
            t.requires_grad_(True)
    return state


# ------------------------------------------------------------------ one pass

_NAMES = ("means", "scales", "quats", "colors", "opacities")


def _named(case):
    more = (("viewmat",) if case["pose"] else ()) + (("transforms",) if case["objects"] else ())
    return _NAMES + more


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "adam":
        opt = state["opt"]
        opt.step(state["grads"])
        return {"params": opt.params, "mu": opt.mu, "nu": opt.nu}
    if kind == "mcmc":
        new, reset = mcmc.relocate(state["key"], *state["params"], state["binoms"])
        means = mcmc.inject_noise(state["key"], new[0], new[1], new[2], new[4], 50.0)
        return {"means": means, "log_scales": new[1], "quats": new[2], "colors": new[3],
                "opacities": new[4], "reset": reset}
    if kind == "train":
        step = state["step"]
        loss = step()
        return {"loss": loss, "params": step.params, "mu": step.opt.mu, "nu": step.opt.nu}
    splat, cam = state["leaves"][:5], state["camera"]
    views = {"viewmat": state["viewmat"], "background": state["background"]}
    if kind == "view":
        with torch.no_grad():
            image, depth = splax_amd.render(*splat, antialiased=case["antialiased"],
                                            render_depth=case["depth"], **views, **cam)
        return {"image": image, "depth": depth}
    if kind == "fit":
        loss, image = splax_amd.render_loss(*splat, target=state["target"], loss=case["loss"],
                                            **views, **cam)
        out = {"loss": loss, "image": image}
    elif kind == "stages":
        means, scales, quats, colors, opacities = splat
        xys, depths, radii, conics, _, cum = splax_amd.project(
            means, scales, quats, state["viewmat"], opacities=opacities, **cam)
        image = splax_amd.rasterize(colors, opacities, state["background"], xys, depths, radii,
                                    conics, cum, img_shape=cam["img_shape"])
        loss = l1_loss(image, state["target"])
        out = {"loss": loss, "image": image}
    else:
        image, depth = splax_amd.render(*splat, render_depth=True,
                                        gaussian_transforms=state["transforms"],
                                        gaussian_slices=state["slices"], **views, **cam)
        loss = l1_loss(image, state["target"]) + 0.1 * l1_loss(depth, state["target_depth"])
        out = {"loss": loss, "image": image, "depth": depth}
    grads = torch.autograd.grad(loss, state["leaves"])
    return {**{k: t.detach() for k, t in out.items()}, "grads": dict(zip(_named(case), grads))}


# ------------------------------------------------------------------ what a pass cannot do without

def work(case):
    kind, n, b = case["kind"], case["n"], case["cameras"]
    if kind == "adam":  # p, g, mu, nu read; p, mu, nu written; about 15 operations per value
        return {"bytes": 14 * n * 28, "flops": 14 * n * 15}
    if kind == "mcmc":  # every row read and written once, and the mask; Sigma w per gaussian
        return {"bytes": n * (56 + 56 + 1), "flops": n * 120}
    pixels = b * case["height"] * case["width"]
    # pixel-gaussian pairs: the area where an opacity of about 0.6 stays above 1/255, of the
    # share of the gaussians in view, up to the depth at which a pixel saturates
    _, ls, _, dist = _LAYOUTS[case["layout"]]
    sigma = math.exp(ls[0] + 0.5 * ls[1] ** 2) * case["focal"] / dist
    pairs = min(0.8 * n * b * 31.0 * (sigma ** 2 + 0.3), 40.0 * pixels)
    image = 4 * pixels * (3 + (1 if case["depth"] else 0))
    if kind == "view":
        return {"bytes": 56 * n + image, "flops": 26 * pairs + 300 * n * b}
    # forward and backward: the splat, the targets and the image; the gradients
    step = {"bytes": 56 * n + 2 * image + 56 * n, "flops": 91 * pairs + 900 * n * b}
    if kind == "train":
        step["bytes"] += 14 * n * 28 - 112 * n
        step["flops"] += 14 * n * 15
    return step


def tolerance(case):
    """float32 throughout: about four times what the cases differ by from ``exact``. An image is
    1e-5 from it (a pixel whose alpha lands on the other side of 1/255); gradients under the mean
    square are up to 4.6e-4 (the sums of needle-thin gaussians, multiplied by their conics'
    condition), under L1 up to 2.6e-3 (the sign of a pixel's difference turns)."""
    kind = case["kind"]
    if kind == "adam":
        return {"rel": 4e-7, "max": 1e-5}
    if kind == "mcmc":
        return {"rel": 1e-5, "max": 1e-4, "differ": 1e-5}
    if kind == "view":
        return {"rel": 5e-5, "max": 0.02}
    if kind == "train":  # Adam divides a gradient by its own size: a few signs of zero may turn
        return {"rel": 1e-3, "max": 0.5}
    return {"rel": 1e-2 if case["loss"] == "l1" else 2e-3, "max": 0.1}


# ------------------------------------------------------------------ the same in 64 bits

_ALPHA_MIN, _ALPHA_MAX, _T_MIN = (float(np.float32(v)) for v in (1 / 255, 0.999, 1e-4))


def _key_bits(b, h, w):
    """Depth bits of the packed sort key, or None where the order is by the raw depth."""
    tiles = -(-h // 16) * -(-w // 16)
    bits = 31 - (b - 1).bit_length() - (tiles - 1).bit_length()
    return bits if bits >= 16 else None


def _project64(p, vm, case, transforms, slices):
    """Screen positions, conics, blend opacities and depths of one camera in 64 bits."""
    h, w, f = case["height"], case["width"], case["focal"]
    means, scales, quats, colors, opac = p
    # the rotation's diagonal is 2 w^2 - 1 + 2 v^2, differentiated as 1 - 2 (the other squares):
    # the same for a unit quaternion, and these are that up to rounding
    qw, x, y, z = quats.unbind(1)
    v2 = quats[:, 1:] * quats[:, 1:]
    diagonal = 1 - 2 * (v2.sum(1, keepdim=True) - v2)
    diagonal = diagonal + (2 * (qw * qw)[:, None] - 1 + 2 * v2 - diagonal).detach()
    R = torch.stack([diagonal[:, 0], 2 * (x * y - z * qw), 2 * (x * z + y * qw),
                     2 * (x * y + z * qw), diagonal[:, 1], 2 * (y * z - x * qw),
                     2 * (x * z - y * qw), 2 * (y * z + x * qw), diagonal[:, 2]],
                    1).reshape(-1, 3, 3)
    if transforms is not None:
        ids = torch.full((means.shape[0],), -1, device=means.device)
        for k, (a, e) in enumerate(slices):
            ids[a:e] = k
        tf = torch.cat([transforms, torch.eye(4, dtype=torch.float64, device=means.device)[None]])
        tf = tf[ids]
        means = (tf[:, :3, :3] * means[:, None, :]).sum(-1) + tf[:, :3, 3]
        R = (tf[:, :3, :3, None] * R[:, None, :, :]).sum(2)
    M = R * scales[:, None, :]
    V = (M[:, :, None, :] * M[:, None, :, :]).sum(-1)
    W = vm[:3, :3]
    c = (W[None] * means[:, None, :]).sum(-1) + vm[:3, 3]
    cx, cy, cz = c.unbind(1)
    front = cz.detach() > 0.01
    safe = torch.where(front, cz, torch.ones_like(cz))

    def cov(tx, ty, tz):
        zero = torch.zeros_like(tz)
        J = torch.stack([torch.stack([f / tz, zero, -f * tx / tz ** 2], 1),
                         torch.stack([zero, f / tz, -f * ty / tz ** 2], 1)], 1)
        T = (J[:, :, :, None] * W[None, None]).sum(2)
        TV = (T[:, :, :, None] * V[:, None]).sum(2)
        S = (TV[:, :, None, :] * T[:, None, :, :]).sum(-1)
        return S[:, 0, 0] + 0.3, S[:, 0, 1], S[:, 1, 1] + 0.3

    # the covariance at the clamped position, differentiated at the unclamped one
    lim = [1.3 * 0.5 * s / f for s in (w, h)]
    free = cov(cx, cy, safe)
    with torch.no_grad():
        held = cov(safe * (cx / safe).clamp(-lim[0], lim[0]),
                   safe * (cy / safe).clamp(-lim[1], lim[1]), safe)
    A, B, C = (u + (v - u.detach()) for u, v in zip(free, held))
    det = A * C - B * B
    conic = torch.stack([C / det, -B / det, A / det], 1)
    xy = torch.stack([cx / (safe + 1e-6) * f + w / 2, cy / (safe + 1e-6) * f + h / 2], 1)
    o = opac[:, 0]
    with torch.no_grad():
        t = 2 * torch.log(255 * o.clamp(min=1e-30))
        ok = front & (o >= _ALPHA_MIN) & (t > 0)
        ext = torch.sqrt(t.clamp(min=0)[:, None] * torch.stack([A, C], 1))
        lo = torch.floor((xy - ext) / 16).nan_to_num().clamp(-1, 1 << 20).long()
        hi = torch.floor((xy + ext) / 16).nan_to_num().clamp(-1, 1 << 20).long()
        lim_t = torch.tensor([-(-w // 16) - 1, -(-h // 16) - 1], device=o.device)
        lo, hi = lo.clamp(min=0), torch.minimum(hi, lim_t)
        size = torch.where(ok[:, None], (hi - lo + 1).clamp(min=0), 0)
    if case["antialiased"]:
        a_, b_, c_ = conic.unbind(1)
        o = o * torch.sqrt((1 - 0.3 * (a_ + c_) + 0.09 * (a_ * c_ - b_ * b_)).clamp(0, 1))
    return xy, conic, o, cz, (lo, size)


def _float32_depth(means, vm, transforms, slices):
    """The depth as float32 sums give it: it decides the order of the blend."""
    m = means
    if transforms is not None:
        m = m.clone()
        for k, (a, e) in enumerate(slices):
            t, s = transforms[k], means[a:e]
            for i in range(3):
                m[a:e, i] = ((t[i, 0] * s[:, 0] + t[i, 1] * s[:, 1]) + t[i, 2] * s[:, 2]) + t[i, 3]
    return ((vm[2, 0] * m[:, 0] + vm[2, 1] * m[:, 1]) + vm[2, 2] * m[:, 2]) + vm[2, 3]


def _tile_lists(z32, lo, size, case):
    """Ids of every tile's gaussians front to back, by tiles from the fullest down."""
    h, w = case["height"], case["width"]
    nx, ny = -(-w // 16), -(-h // 16)
    seen = (size.prod(1) > 0).nonzero()[:, 0]
    depth, bits = z32[seen], _key_bits(case["cameras"], h, w)
    if bits is not None and seen.numel():
        span = depth.max() - depth.min()
        top = float((1 << bits) - 1)
        depth = ((depth - depth.min()) / span * top).int().clamp(0, int(top)) if span > 0 \
            else torch.zeros_like(depth)
    seen = seen[torch.sort(depth, stable=True)[1]]
    lo, size = lo[seen], size[seen]
    count = size.prod(1)
    item = torch.repeat_interleave(torch.arange(seen.numel(), device=z32.device), count)
    at = torch.arange(item.numel(), device=z32.device) - (count.cumsum(0) - count)[item]
    tile = (lo[item, 1] + at // size[item, 0]) * nx + lo[item, 0] + at % size[item, 0]
    tile, by = torch.sort(tile, stable=True)
    per = torch.bincount(tile, minlength=nx * ny)
    first = per.cumsum(0) - per
    per, order = torch.sort(per, descending=True)
    return seen[item[by]], first[order], per, order


class _Blend64:
    """The alpha blend of one image, all tiles a step at a time, and its backward."""

    def __init__(self, xy, conic, o, colors, z, lists, case, background):
        self.ids, self.first, per, order = lists
        h, w = case["height"], case["width"]
        nx = -(-w // 16)
        dev = xy.device
        px = torch.arange(256, device=dev)
        self.x = ((order % nx) * 16)[:, None] + px[None] % 16
        self.y = ((order // nx) * 16)[:, None] + px[None] // 16
        self.inside = (self.x < w) & (self.y < h)
        self.pixel = self.y * w + self.x
        self.table = torch.cat([xy, conic, o[:, None], colors, z[:, None]], 1)
        counts = per.cpu().numpy()
        self.active = [int(a) for a in np.searchsorted(-counts, -np.arange(
            counts[0] if len(counts) else 0), side="left")]
        self.bg = background
        self.hw = (h, w)

    def _step(self, k):
        a = self.active[k]
        g = self.ids[self.first[:a] + k]
        r = self.table[g]
        dx = r[:, 0:1] - (self.x[:a] + 0.5)
        dy = r[:, 1:2] - (self.y[:a] + 0.5)
        sigma = 0.5 * (r[:, 2:3] * dx * dx + r[:, 4:5] * dy * dy) + r[:, 3:4] * dx * dy
        raw = r[:, 5:6] * torch.exp(-sigma)
        alpha = raw.clamp(max=_ALPHA_MAX)
        return a, g, r, dx, dy, raw, alpha, (sigma >= 0) & (alpha >= _ALPHA_MIN)

    def forward(self):
        shape = self.x.shape
        new = lambda *s: torch.zeros(*s, dtype=torch.float64, device=self.x.device)  # noqa: E731
        self.T, self.out = 1.0 + new(shape), new(*shape, 4)
        self.last = torch.full(shape, -1, device=self.x.device)
        done = ~self.inside
        for k in range(len(self.active)):
            if k % 64 == 0 and bool(done.all()):
                break
            a, _, r, _, _, _, alpha, ok = self._step(k)
            ok &= ~done[:a]
            after = self.T[:a] * (1 - alpha)
            stop = ok & (after <= _T_MIN)
            done[:a] |= stop
            ok &= ~stop
            weight = torch.where(ok, alpha * self.T[:a], 0.0)
            self.out[:a] += weight[..., None] * r[:, None, 6:10]
            self.T[:a] = torch.where(ok, after, self.T[:a])
            self.last[:a] = torch.where(ok, k, self.last[:a])
        image, depth = new(self.hw[0] * self.hw[1], 3), new(self.hw[0] * self.hw[1])
        at = self.pixel[self.inside]
        image[at] = (self.out[..., :3] + self.T[..., None] * self.bg)[self.inside]
        depth[at] = self.out[..., 3][self.inside]
        return image.reshape(*self.hw, 3), depth.reshape(self.hw)

    def backward(self, v_image, v_depth):
        """Cotangents of the table's columns. A saturated alpha passes none to its exponent."""
        v = torch.cat([v_image.reshape(-1, 3), v_depth.reshape(-1, 1)], 1)
        v = torch.where(self.inside[..., None], v[self.pixel.clamp(max=v.shape[0] - 1)], 0.0)
        T = self.T.clone()
        behind = T * (v[..., :3] * self.bg).sum(-1)  # what the blend puts behind, times v
        grad = torch.zeros_like(self.table)
        for k in range(min(len(self.active), int(self.last.max()) + 1) - 1, -1, -1):
            a, g, r, dx, dy, raw, alpha, ok = self._step(k)
            ok &= k <= self.last[:a]
            alpha = torch.where(ok, alpha, 0.0)
            T[:a] /= 1 - alpha
            dot = (r[:, None, 6:10] * v[:a]).sum(-1)
            v_alpha = T[:a] * dot - behind[:a] / (1 - alpha)
            weight = alpha * T[:a]
            behind[:a] += weight * dot
            geo = ok & (raw <= _ALPHA_MAX)
            v_sigma = torch.where(geo, -raw * v_alpha, 0.0)
            part = torch.stack([
                (v_sigma * (r[:, 2:3] * dx + r[:, 3:4] * dy)).sum(1),
                (v_sigma * (r[:, 4:5] * dy + r[:, 3:4] * dx)).sum(1),
                (0.5 * v_sigma * dx * dx).sum(1), (v_sigma * dx * dy).sum(1),
                (0.5 * v_sigma * dy * dy).sum(1), -v_sigma.sum(1) / r[:, 5]], 1)
            part = torch.cat([part, (weight[..., None] * v[:a]).sum(1)], 1)
            grad.index_add_(0, g, part)
        return grad


def _exact_adam(case, seed):
    params, grads, mu, nu = ({k: t.double() for k, t in d.items()}
                             for d in _adam_inputs(case, _generator(seed)))
    count = _ADAM_COUNT + 1
    for k in params:
        mu[k] = 0.9 * mu[k] + 0.1 * grads[k]
        nu[k] = 0.999 * nu[k] + 0.001 * grads[k] ** 2
        params[k] = params[k] - DEFAULT_LRS[k] * (mu[k] / (1 - 0.9 ** count)) / (
            torch.sqrt(nu[k] / (1 - 0.999 ** count)) + 1e-8)
    return {"params": params, "mu": mu, "nu": nu}


def exact(case, seed):
    kind = case["kind"]
    if kind == "adam":
        return _exact_adam(case, seed)
    if kind in ("mcmc", "train"):  # random draws; decisions that follow the last bit
        return None
    state = prepare(case, seed)
    target, b = state["target"], case["cameras"]
    leaves = [t.detach().double().requires_grad_(kind != "view") for t in state["leaves"]]
    named = dict(zip(_named(case), leaves))
    vms32 = state["viewmat"].detach().reshape(-1, 4, 4)
    tf32 = state["transforms"].detach() if "transforms" in state else None
    bg, slices = state["background"].double(), state.get("slices")
    images, depths, loss = [], [], 0.0
    grads = [torch.zeros_like(t) for t in leaves]
    for i in range(b):
        vms = named["viewmat"].reshape(-1, 4, 4) if case["pose"] else vms32.double()
        xy, conic, o, z, (lo, size) = _project64(leaves[:5], vms[i], case,
                                                 named.get("transforms"), slices)
        z32 = _float32_depth(state["leaves"][0].detach(), vms32[i], tf32, slices)
        blend = _Blend64(xy.detach(), conic.detach(), o.detach(), leaves[3].detach(), z.detach(),
                         _tile_lists(z32, lo, size, case), case, bg)
        image, depth = blend.forward()
        images.append(image)
        depths.append(depth)
        if kind == "view":
            continue
        d = image - target.reshape(-1, *image.shape)[i].double()
        total = float(target.numel())
        v_image = torch.sign(d) / total if case["loss"] == "l1" else 2 * d / total
        loss = loss + (d.abs() if case["loss"] == "l1" else d * d).sum() / total
        v_depth = torch.zeros_like(depth)
        if kind == "objects":
            e = depth - state["target_depth"].double()
            v_depth = 0.1 * torch.sign(e) / e.numel()
            loss = loss + 0.1 * e.abs().mean()
        v = blend.backward(v_image, v_depth)
        # a gaussian that reaches no tile gets no gradient (its conic may not be finite)
        hit = size.prod(1) > 0
        outs = [t[hit] for t in (xy, conic, o, leaves[3], z)]
        vs = [t[hit] for t in (v[:, 0:2], v[:, 2:5], v[:, 5], v[:, 6:9], v[:, 9])]
        part = torch.autograd.grad(outs, leaves, vs, allow_unused=True)
        grads = [a if p is None else a + p for a, p in zip(grads, part)]
        del blend, v, part, outs, vs
    image = torch.stack(images) if b > 1 else images[0]
    depth = torch.stack(depths) if b > 1 else depths[0]
    if kind == "view":
        return {"image": image, "depth": depth if case["depth"] else None}
    out = {"loss": loss, "image": image, "grads": dict(zip(_named(case), grads))}
    if kind == "objects":
        out["depth"] = depth
    return out
