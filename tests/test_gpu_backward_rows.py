"""The backward blend's row walks at the sizes where they can go wrong: sub-block lists of 1 to 5
records (a group takes four steps), tiles whose ranges end inside, at and just past a batch (112
records), records whose alpha is clamped in some batches only, the depth channel's tenth sum, and
images narrower than a tile. Every pixel is reached by every record, so each row's list is the
tile's. Bars: those of test_gpu_sweep.py against the CPU oracle and its float64 truth.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

import splax_amd
import timed_path as TP
from conftest import assert_bit_exact, rel_fro

pytestmark = pytest.mark.gpu


def _scene(n, H, W, seed, opaque_every):
    """n gaussians wider than the image in front of one camera, thin enough (opacity about 1/n)
    that every one of them is blended at most pixels; every ``opaque_every``-th of the rear half
    has opacity 1."""
    rng = np.random.default_rng(seed)
    opac = rng.uniform(0.5, 1.5, n).astype(np.float32) * np.float32(min(0.4, 3.0 / n)) + 0.006
    means = np.stack([rng.uniform(-0.2, 0.2, n), rng.uniform(-0.2, 0.2, n),
                      np.sort(rng.uniform(0.0, 1.0, n))], 1)
    if opaque_every:
        opac[n // 2::opaque_every] = 1.0
    return {
        "means": means.astype(np.float32),
        "scales": rng.uniform(0.4, 0.9, (n, 3)).astype(np.float32),
        "quats": np.tile(np.array([1, 0, 0, 0], np.float32), (n, 1)),
        "colors": rng.uniform(0, 1, (n, 3)).astype(np.float32),
        "opac": opac.reshape(n, 1), "bg": np.ones(3, np.float32), "img_shape": (H, W),
        "f": (20.0, 20.0), "c": (W / 2, H / 2),
        "vm": np.block([[np.eye(3), np.array([[0.0], [0.0], [3.0]])],
                        [np.zeros((1, 3)), np.ones((1, 1))]]).astype(np.float32),
    }


@pytest.mark.parametrize("depth", [False, True])
@pytest.mark.parametrize("n,H,W,opaque_every", [
    (2, 16, 16, 0), (3, 16, 16, 1), (4, 5, 3, 0), (5, 16, 16, 2), (111, 16, 16, 0),
    (112, 16, 16, 40), (113, 17, 15, 0), (224, 16, 16, 0), (225, 16, 33, 112), (340, 9, 16, 150),
])
def test_row_walks_match_oracle(n, H, W, opaque_every, depth):
    sc = _scene(n, H, W, 31 * n + H, opaque_every)
    rng = np.random.default_rng(n)
    w = rng.uniform(-1, 1, (H, W, 3)).astype(np.float32)
    wd = rng.uniform(-1, 1, (H, W)).astype(np.float32)
    t = lambda a, g=False: torch.from_numpy(np.ascontiguousarray(a)).cuda().requires_grad_(g)  # noqa: E731
    p = {k: t(sc[k], True) for k in ("means", "scales", "quats", "colors", "opac")}
    img, dep = splax_amd.render(*p.values(), viewmat=t(sc["vm"]), background=t(sc["bg"]),
                                img_shape=(H, W), f=sc["f"], render_depth=depth)
    loss = (img * t(w)).sum()
    if depth:
        loss = loss + (dep * t(wd)).sum()
    loss.backward()
    kw = {"wd": wd} if depth else {}
    ref, rg, cond = TP.weighted_chain(sc, w, vm=sc["vm"], **kw)
    _, tg, _ = TP.weighted_chain(sc, w, vm=sc["vm"], truth=True, **kw)
    image = ref[0] if depth else ref
    got = img.detach().cpu().numpy()
    assert_bit_exact(got, image.reshape(got.shape), "image")
    for k, v in p.items():
        g = v.grad.cpu().numpy().astype(np.float64)
        r = np.asarray(rg[k], np.float64).reshape(g.shape)
        truth = np.asarray(tg[k], np.float64).reshape(g.shape)
        assert rel_fro(g, r) < 1e-4, (k, rel_fro(g, r))
        for (lo, hi), (cnt, eg, eo) in zip(TP.BANDS, TP.band_errors(g, r, truth, cond)):
            if cnt >= 32:
                assert eg <= max(TP.FACTOR * eo, 1e-5), (k, lo, cnt, eg, eo)
