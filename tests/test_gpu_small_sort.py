"""The small sort at the edges of its partitions and of the size up to which it is taken, and the
projection's chunk sizes at the edge between them, against the CPU oracle bit for bit.

Every gaussian covers exactly one tile, so n gaussians are n intersections."""

from __future__ import annotations

import numpy as np
import pytest
import torch

import splax_amd
from conftest import assert_bit_exact
from oracle import oracle as O
from splax_amd import _lib, _ops
from splax_amd.scenes import make_scene

pytestmark = pytest.mark.gpu

HW = (250, 330)


def _t(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def _dots(n, seed):
    """n one-tile gaussians at random tile centres, a few depths shared by many."""
    rng = np.random.default_rng(seed)
    tiles = np.stack([rng.integers(0, HW[1] // 16, n), rng.integers(0, HW[0] // 16, n)], 1)
    xys = (16 * tiles + 8).astype(np.float32)
    depths = rng.choice(rng.uniform(1, 9, max(2, n // 3)).astype(np.float32), n)
    conics = np.tile(np.array([1.0, 0.0, 1.0], np.float32), (n, 1))
    opac = rng.uniform(0.1, 1.0, n).astype(np.float32)
    return xys, depths, np.full(n, 4, np.int32), conics, opac, np.arange(1, n + 1, dtype=np.int32)


@pytest.mark.parametrize("wide", [False, True])
@pytest.mark.parametrize("n", [1, 2, 63, 1023, 1024, 1025, 5000, 81919, 81920, 81921])
def test_small_sort_edges(n, wide):
    xys, depths, radii, conics, opac, cum = _dots(n, n)
    _lib.set_wide_keys(wide)
    O.set_wide_keys(wide)
    try:
        rk, rid, rbins = O.sort_and_bin(xys, depths, radii, conics, opac, cum, n=n, B=1,
                                        img_shape=HW)
        gk, gid, gbins = _ops.sort_and_bin(_t(xys), _t(depths), _t(radii), _t(conics), _t(opac),
                                           _t(cum), n=n, B=1, img_shape=HW)
        # the kept forward: 16-bit key halves after two passes, positions, a bound above the count
        *_, kept, _ = _ops.rasterize_fwd_keep(
            _t(np.full((n, 3), 0.5, np.float32)), _t(opac), _t(opac),
            _t(np.zeros((1, 3), np.float32)), _t(xys), _t(depths), _t(radii), _t(conics),
            _t(cum), n=n, B=1, img_shape=HW)
    finally:
        _lib.set_wide_keys(False)
        O.set_wide_keys(False)
    assert_bit_exact(gk.cpu().numpy(), rk, "keys")
    assert_bit_exact(gid.cpu().numpy(), rid, "ids")
    assert_bit_exact(gbins.cpu().numpy(), rbins, "bins")
    assert kept.M == n
    assert_bit_exact(kept.ids.cpu().numpy()[:n], rid, "kept ids")
    assert_bit_exact(kept.bins.cpu().numpy(), rbins, "kept bins")
    # one intersection per gaussian: the emission position is the id
    assert_bit_exact(kept.pos.cpu().numpy()[:n], rid, "positions")


@pytest.mark.parametrize("n,B", [(255, 2), (256, 3), (257, 2), (1000, 5), (131072, 2),
                                 (131073, 2)])
def test_projection_chunks(n, B):
    """Images whose edges fall inside 256- and 1024-item chunks: prefix, count and (through the
    packed keys) depth range."""
    s = make_scene(3, n=n)
    vm = np.ascontiguousarray(s.viewmats[:B])
    q = np.roll(s.quats, -1, axis=-1)
    ref = O.project_fwd(s.means, s.scales, q, vm.reshape(-1, 4), s.opacities, n=n, total=B * n,
                        img_shape=s.img_shape, f=s.f, c=s.c)
    rk, rid, rbins = O.sort_and_bin(*ref[:4], s.opacities, ref[5], n=n, B=B,
                                    img_shape=s.img_shape)
    tf, tids = torch.zeros((1, 4, 4)).cuda(), torch.full((1,), -1, dtype=torch.int32).cuda()
    _, _, _, kept, _ = _ops.render_fwd(
        _t(s.means), _t(s.scales), _t(s.quats), _t(s.colors), _t(s.opacities).reshape(-1),
        _t(vm.reshape(-1, 4)), _t(s.background[None]), tf, tids, n=n, B=B, num_transforms=1,
        has_transforms=False, img_shape=s.img_shape, f=s.f, c=s.c, glob_scale=1.0,
        clip_thresh=0.01)
    assert kept.M == rid.size
    assert_bit_exact(kept.cum.cpu().numpy(), ref[5].ravel(), "cum")
    assert_bit_exact(kept.sort.ids.cpu().numpy()[:kept.M], rid, "ids")
    assert_bit_exact(kept.sort.bins.cpu().numpy(), rbins, "bins")
    xys, _, _, _, _, cum = splax_amd.project(
        _t(s.means), _t(s.scales), _t(s.quats), _t(vm), opacities=_t(s.opacities).reshape(-1),
        img_shape=s.img_shape, f=s.f)
    assert_bit_exact(cum.cpu().numpy().ravel(), ref[5].ravel(), "project cum")
