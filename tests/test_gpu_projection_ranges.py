"""The projection and the key emission at the edges of their number ranges and sizes, against the CPU
oracle bit for bit: operands inside and outside the ranges of the shared-reciprocal divisions and
the short square root, keys staged in LDS and stored directly, chunk scans of one to several
spans."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from conftest import assert_bit_exact
from oracle import oracle as O
from splax_amd import _lib, _ops
from splax_amd.scenes import make_scene

pytestmark = pytest.mark.gpu

HW = (250, 330)


def _t(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def _project(means, scales, quats, vm, opac, *, n, B, hw, f, c, clip=0.01):
    tf, tids = torch.zeros((1, 4, 4)).cuda(), torch.full((1,), -1, dtype=torch.int32).cuda()
    return _ops.project_fwd(_t(means), _t(scales), _t(quats), _t(vm), _t(opac), tf, tids, n=n,
                            total=B * n, num_transforms=1, has_transforms=False, img_shape=hw,
                            f=f, c=c, glob_scale=1.0, clip_thresh=clip)


def _same(a, b, what):
    for x, y, name in zip(a, b, ("xys", "depths", "radii", "conics", "num_tiles_hit", "cum")):
        assert_bit_exact(x.cpu().numpy().reshape(np.asarray(y).shape), y, f"{what} {name}")


@pytest.mark.parametrize("decades", [3, 12, 20])
def test_operand_ranges(decades):
    """Depths, offsets and scales over up to 40 decades (2^-66 to 2^66), zeros among the offsets,
    spheres (b near zero), opacities at and beside 1/255 and far above 1."""
    rng = np.random.default_rng(decades)
    n = 20_000
    z = 10.0 ** rng.uniform(-decades, decades, n)
    xy = rng.uniform(-0.6, 0.6, (n, 2)) * z[:, None]
    xy[rng.random((n, 2)) < 0.05] = 0.0
    xy[rng.random((n, 2)) < 0.05] *= 1e-19
    means = np.concatenate([xy, z[:, None]], 1).astype(np.float32)
    scales = (z[:, None] * 10.0 ** rng.uniform(-4, 1, (n, 3))).astype(np.float32)
    scales[:2000] = scales[:2000, :1]  # spheres
    scales[2000:4000] = 10.0 ** rng.uniform(-decades, decades, (2000, 3))
    q = rng.normal(size=(n, 4))
    q = (q / np.linalg.norm(q, axis=1, keepdims=True)).astype(np.float32)
    q[1000:1500] = [0, 0, 0, 1]
    opac = rng.uniform(0.0, 1.0, n).astype(np.float32)
    edge = np.float32(1 / 255)
    opac[::7] = edge
    opac[1::7] = np.nextafter(edge, np.float32(1))
    opac[2::49] = 1e25
    vm = np.eye(4, dtype=np.float32)
    kw = dict(f=(300.0, 290.0), c=(165.0, 125.0))
    ref = O.project_fwd(means, scales, q, vm, opac, n=n, total=n, img_shape=HW,
                        clip_thresh=1e-25, **kw)
    got = _project(means, scales, q, vm, opac, n=n, B=1, hw=HW, clip=1e-25, **kw)
    _same(got, ref, f"{decades} decades")
    assert (ref[2] > 0).sum() > n // 4
    for wide in (False, True):
        _lib.set_wide_keys(wide)
        O.set_wide_keys(wide)
        try:
            rk, rid, _ = O.sort_and_bin(*ref[:4], opac, ref[5], n=n, B=1, img_shape=HW)
            gk, gid, _ = _ops.sort_and_bin(*got[:4], _t(opac), got[5], n=n, B=1, img_shape=HW)
        finally:
            _lib.set_wide_keys(False)
            O.set_wide_keys(False)
        assert_bit_exact(gk.cpu().numpy(), rk, "keys")
        assert_bit_exact(gid.cpu().numpy(), rid, "ids")


@pytest.mark.parametrize("wide", [False, True])
@pytest.mark.parametrize("n", [262_144, 262_145, 262_400])
def test_staged_emission(n, wide):
    """Workgroups with no key, a few, and more than the staged ones, on both sides of the item count
    from which keys are staged."""
    s = make_scene(3, n=n)
    scales = (s.scales * 0.05).astype(np.float32)
    scales[1000:1300] *= 200.0       # large ellipses across two workgroups
    scales[n - 100:] *= 200.0        # and in the last one
    opac = s.opacities.reshape(-1).copy()
    opac[5120:8192] = 0.0            # workgroups without a key
    q = np.roll(s.quats, -1, axis=-1)
    vm = s.viewmats[0]
    kw = dict(f=s.f, c=s.c)
    ref = O.project_fwd(s.means, scales, q, vm, opac, n=n, total=n, img_shape=s.img_shape, **kw)
    got = _project(s.means, scales, q, vm, opac, n=n, B=1, hw=s.img_shape, **kw)
    _same(got, ref, f"{n} items")
    per = np.add.reduceat(np.asarray(ref[4]).reshape(-1), np.arange(0, n, 256))
    assert per.max() > 2048 and per.min() == 0
    _lib.set_wide_keys(wide)
    O.set_wide_keys(wide)
    try:
        rk, rid, rbins = O.sort_and_bin(*ref[:4], opac, ref[5], n=n, B=1, img_shape=s.img_shape)
        gk, gid, gbins = _ops.sort_and_bin(*got[:4], _t(opac), got[5], n=n, B=1,
                                           img_shape=s.img_shape)
    finally:
        _lib.set_wide_keys(False)
        O.set_wide_keys(False)
    assert_bit_exact(gk.cpu().numpy(), rk, "keys")
    assert_bit_exact(gid.cpu().numpy(), rid, "ids")
    assert_bit_exact(gbins.cpu().numpy(), rbins, "bins")


@pytest.mark.parametrize("total", [256 * 4096, 256 * 4096 + 1, 256 * 16384 + 1,
                                   256 * 3 * 16384 + 255, 256 * 3 * 16384 + 257])
def test_chunk_scan_spans(total):
    """cum_tiles_hit is the running sum of num_tiles_hit at one, four and twelve spans of chunks and
    past them."""
    g = torch.Generator("cuda").manual_seed(total)
    means = torch.rand((total, 3), device="cuda", generator=g) * 2 - 1
    means[:, 2] += 3
    scales = torch.full((total, 3), 0.01, device="cuda")
    quats = torch.tensor([[0.0, 0.0, 0.0, 1.0]], device="cuda").expand(total, 4).contiguous()
    opac = torch.full((total,), 0.5, device="cuda")
    tf, tids = torch.zeros((1, 4, 4)).cuda(), torch.full((1,), -1, dtype=torch.int32).cuda()
    out = _ops.project_fwd(means, scales, quats, torch.eye(4, device="cuda"), opac, tf, tids,
                           n=total, total=total, num_transforms=1, has_transforms=False,
                           img_shape=HW, f=(300.0, 300.0), c=(165.0, 125.0), glob_scale=1.0,
                           clip_thresh=0.01)
    nth, cum = out[4].reshape(-1), out[5].reshape(-1)
    assert int(nth.max()) > 1
    assert torch.equal(cum, torch.cumsum(nth, 0, dtype=torch.int32))
