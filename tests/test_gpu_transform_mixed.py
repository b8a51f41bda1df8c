"""The transform gradient where a wave holds many transforms (ids in any order, more transforms
than a wave has lanes, none moved in some waves) against the CPU oracle, and the GPU's slice ids
against the CPU's past one launch's 64 slices."""

from __future__ import annotations

import numpy as np
import pytest
import torch

import splax_amd
from oracle import oracle as O
from splax_amd import _ops
from test_gpu_transforms import C, F, HW, _grad_compare, _np, _scene, _t, _transforms, _viewmats

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,K", [(63, 2), (256, 64), (257, 5), (1000, 130)])
def test_mixed_ids_gradient_matches_oracle(n, K):
    rng, means, scales, quats, opac = _scene(n, n + K)
    ids = rng.integers(-1, K + 1, n).astype(np.int32)  # -1 and K are static
    ids[64:128] = -1
    tf, vms = _transforms(rng, K), _viewmats(1)
    q = np.roll(quats, -1, axis=-1)
    _, _, radii, conics, _, _ = O.project_fwd(
        means, scales, q, vms.reshape(-1, 4), opac, n=n, total=n, img_shape=HW, f=F, c=C,
        transforms=tf, transform_ids=ids, num_transforms=K)
    v_xy = rng.normal(size=(n, 2)).astype(np.float32)
    v_depth = rng.normal(size=n).astype(np.float32)
    v_conic = rng.normal(size=(n, 3)).astype(np.float32)
    ref = O.project_bwd(means, scales, q, vms.reshape(-1, 4), radii, conics, v_xy, v_depth,
                        v_conic, n=n, B=1, f=F, transforms=tf, transform_ids=ids,
                        num_transforms=K)
    got = _ops.project_bwd(_t(means), _t(scales), _t(q), _t(vms).reshape(-1, 4), _t(radii),
                           _t(conics), _t(v_xy), _t(v_depth), _t(v_conic), _t(tf), _t(ids), n=n,
                           B=1, num_transforms=K, has_transforms=True, f=F, glob_scale=1.0)
    _grad_compare(_np(got[4]).reshape(ref[4].shape), ref[4], "v_transforms")


@pytest.mark.parametrize("n,k", [(1, 1), (300, 12), (1000, 64), (1000, 65), (4000, 200)])
def test_slice_ids_equal_the_cpu(n, k):
    edges = np.sort(np.random.default_rng(k).choice(n + 1, size=min(2 * k, n + 1), replace=False))
    slices = [(int(a), int(b)) for a, b in zip(edges[::2], edges[1::2])]
    np.random.default_rng(k + 1).shuffle(slices)
    got = splax_amd.transform_ids(n, slices, device="cuda")
    assert got.dtype == torch.int32 and got.device.type == "cuda"
    assert torch.equal(got.cpu(), splax_amd.transform_ids(n, slices))
    assert (splax_amd.transform_ids(n, [], device="cuda") == -1).all()
