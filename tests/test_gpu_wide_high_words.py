"""64-bit keys sorted by their high words after the depth passes (kept forwards) against whole keys
(splat_sort_and_bin) and the CPU oracle, bit for bit, beside the small sort's limit, in both
partition sizes, and where no tile or image bits are left to sort."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from conftest import assert_bit_exact
from oracle import oracle as O
from splax_amd import _lib, _ops
from test_gpu_small_sort import _t

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,B,hw", [(81_920, 1, (250, 330)), (81_921, 1, (250, 330)),
                                    (90_000, 1, (16, 16)), (100_003, 3, (250, 330)),
                                    (1_048_575, 1, (250, 330)), (350_001, 3, (16, 16))])
def test_wide_high_words(n, B, hw):
    rng = np.random.default_rng(n)
    total = B * n
    tiles = np.stack([rng.integers(0, max(hw[1] // 16, 1), total),
                      rng.integers(0, max(hw[0] // 16, 1), total)], 1)
    xys = (16 * tiles + 8).astype(np.float32)
    depths = rng.choice(rng.uniform(0.01, 900, n // 3).astype(np.float32), total)
    conics = np.tile(np.array([1.0, 0.0, 1.0], np.float32), (total, 1))
    opac = rng.uniform(0.1, 1.0, n).astype(np.float32)
    radii = np.full(total, 4, np.int32)
    cum = np.arange(1, total + 1, dtype=np.int32)
    _lib.set_wide_keys(True)
    O.set_wide_keys(True)
    try:
        rk, rid, rbins = O.sort_and_bin(xys, depths, radii, conics, opac, cum, n=n, B=B,
                                        img_shape=hw)
        args = [_t(a) for a in (xys, depths, radii, conics)]
        gk, gid, gbins = _ops.sort_and_bin(*args, _t(opac), _t(cum), n=n, B=B, img_shape=hw)
        *_, kept, _ = _ops.rasterize_fwd_keep(
            _t(np.full((n, 3), 0.5, np.float32)), _t(opac), _t(opac),
            _t(np.zeros((1, 3), np.float32)), *args, _t(cum), n=n, B=B, img_shape=hw)
        torch.cuda.synchronize()
    finally:
        _lib.set_wide_keys(False)
        O.set_wide_keys(False)
    assert_bit_exact(gk.cpu().numpy(), rk, "keys")
    assert_bit_exact(gid.cpu().numpy(), rid, "ids")
    assert_bit_exact(gbins.cpu().numpy(), rbins, "bins")
    assert kept.M == total
    assert_bit_exact(kept.ids.cpu().numpy()[:total], rid, "kept ids")
    assert_bit_exact(kept.bins.cpu().numpy(), rbins, "kept bins")
    assert_bit_exact(kept.pos.cpu().numpy()[:total], rid, "positions")
