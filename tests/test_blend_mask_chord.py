"""The blends' sub-block masks from clamped chord heights (CPU only).

`subblock_mask` (csrc/blend.hip) evaluates the chord of a record's ellipse at the heights of its
extreme points clamped to each band, from fields the record pack forms (`pack_record`,
csrc/splat_common.hpp). Both are restated here step by step in float32, with every hardware
reciprocal and square root off by its 1 ulp in either direction, and checked against the brute
force of the blend's own sigma test over all 256 pixel centres: no sub-block that a pixel centre
reaches is dropped. Mirroring the extreme point's height in the restated mask breaks that.
"""

from __future__ import annotations

import numpy as np
import pytest

from test_blend_masks import (BW, _fma, _scene_records, _synthetic_records, _tiles_of, f32,
                              mask_tight, reach)


def _ulp(v, by):
    """v moved by `by` units in the last place."""
    v = v.astype(f32)
    return np.nextafter(v, f32(by) * f32(np.inf), dtype=f32) if by else v


def chord_fields(R, by):
    with np.errstate(all="ignore"):
        a, b, c = (f32(2) * R["ha"]).astype(f32), R["b"], (f32(2) * R["hc"]).astype(f32)
        smax = R["smax"]
        det = (a * c - b * b).astype(f32)
        tr = (a + c).astype(f32)
        k = (f32(2) * smax * _ulp(f32(1) / det, by)).astype(f32)
        box = (a > 0) & (c > 0) & (det > 0) & (tr * tr < f32(1e4) * det) & (k * tr < f32(1e30))
        ex = (_ulp(np.sqrt(k * c), by) * f32(1.01)).astype(f32)
        ia4 = (f32(0.25) * _ulp(f32(1) / a, by)).astype(f32)
        m = _fma(f32(2.5e-4), ex, f32(2.5e-3))
        d = ((det * ia4).astype(f32) * ia4).astype(f32)
        dy_r = (-(b * ex).astype(f32) * _ulp(f32(1) / c, by)).astype(f32)
    none = ~(smax >= 0)
    box &= ~none
    z = np.zeros_like(a)
    return dict(ia4=np.where(box, ia4, none.astype(f32)),
                m=np.where(box, m, np.where(none, z, f32(1e30))),
                d=np.where(box, d, z), dy_r=np.where(box, dy_r, z))


def mask_chord(R, F, tx, ty, by=0, peak_sign=1):
    m, d = F["m"], F["d"]
    p = ((f32(0.5) * f32(1.0201)) * R["smax"] * F["ia4"]).astype(f32)
    s = (-R["b"] * F["ia4"]).astype(f32)
    dy_r = (f32(peak_sign) * F["dy_r"]).astype(f32)
    bx = (((np.asarray(tx) * BW).astype(f32) + f32(0.5)) - R["x"]).astype(f32)
    by_ = (((np.asarray(ty) * BW).astype(f32) + f32(0.5)) - R["y"]).astype(f32)
    kr = _fma(bx, f32(-0.25), (m + f32(1)).astype(f32))
    kl = _fma(bx, f32(0.25), (m + f32(4.75)).astype(f32))
    mask = np.zeros(bx.shape, np.uint32)
    with np.errstate(all="ignore"):
        for j in range(4):
            y0, y1 = (by_ + f32(4 * j)).astype(f32), (by_ + f32(4 * j + 3)).astype(f32)
            n = []
            for sgn, kk in ((1, kr), (-1, kl)):
                t = np.clip(f32(sgn) * dy_r, y0, y1).astype(f32)
                w = _ulp(np.sqrt(_fma(-(d * t).astype(f32), t, p)), by)
                h = _fma(f32(sgn) * s, t, (w + kk).astype(f32))
                n.append(np.nan_to_num(np.clip(h, 0, 4), nan=0.0).astype(np.uint32))
            nr, nl = n
            width = np.maximum((nr + nl).astype(np.int64) - 4, 0)
            mask |= (((1 << width) - 1) << (4 * j + 4 - nl.astype(np.int64))).astype(np.uint32)
    return mask


def _records():
    rng = np.random.default_rng(3)
    return (_scene_records(2, 60_000, rng, 1500), _scene_records(1, 30_000, rng, 800),
            _synthetic_records(rng, 3000))


@pytest.mark.parametrize("ulp", [0, 1, -1])
def test_chord_mask_keeps_every_sub_block_a_pixel_reaches(ulp):
    for R in _records():
        idx, tx, ty = _tiles_of(R)
        F = {k: v[idx] for k, v in chord_fields(R, ulp).items()}
        R = {k: v[idx] for k, v in R.items()}
        got = mask_chord(R, F, tx, ty, by=ulp)
        missed = reach(R, tx, ty) & ~got
        assert not missed.any(), f"{int((missed != 0).sum())} (record, tile) pairs lose a sub-block"
        # as tight as the chords at the band's ends: both bound the same extent
        kept = [int(np.unpackbits(v.astype(np.uint32).view(np.uint8)).sum())
                for v in (got, mask_tight(R, tx, ty))]
        assert kept[0] <= 1.001 * kept[1], kept


def test_mirrored_extreme_point_loses_sub_blocks():
    R = _synthetic_records(np.random.default_rng(4), 1500)
    idx, tx, ty = _tiles_of(R)
    F = {k: v[idx] for k, v in chord_fields(R, 0).items()}
    R = {k: v[idx] for k, v in R.items()}
    assert (reach(R, tx, ty) & ~mask_chord(R, F, tx, ty, peak_sign=-1)).any()


def test_records_without_a_chord():
    """An opacity no pixel accepts keeps nothing; a conic past the conditioning limit everything."""
    from test_blend_masks import pack
    R = pack([20, 20.3], [20, 20.6], [1.0, 1.0], [0.0, 0.99999], [1.0, 1.0], [1e-3, 0.9])
    F = chord_fields(R, 0)
    assert mask_chord(R, F, np.array([1, 1]), np.array([1, 1])).tolist() == [0, 0xFFFF]
