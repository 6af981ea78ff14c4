"""The sines and cosines a float32 forward takes, read off its own output.

With unit and zero bond lengths and the default frame a coordinate is one sine or cosine rounded to
float32, which differs from the correctly rounded one only where the double it came from lies on the
other side of a rounding boundary: for an error of e about e / 2^-24 of the values do (the largest
binade; fewer at smaller values).  A first angle's 1.4e-14 leaves about 2e-7 of them, a huge angle's
3e-16 none, an error of 1e-11 about 1e-4.  Bars: 1e-5 of the values.
"""

from __future__ import annotations

import numpy as np
import pytest

SHAPES = [(1 << 20, 4), (60000, 135)]  # packed chains, one chain per workgroup


def _angles(batch, huge, seed):
    rng = np.random.default_rng(seed)
    if not huge:
        return rng.uniform(0.2, 2.9, batch).astype(np.float32)
    sign = rng.choice([-1.0, 1.0], batch)
    return (sign * 2.0 ** rng.uniform(16.001, 127.9, batch)).astype(np.float32)


def _forward(device, batch, points, lengths, first_angle, angle, dihedral):
    import torch

    import cufk_amd

    L = torch.zeros(batch, points - 1, device=device)
    for k, v in lengths.items():
        L[:, k] = v
    A = torch.full((batch, points - 2), float(np.float32(np.pi / 2)), device=device)
    D = torch.zeros(batch, points - 3, device=device)
    for dst, v in ((A[:, 0], first_angle), (A[:, 1], angle), (D[:, 0], dihedral)):
        if v is not None:
            dst.copy_(torch.from_numpy(v))
    return cufk_amd.reconstruct(L, A, D).cpu().numpy()


@pytest.mark.gpu
@pytest.mark.parametrize("batch,points", SHAPES)
@pytest.mark.parametrize("huge", [True, False])
def test_first_angle(device, batch, points, huge):
    """x2 = (-cos, sin, 0) of the first angle for bonds (0, 1)."""
    a = _angles(batch, huge, 1)
    x2 = _forward(device, batch, points, {1: 1.0}, a, None, None)[:, 2]
    s, c = np.sin(a.astype(np.float64)), np.cos(a.astype(np.float64))
    keep = np.abs(s) > 0.1  # the frame is a right one for a positive sine
    wrong = (x2[keep, 1] != s[keep].astype(np.float32)).mean(), (x2[keep, 0] != (-c[keep]).astype(np.float32)).mean()
    print("differ", wrong)
    assert max(wrong) <= 1e-5 + 2 / batch


@pytest.mark.gpu
@pytest.mark.parametrize("batch,points", SHAPES)
def test_huge_dihedral(device, batch, points):
    """x3 - x2 stands on the first plane by sin(dihedral) for a unit third bond and right angles."""
    d = _angles(batch, True, 2)
    x3 = _forward(device, batch, points, {2: 1.0}, None, None, d)[:, 3]
    wrong = (x3[:, 2] != np.sin(d.astype(np.float64)).astype(np.float32)).mean()
    print("differ", wrong)
    assert wrong <= 1e-5 + 2 / batch
