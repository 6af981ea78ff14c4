"""The forward's plans and row windows at their edges, and angles beyond the table's range.

Every plan edge (256, 512, 768, 1024 and 1536 steps, and the batch sizes at which a chain takes fewer
waves), chains shorter than one vector of a row, and one-element cuts of the last vector, against the
float64 oracle on the same rounded inputs.  Bars: float32 1e-5 nm RMS and 1e-4 nm at most (the
acceptance bar at N = 2049, where 2046 roundings of 2^-24 at a 10 nm extent accumulate); half types one
rounding of a coordinate, 2^-8 (bfloat16) and 2^-11 (float16) of the largest, plus the float32 bar;
float64 1e-12.
"""

from __future__ import annotations

import re
from pathlib import Path

import numpy as np
import pytest

from oracle import nerf64 as o

SRC = Path(__file__).resolve().parent.parent / "cufk_amd" / "csrc" / "chain_ops.h"
BARS = {"float32": 0.0, "bfloat16": 2.0**-8, "float16": 2.0**-11}


def _check(device, dtype, batch, points, seed, huge=False):
    import torch

    import cufk_amd

    pick = sorted({0, batch // 2, batch - 1})
    d = o.synthetic_inputs(len(pick), points, seed=seed, anchors=True)
    if huge:  # a few angles far beyond one turn, of both signs, among ordinary ones
        rng = np.random.default_rng(seed)
        d["dihedrals"][0, rng.integers(0, points - 3, 3)] = [7.0e4, -3.0e9, 2.5e37]
        d["angles"][-1, 1 + rng.integers(0, points - 3, 2)] = [65537.5, -1.2e20]
    tdtype = getattr(torch, dtype)
    rows, rounded = {}, {}
    for k in ("lengths", "angles", "dihedrals"):
        small = torch.tensor(d[k], device=device).to(tdtype)
        rounded[k] = small.double().cpu().numpy()
        full = small[:1].expand(batch, -1).clone()
        full[pick] = small
        rows[k] = full
    an = {k: torch.tensor(d[k], device=device).to(tdtype) for k in ("p0", "first_direction", "initial_normal")}
    got = cufk_amd.reconstruct(*rows.values(), *an.values())[pick].double().cpu().numpy()
    want = o.reconstruct_forward(*rounded.values(), **{k: v.double().cpu().numpy() for k, v in an.items()})
    err = np.abs(got - want)
    if dtype == "float64":
        assert err.max() <= 1e-12
    else:
        rounding = BARS[dtype] * np.abs(want).max()
        assert np.sqrt((err**2).sum(-1).mean(-1)).max() <= 1e-5 + rounding and err.max() <= 1e-4 + rounding


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", ["float32", "bfloat16", "float16", "float64"])
@pytest.mark.parametrize("steps", [1, 2, 3, 4, 5, 8, 255, 256, 257, 512, 513, 514, 768, 769, 1024, 1025, 1536, 1537, 2048])
def test_plan_edges_small_batches(device, dtype, steps):
    _check(device, dtype, 3, steps + 3, seed=steps)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", ["float32", "bfloat16", "float16"])
@pytest.mark.parametrize("batch,steps", [(2048, 300), (2049, 300), (2049, 511), (2048, 520), (2049, 520), (2049, 765),
                                         (2049, 768), (1024, 800), (1025, 801), (2049, 1023)])
def test_plan_edges_large_batches(device, dtype, batch, steps):
    _check(device, dtype, batch, steps + 3, seed=steps)


@pytest.mark.gpu
@pytest.mark.parametrize("batch,steps", [(2, 100), (2, 400), (2049, 400), (2049, 700), (2, 900), (2, 2046)])
def test_huge_angles(device, batch, steps):
    _check(device, "float32", batch, steps + 3, seed=7, huge=True)


def test_huge_reduction_constants_and_steps():
    """reduce_huge's words are the bits of 1/(2 pi), and its integer steps give x mod one 64th of a
    half turn to 1e-17."""
    from mpmath import floor, mp, mpf, nint, pi

    text = SRC.read_text()
    words = [int(w, 16) for w in re.findall(r"0x([0-9a-f]{8})u", re.search(r"kInverseTurn\[\] = \{0u, (.*?)\};", text).group(1))]
    scale = float(re.search(r"static_cast<double>\(rest\) \* (\S+);", text).group(1))
    mp.prec = 600
    assert words == [int(floor(mpf(2) ** (32 * (i + 1)) / (2 * pi))) & 0xFFFFFFFF for i in range(len(words))]
    assert scale == float(2 * pi / mpf(2) ** 64)
    table = [0, *words]
    rng = np.random.default_rng(0)
    xs = np.concatenate([2.0 ** rng.uniform(16.0, 127.9, 300), [65536.5, 3.4028235e38]]).astype(np.float32)
    for x in xs:
        bits = int(x.view(np.uint32))
        exponent, m = bits >> 23, (bits & 0x7FFFFF) | 0x800000
        at = min(exponent, 254) - 150 + 32
        w, sh = table[at >> 5:], at & 31
        word = lambda i: (((w[i] << 32 | w[i + 1]) << sh) >> 32) & 0xFFFFFFFF  # noqa: E731,B023
        turn = (m * (word(0) << 64 | word(1) << 32 | word(2)) >> 32) & (2**64 - 1)
        k = (turn + 2**56) % 2**64 >> 57
        rest = (turn - (k << 57) + 2**63) % 2**64 - 2**63
        exact = mpf(float(x)) * 64 / pi
        want = (exact - nint(exact)) * pi / 64
        assert k == int(nint(exact)) % 128 and abs(rest * scale - want) < 1e-17, x
