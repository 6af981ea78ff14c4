"""The backward over saved rows at its edges: every plan edge, chains shorter than one vector of a row,
one-element cuts of the last vector, regular and refused (exact path) chains side by side, as the kept
flags say, with and without anchors' gradients.  Against the float64 oracle on the same rounded inputs,
relative to the chain's largest gradient.

Bars: float32 5e-5 (the suite's gradient bar at N = 2049: suffix sums of up to 2049 float moments, each
rounded at 2^-24 of the chain's extent), half types one rounding of a gradient (2^-8, 2^-11) on top,
float64 1e-9.
"""

from __future__ import annotations

import numpy as np
import pytest

from oracle import nerf64 as o
from test_gpu_parity import _abi, _flagged_forward, _shadow_forward

ROUNDING = {"float32": 0.0, "bfloat16": 2.0**-8, "float16": 2.0**-11}


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", ["float32", "bfloat16", "float16", "float64"])
@pytest.mark.parametrize("batch,steps", [(4, s) for s in (1, 2, 3, 4, 5, 7, 8, 9, 255, 256, 257, 511, 512, 513, 767, 768,
                                                         769, 1024, 1025, 1536, 1537, 2047, 2048)]
                         + [(4100, 300), (4100, 512), (2050, 520), (2050, 1021)])
def test_saved_backward_runs(device, dtype, batch, steps):
    import torch

    import cufk_amd

    tdtype = getattr(torch, dtype)
    pick = [0, 1, batch - 2, batch - 1]
    d = o.synthetic_inputs(4, steps + 3, seed=steps, anchors=True)
    straight = np.pi - 0.004 if tdtype == torch.float64 else 2.9  # sines 0.004 and 0.24, refused below 0.01 and 0.5
    d["angles"][1, steps // 2] = straight
    d["dihedrals"][3, steps - 1] = 7.0e4 if tdtype != torch.float16 else 3.0e4
    rows, rounded = {}, {}
    for k in ("lengths", "angles", "dihedrals", "grad"):
        small = torch.tensor(d[k], device=device).to(tdtype)
        rounded[k] = small.double().cpu().numpy()
        full = small[:1].expand(batch, *small.shape[1:]).clone()
        full[pick] = small
        rows[k] = full
    an = {k: torch.tensor(d[k], device=device).to(tdtype) for k in ("p0", "first_direction", "initial_normal")}
    forward = _flagged_forward if tdtype in (torch.float32, torch.float64) else _shadow_forward
    flags = forward(_abi(), *(rows[k] for k in ("lengths", "angles", "dihedrals")), tuple(an.values()))[-1]
    if flags is not None:
        assert flags[pick].cpu().tolist() == [1, 0, 1, 1]
    anchors = batch == 4 and steps % 2 == 1
    wrt = [rows[k].requires_grad_(True) for k in ("lengths", "angles", "dihedrals")]
    wrt += [v.requires_grad_(True) for v in an.values()] if anchors else []
    xyz = cufk_amd.reconstruct(*wrt[:3], *an.values(), anchor_grads=anchors)
    got = torch.autograd.grad(xyz, wrt, rows["grad"])
    frame = {k: v.detach().double().cpu().numpy() for k, v in an.items()}
    want = list(o.reconstruct_backward(*rounded.values(), **frame))
    want += list(o.anchor_gradients(*rounded.values(), **frame)) if anchors else []
    bar = 1e-9 if dtype == "float64" else 5e-5 + ROUNDING[dtype]
    for i, (a, b) in enumerate(zip(got, want, strict=True)):
        a = a.double().cpu().numpy()
        err = np.abs((a[pick] if i < 3 else a) - b).max(-1)
        assert (err <= bar * np.maximum(1.0, np.abs(b).max(-1))).all(), (i, err)
