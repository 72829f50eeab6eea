"""How far the prompt attention is from 64 bits, where one key holds much of a
row's weight.

A bf16 value is rounded by an ulp of 2^-7 times its power of two: rms 2^-7 /
sqrt(12), over a mean square of about 1.5^2 in [1, 2) 1.6e-3 relative.  The output's
rounding alone is that.  A weight near 1 that is rounded too adds as much again in
quadrature (2.2e-3); with the row's maximum as the softmax's reference the heaviest
weight is 1 exactly and only the others' share is added.  The bound of 1.95e-3 lies
between the two: sqrt(1.6^2 + 1.1^2).  In the second case the scores grow along the
keys, so that every row's maximum moves many times."""
from __future__ import annotations

import pytest
import torch

from tests.test_gpu_attn_prefill import D, _run_prefill

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("Hq,Hkv", [(8, 2), (6, 2), (4, 2), (4, 4)])
@pytest.mark.parametrize("std,ramp", [(3.0, (1.0, 1.0)), (2.0, (0.3, 1.5))])
def test_heaviest_weight_is_not_rounded(device, Hq, Hkv, std, ramp):
    P, L0 = 256, 1024
    S, Smax = L0 + P, L0 + P
    g = torch.Generator().manual_seed(Hq)
    q = (std * torch.randn(P, Hq, D, generator=g)).bfloat16()
    keys = torch.randn(Hkv, S, D, generator=g) * torch.linspace(*ramp, S)[None, :, None]
    keys, vals = keys.bfloat16(), torch.randn(Hkv, S, D, generator=g).bfloat16()
    gates = torch.full((P, 2 * Hq * D), 30.0).bfloat16()  # sigmoid 1
    got = _run_prefill(device, q, keys, vals.transpose(1, 2).contiguous(), gates, L0, P, Hq, Hkv, Smax,
                       D ** -0.5).double().view(P, Hq, D)
    pos, rows = torch.arange(S), L0 + torch.arange(P)
    num = den = 0.0
    for h in range(Hq):
        k, v = keys[h // (Hq // Hkv)].double(), vals[h // (Hq // Hkv)].double()
        s = (q[:, h].double() @ k.t()) * D ** -0.5
        ref = torch.softmax(s.masked_fill(pos[None] > rows[:, None], float("-inf")), -1) @ v
        num += (got[:, h] - ref).pow(2).sum().item()
        den += ref.pow(2).sum().item()
    err = (num / den) ** 0.5
    print(f"[attn precision] {Hq}:{Hkv} std {std} ramp {ramp}: {err:.2e}", flush=True)
    assert err <= 1.95e-3
