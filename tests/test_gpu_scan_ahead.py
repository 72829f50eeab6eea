"""The scan's long walks (state in and final over 72 MB, at least 4 tokens, heads
of up to 128: each workgroup loads the lines of its next items ahead) against the
same sequences in short calls: a sequence's rows depend on nothing else, so out,
final state and tape must be the same bits.  Head dims with rows of one to four
lines, more than 32 tokens, strided q / k / v rows, ragged lengths, the state-only
replay, and long walks of 3 tokens and of 256-wide heads, which load nothing
ahead."""
from __future__ import annotations

import pytest
import torch

import dflash_mlx
from dflash_mlx.gated_delta import _scan

pytestmark = pytest.mark.gpu


def _inputs(device, B, T, Hk, Hv, D, seed, strided=False):
    g = torch.Generator(device=device).manual_seed(seed)
    r = lambda *s: torch.randn(*s, generator=g, device=device)  # noqa: E731
    if strided:  # views of one [B, T, C] activation buffer
        buf = (0.1 * r(B, T, (2 * Hk + Hv) * D)).bfloat16()
        q = buf[..., :Hk * D].unflatten(-1, (Hk, D))
        k = buf[..., Hk * D:2 * Hk * D].unflatten(-1, (Hk, D))
        v = buf[..., 2 * Hk * D:].unflatten(-1, (Hv, D))
    else:
        q, k = (0.1 * r(B, T, Hk, D)).bfloat16(), (0.1 * r(B, T, Hk, D)).bfloat16()
        v = r(B, T, Hv, D).bfloat16()
    gd, beta = torch.sigmoid(r(B, T, Hv)), torch.sigmoid(r(B, T, Hv))
    return [q, k, v, gd, beta, 0.05 * r(B, Hv, D, D)]


@pytest.mark.parametrize("B,T,Hk,Hv,D,strided", [
    (19, 5, 16, 32, 128, False), (24, 4, 16, 32, 128, True), (74, 6, 16, 32, 64, False),
    (34, 5, 8, 32, 96, True), (290, 4, 16, 32, 32, False), (20, 37, 4, 32, 128, False),
    (24, 3, 16, 32, 128, True), (10, 5, 8, 16, 256, False)])
def test_long_walk_matches_short_calls(device, B, T, Hk, Hv, D, strided):
    assert B * Hv * D * D * 8 > 72 << 20
    print(f"[scan ahead] B={B} T={T} Hk={Hk} Hv={Hv} D={D}", flush=True)
    x = _inputs(device, B, T, Hk, Hv, D, seed=B + D, strided=strided)
    out, fin, tape = dflash_mlx.gated_delta_verify(*x)
    for b in range(0, B, 4):
        o, f, t = dflash_mlx.gated_delta_verify(*[y[b:b + 4] for y in x])
        assert torch.equal(out[b:b + 4], o) and torch.equal(fin[b:b + 4], f)
        assert torch.equal(tape[:, b:b + 4], t)


def test_long_walk_lengths_and_replay(device):
    B, T = 20, 6
    x = _inputs(device, B, T, 16, 32, 128, seed=4)
    lens = torch.arange(B, device=device, dtype=torch.int32) % (T + 2)
    fin = dflash_mlx.advance_gated_delta_states(x[5], x[1], x[2], x[3], x[4], lengths=lens)
    for b in range(0, B, 5):
        want = dflash_mlx.advance_gated_delta_states(x[5][b:b + 5], x[1][b:b + 5], x[2][b:b + 5],
                                                     x[3][b:b + 5], x[4][b:b + 5],
                                                     lengths=lens[b:b + 5])
        assert torch.equal(fin[b:b + 5], want)
    out, f2, _ = _scan(*x, want_out=True, want_tape=False)
    assert torch.equal(out[:4], _scan(*[y[:4] for y in x], want_out=True, want_tape=False)[0])
