"""GPU parity of the prompt attention at the edges of its tiles, against the
fp32 reference of test_gpu_attn_prefill.py.

32-row blocks (P one below, at and above; 1, 2 and 4 blocks a workgroup, the last
ones past the end), turns of 128 keys whose second half
is empty, partly visible or past the cache's end (Smax an odd multiple of 64),
1 to 4 query heads a KV head, KV head counts that do and do not divide the 8
XCDs (the two block orders), gates and outputs off 16-byte boundaries, and
scores that grow by far more than the rescale threshold from tile to tile.
Probabilities and outputs are rounded to bf16 (2^-9 relative each): 1e-2 of the
largest output covers both with the fp32 sums.
"""
from __future__ import annotations

import pytest
import torch

from dflash_mlx import _lib
from tests import test_gpu_model_ops as model_ops
from tests.test_gpu_attn_prefill import D, _make, _reference, _run_prefill

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("P,L0,Hq,Hkv,Smax", [
    (31, 0, 4, 4, 64), (32, 33, 6, 3, 128), (33, 95, 16, 4, 192), (65, 127, 15, 5, 192),
    (97, 0, 2, 1, 128), (128, 0, 8, 8, 128), (129, 191, 3, 3, 320), (160, 96, 20, 5, 256),
    (1, 300, 8, 8, 320), (33, 0, 5, 5, 64), (64, 64, 16, 8, 128), (65, 0, 6, 3, 128), (257, 70, 4, 4, 384),
    (700, 68, 16, 4, 768)])
def test_tiles(device, P, L0, Hq, Hkv, Smax):
    print(f"[attn prefill tiles] P={P} L0={L0} Hq={Hq} Hkv={Hkv} Smax={Smax}", flush=True)
    scale = D ** -0.5
    q, keys, vals, gates, kc, vt = _make(device, P, L0, Hq, Hkv, Smax, seed=P + L0)
    got = _run_prefill(device, q, kc, vt, gates, L0, P, Hq, Hkv, Smax, scale).float()
    ref = _reference(q, keys, vals, gates, L0, Hq, Hkv, scale)
    assert torch.isfinite(got).all()
    assert (got - ref).abs().max().item() <= 1e-2 * ref.abs().max().item()


def test_growing_scores(device):
    """Keys scaled up along the sequence: a row's max grows by hundreds of log2
    units over the tiles, so O is rescaled again and again."""
    P, L0, Hq, Hkv, Smax = 40, 400, 8, 2, 448
    q, keys, vals, gates, kc, vt = _make(device, P, L0, Hq, Hkv, Smax, seed=3)
    ramp = torch.linspace(0.1, 40.0, L0 + P)[None, :, None]
    keys = (keys.float() * ramp).bfloat16()
    kc[:, :L0 + P] = keys
    got = _run_prefill(device, q, kc, vt, gates, L0, P, Hq, Hkv, Smax, D ** -0.5).float()
    ref = _reference(q, keys, vals, gates, L0, Hq, Hkv, D ** -0.5)
    assert torch.isfinite(got).all()
    assert (got - ref).abs().max().item() <= 1e-2 * ref.abs().max().item()


@pytest.mark.parametrize("scale", [-0.5, 0.0, -1e-3])
def test_scale_without_a_positive_sign(device, scale):
    """Scales the softmax takes as they are: a negative one turns the order of
    the scores round, zero weighs the visible keys alike."""
    P, L0, Hq, Hkv, Smax = 45, 150, 8, 2, 256
    q, keys, vals, gates, kc, vt = _make(device, P, L0, Hq, Hkv, Smax, seed=5)
    got = _run_prefill(device, q, kc, vt, gates, L0, P, Hq, Hkv, Smax, scale).float()
    ref = _reference(q, keys, vals, gates, L0, Hq, Hkv, scale)
    assert torch.isfinite(got).all()
    assert (got - ref).abs().max().item() <= 1e-2 * ref.abs().max().item()


@pytest.mark.parametrize("gate_off,gate_pad,out_off", [(1, 0, 0), (0, 3, 0), (0, 0, 1)])
def test_unaligned_gate_and_output(device, gate_off, gate_pad, out_off):
    """Gate rows and outputs on 2-byte boundaries give the aligned call's bits."""
    P, L0, Hq, Hkv, Smax = 37, 70, 8, 2, 128
    scale = D ** -0.5
    q, keys, vals, gates, kc, vt = _make(device, P, L0, Hq, Hkv, Smax, seed=9)
    want = _run_prefill(device, q, kc, vt, gates, L0, P, Hq, Hkv, Smax, scale)
    W = gates.shape[1]
    buf = torch.zeros(P * (W + gate_pad) + 8, dtype=torch.bfloat16, device=device)
    gd = buf[gate_off:gate_off + P * (W + gate_pad)].view(P, W + gate_pad)
    gd[:, :W] = gates.to(device)
    ob = torch.full((P * Hq * D + 8,), float("nan"), dtype=torch.bfloat16, device=device)
    out = ob[out_off:out_off + P * Hq * D]
    qd, kd, vd = (t.to(device) for t in (q, kc, vt))
    lens = torch.tensor([L0], dtype=torch.int32, device=device)
    _lib.call("dflash_attn_prefill", qd.data_ptr(), kd.data_ptr(), vd.data_ptr(), lens.data_ptr(),
              gd.data_ptr(), gd.stride(0), out.data_ptr(), P, Hq, Hkv, D, Smax, scale,
              _lib.stream_handle(device))
    torch.cuda.synchronize()
    assert torch.equal(out.view(P, Hq * D).cpu(), want)
    assert torch.isnan(ob[:out_off].float()).all() and torch.isnan(ob[out_off + P * Hq * D:].float()).all()


@pytest.mark.parametrize("B,T,lens", [(1, 420, [37]), (1, 1300, [1000]), (3, 333, [7, 64, 2001]),
                                      (2, 2100, [0, 5])])
def test_prep_rows(device, B, T, lens):
    """Long inputs walk a token's heads in one wave (2 heads, 6 with a last wave
    of 2, 4, all 20): the oracle's bits, as for the short ones."""
    model_ops.test_attn_prep_norm_rope_and_cache_append(device, B, T, lens)


def test_prep_rows_outside_the_cache(device):
    """A long input that runs past the cache sets its overflow word and writes
    what fits, as calls of 32 tokens do."""
    Hq, Hkv, Smax, T, rot = 6, 3, 1024, 1100, 64
    g = torch.Generator(device=device).manual_seed(4)
    r = lambda *s: torch.randn(*s, generator=g, device=device).bfloat16()  # noqa: E731
    rows = (2 * Hq + 2 * Hkv) * D
    proj, qn, kn = r(T, rows), r(D), r(D)

    def prep(step):
        kc = torch.zeros(Hkv, Smax, D, dtype=torch.bfloat16, device=device)
        vt = torch.zeros(Hkv, D, Smax, dtype=torch.bfloat16, device=device)
        q = torch.empty(T, Hq, D, dtype=torch.bfloat16, device=device)
        over = torch.zeros(1, dtype=torch.int32, device=device)
        for t in range(0, T, step):
            n = min(step, T - t)
            lens = torch.tensor([100 + t], dtype=torch.int32, device=device)
            _lib.call("dflash_attn_prep", proj[t:].data_ptr(), rows, qn.data_ptr(), kn.data_ptr(),
                      lens.data_ptr(), kc.data_ptr(), vt.data_ptr(), q[t:].data_ptr(), over.data_ptr(),
                      1, n, Hq, Hkv, D, Smax, rot, 1e5, 1e-6, _lib.stream_handle(device))
            torch.cuda.synchronize()
        return q, kc, vt, over

    for a, b in zip(prep(T), prep(32)):
        assert torch.equal(a, b)
    assert int(prep(T)[3]) == 1
