"""What the scan ops refuse and accept: the quick acceptance check must say no
to every input that the explaining check raises for, and strided, bf16-gated or
non-contiguous inputs must give the plain call's bits."""
from __future__ import annotations

import pytest
import torch

import dflash_mlx
from dflash_mlx.gated_delta import _accepts, _explain_scan_inputs

pytestmark = pytest.mark.gpu


def _good(device):
    g = torch.Generator(device=device).manual_seed(0)
    r = lambda *s: torch.randn(*s, generator=g, device=device)  # noqa: E731
    B, T, Hk, Hv, D = 2, 3, 2, 4, 64
    return dict(q=(0.1 * r(B, T, Hk, D)).bfloat16(), k=(0.1 * r(B, T, Hk, D)).bfloat16(),
                v=r(B, T, Hv, D).bfloat16(), g=torch.sigmoid(r(B, T, Hv)),
                beta=torch.sigmoid(r(B, T, Hv)), state=r(B, Hv, D, D))


@pytest.mark.parametrize("name,change,error", [
    ("q", lambda t: t[:, :2], ValueError), ("q", lambda t: t.float(), TypeError),
    ("q", lambda t: t.cpu(), ValueError), ("k", lambda t: t[0], ValueError),
    ("k", lambda t: t.half(), TypeError), ("k", lambda t: t.cpu(), ValueError),
    ("v", lambda t: t[:1], ValueError), ("v", lambda t: t[:, :, :3], ValueError),
    ("v", lambda t: t.float(), TypeError), ("g", lambda t: t[..., :2], ValueError),
    ("g", lambda t: t.cpu(), ValueError), ("beta", lambda t: t[:, :1], ValueError),
    ("beta", lambda t: t.cpu(), ValueError), ("state", lambda t: t[:, :2], ValueError),
    ("state", lambda t: t.cpu(), ValueError), ("state", lambda t: t.double(), TypeError)])
def test_refused(device, name, change, error):
    x = _good(device)
    assert _accepts(**x)
    x[name] = change(x[name])
    if not (name == "state" and error is TypeError):  # its dtype is checked later
        assert not _accepts(**x)
        with pytest.raises(error):
            _explain_scan_inputs(**x)
    with pytest.raises(error):
        dflash_mlx.gated_delta_kernel(**x)


def test_accepted_forms(device):
    x = _good(device)
    want = dflash_mlx.gated_delta_verify(**x)
    y = dict(x)
    for n in ("q", "k", "v"):  # innermost dimension not unit-stride
        y[n] = x[n].transpose(2, 3).contiguous().transpose(2, 3)
    y["g"] = x["g"].transpose(1, 2).contiguous().transpose(1, 2)
    y["state"] = x["state"].transpose(2, 3).contiguous().transpose(2, 3)
    for a, b in zip(dflash_mlx.gated_delta_verify(**y), want):
        assert torch.equal(a, b)
    z = dict(x, beta=x["beta"].bfloat16())
    w = dict(x, beta=x["beta"].bfloat16().float())
    for a, b in zip(dflash_mlx.gated_delta_verify(**z), dflash_mlx.gated_delta_verify(**w)):
        assert torch.equal(a, b)


def test_current_stream_is_used(device):
    """A call under a side stream runs on it (after the work queued there)."""
    x = _good(device)
    want = dflash_mlx.gated_delta_verify(**x)
    torch.cuda.synchronize()
    s = torch.cuda.Stream(device)
    state = torch.full_like(x["state"], float("nan"))
    big = torch.randn(4096, 4096, device=device)
    torch.cuda.synchronize()
    with torch.cuda.stream(s):
        for _ in range(20):
            big = big @ big * 1e-3
        state.copy_(x["state"])  # behind the products; another stream would read NaN
        got = dflash_mlx.gated_delta_verify(**dict(x, state=state))
    s.synchronize()
    for a, b in zip(got, want):
        assert torch.equal(a, b)
