"""Host side of the prompt pass (CPU tensors, no kernel runs): which token and
output tensors its kernels are given as they are, and which go through the
pass's own buffers, whose copies refuse a shape that does not fit."""
from __future__ import annotations

from types import SimpleNamespace

import pytest
import torch

from dflash_mlx import prefill
from dflash_mlx.gdn_layer import GatedDeltaConfig
from dflash_mlx.prefill import HybridPrefill

P, H = 6, 8


@pytest.fixture
def calls(monkeypatch):
    seen = []
    monkeypatch.setattr(prefill._lib, "call", lambda fn, *args: seen.append((fn, args)))
    return seen


def _pass():
    """A pass over no layers: embedding + norm, then the outputs' hand-over."""
    pre = HybridPrefill.__new__(HybridPrefill)
    pre.cfg = SimpleNamespace(hidden_size=H, intermediate_size=16, num_hidden_layers=0, vocab_size=32,
                              num_attention_heads=1, num_key_value_heads=1, head_dim=128,
                              attn_proj_rows=512, rms_norm_eps=1e-6, linear=GatedDeltaConfig())
    one = torch.zeros(H)
    pre.run = SimpleNamespace(device=torch.device("cpu"), capture_layers=(), keep=torch.zeros(1),
                              w=SimpleNamespace(embed=one, layers=[{"ln_in": one}], final_norm=one))
    pre.w, pre.rows_cap, pre.in_stride = [], 16, 16
    pre.tokens = torch.full((16,), -1, dtype=torch.int32)
    pre.proj = pre.act = torch.zeros(16)
    pre.h, pre.xn = torch.zeros(16, H), torch.arange(16 * H).view(16, H).bfloat16()
    return pre


TOKENS = torch.arange(P, dtype=torch.int32)


@pytest.mark.parametrize("tokens,as_is", [
    (TOKENS, True), (TOKENS.long(), False), (torch.arange(2 * P, dtype=torch.int32)[::2], False)])
def test_tokens(calls, tokens, as_is):
    pre = _pass()
    pre._pass(tokens, P, None, torch.empty(P, H, dtype=torch.bfloat16), None)
    assert calls[0][0] == "dflash_embed_rmsnorm"
    assert calls[0][1][1] == (tokens if as_is else pre.tokens).data_ptr()
    if not as_is:
        assert torch.equal(pre.tokens[:P].long(), tokens.long())


@pytest.mark.parametrize("tokens", [TOKENS[None], TOKENS[:, None], TOKENS[:P - 1], TOKENS[:0]])
def test_tokens_of_another_shape_are_refused(calls, tokens):
    with pytest.raises(RuntimeError):
        _pass()._pass(tokens, P, None, torch.empty(P, H, dtype=torch.bfloat16), None)
    assert not calls


@pytest.mark.parametrize("out", [
    torch.empty(P - 1, H, dtype=torch.bfloat16), torch.empty(P, H - 1, dtype=torch.bfloat16),
    torch.empty(P * H, dtype=torch.bfloat16), torch.empty(1, H, dtype=torch.bfloat16)])
def test_outputs_of_another_shape_are_refused(calls, out):
    with pytest.raises(RuntimeError):
        _pass()._pass(TOKENS, P, None, out, None)


@pytest.mark.parametrize("out", [
    torch.empty(P, H), torch.empty(P, 2 * H, dtype=torch.bfloat16)[:, ::2],
    torch.empty(P * H + 1, dtype=torch.bfloat16)[1:].view(P, H)])
def test_outputs_of_another_layout_get_a_copy(calls, out):
    pre = _pass()
    pre._pass(TOKENS, P, None, out, None)
    assert torch.equal(out.float(), pre.xn[:P].float())
