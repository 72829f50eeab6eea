"""Cache entries put into a hybrid target's cache from outside, as the next
forward takes them: the windows and states of every gated-delta layer equal
their entries, whatever form those have, and nothing is kept of the last block.
A block of 20 tokens then gives the bits of a cache that held them all along."""
from __future__ import annotations

import pytest
import torch

from dflash_mlx.gdn_layer import GatedDeltaConfig
from dflash_mlx.hybrid_model import HybridConfig, HybridWeights
from dflash_mlx.target import HybridTargetModel

pytestmark = pytest.mark.gpu

CFG = HybridConfig(hidden_size=256, num_hidden_layers=4, intermediate_size=512, vocab_size=1024,
                   num_attention_heads=4, num_key_value_heads=1, head_dim=128,
                   linear=GatedDeltaConfig(linear_num_key_heads=2, linear_num_value_heads=4))


def _strided(t):
    return t.transpose(1, 2).contiguous().transpose(1, 2)


def _misaligned(t):
    buf = torch.empty(t.numel() + 1, dtype=t.dtype, device=t.device)
    out = buf[1:].view(t.shape)
    out.copy_(t)
    return out


@pytest.fixture(scope="module")
def model(device):
    return HybridTargetModel(CFG, HybridWeights.random(CFG, device, seed=5, on_device=False), device,
                             max_seq_len=256, block_size=16)


@pytest.mark.parametrize("form", ["plain", "some", "strided", "misaligned", "bf16", "none", "given on", "mixed"])
def test_entries(model, device, form):
    toks = torch.randint(0, CFG.vocab_size, (1, 60), generator=torch.Generator().manual_seed(6),
                         dtype=torch.int32).to(device)
    cache = model.make_cache()
    model.forward_dflash(toks[:, :40], cache, [])
    snap = model.snapshot_linear_caches(cache)
    model.forward_dflash(toks[:, 40:52], cache, [])  # a block: its tape and keep counts stay behind
    lin = cache.linear_idx
    for i in (lin[1:2] if form == "some" else lin):
        conv, state = snap[i]
        if form == "mixed":  # the types of windows and states differ from layer to layer
            conv, state = (conv.float(), state.bfloat16()) if i == lin[1] else (conv, state)
        change = {"strided": _strided, "misaligned": _misaligned,
                  "bf16": lambda t: t.bfloat16(), "none": lambda t: None}.get(form, lambda t: t)
        cache[i][0], cache[i][1] = change(conv), change(state)
    if form == "given on":  # the first layer's buffers as the second layer's entry
        cache[lin[1]][0], cache[lin[1]][1] = cache.runner.conv[0], cache.runner.state[0]
    # what plain copies in layer order give
    run = cache.runner
    want = []
    for j, bufs in ((0, run.conv), (1, run.state)):
        now = [b.clone() for b in bufs]
        for gi, i in enumerate(lin):
            e = cache[i][j]
            own = next((k for k, b in enumerate(bufs) if e is not None and e.data_ptr() == b.data_ptr()), None)
            now[gi] = (torch.zeros_like(now[gi]) if e is None else now[own].clone() if own is not None
                       else e.reshape(now[gi].shape).to(now[gi].dtype))
        want.append([t.clone() for t in now])
    model._sync_in(cache, 1)
    torch.cuda.synchronize()
    for bufs, ref in zip((run.conv, run.state), want):
        for b, r in zip(bufs, ref):
            assert torch.equal(b, r)
    assert run.keep.tolist() == [0]
    other = model.make_cache()
    for gi, i in enumerate(lin):
        other[i][0], other[i][1] = want[0][gi], want[1][gi]
    for kv, src in zip((other[i] for i in other.attn_idx), (cache[i] for i in cache.attn_idx)):
        kv.offset = src.offset
    for a, b in zip(other.runner.k_cache + other.runner.vt_cache, run.k_cache + run.vt_cache):
        a.copy_(b)
    for a, b in zip(model.forward_dflash(toks[:, :20], cache, [1, 3]),
                    model.forward_dflash(toks[:, :20], other, [1, 3])):
        assert torch.equal(a, b)
    for a, b in zip(lin, other.linear_idx):
        assert torch.equal(cache[a][0], other[b][0]) and torch.equal(cache[a][1], other[b][1])
