"""Which cache entries HybridTargetModel takes into a runner and in which order
(CPU tensors and a stand-in runner without the gather launch): what one loop
over the layers, window before state, gives, and nothing at all for an entry
that does not fit."""
from __future__ import annotations

import itertools
from types import SimpleNamespace

import pytest
import torch

from dflash_mlx.cache import ArraysCache
from dflash_mlx.target import HybridTargetModel

MODEL = SimpleNamespace(max_seq_len=8, _moves=HybridTargetModel._moves,
                        _copy_in=HybridTargetModel._copy_in)


class _Cache(list):
    pass


def _cache(layers=3):
    conv = torch.arange(1.0, layers + 1).view(-1, 1, 1, 1).expand(layers, 1, 3, 4).clone()
    run = SimpleNamespace(conv=list(conv.unbind(0)), keep=torch.full((1,), 5, dtype=torch.int32),
                          state=[torch.full((1, 2, 2, 4), 10.0 + i) for i in range(layers)],
                          load_states=lambda srcs: False, Smax=64)
    cache = _Cache()
    for c, s in zip(run.conv, run.state):
        e = ArraysCache(size=2)
        e[0], e[1] = c, s
        cache.append(e)
    cache.runner, cache.linear_idx, cache.attn_idx = run, list(range(layers)), []
    cache._installed = [(e[0], e[1]) for e in cache]
    return cache


@pytest.mark.parametrize("forms", itertools.product(["keep", "none", "new", "first", "last"], repeat=3))
def test_entries_are_taken_in_layer_order(forms):
    cache = _cache()
    run = cache.runner
    for i, form in enumerate(forms):
        if form == "none":
            cache[i][0], cache[i][1] = None, None
        elif form == "new":
            cache[i][0], cache[i][1] = torch.full((1, 3, 4), -1.0 - i), torch.full((1, 2, 2, 4), -7.0 - i)
        elif form != "keep":
            j = 0 if form == "first" else 2
            cache[i][0], cache[i][1] = run.conv[j], run.state[j]
    # one loop over the layers, on copies
    now = [[b.clone() for b in bufs] for bufs in (run.conv, run.state)]
    for i, form in enumerate(forms):
        for j in range(2):
            if form == "none":
                now[j][i].zero_()
            elif form == "new":
                now[j][i].copy_(cache[i][j])
            elif form != "keep":
                now[j][i].copy_(now[j][0 if form == "first" else 2])
    HybridTargetModel._sync_in(MODEL, cache, 1)
    for bufs, want in zip((run.conv, run.state), now):
        for b, w in zip(bufs, want):
            assert torch.equal(b, w), forms
    foreign = any(f in ("none", "new") or f == "first" and i != 0 or f == "last" and i != 2
                  for i, f in enumerate(forms))
    assert int(run.keep) == (0 if foreign else 5)


@pytest.mark.parametrize("dtypes", itertools.product([torch.bfloat16, torch.float32], repeat=3))
def test_foreach_copies_hold_one_type(monkeypatch, dtypes):
    """Entries of several types: a foreach copy over mixed types has given wrong
    values on the device, so each one holds a single type."""
    cache = _cache()
    run = cache.runner
    run.conv = [c.bfloat16() for c in run.conv]
    want = []
    for i, dt in enumerate(dtypes):
        cache[i][0], cache[i][1] = torch.full((1, 3, 4), -1.5 - i, dtype=dt), torch.full((1, 2, 2, 4), -7.5 - i, dtype=dt)
        want.append((-1.5 - i, -7.5 - i))
    real = torch._foreach_copy_

    def checked(dsts, srcs):
        assert len({t.dtype for t in (*dsts, *srcs)}) == 1
        real(dsts, srcs)

    monkeypatch.setattr(torch, "_foreach_copy_", checked)
    HybridTargetModel._sync_in(MODEL, cache, 1)
    for conv, state, (c, s) in zip(run.conv, run.state, want):
        assert bool((conv == c).all()) and bool((state == s).all())


@pytest.mark.parametrize("layer", [0, 1, 2])
@pytest.mark.parametrize("which", [0, 1])
def test_refused_entry_changes_nothing(layer, which):
    """An entry of another size is refused with the runner and the cache as
    they were (what the last block kept included): put right, the cache goes on."""
    cache = _cache()
    run = cache.runner
    before = [b.clone() for b in (*run.conv, *run.state)]
    window, good = cache[0][0], cache[layer][which]
    cache[0][0] = None
    cache[layer][which] = torch.zeros(5)
    with pytest.raises(RuntimeError):
        HybridTargetModel._sync_in(MODEL, cache, 1)
    assert int(run.keep) == 5
    for b, w in zip((*run.conv, *run.state), before):
        assert torch.equal(b, w)
    cache[0][0] = window
    cache[layer][which] = good
    HybridTargetModel._sync_in(MODEL, cache, 1)
    assert int(run.keep) == 5
