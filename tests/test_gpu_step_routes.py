"""The verify step of several sequences on the GPU: which launches its plan
holds, and its results against the CPU oracle of the whole step
(oracle/hybrid_oracle.model_step), with the bounds of test_gpu_hybrid.py.

Three and four sequences of 4 and of 32 value heads (below and above one scan
workgroup a compute unit: prologue inside the scan, or a launch of its own),
48 and 64 rows (projections on the block GEMMs; LM head on the tiled kernel up to
48 rows and the block form above), ragged lengths."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from dflash_mlx.gdn_layer import GatedDeltaConfig
from dflash_mlx.hybrid_model import HybridConfig, HybridVerifyRunner, HybridWeights, fuse_prologue
from oracle import hybrid_oracle as ho
from oracle import oracle as gdn_oracle
from tests.test_gpu_hybrid import _initial_state, _logits, _np, _np_weights, _runner

pytestmark = pytest.mark.gpu


def _cfg(hk, hv):
    return HybridConfig(hidden_size=256, num_hidden_layers=4, intermediate_size=512, vocab_size=1024,
                        num_attention_heads=4, num_key_value_heads=1, head_dim=128,
                        linear=GatedDeltaConfig(linear_num_key_heads=hk, linear_num_value_heads=hv))


def _cus(device):
    return torch.cuda.get_device_properties(device).multi_processor_count


@pytest.mark.parametrize("B,T,hk,hv", [(3, 16, 2, 4), (4, 16, 2, 4), (3, 16, 16, 32), (4, 16, 16, 32)])
def test_step_of_several_sequences_matches_oracle(device, B, T, hk, hv):
    cfg, Smax = _cfg(hk, hv), 256
    w = HybridWeights.random(cfg, device, seed=51, on_device=False)
    st = _initial_state(cfg, B, [20, 100, 1, 63][:B], seed=52)
    tokens = torch.randint(0, cfg.vocab_size, (B, T), generator=torch.Generator().manual_seed(53),
                           dtype=torch.int32)
    run = _runner(cfg, w, st, B, T, Smax, device)
    names = [fn for fn, _ in run._plan(T).fwd]
    fused = fuse_prologue(B, hv, 128, _cus(device))
    assert fused == (hv == 4) and run.fused_prologue == fused
    assert names.count("dflash_gdn_prologue_scan_rollback") == (3 if fused else 0)
    assert names.count("dflash_gdn_prologue") == (0 if fused else 3)
    assert "dflash_gemm_bf16_swiglu_tiled" in names and "dflash_gemm_bf16_tiled_residual_norm" not in names
    assert run._plan(T).lm[0] == "dflash_lm_head_greedy_accept_tiled"
    print(f"[step routes] B={B} T={T} Hv={hv}", flush=True)
    run.tokens.copy_(tokens)
    run.forward_accept()
    torch.cuda.synchronize()
    o_state = dict(lens=np.array(st["lens"]), conv=[_np(c) for c in st["conv"]],
                   rec=[_np(s) for s in st["rec"]], k=[_np(k) for k in st["k"]],
                   v=[_np(v) for v in st["v"]])
    ref = ho.model_step(cfg, _np_weights(w), o_state, tokens.numpy(), cfg.rms_norm_eps)
    rel = lambda a, b: np.max(np.abs(a - b)) / np.max(np.abs(b))  # noqa: E731
    hid = rel(_np(run.xn).reshape(B, T, -1), ref["hidden"])
    logits = rel(_np(_logits(run)), ref["logits"])
    tape = rel(_np(run.tape[0]), ref["tape"][0])
    print(f"  hidden rel {hid:.2e}  logits rel {logits:.2e}  tape[0] rel {tape:.2e}", flush=True)
    assert hid <= 3e-2 and logits <= 3e-2 and tape <= 1e-2
    post, toks = run.posterior.cpu().numpy(), tokens.numpy()
    for b in range(B):
        m = gdn_oracle.longest_prefix_match(toks[b, 1:], post[b, :-1])
        assert int(run.matched[b]) == m and int(run.bonus[b]) == post[b, m]
    srt = np.sort(ref["logits"], axis=-1)
    clear = (srt[..., -1] - srt[..., -2]) > 0.1 * np.max(np.abs(ref["logits"]))
    assert clear.any() and np.array_equal(post[clear], ref["posterior"][clear])


@pytest.mark.parametrize("B,hk,hv", [(1, 16, 32), (2, 8, 16), (4, 8, 8), (2, 16, 32), (1, 16, 64), (2, 16, 48)])
def test_prologue_rule_counts_workgroups(device, B, hk, hv):
    """The scan computes its prologue while each of its workgroups (8 a value
    head) has a compute unit of its own; asked not to, it never does."""
    cfg = _cfg(hk, hv)
    w = HybridWeights.random(cfg, device, seed=3, on_device=True)
    for asked in (True, False):
        run = HybridVerifyRunner(cfg, w, B, 4, 64, device, fused_prologue=asked)
        want = asked and B * hv * 8 <= _cus(device)
        names = [fn for fn, _ in run._plan(4).fwd]
        assert run.fused_prologue == want
        assert ("dflash_gdn_prologue_scan_rollback" in names) == want
        assert ("dflash_gdn_prologue" in names) != want
