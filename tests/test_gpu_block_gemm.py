"""GPU parity of the block GEMMs (16 < M <= 128 rows over fragment-tiled
weights) against an fp32 torch product of the same bf16 inputs.

Bounds: a bf16 output within one rounding of the reference (2^-8 |ref|) plus
1e-3 of its rms for fp32 sums in another order; the gated output within two
roundings (silu of an fp32 product, then one rounding); fp32 partials summed
within 1e-4 of the rms.  Sizes: both sides of every column-tile count (16-row
steps up to 128), weight tiles cut short (N not a multiple of 64 or 96, N = 16),
K of one k-step (three idle waves), of odd quarters and of every turn remainder,
activation rows further apart than K, split ranges with idle waves; more than
64 rows on 4 row tiles at 4, 5 and 7 k-steps a wave (one activation step in
flight), 8 with a last wave of 7, and 8 (two in flight).
"""
from __future__ import annotations

import pytest
import torch

from dflash_mlx import _lib
from dflash_mlx import prefill as pf
from dflash_mlx.gdn_layer import GatedDeltaConfig
from dflash_mlx.hybrid_model import HybridConfig, HybridVerifyRunner, HybridWeights
from dflash_mlx.prefill import HybridPrefill
from dflash_mlx.runtime import lm_head_greedy_accept, tile_weight

pytestmark = pytest.mark.gpu


def _block(device, x, wt, out, part, nsplit, M, N, K, swiglu=0):
    _lib.call("dflash_gemm_bf16_tiled_block", x.data_ptr(), x.stride(0), wt.data_ptr(),
              _lib.ptr(out), 0 if out is None else out.stride(0), _lib.ptr(part), nsplit, M, N, K,
              swiglu, _lib.stream_handle(device))
    torch.cuda.synchronize()


@pytest.mark.parametrize("M,N,K,nsplit,pad", [
    (17, 16, 64, 0, 0), (32, 272, 128, 0, 8), (33, 1040, 320, 0, 0), (48, 96, 192, 0, 0),
    (49, 4112, 576, 0, 64), (64, 12352, 2560, 0, 0), (65, 160, 1088, 0, 0), (96, 5120, 640, 0, 0),
    (97, 18432, 448, 0, 0), (128, 2576, 2560, 0, 16), (1, 48, 64, 0, 0), (128, 2560, 9216, 6, 0),
    (65, 2560, 4096, 6, 0), (31, 80, 320, 4, 0), (100, 16, 64, 3, 0),
    (97, 12352, 1024, 0, 0), (128, 12352, 1088, 0, 8), (81, 12352, 1280, 0, 0),
    (97, 12352, 1792, 0, 0), (128, 12352, 1984, 0, 8), (81, 12352, 2048, 0, 0)])
def test_block_gemm(device, M, N, K, nsplit, pad):
    print(f"[block gemm] M={M} N={N} K={K} nsplit={nsplit} pad={pad}", flush=True)
    g = torch.Generator(device=device).manual_seed(M + 3 * N + K)
    x = torch.randn(M, K + pad, generator=g, device=device).bfloat16()[:, :K]
    w = (0.02 * torch.randn(N, K, generator=g, device=device)).bfloat16()
    ref = x.float() @ w.float().t()
    scale = ref.pow(2).mean().sqrt().item()
    if nsplit:
        used = int(_lib.load().dflash_gemm_splits(K, nsplit))
        part = torch.full((used, M, N), float("nan"), device=device)
        _block(device, x, tile_weight(w), None, part, nsplit, M, N, K)
        assert (part.sum(0) - ref).abs().max().item() <= 1e-4 * scale + 1e-5
    else:
        out = torch.full((M, N + 8), float("nan"), device=device).bfloat16()
        _block(device, x, tile_weight(w), out, None, 0, M, N, K)
        err = ((out[:, :N].float() - ref).abs() - 2 ** -8 * ref.abs()).max().item()
        assert err <= 1e-3 * scale, err
        assert torch.isnan(out[:, N:].float()).all()  # nothing past the row


@pytest.mark.parametrize("M,I,K", [(20, 16, 64), (64, 9216, 2560), (113, 528, 704), (128, 48, 128)])
def test_block_gemm_swiglu(device, M, I, K):
    print(f"[block gemm swiglu] M={M} I={I} K={K}", flush=True)
    g = torch.Generator(device=device).manual_seed(M + I + K)
    x = torch.randn(M, K, generator=g, device=device).bfloat16()
    w = (0.05 * torch.randn(2 * I, K, generator=g, device=device)).bfloat16()
    pairs = w.view(2, I // 16, 16, K).transpose(0, 1).reshape(2 * I, K).contiguous()
    out = torch.full((M, I), float("nan"), device=device).bfloat16()
    _block(device, x, tile_weight(pairs), out, None, 0, M, 2 * I, K, 1)
    gu = x.float() @ w.float().t()
    ref = torch.nn.functional.silu(gu[:, :I]) * gu[:, I:]
    err = ((out.float() - ref).abs() - 2 ** -7 * ref.abs()).max().item()
    assert err <= 1e-3 * ref.pow(2).mean().sqrt().item()


@pytest.mark.parametrize("B,N,V,H", [(1, 17, 16, 64), (2, 16, 1040, 192), (3, 11, 4112, 640),
                                     (4, 16, 2576, 2560), (7, 7, 128, 128)])
def test_lm_head_block_rows(device, B, N, V, H):
    """17 to 64 hidden rows over the tiled head: the planted winner of each row
    (a margin far above the sums' rounding), the vocabulary's last tile cut
    short, and no index past V."""
    g = torch.Generator(device=device).manual_seed(V + H)
    w = (0.02 * torch.randn(V, H, generator=g, device=device)).bfloat16()
    win = torch.randint(0, V, (B, N), generator=g, device=device)
    win[0, 0], win[-1, -1] = V - 1, 0
    hidden = (torch.randn(B, N, H, generator=g, device=device) * 0.1 + 50 * w[win].float()).bfloat16()
    want = (hidden.double().reshape(-1, H) @ w.double().t()).argmax(-1).view(B, N)
    post, matched, bonus = lm_head_greedy_accept(hidden, w, win.int()[:, 1:], weight_tiled=tile_weight(w))
    assert torch.equal(post.long(), want)
    lead = (want[:, :-1] == win[:, 1:]).int().cumprod(1).sum(1).int()
    assert torch.equal(matched, lead)
    assert torch.equal(bonus.long(), want.gather(1, lead.long()[:, None])[:, 0])


def test_block_gemm_refuses(device):
    f = _lib.load().dflash_gemm_bf16_tiled_block
    d = torch.zeros(1 << 16, dtype=torch.bfloat16, device=device).data_ptr()
    st = _lib.stream_handle(device)
    assert f(d, 64, d, d, 64, None, 0, 129, 64, 64, 0, st) == -2   # rows
    assert f(d, 64, d, d, 64, None, 0, 32, 40, 64, 0, st) == -2    # N % 16
    assert f(d, 64, d, d, 64, None, 0, 32, 48, 64, 1, st) == -2    # gated N % 32
    assert f(d, 64, d, d, 64, None, 0, 32, 64, 96, 0, st) == -2    # K % 64
    assert f(d, 32, d, d, 64, None, 0, 32, 64, 64, 0, st) == -2    # row stride
    assert f(d, 64, d, None, 0, None, 4, 32, 64, 64, 0, st) == -1  # no partials
    assert f(d + 2, 64, d, d, 64, None, 0, 32, 64, 64, 0, st) == -4
    assert f(d, 64, d, d, 64, None, 0, 0, 64, 64, 0, st) == 0


def test_short_prompt_after_a_long_one(device):
    """A 40-row pass gives the same bits in fresh buffers and in those of a
    300-row pass before it (its K splits do not depend on what ran before)."""
    cfg = HybridConfig(hidden_size=256, num_hidden_layers=4, intermediate_size=512, vocab_size=1024,
                       num_attention_heads=4, num_key_value_heads=1, head_dim=128,
                       linear=GatedDeltaConfig(linear_num_key_heads=2, linear_num_value_heads=4))
    w = HybridWeights.random(cfg, device, seed=23, on_device=False)
    toks = torch.randint(0, cfg.vocab_size, (300,), generator=torch.Generator().manual_seed(1),
                         dtype=torch.int32).to(device)
    outs = []
    for first in (0, 300):
        run = HybridVerifyRunner(cfg, w, 1, 16, 512, device)
        pre = HybridPrefill(run)
        out = torch.empty(300, cfg.hidden_size, dtype=torch.bfloat16, device=device)
        if first:
            pre._ensure(first)
        pre.forward(toks[:40], out[:40], None)
        torch.cuda.synchronize()
        outs.append(out[:40].cpu())
    assert torch.isfinite(outs[0].float()).all()
    assert torch.equal(*outs)


@pytest.mark.parametrize("kind,N,K", [("gate", 33024, 128), ("plain", 33040, 192), ("residual", 5120, 15616),
                                      ("residual", 5120, 640)])
@pytest.mark.parametrize("side", [0, 1])
def test_block_and_tile_routes_of_the_prompt_pass(device, monkeypatch, kind, N, K, side):
    """A prompt's projection on both sides of the row count where its route
    changes: the planned kernels, and an fp32 product."""
    cus = torch.cuda.get_device_properties(device).multi_processor_count
    P = pf.block_rows(kind == "residual", N, K, cus) + side
    if cus == 256:
        assert P - side == (128 if K == 640 else 96 if kind == "residual" else 80)
    print(f"[prompt routes] {kind} N={N} K={K} P={P}", flush=True)
    g = torch.Generator(device=device).manual_seed(N + P)
    x = torch.randn(P, K, generator=g, device=device).bfloat16()
    w = (0.05 * torch.randn(N, K, generator=g, device=device)).bfloat16()
    ref = x.float() @ w.float().t()
    pre = HybridPrefill.__new__(HybridPrefill)
    pre.cus, pre.cfg = cus, HybridConfig(hidden_size=N)
    pre.r = torch.full((P, N), float("nan"), dtype=torch.bfloat16, device=device)
    floats = pf.partial_floats(kind == "residual", N, K, P, cus)
    pre.part = torch.full((max(floats, 4),), float("nan"), device=device)
    paired = w.view(2, N // 32, 16, K).transpose(0, 1).reshape(N, K).contiguous() if kind == "gate" else w
    weight = (tile_weight(paired), N)
    calls, real = [], _lib.call
    monkeypatch.setattr(pf._lib, "call", lambda fn, *a: (calls.append(fn), real(fn, *a)))
    st = _lib.stream_handle(device)
    if kind == "residual":
        used = pre._to_residual(weight, x.data_ptr(), K, P, st)
        got = pre.part[:used * P * N].view(used, P, N).sum(0) if used else pre.r.float()
    else:
        got = torch.full((P, N // 2 if kind == "gate" else N), float("nan"), dtype=torch.bfloat16, device=device)
        pre._bf16_proj(weight, x.data_ptr(), K, P, got.data_ptr(), got.shape[1], kind == "gate", st)
        got = got.float()
        if kind == "gate":
            ref = torch.nn.functional.silu(ref[:, :N // 2]) * ref[:, N // 2:]
    torch.cuda.synchronize()
    assert (calls[0] == "dflash_gemm_bf16_tiled_block") == (side == 0), calls
    scale = ref.pow(2).mean().sqrt().item()
    err = ((got - ref).abs() - 2 ** -7 * ref.abs()).max().item()  # two bf16 roundings
    assert err <= 1e-3 * scale, err


@pytest.fixture(scope="module")
def far(device):
    """(hidden rows, the same rows packed): 49 rows of 128 more than 2^28 elements
    apart, past the block kernels' 32-bit offsets."""
    stride, g = (1 << 28) + 8, torch.Generator(device=device).manual_seed(17)
    x = torch.randn(49, 128, generator=g, device=device).bfloat16()
    apart = torch.empty(48 * stride + 128, dtype=torch.bfloat16, device=device)
    apart = apart.as_strided((49, 128), (stride, 1))
    apart.copy_(x)
    yield apart, x
    del apart
    torch.cuda.empty_cache()


@pytest.mark.parametrize("M,nsplit", [(17, 1), (49, 1), (33, 2)])
def test_rows_far_apart(device, far, M, nsplit):
    """The verify projections' bits do not depend on the rows' distance."""
    N, K = 1040, 128
    g = torch.Generator(device=device).manual_seed(M)
    wt = tile_weight((0.05 * torch.randn(N, K, generator=g, device=device)).bfloat16())
    outs = []
    for x in far:
        out = torch.full((nsplit, M, N), float("nan"), dtype=torch.float32 if nsplit > 1 else torch.bfloat16,
                         device=device)
        _lib.call("dflash_gemm_bf16_tiled", x.data_ptr(), x.stride(0), wt.data_ptr(), out.data_ptr(), N, M,
                  N, K, nsplit, 32, 4, None, 0, _lib.stream_handle(device))
        outs.append(out)
    gated = []
    for x in far:
        out = torch.full((M, 512), float("nan"), dtype=torch.bfloat16, device=device)
        _lib.call("dflash_gemm_bf16_swiglu_tiled", x.data_ptr(), x.stride(0), wt.data_ptr(), out.data_ptr(),
                  512, M, 1024, K, 4, None, 0, _lib.stream_handle(device))
        gated.append(out)
    torch.cuda.synchronize()
    for a, b in (outs, gated):
        assert not torch.isnan(b.float()).any()
        assert torch.equal(a, b)


def test_lm_head_rows_far_apart(device, far):
    V, H = 1040, 128
    g = torch.Generator(device=device).manual_seed(1)
    w = (0.05 * torch.randn(V, H, generator=g, device=device)).bfloat16()
    win = torch.randint(0, V, (49,), generator=g, device=device)
    for x in far:
        x.copy_((0.1 * far[1].float() + 50 * w[win].float()).bfloat16())
        post, _, _ = lm_head_greedy_accept(x.unsqueeze(0), w, win[None, 1:].int(), weight_tiled=tile_weight(w))
        assert torch.equal(post[0].long(), win)


def test_more_weight_rows_than_the_block_kernel_s_offsets(device):
    N, K, M = (1 << 24) + 16, 64, 17
    g = torch.Generator(device=device).manual_seed(5)
    w = torch.randn(N, K, generator=g, device=device, dtype=torch.bfloat16)
    x = torch.randn(M, K, generator=g, device=device).bfloat16()
    out = torch.empty(M, N, dtype=torch.bfloat16, device=device)
    wt = tile_weight(w)
    _lib.call("dflash_gemm_bf16_tiled", x.data_ptr(), K, wt.data_ptr(), out.data_ptr(), N, M, N, K, 1, 32,
              4, None, 0, _lib.stream_handle(device))
    for cols in (slice(0, 4096), slice(N - 4096, N)):  # the first and last weight rows, by the block kernel
        part = torch.empty(M, 4096, dtype=torch.bfloat16, device=device)
        _block(device, x, tile_weight(w[cols].contiguous()), part, None, 0, M, 4096, K)
        assert torch.equal(out[:, cols], part)


@pytest.fixture(scope="module")
def wide(device):
    cfg = HybridConfig(num_hidden_layers=4, vocab_size=1024)
    return cfg, HybridWeights.random(cfg, device, seed=29, on_device=True)


@pytest.mark.parametrize("first,rows", [(6144, 300), (777, 250), (3000, 1000), (6144, 128)])
def test_prompt_after_a_longer_one(device, wide, first, rows):
    """The same at the 4B target's widths, for prompts whose plans split K in
    other ways (300: 8 ways and 4) than the longer one's before it."""
    cfg, w = wide
    print(f"[prompt order] {rows} rows after {first}", flush=True)
    toks = torch.randint(0, cfg.vocab_size, (rows,), generator=torch.Generator().manual_seed(2),
                         dtype=torch.int32).to(device)
    outs = []
    for cap in (0, first):
        pre = HybridPrefill(HybridVerifyRunner(cfg, w, 1, 16, 1024, device))
        if cap:
            pre._ensure(cap)
        out = torch.empty(rows, cfg.hidden_size, dtype=torch.bfloat16, device=device)
        pre.forward(toks, out, None)
        torch.cuda.synchronize()
        outs.append(out.cpu())
    assert torch.isfinite(outs[0].float()).all()
    assert torch.equal(*outs)
