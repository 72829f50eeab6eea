"""The prompt pass's split-K partials (host side): the buffer sized for a prompt
of some length holds what the plan of every shorter prompt writes, so that a
projection's K splits, and with them its bits, never depend on what ran before."""
from __future__ import annotations

import pytest

from dflash_mlx import prefill as pf


def _writes(residual, N, K, P, cus):
    """fp32 partials of one projection over P rows, from the plan functions."""
    nks = K // 64
    used = lambda s: -(-nks // -(-nks // min(s, nks)))  # noqa: E731  (dflash_gemm_splits)
    block = P <= pf.block_rows(residual, N, K, cus)
    if residual:
        s = pf.block_splits(N, cus, K) if block else pf.residual_splits(N, P, cus, K)
        return used(s) * P * N if s > 1 else 0
    if block:
        return 0
    s = pf.prompt_splits(N, P, cus)
    if s > 1:
        return used(s) * P * N
    tail = pf.tail_split(N, P, cus, K)
    return used(tail[1]) * P * (N - tail[0]) if tail else 0


SHAPES = [(True, 2560, 4096), (True, 2560, 2048), (True, 2560, 9216), (False, 12352, 2560),
          (False, 5120, 2560), (False, 18432, 2560), (True, 256, 512), (False, 1040, 256),
          (True, 7168, 18432), (False, 36864, 7168), (True, 64, 64)]


@pytest.mark.parametrize("cus", [256, 304, 64])
@pytest.mark.parametrize("residual,N,K", SHAPES)
def test_every_shorter_prompt_fits(residual, N, K, cus):
    writes = [0] + [_writes(residual, N, K, P, cus) for P in range(1, 8193)]
    most = 0
    sizes = {1, 16, 40, 80, 81, 97, 100, 128, 129, 300, 777, 1023, 2049, 3000, 6144, 8192}
    for P in range(1, 8193):
        most = max(most, writes[P])
        if P in sizes:
            assert pf.partial_floats(residual, N, K, P, cus) >= most, P
    # no more than a unit's 256 x 256 tile each above what is needed
    assert pf.partial_floats(residual, N, K, 8192, cus) <= max(most, 256 * 256 * cus)


@pytest.mark.parametrize("K", [64, 128, 576, 2560, 4096, 9216])
def test_splits_used_is_the_library_s(K):
    from dflash_mlx import _lib

    lib = _lib.load()
    for s in range(1, 40):
        assert pf.splits_used(K, s) == lib.dflash_gemm_splits(K, s)
