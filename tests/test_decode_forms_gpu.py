"""Decode forms that a launch's size selects (early refill, non-temporal loads): a row's bits are the same in each."""
import numpy as np
import pytest
import torch

import dgx_attn as A

pytestmark = pytest.mark.gpu

TORCH = {0: torch.float32, 1: torch.float16, 2: torch.bfloat16}


def _batch(B, ML, nq, nkv, hd, kvdt, seed):
    rng = np.random.default_rng(seed)
    pos = rng.integers(0, ML, B).astype(np.int32)
    pos[0], pos[1], pos[2] = 0, 15, ML - 1                  # one key, one whole tile, every chunk
    g = torch.Generator(device="cuda").manual_seed(seed)
    Q = torch.randn(B, nq, hd, device="cuda", generator=g).to(TORCH[kvdt])
    K, V = (torch.randn(B, ML, nkv, hd, device="cuda", generator=g).to(TORCH[kvdt]) for _ in range(2))
    return pos, Q, K, V


# Against up to 32 (HD 256) or 36 (HD 512) workgroups of a row alone: 1280 and 1152, past two per CU, and 288 MB of caches,
# past the last-level cache.
@pytest.mark.parametrize("kvdt", [1, 2])
@pytest.mark.parametrize("B,ML,nq,nkv,hd,chunk", [(40, 2048, 24, 4, 256, 256), (8, 17600, 16, 1, 512, 512)])
def test_batch_rows_equal_rows_alone(B, ML, nq, nkv, hd, chunk, kvdt):
    pos, Q, K, V = _batch(B, ML, nq, nkv, hd, kvdt, B + kvdt)
    stride = ML * nkv * hd
    A.split_reserve(B, nq, ML, hd)
    O, lse = torch.full((B, nq, hd), float("nan"), device="cuda"), torch.full((B, nq), float("nan"), device="cuda")
    A.attn_batch(Q, K, V, O, B, 1, nq, nkv, hd, torch.from_numpy(pos).cuda(), stride, ML - 1, chunk=chunk, lse=lse)
    assert torch.isfinite(O).all() and torch.isfinite(lse).all(), "a row was not written"
    for b in range(B):
        Ob, lb = torch.empty_like(O[b]), torch.empty_like(lse[b])
        A.attn_batch(Q[b], K[b], V[b], Ob, 1, 1, nq, nkv, hd, torch.from_numpy(pos[b:b + 1]).cuda(), 0, int(pos[b]), chunk=chunk,
                     lse=lb)
        assert torch.equal(O[b], Ob) and torch.equal(lse[b], lb), f"row {b} at {pos[b]}"


@pytest.mark.parametrize("B,ML,nq,nkv,hd", [(40, 2048, 24, 4, 256), (36, 4096, 16, 4, 128)])
def test_fp32_batch_rows_equal_rows_alone(B, ML, nq, nkv, hd):
    """640 and 1152 workgroups of the fp32 kernel against up to 32 of a row alone."""
    pos, Q, K, V = _batch(B, ML, nq, nkv, hd, 0, B)
    A.flash_reserve_partials(B * nq * (ML // 512), hd)
    O = torch.full((B, nq, hd), float("nan"), device="cuda")
    A.attn_decode_batch(Q, K, V, O, B, nq, nkv, hd, 0, ML * nkv * hd, base_b=torch.from_numpy(pos).cuda())
    assert torch.isfinite(O).all(), "a row was not written"
    for b in range(B):
        Ob = torch.empty_like(O[b])
        A.attn_decode(Q[b], K[b], V[b], Ob, 1, nq, nkv, hd, int(pos[b]))
        assert torch.equal(O[b], Ob), f"row {b} at {pos[b]}"
