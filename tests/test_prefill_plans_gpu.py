"""Prefill work plans: whatever tile shape, item form (one tile, half a tile, a causal pair) and item-to-XCD mapping a
launch gets, a row's bits are those of the same row in a short launch, and every row is written."""
import pytest
import torch

import dgx_attn as A

pytestmark = pytest.mark.gpu

TORCH = {1: torch.float16, 2: torch.bfloat16}


def _ref(Q, K, V, base, window, scale):
    """fp32 attention of Q [T, NQ, HD] over K / V [n, NKV, HD], token t at base + t."""
    T, NQ, HD = Q.shape
    G = NQ // K.shape[1]
    j = torch.arange(K.shape[0], device="cuda")
    p = base + torch.arange(T, device="cuda")
    ok = j[None, :] <= p[:, None]
    if window:
        ok &= j[None, :] > p[:, None] - window
    out = torch.empty(T, NQ, HD, device="cuda")
    for h in range(NQ):
        s = (Q[:, h].float() @ K[:, h // G].float().t().contiguous()) * scale
        out[:, h] = torch.softmax(s.masked_fill(~ok, float("-inf")), -1) @ V[:, h // G].float().contiguous()
    return out


# T, base, window, heads, head dim, cache type, fp32 Q / O, chunk of the short launches. At 256 CUs: the 128-row tile, the
# 96-row tile, pairs, half tiles, 64-row tiles with several rounds, HD 128 and 512.
@pytest.mark.parametrize("T,base,window,nq,nkv,hd,kvdt,f32", [
    (4096, 0, 1024, 16, 8, 256, 2, False), (4000, 131, 700, 16, 8, 256, 1, True), (1377, 0, 0, 24, 4, 256, 1, True),
    (1024, 0, 0, 16, 8, 256, 2, False), (333, 71, 0, 24, 4, 256, 2, True), (2600, 0, 0, 16, 8, 256, 2, False),
    (1500, 0, 0, 16, 4, 128, 1, False), (1100, 0, 0, 16, 1, 512, 2, False), (2048, 0, 512, 16, 1, 512, 1, True)])
def test_row_bits_do_not_depend_on_the_plan(T, base, window, nq, nkv, hd, kvdt, f32):
    g = torch.Generator(device="cuda").manual_seed(T + hd)
    qt = torch.float32 if f32 else TORCH[kvdt]
    Q = torch.randn(T, nq, hd, device="cuda", generator=g).to(qt)
    K = torch.randn(base + T, nkv, hd, device="cuda", generator=g).to(TORCH[kvdt])
    V = torch.randn(base + T, nkv, hd, device="cuda", generator=g).to(TORCH[kvdt])
    O = torch.full_like(Q, float("nan"))
    lse = torch.full((T, nq), float("nan"), device="cuda")
    A.attn_prefill(Q, K, V, O, 1, T, nq, nkv, hd, base=base, window=window, lse=lse)
    assert torch.isfinite(O.float()).all() and torch.isfinite(lse).all(), "a row was not written"
    for t0, n in ((0, 1), (T // 3, 37), (T // 2 + 5, 150), (T - 7, 7)):
        Os = torch.empty(n, nq, hd, device="cuda", dtype=qt)
        ls = torch.empty(n, nq, device="cuda")
        A.attn_prefill(Q[t0:t0 + n], K, V, Os, 1, n, nq, nkv, hd, base=base + t0, window=window, lse=ls)
        assert torch.equal(O[t0:t0 + n], Os) and torch.equal(lse[t0:t0 + n], ls), f"rows {t0}..{t0 + n - 1}"
        r = _ref(Q[t0:t0 + n].to(TORCH[kvdt]), K[:base + t0 + n], V[:base + t0 + n], base + t0, window, hd ** -0.5)
        # 16-bit output: half an ulp of |O| < 4 (bf16 1.6e-2 / 2, f16 2e-3 / 2); f16 probabilities 2^-12 of |V| <= 5
        assert (Os.float() - r).abs().max().item() <= (2e-3 if f32 or kvdt == 1 else 1e-2)


@pytest.mark.parametrize("nseq,nq,nkv", [(1, 8, 1), (1, 16, 16), (1, 12, 3), (3, 8, 4), (5, 2, 1), (2, 16, 8), (7, 24, 4)])
@pytest.mark.parametrize("T,split", [(40, 0), (333, 0), (333, 128)])
def test_every_head_count_is_mapped(nseq, nq, nkv, T, split):
    """1 to 28 (sequence, KV head) pairs: divisors and multiples of the 8 XCDs, and counts that are neither."""
    HD, base, ML = 256, 70, 512
    g = torch.Generator(device="cuda").manual_seed(nseq * 100 + nq)
    Q = torch.randn(nseq, T, nq, HD, device="cuda", generator=g).half()
    K = torch.randn(nseq, ML, nkv, HD, device="cuda", generator=g).half()
    V = torch.randn(nseq, ML, nkv, HD, device="cuda", generator=g).half()
    O = torch.full_like(Q, float("nan"))
    bb = torch.tensor([base - 3 * s for s in range(nseq)], dtype=torch.int32, device="cuda")
    A.attn_prefill(Q, K, V, O, nseq, T, nq, nkv, HD, base_b=bb, kv_stride=ML * nkv * HD, max_pos=base + T - 1, kv_split=split)
    for s in range(nseq):
        b = base - 3 * s
        r = _ref(Q[s], K[s, :b + T], V[s, :b + T], b, 0, HD ** -0.5)
        assert (O[s].float() - r).abs().max().item() <= 2e-3, f"sequence {s}"      # as above, f16


@pytest.mark.parametrize("kvdt,off", [(1, 1), (2, 3), (2, 4)])
def test_q_off_a_16_byte_boundary(kvdt, off):
    T, nq, nkv, HD = 100, 24, 4, 256
    g = torch.Generator(device="cuda").manual_seed(9)
    buf = torch.randn(off + T * nq * HD, device="cuda", generator=g).to(TORCH[kvdt])
    K = torch.randn(T, nkv, HD, device="cuda", generator=g).to(TORCH[kvdt])
    V = torch.randn(T, nkv, HD, device="cuda", generator=g).to(TORCH[kvdt])
    Q = buf[off:].clone()
    O, Ou = torch.empty_like(Q), torch.empty_like(Q)
    A.attn_prefill(Q, K, V, O, 1, T, nq, nkv, HD)
    A.attn_prefill(buf[off:], K, V, Ou, 1, T, nq, nkv, HD)
    assert torch.equal(O, Ou)
