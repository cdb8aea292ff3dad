"""Verify and tree runs on the tile kernel: edges of the tiles (16-row blocks, 32 and 64 rows, several token tiles), of the
64-key steps and of the chunks, one to many sequences, against fp32 attention; runs over several chunks and sequences against
each sequence alone."""
import numpy as np
import pytest
import torch

import dgx_attn as A

pytestmark = pytest.mark.gpu

TORCH = {1: torch.float16, 2: torch.bfloat16}


def _ref(Q, K, V, base, window, anc):
    T, NQ, HD = Q.shape
    G = NQ // K.shape[1]
    n = base + T
    j, p = torch.arange(n, device="cuda"), base + torch.arange(T, device="cuda")
    ok = j[None, :] <= p[:, None]
    if window:
        ok &= j[None, :] > p[:, None] - window
    if anc is not None:
        d = j - base
        bits = torch.from_numpy(anc.astype(np.int64)).cuda()
        ok &= (d < 0)[None, :] | ((d < 32)[None, :] & ((bits[:, None] >> d.clamp(0, 31)[None, :]) & 1).bool())
    out = torch.empty(T, NQ, HD, device="cuda")
    for h in range(NQ):
        s = (Q[:, h].float() @ K[:n, h // G].float().t().contiguous()) * HD ** -0.5
        out[:, h] = torch.softmax(s.masked_fill(~ok, float("-inf")), -1) @ V[:n, h // G].float().contiguous()
    return out


# T x GRP rows: 17 (one past a block), 32, 33, 48, 64, 65 and 96 (two token tiles), 200, 36 (GRP 36)
SHAPES = [(17, 1, 1, 256), (16, 2, 1, 128), (11, 6, 2, 256), (8, 24, 4, 256), (16, 16, 4, 128), (13, 10, 2, 256),
          (16, 24, 4, 256), (25, 16, 2, 128), (1, 36, 1, 256)]
# 24 sequences of 64-key chunks are more items than run at once: a workgroup takes several chunks in turn; 70 sequences
# (the smaller shapes) are more than a wave's lanes.
BATCHES = [(1, 64, 0), (3, 96, 0), (70, 256, 0), (5, 160, 100), (24, 64, 0), (24, 64, 300)]


@pytest.mark.parametrize("kvdt", [1, 2])
@pytest.mark.parametrize("T,nq,nkv,hd,B,chunk,window", [s + b for s in SHAPES for b in BATCHES if b[0] < 70 or s[0] * s[1] <= 200])
def test_verify_tile_against_fp32(T, nq, nkv, hd, kvdt, B, chunk, window):
    rng = np.random.default_rng(T * 100 + B)
    base = rng.integers(0, 700, B).astype(np.int32)
    base[0] = (0, 63, 64, 95, 160)[B % 5]                   # around step and chunk edges
    ML = 768
    g = torch.Generator(device="cuda").manual_seed(T + B)
    dt = TORCH[kvdt]
    Q = torch.randn(B, T, nq, hd, device="cuda", generator=g).to(dt)
    K = torch.randn(B, ML, nkv, hd, device="cuda", generator=g).to(dt)
    V = torch.randn(B, ML, nkv, hd, device="cuda", generator=g).to(dt)
    anc = None
    if T <= 32 and not window:
        anc = np.array([[(1 << t) | (1 << (t // 2)) | 1 for t in range(T)] for _ in range(B)], np.uint32)
    ancd = None if anc is None else torch.from_numpy(anc.reshape(-1).view(np.int32)).cuda()
    max_pos = int(base.max()) + T - 1
    A.split_reserve(B * T * max(1, -(-A.split_chunk() // chunk)), nq, max_pos + 1, hd)
    O = torch.full((B, T, nq, hd), float("nan"), device="cuda")
    A.attn_batch(Q, K, V, O, B, T, nq, nkv, hd, torch.from_numpy(base).cuda(), ML * nkv * hd, max_pos, chunk=chunk, anc=ancd,
                 window=window)
    for b in sorted({0, B // 2, B - 1}):
        r = _ref(Q[b], K[b], V[b], int(base[b]), window, None if anc is None else anc[b])
        # fp32 output: what is left is the 16-bit P, 2^-12 (f16) of |V| <= 5, and fp32 sums
        assert (O[b] - r).abs().max().item() <= 2e-3, f"sequence {b} at {base[b]}"
    assert torch.isfinite(O).all(), "a row was not written"


def test_ring_that_was_never_filled():
    """Rows of the ring past the last key hold NaN: they are not read."""
    B, T, nq, nkv, hd, cap, W = 2, 8, 24, 4, 256, 512, 400
    g = torch.Generator(device="cuda").manual_seed(3)
    base = torch.tensor([5, 90], dtype=torch.int32, device="cuda")
    Q = torch.randn(B, T, nq, hd, device="cuda", generator=g).half()
    K = torch.full((B, cap, nkv, hd), float("nan"), device="cuda").half()
    V = K.clone()
    for b, n in enumerate((13, 98)):
        K[b, :n] = torch.randn(n, nkv, hd, device="cuda", generator=g).half()
        V[b, :n] = torch.randn(n, nkv, hd, device="cuda", generator=g).half()
    A.split_reserve(B * T, nq, 98, hd)
    O = torch.empty(B, T, nq, hd, device="cuda")
    A.attn_batch_ex(Q, O, B, T, nq, nkv, hd, base, 97, K=K, V=V, kv_stride=cap * nkv * hd, window=W, kv_cap=cap)
    for b in range(B):
        r = _ref(Q[b], K[b], V[b], int(base[b]), W, None)
        assert (O[b] - r).abs().max().item() <= 2e-3        # as above


@pytest.mark.parametrize("runs", [0, 1])
@pytest.mark.parametrize("T,nq,nkv,hd,chunk,cap", [(8, 24, 4, 256, 640, 0), (8, 24, 4, 256, 96, 0), (12, 16, 4, 128, 128, 512),
                                                   (30, 16, 8, 256, 256, 512), (1, 24, 4, 256, 256, 0)])
def test_rows_below_the_window_are_not_read(T, nq, nkv, hd, chunk, cap, runs):
    """A cache (or ring) filled from the first window on only, to whole 16-key blocks: NaN lies below."""
    W, base = 300, torch.tensor([1000, 333, 2047, 1024], dtype=torch.int32)
    B, ML = 4, cap or 2304
    g = torch.Generator(device="cuda").manual_seed(T + chunk)
    Q = torch.randn(B, T, nq, hd, device="cuda", generator=g).half()
    kv = [torch.randn(B, 2304, nkv, hd, device="cuda", generator=g).half() for _ in range(2)]
    K, V = (torch.full((B, ML, nkv, hd), float("nan"), device="cuda").half() for _ in range(2))
    for b, n in enumerate(base.tolist()):
        j = torch.arange((n - W + 1) // 16 * 16, n + T, device="cuda")
        K[b, j % ML], V[b, j % ML] = kv[0][b, j], kv[1][b, j]
    max_pos = int(base.max()) + T - 1
    A.split_reserve(B * T * max(1, -(-A.split_chunk() // chunk)), nq, max_pos + 1, hd)
    O = torch.empty(B, T, nq, hd, device="cuda")
    prev = A.verify_runs(runs)
    try:
        A.attn_batch_ex(Q, O, B, T, nq, nkv, hd, base.cuda(), max_pos, K=K, V=V, kv_stride=ML * nkv * hd, window=W, chunk=chunk,
                        kv_cap=cap)
    finally:
        A.verify_runs(prev)
    for b in range(B):
        r = _ref(Q[b], kv[0][b], kv[1][b], int(base[b]), W, None)
        assert (O[b] - r).abs().max().item() <= 2e-3, f"sequence {b}"        # as above


# Workgroups at once: 256 (HD 256) or 512 (HD 128) over KV heads x tiles. Chunks that outnumber them, with more or fewer
# sequences than runs, and a count of KV heads x tiles that does not divide the device.
@pytest.mark.parametrize("B,T,nq,nkv,hd,chunk,hi,window", [
    (40, 8, 24, 4, 256, 64, 900, 0), (64, 8, 24, 4, 256, 64, 600, 0), (65, 8, 24, 4, 256, 64, 600, 0),
    (130, 9, 16, 4, 128, 64, 700, 0), (9, 30, 24, 3, 256, 96, 2000, 0), (33, 20, 16, 8, 256, 64, 900, 300),
    (3, 32, 48, 24, 256, 64, 500, 0), (2, 8, 24, 4, 256, 64, 9000, 0), (5, 1, 40, 1, 256, 32, 9000, 0)])
def test_runs_do_not_show_in_the_bits(B, T, nq, nkv, hd, chunk, hi, window):
    rng = np.random.default_rng(B)
    base = rng.integers(0, hi, B).astype(np.int32)
    base[rng.integers(0, B, B // 3)] = 0                    # several one-chunk sequences
    base[B // 2] = hi
    ML, max_pos = hi + T, hi + T - 1
    g = torch.Generator(device="cuda").manual_seed(B + T)
    Q = torch.randn(B, T, nq, hd, device="cuda", generator=g).half()
    K, V = (torch.randn(B, ML, nkv, hd, device="cuda", generator=g).half() for _ in range(2))
    A.split_reserve(B * T * -(-A.split_chunk() // chunk), nq, max_pos + 1, hd)
    O, lse = torch.full((B, T, nq, hd), float("nan"), device="cuda"), torch.full((B, T, nq), float("nan"), device="cuda")
    A.attn_batch(Q, K, V, O, B, T, nq, nkv, hd, torch.from_numpy(base).cuda(), ML * nkv * hd, max_pos, chunk=chunk, window=window,
                 lse=lse)
    assert torch.isfinite(O).all() and torch.isfinite(lse).all(), "a row was not written"
    for b in range(B):
        Ob, lb = torch.empty_like(O[b]), torch.empty_like(lse[b])
        A.attn_batch(Q[b], K[b], V[b], Ob, 1, T, nq, nkv, hd, torch.from_numpy(base[b:b + 1]).cuda(), 0, int(base[b]) + T - 1,
                     chunk=chunk, window=window, lse=lb)
        assert torch.equal(O[b], Ob) and torch.equal(lse[b], lb), f"sequence {b} at {base[b]}"
    r = _ref(Q[B // 2], K[B // 2], V[B // 2], hi, window, None)
    assert (O[B // 2] - r).abs().max().item() <= 2e-3       # as above
