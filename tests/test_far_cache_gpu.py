"""Caches whose K (or V) of one sequence passes 2 and 4 GiB: every entry point reads the right rows there."""
import pytest
import torch

import dgx_attn as A

pytestmark = pytest.mark.gpu

TORCH = {0: torch.float32, 1: torch.float16, 2: torch.bfloat16}
ROW = 4096                                  # bytes of a cache row, so row 2^20 starts at byte 2^32
FAR, ROWS, W = 1 << 20, (1 << 20) + 1088, 300


@pytest.fixture(scope="module")
def buf():
    """One buffer serves as K and as V; rows that no test attends hold 3."""
    b = torch.full((ROWS * ROW // 2,), 3.0, device="cuda", dtype=torch.float16)
    yield b
    del b
    torch.cuda.empty_cache()


def _cache(buf, kvdt, hd, first, n, seed):
    """The buffer as a cache [rows, heads, hd] with rows [first, first + n) drawn, the others 3."""
    dt = TORCH[kvdt]
    es = dt.itemsize
    kv = buf.view(dt).view(ROWS, ROW // es // hd, hd)
    g = torch.Generator(device="cuda").manual_seed(seed)
    kv.fill_(3.0)
    kv[first:first + n] = torch.randn(n, *kv.shape[1:], device="cuda", generator=g).to(dt)
    return kv


def _ref(Q, kv, pos0, window, first):
    """fp32 attention of Q [T, NQ, HD] at positions pos0 + t over kv, whose row 0 is key `first`."""
    T, NQ, HD = Q.shape
    G = NQ // kv.shape[1]
    j = first + torch.arange(kv.shape[0], device="cuda")
    p = pos0 + torch.arange(T, device="cuda")
    ok = (j[None, :] <= p[:, None]) & (j[None, :] > p[:, None] - window)
    out = torch.empty(T, NQ, HD, device="cuda")
    for h in range(NQ):
        k = kv[:, h // G].float().contiguous()
        s = (Q[:, h].float() @ k.t().contiguous()) * HD ** -0.5
        out[:, h] = torch.softmax(s.masked_fill(~ok, float("-inf")), -1) @ k
    return out


# Rows around byte 2^31 (row 600000), across byte 2^32, and past it.
@pytest.mark.parametrize("base", [600000, FAR - 40, FAR + 900])
@pytest.mark.parametrize("kind,hd,nq,kvdt,T", [
    ("decode", 256, 16, 1, 1), ("verify", 256, 16, 1, 9), ("verify", 256, 24, 2, 13), ("verify", 128, 32, 1, 12),
    ("flash", 256, 16, 2, 11), ("flash", 512, 16, 1, 7), ("prefill", 256, 16, 2, 100), ("prefill", 128, 32, 1, 100),
    ("prefill", 512, 16, 2, 70), ("prefill", 256, 16, 0, 75), ("split", 256, 16, 1, 100), ("v2", 256, 24, 1, 150)])
def test_rows_past_32_bit_offsets(buf, kind, hd, nq, kvdt, T, base):
    nkv, C = ROW // TORCH[kvdt].itemsize // hd, 640
    kv = _cache(buf, kvdt, hd, base - W, W + T, base + hd)
    fp32 = kind in ("flash", "v2") or kvdt == 0
    g = torch.Generator(device="cuda").manual_seed(T)
    Q = torch.randn(T, nq, hd, device="cuda", generator=g).to(torch.float32 if fp32 else TORCH[kvdt])

    def call(cache, b):
        O = torch.full((T, nq, hd), float("nan"), device="cuda", dtype=torch.float32 if kind == "verify" else Q.dtype)
        if kind in ("decode", "verify"):
            pos = torch.tensor([b], dtype=torch.int32, device="cuda")
            A.split_reserve(T * max(1, -(-A.split_chunk() // C)), nq, b + T, hd)
            A.attn_batch(Q, cache, cache, O, 1, T, nq, nkv, hd, pos, 0, b + T - 1, chunk=C, window=W)
        elif kind == "flash":
            A.flash_attn(Q, cache, cache, O, T, nq, nkv, hd, b, window=W)
        elif kind == "v2":
            A.flash_attn_v2(Q, cache, cache, O, T, nq, nkv, hd, b, window=W)
        else:
            A.attn_prefill(Q, cache, cache, O, 1, T, nq, nkv, hd, base=b, window=W, kv_split=C if kind == "split" else 0)
        return O

    O = call(kv, base)
    D = (base - W) // 2560 * 2560               # a multiple of every chunk, split and step: the same boundaries
    assert torch.equal(O, call(kv[D:], base - D)), "not the bits of the same rows in a short cache"
    r = _ref(Q.to(TORCH[kvdt]) if kvdt else Q.bfloat16(), kv[base - W:base + T] if kvdt else kv[base - W:base + T].bfloat16(),
             base, W, base - W)
    # half an ulp of |O| < 4 in the output type (bf16 8e-3, f16 1e-3), f16 probabilities 2^-12 of |V| <= 5
    assert (O.float() - r).abs().max().item() <= (1e-2 if O.dtype == torch.bfloat16 else 2e-3)


@pytest.mark.parametrize("T", [9, 100])
def test_ring_past_32_bit_offsets(buf, T):
    """A ring of more than 4 GiB: rows past byte 2^32 up to its end, then row 0."""
    cap, nq, nkv, hd = ROWS, 16, 8, 256
    base = 2 * cap - 30                          # keys base - W .. base + T - 1 sit in rows cap - 330 .. cap - 1, 0 ..
    kv = _cache(buf, 1, hd, 0, 200, 5)
    g = torch.Generator(device="cuda").manual_seed(6)
    kv[cap - 400:] = torch.randn(400, nkv, hd, device="cuda", generator=g).half()
    Q = torch.randn(T, nq, hd, device="cuda", generator=g).half()
    O = torch.full((T, nq, hd), float("nan"), device="cuda", dtype=torch.float16)
    if T < 32:
        C = 640
        A.split_reserve(T * max(1, -(-A.split_chunk() // C)), nq, base + T, hd)
        A.attn_batch_ex(Q, O, 1, T, nq, nkv, hd, torch.tensor([base], dtype=torch.int32, device="cuda"), base + T - 1, K=kv, V=kv,
                        chunk=C, window=W, kv_cap=cap)
    else:
        A.attn_prefill(Q, kv, kv, O, 1, T, nq, nkv, hd, base=base, window=W, kv_cap=cap)
    rows = torch.arange(base - W, base + T, device="cuda") % cap
    assert (O.float() - _ref(Q, kv[rows], base, W, base - W)).abs().max().item() <= 2e-3        # as above, f16
