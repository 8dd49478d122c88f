"""Prompt attention (attn_prefill_kernel, csrc/kernels/attention.hip) where its tiles of 64 queries and 64 keys, the two halves
of the keys and the wide heads' layouts end; every key visible to every query (the vision tower)."""
import math

import pytest
import torch

from test_kernels_gpu import C, S, rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D", [64, 80, 96, 112, 128, 256])
@pytest.mark.parametrize("start,NQ,window,whole", [
    (0, 16, 0, False), (0, 63, 0, False), (0, 65, 0, False), (31, 64, 0, False), (129, 33, 0, False),
    (0, 577, 0, True), (70, 321, 32, False), (3, 200, 97, False), (0, 1100, 0, False), (0, 16, 0, True), (0, 32, 0, False),
    (1, 32, 0, False), (15, 17, 0, True), (100, 16, 12, False), (96, 20, 13, False)])
def test_prefill_attention(D, start, NQ, window, whole):
    """Queries, keys and weights are fp16 with float32 sums: the result is off by a few 2^-11 of its size (3e-3, as for the
    decode kernels); keys and values come from the cache as they are stored."""
    kv, G, bs = (2, 4, 16) if NQ < 1000 else (8, 4, 16)  # the long one: more blocks than run at once
    H, total = kv * G, start + NQ
    blocks = (total + bs - 1) // bs
    torch.manual_seed(D + NQ)
    kc, vc = (torch.randn(blocks + 5, kv, bs, D, device="cuda").half() for _ in range(2))
    bt = torch.randperm(blocks + 5, device="cuda")[:blocks].view(1, blocks).int()
    q = torch.randn(NQ, H * D, device="cuda")
    pos = torch.arange(start, start + NQ, device="cuda")
    qlen = torch.full_like(pos, total) if whole else pos + 1
    out = torch.full((NQ + 1, H * D), 7.0, device="cuda")
    ql, seq = qlen.int(), torch.zeros(NQ, device="cuda", dtype=torch.int32)
    C().attention(q.data_ptr(), H * D, kc.data_ptr(), vc.data_ptr(), bt.data_ptr(), blocks, seq.data_ptr(), ql.data_ptr(), NQ, H, kv, D, bs,
                  1 / math.sqrt(D), window, out.data_ptr(), H * D, 0, 1, 0, S(), prefill=1)
    torch.cuda.synchronize()
    t = torch.arange(total, device="cuda")
    rows = lambda c: c.float()[bt[0][t // bs].long(), :, t % bs].repeat_interleave(G, 1).transpose(0, 1).contiguous()  # noqa: E731
    s = torch.matmul(q.view(NQ, H, D).transpose(0, 1).contiguous(), rows(kc).transpose(1, 2).contiguous()) / math.sqrt(D)
    seen = t[None] < qlen[:, None]
    if window:
        seen &= t[None] >= qlen[:, None] - window
    want = torch.matmul(torch.softmax(s.masked_fill(~seen, float("-inf")), -1), rows(vc)).transpose(0, 1).reshape(NQ, -1)
    assert rel(out[:NQ], want) < 3e-3 and bool((out[NQ] == 7.0).all())
