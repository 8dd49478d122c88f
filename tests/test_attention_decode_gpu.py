"""Decode attention: heads per block, block order and the split count over rows, groups and ragged lengths."""
import pytest
import torch

from ollama_operator_amd.ops import native

pytestmark = pytest.mark.gpu


def check(H, Hkv, lens, window, splits, mb=None):
    """Against float64. Score, weight and sum are float32 chains of at most 4,700 terms of one sign or 128 of both: some 2e-6 of the
    result; the bound is five times that."""
    D, bs, G, NQ = 128, 16, H // Hkv, len(lens)
    mb = mb or (max(lens) + bs - 1) // bs
    nblk = NQ * mb
    gen = torch.Generator("cuda").manual_seed(H + NQ)
    kc = torch.randn(nblk, Hkv, bs, D, device="cuda", generator=gen, dtype=torch.float16)
    vc = torch.randn(nblk, Hkv, bs, D, device="cuda", generator=gen, dtype=torch.float16)
    bt = torch.randperm(nblk, device="cuda", generator=gen).view(NQ, mb).int()
    q = torch.randn(NQ, H * D, device="cuda", generator=gen)
    seq = torch.arange(NQ - 1, -1, -1, device="cuda", dtype=torch.int32)  # query i reads table row NQ - 1 - i
    qlen = torch.tensor(lens, device="cuda", dtype=torch.int32)
    refs = []
    for i, n in enumerate(lens):
        t = torch.arange(max(0, n - window) if window else 0, n, device="cuda")
        b = bt[NQ - 1 - i][t // bs].long()
        k, v = kc[b, :, t % bs].double(), vc[b, :, t % bs].double()  # [n, Hkv, D]
        s = (k[:, :, None] * q[i].view(Hkv, G, D).double()).sum(-1) * D ** -0.5
        refs.append((torch.softmax(s, 0)[..., None] * v[:, :, None]).sum(0).reshape(-1))
    out = torch.empty(NQ, H * D, device="cuda")
    for S in splits:
        ws = torch.full((max(1, native().attention_ws_floats(NQ, H, D, S)),), float("nan"), device="cuda")
        cnt = torch.zeros(NQ * H, device="cuda", dtype=torch.int32)
        for _ in range(2):  # the tickets re-arm themselves
            out.fill_(float("nan"))
            native().attention(q.data_ptr(), H * D, kc.data_ptr(), vc.data_ptr(), bt.data_ptr(), mb, seq.data_ptr(), qlen.data_ptr(), NQ,
                               H, Hkv, D, bs, D ** -0.5, window, out.data_ptr(), H * D, ws.data_ptr(), S, cnt.data_ptr(),
                               torch.cuda.current_stream().cuda_stream)
        assert int(cnt.abs().sum()) == 0
        for i, n in enumerate(lens):
            err = float((out[i].double() - refs[i]).norm() / refs[i].norm())
            assert err < 1e-5, (S, i, n, err)


@pytest.mark.parametrize("window", [0, 700])
@pytest.mark.parametrize("H,Hkv,NQ", [(32, 8, 1), (32, 8, 3), (32, 8, 8), (32, 8, 17), (32, 32, 5), (32, 32, 8), (24, 8, 12), (64, 8, 24),
                                      (20, 2, 9)])
def test_rows_groups_and_lengths(H, Hkv, NQ, window):
    """Lengths lie around one split (512 keys), two, and a split more per 4,096."""
    some = [511, 1, 4700, 513, 37, 768, 769, 4097, 128]
    lens = [some[i % len(some)] if i < 9 else 1 + 97 * i % 600 for i in range(NQ)]
    check(H, Hkv, lens, window, sorted({1, 7, max(1, min(32, 512 // (NQ * Hkv)))}), mb=300)


@pytest.mark.parametrize("H,Hkv,NQ", [(32, 8, 1), (32, 8, 9), (32, 8, 12), (32, 8, 17), (32, 32, 3), (32, 32, 5), (64, 8, 17), (8, 8, 70)])
@pytest.mark.parametrize("n", [513, 700, 2304, 2600])
def test_rows_of_one_length(H, Hkv, NQ, n):
    """Lengths within a quarter of their mean, among them the last that takes the short rows' splits and longer ones; more rows than a
    wave has lanes; and the same rows beside one of another length, which leaves some of them on either rule."""
    S = max(1, min(32, 512 // (NQ * Hkv)))
    check(H, Hkv, [n + 7 * i % 61 for i in range(NQ)], 0, [S, 5])
    check(H, Hkv, [40] + [n - 5 * i % 300 for i in range(1, NQ)], 0, [S])
