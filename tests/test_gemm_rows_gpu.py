"""Prompt portions of 16 .. 64 rows (csrc/kernels/gemm_rows.hip) and of 65 .. 127 (the 128-row tiles of gemm_dq.hip): every quant
type against a float32 product on the dequantised weights, where rows, columns, super-blocks and the waves' shares of K end, the
epilogues that pair rows, and what the kernels leave to others. Launch counters say which kernel ran."""
import math

import pytest
import torch

from ollama_operator_amd.gguf import GGMLType
from test_kernels_gpu import QM, QTYPES, C, S, rel

pytestmark = pytest.mark.gpu
p = lambda t: t.data_ptr() if t is not None else 0  # noqa: E731


def run(m, x, y, epi=0, norm=0, nw=None, bias=None, extra=None, rows=0, kernel=""):
    """rows: rows that the fp16 workspace holds (0: whole row tiles); kernel: the launch counter that moves, and no other."""
    B, K = x.shape
    xws = torch.empty((rows or (B + 15) // 16 * 16) * ((K + 255) // 256 * 256), device="cuda", dtype=torch.float16)
    d = dict(extra or {}, xws=xws.data_ptr(), xws_elems=xws.numel())
    on = C().dq_gemm_enabled()
    C().set_dq_gemm(1)
    C().reset_launch_counts()
    C().gemv(m.tup, B, p(x), K, norm, p(nw), 0, 1e-5, epi, p(y), y.shape[1], p(bias), 0, d, S())
    torch.cuda.synchronize()
    C().set_dq_gemm(int(on))
    n = C().launch_counts()
    kernel = kernel or ("gemm_rows" if B <= 64 else "dq_gemm")
    assert {k: v for k, v in n.items() if v} == {kernel: 1}, n


@pytest.mark.parametrize("qt", QTYPES)
@pytest.mark.parametrize("N,K", [(1, 256), (40, 288), (450, 1280), (4096, 4096), (8200, 768), (16400, 512), (3200, 8640)])
def test_rows(qt, N, K):
    """fp16 products with float32 sums against float32 on the same dequantised weights: both operands are rounded to fp16
    (2^-11 each, as in the larger GEMMs), so the result is off by about 2^-11 of its size."""
    if K % 256 and qt in (GGMLType.Q4_K, GGMLType.Q5_K, GGMLType.Q6_K):
        pytest.skip("k-quant rows are whole super-blocks")
    m = QM(qt, N, K, seed=K)
    for B in (16, 17, 33, 48, 64, 65, 100, 127):
        x = torch.randn(B, K, device="cuda")
        y = torch.full((B, N + 3), 9.0, device="cuda")
        run(m, x, y)
        assert rel(y[:, :N], x @ m.w.T) < 2e-3, B
        assert bool((y[:, N:] == 9.0).all())


@pytest.mark.parametrize("B", [16, 50, 127])
def test_rows_epilogues(B):
    N, K = 512, 1024
    m = QM(GGMLType.Q4_K, N, K, seed=B)
    x, nw, bias = torch.randn(B, K, device="cuda"), torch.rand(K, device="cuda") + 0.5, torch.randn(N, device="cuda")
    h = x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + 1e-5) * nw
    y0 = torch.randn(B, N, device="cuda")
    y = y0.clone()
    run(m, x, y, epi=1, norm=1, nw=nw, bias=bias)  # residual add of a normed product
    assert rel(y - y0, h @ m.w.T + bias) < 2e-3
    y = torch.zeros(B, N // 2, device="cuda")
    run(m, x, y, epi=2, norm=1, nw=nw)  # gate and up rows in turn
    z = h @ m.w.T
    assert rel(y, torch.nn.functional.silu(z[:, 0::2]) * z[:, 1::2]) < 4e-3
    # q | k | v with a rotation of row pairs and the scatter into a paged cache
    D, heads, kv, bs = 64, 4, 2, 16
    blocks = (B + bs - 1) // bs
    kc, vc = (torch.zeros(blocks, kv, bs, D, device="cuda", dtype=torch.float16) for _ in range(2))
    pos = torch.arange(B, device="cuda", dtype=torch.int32)
    freq = (1e4 ** (-torch.arange(0, D, 2, device="cuda").double() / D)).float()
    q = torch.zeros(B, heads * D, device="cuda")
    run(m, x, q, epi=4, norm=1, nw=nw, extra=dict(pos=p(pos), slot=p(pos), kc=p(kc), vc=p(vc), inv_freq=p(freq), Eq=heads * D,
                                                  Ekv=kv * D, D=D, n_rot=D, n_kv=kv, bs=bs))
    ang = pos.float()[:, None, None] * freq

    def turn(t):
        u, v = t[..., 0::2], t[..., 1::2]
        return torch.stack([u * torch.cos(ang) - v * torch.sin(ang), u * torch.sin(ang) + v * torch.cos(ang)], -1).reshape(t.shape)

    zq, zk, zv = z.split([heads * D, kv * D, kv * D], 1)
    assert rel(q, turn(zq.view(B, heads, D)).reshape(B, -1)) < 2e-3
    seen = lambda c: c.permute(0, 2, 1, 3).reshape(blocks * bs, kv, D)[:B].float()  # noqa: E731
    assert rel(seen(kc), turn(zk.view(B, kv, D))) < 3e-3 and rel(seen(vc), zv.view(B, kv, D)) < 3e-3
    assert math.isfinite(float(kc.float().abs().max()))


@pytest.mark.parametrize("qt", QTYPES)
@pytest.mark.parametrize("K", [256, 768, 1280, 2304])
def test_activations_past_fp16(qt, K):
    """An activation that overflows fp16 (its rows' products are infinite, or no number where the weight is 0) in the last
    super-block, which the lane groups past a count that is no multiple of four load too: the same infinities as the product
    of the rounded operands gives, and rows without one stay finite."""
    m = QM(qt, 96, K, seed=K)
    for B in (16, 33, 64):
        x = torch.randn(B, K, device="cuda")
        x[B // 2, K - 7] = 1e6
        y = torch.zeros(B, 96, device="cuda")
        run(m, x, y)
        want = x.half().double() @ m.w.double().T
        assert bool((torch.isnan(y) == torch.isnan(want)).all()) and bool((torch.isinf(y) == torch.isinf(want)).all())
        inf = torch.isinf(want)
        assert bool((y[inf].double() == want[inf]).all())
        rows = torch.arange(B, device="cuda") != B // 2
        assert rel(y[rows], want[rows].float()) < 2e-3


@pytest.mark.parametrize("B", [17, 33, 63])
def test_short_workspace(B):
    """A workspace without room for the last row tile (the caller's rows only): the 128 x 128 tile kernel takes the call."""
    m = QM(GGMLType.Q4_K, 200, 1024, seed=B)
    x, y = torch.randn(B, 1024, device="cuda"), torch.zeros(B, 200, device="cuda")
    run(m, x, y, rows=B, kernel="gemm_tile")
    assert rel(y, x @ m.w.T) < 2e-3


@pytest.mark.parametrize("qt", [GGMLType.Q4_0, GGMLType.Q6_K])
@pytest.mark.parametrize("B", [16, 64, 65, 130])
def test_wide_rows(qt, B):
    """The preparation keeps a row of activations in LDS, 160 KB: K = 40,704 is the last that fits, a wider matrix goes to the
    tile kernel. (32-wide blocks: K need not be whole super-blocks.)"""
    for K, kernel in ((40704, ""), (40736 if qt == GGMLType.Q4_0 else 40960, "gemm_tile"), (45056, "gemm_tile")):
        m = QM(qt, 40, K, seed=B)
        x, y = torch.randn(B, K, device="cuda"), torch.zeros(B, 40, device="cuda")
        run(m, x, y, kernel=kernel)
        assert rel(y, x @ m.w.T) < 2e-3, K


@pytest.mark.parametrize("qt", QTYPES)
@pytest.mark.parametrize("N,K", [(130, 1024), (256, 2304), (1024, 4096), (4096, 4096), (512, 11008), (2048, 11008), (22016, 512)])
def test_split_k(qt, N, K):
    """65 .. 127 rows with room for partial sums: narrow matrices split K up to 16 ways, shares of unequal length among them, and
    add the shares up in a second launch. Limits as above."""
    m = QM(qt, N, K, seed=N)
    gws = torch.full((16 * 127 * N,), float("nan"), device="cuda")
    for B in (65, 96, 127):
        x, y = torch.randn(B, K, device="cuda"), torch.full((B, N + 3), 9.0, device="cuda")
        run(m, x, y, extra=dict(gws=p(gws), gws_elems=gws.numel()))
        assert rel(y[:, :N], x @ m.w.T) < 2e-3, B
        assert bool((y[:, N:] == 9.0).all())
