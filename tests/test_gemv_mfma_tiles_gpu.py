"""The batched decode GEMV with one, two and three row tiles a block, at every epilogue that has a kernel of its own: stores and gated
outputs, residual adds (with the next projection's input and without), q k v, and the launch of two matrices. Every product is
counted, so one that another kernel took fails."""
import pytest
import torch

from ollama_operator_amd.engine.runner import Runner
from ollama_operator_amd.gguf import GGMLType
from ollama_operator_amd.gguf.constants import FileType
from ollama_operator_amd.models.config import preset
from ollama_operator_amd.models.random_init import write_random_gguf
from test_gemv_mfma_gpu import QMM, f16_rows
from test_kernels_gpu import C, gemv, rel

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def counted():
    """products() -> those that ran on these kernels since the last call"""
    C().reset_launch_counts()

    def products():
        n = C().launch_counts()
        C().reset_launch_counts()
        assert all(n[k] == 0 for k in n if k.startswith("gem") and k != "gemv_mb"), n
        return n["gemv_mb"]
    yield products


@pytest.mark.parametrize("rows16", [False, True], ids=["float32 rows", "fp16 rows"])
@pytest.mark.parametrize("B", [3, 16])
@pytest.mark.parametrize("qt,N,K", [(GGMLType.Q4_K, 4096, 1024), (GGMLType.Q4_K, 4112, 1024), (GGMLType.Q8_0, 8250, 2304),
                                    (GGMLType.Q6_K, 8250, 2304), (GGMLType.Q4_0, 8250, 2304), (GGMLType.Q4_K, 4150, 6144),
                                    (GGMLType.Q8_0, 4150, 6144)])
def test_tiles_and_epilogues(qt, N, K, B, rows16, counted):
    """256 blocks: 4,096 rows are a tile for each, 4,112 two for one of them, 8,250 two to three, the last partial. Weights are
    fp16(scale * code) and the sums float32: an error of 2^-11 a weight at most, 3e-4 in all; the bound is that of the other tests."""
    if not rows16 and B == 16 and K > 4096:
        B = 8  # 16 fp16 rows do not fit the LDS
    m = QMM(qt, N, K, seed=N + B)
    x = torch.randn(B, K, device="cuda")
    extra = {}
    if rows16:
        x = x.half().float()
        x16 = f16_rows(x, (K + 255) // 256 * 256, 0)  # nothing is read past the last row
        extra = dict(x16=x16.data_ptr(), ld16=x16.shape[1])
    ref = x @ m.w.T
    bias = torch.randn(N, device="cuda")
    y0 = torch.randn(B, N, device="cuda")
    for b in (None, bias):
        rb = ref if b is None else ref + b
        y = torch.full((B, N), float("nan"), device="cuda")
        gemv(m, x, y=y, bias=b, extra=dict(extra))
        assert rel(y, rb) < 4e-3
        y = y0.clone()
        gemv(m, x, epi=1, y=y, bias=b, extra=dict(extra))
        assert rel(y, y0 + rb) < 4e-3
    y = torch.full((B, N // 2), float("nan"), device="cuda")
    gemv(m, x, epi=2, y=y, extra=dict(extra))
    assert rel(y, torch.nn.functional.silu(ref[:, 0::2]) * ref[:, 1::2]) < 8e-3
    assert counted() == 5


@pytest.mark.parametrize("biased", [False, True])
@pytest.mark.parametrize("B", [3, 16])
@pytest.mark.parametrize("qt,H,Hkv,K", [(GGMLType.Q4_K, 16, 8, 4096), (GGMLType.Q4_K, 32, 32, 2304), (GGMLType.Q6_K, 32, 8, 4096),
                                        (GGMLType.Q8_0, 32, 8, 2304), (GGMLType.Q4_0, 16, 8, 1024), (GGMLType.Q4_K, 32, 8, 6144)])
def test_qkv_on_fp16_rows(qt, H, Hkv, K, B, biased, counted):
    """q k v on the decode chain's rows, one to three tiles a block, against float64. Products as above (2^-11 a weight, 4e-3 allowed);
    q is kept in float32, the cache adds a rounding to fp16 (2^-11) to a turned pair."""
    D, n_rot, bs = 128, 128, 16
    Eq, Ekv = H * D, Hkv * D
    m = QMM(qt, Eq + 2 * Ekv, K, seed=K + H)
    x = torch.randn(B, K, device="cuda").half().float()
    x16 = f16_rows(x, (K + 255) // 256 * 256, 0)
    bias = torch.randn(Eq + 2 * Ekv, device="cuda") if biased else None
    pos = torch.arange(B, device="cuda", dtype=torch.int32) * 37 + 5
    slot = torch.randperm(20 * bs, device="cuda")[:B].int()
    inv = (10000.0 ** (-torch.arange(0, n_rot // 2, dtype=torch.float64) * 2 / n_rot)).float().cuda()
    q = torch.zeros(B, Eq, device="cuda")
    kc = torch.zeros(20, Hkv, bs, D, device="cuda", dtype=torch.float16)
    vc = torch.zeros_like(kc)
    gemv(m, x, epi=4, y=q, bias=bias, extra=dict(
        x16=x16.data_ptr(), ld16=x16.shape[1], pos=pos.data_ptr(), slot=slot.data_ptr(), kc=kc.data_ptr(), vc=vc.data_ptr(),
        inv_freq=inv.data_ptr(), Eq=Eq, Ekv=Ekv, D=D, n_rot=n_rot, n_kv=Hkv, bs=bs))
    assert counted() == 1
    y = x.double() @ m.w.double().T + (0 if bias is None else bias.double())
    ang = (pos.float()[:, None] * inv).double()
    cs, sn = torch.cos(ang)[:, None], torch.sin(ang)[:, None]

    def turned(t, heads):
        t = t.view(B, heads, D)
        a, b = t[..., 0::2], t[..., 1::2]
        return torch.stack([a * cs - b * sn, a * sn + b * cs], -1).reshape(B, heads, D)

    at = slot.long()
    assert rel(q.view(B, H, D), turned(y[:, :Eq], H)) < 4e-3
    assert rel(kc[at // bs, :, at % bs], turned(y[:, Eq:Eq + Ekv], Hkv)) < 5e-3
    assert rel(vc[at // bs, :, at % bs], y[:, Eq + Ekv:].view(B, Hkv, D)) < 5e-3
    assert int((kc != 0).any(-1).sum()) == int((vc != 0).any(-1).sum()) == B * Hkv  # nothing in other rows


@pytest.mark.parametrize("B", [3, 16])
@pytest.mark.parametrize("qt,N,K", [(GGMLType.Q4_K, 4096, 2304), (GGMLType.Q4_K, 4112, 1024), (GGMLType.Q6_K, 8250, 2304),
                                    (GGMLType.Q4_K, 4150, 6144)])
def test_residual_add_that_feeds_the_next(qt, N, K, B, counted):
    """The residual, fp16(residual * norm weight) and the sums of squares per 16 rows, with up to three tiles a block."""
    m = QMM(qt, N, K, seed=N + K)
    x = torch.randn(B, K, device="cuda").half().float()
    x16 = f16_rows(x, (K + 255) // 256 * 256, 0)
    y0 = torch.randn(B, N, device="cuda") * 4
    y = y0.clone()
    nw = torch.rand(N, device="cuda") + 0.5
    nt = (N + 15) // 16
    e16 = torch.zeros(B + 1, N, device="cuda", dtype=torch.float16)
    st = torch.full((16, nt), -1.0, device="cuda")
    gemv(m, x, epi=1, y=y, extra=dict(x16=x16.data_ptr(), ld16=x16.shape[1], emit16=e16.data_ptr(), ld_emit=N, emit_nw=nw.data_ptr(),
                                      emit_stat=st.data_ptr()))
    assert counted() == 1
    assert rel(y, y0 + x @ m.w.T) < 4e-3
    assert rel(e16[:B].float(), y * nw) < 1e-3 and float(e16[B].abs().max()) == 0.0
    sq = torch.nn.functional.pad(y.double().pow(2), (0, 16 * nt - N)).view(B, nt, 16).sum(-1)
    assert torch.allclose(st[:B].double(), sq, rtol=1e-5) and bool((st[B:] == -1).all())


@pytest.mark.parametrize("E", [512, 2304, 4096])
@pytest.mark.parametrize("B", [4, 16])
def test_two_matrices_in_one_launch(tmp_path, E, B):
    """q, k in Q4_K and v in Q6_K: the second layer's q k v is one launch on the chain's rows, of one and two super-blocks a wave. The
    step's logits against the int8 GEMV's (2e-2, as for other models), and every projection of the step counted once."""
    path = str(tmp_path / "m.gguf")
    write_random_gguf(path, preset("tiny-llama", n_embd=E, n_ff=512, n_layer=2, n_head=E // 128, n_head_kv=E // 128, n_rot=128,
                                   ctx_len=128), FileType.MOSTLY_Q4_K_M, seed=E)
    g = Runner(path, device="cuda", max_batch=64, max_seqs=16, ctx=128, use_graphs=False)
    assert [bool(g.w.layers[i].get("wv")) for i in (0, 1)] == [False, True] and g.exe.exe.mb_chain
    prompts = [[1] + [3 + (7 * i + j * j) % 400 for j in range(4 + i)] for i in range(B)]
    sids = [g.new_sequence() for _ in prompts]
    for sid, p in zip(sids, prompts):
        g.prefill(sid, p)
    out = []
    for on in (1, 0):
        C().set_mb_enable(on)
        try:
            g.set_tokens(list(range(7, 7 + B)))
            C().reset_launch_counts()
            g.decode_batch(sids, [len(p) for p in prompts])
            torch.cuda.synchronize()
            n = C().launch_counts()["gemv_mb"]
        finally:
            C().set_mb_enable(1)
        assert n == (9 if on else 0), n  # q k v, o, gate up, down of two layers and the head
        out.append(g.logits[:B, :g.cfg.n_vocab].float().cpu())
    assert rel(out[0], out[1]) < 2e-2
    g.close()
