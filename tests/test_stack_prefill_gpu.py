"""Prompt-portion kernels of layer-list models at the sizes where their tiles end: the matrix-core attention (64 query
rows x 64 keys per tile) against the float64 implementation in `bizulix_oracle.py`."""
import numpy as np
import pytest
import torch

import bizulix_cases as bc
from ollama_operator_amd.ops import stack_native

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim,heads,kv", [(64, 4, 1), (96, 2, 2), (128, 4, 2)])
@pytest.mark.parametrize("cap", [0.0, 20.0])
def test_flash_prefill_tile_edges(tmp_path, dim, heads, kv, cap):
    """One attention layer, prompts that end around tile and group edges, whole and in two portions, and two sequences
    whose rows share a step. Rounding: the layer's input, q / k / v, the outputs and the head's input are bfloat16 (2^-9
    each, five roundings): a row's logits stay within 1e-2 of their spread."""
    m = bc.Model(tmp_path, bc.config([(bc.attn(heads=heads, kv_heads=kv, dim=dim, vdim=dim, scale=dim ** -0.5, softcap=cap), None)],
                                     cap=0.0))
    r = m.runner("cuda", "bfloat16", max_batch=512, kv_tokens=2048)
    toks = bc.tokens(300, 96, seed=dim)
    want, _ = m.oracle(toks)
    for n in (17, 31, 32, 33, 63, 64, 65, 95, 97, 128, 129, 193, 300):
        for cuts in ([n], [max(1, n // 3), n], [n - 1, n]):
            got = bc.run_cuts(r, toks[:n], cuts)
            e = bc.rel_err(got, want[:n])
            assert e.max() < 1e-2, f"{n} rows cut at {cuts}: row {int(e.argmax())} off by {e.max():.3g}"
    a, b = r.new_sequence(), r.new_sequence()
    r.step_entries([(a, toks[:40], [])])
    out = r.step_entries([(a, toks[40:140], list(range(100))), (b, toks[:70], list(range(70)))]).float().cpu().numpy()
    e = bc.rel_err(out, np.concatenate([want[40:140], want[:70]]))
    assert e.max() < 1e-2, f"two sequences in a step: row {int(e.argmax())} off by {e.max():.3g}"


# rows x columns x K: up to 16 / 64 rows (one and several columns per block, K no multiple of 32 x 8 waves); the tiles from
# 64 x 64 to 256 x 256 with ragged last rows and columns, one step of K, odd step counts, K no multiple of 64; short K (to 64
# at 17 .. 64 rows, to 256 above) in small and large tiles; up to 511, and no multiple of 64 beyond; few rows of many columns
GEMMS = [(9, 1, 8), (16, 4100, 264), (16, 40, 72), (17, 33, 2048), (64, 4100, 1032), (64, 15, 96), (65, 64, 64), (65, 65, 72),
         (100, 700, 192), (129, 1024, 704), (300, 3600, 1024), (500, 7177, 2048), (1000, 2048, 2048), (1030, 7177, 2048),
         (2000, 7177, 2112), (2048, 1030, 200), (4096, 2048, 1088), (17, 70, 8), (64, 4100, 64), (33, 65, 72), (65, 100, 8),
         (70, 1030, 256), (2050, 4100, 40), (2048, 4096, 256), (65, 33, 264), (1030, 4100, 320), (64, 8200, 448), (66, 130, 504),
         (65, 40, 520), (1030, 4100, 1032), (3000, 700, 584), (2050, 2100, 520), (17, 8192, 512), (64, 8200, 1088), (33, 9000, 72),
         (50, 8193, 64)]


@pytest.mark.parametrize("M,N,K", GEMMS)
def test_gemm_tiles(M, N, K):
    """Every tile of the bfloat16 products against float64, three epilogues. The operands' products are exact in float32;
    sums of K of them in any order stay within K 2^-24 of the sum of magnitudes (about K times the operands' mean square)."""
    C, s = stack_native(), torch.cuda.current_stream().cuda_stream
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    lda = K + 24  # rows with other columns behind them
    a = torch.randn(M, lda, device="cuda", generator=g).bfloat16()
    w = torch.randn(N, K, device="cuda", generator=g).bfloat16()
    add, res = (torch.randn(M, N, device="cuda", generator=g) for _ in range(2))
    ref = a[:, :K].double() @ w.double().T
    lim = 2.0 ** -24 * K * K ** 0.5 + 1e-5
    p = dict(A=a.data_ptr(), lda=lda, W=w.data_ptr(), M=M, N=N, K=K, ldc=N, f32=0)
    out = torch.full((M, N), 7.0, device="cuda")
    C.gemm(dict(p, C=out.data_ptr(), epi=0), s)
    assert float((out.double() - ref).abs().max()) < lim
    want = res.double() + 0.5 * (ref + add.double())
    C.gemm(dict(p, C=res.data_ptr(), epi=1, mult=0.5, add=add.data_ptr()), s)
    assert float((res.double() - want).abs().max()) < lim
    C.gemm(dict(p, C=out.data_ptr(), epi=2, cap=5.0), s)
    assert float((out.double() - 5.0 * torch.tanh(ref / 5.0)).abs().max()) < lim + 1e-5


@pytest.mark.parametrize("rows,experts,ff", [(40, 6, 24), (150, 4, 72), (500, 4, 64), (700, 3, 40), (60, 40, 448), (200, 40, 424)])
def test_grouped_experts(tmp_path, rows, experts, ff):
    """Routed feed-forwards with few, some and many rows per expert (64-row and 128-row tiles, few and many blocks; K = ff and
    K = 64 with and without a remainder of 64) against the float64 implementation."""
    m = bc.Model(tmp_path, bc.config([(bc.attn(dim=16, vdim=16), bc.moe(experts=experts, top=2, ff=ff, shared_ff=0))], cap=0.0))
    r = m.runner("cuda", "bfloat16", max_batch=1024, kv_tokens=2048)
    toks = bc.tokens(rows, 96, seed=rows)
    want, _ = m.oracle(toks)
    bc.check(bc.run_cuts(r, toks, [rows]), want, "bfloat16", f"{rows} rows, {experts} experts of {ff}")


@pytest.mark.parametrize("dim,vdim", [(64, 64), (72, 44), (96, 96), (128, 128), (40, 120), (64, 200), (24, 30)])
@pytest.mark.parametrize("dtype", ["bfloat16", "float32"])
def test_decode_attention(tmp_path, dim, vdim, dtype):
    """Single rows over 1 .. 300 keys, where the groups of 64 keys and the rounds of four waves end: values requested ahead of
    the scores (16-bit, up to 128 dims), value rows no multiple of a piece, wide ones. Limits as for the prompts; in
    float32 the oracle's (2^-24 per operation, some hundred of them in a row)."""
    m = bc.Model(tmp_path, bc.config([(bc.attn(heads=2, kv_heads=1, dim=dim, vdim=vdim, scale=dim ** -0.5), None)], cap=0.0))
    r = m.runner("cuda", dtype, max_batch=512, kv_tokens=2048)
    toks = bc.tokens(300, 96, seed=dim + vdim)
    want, _ = m.oracle(toks)
    for n in (1, 2, 63, 64, 65, 128, 129, 255, 256, 257, 300):
        got = bc.run_cuts(r, toks[:n], [n] if n == 1 else [n - 1, n])
        e = bc.rel_err(got[-1:], want[n - 1:n])
        assert e.max() < (1e-2 if dtype == "bfloat16" else 1e-4), f"{n} keys: off by {e.max():.3g}"


@pytest.mark.parametrize("dim,vdim", [(64, 64), (192, 64), (256, 128), (192, 160)])
def test_many_single_rows(tmp_path, dim, vdim):
    """A step of 20 sequences with a row each (decode steps of more than 16 users), short and long contexts side by side: on query
    tiles, or wide keys on a block per row and head. Limits as for the prompts."""
    m = bc.Model(tmp_path, bc.config([(bc.attn(heads=4, kv_heads=2, dim=dim, vdim=vdim, scale=dim ** -0.5), None)], cap=0.0))
    r = m.runner("cuda", "bfloat16", max_batch=512, max_seqs=20, kv_tokens=4096)
    toks = bc.tokens(300, 96, seed=dim + vdim)
    want, _ = m.oracle(toks)
    ctx = [1, 2, 31, 32, 33, 63, 64, 65, 299] + list(range(100, 111))
    ids = [r.new_sequence() for _ in ctx]
    for i, n in zip(ids, ctx):
        r.step_entries([(i, toks[:n], [])])
    out = r.step_entries([(i, [toks[n]], [0]) for i, n in zip(ids, ctx)]).float().cpu().numpy()
    e = bc.rel_err(out, want[ctx])
    assert e.max() < 1e-2, f"{ctx[int(e.argmax())]} keys: off by {e.max():.3g}"
