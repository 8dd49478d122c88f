"""Prompt-portion kernels of layer-list models at the sizes where their tiles end: the matrix-core attention (64 query
rows x 64 keys per tile) against the float64 implementation in `bizulix_oracle.py`."""
import numpy as np
import pytest

import bizulix_cases as bc

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
