"""Query heads per block of the decode attention: the rule, by rows, group and the mean length, and the steps that follow it."""
import numpy as np
import pytest
import torch

from ollama_operator_amd.engine.runner import Runner
from ollama_operator_amd.engine.sampling import SamplingOptions
from ollama_operator_amd.ops import native


@pytest.mark.parametrize("NQ,H,n_kv,D,short,grown", [
    (4, 32, 8, 128, 1, 1), (8, 32, 8, 128, 1, 4), (15, 32, 8, 128, 1, 4), (16, 32, 8, 128, 2, 4), (32, 32, 8, 128, 4, 4),
    (8, 64, 8, 128, 2, 4), (64, 64, 8, 64, 4, 4), (8, 32, 32, 128, 1, 1), (12, 24, 8, 128, 1, 1), (8, 48, 8, 128, 1, 2),
    (32, 32, 8, 256, 2, 2), (32, 32, 8, 80, 2, 2), (32, 4, 2, 64, 1, 2)])
def test_rule(NQ, H, n_kv, D, short, grown):
    heads = native().attention_heads
    assert heads(NQ, H, n_kv, D, 1) == heads(NQ, H, n_kv, D, 1300) == short
    assert heads(NQ, H, n_kv, D, 1301) == heads(NQ, H, n_kv, D, 1 << 40) == grown
    assert (H // n_kv) % short == 0 and (H // n_kv) % grown == 0


@pytest.mark.parametrize("H,n_kv", [(32, 0), (4, 8), (32, 5), (32, -1)])
def test_heads_without_groups_are_refused(H, n_kv):
    with pytest.raises(RuntimeError, match="multiple of n_kv"):
        native().attention_heads(8, H, n_kv, 128, 100)


def test_even_rows_fill_whole_rounds():
    """Splits of rows of one length: no few blocks past a round of 256, which would take a round for themselves."""
    splits = native().attention_even_splits
    assert [splits(b, 1500, 16) for b in (32, 64, 72, 96, 128, 160, 200, 256, 257)] == [8, 4, 3, 2, 2, 1, 1, 1, 1]
    assert [splits(b, 4000, 3) for b in (136, 160, 192, 272)] == [3, 3, 1, 3]  # long rows: two or four rounds of thirds
    for b in range(1, 600):
        for keys in (1500, 4000):
            k = splits(b, keys, 8)
            rounds = -(-b * k // 256)
            # one split more would not fit the rounds that there are, and (256 // 86 = 2) two thirds of them are busy
            assert k in (1, 8) or (b * (k + 1) > 256 * rounds and b * k > 256 * rounds * 2 / 3), (b, keys, k)


@pytest.mark.gpu
@pytest.mark.parametrize("graphs", [True, False])
def test_steps_follow_the_lengths(tiny_models, monkeypatch, graphs):
    """A step graph per choice, taken by the rows' positions; results as with one head throughout. Sums of the same float32 terms in
    another order, through two layers of 16-bit products: 1e-3 (single steps of other batch sizes are allowed 3e-2)."""
    B, O = 32, SamplingOptions(temperature=0)
    rng = np.random.default_rng(2)
    prompts = [[1] + [int(x) for x in rng.integers(3, 500, 5 + i % 7)] for i in range(B)]

    def run(rule):
        r = Runner(tiny_models["tiny-llama"], device="cuda", max_batch=256, max_seqs=B, ctx=64, use_graphs=graphs)
        asked = []
        monkeypatch.setattr(r, "decode_heads", rule)
        if graphs:
            r.capture_batch_graphs(2)
        sids = [r.new_sequence() for _ in prompts]
        for sid, p in zip(sids, prompts):
            r.prefill(sid, p)
        r.recompose([(O, p + [7], 0, 0) for p in prompts], [7] * B)
        out = []
        for step in range(4):
            r.decode_batch(sids, [len(p) + step for p in prompts])
            torch.cuda.synchronize()
            out.append(r.logits[:B, :r.cfg.n_vocab].float().cpu())
            asked.append(r._decode_heads)
        keys = [k for k in r.graphs if k[0] == B]
        r.close()
        return out, keys, asked

    one, k1, _ = run(lambda poss: 1)
    two, k2, after = run(lambda poss: 1 if min(poss) < 8 else 2)
    assert after == [0] * 4  # nothing of a step's choice stays
    if graphs:
        assert {k[4] for k in k1} == {1} and {k[4] for k in k2} == {1, 2}
    for a, b in zip(one, two):
        assert float((a - b).norm() / a.norm()) < 1e-3


@pytest.mark.gpu
def test_the_step_asks_for_the_mean_length(tiny_models):
    r = Runner(tiny_models["tiny-llama"], device="cuda", max_batch=64, max_seqs=2, ctx=64)
    assert r.decode_heads([5] * 31) == 0  # fewer than 64 blocks
    assert r.decode_heads([1299] * 32) == 1 and r.decode_heads([1300] * 32) == 2
    assert r.decode_heads([0] * 16 + [2700] * 16) == 2 and r.decode_heads([0] * 24 + [4000] * 8) == 1
    r.cfg.sliding_window = 600
    assert r.decode_heads([9000] * 32) == 1
    r.close()
