"""Single stage calls of the native executor: a layer's attention stage works on the positions it is given, whatever ran before."""
import numpy as np
import pytest
import torch

from ollama_operator_amd.engine.runner import Runner

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B", [16, 70])  # the products of up to 64 rows, and the tiles
def test_attention_stage_of_a_later_layer_uses_its_own_positions(tiny_models, B):
    r = Runner(tiny_models["tiny-llama"], device="cuda", max_batch=128, max_seqs=1, ctx=256)
    sid = r.new_sequence()
    r.kv.reserve(sid, 256)
    r._sync_block_table(sid)
    rows = torch.randn(B, r.resid.shape[1], device="cuda", generator=torch.Generator("cuda").manual_seed(1))

    def inputs(start):
        pos = np.arange(start, start + B)
        z = np.zeros(B, np.int32)
        r._upload(np.stack([pos, r._slots(sid, pos), pos + 1, z, z]).astype(np.int32), np.full(B, 5, np.int64))

    def stage(layer):
        r.resid[:B] = rows
        r.exe.run("attn", layer, B, prefill=True)
        return r.qbuf[:B].clone()

    last = r.cfg.n_layer - 1
    inputs(150)
    r.exe.run("embed", 0, B)
    stage(0)
    want = stage(last)  # behind layer 0 on the same positions
    inputs(0)
    r.exe.run("embed", 0, B)
    other = stage(0), stage(last)
    inputs(150)
    got = stage(last)   # behind a pass on others
    assert torch.equal(got, want)
    assert not torch.equal(got, other[1])
    r.close()
