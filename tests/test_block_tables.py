"""Block-table rows of several sequences in one upload: after every admission the device's rows are the host's."""
import numpy as np
import pytest

from ollama_operator_amd.engine.kv_cache import OutOfBlocks
from ollama_operator_amd.engine.runner import Runner
from ollama_operator_amd.engine.sampling import SamplingOptions

O = SamplingOptions(temperature=0)


def same(r, sids):
    t = r.d_block_table.cpu().numpy()
    for sid in sids:
        s = r.kv.seqs[sid]
        assert s.blocks and list(t[s.row, :len(s.blocks)]) == s.blocks, sid


def admit(r, lens, rng):
    sids = [r.new_sequence() for _ in lens]
    items = []
    for sid, n in zip(sids, lens):
        p = [1] + [int(x) for x in rng.integers(3, 500, n - 1)]
        items.append((sid, 0, p, O, p, 0))
    r.admit_many(items)
    return sids


@pytest.mark.parametrize("words", [None, 0], ids=["one copy", "row by row"])
@pytest.mark.parametrize("device", ["cpu", pytest.param("cuda", marks=pytest.mark.gpu)])
def test_rows_follow_admissions(tiny_models, device, words):
    """Sequences between the admitted ones keep their rows; freed rows are taken again; rows grow in a step."""
    r = Runner(tiny_models["tiny-llama"], device=device, max_batch=64, max_seqs=8, ctx=128)
    if words is not None and r._ring is not None:
        r._ring.words = words
    rng = np.random.default_rng(3)
    a = admit(r, [20, 3, 30, 2], rng)
    same(r, a)
    for sid in a[::2]:
        r.free_sequence(sid)
    live = a[1::2]
    b = admit(r, [17, 16, 1, 30], rng)  # rows around those that run on, other blocks than before
    same(r, live + b)
    sids = live + b
    out = r.step_entries([(sid, [5, 6], [1]) for sid in sids])
    assert out.shape[0] == len(sids)
    same(r, sids)
    r.recompose([(O, [1, 7], 0, 0)] * len(sids), [7] * len(sids))
    for _ in range(3):  # some of the rows cross into a new block
        r.decode_batch(sids, [r.kv.seqs[s].length for s in sids])
        for s in sids:
            r.kv.seqs[s].tokens.append(7)
    same(r, sids)


@pytest.mark.parametrize("device", ["cpu", pytest.param("cuda", marks=pytest.mark.gpu)])
def test_a_refused_row_leaves_the_others_in_place(tiny_models, device):
    """What was reserved before a later sequence found no blocks is on the device: nothing asks for it again."""
    r = Runner(tiny_models["tiny-llama"], device=device, max_batch=64, max_seqs=4, ctx=128)
    rng = np.random.default_rng(4)
    a = admit(r, [r.block_size, 2 * r.block_size, r.block_size], rng)
    last = r.kv.seqs[a[-1]]
    r.kv.max_blocks = 5
    last.blocks += [r.kv.alloc.alloc() for _ in range(4)]  # at the limit of a sequence
    with pytest.raises(OutOfBlocks):
        r.decode_batch(a, [r.block_size, 2 * r.block_size, 5 * r.block_size])
    same(r, a[:2])
    assert len(r.kv.seqs[a[0]].blocks) > 1
    with pytest.raises(OutOfBlocks):
        r.admit_many([(a[0], r.block_size, [5] * 3, O, [1] * r.block_size, 0), (a[2], r.block_size, [5] * 90, O, [1] * r.block_size, 0)])
    same(r, a[:2])


@pytest.mark.parametrize("device", ["cpu", pytest.param("cuda", marks=pytest.mark.gpu)])
def test_a_reservation_that_fails_midway_leaves_its_blocks_on_the_device(tiny_models, device):
    """The pool runs out within a row's reservation: the blocks it took are the row's, and a step that needs no more goes through."""
    r = Runner(tiny_models["tiny-llama"], device=device, max_batch=64, max_seqs=4, ctx=128, kv_tokens=6 * 16)
    assert r.block_size == 16
    a = admit(r, [16, 16, 16], np.random.default_rng(5))
    poss = [16, 16, 16]
    r.recompose([(O, [1, 7], 0, 0)] * 3, [7] * 3)
    r.d_block_table[:] = -1  # whatever is not uploaded again is no page
    for sid in a:
        r._sync_block_table(sid)
    with pytest.raises(OutOfBlocks):
        r.decode_batch(a, poss)  # asks for four blocks a row: three are left
    s = r.kv.seqs[a[0]]
    assert len(s.blocks) > 1 and r.kv.alloc.n_free == 0
    same(r, a)
    r.free_sequence(a[2])
    with pytest.raises(OutOfBlocks):
        r.admit_many([(a[1], 16, [5] * 40, O, [1] * 16, 0), (r.new_sequence(), 0, [5] * 60, O, [5] * 60, 0)])
    same(r, a[:2])
    with pytest.raises(OutOfBlocks):
        r.step_entries([(a[1], [5] * 90, [1])])
    same(r, a[:2])
