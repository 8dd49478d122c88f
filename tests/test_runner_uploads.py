"""Uploads of a runner's step inputs and sampler state: what arrives on the device, for few and many rows."""
import numpy as np
import pytest
import torch

from ollama_operator_amd.engine.runner import HIST_CAP, Runner
from ollama_operator_amd.engine.sampling import SamplingOptions
from ollama_operator_amd.gguf.constants import FileType
from ollama_operator_amd.models.config import preset
from ollama_operator_amd.models.random_init import write_random_gguf

def make(tmp_path_factory, device):
    path = str(tmp_path_factory.mktemp("m") / "tiny.gguf")
    write_random_gguf(path, preset("tiny-llama"), FileType.MOSTLY_Q4_0, seed=3)
    r = Runner(path, device=device, max_batch=80, max_seqs=3)
    yield r
    r.close()


@pytest.fixture(scope="module")
def runner(tmp_path_factory):
    yield from make(tmp_path_factory, "cuda:0")


@pytest.fixture(scope="module")
def cpu_runner(tmp_path_factory):
    yield from make(tmp_path_factory, "cpu")


ROWS = [(1, 0), (1, 79), (3, 5), (64, 0), (65, 2), (80, 0)]


@pytest.mark.gpu
@pytest.mark.parametrize("n,first", ROWS)
def test_sampler_rows(runner, n, first):
    check_sampler_rows(runner, n, first)


@pytest.mark.parametrize("n,first", ROWS)
def test_sampler_rows_cpu(cpu_runner, n, first):
    check_sampler_rows(cpu_runner, n, first)


def check_sampler_rows(r, n, first):
    rng = np.random.default_rng(n + first)
    first = min(first, 80 - n)
    r.s_temp.fill_(-1.0)
    rows = [(SamplingOptions(temperature=0.5 + i, top_k=i, top_p=0.25 * (i % 4), min_p=0.01 * i, repeat_penalty=1.0 + i,
                             repeat_last_n=2 * i, presence_penalty=-0.5 * i, frequency_penalty=0.125 * i),
             rng.integers(-2, 500, [0, 1, 255, 256, 300][i % 5]).tolist(), [7, (1 << 64) - 1, 1 << 63, (1 << 63) - 1][i % 4], 3 * i)
            for i in range(n)]
    r._set_samplers(rows, first)
    for i, (o, hist, seed, step) in enumerate(rows):
        b = first + i
        got = [float(t[b]) for t in (r.s_temp, r.s_topp, r.s_minp, r.s_rpen, r.s_ppen, r.s_fpen)]
        want = [np.float32(v) for v in (o.temperature, o.top_p, o.min_p, o.repeat_penalty, o.presence_penalty, o.frequency_penalty)]
        assert got == [float(v) for v in want]
        h = [t for t in hist if t >= 0][-HIST_CAP:]
        assert [int(t[b]) for t in (r.s_topk, r.s_lastn, r.s_step, r.s_hcount)] == [o.top_k, o.repeat_last_n, step, len(h)]
        assert int(r.s_seed[b]) % (1 << 64) == seed
        assert r.s_hist[b].tolist() == h + [0] * (HIST_CAP - len(h))
    others = [b for b in range(80) if not first <= b < first + n]
    assert all(float(r.s_temp[b]) == -1.0 for b in others)
    for o, hist, seed in ((dict(temperature=1e300), [], 0), (dict(top_k=1 << 31), [], 0), (dict(repeat_last_n=-(1 << 31) - 1), [], 0),
                          ({}, [1, 1 << 31], 0), ({}, [], 1 << 64), ({}, [], -(1 << 63) - 1)):
        with pytest.raises(RuntimeError):  # what the arrays cannot hold
            r._set_samplers([(SamplingOptions(**o), hist, seed, 0)])


@pytest.mark.gpu
@pytest.mark.parametrize("B,nt", [(1, 0), (1, 1), (79, 79), (80, 80), (0, 5), (3, 0)])
def test_step_inputs(runner, B, nt):
    """Uploads in a row that the device has not read yet: each arrives whole and in order."""
    r, rng = runner, np.random.default_rng(B)
    seen = []
    for _ in range(20):  # more than the ring's slots
        arr, toks = rng.integers(0, 1 << 30, (5, B)).astype(np.int32), rng.integers(0, 500, nt).astype(np.int32)
        r._upload(arr, toks if nt else None)
        seen.append((arr, toks, r.d_step.clone()))
    torch.cuda.synchronize()
    for arr, toks, got in seen:
        assert np.array_equal(got[:5, :B].cpu().numpy(), arr)
        assert got[5, :nt].tolist() == toks.tolist()
