"""Routed experts of a prompt in one launch per matrix (csrc/kernels/gemm_dq_moe.hip): every weight type, few and many rows,
tiles that end inside an expert's rows."""
import numpy as np
import pytest

from ollama_operator_amd.engine.runner import Runner
from ollama_operator_amd.gguf.constants import FileType
from ollama_operator_amd.models.config import preset
from ollama_operator_amd.models.random_init import write_random_gguf
from ollama_operator_amd.ops import native

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ft,n_ff,rows,n_embd", [
    (FileType.MOSTLY_Q4_K_M, 8192, 260, 512), (FileType.MOSTLY_Q4_K_M, 3840, 577, 512), (FileType.MOSTLY_Q5_K_S, 8192, 257, 512),
    (FileType.MOSTLY_Q4_0, 8192, 321, 512), (FileType.MOSTLY_Q8_0, 3840, 640, 512), (FileType.MOSTLY_Q6_K, 8192, 300, 512),
    (FileType.MOSTLY_Q4_K_M, 1024, 17, 512), (FileType.MOSTLY_Q4_0, 1280, 129, 512),
    # widths that are no multiple of 256 (padded K) nor of 128 (the last columns of an expert's tile), a full portion among them
    (FileType.MOSTLY_Q4_0, 1056, 640, 576), (FileType.MOSTLY_Q8_0, 1056, 101, 576), (FileType.MOSTLY_Q4_0, 2144, 40, 1088),
    (FileType.MOSTLY_Q8_0, 1120, 640, 1088),
    # up to 128 rows an expert on average (tiles in halves): at the limit some experts have more, the second half of a tile a few
    (FileType.MOSTLY_Q4_K_M, 1024, 256, 512), (FileType.MOSTLY_Q5_K_S, 1280, 250, 512), (FileType.MOSTLY_Q6_K, 1280, 256, 512),
    (FileType.MOSTLY_Q6_K, 1024, 33, 512), (FileType.MOSTLY_Q8_0, 1056, 256, 576), (FileType.MOSTLY_Q4_0, 1056, 255, 576)])
def test_grouped_experts(tmp_path, ft, n_ff, rows, n_embd):
    """Against float32 on the CPU, beside the path that is taken with these kernels switched off: both round the same two
    operands to fp16 and add in float32, so neither may be further from float32 than the other by more than the order of sums
    and the atomics' order explain (a fifth)."""
    path = str(tmp_path / "m.gguf")
    heads = dict(n_head=8) if n_embd == 512 else dict(n_head=n_embd // 64, n_head_kv=1)
    write_random_gguf(path, preset("tiny-mixtral", n_embd=n_embd, n_ff=n_ff, n_layer=1, ctx_len=768, **heads), ft, seed=int(ft))
    rng = np.random.default_rng(rows)
    toks = [1] + [int(x) for x in rng.integers(3, 500, rows - 1)]
    C = native()

    def logits(device):
        r = Runner(path, device=device, max_batch=640, max_seqs=2, ctx=704)
        C.reset_launch_counts()
        r.prefill(r.new_sequence(), toks)
        out = r.logits[0, :r.cfg.n_vocab].double().cpu()
        n = C.launch_counts() if device == "cuda" else None
        r.close()
        return out, n

    want, _ = logits("cpu")
    on = C.dq_gemm_enabled()
    C.set_dq_gemm(1)
    got, n = logits("cuda")
    C.set_dq_gemm(0)
    old, m = logits("cuda")
    C.set_dq_gemm(int(on))
    # gate|up and down: dq_gemm; q|k|v (one launch, or v apart) and o: the same tiles from 65 rows, gemm_rows.hip below
    assert n["gemm_tile"] == 0, n
    assert n["dq_gemm"] >= 4 and n["gemm_rows"] == 0 if rows > 64 else n["dq_gemm"] == 2 and n["gemm_rows"] >= 2, n
    assert m["dq_gemm"] == m["gemm_rows"] == 0, m
    err = lambda v: float((v - want).norm() / want.norm())  # noqa: E731
    print(err(got), err(old))
    assert err(got) < 1.2 * err(old) + 1e-4


def test_grouped_experts_need_no_library(tmp_path, monkeypatch):
    """The grouped launches run for a runner of a few rows, with the library path switched off or on, and bring no workspace of
    the library's along; experts they leave (gate and up of under 2,048 rows) keep theirs."""
    C = native()

    def load(n_ff, max_batch, lib):
        path = str(tmp_path / f"m{n_ff}.gguf")
        write_random_gguf(path, preset("tiny-mixtral", n_embd=512, n_ff=n_ff, n_layer=1, n_head=8, ctx_len=512), FileType.MOSTLY_Q4_0,
                          seed=1)
        old = C.moe_lib_min_m()
        C.set_moe_lib_min_m(lib)
        try:
            r = Runner(path, device="cuda", max_batch=max_batch, max_seqs=2, ctx=512)
            C.reset_launch_counts()
            r.prefill(r.new_sequence(), list(range(3, 43)))
            return C.launch_counts()["dq_gemm"], r.w16 is not None, r.yws is not None, r.moe_y.numel() if r.moe_y is not None else 0
        finally:
            C.set_moe_lib_min_m(old)

    for max_batch, lib in ((64, 256), (512, 256), (64, 0)):
        assert load(1024, max_batch, lib) == (2, False, False, max_batch * 2 * 512)
    assert load(512, 512, 256) == (0, True, True, 0)
    assert load(512, 512, 0) == (0, False, False, 0)
