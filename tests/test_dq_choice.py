"""Tile and K split of the dequantising prompt products (csrc/kernels/gemm_dq.hip): what is forced is what runs, or an error."""
import pytest

from ollama_operator_amd.gguf import GGMLType
from ollama_operator_amd.ops import native

Q4K, Q6K = int(GGMLType.Q4_K), int(GGMLType.Q6_K)
GWS = 3 << 27


@pytest.fixture(autouse=True)
def _auto():
    yield
    native().set_dq_tuning(-1, 0)


@pytest.mark.parametrize("M,N,K", [(65, 1024, 4096), (509, 28672, 4096), (2048, 22016, 4096), (2048, 4096, 11008)])
@pytest.mark.parametrize("qt", [Q4K, Q6K])
def test_forced_choices_run(qt, M, N, K):
    C = native()
    for tile in range(4):
        for sk in (1, 2, 3, 5, 7):  # also splits that the rule never takes, and more blocks than it allows
            C.set_dq_tuning(tile, sk)
            assert C.dq_choice(qt, M, N, K, GWS) == (tile, sk)
        C.set_dq_tuning(tile, 0)
        assert C.dq_choice(qt, M, N, K, GWS)[0] == tile
    C.set_dq_tuning(-1, 0)
    tile, sk = C.dq_choice(qt, M, N, K, GWS)
    assert 0 <= tile <= 3 and sk in (1, 2, 3, 4, 6, 8) and sk * M * N <= GWS


@pytest.mark.parametrize("K,gws,sk", [(512, GWS, 3), (4096, 0, 2), (4096, 3 * 65 * 1024 - 1, 3)])
def test_a_forced_split_that_does_not_fit_is_refused(K, gws, sk):
    C = native()
    C.set_dq_tuning(0, sk)
    with pytest.raises(RuntimeError, match="splits of K"):
        C.dq_choice(Q4K, 65, 1024, K, gws)
    C.set_dq_tuning(0, 1)
    assert C.dq_choice(Q4K, 65, 1024, K, gws) == (0, 1)
    C.set_dq_tuning(-1, 0)
    C.dq_choice(Q4K, 65, 1024, K, gws)
