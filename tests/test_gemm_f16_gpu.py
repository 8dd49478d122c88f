"""fp16 weights times prompt-sized activations (csrc/kernels/gemm_f16.hip): every tile, the last rows and columns of a matrix,
norms and epilogues."""
import pytest
import torch

from test_kernels_gpu import C, S, rel

pytestmark = pytest.mark.gpu
p = lambda t: t.data_ptr() if t is not None else 0  # noqa: E731


def run(w, K, x, y, epi=0, norm=0, nw=None, nb=None, bias=None, row_offset=0):
    B = x.shape[0]
    xws = torch.empty(B * w.shape[1], device="cuda", dtype=torch.float16)
    C().reset_launch_counts()
    C().gemv((p(w), 0, 0, 0, w.shape[0], K, 1), B, p(x), x.shape[1], norm, p(nw), p(nb), 1e-5, epi, p(y), y.shape[1], p(bias), row_offset,
             dict(xws=p(xws), xws_elems=xws.numel()), S())
    torch.cuda.synchronize()
    assert C().launch_counts()["dq_gemm"] == 1


@pytest.mark.parametrize("B,N,K", [(128, 1, 64), (129, 70, 588), (577, 1024, 1024), (577, 3072, 1024), (576, 4096, 4096), (2000, 4100, 512),
                                   (4099, 8200, 256), (300, 130, 4360)])
def test_gemm_f16(B, N, K):
    """Activations are rounded to fp16 (2^-11 of each, in quadrature over K) and added in float32: against float32 products of
    the rounded operands only the order of the sums is left, 2^-24 sqrt(K) of the result's size and the matrix cores' own
    rounding; 2e-5 holds both. Weights come with K padded to 256 with zeros."""
    torch.manual_seed(N)
    Kp = (K + 255) // 256 * 256
    w = torch.zeros(N, Kp, device="cuda", dtype=torch.float16)
    w[:, :K] = torch.randn(N, K, device="cuda") / K ** 0.5
    x, bias = torch.randn(B, K, device="cuda"), torch.randn(N, device="cuda")
    z = x.half().double() @ w[:, :K].double().T + bias.double()
    y = torch.full((B, N + 3), 9.0, device="cuda")
    run(w, K, x, y, bias=bias)
    assert rel(y[:, :N], z.float()) < 2e-5 and bool((y[:, N:] == 9.0).all())
    y = y0 = torch.randn(B, N, device="cuda")
    y = y0.clone()
    run(w, K, x, y, epi=1, bias=bias)
    assert rel(y, (z + y0.double()).float()) < 2e-5
    y = torch.empty(B, N, device="cuda")
    run(w, K, x, y, epi=6, bias=bias)
    assert rel(y, torch.nn.functional.gelu(z).float()) < 2e-5
    run(w, K, x, y, epi=7, bias=bias)
    assert rel(y, (z * torch.sigmoid(1.702 * z)).float()) < 2e-5
    nw, nb = torch.rand(K, device="cuda") + 0.5, torch.randn(K, device="cuda")
    run(w, K, x, y, norm=2, nw=nw, nb=nb, bias=bias)  # the normed rows are rounded after the norm: 2^-11 each
    h = torch.nn.functional.layer_norm(x, (K,), nw, nb, 1e-5)
    assert rel(y, (h.double() @ w[:, :K].double().T + bias.double()).float()) < 1e-3
    if N % 2 == 0:
        y = torch.empty(B, N // 2, device="cuda")
        run(w, K, x, y, epi=2)
        g = z - bias.double()
        assert rel(y, (torch.nn.functional.silu(g[:, 0::2]) * g[:, 1::2]).float()) < 4e-5


@pytest.mark.parametrize("B,N,K,at", [(128, 70, 588, 5), (577, 1024, 1024, 2048), (300, 130, 4360, 1)])
def test_rows_of_a_concatenated_matrix(B, N, K, at):
    """The matrix is rows at .. at + N - 1 of a concatenated one: outputs and biases sit there, the columns beside them stay.
    Tolerance as above."""
    torch.manual_seed(at)
    w = torch.zeros(N, (K + 255) // 256 * 256, device="cuda", dtype=torch.float16)
    w[:, :K] = torch.randn(N, K, device="cuda") / K ** 0.5
    x, bias = torch.randn(B, K, device="cuda"), torch.randn(at + N, device="cuda")
    y = torch.full((B, at + N + 3), 9.0, device="cuda")
    run(w, K, x, y, bias=bias, row_offset=at)
    z = x.half().double() @ w[:, :K].double().T + bias[at:].double()
    assert rel(y[:, at:at + N], z.float()) < 2e-5
    assert bool((y[:, :at] == 9.0).all()) and bool((y[:, at + N:] == 9.0).all())
