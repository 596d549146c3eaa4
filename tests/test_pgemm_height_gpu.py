"""The prefill GEMM's tile heights (160, 192, 224, 256 rows, by how the tiles fill the chip) and epilogues at
the edges of their rows, against 64-bit products: a fp32 sum of K exact terms is off by at most
K 2^-24 sum |x w|, a bf16 result by 2^-8 of its value more."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N,K", [(M, 28672, 256) for M in (320, 321, 384, 385, 448, 449, 512, 513)] +
                         [(1, 256, 256), (159, 512, 512), (160, 512, 512), (161, 512, 512), (1300, 1024, 512)])
def test_products(M, N, K):
    from docqa_amd import ops

    assert ops.load_native(build_if_missing=True)
    T = torch.ops.docqa
    g = torch.Generator(device="cuda").manual_seed(M + N)
    x = torch.randn(M, K, device="cuda", generator=g).bfloat16()
    w = (torch.randn(N, K, device="cuda", generator=g) * K ** -0.5).bfloat16()
    want = x.double() @ w.double().t()
    eps = K * 2.0 ** -24 * (x.double().abs() @ w.double().abs().t())
    for S in (1, 2):
        P = T.pgemm_partial(x, w, S)
        assert P.shape == (S, M, N) and bool(((P.double().sum(0) - want).abs() <= eps).all())
    P = T.pgemm_partial(x, w, 1)[0]
    # the other epilogues are these sums', rounded and activated
    assert torch.equal(T.pgemm(x, w, 0), P.bfloat16())
    assert torch.equal(T.pgemm(x, w, 3), (P.clamp_min(0) ** 2).bfloat16())
    ref = torch.nn.functional.gelu(P.double(), approximate="tanh")
    assert bool(((T.pgemm(x, w, 4).double() - ref).abs() <= 2.0 ** -8 * ref.abs() + 1e-5).all())
    gate, up = P.bfloat16().double().view(M, -1, 2, 8).unbind(2)
    ref = (gate * torch.sigmoid(gate) * up).reshape(M, -1)
    assert bool(((T.pgemm(x, w, 1).double() - ref).abs() <= 2.0 ** -8 * ref.abs() + 1e-5).all())
