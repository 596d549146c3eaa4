"""The 5..128-row decode products: every tile and epilogue at the edges of its rows, against 64-bit products.

A fp32 sum of K terms of bf16 x bf16 (exact in fp32) differs from the true one by at most K 2^-24 sum |x w|,
whatever its order; a bf16 result by half an ulp (2^-9 of the value, 2^-8 where it rounds up a binade) more."""
import pytest
import torch

pytestmark = pytest.mark.gpu

ROWS = [4, 5, 16, 17, 31, 32, 33, 64, 65, 97, 128]
# N, K, S: one tile of either width; an odd count; more than two workgroups a CU; 128-wide tiles; slices
SHAPES = [(64, 512, 1), (128, 1024, 2), (192, 512, 1), (16640, 512, 1), (24576, 512, 1), (6144, 2048, 4), (320, 4096, 8)]


def _inputs(M, N, K):
    g = torch.Generator(device="cuda").manual_seed(M * 131 + N + K)
    x = torch.randn(M * K + 1, device="cuda", generator=g).bfloat16()[M % 2:][:M * K].view(M, K)   # odd rows: 2-byte offset
    w = (torch.randn(N, K, device="cuda", generator=g) * K ** -0.5).bfloat16()
    return x, w, x.double() @ w.double().t(), K * 2.0 ** -24 * (x.double().abs() @ w.double().abs().t())


@pytest.mark.parametrize("N,K,S", SHAPES)
@pytest.mark.parametrize("M", ROWS)
def test_products(M, N, K, S):
    from docqa_amd import ops

    assert ops.load_native(build_if_missing=True)
    T = torch.ops.docqa
    x, w, want, eps = _inputs(M, N, K)
    P = T.dgemm_partial(x, w, S, 64)
    assert P.shape == (S, M, N) and bool(((P.double().sum(0) - want).abs() <= eps).all())
    y = T.dgemm(x, w, S).double()
    assert bool(((y - want).abs() <= eps + 2.0 ** -8 * want.abs() + 1e-30).all())
    if S == 1:
        ids, vals = T.dgemm_argmax_val(x, w, N - 3)
        y = T.dgemm(x, w, 1)[:, :N - 3].float()
        assert torch.equal(vals.view(-1), y.max(1).values) and torch.equal(ids.view(-1), (y == vals.view(-1, 1)).int().argmax(1))


@pytest.mark.parametrize("N,K", [(64, 512), (16640, 512), (24576, 512), (22400, 512)])
@pytest.mark.parametrize("M", ROWS)
def test_glu(M, N, K):
    from docqa_amd import ops

    assert ops.load_native(build_if_missing=True)
    x, w, want, eps = _inputs(M, N, K)
    a, b = want.view(M, -1, 2, 8)[:, :, 0].reshape(M, -1), want.view(M, -1, 2, 8)[:, :, 1].reshape(M, -1)
    ea, eb = (e.reshape(M, -1) for e in eps.view(M, -1, 2, 8).unbind(2))
    # gate and up are rounded to bf16 before the product; |silu'| <= 1.1, |silu(a)| <= |a|; the result's own rounding
    ra, rb = ea + 2.0 ** -8 * a.abs(), eb + 2.0 ** -8 * b.abs()
    ref = a * torch.sigmoid(a) * b
    bound = 1.1 * ra * (b.abs() + rb) + a.abs() * rb + 2.0 ** -8 * (ref.abs() + ra * b.abs()) + 1e-6
    assert bool(((torch.ops.docqa.dgemm_glu(x, w).double() - ref).abs() <= bound).all())


@pytest.mark.parametrize("M", [17, 64, 128])
def test_activations(M):
    from docqa_amd import ops

    assert ops.load_native(build_if_missing=True)
    for act in ("relu2", "gelu_tanh"):
        x, w, want, eps = _inputs(M - M % 2, 192, 512)
        got = ops.act_linear(x, w, act, decode=True).double()
        ref = want.relu() ** 2 if act == "relu2" else torch.nn.functional.gelu(want, approximate="tanh")
        slope = 2 * (want.abs() + eps) if act == "relu2" else 1.2
        assert bool(((got - ref).abs() <= slope * eps + 2.0 ** -8 * ref.abs() + 1e-5).all())
