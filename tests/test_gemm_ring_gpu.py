"""The encoder GEMM's tiles (csrc/kernels/gemm.hip): K-tile counts around their rings, row remainders,
every epilogue, against 64-bit products."""
import pytest
import torch

from docqa_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N,K", [
    (256 * 128, 256, 64), (256 * 127 + 1, 256, 128), (256 * 85 + 255, 384, 192), (256 * 86 - 31, 384, 320),
    (256 * 28 + 129, 1152, 384), (256 * 14 + 37, 2304, 768), (256 * 43 + 5, 768, 3072),
    # 192-row tiles of the ring, in one round and in more
    (4500, 2304, 64), (192 * 23 - 1, 2304, 192), (192 * 114 + 5, 768, 128), (192 * 14 - 60, 2304, 320), (2689, 2304, 768),
    # 32 x 32 and 64 x 64 tiles (K not a multiple of 128: the latter), 1 .. 6 stages, one row
    (1, 128, 128), (24, 384, 256), (33, 1152, 384), (128, 768, 512), (31, 128, 640), (1, 128, 64), (65, 256, 192),
    (300, 2304, 768), (1000, 768, 3072), (700, 3072, 320), (129, 128, 448),
])
@pytest.mark.parametrize("epi", [ops.EPI_NONE, ops.EPI_BIAS, ops.EPI_BIAS_GELU, ops.EPI_BIAS_RES])
def test_products(M, N, K, epi):
    g = torch.Generator(device="cuda").manual_seed(M + K)

    def rnd(*s, std=1.0):
        return torch.empty(*s, device="cuda", dtype=torch.bfloat16).normal_(0, std, generator=g)

    x, w, b, r = rnd(M, K), rnd(N, K, std=K ** -0.5), rnd(N), rnd(M, N)
    got = ops.linear_fused(x, w, None if epi == ops.EPI_NONE else b, r if epi == ops.EPI_BIAS_RES else None, epi)
    ref = x.double() @ w.double().T
    if epi != ops.EPI_NONE:
        ref += b.double()
    if epi == ops.EPI_BIAS_GELU:
        ref = torch.nn.functional.gelu(ref)
    if epi == ops.EPI_BIAS_RES:
        ref += r.double()
    # one rounding to bf16 of fp32 sums of K products of about 1 / sqrt(K) each
    err = (got.double() - ref).abs()
    assert (err <= 2.0 ** -8 * ref.abs() + 2.0 ** -18 * K ** 0.5).all()


@pytest.mark.parametrize("M", [512, 12 * 1024, 256 * 129])      # 64 x 64, 128 x 128, ring
def test_gelu_tails(M):
    """x Phi(x) keeps its relative precision where 1 + erf(x / sqrt 2) has lost it."""
    v = torch.linspace(-9, 9, M).to(torch.bfloat16)
    x, w = torch.zeros(M, 64, dtype=torch.bfloat16), torch.zeros(256, 64, dtype=torch.bfloat16)
    x[:, 0], w[:, 0] = v, 1
    got = ops.linear_fused(x.cuda(), w.cuda(), torch.zeros(256, device="cuda", dtype=torch.bfloat16), None, ops.EPI_BIAS_GELU)
    d = v.double()
    ref = d * 0.5 * torch.special.erfc(-d / 2 ** 0.5)
    err = (got[:, 0].cpu().double() - ref).abs()
    # half a unit in the last of bf16's 8 bits is at most 2^-8 of the value; fp32 adds 4e-6 < 2^-17
    assert (err <= (2.0 ** -8 + 2.0 ** -17) * ref.abs()).all() and torch.equal(got[:, 0], got[:, 255])
