"""Prefill attention at the edges of its 64-key and 32..128-row tiles, masked and whole tiles, any sign of scale,
against 64-bit softmax.  Weights are rounded to bf16 (2^-9 of each) and so is the result; scores are fp32 sums
of D exact products: 2^-8 (sum w |v| + |o|) covers both, and D 2^-24 sum |q k| scale of a score's error is
beneath it at these sizes."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _reference(qkv, lens, Hq, Hkv, D, scale, causal):
    q, k, v = qkv.double().view(sum(lens), -1, D).split([Hq, Hkv, Hkv], 1)
    out, bound, t = [], [], 0
    for n in lens:
        qq = q[t:t + n].transpose(0, 1)
        kk, vv = (x[t:t + n].repeat_interleave(Hq // Hkv, 1).transpose(0, 1).contiguous() for x in (k, v))
        s = (qq @ kk.transpose(1, 2).contiguous()) * scale
        if causal:
            s = s.masked_fill(torch.ones(n, n, device=s.device, dtype=torch.bool).triu(1), float("-inf"))
        w = s.softmax(-1)
        o = w @ vv
        out.append(o.transpose(0, 1).reshape(n, Hq * D))
        bound.append((2.0 ** -8 * (w @ vv.abs() + o.abs())).transpose(0, 1).reshape(n, Hq * D))
        t += n
    return torch.cat(out), torch.cat(bound) + 1e-5


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("Hq,Hkv,D", [(3, 3, 32), (2, 2, 64), (2, 1, 128), (4, 1, 128), (16, 2, 128)])
@pytest.mark.parametrize("sign", [1, -1, 0])
def test_lengths(Hq, Hkv, D, causal, sign):
    from docqa_amd import ops

    assert ops.load_native(build_if_missing=True)
    lens = [1, 31, 33, 63, 0, 64, 65, 127, 128, 129, 200]
    g = torch.Generator(device="cuda").manual_seed(D + Hq)
    qkv = torch.randn(sum(lens), (Hq + 2 * Hkv) * D, device="cuda", generator=g).bfloat16()
    cu = torch.tensor([0] + torch.tensor(lens).cumsum(0).tolist(), dtype=torch.int32, device="cuda")
    got = ops.flash_prefill(qkv, cu, max(lens), Hq, Hkv, D, sign * D ** -0.5, causal)
    want, bound = _reference(qkv, lens, Hq, Hkv, D, sign * D ** -0.5, causal)
    assert bool(((got.double() - want).abs() <= bound).all())


def test_infinite_scores():
    """A key whose scores are -inf has no weight; one whose score is +inf leaves its queries without a number;
    sequences beside them are untouched."""
    from docqa_amd import ops

    assert ops.load_native(build_if_missing=True)
    D, lens = 64, [70, 70, 70]
    g = torch.Generator(device="cuda").manual_seed(1)
    qkv = torch.randn(210, 3 * D, device="cuda", generator=g).bfloat16()
    qkv[:, 0] = 1.0                                  # every query's first element
    qkv[3, D], qkv[3, D + 1:2 * D] = float("-inf"), 0.0
    qkv[73, D], qkv[73, D + 1:2 * D] = float("inf"), 0.0
    cu = torch.tensor([0, 70, 140, 210], dtype=torch.int32, device="cuda")
    got = ops.flash_prefill(qkv, cu, 70, 1, 1, D, 0.125, False)
    want, bound = _reference(qkv, lens, 1, 1, D, 0.125, False)
    assert bool(got[70:140].isnan().all()) and bool(want[70:140].isnan().all())
    for s in (slice(0, 70), slice(140, 210)):
        assert bool(((got[s].double() - want[s]).abs() <= bound[s]).all())
