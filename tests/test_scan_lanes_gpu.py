"""The selective scan with a channel's states spread over lanes: at the edges of its channel tiles and token
blocks, against the recurrence in 64 bits and against the scan in chunks."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("C,N,lens", [(2, 1, [1]), (30, 5, [15, 16, 17, 0, 33]), (62, 16, [1, 2, 31, 32]), (130, 16, [3, 48]),
                                      (8192, 16, [2, 0, 1, 17, 16, 5, 9])])
def test_whole_sequences(C, N, lens, dtype):
    from docqa_amd import ops

    assert ops.load_native(build_if_missing=True)
    T, B, Np, dev = sum(lens), len(lens), (N + 3) // 4 * 4, "cuda"
    g = torch.Generator(device=dev).manual_seed(C + N)
    r = lambda *s: torch.randn(*s, device=dev, generator=g)  # noqa: E731
    x, dt, bc = r(T, C).to(dtype), (r(T, C) * 2 - 1).to(dtype), r(T, 2 * N + 3).to(dtype)
    z = r(T, 2 * C).to(dtype)[:, C:]
    A2, D, db = torch.zeros(C, Np, device=dev), r(C), r(C)
    A2[:, :N] = -torch.exp(torch.rand(C, N, device=dev, generator=g) * 3 - 2) * 1.4427
    S0 = r(B + 1, C, Np)
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=dev)  # noqa: E731
    cu = [0]
    for n in lens:
        cu.append(cu[-1] + n)
    slots = [B - b if b != 1 else -1 for b in range(B)]          # the second sequence has none
    ctx = [7 * (b % 3 == 0) for b in range(B)]
    assert ops.scan_whole(x, dt, N, z, max(lens)) or z.data_ptr() % 8
    S, Sc = S0.clone(), S0.clone()
    args = (x, dt, bc, 1, N + 1, N, z, A2, D, db)
    y = ops.selective_scan(*args, S, i32(slots), i32(cu), i32(ctx), max(lens))
    yc = ops.selective_scan(*args, Sc, i32(slots), i32(cu), i32(ctx), max(lens), 8)
    d = torch.nn.functional.softplus(dt.double() + db.double())
    for b, n in enumerate(lens):
        s = S0[slots[b]].double() if ctx[b] and slots[b] >= 0 else torch.zeros(C, Np, device=dev, dtype=torch.float64)
        # m: the same sums of absolute values, which bound what fp32 rounding (2^-24 a step, a decay's exponent
        # up to 2^5 with 2^-24 of it, ten steps a token's path) can have added up to
        m = s.abs()
        for t in range(cu[b], cu[b + 1]):
            e = torch.exp2(d[t][:, None] * A2.double())[:, :N]
            Bv, Cv = bc[t, 1:N + 1].double(), bc[t, N + 1:2 * N + 1].double()
            u = (d[t] * x[t].double())[:, None] * Bv
            s[:, :N], m[:, :N] = e * s[:, :N] + u, e * m[:, :N] + u.abs()
            gate = torch.nn.functional.silu(z[t].double())
            want = ((s[:, :N] * Cv).sum(1) + D.double() * x[t].double()) * gate
            size = ((m[:, :N] * Cv.abs()).sum(1) + (D.double() * x[t].double()).abs()) * gate.abs()
            tol = size * 2.0 ** -17 + want.abs() * (2.0 ** -8 if dtype == torch.bfloat16 else 0) + 1e-30
            assert bool(((y[t].double() - want).abs() <= tol).all()) and bool(((yc[t].double() - want).abs() <= tol).all())
        if slots[b] >= 0 and n:
            assert bool(((S[slots[b], :, :N].double() - s[:, :N]).abs() <= m[:, :N] * 2.0 ** -17 + 1e-30).all())
        elif slots[b] >= 0:
            assert torch.equal(S[slots[b]], S0[slots[b]])
    assert torch.equal(S[0], S0[0])
