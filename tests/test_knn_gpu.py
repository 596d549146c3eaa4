"""Flat search on the GPU at the edges of its tiles and pieces (csrc/kernels/knn.hip,
docqa_dist.h) against 64-bit distances."""
import pytest
import torch

from docqa_amd import ops

pytestmark = pytest.mark.gpu


def _check(xb, xq, k, ip, offset=0):
    norms = (xb.float() ** 2).sum(1)
    D, I = ops.knn(xb, norms, xq, k, ip, offset)
    q64 = xq.to(xb.dtype).double()
    dot = q64 @ xb.double().T
    exact = dot if ip else (xq.double() ** 2).sum(1, keepdim=True) + norms.double() - 2 * dot
    n = min(k, xb.shape[0])
    ref = exact.topk(n, 1, largest=ip)[0]
    # fp32: d products of sums below |x| |q| each round by 2^-24, and ||x||^2 + ||q||^2 once more
    tol = 2.0 ** -22 * xb.shape[1] ** 0.5 * float(xb.float().norm(dim=1).max() * xq.norm(dim=1).max() + norms.max())
    assert (D[:, :n].double() - ref).abs().max() <= tol
    got = exact.gather(1, I[:, :n] - offset)
    assert (got - ref).abs().max() <= 2 * tol
    assert all(len(set(r)) == n for r in I[:, :n].tolist())
    assert (I[:, n:] == -1).all()
    assert (D[:, n:].abs() > 3e38).all()


@pytest.mark.parametrize("N,nq,d", [
    (1, 1, 8), (31, 3, 24), (32, 33, 40), (33, 1, 384), (2647, 1, 384), (2647, 256, 384),      # small workgroups
    (32641, 1, 104), (40000, 31, 72), (32700, 33, 40), (17000, 65, 48), (33000, 129, 56),      # each tile width
    (66000, 40, 72), (65537, 64, 40), (70000, 33, 32), (33000, 200, 8),                        # and its row ends
])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("k,ip", [(1, False), (10, True), (64, False)])
def test_knn_tile_edges(N, nq, d, dtype, k, ip):
    if dtype == torch.bfloat16:
        d = d // 16 * 16 + 16
    g = torch.Generator(device="cuda").manual_seed(N + nq)
    xb = torch.randn(N, d, device="cuda", generator=g).to(dtype)
    xq = torch.randn(nq, d, device="cuda", generator=g)
    _check(xb, xq, k, ip, offset=7)


def test_knn_pieces():
    """More distances than the workspace holds: pieces of rows with the best carried along,
    and of queries."""
    g = torch.Generator(device="cuda").manual_seed(0)
    xb, xq = torch.randn(300_000, 8, device="cuda", generator=g), torch.randn(520, 8, device="cuda", generator=g)
    _check(xb, xq, 40, False)
    xb, xq = torch.randn(70, 8, device="cuda", generator=g), torch.randn(1_500_000, 8, device="cuda", generator=g)
    norms = (xb ** 2).sum(1)
    D, I = ops.knn(xb, norms, xq, 1, False, 0)
    ref = torch.cdist(xq, xb) ** 2
    assert (D - ref.min(1, keepdim=True)[0]).abs().max() < 1e-4
    assert (ref.gather(1, I) - D).abs().max() < 1e-4


def test_knn_ties_missing_and_unaligned():
    """Equal rows by the thousand keep the lower id; NaN and infinite rows are never found;
    views that start off a 16-byte boundary are taken."""
    row = torch.randn(1, 64, device="cuda")
    xb = row.repeat(50_000, 1)
    q = torch.randn(5, 64, device="cuda")
    for n in (50_000, 3000):
        D, I = ops.knn(xb[:n], (xb[:n] ** 2).sum(1), q, 20, False, 0)
        assert I.tolist() == [list(range(20))] * 5
    far = torch.randn(300, 64, device="cuda")
    far[::2] = float("nan")
    far[1::4] = float("inf")
    D, I = ops.knn(far, (far ** 2).sum(1), q, 64, False, 0)
    keep = [i for i in range(300) if i % 2 and i % 4 != 1]
    assert all(set(r) <= set(keep) and len(set(r)) == 64 for r in I.tolist())
    flat = torch.randn(200 * 64 + 1, device="cuda")
    xb = flat[1:].view(200, 64)
    _check(xb, torch.randn(4 * 64 + 1, device="cuda")[1:].view(4, 64), 3, False)


@pytest.mark.parametrize("n,nq,d", [(1, 1, 8), (768, 64, 768), (1024, 33, 768), (4096, 1000, 40), (70, 9000, 1280)])
def test_fp32_product(n, nq, d):
    x, w = torch.randn(nq, d, device="cuda"), torch.randn(n, d, device="cuda")
    got = ops.fp32_matmul_nt(x, w).double()
    ref = x.double() @ w.double().T
    assert (got - ref).abs().max() <= 2.0 ** -22 * d ** 0.5 * float(x.norm(dim=1).max() * w.norm(dim=1).max())


def test_ivfpq_equal_distances_by_the_thousand():
    """Every stored vector at one distance: partial lists whose merge holds more equal entries
    than its buffer still give k different vectors."""
    from docqa_amd.index.ivfpq import IVFPQIndex

    idx = IVFPQIndex(64, 64, 16, device="cuda")
    idx.centroids, idx.pq = torch.zeros(64, 64, device="cuda"), torch.zeros(16, 256, 4, device="cuda")
    n = 64 * 100
    idx.codes = torch.randint(0, 256, (n, 16), device="cuda", dtype=torch.uint8)
    idx.ids, idx.ntotal = torch.arange(n, device="cuda") + 5, n
    idx.list_off = torch.arange(65, device="cuda") * 100
    q = torch.randn(3, 64, device="cuda")
    for k in (1, 64):
        D, I = idx.search(q, k, nprobe=64)
        assert (D - (q ** 2).sum(1, keepdim=True)).abs().max() < 1e-3       # fp16 tables of zeros: fp32 rounding
        assert all(len(set(r)) == k and min(r) >= 5 and max(r) < n + 5 for r in I.tolist())


@pytest.mark.parametrize("d,dtype", [(37, torch.float32), (64, torch.float32), (768, torch.bfloat16), (10, torch.bfloat16)])
@pytest.mark.parametrize("metric", ["l2", "ip"])
def test_refine_widths(d, dtype, metric):
    from docqa_amd.index.refine import RefineFlat

    x = torch.randn(500, d, device="cuda").to(dtype)
    q = torch.randn(5, d, device="cuda")
    cand = torch.stack([torch.randperm(500, device="cuda")[:57] for _ in range(5)])
    cand[:, 3] = -1
    D, I = ops._native().refine_flat(x, q, cand, 9, metric == "ip")
    D2, I2 = RefineFlat(None, x, metric).rerank(q, cand, 9)
    # (sums of d products in another order; random distances are further apart than that)
    assert torch.equal(I, I2) and torch.allclose(D, D2, rtol=1e-4, atol=1e-4)


def test_row_norms():
    x = torch.randn(1001, 37, device="cuda")
    assert torch.allclose(ops.row_norms(x), (x ** 2).sum(1), rtol=1e-5)


@pytest.mark.parametrize("ip", [False, True])
@pytest.mark.parametrize("nq,N", [(150, 33000), (50, 66000)])
def test_knn_values_at_the_ends(nq, N, ip):
    """Wide batches multiply fp32 as bf16 parts: rows and queries of infinities, NaN, values beyond bf16's largest,
    products beyond fp32's and tiny ones come out as the narrow batches' fp32 products make them."""
    g = torch.Generator(device="cuda").manual_seed(nq)
    d = 40
    xb, xq = torch.randn(N, d, device="cuda", generator=g), torch.randn(nq, d, device="cuda", generator=g)
    inf, big = float("inf"), 3.4e38
    xb[5, 3], xb[40, 7], xb[41], xb[100, 0], xb[N - 1, 39] = inf, -inf, float("nan"), big, inf
    xb[200], xb[300, :20], xb[300, 20:] = 1e30, 1e30, -1e30
    xb[400] *= 1e-30
    xq[1, 3], xq[2], xq[3, 0], xq[4], xq[nq - 1, 5] = -inf, 1e20, big, 1e-30, float("nan")
    norms = (xb ** 2).sum(1)
    D, I = ops.knn(xb, norms, xq, 20, ip, 0)
    parts = [ops.knn(xb, norms, xq[i:i + 25], 20, ip, 0) for i in range(0, nq, 25)]
    Dn, In = torch.cat([p[0] for p in parts]), torch.cat([p[1] for p in parts])
    assert torch.equal(D.isfinite(), Dn.isfinite()) and torch.equal(I < 0, In < 0)
    assert torch.equal(D[~D.isfinite()].nan_to_num(1.0), Dn[~Dn.isfinite()].nan_to_num(1.0))
    # 40 products and the norms, each rounded by 2^-24 on either side
    size = (xq.double() ** 2).sum(1, keepdim=True).nan_to_num(0, 0, 0) + 2000 + Dn.double().abs().nan_to_num(0, 0, 0)
    assert bool(((D.double() - Dn.double()).abs().nan_to_num(0, 0, 0) <= 40 * 2.0 ** -22 * size).all())
    ordinary = torch.arange(5, nq - 1, device="cuda")
    assert torch.equal((I == 400)[ordinary], (In == 400)[ordinary])
