"""The encoder stack issued by one call computes what the op-by-op path does, byte for byte: positions taken from
the sequence starts on the device, and for few rows the normalisations inside the products behind them."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("preset", ["tiny-bert", "minilm-l6", "bge-base"])
@pytest.mark.parametrize("lengths", [[1], [24], [0, 3, 0, 0, 70, 1, 0], [2] * 63 + [5], [1, 3] * 40, [100, 124], [120] * 4, [0, 1, 2] * 1500],
                         ids=["one", "question", "empty", "64", "80", "224", "480", "4500"])
def test_stack_equals_its_ops(preset, lengths):
    from docqa_amd import ops
    from docqa_amd.models.bert import BertConfig, BertEncoder, pack, packed_positions

    enc = BertEncoder(BertConfig.preset(preset), device="cuda", seed=5)
    g = torch.Generator().manual_seed(len(lengths))
    ids, cu, longest = pack([torch.randint(0, 4000, (n,), generator=g).tolist() for n in lengths], 128, "cuda")
    assert ids.shape[0] == sum(lengths) and cu.tolist()[-1] == sum(lengths)
    pos = packed_positions(cu, ids.shape[0])
    got = enc.hidden_states(ids, cu, longest)
    given = enc.hidden_states(ids, cu, longest, pos.flip(0).contiguous())
    for want_pos, have in ((pos, got), (pos.flip(0).contiguous(), given)):
        h = ops.bert_embed_ln(ids, want_pos, None, enc.wte, enc.wpe, enc.wtt, enc.emb_g, enc.emb_b, enc.cfg.eps)
        for L in enc.layers:
            qkv = ops.linear_fused(h, L["qkv_w"], L["qkv_b"], None, ops.EPI_BIAS)
            a = ops.flash_prefill(qkv, cu, longest, enc.cfg.heads, enc.cfg.heads, enc.cfg.head_dim, enc.scale, False)
            h = ops.layernorm(ops.linear_fused(a, L["o_w"], L["o_b"], h, ops.EPI_BIAS_RES), None, L["ln1_g"], L["ln1_b"],
                              enc.cfg.eps)
            u = ops.linear_fused(h, L["up_w"], L["up_b"], None, ops.EPI_BIAS_GELU)
            h = ops.layernorm(ops.linear_fused(u, L["down_w"], L["down_b"], h, ops.EPI_BIAS_RES), None, L["ln2_g"],
                              L["ln2_b"], enc.cfg.eps)
        assert torch.equal(have, h)


def test_pack_takes_what_torch_takes():
    from docqa_amd.models.bert import pack

    ids, cu, longest = pack([[1, 2, 3], [], [True, torch.tensor(7)], [2.0, 5]], 2, "cpu")
    assert ids.tolist() == [1, 2, 1, 7, 2, 5] and cu.tolist() == [0, 2, 2, 4, 6] and longest == 2
    assert ids.dtype == cu.dtype == torch.int32
    assert [t.tolist() for t in pack([], 8, "cpu")[:2]] == [[], [0]]


@pytest.mark.parametrize("H", [8, 384, 512, 520, 1024])
def test_pool_lengths(H):
    from docqa_amd import ops

    lens = [1, 0, 7, 8, 33, 2, 70]
    cu = torch.tensor([0] + torch.tensor(lens).cumsum(0).tolist(), dtype=torch.int32, device="cuda")
    h = torch.randn(sum(lens), H, device="cuda", dtype=torch.bfloat16)
    for mean in (True, False):
        got = ops.pool_l2(h, cu, mean, False)
        for b, n in enumerate(lens):
            x = h[int(cu[b]):int(cu[b]) + n].double()
            want = (x.mean(0) if mean else x[0]) if n else torch.zeros(H, device="cuda", dtype=torch.float64)
            # sums of n bf16 values in fp32, once divided
            assert bool(((got[b].double() - want).abs() <= (n + 2) * 2.0 ** -24 * (x.abs().mean(0) if n else 0)).all())
