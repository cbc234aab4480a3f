"""Query blocks left over after whole rounds of the card are shared by four waves each
(`shared_from` in csrc/attn_fwd.hip): launches on both sides of the rule's lines."""
import math

import pytest
import torch

from oracle.attention import masked_attention
from oracle.pooling import pooled_attention
from sparseattnfunctions_amd._kv import kv_list_from_mask
from sparseattnfunctions_amd.utils.attn_pooling_kernel import attn_with_pooling
from sparseattnfunctions_amd.utils.block_sparse_attn_kernel import block_sparse_attention, shares_text_rows

pytestmark = pytest.mark.gpu


# 10 query blocks per head: 704 slots (all shared), 710 items (none), 1 024 slots (none), 1 040
# items (the last of each XCD's range shared), 2 560 items (512 slots shared).
@pytest.mark.parametrize("H", [1, 70, 71, 102, 104, 256])
@pytest.mark.parametrize("dtype,biased", [(torch.bfloat16, False), (torch.bfloat16, True), (torch.float16, False)])
def test_lists_of_every_length(H, dtype, biased):
    print(f"case shared items H={H} {dtype} biased={biased}", flush=True)
    dev, L = torch.device("cuda:0"), 617
    nb = math.ceil(L / 64)
    g = torch.Generator().manual_seed(H)
    q, k, v = (torch.randn(1, H, L, 64, generator=g) for _ in range(3))
    mask = torch.rand(1, H, nb, nb, generator=g) < 0.4
    for m in range(nb):  # the last head's rows keep 0, 1, 2, ... blocks: fewer than the waves, too
        mask[0, H - 1, m] = torch.arange(nb) < m
    q[0, 0] *= 40  # scores of several hundred: the running-maximum pass
    q, k, v = (t.to(dtype) for t in (q, k, v))
    bias = torch.randn(1, H, L, generator=g) if biased else None
    kv = kv_list_from_mask(mask.to(dev), 1, H, nb, nb)
    out = block_sparse_attention(q.to(dev), k.to(dev), v.to(dev), kv, 0.125,
                                 key_bias=None if bias is None else bias.to(dev))
    heads = sorted({(0, h) for h in (0, H - 1, H // 8, H // 2)})
    want = masked_attention(q, k, v, mask, 0.125, key_bias=bias, heads=heads)
    for b, h in heads:
        err = (out[b, h].cpu().double() - want[b, h]).abs()
        assert err.max() <= 2e-2 and err.mean() <= 2e-3, (h, err.max().item())
    assert torch.all(out[0, H - 1, :64] == 0)  # an empty list


@pytest.mark.parametrize("H,block,causal", [(1, 64, False), (70, 32, False), (104, 64, False), (104, 64, True)])
def test_pooled_map(H, block, causal):
    print(f"case shared items pooled H={H} block={block} causal={causal}", flush=True)
    dev, L = torch.device("cuda:0"), 617
    g = torch.Generator().manual_seed(H + block)
    q, k, v = (torch.randn(1, H, L, 64, generator=g).bfloat16() for _ in range(3))
    o, po = attn_with_pooling(q.to(dev), k.to(dev), v.to(dev), causal, 0.125, block)
    for h in {0, H // 8, H - 1}:
        want_o, want_po = pooled_attention(*(t[:, h:h + 1] for t in (q, k, v)), causal, 0.125, block)
        err = (o[:, h:h + 1].cpu().double() - want_o).abs()
        assert err.max() <= 2e-2 and err.mean() <= 2e-3
        assert torch.allclose(po[:, h:h + 1].cpu().double(), want_po, rtol=5e-3, atol=1e-9)


# Text rows in groups of their own before rows of one wave each: remainders shared (the
# text rows apart) and not, and every row a text row.
@pytest.mark.parametrize("H,text", [(71, 2), (74, 3), (90, 2), (104, 1), (72, 10)])
@pytest.mark.parametrize("mode", ["bf16", "fp16", "bias", "fp16 scores", "biased fp16 scores", "row maps"])
def test_shared_text_rows(H, text, mode):
    print(f"case shared text rows H={H} text={text} {mode}", flush=True)
    dev, L = torch.device("cuda:0"), 617
    nb = math.ceil(L / 64)
    g = torch.Generator().manual_seed(H)
    dtype = torch.float16 if mode == "fp16" else torch.bfloat16
    q, k, v = (torch.randn(1, H, L, 64, generator=g) for _ in range(3))
    q[0, 0] *= 40  # the running-maximum pass, and past the fp16 scores' bound
    q, k, v = (t.to(dtype) for t in (q, k, v))
    mask = torch.rand(1, H, nb, nb, generator=g) < 0.4
    mask[:, :, :text] = True
    mask[0, H - 1, 0] = False
    bias = torch.randn(1, H, L, generator=g) if "bias" in mode else None
    rows = torch.randperm(L, generator=g).int() if mode == "row maps" else None
    kv = kv_list_from_mask(mask.to(dev), 1, H, nb, nb)
    kv.row_blocks = 1  # below the rule's lines
    assert shares_text_rows(H * nb, nb, text, kv.row_blocks, 64)
    opts = dict(q_rows=rows.to(dev), o_rows=rows.to(dev)) if rows is not None else {}
    out = block_sparse_attention(q.to(dev), k.to(dev), v.to(dev), kv, 0.125, n_text_blocks=text,
                                 key_bias=None if bias is None else bias.to(dev),
                                 fp16_scores="fp16 scores" in mode or None, **opts)
    heads = sorted({(0, h) for h in (0, H - 1, H // 8, H // 2)})
    if rows is not None:
        out, q = out[:, :, rows.long().to(dev)], q[:, :, rows.long()]
    want = masked_attention(q, k, v, mask, 0.125, key_bias=bias, heads=heads)
    for b, h in heads:
        err = (out[b, h].cpu().double() - want[b, h]).abs()
        assert err.max() <= 2e-2 and err.mean() <= 2e-3, (h, err.max().item())
    assert torch.all(out[0, H - 1, :64] == 0)  # an empty list
