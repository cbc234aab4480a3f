"""Query blocks left over after whole rounds of the card are shared by four waves each
(`shared_from` in csrc/attn_fwd.hip): launches on both sides of the rule's lines."""
import ctypes
import math

import pytest
import torch

from oracle.attention import masked_attention
from oracle.pooling import pooled_attention
from sparseattnfunctions_amd import _lib
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


# Remainders whose short lists keep one wave each (`share_min`): 704 of 704 slots (from 20 tiles on),
# 416 of 1 440 (16), 512 of 2 560 (8) and 320 of 2 368 (8), in groups of both kinds; and lists that
# are all shorter, decided by their width.
@pytest.mark.parametrize("H,nkb", [(70, 24), (144, 24), (256, 24), (236, 24), (70, 19), (144, 8), (256, 7)])
@pytest.mark.parametrize("mode", ["bf16", "bias", "fp16", "plain order", "text rows"])
def test_short_lists_keep_one_wave(H, nkb, mode):
    print(f"case shared items short lists H={H} nkb={nkb} {mode}", flush=True)
    dev, Lq, Lk = torch.device("cuda:0"), 617, 64 * nkb - 5
    nqb = math.ceil(Lq / 64)
    g = torch.Generator().manual_seed(H + nkb)
    dtype = torch.float16 if mode == "fp16" else torch.bfloat16
    q, k, v = (torch.randn(1, H, L, 64, generator=g).to(dtype) for L in (Lq, Lk, Lk))
    # heads of empty and short lists, of long ones, and of both in one group
    longest = torch.tensor([3, nkb, 12, 0])[torch.arange(H) % 4]
    count = (torch.rand(H, nqb, generator=g) * (longest[:, None] + 1)).long()
    count[:, 4] = longest
    mask = torch.arange(nkb) < count[..., None].clamp(max=nkb)
    text = 1 if mode == "text rows" else 0
    mask[:, :text] = True
    mask = mask[None]
    bias = torch.randn(1, H, Lk, generator=g) if mode == "bias" else None
    kv = kv_list_from_mask(mask.to(dev), 1, H, nqb, nkb)
    if text:
        kv.row_blocks = 0.1
    out = torch.full((1, H, Lq, 64), math.nan, dtype=dtype, device=dev)
    if mode == "plain order":  # no work order: the items by index
        lib, st = _lib.load(), [_lib.i64(*t.to(dev).stride()[:3]) for t in (q, k, v)]
        d = [t.to(dev) for t in (q, k, v)]
        _lib.check(lib.sa_block_sparse_fwd(d[0].data_ptr(), st[0], d[1].data_ptr(), st[1], d[2].data_ptr(), st[2],
                                           out.data_ptr(), st[0], 1, H, Lq, Lk, 64, kv.idx.data_ptr(),
                                           kv.cnt.data_ptr(), kv.max_cnt, None, None, 0.125, None, 0,
                                           _lib.stream_of(out)), "sa_block_sparse_fwd")
    else:
        block_sparse_attention(q.to(dev), k.to(dev), v.to(dev), kv, 0.125, out=out, n_text_blocks=text,
                               key_bias=None if bias is None else bias.to(dev))
    assert torch.isfinite(out).all()
    heads = sorted({(0, h) for h in (0, 1, 2, 3, H // 2 + 1, H - 2, H - 1)})
    want = masked_attention(q, k, v, mask, 0.125, key_bias=bias, heads=heads)
    for b, h in heads:
        err = (out[b, h].cpu().double() - want[b, h].nan_to_num()).abs()
        assert err.max() <= 2e-2 and err.mean() <= 2e-3, (h, err.max().item())


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


# Causal maps on both sides of the lines between index order and ranges (`xcd_ranges_pay`): 1 600
# and 2 160 items of heads that deal out evenly, 2 870 and 2 890 of others, and dense maps whose
# remainder is not shared.
@pytest.mark.parametrize("H,block,causal", [(160, 64, True), (216, 32, True), (287, 64, True), (289, 128, True),
                                            (85, 64, False), (85, 32, False), (85, 128, False)])
def test_pooled_map_placement(H, block, causal):
    print(f"case pooled placement H={H} block={block} causal={causal}", flush=True)
    dev, L = torch.device("cuda:0"), 617
    g = torch.Generator().manual_seed(H + block)
    q, k, v = (torch.randn(1, H, L, 64, generator=g).bfloat16() for _ in range(3))
    o, po = attn_with_pooling(q.to(dev), k.to(dev), v.to(dev), causal, 0.125, block)
    for h in {0, H // 8, H // 2, H - 1}:
        want_o, want_po = pooled_attention(*(t[:, h:h + 1] for t in (q, k, v)), causal, 0.125, block)
        err = (o[:, h:h + 1].cpu().double() - want_o).abs()
        assert err.max() <= 2e-2 and err.mean() <= 2e-3
        assert torch.allclose(po[:, h:h + 1].cpu().double(), want_po, rtol=5e-3, atol=1e-9)
    assert torch.isfinite(o).all() and torch.isfinite(po).all()
    # a head's rows do not depend on where they run
    alone, alone_po = attn_with_pooling(*(t[:, :1].to(dev) for t in (q, k, v)), causal, 0.125, block)
    assert (o[:, :1] - alone).abs().max() <= 2e-2 and torch.allclose(po[:, :1], alone_po, rtol=5e-3, atol=1e-9)


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


def _text_rows_everywhere(dev, H, nb, text, tail, dtype=torch.bfloat16, D=64):
    """q, k, v of nb blocks, the last of `tail` tokens; lists of the text blocks, one block of the
    row's own and every block for text rows, and those lists' mask."""
    L = 64 * (nb - 1) + tail
    g = torch.Generator(dev).manual_seed(H * nb)
    q, k, v = (torch.randn(1, H, L, D, device=dev, generator=g).to(dtype) for _ in range(3))
    mask = torch.eye(nb, dtype=torch.bool, device=dev).repeat(1, H, 1, 1)
    mask[:, :, :text] = True
    mask[:, :, :, :text] = True
    kv = kv_list_from_mask(mask, 1, H, nb, nb)
    kv.row_blocks = text + 1
    return q, k, v, kv, mask


def _rows_in_64_bits(q, k, v, mask, rows, bias=None):
    """Outputs of query blocks `rows` of every head, [H, 64 len(rows), D]."""
    out = []
    for h in range(q.shape[1]):
        idx = torch.cat([torch.arange(64 * r, min(64 * r + 64, q.shape[2]), device=q.device) for r in rows])
        s = q[0, h, idx].double() @ k[0, h].double().T.contiguous() * 0.125
        if bias is not None:
            s += bias[0, h].double()
        keep = mask[0, h, idx // 64].repeat_interleave(64, dim=1)[:, :k.shape[2]]
        out.append(torch.softmax(s.masked_fill(~keep, -math.inf), dim=-1) @ v[0, h].double())
    return torch.stack(out), idx


# One text block per head, one or no head starting in each XCD's range of 1 mod 4 items: the text
# rows' groups would fit the slots of the order without them (1 760, 1 792, 1 760; with a bias,
# which never takes key-range parts, 1 024), of which no remainder is shared.
@pytest.mark.parametrize("H,nb,biased", [(8, 217, False), (8, 221, False), (7, 247, False), (8, 125, True)])
def test_one_text_row_per_range(H, nb, biased):
    print(f"case shared items one text row per range H={H} nb={nb} biased={biased}", flush=True)
    dev = torch.device("cuda:0")
    q, k, v, kv, mask = _text_rows_everywhere(dev, H, nb, 1, 2)
    assert shares_text_rows(H * nb, nb, 1, kv.row_blocks, 64)
    bias = torch.randn(1, H, q.shape[2], device=dev) if biased else None
    out = torch.full_like(q, math.nan)
    block_sparse_attention(q, k, v, kv, 0.125, key_bias=bias, n_text_blocks=1, out=out)
    assert torch.isfinite(out).all()
    want, idx = _rows_in_64_bits(q, k, v, mask, (0, 1, nb - 1), bias)
    err = (out[0][:, idx].double() - want).abs()
    assert err.max() <= 2e-2 and err.mean() <= 2e-3, err.max().item()
    kv.row_blocks = None  # the same lists without shared text rows
    plain = block_sparse_attention(q, k, v, kv, 0.125, key_bias=bias, n_text_blocks=1)
    assert (out - plain).abs().max() <= 2e-2


# Token masks with text rows in groups of their own: one text block that would fit the plain order's
# 736, 960 and 1 024 slots, and two.
@pytest.mark.parametrize("config,H", [
    (dict(kernel_size=(1, 3, 3), tile_size=(12, 3, 3), img_size=(12, 21, 36), text_length=51), 5),
    (dict(kernel_size=(1, 5, 5), tile_size=(11, 3, 3), img_size=(11, 27, 33), text_length=58), 6),
    (dict(kernel_size=(1, 5, 5), tile_size=(11, 3, 3), img_size=(11, 24, 30), text_length=49), 8),
    (dict(kernel_size=(1, 3, 3), tile_size=(12, 3, 3), img_size=(12, 21, 36), text_length=100), 5),
])
def test_text_rows_beside_token_masks(config, H):
    print(f"case shared items sliding {config} H={H}", flush=True)
    from sparseattnfunctions_amd._kv import KVList
    from sparseattnfunctions_amd.SildingTileAttention import SildingTileAttention

    dev, text = torch.device("cuda:0"), config["text_length"]
    layer = SildingTileAttention(config)
    T, Hp, Wp = config["img_size"]
    L = text + T * Hp * Wp
    g = torch.Generator(dev).manual_seed(H)
    q, k, v = (torch.randn(1, H, L, 64, device=dev, generator=g).bfloat16() for _ in range(3))
    lay = layer._get_layout(dev)
    assert shares_text_rows(H * lay.nb, lay.nb, lay.text_blocks, lay.row_blocks, 64, True)
    out = torch.full_like(q, math.nan)
    kv = KVList(lay.kv_idx, lay.kv_cnt, 1, 1, lay.nb, lay.nb, row_blocks=lay.row_blocks)
    opts = dict(n_text_blocks=lay.text_blocks, tile_masks=(lay.kv_slot, lay.masks, True))
    block_sparse_attention(q, k, v, kv, 0.125, out=out, **opts)
    assert torch.isfinite(out).all()
    kv.row_blocks = None
    plain = block_sparse_attention(q, k, v, kv, 0.125, **opts)
    assert (out - plain).abs().max() <= 2e-2
    want = torch.stack([torch.softmax(q[0, h, :text].double() @ k[0, h].double().T.contiguous() / 8, dim=-1)
                        @ v[0, h].double() for h in range(H)])
    err = (layer(q, k, v)[0, :, :text].double() - want).abs()
    assert err.max() <= 2e-2 and err.mean() <= 2e-3, err.max().item()


# Kernels that never share an item run a long order's in the group's first slot: the plain order's
# bits.
@pytest.mark.parametrize("dtype,D,terms", [(torch.bfloat16, 128, False), (torch.float16, 128, False),
                                           (torch.float32, 64, False), (torch.float32, 128, False),
                                           (torch.float32, 64, True), (torch.float32, 128, True)])
@pytest.mark.parametrize("H,nb", [(3, 9), (8, 13)])
def test_long_order_in_kernels_that_do_not_share(dtype, D, terms, H, nb):
    print(f"case long order unshared {dtype} D={D} terms={terms} H={H} nb={nb}", flush=True)
    dev, lib = torch.device("cuda:0"), _lib.load()
    q, k, v, kv, _ = _text_rows_everywhere(dev, H, nb, 2, 33, dtype, D)
    L, st = q.shape[2], _lib.i64(*q.stride()[:3])
    ws = None
    if terms:
        n = ctypes.c_int64(0)
        _lib.check(lib.sa_block_sparse_fwd_f32_terms_workspace(1, H, L, D, ctypes.byref(n)), "workspace")
        ws = torch.empty(n.value, dtype=torch.uint8, device=dev)
    outs = []
    for name in ("sa_attn_work_order", "sa_attn_work_order_long"):
        n = ctypes.c_int64(0)
        build = getattr(lib, name)
        _lib.check(build(1, H, nb, 2, 8, None, ctypes.byref(n)), name)
        order = torch.empty(n.value, dtype=torch.int32)
        _lib.check(build(1, H, nb, 2, 8, order.data_ptr(), ctypes.byref(n)), name)
        order = order.to(dev)
        out = torch.full_like(q, math.nan)
        args = [q.data_ptr(), st, k.data_ptr(), st, v.data_ptr(), st, out.data_ptr(), st, 1, H, L, L, D,
                kv.idx.data_ptr(), kv.cnt.data_ptr(), kv.max_cnt]
        if terms:
            rc = lib.sa_block_sparse_fwd_f32_terms(*args, 0.125, order.data_ptr(), order.numel(), ws.data_ptr(),
                                                   ws.numel(), _lib.stream_of(q))
        else:
            fn = {torch.bfloat16: "sa_block_sparse_fwd", torch.float16: "sa_block_sparse_fwd_f16",
                  torch.float32: "sa_block_sparse_fwd_f32"}[dtype]
            rc = getattr(lib, fn)(*args, None, None, 0.125, order.data_ptr(), order.numel(), _lib.stream_of(q))
        _lib.check(rc, name)
        outs.append(out)
    torch.cuda.synchronize()
    assert torch.isfinite(outs[0]).all() and torch.equal(outs[0], outs[1])
