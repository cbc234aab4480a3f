"""fp32 attention on split bf16 operands (`sa_block_sparse_fwd_f32_terms`): edges of its tiles,
units and rules, against the fp64 oracle and the fp32 kernel without a workspace."""
import math

import pytest
import torch

from oracle.attention import masked_attention
from oracle.pooling import pooled_attention
from sparseattnfunctions_amd._kv import kv_list_from_mask
from sparseattnfunctions_amd.utils import block_sparse_attn_kernel as bsk
from sparseattnfunctions_amd.utils.attn_pooling_kernel import attn_with_pooling

pytestmark = pytest.mark.gpu


@pytest.fixture
def dev():
    return torch.device("cuda:0")


def _plain(monkeypatch, *args):
    """The same call through `sa_block_sparse_fwd_f32`."""
    with monkeypatch.context() as m:
        m.setattr(bsk, "F32_TERMS_BLOCKS", 1 << 30)
        return bsk.block_sparse_attention(*args)


def _lists(B, H, Lq, Lk, keep, seed, dev):
    nqb, nkb = math.ceil(Lq / 64), math.ceil(Lk / 64)
    mask = torch.rand(B, H, nqb, nkb, generator=torch.Generator().manual_seed(seed)) < keep
    mask[..., 0] = True
    return mask, kv_list_from_mask(mask.to(dev), B, H, nqb, nkb)


def _rand(seed, *shape):
    return torch.randn(*shape, generator=torch.Generator().manual_seed(seed))


# Units shared by four waves and units of one wave (more than 6 144 of them), partial first and
# last tiles, lists shorter than the four waves.
@pytest.mark.parametrize("B,H,Lq,Lk,D,keep", [
    (1, 1, 512, 512, 64, 1.0), (2, 3, 449, 321, 64, 0.9), (1, 2, 1000, 65, 64, 1.0), (1, 1, 2049, 2047, 64, 0.4),
    (1, 40, 9900, 700, 64, 0.7), (1, 2, 450, 1001, 128, 0.6), (1, 40, 5000, 450, 128, 0.8),
])
def test_errors_no_larger_than_the_fp32_kernels(dev, monkeypatch, B, H, Lq, Lk, D, keep):
    print(f"case terms {B} {H} {Lq} {Lk} {D} {keep}", flush=True)
    q, k, v = _rand(1, B, H, Lq, D), _rand(2, B, H, Lk, D), _rand(3, B, H, Lk, D)
    mask, kv = _lists(B, H, Lq, Lk, keep, Lq + Lk, dev)
    args = (q.to(dev), k.to(dev), v.to(dev), kv, 1 / math.sqrt(D))
    heads = [(b, h) for b in range(B) for h in range(0, H, 13)]
    want = masked_attention(q, k, v, mask, 1 / math.sqrt(D), heads=heads)
    new, old = (x.cpu().double() for x in (bsk.block_sparse_attention(*args), _plain(monkeypatch, *args)))
    for b, h in heads:
        e_new, e_old = (x[b, h] - want[b, h] for x in (new, old))
        # both round about 1e-6 of a unit-variance v; 5 % covers the spread of so few rows
        assert e_new.norm() <= 1.05 * e_old.norm(), (e_new.norm().item(), e_old.norm().item())
        assert e_new.abs().max() <= 2e-5
    assert (new - old).abs().max() <= 4e-5


# Rows, keys and values that the split operands cannot carry run in fp32: the same bits.
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("where,value", [("k", float("inf")), ("k", -2.0 ** 61), ("v", float("nan")),
                                          ("v", 2.0 ** 100), ("tiny v", 2.0 ** -90), ("q", 2.0 ** 60),
                                          ("q", float("-inf"))])
def test_out_of_range_operands(dev, monkeypatch, D, where, value):
    print(f"case terms out of range {D} {where} {value}", flush=True)
    # one wave per unit, so that both kernels visit the tiles of a row in the same order
    B, H, L = 1, 26 if D == 64 else 13, 15360
    q, k, v = (_rand(i, B, H, L, D).to(dev) for i in (4, 5, 6))
    t = {"k": k, "v": v, "q": q, "tiny v": v}[where]
    if where == "tiny v":
        t[0, 0] *= value
    else:
        t[0, 0, 70, 3] = value
    nb = L // 64
    mask = torch.zeros(1, 1, nb, nb, dtype=torch.bool)
    mask[..., :4] = True
    kv = kv_list_from_mask(mask.to(dev), B, H, nb, nb)
    args = (q, k, v, kv, 0.125)
    new, old = bsk.block_sparse_attention(*args), _plain(monkeypatch, *args)
    # a wave owns 64 query rows (32 at head dim 128) and decides for them
    rows = slice(64, 128 if D == 64 else 96) if where == "q" else slice(None)
    assert torch.equal(new[0, 0, rows].isnan(), old[0, 0, rows].isnan())
    assert torch.equal(new[0, 0, rows].nan_to_num(), old[0, 0, rows].nan_to_num())
    assert not torch.equal(new[0, 1], old[0, 1])  # the other heads took the split operands


# A block, column or element of small values inside an ordinary head: their low terms would leave
# bf16's range (and a query row's its own), so the head (or row group) runs in fp32: the same bits.
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("where,value", [("v block", 2.0 ** -115), ("v column", 2.0 ** -110), ("v", 2.0 ** -140),
                                          ("k", -2.0 ** -100), ("q", 2.0 ** -90)])
def test_small_values_in_an_ordinary_head(dev, monkeypatch, D, where, value):
    print(f"case terms small values {D} {where} {value}", flush=True)
    # one wave per unit, so that both kernels visit the tiles of a row in the same order
    B, H, L = 1, 26 if D == 64 else 13, 15360
    q, k, v = (_rand(i, B, H, L, D).to(dev) for i in (4, 5, 6))
    v[0, 1, 128:192] = 0  # zeros are no small values
    if where == "v block":
        v[0, 0, 64:128] *= value
    elif where == "v column":
        v[0, 0, :, 5] *= value
    else:
        {"v": v, "k": k, "q": q}[where][0, 0, 70, 3] = value
    nb = L // 64
    mask = torch.zeros(1, 1, nb, nb, dtype=torch.bool)
    mask[..., :4] = True
    mask[..., 7, :] = torch.arange(nb) == 1  # a row of the small block alone
    kv = kv_list_from_mask(mask.to(dev), B, H, nb, nb)
    args = (q, k, v, kv, 0.125)
    new, old = bsk.block_sparse_attention(*args), _plain(monkeypatch, *args)
    rows = slice(64, 128 if D == 64 else 96) if where == "q" else slice(None)
    assert torch.equal(new[0, 0, rows], old[0, 0, rows])
    assert not torch.equal(new[0, 1], old[0, 1])  # the other heads took the split operands
    if where.startswith("v "):
        s = q[0, 0, 448:512].double() @ k[0, 0, 64:128].double().T.contiguous() * 0.125
        want = torch.softmax(s, dim=-1) @ v[0, 0, 64:128].double()
        cols = slice(5, 6) if where == "v column" else slice(None)
        got, want = new[0, 0, 448:512, cols].double(), want[:, cols]
        assert (got - want).norm() <= 4e-6 * want.norm()  # a few fp32 roundings of 64 products


def test_short_lists_and_strided_rows(dev, monkeypatch):
    # head 0: one tile per key block (fp32 bits); head 1: five; BLHD views
    print("case terms short lists", flush=True)
    B, L, H = 1, 64 * 3100, 2
    q, k, v = (_rand(i, B, L, H, 64).to(dev).permute(0, 2, 1, 3) for i in (7, 8, 9))
    nb = L // 64
    mask = torch.eye(nb, dtype=torch.bool).repeat(1, H, 1, 1)
    mask[:, 1, :, :5] = True
    kv = kv_list_from_mask(mask.to(dev), B, H, nb, nb)
    args = (q, k, v, kv, 0.125)
    new, old = bsk.block_sparse_attention(*args), _plain(monkeypatch, *args)
    assert torch.equal(new[:, 0], old[:, 0])
    assert not torch.equal(new[:, 1], old[:, 1])
    assert (new - old).abs().max() <= 4e-5


# Heads with too few tiles per key block beside one that takes the split operands, past the size from
# which the fp32 kernel runs them: its bits. Groups of four units that straddle heads, an empty list,
# an order with text rows first. (At head dim 128 they stay in the split operands' kernel.)
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("H,Lq,Lk,text", [(27, 64 * 41 - 7, 64 * 41 - 7, 0), (47, 64 * 23, 64 * 23 + 1, 0),
                                          (83, 64 * 13 - 1, 64 * 13 - 1, 1), (160, 64 * 40, 64 * 40, 0)])
def test_heads_of_short_lists(dev, monkeypatch, D, H, Lq, Lk, text):
    print(f"case terms heads of short lists D={D} H={H} {Lq} {Lk} text={text}", flush=True)
    nqb, nkb = math.ceil(Lq / 64), math.ceil(Lk / 64)
    q, k, v = _rand(1, 1, H, Lq, D).to(dev), _rand(2, 1, H, Lk, D).to(dev), _rand(3, 1, H, Lk, D).to(dev)
    i, j = torch.arange(nqb)[:, None], torch.arange(nkb)
    mask = (i % nkb == j).repeat(1, H, 1, 1)
    mask[:, 1] = True  # the one head of long lists
    mask[0, 2, 3] = False  # an empty list
    kv = kv_list_from_mask(mask.to(dev), 1, H, nqb, nkb)
    args = (q, k, v, kv, 0.125, None, None, text)
    new, old = bsk.block_sparse_attention(*args), _plain(monkeypatch, *args)
    short = [h for h in range(H) if h != 1]
    if D == 64:
        assert torch.equal(new[:, short], old[:, short])
    assert torch.all(new[0, 2, 192:256] == 0)
    assert not torch.equal(new[:, 1], old[:, 1])
    assert (new - old).abs().max() <= 4e-5


# Few query blocks (up to 128): every head is split, those of one tile per key block too.
def test_short_lists_of_a_small_launch(dev, monkeypatch):
    print("case terms short lists of a small launch", flush=True)
    q, k, v = (_rand(i, 1, 3, 1000, 64) for i in (7, 8, 9))
    mask = torch.eye(16, dtype=torch.bool).repeat(1, 3, 1, 1)
    mask[0, 1, 5] = False
    kv = kv_list_from_mask(mask.to(dev), 1, 3, 16, 16)
    args = (q.to(dev), k.to(dev), v.to(dev), kv, 0.125)
    new, old = bsk.block_sparse_attention(*args), _plain(monkeypatch, *args)
    want = masked_attention(q, k, v, mask, 0.125)
    assert (new.cpu().double() - want).abs().max() <= 2e-5 and torch.all(new[0, 1, 320:384] == 0)
    assert not torch.equal(new, old)


# The pooled map beside one-wave units (more than 6 144) and shared ones, partial last blocks,
# grouped key heads; bars of the fp32 pooling tests.
@pytest.mark.parametrize("H,Hk,L,D,bs,causal", [(130, 130, 3077, 64, 64, False), (130, 65, 3077, 64, 32, True),
                                                 (66, 33, 3077, 128, 128, True), (66, 66, 3077, 128, 32, False),
                                                 (2, 1, 515, 64, 128, False), (2, 2, 577, 128, 64, True)])
def test_pooled_map(dev, H, Hk, L, D, bs, causal):
    print(f"case terms pooled {H} {Hk} {L} {D} {bs} {causal}", flush=True)
    q, k, v = _rand(1, 1, H, L, D), _rand(2, 1, Hk, L, D), _rand(3, 1, Hk, L, D)
    o, po = attn_with_pooling(q.to(dev), k.to(dev), v.to(dev), causal, 1 / math.sqrt(D), bs)
    for h in (0, H - 1):
        hk = h // (H // Hk)
        want_o, want_po = pooled_attention(q[:, h:h + 1], k[:, hk:hk + 1], v[:, hk:hk + 1], causal, 1 / math.sqrt(D),
                                           bs)
        err = (o[:, h:h + 1].cpu().double() - want_o).abs()
        assert err.max() <= 2e-5 and err.mean() <= 2e-6
        assert torch.allclose(po[:, h:h + 1].cpu().double(), want_po, rtol=2e-5, atol=1e-9)
