"""The judges' kernels at their edges: `sa_topk_mass` (histogram selection without written
probabilities) and `sa_pattern_sim_gram_ws` (one walk over the keys)."""
import pytest
import torch

from sparseattnfunctions_amd import _lib
from sparseattnfunctions_amd import partern_attention as pa

pytestmark = pytest.mark.gpu


@pytest.fixture
def dev():
    return torch.device("cuda:0")


def _rows(kind, BH, n, seed, dev):
    g = torch.Generator().manual_seed(seed)
    q, k = torch.randn(1, BH, 40, 64, generator=g), torch.randn(1, BH, n, 64, generator=g)
    if kind == "peaked":  # e spans 2^-100 .. 1: several divisions of the K-th entry's bin
        q *= 8
    elif kind == "uniform":  # one pattern, every entry a tie
        q *= 0
    elif kind == "two values":  # two patterns
        k = torch.sign(k[..., :1]).expand(1, BH, n, 64).contiguous()
    elif kind == "underflow":  # most e are 0
        q *= 300
    return q.bfloat16().to(dev), k.bfloat16().to(dev)


@pytest.mark.parametrize("kind", ["normal", "peaked", "uniform", "two values", "underflow"])
@pytest.mark.parametrize("n,K,rows", [(1, 1, 1), (31, 6, 33), (32, 32, 32), (1000, 200, 40), (16384, 3276, 7)])
def test_topk_mass(dev, kind, n, K, rows):
    print(f"case topk_mass {kind} n={n} K={K} rows={rows}", flush=True)
    BH = 9  # heads are dealt to XCDs by eights: a second, partial group
    q, k = _rows(kind, BH, n, n + rows, dev)
    qs = pa._compact(q, torch.arange(rows), pa._pad32(rows))
    ks = pa._key_operands(k, torch.arange(n), pa._pad32(n))
    share = torch.full((BH, rows), -1.0, device=dev)
    _lib.check(_lib.load().sa_topk_mass(qs.data_ptr(), ks.data_ptr(), BH, rows, qs.shape[1], n, pa._pad32(n), 0.125,
                                        K, share.data_ptr(), _lib.stream_of(q)), "sa_topk_mass")
    p = torch.softmax(q[0, :, :rows].double() @ k[0].double().transpose(1, 2).contiguous() / 8, dim=-1)
    want = p.topk(K, dim=-1).values.sum(-1)
    # fp32 scores: a logit of some hundred carries 2^-24 of itself into each exp2
    assert torch.allclose(share.double(), want, rtol=2e-5 if kind in ("peaked", "underflow") else 2e-6, atol=0)
    again = torch.empty_like(share)
    _lib.check(_lib.load().sa_topk_mass(qs.data_ptr(), ks.data_ptr(), BH, rows, qs.shape[1], n, pa._pad32(n), 0.125,
                                        K, again.data_ptr(), _lib.stream_of(q)), "sa_topk_mass")
    assert torch.equal(share, again)  # whatever the order of the lists


# Rows of equal scores so large that their scaled maximum, rounded, leaves a remainder: every entry is
# the row's largest, so the K largest hold K / n of the mass.
@pytest.mark.parametrize("n,K", [(100, 20), (1000, 200), (16384, 3276)])
@pytest.mark.parametrize("x,y", [(10, 9), (300, 70), (-3, 1000), (2.0 ** 20, 2.0 ** 19 + 4096)])
def test_topk_mass_of_large_equal_scores(dev, n, K, x, y):
    print(f"case topk_mass equal scores {x} * {y} n={n} K={K}", flush=True)
    q = torch.full((1, 3, 33, 64), float(x)).bfloat16().to(dev)
    k = torch.full((1, 3, n, 64), float(y)).bfloat16().to(dev)
    qs = pa._compact(q, torch.arange(33), 64)
    ks = pa._key_operands(k, torch.arange(n), pa._pad32(n))
    share = torch.full((3, 33), -1.0, device=dev)
    _lib.check(_lib.load().sa_topk_mass(qs.data_ptr(), ks.data_ptr(), 3, 33, 64, n, pa._pad32(n), 0.125, K,
                                        share.data_ptr(), _lib.stream_of(q)), "sa_topk_mass")
    assert torch.allclose(share.double(), torch.full_like(share, K / n, dtype=torch.float64), rtol=2e-6, atol=0)


# Frames of one tile, of a tile and a remainder, and of many; text shorter than a tile, of many
# tiles and absent; scores whose sums leave the first walk's range (a second walk).
@pytest.mark.parametrize("F,ns,T,amp", [(1, 5, 0, 1.0), (4, 32, 7, 1.0), (11, 37, 224, 1.0), (12, 9, 33, 1.0),
                                         (3, 70, 40, 25.0), (11, 40, 0, 25.0)])
def test_sim_gram_one_walk(dev, F, ns, T, amp):
    print(f"case sim_gram F={F} ns={ns} T={T} amp={amp}", flush=True)
    geo = pa.PatternGeometry(frames=F, height=10, width=12, text_length=T, sample_num=ns)
    g = torch.Generator().manual_seed(F * ns)
    q = (torch.randn(1, 3, geo.L, 64, generator=g) * amp).bfloat16().to(dev)
    k = torch.randn(1, 3, geo.L, 64, generator=g).bfloat16().to(dev)
    _, ik = pa.get_indexs(geo)
    one = pa._similarity_gram(q, k, geo, ik)
    qs, ks, two = pa._similarity_inputs(q, k, geo, ik)
    _lib.check(_lib.load().sa_pattern_sim_gram(qs.data_ptr(), ks.data_ptr(), 3, F, ns, T, qs.shape[1], ks.shape[1],
                                               0.125, pa.composition_bias(geo), two.data_ptr(), _lib.stream_of(q)),
               "sa_pattern_sim_gram")
    probs = pa._similarity_gram_via_probs(q, k, geo, ik)
    # products of two probabilities: 2^-126 of the largest are lost
    assert torch.allclose(two, probs, rtol=4e-5, atol=1e-9), (two - probs).abs().max()
    assert torch.allclose(one, probs, rtol=4e-5, atol=1e-9), (one - probs).abs().max()


def test_judge_without_memory_for_the_workspace(dev, monkeypatch):
    print("case unified_judge without the Gram workspace", flush=True)
    geo = pa.PatternGeometry(frames=5, height=20, width=24, text_length=30, sample_num=100)
    g = torch.Generator().manual_seed(3)
    q, k = (torch.randn(1, 6, geo.L, 64, generator=g) for _ in range(2))
    for x in (q, k):  # half of the heads repeat one frame
        frames = x[:, :3, 30:].view(1, 3, 5, 480, 64)
        frames.copy_(frames[:, :, :1] + 0.1 * frames)
    q, k = q.bfloat16().to(dev), k.bfloat16().to(dev)
    torch.manual_seed(3)
    draws = (torch.randperm(geo.S)[:100], pa.get_indexs(geo)[1], pa.get_indexs(geo)[1])
    want = pa.unified_judge(q, k, geo, draws)
    _, sim = pa.judge_similarity(q, k, geo, draws[1], return_sim=True)
    empty, refused = torch.empty, []

    def full(*size, **kw):
        if kw.get("dtype") == torch.uint8:
            refused.append(size)
            raise torch.cuda.OutOfMemoryError("no memory")
        return empty(*size, **kw)

    monkeypatch.setattr(torch, "empty", full)
    got = pa.unified_judge(q, k, geo, draws)
    _, sim2 = pa.judge_similarity(q, k, geo, draws[1], return_sim=True)
    assert len(refused) == 3
    assert torch.equal(got, want) and want.any() and not want.all()
    assert torch.allclose(sim, sim2, rtol=4e-5)  # products of fp32 probabilities, as above
