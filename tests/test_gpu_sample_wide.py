"""Sampling over wide vocabularies: lists that follow from the maxima of a row's shares, lists by exponent, draws without a list."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def k():
    from easy_gpt.cpp_amd import kernels

    return kernels.backend()


def draw(k, logits, temperature, top_k, top_p, uniform):
    r = logits.shape[0]
    row = lambda v, dt=torch.float32: torch.full((r,), v, dtype=dt, device="cuda") if not torch.is_tensor(v) else v.cuda()  # noqa: E731
    out = torch.full((r,), -7, dtype=torch.int32, device="cuda")
    k.sample(logits, row(temperature), row(top_k, torch.int32), row(top_p), row(uniform), out)
    return out.cpu().long()


def check(logits, temperature, top_k, top_p, uniform, tokens):
    """Every token is one that the cuts leave, and the drawn point lies in its part of the kept mass.  Weights are float32
    exponentials (a unit in the last place of 2^-23, times the argument), sums of some thousand of them are off by 1e-4 at most."""
    for x, u, tok in zip(logits.double().cpu(), uniform.double().tolist(), tokens.tolist()):
        w = torch.exp((x - x.max()) / temperature)
        kept = torch.ones_like(w, dtype=torch.bool)
        if 0 < top_k < w.numel():
            kept = w >= torch.topk(w, top_k).values[-1] * (1 - 1e-5)
        if 0 < top_p < 1:
            v = torch.where(kept, w, 0)
            values, which = torch.unique(w, return_inverse=True)          # ascending; equals stay or go together
            mass = torch.zeros_like(values).scatter_add_(0, which, v)
            above = (v.sum() - torch.cumsum(mass, 0))[which]
            kept = kept & (above <= top_p * v.sum() * (1 + 1e-5))
        assert kept[tok], (tok, float(w[tok]))
        v = torch.where(kept, w, 0)
        cum, total = torch.cumsum(v, 0), v.sum()
        assert cum[tok] - v[tok] <= (u + 1e-4) * total and cum[tok] >= (u - 1e-4) * total, (tok, u)


@pytest.mark.parametrize("vocab", [8192, 8195, 32768, 151936, 200003])
@pytest.mark.parametrize("top_k,top_p,temperature", [(1, 1.0, 0.7), (20, 0.95, 0.8), (32, 1.0, 1.0), (33, 0.9, 4.0), (128, 0.8, 1.0), (129, 0.9, 1.0),
                                                     (0, 0.9, 1.0), (0, 1.0, 1.0), (50, 0.95, 0.02), (20, 0.9, 0.004)])
def test_tokens_are_those_of_the_cuts(k, vocab, top_k, top_p, temperature):
    g = torch.Generator().manual_seed(vocab + top_k)
    logits = torch.randn(6, vocab, generator=g) * 2.5
    logits[1, 77] += 25.0                                        # one token far above the others
    logits[2, : vocab // 2] = -30.0
    logits[3] = torch.round(logits[3])                           # many equals
    logits[4, ::2] = float("-inf")
    uniform = torch.tensor([0.0, 0.3, 0.5, 0.77, 0.9, 0.999])
    tokens = draw(k, logits.cuda(), temperature, top_k, top_p, uniform)
    check(logits, temperature, top_k, top_p, uniform, tokens)


def test_more_equals_than_a_list_takes(k):
    # 3,000 tokens share the largest value: with ties whole all are kept, and the draw walks the row
    vocab = 40000
    logits = torch.randn(3, vocab, generator=torch.Generator().manual_seed(1))
    at = torch.randperm(vocab, generator=torch.Generator().manual_seed(2))[:3000]
    logits[:, at] = 9.0
    uniform = torch.tensor([0.01, 0.4, 0.98])
    for top_k, top_p in ((20, 1.0), (20, 0.9), (100, 0.5)):
        tokens = draw(k, logits.cuda(), 1.0, top_k, top_p, uniform)
        ordered = torch.sort(at).values
        for u, tok in zip(uniform.tolist(), tokens.tolist()):
            place = int((ordered == tok).nonzero()[0, 0])        # one of them, and the one at the drawn place
            assert abs(place - u * 3000) <= 2, (top_k, top_p, place, u)


def test_rows_of_each_kind_beside_each_other(k):
    # the same token whatever the rows beside it ask for: greedy, a list by the maxima, lists by exponent, no list
    logits = torch.randn(6, 50000, generator=torch.Generator().manual_seed(3)) * 3
    temperature, top_p = torch.tensor([0.0, 0.8, 1.0, 1.2, 1.0, 0.9]), torch.tensor([1.0, 0.95, 0.9, 1.0, 0.8, 1.0])
    top_k, uniform = torch.tensor([5, 20, 0, 0, 500, 128], dtype=torch.int32), torch.tensor([0.5, 0.1, 0.6, 0.7, 0.2, 0.95])
    together = draw(k, logits.cuda(), temperature, top_k, top_p, uniform)
    assert together[0] == logits[0].argmax()
    for r in range(6):
        alone = draw(k, logits[r : r + 1].cuda(), temperature[r : r + 1], top_k[r : r + 1], top_p[r : r + 1], uniform[r : r + 1])
        assert alone[0] == together[r], r


@pytest.mark.parametrize("first", [0, 7, 31])
def test_a_share_of_nothing_but_nan(k, first):
    # the row's maximum is that of the other shares, wherever the one without a number lies and wherever the maximum does
    vocab = 20000
    piece = -(-vocab // 32)
    for at in (3, 9000, vocab - 1):
        if at // piece == first:
            continue
        logits = torch.randn(3, vocab, generator=torch.Generator().manual_seed(at))
        logits[:, at] = 40.0
        logits[1, :] = float("-inf")
        logits[1, at] = -3.0
        logits[2, :] = float("-inf")
        logits[:, first * piece : (first + 1) * piece] = float("nan")
        least = 0 if first else piece                               # of the last row: its first token that is a number
        for top_k, top_p in ((20, 0.9), (200, 0.9), (0, 0.9), (0, 1.0)):
            for temperature in (0.0, 1.0):
                assert draw(k, logits.cuda(), temperature, top_k, top_p, torch.tensor([0.5] * 3)).tolist() == [at, at, least], (at, top_k, top_p)
        out = torch.full((3,), -7, dtype=torch.int32, device="cuda")
        k.argmax(logits.cuda(), out)
        assert out.tolist() == [at, at, least]


@pytest.mark.parametrize("top_k,top_p", [(20, 0.9), (200, 0.9), (0, 0.9), (0, 1.0)])
def test_numbers_that_are_none(k, top_k, top_p):
    # a NaN is never drawn; an infinity is; a row of nothing but NaN or minus infinity gives its first token
    logits = torch.randn(4, 20000, generator=torch.Generator().manual_seed(4))
    logits[0, 5::7] = float("nan")
    logits[1, 1234] = float("inf")
    logits[2] = float("nan")
    logits[3] = float("-inf")
    tokens = draw(k, logits.cuda(), 1.0, top_k, top_p, torch.tensor([0.5, 0.5, 0.5, 0.5])).tolist()
    assert 0 <= tokens[0] < 20000 and (tokens[0] - 5) % 7 != 0
    assert tokens[1:] == [1234, 0, 0]
