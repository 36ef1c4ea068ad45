"""Decoded tokens whose keys are dealt out by the contexts' lengths: the table, and the attention that goes by it."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.fixture(scope="module")
def k():
    from easy_gpt.cpp_amd import kernels

    return kernels.backend()


def ints(x):
    return torch.tensor(x, dtype=torch.int32, device=DEV)


LENGTHS = {
    "even": [700] * 17, "uneven": [1 + 37 * i for i in range(40)], "one long": [4000] + [3] * 30, "edges": [1, 15, 16, 17, 31, 32, 33, 64, 65] * 4,
    "as many as slots": [100 + i for i in range(64)],
}


def table_of(k, lens, slots, window, q_len=None):
    kv, start = ints(lens), ints(list(range(len(lens))))
    table = torch.full((slots * 8 + len(lens) * 2,), -9, dtype=torch.int32, device=DEV)
    k._run("egpt_decode_ranges", kv.data_ptr(), start.data_ptr(), k._ptr(q_len), len(lens), slots, window, table.data_ptr(), k._stream())
    t = table.cpu()
    return t[: slots * 8].view(slots, 8).tolist(), t[slots * 8 :].view(-1, 2).tolist()


@pytest.mark.parametrize("lens", LENGTHS.values(), ids=LENGTHS.keys())
@pytest.mark.parametrize("slots", [64, 128, 256])
@pytest.mark.parametrize("window", [0, 100])
def test_the_table_deals_out_every_block_once(k, lens, slots, window):
    one = [i % 5 != 2 for i in range(len(lens))]
    for q_len in (None, ints([1 if o else 7 for o in one])):
        entries, requests = table_of(k, lens, slots, window, q_len)
        at = 0
        for i, (n, (first, parts)) in enumerate(zip(lens, requests)):
            if q_len is not None and not one[i]:
                assert parts == 0
                continue
            assert first == at and 1 <= parts <= 64
            low = max(0, n - window) // 32 if window else 0
            for j in range(parts):
                b, begin, end, kv, tok, count = entries[at + j][:6]
                assert (b, begin, kv, tok, count) == (i, low, n, i, parts) and begin < end
                low = end
            assert low == (n - 1) // 32 + 1
            at += parts
        assert at <= slots and all(e[0] == -1 for e in entries[at:])
        # no workgroup has more than the least that all of them could do with
        most = max(e[2] - e[1] for e in entries[:at])
        blocks = [end for end in ((n - 1) // 32 + 1 - (max(0, n - window) // 32 if window else 0) for i, n in enumerate(lens) if q_len is None or one[i])]
        least = max(8, -(-max(blocks) // 64))
        assert most <= least or sum(-(-b // (most - 1)) for b in blocks) > slots


@pytest.mark.parametrize("hd,nq,nkv", [(64, 14, 2), (128, 6, 2), (64, 4, 1)])
@pytest.mark.parametrize("lens", LENGTHS.values(), ids=LENGTHS.keys())
@pytest.mark.parametrize("window", [0, 100])
def test_attention_dealt_out_and_in_equal_ranges(k, hd, nq, nkv, lens, window):
    # both round a probability to bfloat16 and the result once: each within 2^-8 of the largest value
    g = torch.Generator().manual_seed(len(lens) + hd)
    ps, b, width = 16, len(lens), (nq + 2 * nkv) * hd
    pages = sum(-(-n // ps) for n in lens)
    table, at, order = torch.full((b, -(-max(lens) // ps)), -1, dtype=torch.int32), 0, torch.randperm(pages, generator=g)
    for i, n in enumerate(lens):
        m = -(-n // ps)
        table[i, :m] = order[at : at + m].to(torch.int32)
        at += m
    kc = torch.randn(pages, nkv, ps, hd, generator=g).bfloat16().to(DEV)
    vc = torch.randn(pages, nkv, hd, ps, generator=g).bfloat16().to(DEV)
    kv, start = ints(lens), ints(list(range(b)))
    slots = ints([int(table[i, (n - 1) // ps]) * ps + (n - 1) % ps for i, n in enumerate(lens)])
    inv = (1.0 / torch.pow(torch.tensor(1e4), 2.0 * torch.arange(hd // 2) / hd)).to(DEV)
    prod = torch.randn(3, b, width, generator=g).to(DEV)
    tab = table.to(DEV)
    n_slots = 256 // nkv
    ranges = torch.empty(n_slots * 8 + b * 2, dtype=torch.int32, device=DEV)
    outs, caches = [], []
    for dealt in (None, ranges):
        kk, vv, out = kc.clone(), vc.clone(), torch.full((b, nq * hd), float("nan"), dtype=torch.bfloat16, device=DEV)
        if dealt is not None:
            k._run("egpt_decode_ranges", kv.data_ptr(), start.data_ptr(), None, b, n_slots, window, dealt.data_ptr(), k._stream())
        assert k.attention_decode_fused(prod, None, 0, 0.0, None, kv - 1, inv, hd, slots, out, kk, vv, tab, start, kv, nq, nkv, hd, ps,
                                        hd ** -0.5, window, max(lens), combine=True, ranges=dealt) is None
        outs.append(out.double())
        caches.append((kk, vv))
    assert torch.equal(caches[0][0], caches[1][0]) and torch.equal(caches[0][1], caches[1][1])
    assert (outs[0] - outs[1]).abs().max() <= 2.0 ** -7 * max(float(vc.abs().max()), float(caches[0][1].abs().max()))


@pytest.mark.parametrize("hd,nq,nkv", [(64, 14, 2), (128, 6, 2)])
@pytest.mark.parametrize("portions", [[(40, 40)], [(70, 600), (2, 2)], []])
def test_a_mixed_step_dealt_out(k, hd, nq, nkv, portions):
    g = torch.Generator().manual_seed(hd)
    ps, single = 16, [5, 1500, 33, 900, 16, 2000, 64]
    q_len = [1] * 4 + [n for n, _ in portions] + [1] * 3 + [0]
    lens = single[:4] + [n for _, n in portions] + single[4:] + [0]
    b, t, width = len(lens), sum(q_len), (nq + 2 * nkv) * hd
    pages = sum(-(-n // ps) for n in lens)
    table, at, order = torch.full((b, -(-max(lens) // ps)), -1, dtype=torch.int32), 0, torch.randperm(pages, generator=g)
    for i, n in enumerate(lens):
        m = -(-n // ps)
        table[i, :m] = order[at : at + m].to(torch.int32)
        at += m
    kc = torch.randn(pages, nkv, ps, hd, generator=g).bfloat16().to(DEV)
    vc = torch.randn(pages, nkv, hd, ps, generator=g).bfloat16().to(DEV)
    qkv = torch.randn(t, width, generator=g).bfloat16().to(DEV)
    q_start = ints([sum(q_len[:i]) for i in range(b)])
    ql, kv, tab = ints(q_len), ints(lens), table.to(DEV)
    n_slots = 256 // nkv
    ranges = torch.empty(n_slots * 8 + b * 2, dtype=torch.int32, device=DEV)
    k._run("egpt_decode_ranges", kv.data_ptr(), q_start.data_ptr(), ql.data_ptr(), b, n_slots, 0, ranges.data_ptr(), k._stream())
    outs = []
    for dealt in (None, ranges):
        out = torch.full((t, nq * hd), float("nan"), dtype=torch.bfloat16, device=DEV)
        k.paged_attention(qkv, out, kc, vc, tab, q_start, ql, kv, nq, nkv, hd, ps, hd ** -0.5, 0, max(max(q_len), 2), max(lens), ranges=dealt,
                          portion_kv=max((n for _, n in portions), default=0) if dealt is not None else None)
        outs.append(out.double())
    assert (outs[0] - outs[1]).abs().max() <= 2.0 ** -7 * float(vc.abs().max())
