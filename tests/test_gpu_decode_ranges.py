"""Decoded tokens whose keys are dealt out by the contexts' lengths: the table, and the attention that goes by it."""
import pytest
import torch

import helpers as H
from conftest import TINY
from easy_gpt.cpp_amd.engine import Engine
from easy_gpt.cpp_amd.weights import write_random_model

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
    "as many as slots": [100 + i for i in range(64)], "very long": [20000] + [300] * 19,
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


def attention64(q, kc, vc, table, n, window, scale):
    """q float64 [m, nq, hd], the last m of a request's n tokens: attention over its pages, float64 [m, nq * hd]."""
    ps, nkv, m, nq = kc.shape[2], kc.shape[1], q.shape[0], q.shape[1]
    pages = table[: -(-n // ps)].long()
    keys = kc[pages].transpose(0, 1).reshape(nkv, -1, kc.shape[3])[:, :n].double().repeat_interleave(nq // nkv, 0)
    values = vc[pages].permute(1, 0, 3, 2).reshape(nkv, -1, vc.shape[2])[:, :n].double().repeat_interleave(nq // nkv, 0)
    s = torch.matmul(q.transpose(0, 1).contiguous(), keys.transpose(1, 2).contiguous()) * scale
    at, far = torch.arange(n, device=q.device), torch.arange(n - m, n, device=q.device)[:, None]
    s.masked_fill_((at > far) | (at <= far - window if window else torch.zeros_like(at > far)), float("-inf"))
    return torch.matmul(torch.softmax(s, -1), values).transpose(0, 1).reshape(m, -1)


def assert_near(out, want, hd):
    """Of every head of every token: the result is rounded once, and its probabilities before, to bfloat16, half a unit of 2^-8 each.  The
    values are random, so the probabilities' errors add up like the result itself does: 2^-9 / sqrt(3) of its length from either
    rounding, 2^-9.3 together.  The line stands five times above; a block of 32 keys left out of 20,000 would be 2^-4.6."""
    out, want = out.double().view(-1, hd), want.view(-1, hd)
    assert ((out - want).norm(dim=1) <= 2.0 ** -7 * want.norm(dim=1)).all()


@pytest.mark.parametrize("hd,nq,nkv", [(64, 14, 2), (128, 6, 2), (64, 4, 1)])
@pytest.mark.parametrize("lens", LENGTHS.values(), ids=LENGTHS.keys())
@pytest.mark.parametrize("window", [0, 100])
def test_attention_dealt_out_and_in_equal_ranges(k, hd, nq, nkv, lens, window):
    # (the product is a single part of bfloat16 numbers and nothing turns, so that queries, keys and values are the reference's)
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
    inv = torch.zeros(hd // 2, device=DEV)
    prod = torch.zeros(3, b, width, device=DEV)
    prod[1] = torch.randn(b, width, generator=g).bfloat16().float().to(DEV)
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
        outs.append(out)
        caches.append((kk, vv))
    assert torch.equal(caches[0][0], caches[1][0]) and torch.equal(caches[0][1], caches[1][1])
    kk, vv = caches[0]
    own = prod[1].double().view(b, nq + 2 * nkv, hd)
    where, off = (slots // ps).long(), (slots % ps).long()
    assert torch.equal(kk[where, :, off].double(), own[:, nq : nq + nkv]) and torch.equal(vv[where, :, :, off].double(), own[:, nq + nkv :])
    want = torch.cat([attention64(own[i : i + 1, :nq], kk, vv, tab[i], n, window, hd ** -0.5) for i, n in enumerate(lens)])
    for out in outs:
        assert_near(out, want, hd)


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
    heads = qkv.double().view(t, -1, hd)[:, :nq]
    want = torch.cat([attention64(heads[s : s + m], kc, vc, tab[i], n, 0, hd ** -0.5)
                      for i, (s, m, n) in enumerate(zip(q_start.tolist(), q_len, lens)) if m])
    for dealt in (None, ranges):
        out = torch.full((t, nq * hd), float("nan"), dtype=torch.bfloat16, device=DEV)
        k.paged_attention(qkv, out, kc, vc, tab, q_start, ql, kv, nq, nkv, hd, ps, hd ** -0.5, 0, max(max(q_len), 2), max(lens), ranges=dealt,
                          portion_kv=max((n for _, n in portions), default=0) if dealt is not None else None)
        assert_near(out, want, hd)


@pytest.fixture(scope="module")
def long_models(tmp_path_factory):
    """The tiny models with head sizes 64 (an upper layer of it looks back 40 tokens) and 128, for contexts of some thousand tokens, with
    peaked attention."""
    out = {}
    for name in "DE":
        plain, sharp = (str(tmp_path_factory.mktemp(f"{kind}_{name}")) for kind in ("long", "long_sharp"))
        write_random_model(plain, dict(TINY[name][0], max_position_embeddings=4096), 90 + ord(name))
        out[name] = H.sharpen_attention(plain, sharp, 6.0)
    return out


@pytest.fixture()
def launched(monkeypatch):
    """The names of the entry points that the backend calls."""
    from easy_gpt.cpp_amd import kernels
    from easy_gpt.cpp_amd.kernels import hip

    kernels.use_backend(None)
    names, run = [], hip.HipKernels._run
    monkeypatch.setattr(hip.HipKernels, "_run", lambda self, name, *args: names.append(name) or run(self, name, *args))
    return names


@pytest.mark.parametrize("dtype,name", [("bfloat16", "D"), ("bfloat16", "E"), ("float32", "D")])
def test_uneven_contexts_through_the_engine(long_models, launched, dtype, name):
    # 20 conversations, one of them long, then the long one over and a shorter one in its place; every step is compared with the plain
    # implementation, and all but the first of a shape are replays of one graph while the contexts grow
    lens = [640] + [12 + 3 * i for i in range(19)]
    steps = 6
    vocab = TINY[name][0]["vocab_size"]
    reqs = H.make_requests(vocab, [n + steps for n in lens] + [330 + steps], seed=17)
    ids = list(reqs)
    trace = [H.step_record(0, [(rid, reqs[rid][:n], [n - 1]) for rid, n in zip(ids, lens)])]
    for s in range(steps):
        trace.append(H.step_record(1 + s, [(rid, [reqs[rid][n + s]], [0]) for rid, n in zip(ids, lens)], ids[:1] if s == steps - 1 else []))
    trace.append(H.step_record(9, [(ids[-1], reqs[ids[-1]][:330], [329])]))
    short = {rid: reqs[rid] + H.make_requests(vocab, [3], seed=len(reqs[rid]))["r0"] for rid in ids[1:-1]}
    for s in range(3):
        entries = [(rid, [short[rid][n + steps + s]], [0]) for rid, n in zip(ids[1:-1], lens[1:])]
        trace.append(H.step_record(10 + s, entries + [(ids[-1], [reqs[ids[-1]][330 + s]], [0])]))
    ref = H.plain_rows(long_models[name], {**reqs, **short}, bf16_weights=dtype == "bfloat16")
    eng = Engine.from_dir(long_models[name], dtype=dtype, device="cuda:0", page_size=16, max_tokens=4096, max_requests=24)
    rows = H.replay(eng, trace)
    H.assert_rows_match(rows, ref, H.BF16_TOL if dtype == "bfloat16" else H.FP32_TOL, f"uneven contexts {name} {dtype}")
    assert ("egpt_attention_decode_ranged" in launched) == (dtype == "bfloat16")
    assert ("egpt_decode_ranges" in launched) == (dtype == "bfloat16")         # no table where nothing goes by it
    assert all(p.graph is not None for p in eng._decode_plans.values())


@pytest.mark.parametrize("dtype,name,longest", [("bfloat16", "D", 2100), ("bfloat16", "E", 1100), ("float32", "E", 1100)])
def test_a_mixed_step_dealt_out_through_the_engine(long_models, launched, dtype, name, longest):
    # decoded tokens, one of them behind a long context, beside portions of a prompt that grows over three steps of one padded size
    lens, portion = [longest] + [9 + 40 * i for i in range(7)], 70
    reqs = H.make_requests(TINY[name][0]["vocab_size"], [n + 3 for n in lens] + [3 * portion], seed=18)
    ids = list(reqs)
    trace = [H.step_record(0, [(rid, reqs[rid][:n], [n - 1]) for rid, n in zip(ids, lens)])]
    for s in range(3):
        entries = [(rid, [reqs[rid][n + s]], [0]) for rid, n in zip(ids, lens)]
        entries.insert(3, (ids[-1], reqs[ids[-1]][s * portion : (s + 1) * portion], [0, portion - 1]))
        trace.append(H.step_record(1 + s, entries))
    ref = H.plain_rows(long_models[name], reqs, bf16_weights=dtype == "bfloat16")
    eng = Engine.from_dir(long_models[name], dtype=dtype, device="cuda:0", page_size=16, max_tokens=4096, max_requests=16)
    rows = H.replay(eng, trace)
    H.assert_rows_match(rows, ref, H.BF16_TOL if dtype == "bfloat16" else H.FP32_TOL, f"mixed steps {name} {dtype}")
    assert ("egpt_paged_attention_mixed" in launched) == ("egpt_decode_ranges" in launched) == (dtype == "bfloat16")
