"""Attention of decoded tokens with the QKV epilogue folded in, where its arithmetic of places can go wrong: page sizes that are no power
of two, more partial sums than a batch of loads, more heads than the workgroup's threads take in one pass."""
import math

import pytest
import torch

import plain_qwen2 as plain
from test_gpu_kernels import DEV, build_paged, paged_reference, rnd

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def k():
    from easy_gpt.cpp_amd import kernels

    return kernels.backend()


@pytest.mark.parametrize("nq,nkv,hd", [(14, 2, 64), (16, 1, 128), (6, 6, 128)])
@pytest.mark.parametrize("ps", [16, 48, 80, 256])
@pytest.mark.parametrize("parts,squares", [(1, 1), (8, 8), (9, 9), (16, 17), (20, 20), (33, 70)])
@pytest.mark.parametrize("batch,ctx,window", [(1, 2049, 0), (5, 1633, 0), (9, 497, 131), (70, 145, 0)])
def test_places_of_pages_and_partial_sums(k, nq, nkv, hd, ps, parts, squares, batch, ctx, window):
    # the same bits, in the output and in the caches, as the two kernels that it stands for
    dtype = torch.bfloat16
    seqs = [(1, max(1, ctx - 37 * i % ctx)) for i in range(batch)]
    kc, vc, table, _, _ = build_paged(seqs, nkv, hd, ps, dtype, seed=31)
    t, width = batch, (nq + 2 * nkv) * hd
    kv_len = torch.tensor([kv for _, kv in seqs], dtype=torch.int32)
    positions = (kv_len - 1).to(DEV)
    slots = torch.stack([table[b, (int(kv_len[b]) - 1) // ps].cpu() * ps + (int(kv_len[b]) - 1) % ps for b in range(t)]).to(torch.int32).to(DEV)
    prod = rnd(parts, t, width, seed=32)
    row_ss = (torch.rand(squares, t, generator=torch.Generator().manual_seed(33)) * 30 + 1).to(DEV)
    bias = rnd(width, dtype=dtype, seed=34)
    inv_freq = torch.as_tensor(plain.rope_inv_freq(hd, 1e4), dtype=torch.float32).to(DEV)
    q_start = torch.arange(t, dtype=torch.int32, device=DEV)
    q_len = torch.ones(t, dtype=torch.int32, device=DEV)
    kc1, vc1, kc2, vc2 = kc.clone(), vc.clone(), kc.clone(), vc.clone()
    qkv = torch.empty(t, width, dtype=dtype, device=DEV)
    k.qkv_rope_store(prod, bias, positions, inv_freq, hd, slots, kc1, vc1, nq, nkv, hd, ps, out=qkv, row_ss=row_ss, hidden=96, eps=1e-5)
    out1, out2 = (torch.zeros(t, nq * hd, dtype=dtype, device=DEV) for _ in range(2))
    k.paged_attention(qkv, out1, kc1, vc1, table, q_start, q_len, kv_len.to(DEV), nq, nkv, hd, ps, 1.0 / math.sqrt(hd), window, 1,
                      int(kv_len.max()))
    assert k.attention_decode_fused(prod, row_ss, 96, 1e-5, bias, positions, inv_freq, hd, slots, out2, kc2, vc2, table, q_start,
                                    kv_len.to(DEV), nq, nkv, hd, ps, 1.0 / math.sqrt(hd), window, int(kv_len.max())) is None
    assert torch.equal(kc1, kc2) and torch.equal(vc1, vc2)
    assert torch.equal(out1, out2)


@pytest.mark.parametrize("hd,lean", [(64, 0), (64, 1), (64, 2), (128, 0), (128, 1)])
@pytest.mark.parametrize("waves", [1, 2, 3, 4, 7, 8])
@pytest.mark.parametrize("splits", [1, 2])
def test_infinite_values_stay_infinite(k, hd, lean, waves, splits):
    # a value that is infinite makes its feature infinite, and that one alone, whichever wavefront has its key and however many there are
    nq, nkv, ps = 6, 2, 16
    kv = 32 * waves * splits                     # a block of keys for each wavefront
    kc, vc, table, keys, vals = build_paged([(1, kv)], nkv, hd, ps, torch.bfloat16, seed=41)
    qkv = rnd(1, (nq + 2 * nkv) * hd, dtype=torch.bfloat16, seed=42)
    start, context = (torch.tensor([v], dtype=torch.int32, device=DEV) for v in (0, kv))
    for at, feature, sign in ((kv - 2, 5, 1.0), (3, hd - 1, -1.0), (kv // 2, 17, 1.0)):
        vv = vc.clone()
        vv[table[0, at // ps].long(), :, feature, at % ps] = sign * float("inf")
        out, part_o, part_ml = torch.empty(1, nq * hd, dtype=torch.bfloat16, device=DEV), rnd(splits, nq, hd), rnd(splits, nq, 2)
        k._run("egpt_paged_attention_decode", qkv.data_ptr(), out.data_ptr(), part_o.data_ptr(), part_ml.data_ptr(), kc.data_ptr(), vv.data_ptr(),
               table.data_ptr(), table.shape[1], start.data_ptr(), context.data_ptr(), 1, nq, nkv, hd, ps, hd ** -0.5, 0, splits, waves, 1, lean,
               k._stream())
        with_inf = vals[0].double()
        with_inf[at, :, feature] = sign * float("inf")
        want = paged_reference(qkv.double().cpu().view(1, nq + 2 * nkv, hd)[:, :nq], keys[0].double(), with_inf, nq, nkv, hd ** -0.5, 0)[0]
        got = out.double().cpu().view(nq, hd)
        assert torch.isinf(want[:, feature]).all() and torch.equal(got[:, feature], want[:, feature])
        rest = torch.arange(hd) != feature
        assert float((got[:, rest] - want[:, rest]).abs().max()) <= 1.2e-2


def both_ways(k, prod, row_ss, bias, kv_len, caches, table, slots, nq, nkv, hd, ps, window=0):
    """(fused, the two kernels it stands for): output and caches of decoded tokens."""
    t, width = len(kv_len), (nq + 2 * nkv) * hd
    inv_freq = torch.as_tensor(plain.rope_inv_freq(hd, 1e4), dtype=torch.float32).to(DEV)
    kv, start, one = kv_len.to(DEV), torch.arange(t, dtype=torch.int32, device=DEV), torch.ones(t, dtype=torch.int32, device=DEV)
    got = []
    for fused in (True, False):
        kc, vc = (c.clone() for c in caches)
        out = torch.zeros(t, nq * hd, dtype=torch.bfloat16, device=DEV)
        if fused:
            assert k.attention_decode_fused(prod, row_ss, 96, 1e-5, bias, kv - 1, inv_freq, hd, slots, out, kc, vc, table, start, kv, nq, nkv, hd, ps,
                                            hd ** -0.5, window, int(kv_len.max())) is None
        else:
            qkv = torch.empty(t, width, dtype=torch.bfloat16, device=DEV)
            k.qkv_rope_store(prod, bias, kv - 1, inv_freq, hd, slots, kc, vc, nq, nkv, hd, ps, out=qkv, row_ss=row_ss, hidden=96, eps=1e-5)
            k.paged_attention(qkv, out, kc, vc, table, start, one, kv, nq, nkv, hd, ps, hd ** -0.5, window, 1, int(kv_len.max()))
        got.append((out, kc, vc))
    return got


def near(one, other):
    """bfloat16 results of the same sums in another order of blocks (a value may round to its neighbour)."""
    a, b = one.double(), other.double()
    return bool(((a - b).abs() <= 2.0 ** -7 * b.abs() + 2e-3).all())


@pytest.mark.parametrize("nq,nkv,hd", [(14, 2, 64), (16, 1, 128)])
@pytest.mark.parametrize("parts,squares,batch", [(1, 1, 1), (9, 9, 5), (33, 70, 70)])
def test_a_bias_that_begins_between_two_of_four_bytes(k, nq, nkv, hd, parts, squares, batch):
    kv_len = torch.tensor([1 + (577 * i + 900) % 1500 for i in range(batch)], dtype=torch.int32)
    kc, vc, table, _, _ = build_paged([(1, int(n)) for n in kv_len], nkv, hd, 16, torch.bfloat16, seed=51)
    slots = torch.stack([table[b, (int(n) - 1) // 16].cpu() * 16 + (int(n) - 1) % 16 for b, n in enumerate(kv_len)]).to(torch.int32).to(DEV)
    width = (nq + 2 * nkv) * hd
    prod, row_ss = rnd(parts, batch, width, seed=52), rnd(squares, batch, seed=53).abs() * 30 + 1
    bias = rnd(width + 1, dtype=torch.bfloat16, seed=54)[1:]
    assert bias.data_ptr() % 4 == 2
    (out, k1, v1), (want, k2, v2) = both_ways(k, prod, row_ss, bias, kv_len, (kc, vc), table, slots, nq, nkv, hd, 16)
    assert torch.equal(k1, k2) and torch.equal(v1, v2) and near(out, want)


def test_partial_sums_of_more_than_two_gigabytes(k):
    nq, nkv, hd, t, parts = 28, 4, 128, 300, 400
    kv_len = torch.tensor([1 + 7 * i % 90 for i in range(t)], dtype=torch.int32)
    kc, vc, table, _, _ = build_paged([(1, int(n)) for n in kv_len], nkv, hd, 16, torch.bfloat16, seed=61)
    slots = torch.stack([table[b, (int(n) - 1) // 16].cpu() * 16 + (int(n) - 1) % 16 for b, n in enumerate(kv_len)]).to(torch.int32).to(DEV)
    width = (nq + 2 * nkv) * hd
    assert parts * t * width * 4 > 1 << 31
    prod = torch.randn(parts, t, width, device=DEV, generator=torch.Generator(device=DEV).manual_seed(62)) * 0.05
    (out, k1, v1), (want, k2, v2) = both_ways(k, prod, None, rnd(width, dtype=torch.bfloat16, seed=63), kv_len, (kc, vc), table, slots, nq, nkv, hd, 16)
    assert torch.equal(k1, k2) and torch.equal(v1, v2) and near(out, want)


@pytest.mark.parametrize("hd", [64, 128])
def test_a_page_of_more_than_two_gigabytes_a_head(k, hd):
    # one page for a request's whole context: a feature's values lie gigabytes behind the head's first
    nq, nkv, ps = 4, 1, (1 << 31) // (2 * hd) + 16
    kv_len = torch.tensor([77], dtype=torch.int32)
    big = [torch.empty(1, nkv, *shape, dtype=torch.bfloat16, device=DEV) for shape in ((ps, hd), (hd, ps))]
    small = [torch.randn(1, nkv, *shape, device=DEV, generator=torch.Generator(device=DEV).manual_seed(71)).to(torch.bfloat16) for shape in ((80, hd), (hd, 80))]
    big[0][:, :, :80], big[1][..., :80] = small
    width, table, slots = (nq + 2 * nkv) * hd, torch.zeros(1, 1, dtype=torch.int32, device=DEV), torch.tensor([76], dtype=torch.int32, device=DEV)
    prod = rnd(3, 1, width, seed=72)
    both = [both_ways(k, prod, None, None, kv_len, caches, table, slots, nq, nkv, hd, caches[0].shape[2]) for caches in (big, small)]
    for (out, kc, vc), (want, k2, v2) in zip(both[0], both[1]):
        assert torch.equal(kc[:, :, :80], k2) and torch.equal(vc[..., :80], v2) and near(out, want)


@pytest.mark.parametrize("hd,leans", [(64, (0, 1, 2)), (128, (0, 1))])
@pytest.mark.parametrize("kv", [1, 31, 33, 100, 255, 256, 257, 700])
@pytest.mark.parametrize("waves,splits", [(8, 1), (4, 1), (3, 2), (8, 3)])
def test_variants_of_the_kernel_agree(k, hd, leans, kv, waves, splits):
    # rounds of one, two and four blocks of keys, also where a wavefront has fewer: the same bits where it has one block at most, and the same
    # keys in any case (the reference)
    nq, nkv, ps = 6, 2, 48
    kc, vc, table, keys, vals = build_paged([(1, kv)], nkv, hd, ps, torch.bfloat16, seed=81)
    qkv = rnd(1, (nq + 2 * nkv) * hd, dtype=torch.bfloat16, seed=82) * 2
    start, context = (torch.tensor([v], dtype=torch.int32, device=DEV) for v in (0, kv))
    want = paged_reference(qkv.double().cpu().view(1, nq + 2 * nkv, hd)[:, :nq], keys[0].double(), vals[0].double(), nq, nkv, hd ** -0.5, 0)[0]
    outs = []
    for lean in leans:
        out, part_o, part_ml = torch.empty(1, nq * hd, dtype=torch.bfloat16, device=DEV), rnd(splits, nq, hd), rnd(splits, nq, 2)
        k._run("egpt_paged_attention_decode", qkv.data_ptr(), out.data_ptr(), part_o.data_ptr(), part_ml.data_ptr(), kc.data_ptr(), vc.data_ptr(),
               table.data_ptr(), table.shape[1], start.data_ptr(), context.data_ptr(), 1, nq, nkv, hd, ps, hd ** -0.5, 0, splits, waves, 1, lean,
               k._stream())
        outs.append(out)
        assert float((out.double().cpu().view(nq, hd) - want).abs().max()) <= 1.2e-2
    if -(-kv // 32) <= waves * splits:
        assert all(torch.equal(outs[0], o) for o in outs)


@pytest.mark.parametrize("nq,nkv,hd", [(14, 2, 64), (16, 1, 128), (6, 6, 128)])
@pytest.mark.parametrize("ps", [48, 80, 256])
@pytest.mark.parametrize("batch,ctx,window", [(1, 2049, 0), (9, 497, 131), (2, 3000, 700)])
@pytest.mark.parametrize("folded", [True, False])
def test_pages_of_any_sixteens_against_64_bits(k, nq, nkv, hd, ps, batch, ctx, window, folded):
    # queries from so short that hundreds of keys count to so long that a single one has most of a row's weight: what is read from the wrong place,
    # left out or seen twice shows as an error of the size of the values, which are N(0, 1).  Otherwise an output is a mean of values, off by
    # the rounding of probabilities (2^-9 of each) and of the result (2^-9 of up to 4)
    kv_len = torch.tensor([max(1, ctx - 37 * i % ctx) for i in range(batch)], dtype=torch.int32)
    kc, vc, table, keys, vals = build_paged([(1, int(n)) for n in kv_len], nkv, hd, ps, torch.bfloat16, seed=91)
    slots = torch.stack([table[b, (int(n) - 1) // ps].cpu() * ps + (int(n) - 1) % ps for b, n in enumerate(kv_len)]).to(torch.int32).to(DEV)
    width = (nq + 2 * nkv) * hd
    prod = rnd(2, batch, width, seed=92)
    prod[:, :, : nq * hd] *= torch.linspace(1.0, 8.0, nq, device=DEV).repeat_interleave(hd)
    inv_freq = torch.as_tensor(plain.rope_inv_freq(hd, 1e4), dtype=torch.float32).to(DEV)
    kv, start, one = kv_len.to(DEV), torch.arange(batch, dtype=torch.int32, device=DEV), torch.ones(batch, dtype=torch.int32, device=DEV)
    k1, v1 = kc.clone(), vc.clone()
    qkv, out = torch.empty(batch, width, dtype=torch.bfloat16, device=DEV), torch.empty(batch, nq * hd, dtype=torch.bfloat16, device=DEV)
    k.qkv_rope_store(prod, None, kv - 1, inv_freq, hd, slots, k1, v1, nq, nkv, hd, ps, out=qkv)
    if folded:
        assert k.attention_decode_fused(prod, None, 0, 0.0, None, kv - 1, inv_freq, hd, slots, out, kc, vc, table, start, kv, nq, nkv, hd, ps,
                                        hd ** -0.5, window, int(kv_len.max())) is None
    else:
        k.paged_attention(qkv, out, k1, v1, table, start, one, kv, nq, nkv, hd, ps, hd ** -0.5, window, 1, int(kv_len.max()))
    row = qkv.double().cpu().view(batch, nq + 2 * nkv, hd)
    for b in range(batch):
        lo = max(0, int(kv_len[b]) - window) if window else 0
        kk, vv = keys[b].double(), vals[b].double()
        kk[-1], vv[-1] = row[b, nq : nq + nkv], row[b, nq + nkv :]
        q = row[b, :nq].view(nkv, nq // nkv, hd)
        scores = torch.matmul(q, kk[lo:].permute(1, 2, 0).contiguous()) * hd ** -0.5
        want = torch.matmul(torch.softmax(scores, -1), vv[lo:].permute(1, 0, 2).contiguous()).view(nq, hd)
        assert float((out[b].double().cpu().view(nq, hd) - want).abs().max()) <= 3e-2, b
