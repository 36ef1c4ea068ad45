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


@pytest.mark.parametrize("hd,lean", [(64, 0), (64, 1), (128, 0), (128, 1)])
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
