"""Attention of decoded tokens with the QKV epilogue folded in, where its arithmetic of places can go wrong: page sizes that are no power
of two, more partial sums than a batch of loads, more heads than the workgroup's threads take in one pass."""
import math

import pytest
import torch

import plain_qwen2 as plain
from test_gpu_kernels import DEV, build_paged, rnd

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
