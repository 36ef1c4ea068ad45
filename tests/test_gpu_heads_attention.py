"""Prompt attention of heads of 64 and 128 whose queries lie by themselves, with a bias by distance (attention_heads32_kernel), against
float64."""
import math

import pytest
import torch

from easy_gpt.cpp_amd import kernels
from test_gpu_kernels import DEV, build_paged

pytestmark = pytest.mark.gpu


def _reference(q, keys, vals, nq, nkv, scale, window, bias):
    n, kv = q.shape[0], keys.shape[0]
    out = torch.zeros(n, nq, q.shape[2], dtype=torch.float64)
    dist = (torch.arange(kv - n, kv)[:, None] - torch.arange(kv)[None])
    unseen = (dist < 0) | ((dist >= window) if window else torch.zeros_like(dist, dtype=torch.bool))
    for h in range(nq):
        s = q[:, h] @ keys[:, h // (nq // nkv)].t() * scale
        if bias is not None:
            s = s + bias[h][dist.clamp(0, bias.shape[1] - 1)]
        out[:, h] = torch.softmax(s.masked_fill(unseen, -math.inf), 1) @ vals[:, h // (nq // nkv)]
    return out


@pytest.mark.parametrize("hd,row_blocks", [(64, 4), (64, 8), (128, 4), (128, 8)])
@pytest.mark.parametrize("nq,nkv,ps,far,window", [(14, 2, 16, 512, 0), (6, 2, 32, 63, 0), (3, 3, 64, 0, 0), (8, 1, 16, 300, 150), (4, 2, 16, None, 0),
                                                  (4, 2, 64, None, 200)])
def test_heads_with_a_bias_by_distance(hd, row_blocks, nq, nkv, ps, far, window):
    # lengths at and around the tiles and blocks of rows, prefixes, single tokens; distances on both sides of `far`; a bias as large
    # as the scores, and larger ones that make a row's maximum grow along the keys
    k = kernels.backend()
    seqs = [(300, 700), (1, 1), (64, 64), (65, 129), (2, 513), (1, 257), (127, 128), (17, 1000), (260, 260)]
    kc, vc, table, keys, vals = build_paged(seqs, nkv, hd, ps, torch.bfloat16, seed=3)
    g = torch.Generator().manual_seed(hd + nq)
    t = sum(n for n, _ in seqs)
    q = torch.randn(t, nq, hd, generator=g).to(torch.bfloat16)
    q_len = torch.tensor([n for n, _ in seqs], dtype=torch.int32)
    q_start = torch.cumsum(q_len, 0, dtype=torch.int32) - q_len
    kv_len = torch.tensor([n for _, n in seqs], dtype=torch.int32)
    scale = hd ** -0.5
    for size in (1.0, 12.0):
        bias = None if far is None else torch.randn(nq, far + 1, generator=g) * size
        out = torch.full((t, nq * hd), float("nan"), dtype=torch.bfloat16, device=DEV)
        bd = None if bias is None else bias.to(DEV)
        qd, qs, ql, kl = q.to(DEV), q_start.to(DEV), q_len.to(DEV), kv_len.to(DEV)
        k._run("egpt_heads_attention", qd.data_ptr(), out.data_ptr(), kc.data_ptr(), vc.data_ptr(), table.data_ptr(), table.shape[1], qs.data_ptr(),
               ql.data_ptr(), kl.data_ptr(), len(seqs), t, nq, nkv, hd, ps, scale, window, k._ptr(bd), far or 0, row_blocks, k._stream())
        torch.cuda.synchronize()
        got = out.double().cpu().view(t, nq, hd)
        for i, (n, _) in enumerate(seqs):
            s = int(q_start[i])
            want = _reference(q[s : s + n].double(), keys[i].double(), vals[i].double(), nq, nkv, scale, window, None if bias is None else bias.double())
            # bfloat16 probabilities and results, as everywhere in these kernels (values of about one; up to four)
            assert float((got[s : s + n] - want).abs().max()) <= (1.2e-2 if size == 1.0 or far is None else 2.4e-2), (i, size)


@pytest.mark.parametrize("hd,row_blocks", [(64, 4), (64, 8), (128, 8)])
@pytest.mark.parametrize("mask", [-1e10, -1e30, torch.finfo(torch.float32).min, -math.inf])
def test_a_bias_that_stands_for_a_mask(hd, row_blocks, mask):
    # beyond `far` (which the first tiles of long rows see alone), and, where it is a finite number that swallows any score, at the
    # nearest distances too: the first rows see masked keys alone then, all alike
    k = kernels.backend()
    nq, nkv, ps, far = 4, 2, 16, 100
    seqs = [(300, 700), (260, 260), (65, 129)]
    kc, vc, table, keys, vals = build_paged(seqs, nkv, hd, ps, torch.bfloat16, seed=7)
    g = torch.Generator().manual_seed(hd)
    t = sum(n for n, _ in seqs)
    q = torch.randn(t, nq, hd, generator=g).to(torch.bfloat16)
    bias = torch.randn(nq, far + 1, generator=g)
    bias[:3, far] = mask
    bias[1, 50:] = mask
    if -math.inf < mask < -1e20:
        bias[2, :5] = mask
        bias[3] = mask
    q_len = torch.tensor([n for n, _ in seqs], dtype=torch.int32)
    q_start = torch.cumsum(q_len, 0, dtype=torch.int32) - q_len
    out = torch.full((t, nq * hd), float("nan"), dtype=torch.bfloat16, device=DEV)
    bd, qd, qs, ql = bias.to(DEV), q.to(DEV), q_start.to(DEV), q_len.to(DEV)
    kl = torch.tensor([n for _, n in seqs], dtype=torch.int32, device=DEV)
    k._run("egpt_heads_attention", qd.data_ptr(), out.data_ptr(), kc.data_ptr(), vc.data_ptr(), table.data_ptr(), table.shape[1], qs.data_ptr(),
           ql.data_ptr(), kl.data_ptr(), len(seqs), t, nq, nkv, hd, ps, hd ** -0.5, 0, bd.data_ptr(), far, row_blocks, k._stream())
    torch.cuda.synchronize()
    got = out.double().cpu().view(t, nq, hd)
    for i, (n, _) in enumerate(seqs):
        s = int(q_start[i])
        want = _reference(q[s : s + n].double(), keys[i].double(), vals[i].double(), nq, nkv, hd ** -0.5, 0, bias.double())
        assert float((got[s : s + n] - want).abs().max()) <= 1.2e-2, i


def test_tables_that_leave_no_room_are_refused():
    k = kernels.backend()
    p = torch.zeros(1 << 20, device=DEV, dtype=torch.uint8).data_ptr()
    for nq, hd, far in ((64, 64, 1024), (16, 128, 4000), (4, 96, 10), (4, 64, 20000)):
        with pytest.raises(Exception):
            k._run("egpt_heads_attention", p, p, p, p, p, 1, p, p, p, 1, 200, nq, 1, hd, 16, 0.1, 0, p, far, 4, k._stream())


def test_wrapper_takes_it_only_where_it_covers_the_call(monkeypatch):
    k = kernels.backend()
    names = []
    run = type(k)._run
    monkeypatch.setattr(type(k), "_run", lambda self, name, *a: (names.append(name), run(self, name, *a))[1])
    nq, nkv, hd, ps = 4, 2, 64, 16
    kc, vc, table, _, _ = build_paged([(200, 200)], nkv, hd, ps, torch.bfloat16, seed=1)
    q = torch.randn(200, nq * hd, device=DEV).bfloat16()
    out = torch.empty_like(q)
    one = lambda v: torch.tensor([v], dtype=torch.int32, device=DEV)  # noqa: E731
    args = (q, out, kc, vc, table, one(0), one(200), one(200), nq, nkv, hd, hd, ps, 0.125)
    k.window_attention(*args, 0, 0, None, 200, 200)
    k.window_attention(*args, 0, 0, None, 200, 200, dist_bias=torch.zeros(nq, 33, device=DEV))
    assert names == ["egpt_heads_attention"] * 2
    names.clear()
    k.window_attention(*args, 50, 0, None, 200, 200)                                              # a narrow window
    k.window_attention(*args, 0, 0, torch.zeros(nq, device=DEV), 200, 200)                        # a sink
    k.window_attention(*args, 0, 0, None, 200, 200, softcap=30.0)
    k.window_attention(*args, 0, 0, None, 200, 200, slopes=torch.zeros(nq, device=DEV))
    k.window_attention(*args, 0, 0, None, 200, 200, block=64)
    k.window_attention(*args, 200, 4, None, 200, 200)                                             # kept first tokens
    k.window_attention(*args, 0, 0, None, 200, 200, dist_bias=torch.zeros(nq, 20001, device=DEV))  # a table that LDS does not hold
    assert names == ["egpt_window_attention_tiled"] * 7
    # the largest that it does, of a kv head's many heads
    names.clear()
    nq, nkv = 32, 1
    kc, vc, table, _, _ = build_paged([(200, 200)], nkv, hd, ps, torch.bfloat16, seed=1)
    q = torch.randn(200, nq * hd, device=DEV).bfloat16()
    args = (q, torch.empty_like(q), kc, vc, table, one(0), one(200), one(200), nq, nkv, hd, hd, ps, 0.125)
    most = (80 * 1024 // 4) // nq - 163
    for far in (most, most + 1):
        k.window_attention(*args, 0, 0, None, 200, 200, dist_bias=torch.zeros(nq, far + 1, device=DEV))
    assert names == ["egpt_heads_attention", "egpt_window_attention_tiled"]
