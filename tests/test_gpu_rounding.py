"""Roundings that results rest on bit by bit, against the same operations one by one on the CPU."""
import functools

import numpy as np
import pytest
import torch

from test_gpu_kernels import DEV, k  # noqa: F401  (k: the fixture)

pytestmark = pytest.mark.gpu
LOG2E = np.float32(1.4426950408889634)


def bf16(x):
    """float32 -> bits of the nearest bfloat16, ties to even; NaN made quiet."""
    u = np.ascontiguousarray(x, dtype=np.float32).view(np.uint32)
    return np.where((u & 0x7FFFFFFF) > 0x7F800000, (u >> 16) | 0x40, (u.astype(np.uint64) + 0x7FFF + ((u >> 16) & 1)) >> 16).astype(np.uint16)


def combined(own, other, keys, weight, other_first):
    """(own + other * weight) / (keys + keys * weight) as the kernel's operations: one of the two products (own has the factor one) is
    fused with the sum, the other is rounded before it.  (Exact in 64 bits: 24 + 24 bits and a sum of numbers of a size.)"""
    f = np.float32
    product = other.astype(np.float64) * float(weight)
    total = f(own.astype(np.float64) + (product if other_first else f(product).astype(np.float64)))
    return bf16(f(total * (f(1) / (f(keys) + f(f(keys) * f(weight))))))


@functools.lru_cache
def telling_parts():
    """[2 sides][3 values][128] whose weighted sums round to different bfloat16 values by which product is rounded by itself."""
    rng, weight = np.random.default_rng(1), np.float32(2 ** -0.5)
    parts = np.empty((2, 3, 0), np.float32)
    while parts.shape[2] < 128:
        # (8 + 8 + 8 bits: the second and the third value 2^-8 and 2^-16 of the first)
        p = (rng.integers(128, 256, (2, 3, 1 << 21)) * np.array([2.0 ** -7, 2.0 ** -15, 2.0 ** -23])[None, :, None]).astype(np.float32)
        own, other = p.sum(1)
        parts = np.concatenate([parts, p[:, :, combined(own, other, 3, weight, True) != combined(own, other, 3, weight, False)]], 2)
    return parts


@pytest.mark.parametrize("hd,shape", [(64, 122), (64, 124), (64, 142), (128, 122), (128, 142), (64, 42), (64, 44), (64, 22), (64, 24), (128, 42), (128, 22)])
def test_keys_of_two_wavefronts_are_combined_with_the_same_rounding(k, hd, shape):  # noqa: F811
    # One tile of keys: of the first wavefront's three count, with scores of 0.5 and probabilities of one, and of the second's three with
    # scores of 0.  Sums of three values are any 24 bits and exact, the scores' unit is 1 / log2(e), so the second part weighs 2^-0.5, and that
    # product is rounded by itself or not.  The values are some where it shows in the result.
    scale = next(float(s) for s in np.float32(np.log(2)) * (1 + np.float32(2.0 ** -24) * np.arange(-4, 5, dtype=np.float32)) if s * LOG2E == 1)
    weight, parts = np.float32(2 ** -0.5), telling_parts()[:, :, :hd]
    rows, ks, ps = 32, shape % 10, 64
    kv = 64 * ks
    keys, vals = torch.zeros(kv, hd), torch.zeros(kv, hd)
    keys[:, 0] = -8192.0
    for w in range(2):
        for i, at in enumerate((3, 20, 41)):
            keys[64 * w + at] = 0.0
            keys[64 * w + at, 1] = 0.5 if w == 0 else 0.0
            vals[64 * w + at] = torch.from_numpy(parts[w, i])
    # the rows see all keys: their queries stand behind the last one, where a page of keys of no weight follows
    pages = ks + 1
    keys = torch.cat([keys, torch.zeros(ps, hd)])
    keys[kv:, 0] = -8192.0
    vals = torch.cat([vals, torch.zeros(ps, hd)])
    kc = keys.view(pages, 1, ps, hd).to(torch.bfloat16).to(DEV)
    vc = vals.view(pages, 1, ps, hd).permute(0, 1, 3, 2).contiguous().to(torch.bfloat16).to(DEV)
    qkv = torch.zeros(rows, 3 * hd)
    qkv[:, :2] = 1.0
    qkv = qkv.to(torch.bfloat16).to(DEV)
    one = lambda v: torch.tensor([v], dtype=torch.int32, device=DEV)  # noqa: E731
    table, start, length, context = torch.arange(pages, dtype=torch.int32, device=DEV)[None].contiguous(), one(0), one(rows), one(kv + rows)
    out = torch.zeros(rows, hd, dtype=torch.bfloat16, device=DEV)
    k._run("egpt_paged_attention_tiled", qkv.data_ptr(), out.data_ptr(), kc.data_ptr(), vc.data_ptr(), table.data_ptr(), pages, start.data_ptr(),
           length.data_ptr(), context.data_ptr(), 1, rows, 1, 1, hd, ps, scale, 0, shape, 1, None, None, 0, 0, 0, k._stream())
    got = out.cpu().view(torch.int16).numpy().view(np.uint16)
    assert (got == got[0]).all()                              # every row sees the same
    j = np.arange(hd)
    if shape >= 100:                                          # 32-row blocks: which element of its lane a feature is
        element = j % 32 // 8 * 4 + j % 4
        other_first = (j < 32) & (element >= 1) & (element <= 5)
    else:
        other_first = np.ones(hd, bool)
    own, other = parts.sum(1)
    expected = np.where(other_first, combined(own, other, 3, weight, True), combined(own, other, 3, weight, False))
    assert (got[0] == expected).all()


@pytest.mark.parametrize("pairs", [False, True])
def test_rounding_to_bfloat16_is_half_to_even(k, pairs):  # noqa: F811
    # Every upper half of a float32 with the lower halves at which rounding turns, subnormals, the largest numbers, infinities and NaN among them,
    # as values of heads, which the QKV epilogue rounds and does nothing else to: one by one (no rotation), or in pairs (the kernel for many
    # tokens).  (x 1 + 0 stands in front of the rounding: a zero's sign is not asked for.)
    low = np.array([0, 1, 0x7FFF, 0x8000, 0x8001, 0xFFFF], np.uint32)
    bits = ((np.arange(1 << 16, dtype=np.uint32) << 16)[:, None] | low).reshape(96, 4096)
    t, heads, hd = 96, 32, 128
    prod = torch.from_numpy(np.tile(bits, (1, 3)).view(np.float32)).to(DEV)[None].contiguous()
    assert (prod.view(torch.int32)[0, :, :4096].cpu().numpy().view(np.uint32) == bits).all()
    positions = torch.arange(t, dtype=torch.int32, device=DEV)
    slots = positions + 0
    kc, vc = torch.zeros(6, heads, 16, hd, dtype=torch.bfloat16, device=DEV), torch.zeros(6, heads, hd, 16, dtype=torch.bfloat16, device=DEV)
    out = torch.zeros(t, 3 * heads * hd, dtype=torch.bfloat16, device=DEV)
    if pairs:
        inv_freq = torch.ones(hd // 2, device=DEV)
        k.qkv_rope_store(prod, None, positions, inv_freq, hd, slots, kc, vc, heads, heads, hd, 16, out=out, cos_sin=k.rope_table(positions, inv_freq))
    else:
        k.qkv_rope_store(prod, None, positions, None, 0, slots, kc, vc, heads, heads, hd, 16, out=out)
    want = bf16(bits.view(np.float32))
    want = np.where(want == 0x8000, 0, want)
    nan = (want & 0x7FFF) > 0x7F80
    stored = vc.permute(0, 3, 1, 2).reshape(t, heads * hd)
    for got in [out[:, 2 * heads * hd :], stored] + ([] if pairs else [out[:, : heads * hd]]):
        got = got.contiguous().cpu().view(torch.int16).numpy().view(np.uint16)
        got = np.where(got == 0x8000, 0, got)
        assert (((got & 0x7FFF) > 0x7F80) == nan).all()
        assert (got[~nan] == want[~nan]).all()
