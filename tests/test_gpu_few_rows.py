"""The small kernels of a decode step at the edges of their sizes: the norm of few rows, the gate's activation behind partial sums, and the
combination of attention's parts, against plain torch in 64 bits.  What they return is rounded to bfloat16 once, so a value is off by at
most 2^-8 of itself (half a unit in the last of its eight bits); what is added to that is the float32 sums' own error."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
BF16 = 2.0 ** -8


@pytest.fixture(scope="module")
def k():
    from easy_gpt.cpp_amd import kernels

    return kernels.backend()


def draw(*shape, seed):
    return torch.randn(*shape, generator=torch.Generator().manual_seed(seed)).to(DEV)


def close(got, want):
    assert ((got.double() - want).abs() <= BF16 * want.abs() + 1e-6).all()


@pytest.mark.parametrize("hidden", [4, 60, 256, 260, 896, 3584, 4096, 4100])
@pytest.mark.parametrize("splits", [None, 0, 1, 2, 8, 9, 13])
@pytest.mark.parametrize("rows,fixed", [(1, False), (8, True), (31, False), (64, False)])
def test_norm_of_few_rows(k, hidden, splits, rows, fixed):
    h = draw(rows, hidden, seed=hidden)
    w = draw(hidden, seed=1).to(torch.bfloat16)
    delta, add = None, 0.0
    if splits == 0:
        delta = draw(rows, hidden, seed=2).to(torch.bfloat16)
        add = delta.double()
    elif splits:
        delta = draw(splits, rows, hidden, seed=2)
        add = delta.double().sum(0)
    stream = torch.round(h.double() * 2.0 ** 32).to(torch.int64) if fixed else h.clone()
    want_h = h.double() + add
    want = want_h * torch.rsqrt((want_h * want_h).mean(-1, keepdim=True) + 1e-5) * (0.5 + w.double())
    out = torch.empty(rows, hidden, dtype=torch.bfloat16, device=DEV)
    pick = torch.arange(rows - 1, -1, -1, dtype=torch.int32, device=DEV)[: (rows + 1) // 2].contiguous()
    some = torch.empty(len(pick), hidden, dtype=torch.bfloat16, device=DEV)
    kept = stream.clone()
    k.rows_add_rmsnorm(stream, delta, pick, w, 1e-5, some, weight_offset=0.5)
    assert torch.equal(stream, kept)
    k.add_rmsnorm(stream, delta, w, 1e-5, out, weight_offset=0.5)
    got_h = stream.double() * 2.0 ** -32 if fixed else stream.double()
    assert ((got_h - want_h).abs() <= 2e-6 * (want_h.abs() + 1)).all()
    close(out, want)
    close(some, want[pick.long()])


@pytest.mark.parametrize("inter", [4, 252, 1024, 1028, 4864])
@pytest.mark.parametrize("splits", [2, 3, 4, 5, 9])
@pytest.mark.parametrize("rows,squares", [(1, 0), (8, 0), (8, 4), (64, 9)])
@pytest.mark.parametrize("activation", ["silu", "gelu_tanh"])
def test_activation_behind_partial_sums(k, inter, splits, rows, squares, activation):
    z = draw(splits, rows, 2 * inter, seed=inter + splits)
    row_ss = (draw(squares, rows, seed=3).abs() * 30 + 1) if squares else None
    total = z.double().sum(0)
    if squares:
        total = total * torch.rsqrt(row_ss.double().sum(0) / 96 + 1e-5)[:, None]
    g, u = total[:, :inter], total[:, inter:]
    act = g * torch.sigmoid(g) if activation == "silu" else 0.5 * g * (1 + torch.tanh(0.7978845608028654 * (g + 0.044715 * g ** 3)))
    out = torch.empty(rows, inter, dtype=torch.bfloat16, device=DEV)
    k.swiglu(z, out, row_ss=row_ss, hidden=96 if squares else 0, eps=1e-5, activation=activation)
    # (the sums' own rounding, 2^-23 of the largest partial sum, goes through both factors)
    assert ((out.double() - act * u).abs() <= BF16 * (act * u).abs() + 4e-6 * (1 + g.abs()) * (1 + u.abs())).all()


@pytest.mark.parametrize("hd", [16, 64, 96, 128, 256])
@pytest.mark.parametrize("splits", [1, 2, 7, 8, 9, 17, 64])
def test_parts_of_attention_combined(k, hd, splits):
    t, nq = 5, 3
    o, ml = draw(splits, t, nq, hd, seed=hd + splits), draw(splits, t, nq, 2, seed=4)
    ml[..., 1] = ml[..., 1].abs() + 0.5
    ml[..., 0] *= 20
    if splits > 2:                               # parts without a key: their maximum says so, their values may be anything
        ml[1, :, :, 0] = float("-inf")
        ml[1, :, :, 1] = float("nan")
        o[1] = float("nan")
    out = torch.empty(t, nq * hd, dtype=torch.bfloat16, device=DEV)
    k.combine_attention(o, ml, out)
    live = [s for s in range(splits) if not (splits > 2 and s == 1)]
    wgt = torch.exp(ml[live, ..., 0].double() - ml[live, ..., 0].double().max(0).values)
    want = (wgt[..., None] * o[live].double()).sum(0) / (wgt * ml[live, ..., 1].double()).sum(0)[..., None]
    size = (wgt[..., None] * o[live].double().abs()).sum(0) / (wgt * ml[live, ..., 1].double()).sum(0)[..., None]
    assert ((out.view(t, nq, hd).double() - want).abs() <= BF16 * want.abs() + 4e-6 * size).all()
