"""Kernels that take four neighbouring values a thread where operands begin on 16 bytes, against the general kernels, which take the same
operands one value further on: the same numbers but for the order in which a row's statistic is added up (float32: 2e-6 of the row's
size; bfloat16: a value may round to its neighbour, which is 2^-7 of it away at most)."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
DTYPES = [torch.float32, torch.bfloat16]


@pytest.fixture(scope="module")
def k():
    from easy_gpt.cpp_amd import kernels

    return kernels.backend()


def draw(*shape, seed, dtype=torch.float32):
    return torch.randn(*shape, generator=torch.Generator().manual_seed(seed)).to(dtype).to(DEV)


def further(t):
    """The same values, beginning one value behind a 16-byte place."""
    flat = torch.empty(t.numel() + 8, dtype=t.dtype, device=t.device)
    out = flat[1 : 1 + t.numel()].view(t.shape)
    out.copy_(t)
    assert out.data_ptr() % 16
    return out


def alike(a, b, dtype):
    step = 2.0 ** -7 if dtype == torch.bfloat16 else 2e-6
    a, b = a.double(), b.double()
    assert ((a - b).abs() <= step * (b.abs() + (0 if dtype == torch.bfloat16 else b.abs().amax(-1, keepdim=True))) + 1e-6).all()


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("hidden", [4, 252, 256, 260, 896, 2048, 4096, 4100])
@pytest.mark.parametrize("rows,splits", [(1, None), (3, 0), (70, 1), (5, 2), (2, 6)])
def test_layer_norm_and_mean_of_two(k, dtype, hidden, rows, splits):
    h = draw(rows, hidden, seed=1) * 3 + 50.0                 # (a mean much larger than the deviations)
    delta = None if splits is None else draw(rows, hidden, seed=2, dtype=dtype) if splits == 0 else draw(splits, rows, hidden, seed=2)
    w, b = draw(hidden, seed=3, dtype=dtype), draw(hidden, seed=4, dtype=dtype)
    got = []
    for move in (lambda t: t, further):
        hh = move(h.clone())
        out = torch.empty(rows, hidden, dtype=dtype, device=DEV)
        pick = torch.arange(rows - 1, -1, -1, dtype=torch.int32, device=DEV)
        some = torch.empty(rows, hidden, dtype=dtype, device=DEV)
        k.add_layernorm(hh, delta, pick, w, None, 1e-5, some)
        k.add_layernorm(hh, delta, None, w, b, 1e-5, out)
        got.append((hh, out, some))
    assert torch.equal(got[0][0], got[1][0])
    step = 4e-6 * 60 * w.double().abs().max()                  # (the mean's last bits, of values around 50)
    for one, other in zip(got[0][1:], got[1][1:]):
        assert ((one.double() - other.double()).abs() <= (2.0 ** -7 * other.double().abs() if dtype == torch.bfloat16 else 0) + step).all()
    if delta is not None:
        a = delta
        for bias, weight in ((b, w), (None, None)):
            one = k.normed_pair_mean(a, h.to(dtype), bias, None, weight, weight, 1e-5, 0.5, act_dtype=dtype)
            other = k.normed_pair_mean(further(a), h.to(dtype), bias, None, weight, weight, 1e-5, 0.5, act_dtype=dtype)
            alike(one, other, torch.float32)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("nq,nkv,dk,dv", [(14, 2, 64, 64), (1, 1, 4, 8), (3, 3, 20, 12), (16, 4, 128, 128), (24, 4, 128, 128), (5, 0, 64, 64)])
@pytest.mark.parametrize("splits,more,every", [(0, 0, 0), (1, 8, 3), (4, 4, 1024)])
def test_whole_norm_and_store(k, dtype, nq, nkv, dk, dv, splits, more, every):
    t, ps = 37, 16
    used = (nq + nkv) * dk + nkv * dv
    proj = draw(t, used + more, seed=5, dtype=dtype) if splits == 0 else draw(splits, t, used + more, seed=5)
    bias, qw, kw = draw(used, seed=6, dtype=dtype), draw(nq * dk, seed=7, dtype=dtype), draw(max(nkv, 1) * dk, seed=8, dtype=dtype)
    positions = torch.arange(t, dtype=torch.int32, device=DEV)
    slots = torch.randperm(4 * ps, generator=torch.Generator().manual_seed(9))[:t].to(torch.int32).to(DEV) if nkv else None
    got = []
    for move in (lambda x: x, further):
        q = torch.zeros(t, nq * dk, dtype=dtype, device=DEV)
        kc = torch.zeros(4, max(nkv, 1), ps, dk, dtype=dtype, device=DEV)
        vc = torch.zeros(4, max(nkv, 1), dv, ps, dtype=dtype, device=DEV)
        k.whole_norm_store(move(proj), bias, q, qw, kw if nkv else None, 1e-5, positions, 0.1, every, slots, kc, vc, nq, nkv, dk, dv, ps)
        got.append((q, kc, vc))
    for one, other in zip(*got):
        alike(one, other, dtype)
    assert torch.equal(got[0][2], got[1][2])                  # values are stored as they are


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("heads,dv", [(1, 64), (7, 128), (3, 256), (5, 64)])
@pytest.mark.parametrize("splits,gate,weighed", [(0, "silu", True), (1, "sigmoid", True), (3, "factor", False), (4, None, True)])
def test_gates_of_heads(k, dtype, heads, dv, splits, gate, weighed):
    t, n = 41, heads * dv
    x = draw(t, n, seed=10) if splits == 0 else draw(splits, t, n, seed=10)
    g = draw(2, t, n + 12, seed=11) if gate else None
    w = draw(dv, seed=12, dtype=dtype) if weighed else None
    got = []
    for move in (lambda v: v, further):
        out = torch.empty(t, n, dtype=dtype, device=DEV)
        k.head_norm_gate(move(x), w, 1e-5, g, 8 if gate else 0, out, heads, dv, **({"gate_act": gate} if gate else {}))
        got.append(out)
    alike(*got, dtype)
    if gate:
        y = draw(t, n, seed=13, dtype=dtype)
        row_ss = draw(3, t, seed=14).abs() + 1
        for args in ({}, dict(row_ss=row_ss, hidden=96, norm_eps=1e-5)):
            out, other = torch.empty_like(y), torch.empty_like(y)
            k.sigmoid_gate(y, 0, g, 8, out, **args)
            k.sigmoid_gate(further(y), 0, g, 8, other, **args)
            assert torch.equal(out, other)                    # (no statistic: the same operations)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("heads,dv", [(14, 64), (7, 128), (1, 64), (8, 256)])
@pytest.mark.parametrize("splits", [0, 1, 2, 3, 4, 5, 7, 8])
def test_a_row_of_gated_heads_is_the_same_among_few_and_among_many(k, dtype, heads, dv, splits):
    # 250,000 values are the line between a wavefront for a head and quads; the partial sums' loads go by threes and what is left of them
    n = heads * dv
    t = 250000 // n + 3
    x, w, g = draw(max(splits, 1), t, n, seed=20), draw(dv, seed=21, dtype=dtype), draw(max(splits, 1), t, n + 4, seed=22)
    many = torch.empty(t, n, dtype=dtype, device=DEV)
    k.head_norm_gate(x[0] if splits == 0 else x, w, 1e-5, g, 4, many, heads, dv)
    total, gate = x.double().sum(0).view(t, heads, dv), g.double().sum(0)[:, 4:]
    want = (total * torch.rsqrt((total * total).mean(-1, keepdim=True) + 1e-5) * w.double()).view(t, n) * gate * torch.sigmoid(gate)
    step = 2.0 ** -8 if dtype == torch.bfloat16 else 0.0       # (one rounding, and 32-bit sums of values of a size of `splits`)
    assert ((many.double() - want).abs() <= step * want.abs() + 1e-5 * (want.abs() + 1)).all()
    for first, count in ((0, 1), (t - 37, 37), (5, 250000 // n - 4)):
        some = torch.empty(count, n, dtype=dtype, device=DEV)
        rows = slice(first, first + count)
        k.head_norm_gate(x[0, rows].contiguous() if splits == 0 else x[:, rows].contiguous(), w, 1e-5, g[:, rows].contiguous(), 4, some, heads, dv)
        assert torch.equal(some, many[rows])


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("splits", [8, 9, 16, 17])
def test_a_gated_row_is_the_same_among_few_and_among_many(k, dtype, splits):
    # more than eight partial sums of up to 131,072 values go by single values
    n = 2048
    t = 131072 // n + 1
    x, g = draw(t, n, seed=30, dtype=dtype), draw(splits, t, n + 4, seed=31)
    many = torch.empty_like(x)
    k.sigmoid_gate(x, 0, g, 4, many)
    want = x.double() * torch.sigmoid(g.double().sum(0)[:, 4:])
    # one rounding, and sixteen additions of sums below 16, each off by 2^-24 of itself: 1.6e-5 in the gate, a quarter of it in the sigmoid, of x < 5
    step = 2.0 ** -8 if dtype == torch.bfloat16 else 0.0
    assert ((many.double() - want).abs() <= step * want.abs() + 2e-5 * (want.abs() + 1)).all()
    for first, count in ((0, 1), (1, t - 1)):
        some = torch.empty_like(x[:count])
        k.sigmoid_gate(x[first : first + count].contiguous(), 0, g[:, first : first + count].contiguous(), 4, some)
        assert torch.equal(some, many[first : first + count])


@pytest.mark.parametrize("hidden,experts,top,tokens", [(64, 4, 2, 65), (192, 16, 4, 1300), (192, 16, 4, 4200), (896, 16, 4, 90)])
def test_experts_of_many_tokens_into_a_given_sum(k, hidden, experts, top, tokens):
    # a choice's place in its expert's rows is nobody's business: the sums are the same bits whichever way the choices are grouped
    x = draw(tokens, hidden, seed=15, dtype=torch.bfloat16)
    router, up = draw(experts, hidden, seed=16, dtype=torch.bfloat16), draw(experts, 128, hidden, seed=17, dtype=torch.bfloat16) * 0.05
    down = draw(experts, hidden, 64, seed=18, dtype=torch.bfloat16) * 0.05
    want = k.expert_mixture(x, router, None, up, down, top)
    into = torch.full((3, tokens, hidden), 7.0, device=DEV)
    assert k.expert_mixture(x, router, None, up, down, top, out=into[1]).data_ptr() == into[1].data_ptr()
    assert torch.equal(into[1], want) and (into[0] == 7).all() and (into[2] == 7).all()
    few = torch.cat([k.expert_mixture(x[i : i + 64].contiguous(), router, None, up, down, top) for i in range(0, tokens, 64)])
    assert ((want - few).abs() <= 1e-2 * few.abs().amax()).all()


@pytest.mark.parametrize("dtype,m,n,kk", [
    (torch.bfloat16, 65, 128, 256), (torch.bfloat16, 300, 896, 768), (torch.bfloat16, 2048, 896, 896),         # the framework's own kernel
    (torch.bfloat16, 130, 896, 4864), (torch.bfloat16, 2535, 896, 768), (torch.bfloat16, 300, 72, 72),         # the library's
    (torch.bfloat16, 64, 128, 256), (torch.bfloat16, 7, 896, 896), (torch.bfloat16, 100, 64, 36),      # few rows, k no multiple of eight: copied
    (torch.float32, 100, 96, 64), (torch.float32, 700, 896, 768), (torch.float32, 3, 64, 60)])
def test_product_with_room_in_front(k, dtype, m, n, kk):
    x, w = draw(m, kk, seed=30, dtype=dtype), draw(n, kk, seed=31, dtype=dtype) * 0.1
    want = k.product(x, w, unrounded=True)
    want = want if want.dim() == 3 else want.float()[None]
    got = k.product_room(x, w)
    assert got.dtype == torch.float32 and got.is_contiguous() and got.shape == (1 + want.shape[0], m, n)
    got[0].fill_(float("nan"))                                # (the caller's: nothing of the sums lies there)
    assert torch.equal(got[1:], want)
    assert ((got[1:].double().sum(0) - x.double() @ w.double().T).abs() <= 2e-2 * (kk ** 0.5)).all()


def test_whose_products_with_room_are(k, monkeypatch):
    # the sizes above
    run, own = k._run, []
    monkeypatch.setattr(k, "_run", lambda name, *a: (own.append(a[3:6]) if name == "egpt_gemm_rows" else None, run(name, *a))[1])
    for m, n, kk in ((65, 128, 256), (300, 896, 768), (2048, 896, 896), (130, 896, 4864), (2535, 896, 768), (300, 72, 72)):
        k.product_room(draw(m, kk, seed=1, dtype=torch.bfloat16), draw(n, kk, seed=2, dtype=torch.bfloat16))
    assert own == [(65, 128, 256), (300, 896, 768), (2048, 896, 896)]
