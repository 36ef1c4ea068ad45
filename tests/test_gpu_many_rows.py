"""The bfloat16 product for many rows (gemm_rows.hip): every tile at its edges, split k ranges, the activated form."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def k():
    from easy_gpt.cpp_amd import kernels

    return kernels.backend()


def rnd(*shape, seed, scale=1.0):
    g = torch.Generator().manual_seed(seed)
    return (torch.randn(*shape, generator=g) * scale).to(torch.bfloat16).cuda()


def run(k, x, w, shape, splits, kind, act=0):
    m, kk = x.shape
    n = w.shape[0] // (2 if kind == 2 else 1)
    out = torch.full((splits, m, n) if kind == 1 else (m, n), float("nan"), dtype=torch.float32 if kind == 1 else torch.bfloat16,
                     device="cuda")
    k._run("egpt_gemm_rows", x.data_ptr(), w.data_ptr(), out.data_ptr(), m, n, kk, splits, kind, act, shape, k._stream())
    return out


@pytest.mark.parametrize("shape", range(5))
@pytest.mark.parametrize("m,n,kk,splits", [(1, 4, 64, 1), (63, 60, 64, 1), (65, 68, 128, 2), (127, 260, 192, 3), (193, 132, 320, 2),
                                           (257, 516, 448, 4), (300, 1152, 896, 1)])
def test_every_tile_at_its_edges(k, shape, m, n, kk, splits):
    x, w = rnd(m, kk, seed=1), rnd(n, kk, seed=2)
    want = x.double() @ w.double().t()
    # float32 sums of kk products of bfloat16 numbers: at most kk roundings of the sum of magnitudes
    bound = (x.double().abs() @ w.double().abs().t()) * kk * 2.0 ** -24
    parts = run(k, x, w, shape, splits, 1)
    assert ((parts.double().sum(0) - want).abs() <= bound).all()
    rounded = run(k, x, w, shape, 1, 0).double()
    assert ((rounded - want).abs() <= bound + want.abs() * 2.0 ** -8).all()


@pytest.mark.parametrize("shape", range(5))
@pytest.mark.parametrize("act", [0, 1])
@pytest.mark.parametrize("m,n,kk", [(2, 4, 64), (65, 36, 128), (130, 260, 192)])
def test_the_activated_form(k, shape, act, m, n, kk):
    x, w = rnd(m, kk, seed=3), rnd(2 * n, kk, seed=4, scale=0.2)
    both = x.double() @ w.double().t()
    z, u = both[:, :n], both[:, n:]
    gate = z * torch.sigmoid(z) if act == 0 else torch.nn.functional.gelu(z, approximate="tanh")
    out = run(k, x, w, shape, 1, 2, act).double()
    assert ((out - gate * u).abs() <= (gate * u).abs() * 2.0 ** -8 + 1e-4 * (1 + z.abs()) * (1 + u.abs())).all()


@pytest.mark.parametrize("m,n,kk", [(65, 896, 4864), (200, 896, 896), (600, 1152, 896), (70, 104, 64), (130, 136, 192)])
def test_the_backend_chooses_and_sums(k, m, n, kk):
    x, w = rnd(m, kk, seed=5), rnd(n, kk, seed=6, scale=0.1)
    want = x.double() @ w.double().t()
    for unrounded in (False, True):
        got = k.product(x, w, unrounded=unrounded)
        total = got.double().sum(0) if got.dim() == 3 else got.double()
        assert (total - want).abs().max() <= (2.0 ** -8 if got.dim() == 2 else 1e-5) * want.abs().max()


def test_the_norm_adds_partial_sums_of_many_rows(k):
    t, hidden = 70, 104
    h = rnd(t, hidden, seed=7).float()
    weight = rnd(hidden, seed=8)
    for splits in (1, 2, 3, 4, 5, 8):
        delta = torch.randn(splits, t, hidden, generator=torch.Generator().manual_seed(splits)).cuda()
        hh, out = h.clone(), torch.empty((t, hidden), dtype=torch.bfloat16, device="cuda")
        k.add_rmsnorm(hh, delta, weight, 1e-6, out)
        v = h.double() + delta.double().sum(0)
        assert (hh.double() - v).abs().max() <= splits * 2.0 ** -22 * 8
        want = v * torch.rsqrt((v * v).mean(-1, keepdim=True) + 1e-6) * weight.double()
        assert ((out.double() - want).abs() <= want.abs() * 2.0 ** -8 + 1e-5).all()
        rows = torch.tensor(list(range(0, t)) + [3], dtype=torch.int32, device="cuda")
        some = torch.empty((t + 1, hidden), dtype=torch.bfloat16, device="cuda")
        k.rows_add_rmsnorm(h, delta, rows, weight, 1e-6, some)
        assert torch.equal(some, out[rows.long()])
