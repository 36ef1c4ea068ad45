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


@pytest.mark.parametrize("splits", [0, 1, 3])
@pytest.mark.parametrize("which", ["h", "delta", "weight", "out"])
def test_the_norm_of_many_rows_takes_operands_that_begin_anywhere(k, splits, which):
    """One operand a value behind 16 bytes: the values of the aligned call, up to the order of a row's sum of 104 squares."""
    t, hidden = 70, 104

    def place(v, name):
        if name != which:
            return v
        whole = torch.empty(v.numel() + 16, dtype=v.dtype, device="cuda")
        moved = whole[1 : 1 + v.numel()].view(v.shape)
        moved.copy_(v)
        return moved

    h, weight = rnd(t, hidden, seed=7).float(), rnd(hidden, seed=8)
    delta = rnd(t, hidden, seed=9) if splits == 0 else torch.randn(splits, t, hidden, generator=torch.Generator().manual_seed(9)).cuda()
    want_h, want = h.clone(), torch.empty((t, hidden), dtype=torch.bfloat16, device="cuda")
    k.add_rmsnorm(want_h, delta, weight, 1e-6, want)
    got_h, got = place(h.clone(), "h"), place(torch.zeros_like(want), "out")
    k.add_rmsnorm(got_h, place(delta, "delta"), place(weight, "weight"), 1e-6, got)
    assert torch.equal(got_h, want_h)
    assert ((got.double() - want.double()).abs() <= want.double().abs() * 2.0 ** -7).all()


@pytest.mark.parametrize("tile_rows", [64, 128])
@pytest.mark.parametrize("t,top,experts,outputs,hidden,ff", [(1, 1, 1, 1, 64, 64), (5, 3, 4, 6, 128, 64), (150, 2, 5, 7, 64, 192),
                                                             (130, 1, 3, 3, 192, 128), (40, 4, 700, 1000, 64, 64)])
def test_rows_grouped_by_expert(k, tile_rows, t, top, experts, outputs, hidden, ff):
    """Choices from `experts` on have no row; with few choices most experts have none, with one expert in use whole tiles."""
    g = torch.Generator().manual_seed(t)
    chosen = torch.stack([torch.randperm(outputs, generator=g)[:top] for _ in range(t)]).int().cuda()
    if experts == 3:
        chosen[:] = 1
    x, w, down = rnd(t, hidden, seed=1), rnd(experts, 2 * ff, hidden, seed=2, scale=0.2), rnd(experts, hidden, ff, seed=3, scale=0.2)
    n = t * top
    new = lambda *shape, dtype=torch.int32: torch.full(shape, -7, dtype=dtype, device="cuda")  # noqa: E731
    row_token, place, counts, tiles = new(n), new(t, top), new(experts), new(1 + 3 * (n // tile_rows + experts + 1))
    k._run("egpt_moe_group", chosen.data_ptr(), row_token.data_ptr(), place.data_ptr(), tiles.data_ptr(), counts.data_ptr(), t, top,
           experts, tile_rows, k._stream())
    flat = chosen.view(-1).long().cpu()
    kept = flat < experts
    assert torch.equal(counts.cpu().long(), torch.bincount(flat[kept], minlength=experts))
    rows = place.view(-1).cpu().long()
    assert (rows[~kept] == -1).all() and torch.equal(rows[kept].sort().values, torch.arange(int(kept.sum())))
    assert torch.equal(row_token.cpu().long()[rows[kept]], torch.arange(n)[kept] // top)
    table = tiles[1 : 1 + 3 * int(tiles[0])].view(-1, 3).cpu()
    assert int(table[:, 2].sum()) == int(kept.sum()) and int(tiles[0]) == int(((counts.cpu() + tile_rows - 1) // tile_rows).sum())
    x64, w64, d64 = x.double().cpu(), w.double().cpu(), down.double().cpu()
    for kind in (2, 3):
        act, y = new(n, ff, dtype=torch.bfloat16), new(n, hidden, dtype=torch.float32)
        wk = w if kind == 2 else w[:, :ff].contiguous()
        k._run("egpt_moe_rows", x.data_ptr(), wk.data_ptr(), row_token.data_ptr(), tiles.data_ptr(), act.data_ptr(), n, t, ff, hidden,
               experts, tile_rows, kind, 0, k._stream())
        k._run("egpt_moe_rows", act.data_ptr(), down.data_ptr(), None, tiles.data_ptr(), y.data_ptr(), n, n, hidden, ff, experts,
               tile_rows, 1, 0, k._stream())
        for i in kept.nonzero().view(-1).tolist():
            e, r = int(flat[i]), int(rows[i])
            z = w64[e] @ x64[i // top]
            want = z[:ff] * torch.sigmoid(z[:ff]) * z[ff:] if kind == 2 else z[:ff].clamp(min=0) ** 2
            assert ((act[r].double().cpu() - want).abs() <= want.abs() * 2.0 ** -8 + 1e-4).all()
            full = d64[e] @ act[r].double().cpu()
            assert ((y[r].double().cpu() - full).abs() <= 1e-5 * (d64[e].abs() @ act[r].double().cpu().abs()) + 1e-6).all()


@pytest.mark.parametrize("shape", range(7))
@pytest.mark.parametrize("kk,splits", [(128, 1), (192, 1), (256, 1), (384, 2), (448, 2)])
def test_a_workgroup_takes_several_tiles_in_turn(k, shape, kk, splits):
    # more tiles than the CUs hold workgroups, with edges in both directions; two steps (a workgroup per tile), three (all of a
    # tile's loads under the tile before), four, and split ranges of three and of four and three steps
    m, n = ((2049, 9004), (2049, 9004), (2049, 9004), (2300, 4100), (2300, 2052), (2300, 2052), (2300, 4100))[shape]
    x, w = rnd(m, kk, seed=9), rnd(n, kk, seed=10)
    want = x.double() @ w.double().t()
    bound = (x.double().abs() @ w.double().abs().t()) * kk * 2.0 ** -24
    parts = run(k, x, w, shape, splits, 1)
    assert ((parts.double().sum(0) - want).abs() <= bound).all()
    if splits > 1:
        return
    rounded = run(k, x, w, shape, 1, 0)
    assert ((rounded.double() - want).abs() <= bound + want.abs() * 2.0 ** -8).all()
    some = (n // 2) // 8 * 8 + (0 if kk == 192 else 4)             # rounded results leave in eights of columns, or in fours
    w = torch.cat([w[:some] * 0.2, w[:some] * 0.2])
    both = x.double() @ w.double().t()
    z, u = both[:, :some], both[:, some:]
    out = run(k, x, w, shape, 1, 2).double()
    gate = z * torch.sigmoid(z) * u
    assert ((out - gate).abs() <= gate.abs() * 2.0 ** -8 + 1e-4 * (1 + z.abs()) * (1 + u.abs())).all()


@pytest.mark.parametrize("act", [0, 1])
def test_the_activation_over_its_range(k, act):
    # gates from the smallest to the largest, up values of one: the result is the activation itself, off by a few float32
    # roundings (4 units of 2^-23, and as much again of the exponent, whose error is one of the factor) and rounded to
    # bfloat16.  Beyond 87 the exponential leaves float32's normal numbers.
    z = torch.cat([torch.linspace(-12, 12, 385), torch.tensor([1e-30, -1e-30, 1e-6, -40.0, 40.0, -86.5, 86.5, -87.5, 87.5, -95.0, -300.0, 300.0, 1e30,
                                                               -1e30])]).to(torch.bfloat16)
    m = z.numel()
    x = torch.zeros(m, 64, dtype=torch.bfloat16)
    x[:, 0], x[:, 1] = z, 1.0
    w = torch.zeros(16, 64, dtype=torch.bfloat16)
    w[:8, 0], w[8:, 1] = 1.0, 1.0
    out = run(k, x.cuda(), w.cuda(), 4, 1, 2, act).cpu().double()
    zd = z.double()
    y = zd if act == 0 else 1.5957691216057308 * (zd + 0.044715 * zd ** 3)
    want = zd * torch.sigmoid(y)
    off = want.abs() * (2.0 ** -8 + (1 + y.abs().clamp(max=100.0)) * 2.0 ** -21) + 1e-37
    assert ((out - want[:, None]).abs() <= off[:, None]).all()


@pytest.mark.parametrize("shape", [5, 6])
@pytest.mark.parametrize("m,n,kk,splits", [(1, 4, 64, 1), (63, 60, 64, 1), (65, 68, 128, 2), (127, 260, 192, 3), (193, 132, 320, 2),
                                           (257, 516, 448, 4), (300, 1152, 896, 1)])
def test_the_deeper_rings_at_their_edges(k, shape, m, n, kk, splits):
    test_every_tile_at_its_edges(k, shape, m, n, kk, splits)


@pytest.mark.parametrize("shape", [5, 6])
@pytest.mark.parametrize("act", [0, 1])
@pytest.mark.parametrize("m,n,kk", [(2, 4, 64), (65, 36, 128), (130, 260, 192)])
def test_the_deeper_rings_activated(k, shape, act, m, n, kk):
    test_the_activated_form(k, shape, act, m, n, kk)


@pytest.mark.parametrize("m", [17, 33, 64])
@pytest.mark.parametrize("n,kk", [(8, 64), (72, 128), (200, 4864), (896, 576), (2560, 2048), (16392, 192), (33000, 128), (65544, 320)])
def test_a_few_dozen_rows(k, m, n, kk):
    # one tile of rows, by every rule for them: the smallest, ranges of two steps and of more, a last range that is shorter, one tile
    # of 64 columns to a CU and just more, more than 512, and the width from which `linear` takes it for a vocabulary
    x, w = rnd(m, kk, seed=11), rnd(n, kk, seed=12)
    want = x.double() @ w.double().t()
    bound = (x.double().abs() @ w.double().abs().t()) * kk * 2.0 ** -24
    for unrounded in (False, True):
        parts = k.product(x, w, unrounded=unrounded)
        if parts.dim() == 2:                                       # one piece where the library rounds
            assert not unrounded and parts.dtype == torch.bfloat16
            assert ((parts.double() - want).abs() <= bound + want.abs() * 2.0 ** -8).all()
        else:
            assert parts.dtype == torch.float32 and ((parts.double().sum(0) - want).abs() <= bound).all()
    out = torch.empty((m, n), dtype=torch.float32, device="cuda")
    assert ((k.linear(x, w, None, out).double() - want).abs() <= bound).all()
    z, u = want[:, :n // 2], want[:, n // 2:]
    gate = z * torch.sigmoid(z) * u
    act = k.gate_up_swiglu(x, w)
    if act is not None:
        assert ((act.double() - gate).abs() <= gate.abs() * 2.0 ** -8 + 1e-4 * (1 + z.abs()) * (1 + u.abs())).all()


@pytest.mark.parametrize("m", [64, 65, 72, 320, 321, 552, 769, 1025])
@pytest.mark.parametrize("n,kk", [(1152, 896), (2048, 1536), (104, 64), (4608, 3584), (96, 200)])
def test_a_product_in_parts(k, n, kk, m):
    """On both sides of every line of its rule: the parts add up to the product, four at most beyond 64 rows."""
    x, w = rnd(m, kk, seed=7), rnd(n, kk, seed=8, scale=0.1)
    parts = k.product_parts(x, w)
    assert parts.dtype == torch.float32 and parts.shape[1:] == (m, n) and (m <= 64 or parts.shape[0] <= k.rope_parts)
    bound = (x.double().abs() @ w.double().abs().t()) * kk * 2.0 ** -24
    assert ((parts.double().sum(0) - x.double() @ w.double().t()).abs() <= bound).all()


@pytest.mark.parametrize("parts", [2, 3, 4, 5])
@pytest.mark.parametrize("t", [63, 64, 65, 130])
@pytest.mark.parametrize("nq,nkv,hd,biased,shift", [(14, 2, 64, True, 0), (5, 1, 24, False, 0), (3, 3, 128, True, 0), (4, 2, 32, True, 1)])
def test_rotation_of_a_product_in_parts(k, t, nq, nkv, hd, biased, shift, parts):
    """Rows rotated and stored out of partial sums, in whichever kernel takes them: the bits of their sum, added in their order, as one
    float32 array, the cache included; `shift`: an operand that does not begin on 16 bytes."""
    width, ps = (nq + 2 * nkv) * hd, 4
    g = torch.Generator().manual_seed(9)
    prod = torch.randn(parts * t * width + shift, generator=g).cuda()[shift:].view(parts, t, width)
    whole = prod[0].clone()
    for p in range(1, parts):
        whole += prod[p]
    bias = rnd(width, seed=10) if biased else None
    positions = torch.arange(t, dtype=torch.int32, device="cuda") * 3
    inv = (1e4 ** (-2.0 * torch.arange(hd // 2) / hd)).float().cuda()
    slots = torch.randperm(t + 5, generator=g)[:t].to(torch.int32).cuda()
    results = []
    for given in (prod, whole[None]):
        pages = -(-(t + 5) // ps)
        kc = torch.zeros((pages, nkv, ps, hd), dtype=torch.bfloat16, device="cuda")
        vc = torch.zeros((pages, nkv, hd, ps), dtype=torch.bfloat16, device="cuda")
        out = torch.empty((t, width), dtype=torch.bfloat16, device="cuda")
        k.qkv_rope_store(given, bias, positions, inv, hd, slots, kc, vc, nq, nkv, hd, ps, out=out, cos_sin=k.rope_table(positions, inv))
        results.append((out, kc, vc))
    assert all(torch.equal(a, b) for a, b in zip(*results))


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("form", [0, 1, 3, 5])
@pytest.mark.parametrize("t", [64, 77])
@pytest.mark.parametrize("nq,nkv,hd,biased,shift", [(14, 2, 64, True, 0), (5, 1, 24, False, 0), (4, 2, 32, True, 1)])
def test_rotated_rows_are_the_same_bits_in_a_large_and_in_a_small_step(k, t, nq, nkv, hd, biased, shift, form, dtype):
    """Rows of a step of 64 tokens and more against the same rows 16 at a time, which another kernel takes: the result and the cache."""
    width, ps = (nq + 2 * nkv) * hd, 4
    g = torch.Generator().manual_seed(11)
    prod = torch.randn(max(form, 1) * t * width + shift, generator=g).cuda()
    prod[shift::37] = -0.0
    prod = (prod if form else prod.to(dtype))[shift:].view(*((form,) if form else ()), t, width)
    bias = rnd(width, seed=12).to(dtype) if biased else None
    positions = torch.arange(t, dtype=torch.int32, device="cuda") * 5
    inv = (1e4 ** (-2.0 * torch.arange(hd // 2) / hd)).float().cuda()
    cs = k.rope_table(positions, inv)
    slots = torch.randperm(t + 5, generator=g)[:t].to(torch.int32).cuda()
    results = []
    for step in (t, 16):
        pages = -(-(t + 5) // ps)
        kc = torch.zeros((pages, nkv, ps, hd), dtype=dtype, device="cuda")
        vc = torch.zeros((pages, nkv, hd, ps), dtype=dtype, device="cuda")
        out = torch.empty((t, width), dtype=dtype, device="cuda")
        for a in range(0, t, step):
            rows = slice(a, min(t, a + step))
            k.qkv_rope_store(prod if step == t else prod[..., rows, :].contiguous(), bias, positions[rows], inv, hd, slots[rows], kc, vc, nq, nkv, hd, ps, out=out[rows],
                             cos_sin=cs[rows])
        results.append((out, kc, vc))
    whole = torch.int32 if dtype == torch.float32 else torch.int16
    assert all(torch.equal(a.view(whole), b.view(whole)) for a, b in zip(*results))


@pytest.mark.parametrize("m,n,kk", [(577, 896, 896), (1024, 896, 896), (960, 896, 768), (913, 1024, 1024), (448, 1536, 1536), (256, 3584, 3584),
                                    (192, 5120, 5120), (2305, 1024, 8192), (65, 18944, 896)])
def test_sums_that_a_norm_adds_are_not_rounded(k, m, n, kk):
    # also where k is one range: each element within the float32 sum's own error, which a rounding to bfloat16 would exceed
    x, w = rnd(m, kk, seed=31), rnd(n, kk, seed=32, scale=kk ** -0.5)
    got = k.product(x, w)
    assert got.dtype == torch.float32 and got.dim() == 3
    got = got.double().sum(0)
    for a in range(0, m, 256):
        want = x[a : a + 256].double() @ w.double().t()
        assert ((got[a : a + 256] - want).abs() <= (x[a : a + 256].double().abs() @ w.double().abs().t()) * kk * 2.0 ** -24).all()


@pytest.mark.parametrize("act,low,high", [(0, -80.0, -20.0), (0, -20.0, -1.0), (1, -1.0, -0.1)])
def test_an_activation_is_as_good_as_the_general_one(k, act, low, high):
    # The factor beside the gate is one, so the result is the activation rounded: it differs from the correctly rounded one where a
    # rounding line lies between, which for a mean error of e float32 units happens to e / 2^16 of the values.  0.36 to 0.41 units
    # are 6e-6 of them (0.5 with gelu's cubic: 8e-6), some 100 of 4,096 x 4,096; the lines stand four deviations above.  (Arguments
    # below zero: of a large one the activation is all but the argument itself, whose few bits lie on rounding lines.)
    m = n = 4096
    g = torch.Generator().manual_seed(51 + act)
    x, w = torch.zeros(m, 64), torch.zeros(2 * n, 64)
    x[:, 0], x[:, 1], x[:, 2] = (torch.rand(m, generator=g) - 0.5) * (high - low) * 0.5, torch.randn(m, generator=g) * 1e-3, 1.0
    w[:n, 0], w[:n, 1], w[:n, 2] = 1.0, torch.randn(n, generator=g), (torch.rand(n, generator=g) - 0.5) * (high - low) * 0.5 + (low + high) / 2
    w[n:, 2] = 1.0
    x, w = x.bfloat16().cuda(), w.bfloat16().cuda()
    z = run(k, x, w[:n].contiguous(), 0, 1, 1)[0].double()
    out = run(k, x, w, 0, 1, 2, act).double()
    y = z if act == 0 else 1.5957691216057308 * (z + 0.044715 * z * z * z)
    want = z / (1 + torch.exp(-y))
    unit = torch.exp2(torch.floor(torch.log2(want.abs())) - 7)
    want = torch.round(want / unit) * unit
    assert float((out != want).double().mean()) <= (8e-6 if act == 0 else 1.1e-5)


@pytest.mark.parametrize("m", [17, 33, 64])
def test_an_output_matrix_writes_where_it_is_told(k, m):
    # logits that do not begin on 16 bytes; what lies before and behind them stays
    n, kk = 65544, 64
    x, w = rnd(m, kk, seed=61), rnd(n, kk, seed=62)
    store = torch.full((m * n + 8,), -7.0, device="cuda")
    out = store[3 : 3 + m * n].view(m, n)
    assert k.linear(x, w, None, out) is out
    bound = (x.double().abs() @ w.double().abs().t()) * kk * 2.0 ** -24
    assert ((out.double() - x.double() @ w.double().t()).abs() <= bound).all()
    assert (store[:3] == -7).all() and (store[3 + m * n :] == -7).all()
