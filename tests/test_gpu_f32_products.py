"""The float32 product on bfloat16 parts (gemm.hip): the same bits in every kernel and batch, float32's precision, and values that
have no parts."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def k():
    from easy_gpt.cpp_amd import kernels

    return kernels.backend()


def rnd(*shape, seed, scale=1.0):
    return (torch.randn(*shape, generator=torch.Generator().manual_seed(seed)) * scale).cuda()


def few(k, x, w, splits, bias=None):
    out = torch.full((splits, x.shape[0], w.shape[0]), float("nan"), device="cuda")
    k._run("egpt_gemm_f32", x.data_ptr(), w.data_ptr(), k._ptr(bias), out.data_ptr(), x.shape[0], w.shape[0], x.shape[1], splits, k._stream())
    return out


def many(k, x, w, splits, fold, rows, bias=None):
    out = torch.full((1 if fold else splits, x.shape[0], w.shape[0]), float("nan"), device="cuda")
    k._run("egpt_gemm_f32_rows", x.data_ptr(), w.data_ptr(), k._ptr(bias), out.data_ptr(), x.shape[0], w.shape[0], x.shape[1], splits,
           int(fold), rows, k._stream())
    return out


def in_order(parts):
    total = parts[0].clone()
    for p in parts[1:]:
        total += p
    return total


SIZES = [(1, 1, 4, 1), (17, 130, 36, 1), (64, 5, 64, 1), (65, 127, 100, 2), (127, 260, 192, 3), (129, 129, 896, 14), (300, 68, 2052, 11),
         (16, 68, 896, 1), (33, 20, 580, 1)]


@pytest.mark.parametrize("m,n,kk,splits", SIZES)
def test_all_kernels_leave_the_same_bits(k, m, n, kk, splits):
    x, w = rnd(m, kk, seed=1), rnd(n, kk, seed=2)
    want = few(k, x, w, splits)
    for rows in (64, 128):
        assert torch.equal(many(k, x, w, splits, False, rows), want)
        assert torch.equal(many(k, x, w, splits, True, rows)[0], in_order(want))
    bias = rnd(n, seed=3)
    for rows in (64, 128):
        assert torch.equal(many(k, x, w, 1, False, rows, bias), few(k, x, w, 1, bias))
    for r in (0, m // 2, m - 1):                             # and a row alone those of the row in its batch
        assert torch.equal(few(k, x[r : r + 1].contiguous(), w, splits)[:, 0], want[:, r])
    # nearer to 64 bits than a chain of float32 operations: a block of 32 values is rounded once
    exact = x.double() @ w.double().t()
    bound = (x.double().abs() @ w.double().abs().t()) * 2.0 ** -24 * (kk / 32 + splits + 8)
    assert ((in_order(want).double() - exact).abs() <= bound).all()


@pytest.mark.parametrize("m", [5, 70])
def test_a_result_that_is_not_aligned(k, m):
    """Four values are one store only where the result begins at 16 bytes; beside it nothing is written."""
    x, w = rnd(m, 64, seed=8), rnd(36, 64, seed=9)
    want = few(k, x, w, 1)[0]
    for rows in (0, 64, 128):
        whole = torch.full((m * 36 + 8,), 7.0, device="cuda")
        out = whole[1 : 1 + m * 36].view(m, 36)
        k._f32_product(x, w, None, out, 1, (rows, False))
        assert torch.equal(out, want) and whole[0] == 7 and (whole[1 + m * 36 :] == 7).all()


@pytest.mark.parametrize("m", [3, 70, 200, 700, 1900])
@pytest.mark.parametrize("n,kk", [(256, 896), (130, 4864), (1300, 64)])
def test_the_backend_gives_a_row_the_same_bits_in_any_batch(k, m, n, kk):
    x, w = rnd(m, kk, seed=4), rnd(n, kk, seed=5)
    total = in_order(k.product(x, w))
    for r in (0, m - 1):
        assert torch.equal(in_order(k.product(x[r : r + 1].contiguous(), w))[0], total[r])


@pytest.mark.parametrize("kernel", ["few", 64, 128])
def test_values_without_parts(k, kernel):
    """Infinities, NaN and numbers beyond the largest bfloat16 come out as plain float32 gives them, rows beside them as ever."""
    x, w = rnd(40, 96, seed=6), rnd(24, 96, seed=7)
    clean = few(k, x, w, 2)
    x[3, 7], x[5, 1], x[6, 2], x[7, 4], x[8], x[9, 40] = float("inf"), float("nan"), 3.4e38, -float("inf"), 1e25, 1e-39
    x[10, 64] = 3.4028e38
    w2 = w.clone()
    w2[9, 2], w2[11], w2[13, 70], w2[9, 64] = 1e-30, 1e25, float("inf"), 1e-30
    run = (lambda a, b: few(k, a, b, 2)) if kernel == "few" else (lambda a, b: many(k, a, b, 2, False, kernel))
    got = in_order(run(x, w2))
    ref = torch.zeros_like(got)
    for at in (0, 64):                                       # plain float32 in two ranges, product after product
        part = torch.zeros_like(got)
        for i in range(at, min(at + 64, 96)):
            part = part + x[:, i : i + 1] * w2[:, i]
        ref = ref + part
    assert torch.equal(torch.isnan(got), torch.isnan(ref)) and torch.equal(torch.isinf(got), torch.isinf(ref))
    fin = torch.isfinite(ref)
    assert torch.equal(got[~fin & ~torch.isnan(ref)], ref[~fin & ~torch.isnan(ref)])
    scale = (x.double().abs() @ w2.double().abs().t())[fin]
    assert ((got - ref).double().abs()[fin] <= scale * 1e-6).all()
    same = [c for c in range(24) if c not in (9, 11, 13)]
    rows = [r for r in range(40) if r not in (3, 5, 6, 7, 8, 9, 10)]
    assert torch.equal(in_order(run(x, w))[rows], in_order(clean)[rows])
    assert torch.equal(got[rows][:, same], in_order(clean)[rows][:, same])
    if kernel != "few":
        assert torch.equal(many(k, x, w2, 2, True, kernel)[0].nan_to_num(7.0), got.nan_to_num(7.0))


def time_of(f):
    """Microseconds of one call, the shortest of several."""
    f()
    times = []
    for _ in range(8):
        start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        start.record()
        f()
        end.record()
        torch.cuda.synchronize()
        times.append(start.elapsed_time(end) * 1e3)
    return min(times)


@pytest.mark.parametrize("m,most", [(8, 4.0), (1811, 8.0)])
@pytest.mark.parametrize("value", [float("nan"), float("inf"), 3.4e38])
def test_rows_without_parts_stay_cheap(k, m, most, value):
    """A stream that holds NaN or infinities has them in every later product: such rows are added up by wavefronts, tile by tile,
    not by a lane an element (which took 17 and 130 times as long as numbers for eight and for 1,811 rows; now 1.7 and 3.3 times)."""
    x, w = rnd(m, 896, seed=11), rnd(9728, 896, seed=12)
    numbers = time_of(lambda: k.product(x, w))
    x[:, 5] = value
    assert not torch.isfinite(in_order(k.product(x, w))).all()
    assert time_of(lambda: k.product(x, w)) < most * numbers


@pytest.mark.parametrize("m,n,kk,splits", [(1, 16, 4, 1), (17, 130, 36, 1), (65, 127, 100, 2), (130, 260, 580, 3)])
@pytest.mark.parametrize("kernel", ["few", 64, 128])
def test_every_place_of_a_value_without_parts(k, m, n, kk, splits, kernel):
    """One such value at a time, in the first and last row, column and place of k: its row (or column) is NaN or infinite as in
    float64, everything else as it was."""
    run = (lambda a, b: few(k, a, b, splits)) if kernel == "few" else (lambda a, b: many(k, a, b, splits, False, kernel))
    x, w = rnd(m, kk, seed=13), rnd(n, kk, seed=14)
    clean = in_order(run(x, w))
    for where in (0, kk // 2, kk - 1):
        for value in (float("nan"), float("inf")):
            for row in {0, m - 1}:
                bad = x.clone()
                bad[row, where] = value
                got, want = in_order(run(bad, w)), clean.clone()
                want[row] = value * w[:, where]
                assert torch.equal(got.nan_to_num(7.0, 8.0, 9.0), want.nan_to_num(7.0, 8.0, 9.0))
            for col in {0, n - 1}:
                bad = w.clone()
                bad[col, where] = value
                got, want = in_order(run(x, bad)), clean.clone()
                want[:, col] = value * x[:, where]
                assert torch.equal(got.nan_to_num(7.0, 8.0, 9.0), want.nan_to_num(7.0, 8.0, 9.0))


@pytest.mark.parametrize("kernel", ["few", 64, 128])
@pytest.mark.parametrize("small_w", [False, True])
@pytest.mark.parametrize("power", [-100, -112, -120, -124, -126, -128, -132, -140, -146])
def test_small_operands_keep_their_bits(k, kernel, small_w, power):
    """A whole operand of values around 2^power against large partners: float32's error of the product, down into the subnormals
    (whose own bits are the float32 numbers that both sides are given).  A block of 32 values is rounded once and the blocks'
    sum 28 times: 2^-24 sqrt(28 + 1) = 3.2e-7 in the 2-norm, were all roundings of the largest size and of random sign."""
    small, large = rnd(70, 896, seed=15), rnd(130, 896, seed=16) * 2.0 ** 60
    small = (small.double() * 2.0 ** power).float()
    assert small.abs().max() < 2.0 ** (power + 3) and small.abs().max() > 0
    x, w = (large, small) if small_w else (small, large)
    got = few(k, x, w, 1)[0] if kernel == "few" else many(k, x, w, 1, False, kernel)[0]
    exact = x.double() @ w.double().t()
    assert (got.double() - exact).norm() <= 3.2e-7 * exact.norm()


def test_small_operands_beside_others(k):
    """The result's own range: ordinary rows, rows below 2^-126 whose products are subnormal, and rows whose one value below 2^-126
    meets the only value of its column."""
    x, w = rnd(40, 192, seed=17), rnd(48, 192, seed=18)
    clean = few(k, x, w, 1)[0]
    x[3] = (x[3].double() * 2.0 ** -130).float()
    x[7], x[7, 5], w2 = 0.0, 1.2345e-39, w.clone()
    w2[9], w2[9, 5] = 0.0, 3.0
    for run in (lambda a, b: few(k, a, b, 1)[0], lambda a, b: many(k, a, b, 1, False, 64)[0], lambda a, b: many(k, a, b, 1, False, 128)[0]):
        got = run(x, w2)
        exact = x.double() @ w2.double().t()
        # six blocks are rounded, each result to a multiple of 2^-149 at best
        bound = 2.0 ** -24 * 8 * (x.double().abs() @ w2.double().abs().t()) + 7 * 2.0 ** -150
        assert ((got.double() - exact).abs() <= bound).all()
        same = [r for r in range(40) if r not in (3, 7)]
        columns = [c for c in range(48) if c != 9]
        assert torch.equal(got[same][:, columns], clean[same][:, columns])


@pytest.mark.parametrize("act", ["silu", "gelu_tanh"])
@pytest.mark.parametrize("m,inter,kk", [(65, 4, 4), (66, 31, 36), (127, 33, 100), (128, 64, 64), (129, 65, 896), (193, 130, 580), (300, 96, 2052),
                                        (700, 4864, 896)])
def test_the_gated_form_leaves_the_bits_of_product_and_activation(k, m, inter, kk, act):
    x, w = rnd(m, kk, seed=5), rnd(2 * inter, kk, seed=6, scale=kk ** -0.5)
    if kk > 500:
        x[3, 7], w[inter // 2, 11] = float("inf"), float("nan")
    splits = k._f32_splits(2 * inter, kk)
    parts = few(k, x, w, splits)
    want = torch.empty((m, inter), device="cuda")
    k.swiglu(parts, want, activation=act)
    for rows in (64, 128):
        out = torch.full((m, inter), 7.0, device="cuda")
        k._run("egpt_gemm_f32_gated", x.data_ptr(), w.data_ptr(), out.data_ptr(), m, inter, kk, splits, rows, 0 if act == "silu" else 1,
               k._stream())
        assert torch.equal(out.nan_to_num(nan=1e30), want.nan_to_num(nan=1e30)) and torch.equal(out.isnan(), want.isnan())
    got = k.gate_up_rows(x, w, activation=act)
    assert got is None or torch.equal(got.nan_to_num(nan=1e30), want.nan_to_num(nan=1e30))
    assert got is not None or inter < 4864
