"""The rules by which the kernel wrappers choose workgroup shapes and split counts were measured at a few models'
sizes; between and beyond those they choose speed, not results, but what they return must always be something the
kernels take.  Checked here over a grid of sizes, on the CPU (the rules are plain functions of the sizes)."""
import itertools

import pytest
import torch

from emulated_kernels import EmulatedKernels
from easy_gpt.cpp_amd import kernels
from easy_gpt.cpp_amd.engine.engine import _same_portion, _same_spread, _spread
from easy_gpt.cpp_amd.kernels.hip import HipKernels as K

BATCHES = [1, 2, 3, 7, 8, 16, 17, 31, 32, 33, 48, 63, 64, 65, 100, 128, 200, 256, 257, 512, 1000, 4096]
CONTEXTS = [1, 15, 16, 33, 64, 100, 511, 512, 2048, 2049, 4096, 8192, 9216, 32640, 131072, 1000000]


def test_decode_attention_shapes_are_launchable():
    for b, nkv, hd, ctx, combine in itertools.product(BATCHES, [1, 2, 3, 4, 8, 16, 40], [64, 128], CONTEXTS, [True, False]):
        n_splits, n_waves, lean = K._decode_shape(b, nkv, hd, ctx, combine)
        what = (b, nkv, hd, ctx, combine, n_splits, n_waves, lean)
        assert 1 <= n_splits <= 64 and n_waves in (1, 2, 4, 8) and lean in (0, 1), what
        # the kernel's LDS: a wavefront's 16 rows of head size + 2 floats, and the fused variant's queries, key and value
        lds = n_waves * 16 * (hd + 2) * 4 + 18 * hd * 2
        assert lds <= 96 * 1024, what


def test_decode_attention_takes_rounds_of_one_block_where_no_wavefront_has_two():
    for b, nkv, hd, ctx in itertools.product(BATCHES, [1, 2, 3, 4, 8, 16, 40], [64, 128], CONTEXTS + [129, 250, 256, 600]):
        n_splits, n_waves, lean = K._decode_shape(b, nkv, hd, ctx, True)
        one = -(-(-(-ctx // 32)) // (n_splits * n_waves)) == 1
        assert not one or lean == 1, (b, nkv, hd, ctx)
        assert K._decode_form(n_splits, n_waves, lean, hd, ctx) == (2 if one and hd == 64 else lean), (b, nkv, hd, ctx)


def test_shapes_of_new_prompts():
    # (tokens, nq, nkv, head size, page size, longest context) and the workgroup shape, at and around the lines
    for sizes, shape in [((580, 14, 2, 64, 16, 580), 24), ((590, 14, 2, 64, 16, 590), 44), ((1300, 14, 2, 64, 16, 1300), 44), ((1400, 14, 2, 64, 16, 700), 44),
                         ((1755, 14, 2, 64, 16, 1755), 44), ((1756, 14, 2, 64, 16, 1756), 1142), ((1200, 14, 2, 64, 16, 100), 142),
                         ((1100, 14, 2, 64, 16, 100), 44), ((1800, 14, 2, 64, 128, 1800), 44), ((2400, 14, 2, 64, 128, 2400), 42),
                         ((200, 12, 2, 128, 16, 200), 22), ((300, 12, 2, 128, 16, 300), 42), ((400, 12, 2, 128, 16, 400), 142),
                         ((1000, 28, 4, 128, 128, 1000), 42), ((6500, 14, 2, 64, 16, 6500), 1181),
                         ((800, 28, 4, 128, 16, 800), 1142), ((500, 28, 4, 128, 16, 500), 142), ((512, 28, 4, 128, 16, 4096), 1142),
                         ((512, 28, 4, 128, 16, 1000), 142), ((2400, 14, 2, 64, 16, 600), 1142), ((2400, 14, 2, 64, 16, 400), 1181),
                         ((2800, 14, 2, 64, 16, 700), 1181), ((2800, 12, 2, 128, 16, 700), 1181), ((2800, 12, 2, 128, 16, 701), 1142)]:
        assert K._portion_shape(*sizes) == (shape, 1), sizes


def test_split_counts_of_the_products_leave_no_range_empty():
    widths = [64, 72, 896, 1000, 1536, 2048, 3584, 4864, 5120, 8192, 8960, 13824, 18944, 27648, 151936]
    for m, n, k in itertools.product([1, 8, 16, 17, 32, 33, 64], widths, widths):
        s = K._n_splits(m, n, k)
        steps = -(-k // 128)
        assert 1 <= s <= steps and (s - 1) * -(-steps // s) < steps, (m, n, k, s)
    for n, k in itertools.product(widths, widths):
        s = K._f32_splits(n, k)
        steps = -(-k // 64)
        assert 1 <= s <= min(steps, 12) and (s - 1) * -(-steps // s) < steps, (n, k, s)
        s, waves = K._normed_shape(n, k)
        steps = -(-k // 128)
        assert 1 <= s <= steps and (s - 1) * -(-steps // s) < steps and waves in (4, 8, 16), (n, k, s, waves)


def test_which_rows_go_to_the_library_is_monotonic_in_the_rows():
    # up to 16 rows never, beyond 64 always, and a product that goes there at some number of rows goes there at more
    widths = [64, 896, 1536, 2048, 3584, 4608, 5120, 9728, 18944, 151936]
    for n, k in itertools.product(widths, widths):
        rows = (1, 16, 17, 24, 32, 33, 48, 64, 65, 2048)
        goes = [K._library_rows(m, n, k) for m in rows]
        assert goes[:2] == [False, False] and goes[-2:] == [True, True], (n, k, goes)
        assert goes == sorted(goes), (n, k, goes)


def test_products_of_many_rows_leave_their_kernel_where_the_library_is_faster():
    # (rows, n, k) with both sides measured more than the runs differ when the lines were drawn
    own = [(96, 896, 896), (300, 1152, 896), (2048, 896, 896), (200, 512, 1024), (1000, 1024, 1024), (128, 1536, 1536), (200, 2048, 2048),
           (200, 3584, 3584), (200, 4608, 3584), (450 - 2, 5120, 5120), (300, 1024, 2048), (1000, 1024, 4096), (650, 1024, 3072), (1500, 896, 4864),
           (640, 2048, 5632), (1500, 5120, 13824), (2048, 4096, 14336), (3500, 2048, 11008), (3584, 3584, 18944)]
    library = [(2800, 1152, 896), (2800, 512, 1024), (1536, 3072, 1024), (1500, 1536, 1536), (650, 2048, 2048), (1500, 2048, 1536),
               (552, 3584, 3584), (448, 4608, 3584), (1500, 4096, 4096), (320, 4096, 2048), (552, 1024, 2048), (1000, 1024, 2048),
               (1500, 1024, 3072), (1500, 1024, 4096), (1536, 2048, 4096), (5000, 896, 4864), (2048, 5120, 13824), (2500, 4096, 14336),
               (5000, 2048, 11008)]
    for sizes in own:
        assert K._own_rows(*sizes, False), sizes
    for sizes in library:
        assert not K._own_rows(*sizes, False), sizes
    unrounded = [(96, 896, 896), (1500, 1152, 896), (1293, 2752, 896), (85, 768, 768), (65, 256, 256)]
    rounded_only = [(2048, 1152, 896), (96, 1152, 1152), (200, 2048, 2048), (552, 3584, 18944)]
    for sizes in unrounded:
        assert K._own_rows(*sizes, True), sizes
    for sizes in rounded_only:
        assert not K._own_rows(*sizes, True), sizes


def test_gate_and_up_leave_their_kernel_where_the_library_is_faster():
    # (rows, k) with both sides measured more than the runs differ when the lines were drawn, over matrices of 4,096 to 37,888 rows
    for m, k in [(65, 896), (2048, 896), (8191, 896), (1000, 1024), (96, 1536), (2500, 1536), (500, 2048), (2048, 2048), (2500, 2560), (200, 3584),
                 (1200, 3584), (2048, 3584), (2500, 3072), (500, 5120)]:
        assert K._own_gate(m, k), (m, k)
    for m, k in [(70, 3072), (128, 3072), (70, 3584), (300, 4096), (2048, 4096), (4096, 8192), (3500, 3584), (5000, 5120), (8191, 2048), (8191, 3072)]:
        assert not K._own_gate(m, k), (m, k)


def test_a_plan_is_found_once_for_its_sizes():
    for plan, sizes in ((K._rows_plan, (101, 896, 4864, 10)), (K._f32_rows_plan, (101, 896, 4864, 11))):
        first, before = plan(*sizes), plan.cache_info()
        assert all(plan(*sizes) == first for _ in range(24))         # a step's layers
        after = plan.cache_info()
        assert after.hits == before.hits + 24 and after.misses == before.misses and after.maxsize is not None


WIDTHS = [64, 128, 320, 896, 1024, 1152, 1536, 2048, 2752, 3584, 4608, 4864, 8960, 9728, 18944, 37888, 151936]
ROWS = [65, 66, 96, 127, 128, 129, 192, 256, 257, 448, 552, 1000, 1537, 2048, 3584, 4097, 8191, 32768, 100003]


def test_plans_of_many_rows_are_launchable():
    # what egpt_gemm_rows refuses: shapes that do not exist, empty ranges of k, more workgroups than a grid holds
    for m, n, k, (most, form) in itertools.product(ROWS, WIDTHS, [w for w in WIDTHS if w % 64 == 0], ((1, 0), (10, 0), (10, 1), (1, 2))):
        shape, s = K._rows_plan(m, n, k, most, form)
        bm, bn = K._rows_shapes[shape][:2]
        steps = k // 64
        per = -(-steps // s)
        what = (m, n, k, most, form, shape, s)
        assert 1 <= s <= min(most, steps) and (s - 1) * per < steps, what
        assert -(-m // bm) * -(-n // bn) * s <= 0x7FFFFFFF, what


def test_plans_of_the_float32_product_are_launchable():
    # what egpt_gemm_f32 and egpt_gemm_f32_rows refuse; up to 64 rows always the kernel for few, nothing is folded there
    for m, n, k in itertools.product([1, 17, 64] + ROWS, WIDTHS + [5, 36], WIDTHS + [4, 100]):
        for s in {1, K._f32_splits(n, k)}:
            rows, fold = K._f32_rows_plan(m, n, k, s)
            what = (m, n, k, s, rows, fold)
            assert rows in ((0,) if m <= 64 else (0, 64, 128)), what
            assert not fold or (s > 1 and rows), what
            if rows:
                assert -(-m // rows) * -(-n // 128) <= 0x7FFFFFFF, what
            else:
                assert -(-m // 64) <= 65535 and s <= 65535, what


def test_the_rules_for_many_rows_change_sides_once():
    # more rows than a product that goes to the library go there too; a gate product leaves its kernel for good as rows grow,
    # and on large matrices begins with the library
    rows = list(range(65, 9000, 61))
    for n, k, unrounded in itertools.product(WIDTHS, WIDTHS, (False, True)):
        own = [K._own_rows(m, n, k, unrounded) for m in rows]
        assert own == sorted(own, reverse=True), (n, k, unrounded)
    for k in WIDTHS + [3072, 4096, 5120, 8192]:
        own = [K._own_gate(m, k) for m in rows]
        assert sum(a != b for a, b in zip(own, own[1:])) <= 2, k


def test_a_product_comes_back_from_the_library_once_at_most():
    # both rules together: own, then perhaps the library, then perhaps own for good; with a long k no way back
    rows = list(range(65, 20000, 61))
    for n, k, unrounded in itertools.product(WIDTHS + [448, 2688], WIDTHS + [640, 768], (False, True)):
        own = [K._own_many(m, n, k, unrounded) for m in rows]
        assert own[0] or k > 896, (n, k, unrounded)
        assert sum(a != b for a, b in zip(own, own[1:])) <= (2 if 640 < k <= 896 else 0 if 256 <= k <= 640 else 1), (n, k, unrounded)
    # (rows, n, k, unrounded) with both sides measured more than the runs differ
    for sizes in [(2304, 512, 512, False), (8191, 1920, 640, False), (2600, 896, 896, False), (8191, 896, 896, False), (16384, 896, 896, True),
                  (4000, 2688, 896, False), (5000, 2688, 896, True), (5000, 9728, 896, True)]:
        assert K._own_many(*sizes), sizes
    for sizes in [(5000, 896, 896, False), (6000, 896, 896, False), (3300, 768, 768, True), (2048, 2688, 896, True), (2048, 9728, 896, True),
                  (5000, 1024, 1024, False), (8191, 1024, 128, False), (4000, 4096, 64, False)]:
        assert not K._own_many(*sizes), sizes


def test_few_row_plans_are_launchable():
    # what egpt_gemm_rows refuses: an empty range, or splits of a result that is not float32
    for n, k, most in itertools.product(WIDTHS + [8, 16384, 16392, 32776], [w for w in WIDTHS if w % 64 == 0], (1, 8, 16)):
        shape, s = K._few_plan(n, k, most)
        steps = k // 64
        assert 4 <= shape <= 6 and 1 <= s <= most and (s - 1) * -(-steps // s) < steps, (n, k, most)
        assert s == 1 or (s * -(-n // 64) <= 256 and -(-steps // s) >= 2), (n, k, most)


def test_products_in_parts_take_no_more_than_their_reader():
    for m, n, k in itertools.product(ROWS, WIDTHS, [w for w in WIDTHS if w % 64 == 0]):
        shape, s = K._rows_plan(m, n, k, K.rope_parts, 1)
        assert 1 <= s <= K.rope_parts and (s - 1) * -(-(k // 64) // s) < k // 64, (m, n, k, shape, s)
    for n, k in itertools.product(WIDTHS, WIDTHS):
        own = [K._own_parts(m, n, k) for m in ROWS]
        assert own == sorted(own, reverse=True), (n, k)


def test_keys_are_dealt_out_where_a_kernel_reads_the_table():
    f32, bf16 = torch.float32, torch.bfloat16
    # (nq, nkv, hd, page size, requests, longest context, spread)
    assert K.deals_out(bf16, 12, 2, 128, 16, 40, 2048, 1) and K.deals_out(bf16, 14, 2, 64, 16, 32, 8192, 2)
    assert K.deals_out(bf16, 12, 2, 128, 16, 24, 32768, 2)                          # the longer the better
    assert not K.deals_out(f32, 12, 2, 128, 16, 40, 2048, 2)                        # other kernels' dtype, head size, heads, pages
    assert not K.deals_out(bf16, 12, 2, 96, 16, 40, 2048, 2) and not K.deals_out(bf16, 34, 2, 64, 16, 40, 2048, 2)
    assert not K.deals_out(bf16, 12, 2, 128, 8, 40, 2048, 2)
    assert not K.deals_out(bf16, 14, 2, 64, 16, 64, 2048, 1) and not K.deals_out(bf16, 12, 2, 128, 16, 40, 2048, 0)      # even contexts
    assert not K.deals_out(bf16, 12, 2, 128, 16, 16, 2048, 2) and not K.deals_out(bf16, 12, 2, 128, 16, 72, 2048, 2)     # few, many
    # beside portions of prompts
    assert K.deals_out(bf16, 12, 2, 128, 16, 41, 2048) and K.deals_out(bf16, 14, 2, 64, 16, 64, 4096)
    assert not K.deals_out(bf16, 12, 2, 128, 16, 41, 1024) and not K.deals_out(bf16, 14, 2, 64, 16, 64, 2048)
    assert not K.deals_out(f32, 12, 2, 128, 16, 41, 2048) and not K.deals_out(bf16, 12, 2, 128, 48, 41, 2048)
    assert not K.deals_out(bf16, 12, 2, 128, 16, 129, 2048)
    # the kernels' limits: a slot for every request, at most 256 of them
    for nkv, b, spread in itertools.product((1, 2, 3, 4, 8, 40), range(1, 300), (None, 0, 1, 2)):
        if K.deals_out(bf16, nkv, nkv, 128, 16, b, 1 << 15, spread):
            assert b <= 256 // nkv <= 256


def test_how_uneven_contexts_are():
    assert _spread([5000] + [10] * 15) == 0                                         # up to 16 nothing goes by it
    assert _spread([700] * 17) == 0 and _spread([13] * 17 + [18]) == 0
    assert _spread([100] * 19 + [150]) == 1 and _spread([100] * 19 + [268]) == 1
    assert _spread([100] * 19 + [280]) == 2 and _spread([1] * 40 + [4000]) == 2


def attention_of(dtype, heads, kv_heads, head_dim, window=None):
    from easy_gpt.cpp_amd.parts import PartSpec, make_part

    part = make_part("mixer", PartSpec("gq_attention", dict(n_heads=heads, n_kv_heads=kv_heads, head_dim=head_dim, qkv_bias=False, out_bias=False,
                                                            window=window, position=PartSpec("rope_half_split", dict(theta=1e4))), "a."), hidden_size=64)
    width = (heads + 2 * kv_heads) * head_dim
    part.load(lambda name: torch.zeros((heads * head_dim if "q_proj" in name else kv_heads * head_dim, 64) if "o_proj" not in name
                                       else (64, heads * head_dim)), dtype, "cpu")
    assert part.w_qkv.shape == (width, 64)
    return part


class RulesOnly(EmulatedKernels):
    deals_out, portion_choice, window_portion_choice = K.deals_out, K.portion_choice, K.window_portion_choice


@pytest.fixture()
def rules_only():
    kernels.use_backend(RulesOnly())
    yield
    kernels.use_backend(None)


def test_steps_with_the_same_kernels_are_kept_by_the_same_hints(rules_only):
    bf16, f32 = torch.bfloat16, torch.float32
    spread = lambda part, rows, most, s: _same_spread(lambda v: part.step_choices(16, rows, rows, most, v, None), s)  # noqa: E731
    wide, narrow = attention_of(bf16, 12, 2, 128), attention_of(bf16, 14, 2, 64)
    assert [spread(wide, 40, 2048, s) for s in (0, 1, 2)] == [0, 1, 1] and [spread(narrow, 40, 2048, s) for s in (0, 1, 2)] == [0, 0, 2]
    for part, rows in ((attention_of(f32, 12, 2, 128), 40), (attention_of(bf16, 12, 2, 96), 40), (wide, 72), (attention_of(bf16, 40, 2, 64), 40)):
        assert [spread(part, rows, 2048, s) for s in (0, 1, 2)] == [0, 0, 0]

    def portion(part, tokens, longest, most):
        return _same_portion(lambda n: part.step_choices(16, tokens, 8, most, None, n), tokens, longest, most)

    # below the prefixes' line one bound for all, so a prompt of 2,048 tokens in portions of 512 has one graph
    assert {portion(narrow, 512, n, 4096) for n in (512, 600, 1024, 1536, 2048)} == {2048}
    assert {portion(wide, 512, n, 1024) for n in (512, 600, 1024)} == {1024}
    # behind a prefix as many workgroups share the keys as there are CUs for, however far it goes
    assert portion(wide, 512, 600, 4096) == 1024 and portion(wide, 512, 1536, 4096) == 4096 and portion(narrow, 512, 4000, 32768) == 32768
    assert portion(narrow, 64, 2500, 32768) == 4096
    assert {portion(attention_of(f32, 14, 2, 64), 512, n, 32768) for n in (512, 5000, 30000)} == {32768}
    # always a bound, and the choice is that of the context's own bound
    for part, tokens, most in itertools.product((wide, narrow), (64, 192, 512, 2048), (256, 1024, 4096, 32768)):
        for longest in (1, 65, 500, 1025, 2048, 4097, 9000, 32768):
            if longest <= most:
                bound = portion(part, tokens, longest, most)
                own = tokens
                while own < longest:
                    own *= 2
                assert longest <= bound <= most
                assert part.step_choices(16, tokens, 8, most, None, bound) == part.step_choices(16, tokens, 8, most, None, min(own, most))


def test_heads_by_themselves_are_kept_by_what_lies_in_front_of_portions(rules_only):
    from easy_gpt.cpp_amd.parts import PartSpec, make_part

    assert K._heads_portion(96, 96) and K._heads_portion(800, 300) and not K._heads_portion(95, 95) and not K._heads_portion(800, 801)

    def part(dtype, dim=64, **kw):
        p = make_part("mixer", PartSpec("normed_attention", dict(n_heads=4, n_kv_heads=2, key_dim=dim, value_dim=dim, scale=0.1, eps=1e-6, **kw), "a."), hidden_size=32)
        p.load(lambda name: torch.zeros(next(s for s in p.param_specs() if s.name == name).shape), dtype, "cpu")
        return p

    bound = lambda p, tokens, longest, most: _same_portion(lambda n: p.step_choices(16, tokens, 8, most, None, n), tokens, longest, most)  # noqa: E731
    plain = part(torch.bfloat16)
    # two kinds of steps of one size: new prompts, and portions behind a prefix, however long; one where nothing goes by it
    assert bound(plain, 512, 300, 4096) == 512 and {bound(plain, 512, n, 4096) for n in (513, 1024, 4096)} == {4096}
    assert bound(plain, 64, 64, 4096) == bound(plain, 64, 3000, 4096) == 4096
    for other in (part(torch.float32), part(torch.bfloat16, 96), part(torch.bfloat16, sink=True), part(torch.bfloat16, softcap=30.0),
                  part(torch.bfloat16, window=100), part(torch.bfloat16, window=500, keep_first=4), part(torch.bfloat16, gated="heads")):
        assert {bound(other, 512, n, 4096) for n in (300, 513, 4096)} == {4096}
    assert plain.step_choices(16, 40, 40, 4096, 1, None) is None
