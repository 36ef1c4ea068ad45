"""Prompt attention in blocks of 32 rows: the workgroup shapes that prompts take, and what lies in pages beyond a context."""
import pytest
import torch

import test_gpu_decode_ranges as decode_ranges
from test_gpu_kernels import DEV, build_paged, k, run_paged  # noqa: F401  (k: the fixture)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hd,shape", [(64, 181), (128, 142), (128, 181)])
@pytest.mark.parametrize("window,ps,splits", [(0, 16, 1), (0, 64, 3), (100, 32, 1), (300, 16, 2)])
def test_workgroups_of_eight_wavefronts(k, hd, shape, window, ps, splits):  # noqa: F811
    # lengths at and around the tiles (64 or 128 keys) and the blocks of rows (128 or 256), wavefronts without rows, single tokens,
    # prefixes; the error is that of bfloat16 probabilities and results, as for every other shape
    seqs = [(300, 700), (1, 1), (64, 64), (65, 129), (2, 513), (1, 257), (127, 128), (17, 1000), (43, 43)]
    assert run_paged(k, seqs, 6, 2, hd, ps, torch.bfloat16, window=window, tiled_shape=shape, key_splits=splits) <= 1.2e-2
    assert run_paged(k, seqs, 7, 1, hd, ps, torch.bfloat16, window=window, tiled_shape=shape, key_splits=splits, ramp=0.9, seed=3) <= 1.2e-2


@pytest.mark.parametrize("hd,shape", [(64, 1142), (64, 1181), (128, 1142), (128, 1181), (64, 181), (128, 142), (128, 181)])
@pytest.mark.parametrize("ramp", [0.26, 0.9, -0.26, 4.0])
def test_scores_that_grow_along_long_contexts(k, hd, shape, ramp):  # noqa: F811
    # behind 1,536 keys the shapes from 1,000 on rescale a row only when its maximum has grown by 2^8: scores that rise by about 3 (in powers of
    # two) from one 64 keys to the next stay below that for several tiles in a row, a rise of 10 is over it in every tile, 45 by far; falling
    # scores never rescale after the first tile.  Blocks of rows on both sides of the 1,536, one head to a group and sixteen, a window
    seqs = [(300, 2500), (64, 64), (33, 1700), (200, 1600)]
    r = ramp * (hd / 64) ** 0.5
    assert run_paged(k, seqs, 6, 2, hd, 16, torch.bfloat16, tiled_shape=shape, seed=9, ramp=r) <= 1.2e-2
    assert run_paged(k, seqs, 3, 3, hd, 64, torch.bfloat16, window=700, tiled_shape=shape, seed=11, ramp=r) <= 1.2e-2
    assert run_paged(k, [(90, 2400), (1, 77)], 16, 1, hd, 32, torch.bfloat16, tiled_shape=shape, seed=12, ramp=r) <= 1.2e-2


@pytest.mark.parametrize("hd,shape", [(128, 142), (128, 1142), (64, 1142)])
@pytest.mark.parametrize("key_splits", [2, 3, 7])
def test_key_ranges_of_portions_behind_prefixes(k, hd, shape, key_splits):  # noqa: F811
    # prefixes of different lengths (one with fewer tiles of keys than workgroups that share them), a new prompt, a window; the keys' ramp
    # makes every far key count, so a range that is left out or taken twice shows
    seqs = [(70, 1300), (33, 33), (5, 2100), (130, 130), (40, 700)]
    assert run_paged(k, seqs, 6, 2, hd, 16, torch.bfloat16, tiled_shape=shape, key_splits=key_splits, seed=31, ramp=8.0 / 2100) <= 1.2e-2
    assert run_paged(k, seqs, 7, 1, hd, 64, torch.bfloat16, window=500, tiled_shape=shape, key_splits=key_splits, seed=32) <= 1.2e-2
    assert run_paged(k, [(96, 9000), (1, 5000), (40, 12001), (3, 3)], 6, 2, hd, 16, torch.bfloat16, tiled_shape=shape, key_splits=key_splits, seed=5) <= 1.2e-2


@pytest.mark.parametrize("hd,shape", [(64, 142), (64, 181), (128, 142), (128, 181), (64, 121), (128, 141)])
@pytest.mark.parametrize("window,ps", [(0, 16), (0, 64), (70, 32)])
def test_nothing_behind_the_context_counts(k, hd, shape, window, ps):  # noqa: F811
    # slots of a request's last page that hold no token, and pages of nobody, hold no numbers: the same bits
    seqs = [(130, 130), (9, 200), (1, 17), (61, 333)]
    nq, nkv, t = 6, 2, 201
    kc, vc, table, _, _ = build_paged(seqs, nkv, hd, ps, torch.bfloat16, seed=5)
    qkv = torch.randn(t, (nq + 2 * nkv) * hd, generator=torch.Generator().manual_seed(6)).to(torch.bfloat16).to(DEV)
    q_len = torch.tensor([q for q, _ in seqs], dtype=torch.int32)
    q_start = (torch.cumsum(q_len, 0, dtype=torch.int32) - q_len).to(DEV)
    q_len, kv_len = q_len.to(DEV), torch.tensor([kv for _, kv in seqs], dtype=torch.int32, device=DEV)
    outs = []
    for keys, vals in ((kc, vc), (torch.where(kc.abs() > 9e3, float("nan"), kc), torch.where(vc.abs() > 9e3, float("nan"), vc))):
        out = torch.empty(t, nq * hd, dtype=torch.bfloat16, device=DEV)
        k._run("egpt_paged_attention_tiled", qkv.data_ptr(), out.data_ptr(), keys.data_ptr(), vals.data_ptr(), table.data_ptr(), table.shape[1],
               q_start.data_ptr(), q_len.data_ptr(), kv_len.data_ptr(), len(seqs), t, nq, nkv, hd, ps, hd ** -0.5, window, shape, 1, None, None,
               0, 0, 0, k._stream())
        torch.cuda.synchronize()
        outs.append(out)
    assert torch.isfinite(outs[0].float()).all() and torch.equal(outs[0], outs[1])


@pytest.mark.parametrize("hd,least", [(64, 4), (128, 3)])
def test_key_ranges_of_the_fewest_tiles_that_the_rule_asks_for(k, hd, least):  # noqa: F811
    # portions behind a prefix whose tiles of 128 keys are dealt out in ranges of `least`: every workgroup has keys, and one range more
    # than that leaves the others as they were, with nothing for itself
    nq, nkv, ps, n, ranges = 6, 2, 16, 64, 8
    kv = ranges * least * 128
    assert k._portion_shape(n, nq, nkv, hd, ps, 32 * 128) == (1142, 32 // least)
    kc, vc, table, _, _ = build_paged([(n, kv)], nkv, hd, ps, torch.bfloat16, seed=2)
    qkv = torch.randn(n, (nq + 2 * nkv) * hd, generator=torch.Generator().manual_seed(4)).to(torch.bfloat16).to(DEV)
    one = lambda v: torch.tensor([v], dtype=torch.int32, device=DEV)  # noqa: E731
    start, length, context = one(0), one(n), one(kv)
    outs = []
    for splits in (ranges, ranges + 1):
        out = torch.empty(n, nq * hd, dtype=torch.bfloat16, device=DEV)
        part_o, part_ml = torch.empty(splits, n, nq, hd, device=DEV), torch.full((splits, n, nq, 2), 7.0, device=DEV)
        k._run("egpt_paged_attention_tiled", qkv.data_ptr(), out.data_ptr(), kc.data_ptr(), vc.data_ptr(), table.data_ptr(), table.shape[1], start.data_ptr(),
               length.data_ptr(), context.data_ptr(), 1, n, nq, nkv, hd, ps, hd ** -0.5, 0, 142, splits, part_o.data_ptr(), part_ml.data_ptr(), 0, 0, 0, k._stream())
        torch.cuda.synchronize()
        assert torch.isfinite(part_ml[:ranges, -1]).all() and torch.all(part_ml[ranges:, :, :, 0] == float("-inf"))
        outs.append(out)
    assert torch.equal(*outs)


@pytest.mark.parametrize("n", [4, 5, 64, 65, 130])
@pytest.mark.parametrize("hd,dtype,shape,line", [(64, torch.bfloat16, 24, 1.2e-2), (128, torch.bfloat16, 142, 1.2e-2), (48, torch.float32, None, 2e-6)])
def test_a_block_of_rows_finds_its_request_among_many(k, n, hd, dtype, shape, line):  # noqa: F811
    # n requests, the portions at the ends and in the middle: few are searched one after the other, many 64 at a time
    seqs = [(1, 1 + 7 * i % 40) for i in range(n)]
    seqs[0], seqs[n // 2], seqs[n - 1] = (70, 70), (9, 30), (133, 140)
    assert run_paged(k, seqs, 6, 2, hd, 16, dtype, tiled_shape=shape) <= line


@pytest.mark.parametrize("hd,nq,nkv", [(64, 14, 2), (128, 12, 2)])
@pytest.mark.parametrize("portions", [[(300, 900), (129, 129)], [(1000, 1000)], [(1800, 1800)]])
def test_portions_of_several_blocks_beside_decoded_tokens_in_one_launch(k, hd, nq, nkv, portions):  # noqa: F811
    decode_ranges.test_a_mixed_step_dealt_out(k, hd, nq, nkv, portions)


@pytest.mark.parametrize("hd,dtype,line", [(16, torch.float32, 2e-6), (64, torch.float32, 2e-6), (96, torch.bfloat16, 1.2e-2), (256, torch.float32, 2e-6)])
@pytest.mark.parametrize("window", [0, 9])
def test_decoded_tokens_of_one_segment(k, hd, dtype, line, window):  # noqa: F811
    # contexts of at most 64 tokens are one segment, whose result is written as it is; the same rows beside a longer context are folded
    # and have the same bits in float32.  (A score is hd products of size one, added up four at a time and divided by sqrt(hd): off by hd / 4
    # roundings of sums of sqrt(hd) at most, which with few keys to a row goes into the result: 3.8e-6 at 256.)
    line = max(line, hd / 4 * 2.0 ** -24)
    short = [(1, 1), (1, 16), (1, 17), (1, 33), (1, 63), (1, 64)]
    assert run_paged(k, short, 6, 2, hd, 16, dtype, window=window) <= line
    nq, nkv, b = 6, 2, len(short)
    outs = []
    kc, vc, table, _, _ = build_paged(short, nkv, hd, 16, dtype, seed=9)
    qkv = torch.randn(b, (nq + 2 * nkv) * hd, generator=torch.Generator().manual_seed(1)).to(dtype).to(DEV)
    one, start, kv = torch.ones(b, dtype=torch.int32, device=DEV), torch.arange(b, dtype=torch.int32, device=DEV), torch.tensor([n for _, n in short], dtype=torch.int32, device=DEV)
    wide = torch.nn.functional.pad(table, (0, 4), value=-1)
    for longest in (64, 128):                                # the launch's bound alone makes one segment or two
        out = torch.empty(b, nq * hd, dtype=dtype, device=DEV)
        k.paged_attention(qkv, out, kc, vc, wide.contiguous(), start, one, kv, nq, nkv, hd, 16, hd ** -0.5, window, 1, longest)
        outs.append(out)
    assert torch.equal(*outs)


def test_rows_are_rescaled_late_in_blocks_of_32_only(k):  # noqa: F811
    p = torch.zeros(1 << 16, device=DEV, dtype=torch.uint8).data_ptr()
    for shape in (1044, 1024, 1000, 2142):
        with pytest.raises(RuntimeError):
            k._run("egpt_paged_attention_tiled", p, p, p, p, p, 1, p, p, p, 1, 1, 2, 1, 64, 16, 0.1, 0, shape, 1, None, None, 0, 0, 0, k._stream())
    assert run_paged(k, [(64, 2000), (200, 1700)], 6, 2, 64, 16, torch.bfloat16, tiled_shape=1142, ramp=0.9, seed=3) <= 1.2e-2
