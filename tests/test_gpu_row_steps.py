"""Steps of few tokens, laid out as rows: one graph for a number of tokens whatever is wanted of them, and the wanted rows in order."""
import pytest
import torch

import helpers as H
from conftest import TINY

pytestmark = pytest.mark.gpu


def test_one_graph_whatever_is_wanted(tiny_models):
    from easy_gpt.cpp_amd import kernels
    from easy_gpt.cpp_amd.engine import Engine, StepEntry

    kernels.use_backend(None)
    load = lambda graphs: Engine.from_dir(tiny_models["A"], dtype="float32", device="cuda:0", page_size=16, max_tokens=512, max_requests=8, use_graphs=graphs)  # noqa: E731
    eng, plain = load(True), load(False)
    counts = [5, 1, 7]
    texts = list(H.make_requests(TINY["A"][0]["vocab_size"], counts, seed=4).values())
    wants = [[(4,), (0,), (6,)], [(0, 4), (), (2, 3, 6)], [(), (), (1,)], [(4, 0, 0), (0, 0), (6, 6, 5)], [tuple(range(5)), (0,), tuple(range(7))], [(), (), ()],
             [tuple(range(5)) * 2, (0,), tuple(range(7)) * 2], [(3,) * 40, (0,) * 3, ()]]          # also more rows than there are tokens
    for again in range(2):                                   # captured, and replayed
        for want in wants:
            got = []
            for e in (eng, plain):
                for i in range(3):
                    e.add_request(i)
                out = e.step([StepEntry(i, t, w) for i, (t, w) in enumerate(zip(texts, want))])
                got.append(None if out is None else out.clone())
                for i in range(3):
                    e.finish(i)
            if not any(want):
                assert got == [None, None]
                continue
            assert got[0].shape == got[1].shape == (sum(map(len, want)), TINY["A"][0]["vocab_size"])
            assert float((got[0] - got[1]).abs().max()) <= 2e-5 * float(got[1].abs().max()), want       # (the orders of sums of 32 bits)
    assert len(eng._row_plans) == 1 and next(iter(eng._row_plans.values())).graph is not None
