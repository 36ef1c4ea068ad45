"""A mixture's shared branch beside the experts' sum, on the CPU with the tests' stand-in for the kernels: where the backend writes sums in
place the two are one tensor, and a branch that replaces the dense feed-forward's `forward` is still the one that runs."""
import pytest
import torch

from emulated_kernels import EmulatedKernels
from easy_gpt.cpp_amd import kernels
from easy_gpt.cpp_amd.parts.expert_mixture import ExpertMixture
from easy_gpt.cpp_amd.parts.feed_forward import SwiGLU
from easy_gpt.cpp_amd.parts.base import register_part
from easy_gpt.cpp_amd.parts.spec import PartSpec

H, FF, EXPERTS = 32, 16, 4


class InPlace(EmulatedKernels):
    writes_sums_in_place = True

    def expert_mixture(self, *args, out=None, **options):
        sums = super().expert_mixture(*args, **options)
        if out is None:
            return sums
        return out.copy_(sums)


class Doubled(SwiGLU):
    def forward(self, x, ctx=None):
        return 2.0 * super().forward(x, ctx)


register_part("feed_forward", "doubled_for_a_test", Doubled)


@pytest.mark.parametrize("kind", ["swiglu", "doubled_for_a_test"])
@pytest.mark.parametrize("tokens", [3, 64, 65, 200])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_sums_written_in_place_are_the_copied_ones(kind, tokens, dtype):
    shared = PartSpec(kind, {"intermediate_size": 24, "unrounded": True}, prefix="s.")
    part = ExpertMixture("m.", H, EXPERTS, 2, FF, shared=shared, router_bias=False)
    g = torch.Generator().manual_seed(1)
    tensors = {s.name: torch.randn(tuple(s.shape), generator=g) * 0.3 for s in part.param_specs()}
    x = torch.randn(tokens, H, generator=g).to(dtype)
    sums = []
    try:
        for backend in (EmulatedKernels(), InPlace()):
            kernels.use_backend(backend)
            part.load(lambda name: tensors[name], dtype, torch.device("cpu"))
            out = part.forward(x)
            assert out.dtype == torch.float32 and out.shape[1:] == (tokens, H)
            sums.append(out)
    finally:
        kernels.use_backend(None)
    assert sums[0].shape == sums[1].shape and torch.equal(sums[0], sums[1])
