"""The product of many rows that makes queries, keys and values with bias, rotation and the store into the cache at its end
(gemm_rows.hip), against float64."""
import pytest
import torch

from easy_gpt.cpp_amd import kernels

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _case(m, kk, nq, nkv, hd, ps, biased, seed=0):
    g = torch.Generator().manual_seed(seed)
    width = (nq + 2 * nkv) * hd
    x = torch.randn(m, kk, generator=g).to(torch.bfloat16)
    w = (torch.randn(width, kk, generator=g) * kk ** -0.5).to(torch.bfloat16)
    b = torch.randn(width, generator=g).to(torch.bfloat16) if biased else None
    positions = torch.randint(0, 9000, (m,), generator=g, dtype=torch.int32)
    inv = (1.0 / 1e4 ** (torch.arange(hd // 2, dtype=torch.float32) / (hd // 2)))
    pages = -(-m // ps) + 2
    slots = torch.randperm(pages * ps, generator=g)[:m].to(torch.int32)
    slots[m // 2] = -1                                     # a token that is stored nowhere
    # in 64 bits; the angles are float32 products, as the model defines them
    y = x.double() @ w.double().t() + (b.double() if biased else 0.0)
    y = y.view(m, nq + 2 * nkv, hd)
    angle = (positions.float()[:, None] * inv[None]).double()[:, None]
    lo, hi = y[:, : nq + nkv, : hd // 2].clone(), y[:, : nq + nkv, hd // 2 :].clone()
    y[:, : nq + nkv, : hd // 2] = lo * angle.cos() - hi * angle.sin()
    y[:, : nq + nkv, hd // 2 :] = lo * angle.sin() + hi * angle.cos()
    return x, w, b, positions, inv, slots, pages, y


def _check(got, want):
    """Rounded once to bfloat16 (eight significant bits: half a unit is 2^-8 of the value at most), behind float32 sums and cosines (1e-5
    of sums of size one)."""
    assert torch.all((got.double().cpu() - want).abs() <= 2.0 ** -8 * 1.01 * want.abs() + 4e-5), float((got.double().cpu() - want).abs().max())


@pytest.mark.parametrize("m,kk,nq,nkv,hd,ps,biased", [
    (65, 64, 2, 1, 64, 16, True), (129, 128, 3, 1, 32, 16, False), (200, 896, 14, 2, 64, 16, True), (257, 192, 6, 2, 128, 32, True),
    (333, 320, 1, 1, 256, 64, True), (64, 448, 5, 5, 64, 48, False), (511, 256, 12, 2, 128, 16, True), (1, 64, 2, 2, 64, 16, True)])
@pytest.mark.parametrize("shape", range(7))
def test_product_with_rotation_and_store(m, kk, nq, nkv, hd, ps, biased, shape):
    k = kernels.backend()
    x, w, b, positions, inv, slots, pages, want = _case(m, kk, nq, nkv, hd, ps, biased)
    width = (nq + 2 * nkv) * hd
    out = torch.full((m, width), 7.0, dtype=torch.bfloat16, device=DEV)
    kc = torch.full((pages, nkv, ps, hd), 7.0, dtype=torch.bfloat16, device=DEV)
    vc = torch.full((pages, nkv, hd, ps), 7.0, dtype=torch.bfloat16, device=DEV)
    xd, wd, bd, sd = x.to(DEV), w.to(DEV), None if b is None else b.to(DEV), slots.to(DEV)
    cs = k.rope_table(positions.to(DEV), inv.to(DEV))
    k._run("egpt_gemm_rows_rotated", xd.data_ptr(), wd.data_ptr(), k._ptr(bd), cs.data_ptr(), sd.data_ptr(), out.data_ptr(), kc.data_ptr(),
           vc.data_ptr(), m, kk, nq, nkv, hd, ps, shape, k._stream())
    torch.cuda.synchronize()
    _check(out.view(m, -1, hd)[:, :nq], want[:, :nq])
    assert torch.all(out.view(m, -1, hd)[:, nq:] == 7.0)
    stored = slots >= 0
    page, off = (slots[stored] // ps).long(), (slots[stored] % ps).long()
    _check(kc.cpu()[page, :, off], want[stored, nq : nq + nkv])
    _check(vc.cpu()[page, :, :, off], want[stored, nq + nkv :])
    # nothing else was written
    free = torch.ones(pages, ps, dtype=torch.bool)
    free[page, off] = False
    assert torch.all(kc.cpu().transpose(1, 2)[free] == 7.0) and torch.all(vc.cpu().permute(0, 3, 1, 2)[free] == 7.0)


def test_rotated_products_that_are_refused():
    k = kernels.backend()
    p = torch.zeros(1 << 20, device=DEV, dtype=torch.uint8).data_ptr()
    for args in ((70, 60, 2, 1, 64, 16, 4), (70, 64, 2, 1, 48, 16, 4), (70, 64, 2, 1, 512, 16, 4)):
        with pytest.raises(Exception):
            k._run("egpt_gemm_rows_rotated", p, p, None, p, p, p, p, p, *args, k._stream())
    with pytest.raises(Exception):
        k._run("egpt_gemm_rows_rotated", p + 2, p, None, p, p, p, p, p, 70, 64, 2, 1, 64, 16, 4, k._stream())


@pytest.mark.parametrize("m", [65, 200, 700])
def test_wrapper_agrees_with_the_two_kernels(m):
    # product, then bias, rotation and store: the same sums but for the order of a split k range
    k = kernels.backend()
    nq, nkv, hd, ps, kk = 14, 2, 64, 16, 896
    x, w, b, positions, inv, slots, pages, want = _case(m, kk, nq, nkv, hd, ps, True, seed=m)
    new = [torch.zeros((pages, nkv, ps, hd), dtype=torch.bfloat16, device=DEV), torch.zeros((pages, nkv, hd, ps), dtype=torch.bfloat16, device=DEV)]
    xd, wd, bd, sd, pd, fd = x.to(DEV), w.to(DEV), b.to(DEV), slots.to(DEV), positions.to(DEV), inv.to(DEV)
    cs = k.rope_table(pd, fd)
    out = k.product_rotated(xd, wd, bd, cs, sd, *new, nq, nkv, hd, ps)
    assert out is not None
    old = [torch.zeros_like(c) for c in new]
    both = torch.empty_like(out)
    k.qkv_rope_store(k.product_parts(xd, wd), bd, pd, fd, hd, sd, *old, nq, nkv, hd, ps, out=both, cos_sin=cs)
    torch.cuda.synchronize()
    stored = slots >= 0
    page, off = (slots[stored] // ps).long(), (slots[stored] % ps).long()
    for q, kc, vc in ((out, *new), (both, *old)):
        _check(q.view(m, -1, hd)[:, :nq], want[:, :nq])
        _check(kc.cpu()[page, :, off], want[stored, nq : nq + nkv])
        _check(vc.cpu()[page, :, :, off], want[stored, nq + nkv :])
    # float32 sums in another order are off by 1e-5 (values of size one), which takes one in a hundred to the other side of a rounding
    for a, b in ((out.view(m, -1, hd)[:, :nq], both.view(m, -1, hd)[:, :nq]), *zip(new, old)):
        assert float((a != b).float().mean()) <= 0.01 and torch.all((a.double() - b.double()).abs() <= 2.0 ** -7 * 1.01 * b.double().abs() + 4e-5)
    # operands that it does not take
    assert k.product_rotated(xd[:64], wd, bd, cs[:64].contiguous(), sd[:64], *new, nq, nkv, hd, ps) is None
    assert k.product_rotated(xd.float(), wd.float(), bd.float(), cs, sd, *new, nq, nkv, hd, ps) is None
