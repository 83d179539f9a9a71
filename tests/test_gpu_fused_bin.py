"""The fused last FFT pass + binning against the general path (the in-place
transform, then the binning of the stored spectrum, which reads each mode's
bin from a table over |k|^2) over the forms the fused pass takes: a first
radix that is or is not run from registers (radix 4 in FP64, 8 in FP32), odd
and even numbers of stages, columns that leave threads idle, one field and
two, and from eight copies of the LDS bins to one.

Tolerance: in FP64 both paths hold the same modes and differ in the order in
which a bin's c / 2 or more terms of one sign are added, so by at most c 2^-52
of the sum.  In FP32 a length divisible by 16 may run another radix ordering;
each mode then differs by at most 3e-6 of the field's rms mode (the bound of
the FFT's own test), a bin's power by twice that; the other lengths hold the
same modes.  A cross bin's terms have both signs and are bounded by the
geometric mean of the two auto bins."""
import pytest

import genpk_amd


@pytest.mark.gpu
@pytest.mark.parametrize("prec,d", [("f64", d) for d in (8, 20, 24, 64, 72, 100, 128, 200, 256, 360, 480)] +
                         [("f32", d) for d in (8, 20, 24, 40, 72, 120, 128, 200, 320, 360, 512)])
@pytest.mark.parametrize("nrbins", [None, 1000, 4000])
def test_fused_binning_equals_stored_binning(gpu, prec, d, nrbins):
    import torch
    print("CASE", prec, d, nrbins, flush=True)
    g = torch.Generator(device="cuda").manual_seed(d)
    a, b = (genpk_amd.Plan(d, prec) for _ in range(2))
    grids = [torch.randn(p.grid.shape, device="cuda", dtype=p.real_dtype, generator=g) for p in (a, b)]

    def fill():
        for p, x in zip((a, b), grids):
            p.import_density(x)

    fill()
    fp, fcount, fkeffs = a.power(nrbins)
    fill()
    fcross = a.power(nrbins, other=b)[0]
    fill()
    a.r2c(), b.r2c()
    sp, scount, skeffs = a.bin(nrbins)
    saa, sbb, sab = a.bin(nrbins, other=b)[0]
    assert torch.equal(fcount, scount) and torch.equal(fkeffs, skeffs)
    rel = scount.double() * 2.0 ** -52 + (6e-6 if prec == "f32" and d % 16 == 0 else 0.0)
    for got, ref, size in ((fp, sp, sp), (fcross[0], saa, saa), (fcross[1], sbb, sbb), (fcross[2], sab, (saa * sbb).sqrt())):
        assert bool(((got - ref).abs() <= rel * size).all())


@pytest.mark.gpu
@pytest.mark.parametrize("prec,d", [("f64", 36), ("f32", 90)])
def test_stored_binning_without_lds_tables(gpu, prec, d):
    """Two fields with 6700 bins leave no LDS for the window factors and the
    thresholds; one field's bins do.  The bound is the first test's."""
    import torch
    print("CASE", prec, d, flush=True)
    nrbins = 6700
    g = torch.Generator(device="cuda").manual_seed(d)
    a, b = (genpk_amd.Plan(d, prec) for _ in range(2))
    for p in (a, b):
        p.import_density(torch.randn(p.grid.shape, device="cuda", dtype=p.real_dtype, generator=g))
        p.r2c()
    (paa, pbb, _), count, _ = a.bin(nrbins, other=b)
    for p, got in ((a, paa), (b, pbb)):
        ref, c1, _ = p.bin(nrbins)
        assert torch.equal(count, c1)
        assert bool(((got - ref).abs() <= count.double() * 2.0 ** -52 * ref).all())
