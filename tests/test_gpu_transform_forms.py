"""The transform passes' forms by length: the column passes' first stage from
registers or element by element (FP32 x pass over blocks of less than a line,
from d = 514 on), and the z pass's first stage from the tile store for every
radix that a half length can begin with.

Transforms are compared with torch's FP64 FFT within the bars of the other
transform tests (1e-13 of the largest coefficient in FP64, 3e-6 in FP32).  The
forward from the tile store is compared with the same density exported (each
cell rounded once, as the z pass rounds it) and imported again, which takes
the element-wise z pass: in FP64 every spectrum value within 1e-13 of the
largest, in FP32 within 3e-6."""
import pytest

import genpk_amd

TOL = {"f64": 1e-13, "f32": 3e-6}


@pytest.mark.gpu
@pytest.mark.parametrize("prec,d", [("f32", d) for d in (500, 540, 576, 648, 750)] + [("f64", d) for d in (486, 540)])
def test_column_passes_by_length(gpu, prec, d):
    import torch
    print("CASE columns", prec, d, flush=True)
    g = torch.Generator(device="cuda").manual_seed(d)
    x = torch.randn((d, d, d), dtype=torch.float64, device="cuda", generator=g)
    p = genpk_amd.Plan(d, prec)
    p.grid.zero_()
    p.grid[:, :, :d] = x
    p.import_density(p.grid.clone())
    ref = torch.fft.rfftn(x)
    got = p.r2c()
    assert float((got - ref).abs().max()) <= TOL[prec] * float(ref.abs().max())
    del ref
    back = p.c2r()[:, :, :d].double() / d ** 3
    assert float((back - x).abs().max()) <= 10 * TOL[prec] * float(x.abs().max())


# the first radix of the half length: 3, 2, 5, 8, 4, 4, 4, 3, 2, 4, 5, 3 (ordering 1
# begins with the leftover radix, ordering 2 with 4)
@pytest.mark.gpu
@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("d,variant", [(18, 0), (20, 0), (50, 0), (64, 0), (64, 1), (64, 2), (72, 0), (90, 0), (100, 0),
                                       (128, 2), (250, 0), (486, 0)])
def test_forward_from_the_tile_store(gpu, prec, d, variant):
    import torch
    print("CASE tile store", prec, d, variant, genpk_amd.radix_plan(d // 2, variant), flush=True)
    g = torch.Generator(device="cuda").manual_seed(d)
    pos = torch.rand((min(20 * d ** 3, 300000), 3), device="cuda", generator=g) * 100.0
    a, b = (genpk_amd.Plan(d, prec).set_options((16, 32, 32), variant) for _ in range(2))
    a.deposit(pos, 100.0)
    b.import_density(a.export_density().clone())
    got, ref = a.r2c(), b.r2c()
    assert float((got - ref).abs().max()) <= TOL[prec] * float(ref.abs().max())
