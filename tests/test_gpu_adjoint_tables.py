"""The adjoint x pass's weight from LDS tables, at the size where they just fit
(FP64, 1024^3: two column buffers and the twiddles leave room for the window
factors and exactly 1024 bins), and from global memory past it.

From the state that power() leaves, one pass transforms, weights and
transforms back in LDS; from a kept spectrum the weight is a pass of its own
and its tables are read from global memory.  Both hold the same modes up to the
rounding of FP64 transforms (1e-13 of the largest coefficient each way), so
dL/drho agrees within 1e-12 of its largest value."""
import pytest

import genpk_amd


@pytest.mark.gpu
@pytest.mark.parametrize("d,nrbins", [(1024, 1023), (1024, 1024), (1024, 1025), (256, 1), (256, 2), (256, 3000)])
def test_weight_tables(gpu, d, nrbins):
    import torch
    print("CASE", d, nrbins, flush=True)
    n, box = 200000, 100.0
    g = torch.Generator(device="cuda").manual_seed(nrbins)
    pos = torch.rand((n, 3), device="cuda", generator=g) * box
    lam = torch.randn(nrbins, dtype=torch.float64, device="cuda", generator=g)
    p = genpk_amd.Plan(d, "f64")
    p.deposit(pos, box)
    p.power(nrbins, mass=float(n))
    fused = p.adjoint_density(lam, float(n), nrbins)[:, :, :d].clone()
    p.clear()
    p.deposit(pos, box)
    p.r2c()
    p.bin(nrbins, mass=float(n))
    ref = p.adjoint_density(lam, float(n), nrbins)[:, :, :d]
    assert float((fused - ref).abs().max()) <= 1e-12 * float(ref.abs().max())
