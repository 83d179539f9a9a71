"""Deposits over many tiles: above 8192 buckets the directory is cut into
sections of 4096 buckets, a workgroup each.  As in the partition's tests, one
mass makes per-cell sums exact integers in fixed point, so the FP64 densities
under two tile shapes are equal bit for bit (with masses in [0.5, 1) below
2^7), and gradients of one dL/drho depend on no order."""
import pytest

import genpk_amd

BOX = 100.0


def _positions(torch, n, kind):
    g = torch.Generator(device="cuda").manual_seed(n)
    pos = torch.rand((n, 3), device="cuda", generator=g) * BOX
    if kind == "slab":      # in 1/16 of the tiles, each with more records than an item holds
        pos[:, 0] *= 1 / 16
    elif kind == "clump":   # half the records in a few tiles
        pos[: n // 2] = torch.randn((n // 2, 3), device="cuda", generator=g) * 0.5 + 50.0
    return pos.contiguous()


# 8192 buckets are one section still, 16384 four, 2^18 sixty-four; 17^3 and
# 33^3 tiles leave buckets without a tile
@pytest.mark.gpu
@pytest.mark.parametrize("d,tiles,n,kind", [(128, (8, 8, 2), 3000, "spread"), (128, (8, 4, 2), 200000, "clump"),
                                            (128, (4, 4, 4), 1000000, "clump"), (132, (4, 4, 4), 100000, "spread"),
                                            (68, (4, 4, 2), 100000, "clump"), (256, (4, 4, 4), 1 << 20, "spread"),
                                            (128, (4, 4, 4), 40000000, "slab")])
@pytest.mark.parametrize("masses", [False, True])
def test_many_tiles(gpu, d, tiles, n, kind, masses):
    import torch
    print("CASE", d, tiles, n, kind, masses, flush=True)
    pos = _positions(torch, n, kind)
    m = None
    if masses:
        m = torch.rand(n, device="cuda", generator=torch.Generator(device="cuda").manual_seed(3)) * 0.5 + 0.5
    a, b = genpk_amd.Plan(d, "f64").set_options(tiles), genpk_amd.Plan(d, "f64")
    got = []
    for p in (a, b):
        p.clear()
        p.deposit(pos, BOX, m, retain=True)
        got.append(p.export_density().clone())
    if masses:
        few = got[0] < 2.0 ** 7
        assert torch.equal(got[0][few], got[1][few])
        # fuller cells: each of the few sums that form a cell is rounded to FP64 once
        assert bool(((got[0] - got[1]).abs() <= 2.0 ** -48 * got[1].abs()).all())
    else:
        assert torch.equal(got[0], got[1])
    a.clear()
    a.redeposit()
    assert torch.equal(a.export_density(), got[0])
    # deposits added to what the tiles hold: only touched tiles have items
    a.deposit(pos[: n // 3].contiguous(), BOX, None if m is None else m[: n // 3].contiguous())
    b.deposit(pos[: n // 3].contiguous(), BOX, None if m is None else m[: n // 3].contiguous())
    x, y = a.export_density(), b.export_density()
    assert bool(((x - y).abs() <= 2.0 ** -48 * y.abs()).all())
    G = torch.randn(got[0].shape, dtype=torch.float64, device="cuda",
                    generator=torch.Generator(device="cuda").manual_seed(5))
    grads = []
    for p in (a, b):
        p.import_density(G)
        grads.append(p.adjoint_gather(pos, BOX, m))
    assert torch.equal(grads[0][0], grads[1][0]) and torch.equal(grads[0][1], grads[1][1])


# few records in many buckets: the second pass's workgroups take fewer records
# than a sub-chunk, down to one (n <= 256 buckets)
@pytest.mark.gpu
@pytest.mark.parametrize("n", [1, 2, 255, 256, 257, 1000, 40000, 300000])
@pytest.mark.parametrize("d,tiles", [(256, (4, 8, 16)), (320, (16, 32, 32)), (512, (16, 32, 32))])
def test_few_records_in_many_buckets(gpu, d, tiles, n):
    import torch
    print("CASE", d, tiles, n, flush=True)
    pos = _positions(torch, n, "spread")
    a, b = genpk_amd.Plan(d, "f64").set_options(tiles), genpk_amd.Plan(d, "f64").set_options((32, 16, 16))
    got = []
    for p in (a, b):
        p.clear()
        p.deposit(pos, BOX, retain=True)
        got.append(p.export_density().clone())
    assert torch.equal(got[0], got[1])
    grads = []
    for p in (a, b):
        p.import_density(got[0])
        grads.append(p.adjoint_gather(pos, BOX))
    assert torch.equal(grads[0][0], grads[1][0]) and torch.equal(grads[0][1], grads[1][1])
