"""Device memory that a plan's first forward takes.  The record pools hold at
most a sixth (or 2^26 slots) more than the records, and nothing else grows with
the particles by more than a few bytes each: the bound below is the sum of

* the grid and the tile store (17 * 33 * 33 values per tile),
* two pools of n + max(n / 6, 2^26) slots of 12 (with masses 16) bytes, the
  first pass's being n slots where it counts,
* partial tiles of split tiles: 8 * 17 * 33 * 33 bytes for every item of split
  tiles, at most two per 2^17 slots of the last pool (no split is finer here),
* the block lists, 6 bytes for each block of 64 slots or more, so less than a
  quarter of a byte per record, and 64 MB for tables and the allocator's rounding.

The largest case takes about 50 GB."""
import pytest

import genpk_amd

BOX = 100.0


@pytest.mark.gpu
@pytest.mark.parametrize("d,n,masses", [(512, 1 << 27, False), (512, 1 << 27, True), (360, 1 << 27, False),
                                        (1024, 1 << 29, False), (1024, 1 << 30, False)])
def test_first_forward_memory(gpu, d, n, masses):
    import torch
    print("CASE", d, n, masses, flush=True)
    pos = torch.rand((n, 3), device="cuda") * BOX
    m = torch.rand(n, device="cuda") if masses else None
    p = genpk_amd.Plan(d, "f32")
    torch.cuda.synchronize()
    before = torch.cuda.mem_get_info()[0]
    p.clear()
    p.deposit(pos, BOX, m)
    p.power()
    torch.cuda.synchronize()
    taken = before - torch.cuda.mem_get_info()[0]
    tiles = -(-d // 16) * (-(-d // 32)) ** 2
    cells = 17 * 33 * 33
    pool = n + max(n // 6, 1 << 26)
    bound = tiles * cells * 4 + 2 * pool * (16 if masses else 12) + 2 * (pool // (1 << 17) + 1) * cells * 8 + n // 4 + (64 << 20)
    print(f"taken {taken / 1e9:.3f} GB, bound {bound / 1e9:.3f} GB", flush=True)
    assert taken <= bound


@pytest.mark.gpu
def test_partial_tiles_share_the_first_pool(gpu):
    """Where the partition takes two passes the partial tiles of split tiles lie
    in the first pass's pool, which the second pass has read: the bound above
    without them.  A second deposit of clumped particles (split tiles) and one
    from the kept order are equal to the first."""
    import torch
    d, n = 1024, 1 << 30
    print("CASE", d, n, flush=True)
    pos = torch.rand((n, 3), device="cuda") * BOX
    p = genpk_amd.Plan(d, "f32")
    torch.cuda.synchronize()
    before = torch.cuda.mem_get_info()[0]
    p.deposit(pos, BOX)
    torch.cuda.synchronize()
    taken = before - torch.cuda.mem_get_info()[0]
    bound = 65536 * 17 * 33 * 33 * 4 + 2 * (n + n // 6) * 12 + n // 4 + (64 << 20)
    print(f"taken {taken / 1e9:.3f} GB, bound {bound / 1e9:.3f} GB", flush=True)
    assert taken <= bound
    del p, pos
    d, n = 512, 20000000
    pos = (torch.randn((n, 3), device="cuda") * 3.0 + 50.0).contiguous()
    p = genpk_amd.Plan(d, "f64")
    got = []
    for again in (False, False, True):
        p.clear()
        p.redeposit() if again else p.deposit(pos, BOX, retain=True)
        got.append(p.export_density().clone())
    assert torch.equal(got[0], got[1]) and torch.equal(got[0], got[2])
    assert abs(float(got[0].sum()) - n) <= 1e-6 * n
