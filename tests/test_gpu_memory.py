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
