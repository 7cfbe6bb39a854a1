"""Brick pool manager on the GPU (yx_brick_pool_*; CuBrickPoolManager::allocMap,
reaction/voxtree/brickpool/BrickPool.cpp:21-62, and UpdateBrickPool,
reaction/voxtree/density.cu:240-284) against the numpy restatement of its
policy, and compositing over a pool-managed volume against the same volume
packed on the host."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_random_operations_match_policy(yx, oracle_mod, cuda):
    torch = cuda
    rng = np.random.default_rng(21)
    g, brick, cap = 16, 4, 1500
    nb, vox = g ** 3, brick ** 3
    dev = torch.device("cuda", 0)
    table = torch.full((nb,), -1, dtype=torch.int32, device=dev)
    params = torch.zeros((cap * vox, 4), dtype=torch.float32, device=dev)
    pool = yx.composite.BrickPool(table, params, g * brick, brick)
    orc = oracle_mod.BrickPoolOracle(np.full(nb, -1, np.int32), np.zeros((cap * vox, 4), np.float32), brick)
    for step in range(60):
        op = rng.choice(["alloc", "alloc", "release", "update"])
        k = int(rng.integers(1, 400))
        bricks = rng.integers(0, nb, size=k).astype(np.int32)
        bt = torch.from_numpy(bricks).to(dev)
        if op == "alloc":
            try:
                exp_slots, exp_new = orc.alloc(bricks)
                ok = True
            except ValueError:
                ok = False
            if ok:
                slots, new = pool.alloc(bt)
                torch.cuda.synchronize()
                assert new == exp_new, step
                assert np.array_equal(slots.cpu().numpy(), exp_slots), step
            else:
                with pytest.raises(yx.YoxelError):
                    pool.alloc(bt)
        elif op == "release":
            assert pool.release(bt) == orc.release(bricks), step
        else:
            packed = rng.standard_normal((k * vox, 4)).astype(np.float32)
            pool.update(bt, torch.from_numpy(packed).to(dev))
            orc.update(bricks, packed)
        torch.cuda.synchronize()
        assert np.array_equal(table.cpu().numpy(), orc.table), (step, op)
        assert pool.stats() == (int(orc.used.sum()), cap), (step, op)
    assert np.array_equal(params.cpu().numpy(), orc.params)
    # an index outside the table fails and changes nothing
    before = table.clone()
    with pytest.raises(yx.YoxelError):
        pool.alloc(torch.tensor([3, nb], dtype=torch.int32, device=dev))
    assert torch.equal(before, table)


@pytest.mark.parametrize("cap,k", [(1, 1), (63, 64), (64, 64), (65, 63), (257, 255), (320, 257)])
def test_list_and_slot_counts_around_a_mask(yx, oracle_mod, cuda, cap, k):
    """Lists and slot maps that end within, at and after a 64-bit mask; every
    brick listed twice; calls that fail leave nothing behind for the next."""
    torch = cuda
    g, brick = 8, 2
    nb, vox = g ** 3, brick ** 3
    dev = torch.device("cuda", 0)
    table = torch.full((nb,), -1, dtype=torch.int32, device=dev)
    params = torch.zeros((cap * vox, 4), dtype=torch.float32, device=dev)
    pool = yx.composite.BrickPool(table, params, g * brick, brick)
    orc = oracle_mod.BrickPoolOracle(np.full(nb, -1, np.int32), np.zeros((cap * vox, 4), np.float32), brick)
    rng = np.random.default_rng(cap)

    def same():
        torch.cuda.synchronize()
        assert np.array_equal(table.cpu().numpy(), orc.table)
        assert np.array_equal(params.cpu().numpy(), orc.params)
        assert pool.stats() == (int(orc.used.sum()), cap)

    for step in range(4):
        fit = min(k, int((~orc.used).sum()) + int((orc.table >= 0).sum()))
        half = rng.permutation(nb)[:fit].astype(np.int32)
        bricks = np.concatenate([half, half[::-1]])
        bt = torch.from_numpy(bricks).to(dev)
        values = rng.standard_normal((bricks.size * vox, 4)).astype(np.float32)
        vt = torch.from_numpy(values).to(dev)
        for bad in (-1, nb):
            broken = bt.clone()
            broken[0] = bad
            with pytest.raises(yx.YoxelError):
                pool.alloc(broken)
            with pytest.raises(yx.YoxelError):
                pool.update(broken, vt)
        same()
        try:
            slots, new = orc.alloc(bricks)
        except ValueError:
            with pytest.raises(yx.YoxelError):
                pool.alloc(bt)
        else:
            got, got_new = pool.alloc(bt)
            assert got_new == new and np.array_equal(got.cpu().numpy(), slots)
        orc.update(bricks, values)
        pool.update(bt, vt)
        same()
        gone = bricks[: max(1, fit // 2)]
        assert pool.release(torch.from_numpy(gone).to(dev)) == orc.release(gone)
        same()


@pytest.mark.parametrize("cap", [126976, 126977, 209715, 2097152, 2097217])
def test_pools_of_many_slots(yx, oracle_mod, cuda, cap):
    """Slot counts around those where the sum of the used slots (31 chunks of
    4096 items) and the scans of the slots' and the list's masks (32,768 masks
    of 64) need more space or another path; half of the slots used before."""
    torch = cuda
    grid = 64 if cap < 64 ** 3 else 136
    nb = grid ** 3
    dev = torch.device("cuda", 0)
    rng = np.random.default_rng(cap)
    order = rng.permutation(nb).astype(np.int32)
    start = np.full(nb, -1, np.int32)
    start[order[:cap // 2]] = rng.permutation(cap)[:cap // 2]
    table = torch.from_numpy(start).to(dev)
    params = torch.zeros((cap, 4), dtype=torch.float32, device=dev)
    pool = yx.composite.BrickPool(table, params, grid, 1)
    orc = oracle_mod.BrickPoolOracle(start, np.zeros((cap, 4), np.float32), 1)
    assert pool.stats() == (cap // 2, cap)
    gone = order[:cap // 4]
    assert pool.release(torch.from_numpy(gone).to(dev)) == orc.release(gone) == cap // 4
    fresh = order[cap // 8:cap // 8 + cap]  # some have a slot, the others take every free one
    slots, new = pool.alloc(torch.from_numpy(fresh).to(dev))
    exp_slots, exp_new = orc.alloc(fresh)
    assert new == exp_new and np.array_equal(slots.cpu().numpy(), exp_slots)
    assert np.array_equal(table.cpu().numpy(), orc.table)
    assert pool.stats() == (int(orc.used.sum()), cap)
    values = rng.standard_normal((fresh.size, 4)).astype(np.float32)
    pool.update(torch.from_numpy(fresh).to(dev), torch.from_numpy(values).to(dev))
    orc.params[exp_slots] = values  # every listed brick has a slot of its own
    assert np.array_equal(params.cpu().numpy(), orc.params)


def test_update_returns_before_its_copy(yx, cuda):
    """update waits for its check alone; the bricks' copy (256 MB here) runs on
    behind the host. A busy host may find it done by the time it looks, so one
    of several calls is enough."""
    torch = cuda
    dev = torch.device("cuda", 0)
    grid, brick = 256, 8
    nb = (grid // brick) ** 3
    bricks = torch.arange(nb, dtype=torch.int32, device=dev)
    table = torch.full((nb,), -1, dtype=torch.int32, device=dev)
    params = torch.zeros((nb * brick ** 3, 4), dtype=torch.float32, device=dev)
    values = torch.ones_like(params)
    pool = yx.composite.BrickPool(table, params, grid, brick)
    pool.alloc(bricks)
    behind = []
    for _ in range(10):
        torch.cuda.synchronize()
        pool.update(bricks, values)
        behind.append(not torch.cuda.current_stream().query())
    assert any(behind)
    assert torch.equal(params, values)


def test_existing_table_and_bad_table(yx, cuda):
    torch = cuda
    vol = yx.composite.Volume(64, 8, occupancy=0.2, seed=3)
    table, params = vol.to(torch.device("cuda", 0))
    pool = yx.composite.BrickPool(table, params, 64, 8)
    assert pool.stats() == (vol.num_slots, vol.num_slots)
    bad = table.clone()
    live = torch.nonzero(bad >= 0).flatten()
    bad[live[1]] = bad[live[0]]  # one slot for two bricks
    with pytest.raises(yx.YoxelError):
        yx.composite.BrickPool(bad, params, 64, 8)


def test_compositing_over_pool_equals_packed_volume(yx, cuda):
    torch = cuda
    dev = torch.device("cuda", 0)
    grid, brick = 128, 8
    vol = yx.composite.Volume(grid, brick, occupancy=0.1, seed=5)
    table_ref, params_ref = vol.to(dev)
    vox = brick ** 3
    live = np.nonzero(vol.table >= 0)[0].astype(np.int32)
    rng = np.random.default_rng(4)
    order = rng.permutation(live)
    # the same bricks allocated in another order in a pool with spare slots
    cap = vol.num_slots + 37
    table = torch.full_like(table_ref, -1)
    params = torch.zeros((cap * vox, 4), dtype=torch.float32, device=dev)
    pool = yx.composite.BrickPool(table, params, grid, brick)
    bt = torch.from_numpy(order).to(dev)
    slots, new = pool.alloc(bt)
    assert new == live.size
    src = vol.params.reshape(-1, vox, 4)[vol.table[order]]
    pool.update(bt, torch.from_numpy(np.ascontiguousarray(src.reshape(-1, 4))).to(dev))
    comp = yx.composite.Compositor()
    views = torch.from_numpy(yx.composite.orbit_views(3, 60.0, 96, 80)).to(dev)
    a = comp.forward(table_ref, params_ref, grid, brick, views, 96, 80)
    b = comp.forward(table, params, grid, brick, views, 96, 80)
    torch.cuda.synchronize()
    for x, y in zip(a, b):
        assert torch.equal(x, y)
    # free a tenth of the bricks in both; the renders still agree
    drop = order[: live.size // 10]
    pool.release(torch.from_numpy(drop).to(dev))
    t2 = table_ref.clone()
    t2[torch.from_numpy(drop.astype(np.int64)).to(dev)] = -1
    a = comp.forward(t2, params_ref, grid, brick, views, 96, 80)
    b = comp.forward(table, params, grid, brick, views, 96, 80)
    torch.cuda.synchronize()
    for x, y in zip(a, b):
        assert torch.equal(x, y)
    assert pool.stats()[0] == live.size - drop.size
