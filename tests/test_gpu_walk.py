"""Pass A's walk over column groups at the shortest transforms (2^15 and 2^16 bits), which only large batches take:
on both sides of the line, every block with a key and a seed of its own."""
import numpy as np
import pytest

import privacyamplification_amd as P

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lg,count", [(15, 512), (15, 511), (16, 512), (16, 511)])
def test_walk_of_short_transforms(engine, oracle, lg, count):
    import torch
    n, rng = 1 << lg, np.random.default_rng(lg)
    print(f"[case] {count} blocks of 2^{lg} bits", flush=True)
    keys = rng.integers(0, 1 << 32, (count, n // 32 + 1), dtype=np.uint32)
    seeds = rng.integers(0, 1 << 32, (count, n // 32), dtype=np.uint32)
    ms = [int(m) * 32 for m in rng.integers(1, n // 32, count)]
    dk, ds = torch.from_numpy(keys.view(np.int32)).cuda(), torch.from_numpy(seeds.view(np.int32)).cuda()
    out = torch.full((count, n // 8), 0x5A, dtype=torch.uint8, device="cuda")
    blk = (P.PaBlock * count)()
    for i, b in enumerate(blk):
        b.key, b.seed, b.n, b.m, b.flags, b.out = dk[i].data_ptr(), ds[i].data_ptr(), n, ms[i], 3, out[i].data_ptr()
    torch.cuda.synchronize()
    engine.batch_device(blk, 0, 0)
    torch.cuda.synchronize()
    got = out.cpu().numpy()
    for i, m in enumerate(ms):
        ref = oracle.amp_out(keys[i], seeds[i], n, m, True, True, method=oracle.NTT)
        assert np.array_equal(got[i, : m // 8], ref), (lg, count, i, m)
        assert np.all(got[i, m // 8:] == 0x5A), (lg, count, i, m)


@pytest.mark.parametrize("lg,count", [(15, 1024), (16, 1024)])
def test_walk_of_short_transforms_resident(engine, oracle, lg, count):
    import torch
    n, m, rng = 1 << lg, 3 << (lg - 3), np.random.default_rng(lg)
    print(f"[case] {count} blocks of 2^{lg} bits on a resident seed", flush=True)
    keys = rng.integers(0, 1 << 32, (count, n // 32 + 1), dtype=np.uint32)
    seed = rng.integers(0, 1 << 32, n // 32, dtype=np.uint32)
    dk = torch.from_numpy(keys.view(np.int32)).cuda()
    out = torch.zeros((count, m // 8), dtype=torch.uint8, device="cuda")
    sid = engine.seed_put(seed, n, m)
    try:
        blk = (P.PaBlock * count)()
        for i, b in enumerate(blk):
            b.key, b.seed_id, b.n, b.m, b.flags, b.out = dk[i].data_ptr(), sid, n, m, 3, out[i].data_ptr()
        torch.cuda.synchronize()
        engine.batch_device(blk, 0, 0)
        torch.cuda.synchronize()
        got = out.cpu().numpy()
        for i in range(count):
            ref = oracle.amp_out(keys[i], seed, n, m, True, True, method=oracle.NTT)
            assert np.array_equal(got[i], ref), (lg, count, i)
    finally:
        engine.seed_drop(sid)
