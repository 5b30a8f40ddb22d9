"""Blocks whose output lies over their own seed or key (device entry points and batches): short blocks read both
to the end before they write, as long ones do."""
import numpy as np
import pytest

import privacyamplification_amd as P

pytestmark = pytest.mark.gpu
BOTH = P.XOR_KEY_REST | P.COMPRESS


def say(*a):
    print("[case]", *a, flush=True)


# sizes of the direct product with one and with many workgroups, and one of the transform beyond; m <= h, so that
# the key-rest words lie behind the output
@pytest.mark.parametrize("n,m", [(64, 32), (4096, 1536), (16384, 6144), (16384 + 32, 8192), (65536, 24576), (131072, 49152),
                                 (200000, 50016), (262144, 32768), (1 << 20, 393216)])
def test_output_over_an_input(engine, oracle, n, m):
    import torch
    up = lambda a: torch.from_numpy(a.view(np.int32).copy()).cuda()
    key, seed = oracle.synth_bits(0x1A + n, n + 1), oracle.synth_bits(0x1B + m, n)
    ref = {f: oracle.amp_out(key if f == BOTH else key[: (n - m) // 32 + 1].copy(), seed, n, m, f == BOTH, True,
                             method=oracle.DIRECT) for f in (BOTH, P.COMPRESS)}
    sid = engine.seed_put(seed, n, m)
    try:
        for flags in (BOTH, P.COMPRESS):
            for over in ("seed", "key"):
                for how in ("single", "resident", "batch"):
                    if how == "resident" and over == "seed":
                        continue
                    say(f"n={n} m={m} flags={flags} output over the {over}, {how}")
                    k, s = up(key), up(seed)
                    out = s if over == "seed" else k
                    torch.cuda.synchronize()
                    if how == "single":
                        engine.block_device(k.data_ptr(), s.data_ptr(), n, m, flags, out.data_ptr(), 0)
                    elif how == "resident":
                        engine.block_device_seeded(k.data_ptr(), sid, n, m, flags, out.data_ptr(), 0)
                    else:  # a second block apart, so that the group has one of each
                        k2, s2 = up(key), up(seed)
                        o2 = torch.zeros(m // 8, dtype=torch.uint8, device="cuda")
                        torch.cuda.synchronize()
                        blk = (P.PaBlock * 2)()
                        for b, (kk, ss, oo) in zip(blk, ((k, s, out), (k2, s2, o2))):
                            b.key, b.seed, b.n, b.m, b.flags, b.out = kk.data_ptr(), ss.data_ptr(), n, m, flags, oo.data_ptr()
                        engine.batch_device(blk, 0, 0)
                    torch.cuda.synchronize()
                    got = out.cpu().numpy().view(np.uint8)[: m // 8]
                    assert np.array_equal(got, ref[flags]), (n, m, flags, over, how)
                    if how == "batch":
                        assert np.array_equal(o2.cpu().numpy(), ref[flags])
    finally:
        engine.seed_drop(sid)
