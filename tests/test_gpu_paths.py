"""The engine's routes by block size (direct product, one-workgroup, mid-size and large transforms) at
the sizes where each can go wrong, bit for bit against the oracle.  A call with a margin always takes the
transform, so the same block is also compared between the direct product and the transform."""
import numpy as np
import pytest

import privacyamplification_amd as P

pytestmark = pytest.mark.gpu

FLAGS = [P.XOR_KEY_REST | P.COMPRESS, P.COMPRESS, P.XOR_KEY_REST, 0]


def say(*a):
    print("[case]", *a, flush=True)


def _ref(oracle, key, seed, n, m, flags):
    xor, comp = bool(flags & P.XOR_KEY_REST), bool(flags & P.COMPRESS)
    k = key if xor else key[: (n - m) // 32 + 1].copy()
    method = oracle.NTT if n & (n - 1) == 0 and n > 1 << 17 else oracle.DIRECT
    return oracle.amp_out(k, seed, n, m, xor, comp, method=method)


class _Device:
    """One block's buffers on the device, the output guarded by 16 bytes."""

    def __init__(self, key, seed, size):
        import torch
        up = lambda a: torch.from_numpy(a.view(np.int32).copy()).cuda()
        self.size = size
        self.key, self.seed = up(np.concatenate([key, np.zeros(1, np.uint32)])), up(seed)
        self.out = torch.full((size + 16,), 0x5A, dtype=torch.uint8, device="cuda")
        self.margin = torch.zeros(1, dtype=torch.float32, device="cuda")

    def take(self):
        import torch
        torch.cuda.synchronize()
        o = self.out.cpu().numpy()
        assert np.all(o[self.size:] == 0x5A)
        self.out.fill_(0x5A)
        torch.cuda.synchronize()
        return o[: self.size]


# edges of the direct product: one word in, out or both; a key that ends on, before and after a chunk of
# 16 words; the one-workgroup sizes' end at 2^14; the work limit (2^18 with 1/8 and 3/8 out, 200000 bits)
DIRECT = [(64, 32), (96, 32), (96, 64), (1024, 32), (1024, 992), (2048 + 32, 1024), (4096, 1536), (5000 // 32 * 32, 4000),
          (5088, 4576 - 32), (16384, 6144), (16384 + 32, 32), (32768 - 32, 32768 - 64), (32768, 24576), (65536, 6144),
          (96000, 24000), (131072, 49152), (131072 - 32, 65536), (200000, 50016), (262144, 32768), (262144, 98304),
          (262144 - 32, 32), (262144, 262144 - 32)]


@pytest.mark.parametrize("n,m", DIRECT)
def test_direct_product_and_transform_agree(engine, oracle, n, m):
    m = m // 32 * 32
    key, seed = oracle.synth_bits(0xD1 + n, n + 1), oracle.synth_bits(0xD2 + m, n)
    sid = engine.seed_put(seed, n, m)
    try:
        for flags in FLAGS:
            if n & (n - 1) and not flags & P.COMPRESS:
                continue
            say(f"direct n={n} m={m} flags={flags}")
            ref = _ref(oracle, key, seed, n, m, flags)
            d = _Device(key, seed, ref.size)
            blk = (P.PaBlock * 3)()
            for margin in (0, d.margin.data_ptr()):
                engine.block_device(d.key.data_ptr(), d.seed.data_ptr(), n, m, flags, d.out.data_ptr(), 0, margin)
                assert np.array_equal(d.take(), ref), (n, m, flags, "fresh", margin)
                engine.block_device_seeded(d.key.data_ptr(), sid, n, m, flags, d.out.data_ptr(), 0, margin)
                assert np.array_equal(d.take(), ref), (n, m, flags, "resident", margin)
            assert 0 < d.margin.item() < 0.25
            # with another length's block and a shorter one of the same transform in the launch
            other = _Device(oracle.synth_bits(5, 2049), oracle.synth_bits(6, 2048), 96)
            for fresh in (True, False):
                for i, (b, bn, bm) in enumerate(((d, n, m), (other, 2048, 768), (None, 0, 0))):
                    if b is None:
                        continue
                    blk[i].key, blk[i].n, blk[i].m, blk[i].out = b.key.data_ptr(), bn, bm, b.out.data_ptr()
                    blk[i].flags = flags if b is d else 3
                    blk[i].seed = b.seed.data_ptr() if fresh or b is other else None
                    blk[i].seed_id = 0 if fresh or b is other else sid
                arr = (P.PaBlock * 2)(blk[0], blk[1])
                engine.batch_device(arr, P.BATCH_GRAPH, 0)
                assert np.array_equal(d.take(), ref), (n, m, flags, "batch", fresh)
                assert np.array_equal(other.take(), _ref(oracle, oracle.synth_bits(5, 2049), oracle.synth_bits(6, 2048),
                                                         2048, 768, 3))
    finally:
        engine.seed_drop(sid)


# transforms of 3 * 2^k: their shortest and longest blocks at every length, the next longer block (a power of
# two's), one word out and one word of key, and as one batch with both kinds of transform in it
MIXED = [(n, m) for e in range(18, 25) for n, m in
         [((1 << e) + 32, 32), (3 << (e - 1), (3 << (e - 1)) - 32), ((3 << (e - 1)) - 32, 3 << (e - 3)), ((3 << (e - 1)) + 32, 1 << (e - 1))]]


@pytest.mark.parametrize("n,m", MIXED)
def test_mixed_radix_blocks(engine, oracle, n, m):
    key, seed = oracle.synth_bits(0xE1 + n, n + 1), oracle.synth_bits(0xE2 + m, n)
    sid = engine.seed_put(seed, n, m)
    small_n, small_m = (1 << 18) + 64, 1 << 17
    sk, ss = oracle.synth_bits(5, small_n + 1), oracle.synth_bits(6, small_n)
    small_ref = oracle.amp_out(sk, ss, small_n, small_m, True, True, method=oracle.NTT)
    try:
        for flags in (P.XOR_KEY_REST | P.COMPRESS, P.COMPRESS):
            say(f"mixed n={n} m={m} flags={flags}")
            k = key if flags & P.XOR_KEY_REST else key[: (n - m) // 32 + 1].copy()
            ref = oracle.amp_out(k, seed, n, m, bool(flags & P.XOR_KEY_REST), True, method=oracle.NTT)
            d = _Device(key, seed, ref.size)
            args = (n, m, flags, d.out.data_ptr(), 0, d.margin.data_ptr())
            engine.block_device(d.key.data_ptr(), d.seed.data_ptr(), *args)
            assert np.array_equal(d.take(), ref), (n, m, flags, "fresh")
            engine.block_device_seeded(d.key.data_ptr(), sid, *args)
            assert np.array_equal(d.take(), ref), (n, m, flags, "resident")
            assert 0 < d.margin.item() < 0.25
            other = _Device(sk, ss, small_ref.size)
            for fresh in (True, False):
                blk = (P.PaBlock * 3)()
                for i, (b, bn, bm) in enumerate(((d, n, m), (other, small_n, small_m))):
                    blk[i].key, blk[i].n, blk[i].m, blk[i].out = b.key.data_ptr(), bn, bm, b.out.data_ptr()
                    blk[i].flags = flags if b is d else 3
                    blk[i].seed = b.seed.data_ptr() if fresh or b is other else None
                    blk[i].seed_id = 0 if fresh or b is other else sid
                engine.batch_device((P.PaBlock * 2)(blk[0], blk[1]), P.BATCH_GRAPH, 0)
                assert np.array_equal(d.take(), ref), (n, m, flags, "batch", fresh)
                assert np.array_equal(other.take(), small_ref)
        if n <= 1 << 22:
            assert np.array_equal(engine.amplify(key, seed, n, m, False, True), ref), (n, m, "host")
    finally:
        engine.seed_drop(sid)


# batches whose row passes take many rows a workgroup (from 1024 workgroups of 256 threads on) and one block
# fewer; row lengths 2^8 .. 2^11, powers of two and 3 * 2^k.  Same inputs, so every output is the oracle's.
@pytest.mark.parametrize("n,count", [(147456, 128), (147456, 127), (262144, 32), (262144, 31), (1 << 19, 16), (1 << 20, 8),
                                     (1 << 20, 7), (393216, 22), (393216, 21), (786432, 11), (1572864, 3), (1572864, 2)])
def test_batched_rows_per_workgroup(engine, oracle, n, count):
    import torch
    m = 3 * n // 8 // 32 * 32
    key, seed = oracle.synth_bits(0xF1 + n, n + 1), oracle.synth_bits(0xF2, n)
    ref = torch.from_numpy(oracle.amp_out(key, seed, n, m, True, True, method=oracle.NTT).copy()).cuda()
    sid = engine.seed_put(seed, n, m)
    try:
        say(f"rows n={n} count={count}")
        d = _Device(key, seed, count * (m // 8))
        for fresh in (True, False):
            blk = (P.PaBlock * count)()
            for i in range(count):
                blk[i].key, blk[i].n, blk[i].m, blk[i].flags = d.key.data_ptr(), n, m, 3
                blk[i].out = d.out.data_ptr() + i * (m // 8)
                if fresh:
                    blk[i].seed = d.seed.data_ptr()
                else:
                    blk[i].seed_id = sid
            engine.batch_device(blk, 0, 0)
            torch.cuda.synchronize()
            assert torch.equal(d.out[: count * (m // 8)].reshape(count, m // 8), ref.expand(count, -1)), (n, count, fresh)
            d.take()
    finally:
        engine.seed_drop(sid)
