"""Blocks with constant and periodic seeds and keys, bit for bit: such inputs have the largest spectral values
and rounding errors of a transform.  The seed repeats a word pattern, so the product repeats too and follows from
the key's words folded to the pattern's length, at any block length."""
import numpy as np
import pytest

import privacyamplification_amd as P

pytestmark = pytest.mark.gpu


def say(*a):
    print("[case]", *a, flush=True)


@pytest.fixture(scope="module")
def big_engine():
    eng = P.Engine(max_n_log2=29, hbm_budget_bytes=160 << 30)
    yield eng
    eng.close()


def _bits(words):
    return np.unpackbits(np.ascontiguousarray(words).astype(">u4").view(np.uint8))


_rng = np.random.default_rng(0x57)
SEEDS = {
    "zeros": [0], "ones": [0xFFFFFFFF], "alternating bits": [0xAAAAAAAA], "half words": [0x0000FFFF],
    "flat word": [0x8F205B9B], "alternating words": [0, 0xFFFFFFFF], "word blocks": [0] * 16 + [0xFFFFFFFF] * 16,
    "byte counter": list(np.arange(256, dtype=np.uint8).view(">u4").astype(np.uint32)),
    "random words": list(_rng.integers(0, 1 << 32, 64, dtype=np.uint32)),
}


def _keys(nw):
    r = np.random.default_rng(0x6B)
    rnd = lambda: r.integers(0, 1 << 32, nw, dtype=np.uint32)
    yield "random", rnd()
    yield "7/8 ones", rnd() | rnd() | rnd()
    yield "ones", np.full(nw, 0xFFFFFFFF, np.uint32)
    yield "zeros", np.zeros(nw, np.uint32)


def _expected(key, pattern, n, m):
    """The m output bits as OutBytes, key-rest XOR and compression on."""
    h, period = n - m, len(pattern)
    x = key[: h // 32 + 1].copy()
    x[h // 32] &= np.uint32(0x80000000)
    x = np.concatenate([x, np.zeros(-x.size % period, np.uint32)])
    fold = np.bitwise_xor.reduce(x.reshape(-1, period), axis=0)
    f, s = _bits(fold).astype(float), _bits(np.array(pattern, np.uint32)).astype(float)
    y = np.rint(np.fft.irfft(np.fft.rfft(f) * np.fft.rfft(s), f.size)).astype(np.int64) & 1
    y = np.packbits(y.astype(np.uint8))
    y = np.tile(y, m // 8 // y.size + 1)[: m // 8]
    w = key[h // 32:]
    rest = (w[: m // 32] << np.uint32(1)) | (w[1: m // 32 + 1] >> np.uint32(31))
    return y ^ rest.astype(">u4").view(np.uint8)


# every kind of four-step transform: pass A from the words, of 3 * 2^k with three and six classes, and from the bit
# masks with 4 to 32 classes; blocks that fill the transform and blocks that leave part of it
SIZES = [1 << 15, 1 << 18, 3 << 18, 1 << 22, 5 << 21, 1 << 24, 11 << 21, 3 << 23, 1 << 25, 13 << 22, 1 << 26, 1 << 27,
         7 << 25, 1 << 28, 1 << 29]


@pytest.mark.parametrize("n", SIZES)
def test_structured_inputs(big_engine, n):
    import torch
    eng, m = big_engine, 3 * n // 8
    out = torch.empty(m // 8, dtype=torch.uint8, device="cuda")
    margin = torch.zeros(1, dtype=torch.float32, device="cuda")
    for kname, key in _keys(n // 32 + 1):
        dk = torch.from_numpy(key.view(np.int32)).cuda()
        for sname, pattern in SEEDS.items():
            seed = np.tile(np.array(pattern, np.uint32), n // 32 // len(pattern))
            assert seed.size == n // 32
            ds = torch.from_numpy(seed.view(np.int32)).cuda()
            ref = torch.from_numpy(_expected(key, pattern, n, m)).cuda()
            args = (n, m, P.XOR_KEY_REST | P.COMPRESS, out.data_ptr(), 0, margin.data_ptr())
            for how in ("fresh", "resident") if kname == "random" else ("fresh",):
                out.fill_(0x5A)
                margin.zero_()
                torch.cuda.synchronize()
                if how == "fresh":
                    eng.block_device(dk.data_ptr(), ds.data_ptr(), *args)
                else:
                    sid = eng.seed_put(seed, n, m)
                    eng.block_device_seeded(dk.data_ptr(), sid, *args)
                torch.cuda.synchronize()
                if how == "resident":
                    eng.seed_drop(sid)
                wrong = int((out != ref).sum())
                say(f"n={n} key {kname}, seed {sname}, {how}: margin {margin.item():.4f}")
                assert wrong == 0, (n, kname, sname, how, wrong, margin.item())
                assert margin.item() < 0.25, (n, kname, sname, how)
