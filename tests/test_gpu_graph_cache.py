"""The graphs that batches capture: ragged short blocks replay those of their shape class, and their number is
bounded whatever mixes of lengths and counts come."""
import numpy as np
import pytest

import privacyamplification_amd as P

pytestmark = pytest.mark.gpu


def _batch(oracle, shapes, tag):
    """(blocks, buffers, references) of fresh blocks, each with a key and a seed of its own."""
    import torch
    blk, keep = (P.PaBlock * len(shapes))(), []
    for i, (b, (n, m)) in enumerate(zip(blk, shapes)):
        key, seed = oracle.synth_bits(tag + 2 * i, n + 1), oracle.synth_bits(tag + 2 * i + 1, n)
        ref = oracle.amp_out(key, seed, n, m, True, True, method=oracle.DIRECT)
        k, s = (torch.from_numpy(a.view(np.int32).copy()).cuda() for a in (key, seed))
        o = torch.zeros(m // 8, dtype=torch.uint8, device="cuda")
        b.key, b.seed, b.n, b.m, b.flags, b.out = k.data_ptr(), s.data_ptr(), n, m, 3, o.data_ptr()
        keep.append((k, s, o, ref))
    torch.cuda.synchronize()
    return blk, keep


def _check(eng, blk, keep, what):
    import torch
    eng.batch_device(blk, P.BATCH_GRAPH, 0)
    torch.cuda.synchronize()
    for i, (_, _, o, ref) in enumerate(keep):
        assert np.array_equal(o.cpu().numpy(), ref), (what, i)


@pytest.mark.parametrize("lg", [9, 11, 14, 16])
def test_ragged_short_batches_replay(oracle, lg):
    rng = np.random.default_rng(lg)
    print(f"[case] ragged pairs of 2^{lg - 1} .. 2^{lg} bits", flush=True)
    with P.Engine(max_n_log2=20) as eng:
        for rep in range(40):
            shapes = []
            for _ in range(2):
                n = int(rng.integers((1 << (lg - 1)) // 32 + 1, (1 << lg) // 32 + 1)) * 32
                shapes.append((n, int(rng.integers(1, n // 32)) * 32))
            _check(eng, *_batch(oracle, shapes, 0x6C0 + 4 * rep), shapes)
        captured, kept = eng.batch_graphs()
        assert captured <= 16 and kept <= 16  # quarters of the output by quarters of the key


def test_number_of_graphs_is_bounded(oracle):
    print("[case] batches of 1 .. 90 blocks of 64 bits, then the first again", flush=True)
    with P.Engine(max_n_log2=20) as eng:
        blk, keep = _batch(oracle, [(64, 32)] * 90, 0x7C0)
        for count in list(range(1, 91)) + [1, 90, 89]:
            part = (P.PaBlock * count)(*blk[:count])
            for _, _, o, _ in keep:
                o.zero_()
            _check(eng, part, keep[:count], count)
        captured, kept = eng.batch_graphs()
        # the arena may have grown, which drops them all; of the last three batches only the first was dropped
        assert kept <= 64 and captured == 91
