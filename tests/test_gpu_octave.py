"""A block length of 3 * 2^(k-2) and one of 2^k share their workspace and get their tables together: whichever an
engine has served, the other needs no device memory more."""
import numpy as np
import pytest

import privacyamplification_amd as P

pytestmark = pytest.mark.gpu
ORDERS = [(1 << 22, 3 << 20), (3 << 20, 1 << 22), (1 << 22, 2500000), (2500000, 1 << 22)]


def say(*a):
    print("[case]", *a, flush=True)


class _Block:
    def __init__(self, oracle, n, tag):
        import torch
        self.n, self.m = n, 3 * n // 8 // 32 * 32
        key, seed = oracle.synth_bits(tag, n + 1), oracle.synth_bits(tag + 1, n)
        self.host = key, seed
        self.ref = oracle.amp_out(key, seed, n, self.m, True, True, method=oracle.NTT)
        self.key, self.seed = (torch.from_numpy(a.view(np.int32).copy()).cuda() for a in (key, seed))
        self.out = torch.zeros(self.m // 8, dtype=torch.uint8, device="cuda")

    def run(self, eng, stream):
        eng.block_device(self.key.data_ptr(), self.seed.data_ptr(), self.n, self.m, 3, self.out.data_ptr(), stream)

    def check(self):
        import torch
        torch.cuda.synchronize()
        assert np.array_equal(self.out.cpu().numpy(), self.ref), self.n
        self.out.zero_()
        torch.cuda.synchronize()


@pytest.mark.parametrize("first,second", ORDERS)
def test_both_lengths_in_the_budget_of_one(oracle, first, second):
    # 12 MB for the tables that pa_create makes: less than a quarter of either workspace's double
    budget = P.workspace_bytes(first, first // 2 // 32 * 32) + (12 << 20)
    with P.Engine(max_n_log2=22, hbm_budget_bytes=budget) as eng:
        for i, n in enumerate((first, second, first)):
            say(f"budget {budget}, n={n}")
            b = _Block(oracle, n, 0x0C0 + i)
            b.run(eng, 0)
            b.check()
            key, seed = b.host
            assert np.array_equal(eng.amplify(key, seed, n, b.m), b.ref), (n, "host")


@pytest.mark.parametrize("first,second", ORDERS)
def test_captured_after_the_other_length(oracle, first, second):
    import torch
    with P.Engine(max_n_log2=22) as eng:
        warm, b = _Block(oracle, first, 0x0D0), _Block(oracle, second, 0x0D8)
        warm.run(eng, 0)
        warm.check()
        say(f"capture n={second} after n={first}")
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            b.run(eng, torch.cuda.current_stream().cuda_stream)
        for _ in range(3):
            graph.replay()
            b.check()
            warm.run(eng, 0)
            warm.check()
