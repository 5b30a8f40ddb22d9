"""Calls of one length on two streams take effect in the order of the calls, whichever route (direct product or
transform) serves them."""
import numpy as np
import pytest

import privacyamplification_amd as P

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [4096, 16384, 65536, 131072, 1 << 20])
@pytest.mark.parametrize("routes", [(False, False), (True, False), (False, True)])  # with a margin: the transform
def test_second_stream_comes_second(oracle, n, routes):
    import torch
    m = 3 * n // 8
    up = lambda a: torch.from_numpy(a.view(np.int32).copy()).cuda()
    keys = [oracle.synth_bits(0x57 + i, n + 1) for i in range(2)]
    seed = oracle.synth_bits(0x5A, n)
    ref = oracle.amp_out(keys[1], seed, n, m, True, True, method=oracle.NTT if n > 1 << 17 else oracle.DIRECT)
    print(f"[case] n={n} margins {routes}", flush=True)
    with P.Engine(max_n_log2=20) as eng:
        dk, ds = [up(k) for k in keys], up(seed)
        out = torch.zeros(m // 8, dtype=torch.uint8, device="cuda")
        margin = torch.zeros(1, device="cuda")
        streams = [torch.cuda.Stream(), torch.cuda.Stream()]
        big = torch.randn(4096, 4096, device="cuda")

        def run(i):
            eng.block_device(dk[i].data_ptr(), ds.data_ptr(), n, m, 3, out.data_ptr(), streams[i].cuda_stream,
                             margin.data_ptr() if routes[i] else None)

        for i in (1, 0, 1):
            run(i)
        torch.cuda.synchronize()
        for _ in range(3):
            out.zero_()
            torch.cuda.synchronize()
            with torch.cuda.stream(streams[0]):  # some milliseconds ahead of the first block
                for _ in range(8):
                    big = big @ big * 1e-3
            run(0)
            run(1)
            torch.cuda.synchronize()
            assert np.array_equal(out.cpu().numpy(), ref), (n, routes)


def test_first_stream_being_captured(oracle):
    """A short block on a stream that is then captured, and one on another stream meanwhile: neither call fails."""
    import torch
    n, m = 4096, 1536
    up = lambda a: torch.from_numpy(a.view(np.int32).copy()).cuda()
    key, seed = oracle.synth_bits(0x67, n + 1), oracle.synth_bits(0x68, n)
    ref = oracle.amp_out(key, seed, n, m, True, True, method=oracle.DIRECT)
    print("[case] n=4096, capture on the stream of the last block", flush=True)
    with P.Engine(max_n_log2=20) as eng:
        dk, ds = up(key), up(seed)
        outs = [torch.zeros(m // 8, dtype=torch.uint8, device="cuda") for _ in range(2)]
        streams = [torch.cuda.Stream(), torch.cuda.Stream()]
        run = lambda o, s: eng.block_device(dk.data_ptr(), ds.data_ptr(), n, m, 3, outs[o].data_ptr(), s.cuda_stream)
        run(0, streams[1])
        run(0, streams[0])
        torch.cuda.synchronize()
        outs[0].zero_()
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=streams[0], capture_error_mode="relaxed"):
            run(0, streams[0])
            run(1, streams[1])
        for _ in range(3):
            outs[0].zero_()
            graph.replay()
            torch.cuda.synchronize()
            assert np.array_equal(outs[0].cpu().numpy(), ref)
        assert np.array_equal(outs[1].cpu().numpy(), ref)
