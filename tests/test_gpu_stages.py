"""Stage timing names the kernels that ran, by block size and seed mode."""
import numpy as np
import pytest

import privacyamplification_amd as P

pytestmark = pytest.mark.gpu

# n: pass A, pass A' and output; margin: the transform also where the direct product serves
STAGES = [(4096, False, {"k_direct"}), (4096, True, {"k_small"}), (1 << 17, False, {"k_direct"}),
          (1 << 17, True, {"k_mid_fwd", "k_rows", "k_mid_inv"}), (1 << 20, False, {"k_mid_fwd", "k_rows", "k_mid_inv"}),
          (3 << 18, False, {"k_mix_fwd", "k_rows", "k_mix_inv"}), (3 << 23, False, {"k_mix_fwd", "k_rows", "k_mix_inv"}),
          (1 << 24, False, {"k_mid_fwd", "k_rows", "k_mid_inv"}),
          (1 << 25, False, {"k_transpose_bits", "k_fwd_cols", "k_rows", "k_inv_cols", "k_pack"}),
          (1 << 28, False, {"k_transpose_bits", "k_fwd_cols", "k_rows", "k_inv_big1+k_inv_big2", "k_pack"})]


@pytest.mark.parametrize("n,margin,names", STAGES)
def test_stage_names(n, margin, names):
    import torch
    m = 3 * n // 8
    print(f"[case] n={n} margin {margin}", flush=True)
    with P.Engine(max_n_log2=28) as eng:
        key = torch.zeros(n // 32 + 2, dtype=torch.int32, device="cuda")
        seed = torch.zeros(n // 32, dtype=torch.int32, device="cuda")
        out = torch.zeros(m // 8, dtype=torch.uint8, device="cuda")
        mg = torch.zeros(1, dtype=torch.float32, device="cuda")
        torch.cuda.synchronize()
        sid = eng.seed_put(np.zeros(n // 32, np.uint32), n, m)
        args = (n, m, 3, out.data_ptr(), 0, mg.data_ptr() if margin else None)
        eng.stage_timing(True)
        for resident in (False, True):
            if resident:
                eng.block_device_seeded(key.data_ptr(), sid, *args)
            else:
                eng.block_device(key.data_ptr(), seed.data_ptr(), *args)
            st = eng.stage_times()
            assert all(ms > 0 and launches == 1 for ms, launches in st.values())
            assert {s.split("(")[0] for s in st} == names
            operands = "(key)" if resident else "(key+seed)"
            assert all(s.endswith(operands) for s in st if "(" in s), st
