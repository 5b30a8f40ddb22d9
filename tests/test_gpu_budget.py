"""The HBM budget counts everything that a resident seed keeps on the device."""
import pytest

import privacyamplification_amd as P

pytestmark = pytest.mark.gpu


# one-workgroup size, with and without the seed's own words, a length of 3 * 2^k, one that does not fill its transform
@pytest.mark.parametrize("n", [16384, 1 << 18, 1 << 19, 3 << 18, 2500000, 1 << 22])
def test_resident_seeds_stay_in_the_budget(oracle, n):
    m = 3 * n // 8 // 32 * 32
    fixed = P.workspace_bytes(n, m) + (8 << 20)  # the workspace and the tables of pa_create
    budget = fixed + 4 * n * max(100, (1 << 27) // n)  # room for 100 spectra and more, so that a few percent show
    seed = oracle.synth_bits(0xB0, n)
    L = P.transform_len(n, m)
    kept = 4 * L + (L // 8 if L > 1 << 14 else 0) + (n // 8 if L <= 1 << 18 else 0)  # spectrum, prefix words, seed words
    print(f"[case] n={n} budget {budget}, {kept} bytes a seed", flush=True)
    with P.Engine(max_n_log2=22, hbm_budget_bytes=budget) as eng:
        counts = []
        for _ in range(2):  # dropped seeds give back what they took
            ids = []
            with pytest.raises(P.EngineError) as err:
                while True:
                    ids.append(eng.seed_put(seed, n, m))
            assert err.value.status == -4
            counts.append(len(ids))
            for sid in ids:
                eng.seed_drop(sid)
        assert counts[0] == counts[1]
        workspace = P.workspace_bytes(n, m)
        assert 1 <= counts[0] * kept <= budget - workspace, (n, counts, kept)
