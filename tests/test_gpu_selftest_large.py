"""The self-tests whose range follows the engine's largest length, at the lengths beyond the default (2^28, 2^29)."""
import pytest

import privacyamplification_amd as P

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name", ["ToBinaryArray", "SetFirstElementToZero"])
@pytest.mark.parametrize("reverse", [True, False])
def test_selftest_of_the_largest_engine(name, reverse):
    print("[case] selftest", name, "to 2^29, out_reverse_endian", reverse, flush=True)
    with P.Engine(max_n_log2=29, out_reverse_endian=reverse) as eng:
        ok, report = eng.selftest(name)
        assert ok, report
