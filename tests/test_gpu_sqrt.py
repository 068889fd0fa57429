"""GPU test of the library's square root, on whose correct rounding every pass's
bits rest, for every float."""
import pytest

pytestmark = pytest.mark.gpu


def test_every_float(pbf):
    r = pbf.check_sqrt()
    assert r["mismatches"] == 0
    # 2^-96 .. 2^96: 192 binades of 2^23 floats, and the last end
    assert r["fast"] == 192 * 2**23 + 1
