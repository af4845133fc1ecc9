"""When large batches of row-major angles are copied to angle-major order first: the
measured cases on either side of the line."""
import pytest

from mentpy_amd.simulators.hip_simulator import _angle_pass


# (slots, sets, angles per set, inputs, forward copies, sampled copies)
@pytest.mark.parametrize("slots,B,n,S,forward,sampled", [
    (4, 131072, 76, 1, True, False), (4, 65536, 76, 1, False, False), (4, 62000, 156, 1, True, False),
    (4, 72115, 156, 1, True, True), (4, 50632, 316, 1, True, False), (4, 524288, 156, 1, True, True),
    (5, 100000, 95, 1, True, False), (5, 49000, 195, 1, True, False), (5, 40506, 395, 1, False, False),
    (5, 63291, 395, 1, True, True), (6, 106000, 90, 1, False, False), (6, 41000, 234, 1, False, False),
    (6, 111111, 144, 1, True, True), (6, 33755, 474, 1, False, False), (6, 52742, 474, 1, True, False),
    (3, 126000, 75, 1, True, False), (3, 60000, 237, 1, False, False), (4, 60000, 236, 1, True, False),
    (3, 136752, 117, 1, True, True), (2, 524288, 78, 1, False, False),
    (4, 524288, 36, 1, False, False), (4, 524288, 76, 3, False, False), (7, 65536, 273, 1, False, False)])
def test_angle_pass_rule(slots, B, n, S, forward, sampled):
    assert _angle_pass(slots, B, n, S, False) is forward
    assert _angle_pass(slots, B, n, S, True) is sampled
