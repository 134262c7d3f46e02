"""The batch's choice of work units per workgroup: classes whose launches in the
trial steps are all too short for two units a workgroup (under 2048 units, so
that every candidate is the same launch) keep one."""
import pytest

import pgmg_amd as P

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [P.PREC_FP64, P.PREC_MIXED])
@pytest.mark.parametrize("shape", [(33, 33, 33), (40, 50, 60), (17, 60, 30)])
def test_short_launches_keep_one_unit(shape, precision):
    print("case", shape, precision, flush=True)
    with P.Batch(1 << 30, max_slots=2, precision=precision) as b:
        b.admit(*shape, P.FAM_Q1_ANISO, 3, 1e-30, 40)
        assert b.tiles()[0] is None
        for _ in range(10):
            b.step()
        assert set(b.tiles()[0].values()) == {1}
