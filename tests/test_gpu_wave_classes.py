"""k_rc_wave at the edges of its classes: stacks of 2, 25, 32, 33, 48, 49 and 60
columns, r_B up to the class limit and 64, rows per lane (tiles of 200, 512, 513,
1024 rows: 4 and 8 of 8, 9 and 16 of 16).  The problem and the bound of
test_gpu_wide_stacks."""
import pytest

import test_gpu_wide_stacks as wide

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("NB,rc,ra,rb", [(200, 1, 1, 1), (200, 24, 1, 7), (200, 16, 16, 32), (512, 20, 13, 20),
                                         (512, 30, 18, 48), (513, 30, 19, 48), (513, 40, 20, 64), (1024, 31, 29, 10)])
def test_wave_classes(ctx, NB, rc, ra, rb):
    wide.test_wide_stacks(ctx, NB, rc, ra, rb)
