"""The tile rule of the specialised convolutions, on the host: which shapes have
a tile must not depend on the batch or the chip (packed weights are laid out
without either), and no row that one fits falls to the generic kernel."""
import pytest

import rustnn_amd as R


@pytest.mark.parametrize("k,s,p", [(3, 1, 1), (3, 2, 1), (1, 1, 0), (1, 2, 0)])
@pytest.mark.parametrize("dx", [0, 1])
def test_plan_or_none_for_every_batch(k, s, p, dx):
    for cin, cout in ((32, 32), (3, 64), (128, 256)):
        for h in (1, 2, 7, 32, 160):
            for w in range(1, 261):
                sp = R.ConvSpec.make(cin, cout, k, s, p, h, w)
                have = {R.dbg_conv_plan(sp, dx, n, cus) is not None
                        for n in (1, 2, 8, 128) for cus in (1, 256, 304)}
                assert len(have) == 1, (cin, cout, h, w)
                if k == 3 and w <= 254:
                    assert have == {True}, (cin, cout, h, w)


def test_wide_rows_take_two_groups_a_wave():
    for n, h, w, npw in ((1, 160, 160, 2), (1, 3, 250, 2), (1, 40, 128, 1), (1, 32, 32, 1),
                         (128, 32, 32, 2)):
        sp = R.ConvSpec.make(32, 32, 3, 1, 1, h, w)
        assert [R.dbg_conv_plan(sp, d, n)[3] for d in (0, 1)] == [npw, npw], (n, h, w)


def test_strided_tiles_by_items():
    """128 positions from one item a CU on, 32 where 64 idle half of the chip."""
    for n, cin, cout, h, npos, npw in ((128, 32, 64, 32, 128, 2), (128, 64, 128, 16, 64, 1),
                                       (32, 32, 64, 32, 32, 1), (1, 32, 64, 32, 32, 1),
                                       (33, 32, 64, 32, 64, 1), (128, 16, 32, 32, 64, 1)):
        sp = R.ConvSpec.make(cin, cout, 3, 2, 1, h, h)
        plan = R.dbg_conv_plan(sp, 0, n)
        assert (plan[0] * plan[1] * sp.ow, plan[3]) == (npos, npw), (n, cin, h, plan)
