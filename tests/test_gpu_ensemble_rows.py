"""Ensembles whose rows are whole 64-B half lines, are not, and are mixed (the two
kinds of loads of the batched collide): bitwise the boxes alone."""
import pytest

from test_gpu_ensemble import _box, _same

pytestmark = pytest.mark.gpu

WHOLE = [((32, 20, 24), 2, 3.0, 2.5, 2e-5, 1), ((64, 18, 17), 0, 3.0, 5.0, 5e-6, 2)]
RAGGED = [((29, 21, 23), 1, 3.0, 2.5, 2e-5, 3), ((70, 19, 18), 0, 3.0, 5.0, 5e-6, 4)]


@pytest.mark.parametrize("precision", ["fp64", "fp32", "fp32x"])
@pytest.mark.parametrize("cases", [WHOLE, RAGGED, WHOLE[:1] + RAGGED, RAGGED[:1] + WHOLE])
def test_rows_of_either_kind(precision, cases):
    from multiphase_flow_codes_amd.lbm import Ensemble
    alone = [_box(c, precision) for c in cases]
    members = [_box(c, precision) for c in cases]
    ens = Ensemble()
    for lat in members:
        ens.add(lat, 2)
    for block, order in ((256, 1), (64, 0), (128, 1)):
        ens.set_block(block)
        ens.set_tile_order(order)
        ens.step(5)
    ens.sync()
    for a, b in zip(alone, members):
        a.step(2, 15)
        a.sync()
        _same(a, b)
    ens.close()
