"""Launch shapes of the collide with FP64 arithmetic at the edges of their rules:
one wavefront per workgroup in short rows, contiguous ranges per XCD and
non-temporal loads in large lattices without spheres, a workgroup per row in
place.  The same nodes are collided in place by
another shape and in another layout, so both agree bitwise; a box in the
plane-major layout checks the padding of the rows too."""
import numpy as np
import pytest

from helpers import small_params

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,precision,walls", [
    # short rows, more than 4096 tiles
    ((4, 90, 80), "fp64", False), ((5, 66, 65), "fp64", True), ((17, 64, 66), "fp64", False),
    # the last of them and the first of the others
    ((48, 66, 64), "fp64", True), ((49, 64, 66), "fp64", False),
    # 2.5 GiB of populations in two buffers; whole half lines or not; rows too short for ranges
    ((32, 536, 522), "fp64", False), ((33, 530, 512), "fp64", True), ((31, 540, 540), "fp64", False),
    # in place, a workgroup per row of one or two tiles; ranges in longer rows
    ((64, 336, 336), "fp64", False), ((65, 480, 460), "fp64", True), ((256, 240, 236), "fp64", False),
    ((20, 70, 66), "fp32x", False), ((64, 70, 64), "fp32x", True), ((100, 50, 47), "fp32x", False),
])
def test_shapes_agree_bitwise(monkeypatch, n, precision, walls):
    from multiphase_flow_codes_amd.lbm import Lattice
    prm = small_params(n=n, walls=walls, forcing=False, strong_forcing=False, body_force=(2e-5, 0.0, 1e-5))
    rng = np.random.default_rng(sum(n))
    u = [rng.normal(0, 0.01, (n[2], n[1], n[0])) for _ in range(3)]
    got = []
    for storage, layout in (("ab", "rows"), ("aa", "rows"), ("ab", "planes")):
        monkeypatch.setenv("MFC_POP_LAYOUT", layout)
        lat = Lattice(prm, precision, storage=storage)
        lat.upload_macro(None, *u)
        lat.initpop()
        lat.collision_mrt()      # moments from the arrays
        lat.streaming()
        lat.macrovar()
        lat.step(1, 3)
        got.append(lat.download_macro())
        lat.close()
    assert all(np.all(np.isfinite(a)) and np.any(a != u[0]) for a in got[0])
    for other in got[1:]:
        for a, b in zip(got[0], other):
            assert np.array_equal(a, b)
