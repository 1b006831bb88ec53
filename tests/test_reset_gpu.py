"""A context that has run and is reset equals a fresh one value for value, on
grids large enough that only two of the four wavefield sets are cleared and on
small ones, whatever the sets held before: the middle of a step, a large random
state, infinities and NaN."""
import numpy as np
import pytest

import cgfd3d
import scenario
from conftest import assert_same

pytestmark = pytest.mark.gpu


def _sim(sc, prec):
    g = cgfd3d.Simulation(sc["ni"], sc["nj"], sc["nk"], sc["dh"], sc["dt"], sc["nt"], precision=prec)
    g.setup(sc)
    return g


def _same(a, b, what):
    for which, name in ((0, "FW"), (1, "W"), (2, "tW")):
        for c in range(9):
            assert_same(a.get_field(c, which), b.get_field(c, which), f"{what}: {name}[{c}]")
    for axis in range(3):
        for which in (0, 1, 2):
            for c in range(9):
                assert_same(a.get_aux(axis, c, which), b.get_aux(axis, c, which), f"{what}: aux{axis} {which} [{c}]")
    assert_same(a.get_seismo(), b.get_seismo(), f"{what}: seismograms")
    assert_same(a.get_pgv(), b.get_pgv(), f"{what}: PGV")


@pytest.mark.parametrize("prec,ni,nj,nk", [(cgfd3d.FP32, 130, 129, 70), (cgfd3d.FP64, 70, 90, 70), (cgfd3d.FP32, 40, 30, 20)])
@pytest.mark.parametrize("variant", [0, 1, 2])
def test_reset_equals_a_fresh_context(prec, ni, nj, nk, variant):
    sc = scenario.config_random(ni, nj, nk, 8, [5, 4, 4, 6, 5, 0], seed=ni)
    padded = -(-(ni + 3) // 64) * 64 * (nj + 3) * (nk + 8) * (8 if prec == cgfd3d.FP64 else 4)
    assert (36 * padded > 128 << 20) == (ni != 40)  # the larger grids clear in part
    fresh, used = _sim(sc, prec), _sim(sc, prec)
    fresh.set_variant(variant)
    used.set_variant(variant)
    fresh.run(2)
    fresh.run_stages(2)
    rng = np.random.default_rng(1)
    for fill in ("large", "special"):
        st = scenario.random_state((ni + 6, nj + 6, nk + 6), rng)
        for c in range(9):
            a = st[c] * 1e6
            if fill == "special":
                a[::7], a[1::7], a[2::7] = np.nan, np.inf, -np.inf
            used.set_field(c, a)
            for axis in range(3):
                v = rng.standard_normal(used.aux_size(axis)) * (np.nan if fill == "special" else 1e6)
                used.set_aux(axis, c, v.astype(np.float64 if prec == cgfd3d.FP64 else np.float32))
        used.run_stages(4 + 3)  # a whole step and most of another
        used.init()
        used.run(2)
        used.run_stages(2)
        _same(used, fresh, f"after {fill}")
        used.init()
    fresh.close()
    used.close()
