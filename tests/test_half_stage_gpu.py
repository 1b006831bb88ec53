"""The stage kernel's half-system workgroups where they can go wrong: ragged
tiles of either width and precision, z chunks of one plane, launches whose
workgroups fill the XCD order partly, absorbing sides of different depth or
none, against the CPU oracle value for value."""
import numpy as np
import pytest

import cgfd3d
import oracle
import scenario
from conftest import assert_same

pytestmark = pytest.mark.gpu


def _compare(sc, steps, prec, zchunks=0, conindex=None):
    g = cgfd3d.Simulation(sc["ni"], sc["nj"], sc["nk"], sc["dh"], sc["dt"], sc["nt"],
                          precision=cgfd3d.FP64 if prec == 64 else cgfd3d.FP32)
    o = oracle.Oracle(sc["ni"], sc["nj"], sc["nk"], sc["dh"], sc["dt"], sc["nt"], double=prec == 64)
    if conindex:
        sc = dict(sc, conindex=conindex)
    for e in (g, o):
        e.setup(sc)
    if zchunks:
        g.set_tuning(zchunks)
    rng = np.random.default_rng(5)
    for c, a in enumerate(scenario.random_state((sc["ni"] + 6, sc["nj"] + 6, sc["nk"] + 6), rng)):
        g.set_field(c, a)
        o.set_field(c, a)
    for e in (g, o):
        e.run(steps)
    for c in range(9):
        assert_same(g.get_field(c), o.get_field(c), f"FW[{c}]")
        for axis in range(3):
            if g.aux_size(axis):
                assert_same(g.get_aux(axis, c), o.get_aux(axis, c), f"FA{axis}[{c}]")
    assert_same(g.get_seismo(), o.get_seismo(), "seismograms")
    assert_same(g.get_pgv(), o.get_pgv(), "PGV")
    width = g.tile_width()
    g.close()
    return width


# columns one short of, at and one past a tile; rows past one and several rounds
# of the 8 XCDs; layers on one side only, of different depth, on no side
@pytest.mark.parametrize("ni,nj,nk,nabs", [(31, 37, 9, [3, 5, 2, 6, 3, 0]), (65, 18, 12, [0, 7, 4, 0, 2, 0]),
                                           (96, 70, 7, [9, 2, 0, 5, 0, 0]), (129, 9, 11, [0, 0, 0, 0, 4, 0])])
@pytest.mark.parametrize("prec", [32, 64])
@pytest.mark.parametrize("shear", [True, False])
def test_ragged_grids(ni, nj, nk, nabs, prec, shear):
    sc = scenario.config_random(ni, nj, nk, 4, nabs, seed=ni, shear=shear)
    _compare(sc, 4, prec)


@pytest.mark.parametrize("zchunks", [1, 12, 4])
def test_chunk_lengths(zchunks):
    _compare(scenario.config_random(40, 32, 12, 4, [5, 4, 4, 5, 5, 0], seed=8), 4, 32, zchunks)


@pytest.mark.parametrize("ni,nj,nk", [(80, 40, 20), (70, 57, 23)])
@pytest.mark.parametrize("conindex", [None, 12])
def test_fp64_in_narrow_tiles(ni, nj, nk, conindex):
    sc = scenario.config_random(ni, nj, nk, 4, [5, 4, 4, 5, 5, 0], seed=nk, shear=conindex is None)
    assert _compare(sc, 4, 64, conindex=conindex) == 32


# values of one wavefront, one workgroup and past one workgroup's gather
@pytest.mark.parametrize("nrecv", [0, 1, 7, 8, 113, 114])
@pytest.mark.parametrize("graph", [False, True])
def test_trace_gather_and_step_counter(nrecv, graph):
    sc = scenario.config_random(24, 20, 10, 9, [3, 2, 2, 3, 2, 0], seed=3, nrecv=max(nrecv, 2))
    sc["recv_locs"] = sc["recv_locs"][:nrecv]
    g = cgfd3d.Simulation(sc["ni"], sc["nj"], sc["nk"], sc["dh"], sc["dt"], sc["nt"])
    o = oracle.Oracle(sc["ni"], sc["nj"], sc["nk"], sc["dh"], sc["dt"], sc["nt"])
    g.setup(sc)
    o.setup(sc)
    g.set_graph(graph)
    g.run(9)
    o.run(9)
    assert g.step == 9
    for c in range(9):
        assert_same(g.get_field(c), o.get_field(c), f"FW[{c}]")
    if nrecv:
        assert_same(g.get_seismo(), o.get_seismo(), "seismograms")
    g.close()


# grids whose 2-plane chunks are just past what the chip holds of the kernel for
# nine metrics, at it, and whose 3-plane chunks are past it too
@pytest.mark.parametrize("ni,nj,nk,shear,chunks", [(64, 64, 64, True, 22), (64, 64, 48, True, 24), (60, 57, 60, True, 20),
                                                   (64, 64, 96, True, 48), (64, 64, 64, False, 32)])
def test_chunks_of_a_launch_just_past_one_round(ni, nj, nk, shear, chunks):
    sc = scenario.config_random(ni, nj, nk, 1, [5, 4, 4, 5, 5, 0], seed=nk, shear=shear)
    g = cgfd3d.Simulation(ni, nj, nk, sc["dh"], sc["dt"], 1)
    g.setup(sc)
    assert g.metrics_specialized() == (not shear)
    assert g.autotune() == chunks  # with one step there is nothing to time: the default choice
    g.close()
    _compare(sc, 1, 32)


# the width that a context reports can be set on it, in either precision
@pytest.mark.parametrize("prec", [cgfd3d.FP32, cgfd3d.FP64])
@pytest.mark.parametrize("ni,nj,nk,width", [(80, 40, 20, 32), (200, 64, 40, 32), (64, 40, 20, 64), (128, 64, 40, 64)])
def test_reported_tile_width_can_be_set(prec, ni, nj, nk, width):
    g = cgfd3d.Simulation(ni, nj, nk, 100.0, 0.005, 4, precision=prec)
    assert g.tile_width() == width
    for w in (width, 64, 0, width):
        g.set_tile_width(w)
        assert g.tile_width() == (w or width)
    if prec == cgfd3d.FP64 and width == 64:
        with pytest.raises(cgfd3d.CgfdError, match="64-column"):
            g.set_tile_width(32)
    g.close()


# the kernel with a Cartesian part holds as many workgroups as the one for three
# metrics: 2-plane chunks of the same grid fit at once
def test_chunks_of_a_hybrid_grid():
    sc = dict(scenario.config_random(64, 64, 64, 1, [5, 4, 4, 5, 5, 0], seed=9, shear=True), conindex=30)
    g = cgfd3d.Simulation(64, 64, 64, sc["dh"], sc["dt"], 1)
    g.setup(sc)
    assert g.autotune() == 32
    g.close()
