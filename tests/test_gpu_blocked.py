"""The blocked steps (several plain steps per launch) give the single steps'
bits at the sizes where they can go wrong: strips and tiles that end inside
the lattice, segments of uneven length, lattices narrower than a strip."""
import numpy as np
import pytest

import tclb_amd
from tclb_amd import ITER_NORM

from test_gpu_parity import random_case, say

pytestmark = pytest.mark.gpu


def same(a, b):
    return np.array_equal(a, b, equal_nan=True)


@pytest.mark.parametrize("model,storage,nx,ny,k", [
    ("d2q9_SRT", "f64", 1031, 1021, 2),         # 1,031 = 16 strips of 62 and 39 columns
    ("d2q9_drag", "f64", 1031, 1021, 4),
    ("d2q9_SRT_drag", "f64", 57, 18500, 5),     # a second strip of one column: tiles take it
    ("d2q9_SRT_drag", "f64", 50, 21000, 5),     # narrower than a strip of 56: its halo wraps onto itself
    ("d2q9", "f16s", 2053, 2049, 3),            # tiles, with stochastic rounding's cost
    ("d2q9_SRT", "f16s", 2053, 2049, 3),
    ("d2q9_SRT", "f32s", 70001, 61, 5),         # rows that a segment of 12 does not divide
])
def test_marching_waves_are_bit_identical(model, storage, nx, ny, k):
    """Lattices whose k <= 5 steps per launch march (two take tiles), against
    single steps: a whole launch, a shorter rest of steps, stochastic
    rounding in the 16-bit format."""
    say(f"marching waves {model} {storage} {nx}x{ny} k={k}")
    case = random_case(model, nx, ny, 1, seed=7)
    a, b = case.build(storage), case.build(storage)
    if storage == "f16s":
        for lat in (a, b):
            lat.set_stochastic_rounding(True, seed=3)
    a.temporal_blocking, b.temporal_blocking = k, 0
    for n in (k, 2 * k - 1):
        a.iterate(n, ITER_NORM)
        b.iterate(n, ITER_NORM)
        fa = a.get_f()
        if n == k:
            assert np.mean(np.isfinite(fa)) > 0.5
        assert same(fa, b.get_f()), n


@pytest.mark.parametrize("storage,sizes,sr", [
    ("f64", [(700, 601), (61, 500), (901, 800)], False),      # marching waves, 4 steps
    ("f64", [(2050, 1031), (61, 500), (1501, 1405)], False),  # 5 steps
    ("f16s", [(2050, 1031), (61, 500), (1501, 1405)], True),  # 3, each keyed by its own iteration
    ("f64", [(75, 41), (20, 9), (130, 70)], False),           # tiles, one case smaller than a tile
    ("f16s", [(75, 41), (20, 9), (130, 70)], False),
])
def test_blocked_batch_steps_are_bit_identical(storage, sizes, sr):
    """Every case of a batch steps as a lone lattice's single steps, through
    whole launches, rests, graph replays and a case that joins mid-run."""
    say(f"blocked batch {storage} {sizes} sr={sr}")
    cases = [random_case("d2q9_drag", nx, ny, 1, seed=11 + i) for i, (nx, ny) in enumerate(sizes)]
    batch = tclb_amd.Batch("d2q9_drag", storage, 1 << 30)
    lats = []
    for c in cases:
        lat = c.build(storage)
        lat.temporal_blocking = 0
        lat.set_block(256)   # the batch's: Globals are summed by block
        lats.append(lat)
    for x in [batch] + lats if sr else []:
        x.set_stochastic_rounding(True, seed=3)
    ids = [batch.add(c) for c in cases[:2]]
    batch.set_graph_steps(2)
    for step, n in enumerate((1, 7, 24)):
        if step == 1:
            ids.append(batch.add(cases[2]))
        batch.iterate(n)
        for i, lat in zip(ids, lats):
            lat.iterate(n)
            assert same(batch.get_f(i), lat.get_f()), (n, i)
            assert same(batch.globals(i), lat.globals), (n, i)


@pytest.mark.parametrize("model,storage,shape", [
    ("d3q19", "f16s", (71, 15, 10)),          # 10,650 nodes: the last run of 256 is part full
    ("d3q27", "f32", (129, 7, 6)),
    ("d3q27_cumulant", "f64", (1, 300, 2)),   # rows of one node
    ("d2q9_autosym2", "f32s", (255, 9, 1)),
])
def test_plain_steps_on_runs_of_the_linear_index(model, storage, shape):
    """Plain steps on runs of 256 consecutive nodes (the default where rows
    are no multiple of 256) against row segments, alone and in a batch."""
    say(f"flat plain steps {model} {storage} {shape}")
    case = random_case(model, *shape, seed=9)
    a, b = case.build(storage), case.build(storage)
    b.set_block(64)
    batch = tclb_amd.Batch(model, storage, 1 << 26)
    cid = batch.add(case)
    for n in (1, 6):
        for x in (a, b, batch):
            x.iterate(n)
        assert same(a.get_f(), b.get_f()) and same(batch.get_f(cid), b.get_f())
        assert same(a.globals, b.globals) and same(batch.globals(cid), b.globals)


@pytest.mark.parametrize("model,storage,shape", [
    ("d3q19", "f64", (159, 130, 75)),          # written columns that the lattice ends inside of
    ("d3q19_lid", "f32s", (157, 131, 60)),     # rows that start inside a memory line
    ("d3q19", "f32", (256, 91, 64)),
    ("d3q27", "f64", (128, 60, 130)),
    ("d3q27_cumulant_SMAG", "f64", (128, 126, 96)),
])
def test_marching_tiles_are_bit_identical(model, storage, shape):
    """3D lattices that take two steps per launch, against single steps: odd
    and even numbers of plain steps, a change of NodeTypes, the Globals step
    behind them."""
    say(f"marching tiles {model} {storage} {shape}")
    case = random_case(model, *shape, seed=5)
    a, b = case.build(storage), case.build(storage)
    b.temporal_blocking = 0
    for n in (3, 4):
        a.iterate(n)
        b.iterate(n)
        assert a.temporal_blocking == 2 and b.temporal_blocking == 0
        fa = a.get_f()
        assert np.mean(np.isfinite(fa)) > 0.5
        assert same(fa, b.get_f()), n
        assert same(a.globals, b.globals), n
        flags = case.flags.copy()
        v = flags.reshape(-1)
        v[0:5 * v[1::5].size:5] = v[1::5]
        a.set_flags(flags)
        b.set_flags(flags)


def test_single_steps_are_timed_on_runs_and_on_row_segments(capfd, monkeypatch):
    """A lattice whose row segments leave no lane idle times both forms of its
    tiles; one whose rows end inside a block keeps runs, and one that was given
    a block keeps row segments."""
    monkeypatch.setenv("TCLBX_TUNE_LOG", "1")
    for nx, block, forms in ((128, None, {"runs", "row segments"}), (136, None, {"runs"}),
                             (128, 64, {"row segments"}), (256, None, {"row segments"})):
        say(f"forms timed at {nx}, block {block}")
        lat = tclb_amd.Lattice("d3q19", nx, 128, 8192 // nx + 1, "f16s")
        lat.set_flags(np.full((lat.nz, lat.ny, lat.nx), lat.spec.flag("MRT"), np.uint16))
        if block:
            lat.set_block(block)
        lat.init()
        capfd.readouterr()
        lat.prepare()
        log = [line for line in capfd.readouterr().err.splitlines() if "rows per tile on" in line]
        assert {line.split(" on ")[1].split(":")[0] for line in log} == forms, log
        lat.close()


def test_a_set_tile_shape_takes_single_steps():
    """A block or a number of rows per tile that the caller sets is what a 3D
    lattice steps in; 0 gives the choice back, and so does sorted dispatch
    when it is turned off.  The getter says what is in use."""
    say("a set tile shape on a marching lattice")
    case = random_case("d3q19", 159, 130, 75, seed=5)
    a = case.build("f64")
    a.iterate(3)
    assert a.temporal_blocking == 2
    for on, off in ((lambda: a.set_block(64), lambda: a.set_block(0)),
                    (lambda: setattr(a, "rows_per_tile", 2), lambda: setattr(a, "rows_per_tile", 0)),
                    (lambda: setattr(a, "sorted_dispatch", True), lambda: setattr(a, "sorted_dispatch", False))):
        on()
        a.iterate(3)
        assert a.temporal_blocking == 0
        off()
        a.iterate(3)
        assert a.temporal_blocking == 2
    b = case.build("f64")
    b.temporal_blocking = 0
    b.iterate(3 * 7)
    assert same(a.get_f(), b.get_f())


@pytest.mark.parametrize("model,storage,nx,ny,steps", [
    ("d2q9_SRT", "f64", 4, 262144, (0,)),          # a strip or a tile wastes most of its columns
    ("d2q9", "f16s", 4, 2000000, (0,)),
    ("d2q9_SRT_drag", "f64", 8, 131072, (3, 5)),   # tiles, not waves of 64 columns
    ("d2q9_SRT", "f32s", 256, 256, (5,)),
    ("d2q9", "f16s", 1, 1, (0, 3, 5)),
])
def test_steps_per_launch_by_size(model, storage, nx, ny, steps):
    """What a lattice left to itself takes, against single steps' bits."""
    say(f"steps per launch {model} {storage} {nx}x{ny}")
    case = random_case(model, nx, ny, 1, seed=3)
    a, b = case.build(storage), case.build(storage)
    b.temporal_blocking = 0
    for x in (a, b):
        x.iterate(8)
    assert a.temporal_blocking in steps
    assert same(a.get_f(), b.get_f()) and same(a.globals, b.globals)
