"""The cumulant collision without its third order (Omega = 1, the default)
and with it, through the C ABI, on random NodeTypes and boundary conditions."""
import numpy as np
import pytest

import tclb_amd

from conftest import oracle_for_case
from test_gpu_parity import random_case, rel_max, say

pytestmark = pytest.mark.gpu


def with_omega(model, omega, steps=6):
    case = random_case(model, 11, 8, 5, seed=47, steps=steps)
    case.settings = [s for s in case.settings if s[0] != "Omega"] + [("Omega", omega)]
    return case


@pytest.mark.parametrize("model", ["d3q27_cumulant", "d3q27_cumulant_SMAG", "d3q27_cumulant_AVG_IB_SMAG"])
@pytest.mark.parametrize("omega", [1.0, 1.25])
def test_third_order_f64(oracle_mod, model, omega):
    """FP64 against the oracle, to the 1e-12 that its other cases are held to."""
    say(f"third order {model} Omega {omega}")
    case = with_omega(model, omega)
    lat, orc = case.build("f64"), oracle_for_case(oracle_mod, case, "f64")
    for n in (1, 6):
        lat.iterate(n)
        orc.iterate(n)
        assert rel_max(lat.get_f(), orc.get_f()) <= 1e-12, n


@pytest.mark.parametrize("model,storage", [("d3q27_cumulant", "f32"), ("d3q27_cumulant", "f16s"),
                                           ("d3q27_cumulant_SMAG", "f32s"), ("d3q27_cumulant_IB", "bf16s"),
                                           ("d3q27_cumulant_AVG", "f32s")])
def test_left_out_third_order_is_exact(model, storage):
    """Omega = 1 + 2^-40 is 1 in the float collision but not to the test for
    1, so its third order is formed and multiplied by zero: the values must
    be those of Omega = 1, where it is left out."""
    say(f"third order left out {model} {storage}")
    out = []
    for omega in (1.0, 1.0 + 2.0 ** -40):
        lat = with_omega(model, omega).build(storage)
        lat.iterate(7)
        out.append((lat.get_f(), lat.globals))
    assert np.array_equal(out[0][0], out[1][0])
    assert np.array_equal(out[0][1], out[1][1])


def test_timing_of_the_tiles_leaves_the_averages():
    """The averages of a lattice large enough to have its tiles timed
    (2^20 nodes) are those of one whose tiles are given: trial steps, which
    run on the current snapshot, would add to them."""
    nx, ny, nz = 128, 128, 64
    rng = np.random.default_rng(8)
    flags = np.where(rng.random((nz, ny, nx)) < 0.05, 0, tclb_amd.Model("d3q27_cumulant_AVG").flag("MRT"))
    runs = []
    for rows in (0, 1):
        lat = tclb_amd.Lattice("d3q27_cumulant_AVG", nx, ny, nz, "f16s")
        lat.set_flags(flags.astype(np.uint16))
        lat.set_setting("ForceX", 1e-5)
        lat.rows_per_tile = rows
        lat.init()
        if rows == 0:
            lat.prepare()
        lat.iterate(20)
        runs.append(lat.get_averages())
        lat.close()
    assert np.abs(runs[0]["avgP"]).max() > 0 or np.abs(runs[0]["avgUX"]).max() > 0
    for k, v in runs[0].items():
        assert np.array_equal(v, runs[1][k]), k
