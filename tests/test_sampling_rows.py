"""Sampling paths chosen by size: k_finish with 512 threads a node (more nodes than CUs), and
the 64-bit agent search a probe takes when a weight in its chunk reaches 2^32 (a risk of 256).
Bit for bit against the oracle."""

import numpy as np
import pytest

import laser_polio_amd as lp
from cases import make
from oracle.oracle import OracleSim
from test_gpu_parity import _compare


def _edit_risk(sim, kind):
    """Acquisition risks around the 32-bit weight limit, on a spread of slots and whole chunks."""
    risk = sim.people.acq_risk_multiplier
    r = np.random.default_rng(1)
    some = r.choice(len(risk), size=len(risk) // 50, replace=False)
    if kind == "edge":          # weights of 2^32 - 256, exactly 2^32 and one step above
        risk[some] = r.choice(np.array([255.99998, 256.0, 256.00003], np.float32), len(some))
    elif kind == "large":
        risk[some] = r.uniform(300, 4000, len(some)).astype(np.float32)
        risk[5120:5376] = 1000.0
    elif kind == "odd":         # zero, negative and NaN weigh nothing; tiny rounds to 0 or 1
        risk[some] = r.choice(np.array([0.0, -0.0, -3.0, np.nan, 2.9e-8, 3.1e-8], np.float32), len(some))


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["edge", "large", "odd"])
@pytest.mark.parametrize("case", ["small3", "hot", "bignode"])
def test_risk_extremes_match_oracle(case, kind):
    sim = make(case)
    _edit_risk(sim, kind)
    ref = OracleSim(sim.export_tables(), pop0=sim.pars.init_pop).run()
    assert ref.res["new_exposed"].sum() > 0
    sim.run()
    # the risks themselves, NaN equal to NaN; _compare takes the rest
    got, want = sim.people.acq_risk_multiplier, ref.cols.pop("acq_risk_multiplier")
    assert np.array_equal(got, want, equal_nan=True)
    _compare(sim, ref)


@pytest.mark.gpu
@pytest.mark.parametrize("n", [255, 256, 257, 300])
def test_finish_workgroup_size_by_nodes_matches_oracle(n):
    """Around one node per CU (256): many later rounds and take-all nodes in both variants."""
    rng = np.random.default_rng(n)
    xy = rng.uniform(0, 50, (n, 2))
    d = np.sqrt(((xy[:, None, :] - xy[None, :, :]) ** 2).sum(-1))
    sim = make("hot", dur=10, init_pop=rng.integers(50, 1800, n), r0=200, r0_scalars=rng.lognormal(0, 0.3, n),
               init_prev=[3] * n, distances=d, dur_exp=lp.constant(2), dur_inf=lp.constant(3))
    ref = OracleSim(sim.export_tables(), pop0=sim.pars.init_pop).run()
    assert ref.res["new_exposed"].sum() > 0
    sim.run()
    _compare(sim, ref)
