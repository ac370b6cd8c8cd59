"""A batch in which some simulations stop early (no cases left) between RI days: a stopped
simulation's ri_timer stays as its last RI day left it, the others' go on, whichever
comes first in the batch.  Bit for bit against the oracle run of each simulation alone."""

import pytest

import laser_polio_amd as lp
from cases import make
from oracle.oracle import OracleSim
from test_gpu_parity import _compare


def _sim(dies_out, seed):
    over = dict(r0=0.3, init_prev=[4, 0], dur_inf=lp.constant(4), dur_exp=lp.constant(2)) if dies_out else {}
    return make("ri_only", seed=seed, stop_if_no_cases=True, dur=60, sia_schedule=[], **over)


@pytest.mark.gpu
@pytest.mark.parametrize("dies_out", [(True, False), (False, True), (True, True, False)])
@pytest.mark.parametrize("per_call", [0, 10])
def test_stopped_sims_beside_running_ones(dies_out, per_call):
    print(f"[batch stopped] {dies_out} per_call={per_call}", flush=True)
    sims = [_sim(x, 30 + i) for i, x in enumerate(dies_out)]
    refs = [OracleSim(s.export_tables(), pop0=s.pars.init_pop).run() for s in sims]
    for x, ref in zip(dies_out, refs):
        assert (ref.stop_day is not None and 14 < ref.stop_day < 56) if x else ref.stop_day is None
    b = lp.BatchedSims(sims)
    if per_call:
        eng = b.prepare()
        for t in range(0, sims[0].nt, per_call):
            eng.run_days(t, min(sims[0].nt, t + per_call))
            eng.sync()                       # ri_timer written back as of each call's end
        b.stop_days = eng.stop_days()
        b.scatter()
    else:
        b.run()
    for s, ref in zip(sims, refs):
        _compare(s, ref)
    b.close()
