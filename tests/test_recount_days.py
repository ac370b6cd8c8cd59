"""The recount after a host write (lp_invalidate) before each kind of day: births and deaths,
SIA, RI with both, a plain day, and a day with no RI day left ahead (no candidates are listed
then).  Bit for bit against the oracle with the same edit."""

import numpy as np
import pytest

from cases import make
from laser_polio_amd import engine as engmod
from oracle.oracle import OracleSim
from test_gpu_parity import _compare, _host_edit


@pytest.mark.gpu
@pytest.mark.parametrize("stages", [False, True])
@pytest.mark.parametrize("k", [1, 7, 10, 14, 15, 42, 43])
def test_host_edit_before_each_kind_of_day(k, stages):
    sim = make("campaigns")
    ref = OracleSim(sim.export_tables(), pop0=sim.pars.init_pop)
    slots = np.arange(sim.people.seg_begin[1], sim.people.seg_begin[1] + 3000)
    for t in range(0, sim.nt):
        if t == k:
            _host_edit(ref.cols["disease_state"], ref.cols["infection_timer"], ref.cols["acq_risk_multiplier"], slots)
        ref.day(t)
    eng = sim._ensure_engine()
    eng.run_days(0, k)
    eng.sync()
    sim._mark_device_newer()
    p = sim.people
    _host_edit(p.disease_state, p.infection_timer, p.acq_risk_multiplier, slots)
    eng = sim._ensure_engine()          # pushes the edited columns (and invalidates)
    t = k
    if stages:
        for stage in (engmod.STAGE_VITAL, engmod.STAGE_DISEASE, engmod.STAGE_RI, engmod.STAGE_SIA,
                      engmod.STAGE_TRANSMISSION, engmod.STAGE_LOG):
            eng.step(k, stage)
        t = k + 1
    eng.run_days(t, sim.nt)
    eng.sync()
    sim._mark_device_newer()
    _compare(sim, ref)
