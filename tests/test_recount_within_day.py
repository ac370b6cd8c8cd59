"""A host write (lp_invalidate) between two stage calls of one day, before each stage of an RI day
with births and a campaign: the recount that follows has to list the RI candidates for the RI
day ahead, today's before its RI stage and the next one after it.  The next RI day then runs from
the lists, or by stage calls.  Bit for bit against the oracle with the same edit."""

import numpy as np
import pytest

from cases import make
from laser_polio_amd import engine as engmod
from oracle.oracle import OracleSim
from test_gpu_parity import _compare, _host_edit

STAGES = [engmod.STAGE_VITAL, engmod.STAGE_DISEASE, engmod.STAGE_RI, engmod.STAGE_SIA, engmod.STAGE_TRANSMISSION,
          engmod.STAGE_LOG]
# the schedule flags of the stages up to each one, for a day that the oracle runs in two parts
FLAGS = {engmod.STAGE_VITAL: engmod.DAY_VD_STEP | engmod.DAY_VD_COPY, engmod.STAGE_DISEASE: engmod.DAY_DS | engmod.DAY_STOPCHK,
         engmod.STAGE_RI: engmod.DAY_RI, engmod.STAGE_SIA: engmod.DAY_SIA,
         engmod.STAGE_TRANSMISSION: engmod.DAY_TX, engmod.STAGE_LOG: 0}


class EditedDay(OracleSim):
    """The oracle with an edit of the agents before stage `before` of tick `k`."""

    def run_edited(self, k, before, edit):
        self.run(0, k)
        flags = int(self.tb.day_flags[k])
        if before == engmod.STAGE_LOG:
            count = self._count

            def edit_and_count(t):
                if t == k:
                    edit(self.cols)
                count(t)

            self._count = edit_and_count
            self.day(k)
        else:
            first = sum(FLAGS[s] for s in STAGES if s < before)
            self.tb.day_flags[k] = flags & first
            self.day(k)
            edit(self.cols)
            self.tb.day_flags[k] = flags & ~first
            self.day(k)
            self.tb.day_flags[k] = flags
        return self.run(k + 1)


def test_two_part_day_of_the_oracle_is_its_day():
    sim = make("campaigns")
    whole = OracleSim(sim.export_tables(), pop0=sim.pars.init_pop).run()
    for before in STAGES[1:]:
        parts = EditedDay(sim.export_tables(), pop0=sim.pars.init_pop).run_edited(14, before, lambda cols: None)
        for name, rows in whole.res.items():
            assert np.array_equal(parts.res[name], rows), (before, name)
        for name, col in whole.cols.items():
            assert np.array_equal(parts.cols[name], col), (before, name)


@pytest.mark.gpu
@pytest.mark.parametrize("next_ri_by_stages", [False, True])
@pytest.mark.parametrize("before", STAGES[1:])
def test_host_edit_between_the_stages_of_an_ri_day(before, next_ri_by_stages):
    k, k2 = 14, 28
    print(f"[recount within a day] before={before} stages={next_ri_by_stages}", flush=True)
    sim = make("campaigns")
    slots = np.arange(sim.people.seg_begin[1], sim.people.seg_begin[1] + 3000)
    ref = EditedDay(sim.export_tables(), pop0=sim.pars.init_pop).run_edited(
        k, before, lambda c: _host_edit(c["disease_state"], c["infection_timer"], c["acq_risk_multiplier"], slots))
    eng = sim._ensure_engine()
    eng.run_days(0, k)
    for stage in STAGES:
        if stage == before:
            eng.sync()
            sim._mark_device_newer()
            p = sim.people
            _host_edit(p.disease_state, p.infection_timer, p.acq_risk_multiplier, slots)
            eng = sim._ensure_engine()      # pushes the edited columns (and invalidates)
        eng.step(k, stage)
    t = k + 1
    if next_ri_by_stages:
        eng.run_days(t, k2)
        for stage in STAGES:
            eng.step(k2, stage)
        t = k2 + 1
    eng.run_days(t, sim.nt)
    eng.sync()
    sim._mark_device_newer()
    assert ref.res["ri_vaccinated"][[28, 42]].sum() > 0
    _compare(sim, ref)


@pytest.mark.gpu
def test_ri_stage_twice_on_a_tick_lists_each_candidate_once():
    """RI of tick 14 stepped twice in a population of mostly RI candidates (the draws are keyed by
    agent and tick, so the second step changes no agent): the days after it are the oracle's,
    the RI day 28 from the lists."""
    k = 14
    sim = make("campaigns", ri_age_days=(0, 20000))
    p = sim.people
    timers = np.concatenate([p.ri_timer[b:e] for b, e in zip(p.seg_begin, p.live_end, strict=True)])
    assert (timers > 28).mean() > 0.5          # candidates of the lists made on ticks 0 to 14
    print("[ri twice] candidates", int((timers > 28).sum()), flush=True)
    ref = OracleSim(sim.export_tables(), pop0=sim.pars.init_pop).run()
    eng = sim._ensure_engine()
    eng.run_days(0, k)
    for stage in STAGES:
        eng.step(k, stage)
        if stage == engmod.STAGE_RI:
            eng.step(k, stage)
    eng.run_days(k + 1, sim.nt)
    eng.sync()
    sim._mark_device_newer()
    for name in ("ri_vaccinated", "ri_protected", "ri_new_exposed_by_strain", "ipv_vaccinated"):
        ref.res[name][k] = getattr(sim.results, name)[k]       # the second step's row stands
    assert ref.res["ri_vaccinated"][28].sum() > 0
    _compare(sim, ref)
