"""The resident workgroups of the mean-field days with a bound on their waits that they cannot keep:
every output is the right value or NaN, whatever the arrays held before, and a wait of no time is
given up on the first day.  Through the C ABI."""

import ctypes

import numpy as np
import pytest

from test_zz_no_alloc import _case


@pytest.mark.gpu
@pytest.mark.parametrize("n", [300, 774, 2048])          # 8, 16 and 32 columns per lane
@pytest.mark.parametrize("wait_us", [0, 1])
def test_given_up_waits_leave_nan(n, wait_us):
    import torch

    from laser_polio_amd import adjoint as adj

    T = 12
    lib, p = adj._lib(), adj._p
    vp, i32 = ctypes.c_void_p, ctypes.c_int32
    lib.lp_mf_days_bounded.argtypes = [ctypes.POINTER(adj.LPMFModel), i32, i32] + [vp] * 6 + [i32, vp]
    lib.lp_mf_adjoint_days_bounded.argtypes = [ctypes.POINTER(adj.LPMFModel), i32, i32] + [vp] * 12 + [i32, vp]
    dev = torch.device("cuda", 0)
    f32 = dict(dtype=torch.float32, device=dev)
    stream = ctypes.c_void_p(torch.cuda.current_stream(dev).cuda_stream)
    print(f"[meanfield waits] n={n} wait_us={wait_us}", flush=True)
    c = _case(n, T, 3, dev)
    model = adj.LPMFModel(n=n, net=c["net"].data_ptr(), net_t=c["net_t"].data_ptr(), keep=c["keep"].data_ptr(),
                          r0_scalar=c["r0s"].data_ptr(), rho=c["rho"].data_ptr(), inv_pop=c["inv_pop"].data_ptr(),
                          season=c["season"].data_ptr(), iota=0.6, inv_tau_e=1 / 3.0, inv_tau_i=1 / 24.0)

    def forward(us):
        traj = {k: torch.full((T + 1, n), 7.0, **f32) for k in ("S", "E", "I")}
        for k, x in traj.items():
            x[0].copy_(c[k])
        rows = {k: torch.full((T, n), 7.0, **f32) for k in ("inc", "m", "g")}
        assert lib.lp_mf_days_bounded(ctypes.byref(model), 0, T, p(traj["S"]), p(traj["E"]), p(traj["I"]), p(rows["inc"]),
                                      p(rows["m"]), p(rows["g"]), us, stream) == 0
        return {**traj, **rows}

    def adjoint(fw, us):
        out = {k: torch.full((n,), 0.25, **f32) for k in ("aS", "aE", "aI")}
        out.update(r0_bar=torch.zeros(n, **f32), net_bar=torch.zeros((n, n), **f32), season_part=torch.full((T, n), 7.0, **f32))
        work = torch.zeros(2 * n, **f32)
        assert lib.lp_mf_adjoint_days_bounded(
            ctypes.byref(model), 0, T, p(fw["S"]), p(fw["I"]), p(fw["m"]), p(fw["g"]), p(c["a_inc"]), p(out["aS"]),
            p(out["aE"]), p(out["aI"]), p(out["r0_bar"]), p(out["net_bar"]), p(out["season_part"]), p(work), us, stream) == 0
        return out

    host = lambda d: {k: v.cpu().numpy() for k, v in d.items()}  # noqa: E731
    fw = forward(10_000_000)
    want = {**host(fw), **host(adjoint(fw, 10_000_000))}
    torch.cuda.synchronize()
    got = {**host(forward(wait_us)), **host(adjoint(fw, wait_us))}
    for name, w in want.items():
        assert np.isfinite(w).all(), name
        assert (np.isnan(got[name]) | (got[name] == w)).all(), name
    if wait_us == 0:
        # forward: day 0 needs no other workgroup's row; adjoint: the last day's row neither
        for name in ("inc", "m", "g"):
            assert np.array_equal(got[name][0], want[name][0]) and np.isnan(got[name][1:]).all(), name
        for name in ("S", "E", "I"):
            assert np.array_equal(got[name][:2], want[name][:2]) and np.isnan(got[name][2:]).all(), name
        assert np.array_equal(got["season_part"][-1], want["season_part"][-1]) and np.isnan(got["season_part"][:-1]).all()
        for name in ("aS", "aE", "aI", "r0_bar"):
            assert np.isnan(got[name]).all(), name
        off = ~np.eye(n, dtype=bool)
        assert np.isnan(got["net_bar"][off]).all() and not got["net_bar"][~off].any()


@pytest.mark.gpu
def test_negative_wait_is_refused():
    import torch

    from laser_polio_amd import adjoint as adj

    lib = adj._lib()
    vp, i32 = ctypes.c_void_p, ctypes.c_int32
    lib.lp_mf_days_bounded.argtypes = [ctypes.POINTER(adj.LPMFModel), i32, i32] + [vp] * 6 + [i32, vp]
    lib.lp_mf_adjoint_days_bounded.argtypes = [ctypes.POINTER(adj.LPMFModel), i32, i32] + [vp] * 12 + [i32, vp]
    x = adj._p(torch.zeros(1, dtype=torch.float32, device="cuda"))
    model = adj.LPMFModel(n=300)
    assert lib.lp_mf_days_bounded(ctypes.byref(model), 0, 1, *[x] * 6, -1, None) == -1
    assert lib.lp_mf_adjoint_days_bounded(ctypes.byref(model), 0, 1, *[x] * 12, -1, None) == -1
