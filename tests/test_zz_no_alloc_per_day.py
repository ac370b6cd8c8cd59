"""The adjoint that rolls one launch a day, the only form that uses its two work rows: above 2048
nodes and under graph capture, with the rows passed in by the caller and in the library's
fixed array.  Through the C ABI."""

import ctypes

import numpy as np
import pytest

from test_zz_no_alloc import _case


def _setup(n, T, seed):
    import torch

    from laser_polio_amd import adjoint as adj

    lib, p = adj._lib(), adj._p
    vp, i32 = ctypes.c_void_p, ctypes.c_int32
    lib.lp_mf_adjoint_days_noalloc.argtypes = [ctypes.POINTER(adj.LPMFModel), i32, i32] + [vp] * 12
    dev = torch.device("cuda", 0)
    f32 = dict(dtype=torch.float32, device=dev)
    c = _case(n, T, seed, dev)
    model = adj.LPMFModel(n=n, net=c["net"].data_ptr(), net_t=c["net_t"].data_ptr(), keep=c["keep"].data_ptr(),
                          r0_scalar=c["r0s"].data_ptr(), rho=c["rho"].data_ptr(), inv_pop=c["inv_pop"].data_ptr(),
                          season=c["season"].data_ptr(), iota=0.6, inv_tau_e=1 / 3.0, inv_tau_i=1 / 24.0)
    traj = [torch.empty((T + 1, n), **f32) for _ in range(3)]
    for tr, k in zip(traj, ("S", "E", "I")):
        tr[0].copy_(c[k])
    inc, m, g = (torch.empty((T, n), **f32) for _ in range(3))
    stream = ctypes.c_void_p(torch.cuda.current_stream(dev).cuda_stream)
    assert lib.lp_mf_days(ctypes.byref(model), 0, T, *(p(x) for x in traj), p(inc), p(m), p(g), stream) == 0
    out = {k: torch.empty(n, **f32) for k in ("aS", "aE", "aI", "r0_bar")}
    out.update(net_bar=torch.empty((n, n), **f32), season_part=torch.empty((T, n), **f32))
    work = torch.empty(2 * n, **f32)

    def run(noalloc):
        for k in ("aS", "aE", "aI"):
            out[k].fill_(0.25)
        out["r0_bar"].zero_()
        out["net_bar"].zero_()
        s = ctypes.c_void_p(torch.cuda.current_stream(dev).cuda_stream)
        common = (ctypes.byref(model), 0, T, p(traj[0]), p(traj[2]), p(m), p(g), p(c["a_inc"]), *(p(x) for x in out.values()))
        rc = lib.lp_mf_adjoint_days_noalloc(*common, s) if noalloc else lib.lp_mf_adjoint_days(*common, p(work), s)
        assert rc == 0

    return run, out, work, (c, traj, inc, m, g)


def _host(out):
    import torch

    torch.cuda.synchronize()
    return {k: v.cpu().numpy() for k, v in out.items()}


@pytest.mark.gpu
@pytest.mark.parametrize("n,T", [(2049, 5), (2600, 3)])
def test_noalloc_adjoint_above_the_resident_sizes(n, T):
    print(f"[no-alloc] n={n} T={T}", flush=True)
    run, out, work, keep = _setup(n, T, 5)
    work.fill_(float("nan"))
    run(False)
    want = _host(out)
    assert np.isfinite(work.cpu().numpy()).all()          # both rows written: this form ran
    for _ in range(2):
        for x in out.values():
            x.fill_(3.0)
        run(True)
        got = _host(out)
        for k, w in want.items():
            assert np.isfinite(w).all() and np.array_equal(got[k], w), k


@pytest.mark.gpu
@pytest.mark.parametrize("noalloc", [False, True])
@pytest.mark.parametrize("n", [40, 300])
def test_captured_adjoint_replays_to_the_eager_result(n, noalloc):
    import torch

    T = 9
    print(f"[no-alloc] captured n={n} noalloc={noalloc}", flush=True)
    run, out, work, keep = _setup(n, T, 6)
    run(noalloc)
    eager = _host(out)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        run(noalloc)
    # each form rounds about 8 times a day (2^-24 each) on values that carry on to the next
    tol = 2 * 8 * (T + 2) * 2.0**-24
    for k in range(3):
        for x in out.values():
            x.fill_(3.0)
        graph.replay()
        got = _host(out)
        for name, w in eager.items():
            err = np.linalg.norm(got[name].astype(np.float64) - w) / np.linalg.norm(w)
            assert err <= tol, (k, name, err)
