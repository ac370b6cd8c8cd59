"""The three ways the mean-field days are rolled (one workgroup, resident workgroups, a launch per
day) at the edges of their node ranges, against float64; checkpointed segments against a
rollout kept whole; rollouts under graph capture."""

import numpy as np
import pytest
import torch

from laser_polio_amd import adjoint as adj

IOTA, ITE, ITI = 14.0 / 24.0, 1 / 3.0, 1 / 24.0


def _inputs(n, T, seed=0):
    rng = np.random.default_rng([seed, n, T])
    pop = np.round(rng.lognormal(np.log(2e5), 0.6, n))
    net = rng.uniform(0, 1, (n, n)) * (rng.uniform(0, 1, (n, n)) < 0.3)
    np.fill_diagonal(net, 0.0)
    net *= 0.2 / np.maximum(net.sum(axis=1, keepdims=True), 1e-30)
    x = [rng.lognormal(0, 0.3, n), net, 1.0 + 0.4 * np.cos(np.arange(T) / 9.0), np.round(pop * rng.uniform(0.2, 0.4, n)),
         np.round(rng.uniform(0, 50, n)), np.round(rng.uniform(0, 80, n)), rng.uniform(0.8, 1.2, n), 1.0 / pop,
         rng.standard_normal((T, n))]
    return [torch.as_tensor(v, dtype=torch.float32, device="cuda") for v in x]


def _run(fn, x, dtype, **kw):
    *leaves, rho, inv_pop, g = [v.to(dtype) for v in x]
    leaves = [v.clone().requires_grad_(True) for v in leaves]
    inc = fn(*leaves, rho, inv_pop, IOTA, ITE, ITI, **kw)
    inc.backward(g)
    return [inc.detach()] + [torch.zeros_like(v) if v.grad is None else v.grad for v in leaves]


@pytest.mark.gpu
@pytest.mark.parametrize("n", [1, 2, 15, 16, 17, 32, 33, 64, 65, 127, 128, 129, 255, 256, 257, 511, 512, 513, 774, 1023,
                               1024, 1025, 2047, 2048, 2049])
@pytest.mark.parametrize("T", [1, 2, 41])
def test_every_path_matches_float64(n, T):
    print(f"[meanfield] n={n} T={T}", flush=True)
    x = _inputs(n, T)
    got = _run(adj.rollout, x, torch.float32)
    # season per node, so that each node's term of a day's season gradient is known
    x[2] = x[2][:, None].expand(T, n).contiguous()
    want = _run(adj.rollout_reference, x, torch.float64)
    terms = want[3]
    want[3] = terms.sum(dim=1)
    # about 8 roundings a day (2^-24 each) on values that carry on to the next, forward and back
    tol = 2 * 8 * (T + 2) * 2.0**-24
    off = ~torch.eye(n, dtype=torch.bool, device="cuda")
    for name, a, b in zip(("inc", "r0s", "net", "season", "S", "E", "I"), got, want):
        a = a.double()
        if name == "net":
            a, b = a[off], b[off]       # the diagonal (zero in every network) is left alone
        # a day's season gradient sums terms of both signs: its roundings go with their size
        size = terms.abs().sum(dim=1) if name == "season" else b
        err = float((a - b).norm() / size.norm().clamp_min(1e-30)) if b.numel() else 0.0
        assert err <= tol, (name, err, tol)


@pytest.mark.gpu
@pytest.mark.parametrize("n", [40, 300, 2100])
@pytest.mark.parametrize("ck", [1, 7, 30])
def test_checkpointed_segments_match_a_rollout_kept_whole(n, ck, monkeypatch):
    x = _inputs(n, 31)
    whole = _run(adj.rollout, x, torch.float32)
    monkeypatch.setattr(adj, "KEEP_BYTES", 0)
    for a, b in zip(whole, _run(adj.rollout, x, torch.float32, checkpoint=ck)):
        assert torch.equal(a, b)


@pytest.mark.gpu
def test_zero_checkpoint_is_refused():
    with pytest.raises(ValueError):
        _run(adj.rollout, _inputs(5, 4), torch.float32, checkpoint=0)


@pytest.mark.gpu
@pytest.mark.parametrize("n", [40, 300, 2100])
def test_rollout_under_graph_capture(n):
    """Captured rollouts (a launch per day above 256 nodes) replay to the eager result."""
    x = _inputs(n, 9)[:-1]
    with torch.no_grad():
        eager = adj.rollout(*x, IOTA, ITE, ITI)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            out = adj.rollout(*x, IOTA, ITE, ITI)
        for k in range(3):
            out.zero_()
            graph.replay()
            torch.cuda.synchronize()
            err = float((out - eager).norm() / eager.norm())
            assert err <= 16 * 11 * 2.0**-24, (k, err)


@pytest.mark.gpu
@pytest.mark.parametrize("n", [40, 300, 2100])
def test_days_of_no_or_little_season_match_float64(n):
    """A day's row keeps the season as a factor unless it is below 2^-20: both sides of that
    line, zero and a season of the other sign."""
    print(f"[meanfield] season edges n={n}", flush=True)
    edges = [0.0, 1.0, 2.0**-19, 2.0**-20, 2.0**-21, 0.0, -0.25, 1.5, 1e-12, 1.0]
    T = len(edges)
    x = _inputs(n, T)
    x[2] = torch.tensor(edges, dtype=torch.float32, device="cuda")
    got = _run(adj.rollout, x, torch.float32)
    x[2] = x[2][:, None].expand(T, n).contiguous()
    want = _run(adj.rollout_reference, x, torch.float64)
    terms = want[3]
    want[3] = terms.sum(dim=1)
    tol = 2 * 8 * (T + 2) * 2.0**-24      # as in test_every_path_matches_float64
    off = ~torch.eye(n, dtype=torch.bool, device="cuda")
    for name, a, b in zip(("inc", "r0s", "net", "season", "S", "E", "I"), got, want):
        a = a.double()
        if name == "net":
            a, b = a[off], b[off]
        size = terms.abs().sum(dim=1) if name == "season" else b
        assert float((a - b).norm() / size.norm().clamp_min(1e-30)) <= tol, name
