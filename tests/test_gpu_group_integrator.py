"""The integrator's groups of 64 nodes, partial and full.  The nodes of a
group share barriers, flags and LDS but no arithmetic, so a node's results are
the same to the last bit in any lane and beside any other nodes; a forest's
operations give the same state whichever lane runs them, chained or claimed;
and the four waves of a group compute the right-hand side that one lane does."""
from fractions import Fraction

import numpy as np
import pytest

from galacticus_amd import params as gp, trees as tr, workloads as wl
from galacticus_amd.cooling import synthetic_cie_table

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch_cuda():
    torch = pytest.importorskip("torch")
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return torch


def _evolve(torch, physics, options, y, node_par, t0, t1, h):
    from galacticus_amd.evolver import NodeEvolverBatched
    d = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    n = len(t0)
    ev = NodeEvolverBatched(n, physics, synthetic_cie_table(), **options)
    y, h = d(y), d(h)
    scale = torch.zeros((30, n), dtype=torch.float64, device="cuda")
    counters = torch.zeros(3 * n, dtype=torch.int64, device="cuda")
    status = ev.evolve_device(y, d(node_par), d(t0), d(t1), h, scale=scale, counters=counters)
    torch.cuda.synchronize()
    return y.cpu(), h.cpu(), status.cpu(), scale.cpu(), counters.cpu().view(3, n)


@pytest.mark.parametrize("n", [1, 63, 64, 65, 200])
@pytest.mark.parametrize("kind,operators,options", [
    ("isolated", None, {}), ("isolated", 0, {}), ("isolated", 2, {"enforceNonNegativity": True}),
    ("satellite", None, {"odeToleranceRelative": 1.0e-4})])
def test_results_do_not_depend_on_the_group(torch_cuda, n, kind, operators, options):
    physics = gp.physics_params()
    make = wl.isolated_halos if kind == "isolated" else wl.satellite_halos
    b = make(n, seed=43, params=physics)
    if operators is not None:
        physics[gp.P["nodeOperators"]] = operators
    t1 = b.t_start + 0.1 * (b.t_end - b.t_start)
    t1[5::11] = b.t_start[5::11]          # intervals of zero length among them
    run = lambda i: _evolve(torch_cuda, physics, options, b.y[:, i], b.node_par[:, i], b.t_start[i], t1[i],
                            b.h_step[i])
    together = run(np.arange(n))
    order = np.random.Generator(np.random.PCG64(n)).permutation(n)
    alone = int(order[n // 2])
    for i in (order, np.array([alone]), np.concatenate([order, order])):
        for whole, part in zip(together, run(i)):
            assert torch_cuda.equal(whole[..., torch_cuda.from_numpy(i)], part)
    assert (together[2] == 0).all()


@pytest.mark.parametrize("trees,resolution", [(1, 5.0e10), (1, 2.0e9), (3, 2.0e10), (90, 2.0e10), (300, 1.0e11)])
def test_chained_operations_match_the_waves(torch_cuda, trees, resolution):
    """A single branch, where every operation is chained to the one before; a
    tree, where mergers leave the last to arrive with the successor; and more
    trees than a group has lanes."""
    torch = torch_cuda
    from galacticus_amd.evolver import NodeEvolverBatched
    physics = gp.physics_params()
    cosmo = tr.cosmology(physics)
    t0, t5 = (float(wl.scale_factor_to_cosmic_time(a)) for a in (1.0, 1.0 / 6.0))
    forest = tr.Forest.build_pch(trees, np.geomspace(2.0e11, 2.0e12, trees), t0, cosmo,
                                 tr.pch_params(resolution, t5), seed=trees)
    walk = tr.walk_params(t0, merging_multiplier=0.2)
    schedule = tr.Schedule(forest, cosmo, walk)
    print("nodes", forest.n_nodes, "operations", schedule.n_ops, flush=True)
    y0 = forest.initial_state(cosmo, walk)
    ev = NodeEvolverBatched(forest.n_nodes, physics, synthetic_cie_table())
    out = []
    for executor in ("waves", "graph", "graph"):
        y = torch.from_numpy(y0.copy()).cuda()
        scale = torch.zeros_like(y)
        status = tr.evolve_forest(ev, schedule, y, scale=scale, executor=executor)
        torch.cuda.synchronize()
        out.append((y.cpu(), scale.cpu(), status.cpu()))
    for other in out[1:]:
        assert all(torch.equal(a, b) for a, b in zip(out[0], other))


_fma = np.vectorize(lambda a, b, c: float(Fraction(a) * Fraction(b) + Fraction(c)), otypes=[float])


def _cash_karp_step(rhs, t, y, h):
    """The state after one Cash-Karp step of the derivative rhs(t, y): the tableau in doubles, and each sum with one
    rounding per term in the integrator's order."""
    k1 = rhs(t, y)
    k2 = rhs(_fma(1 / 5, h, t), _fma(h, (1 / 5) * k1, y))
    k3 = rhs(_fma(3 / 10, h, t), _fma(h, _fma(9 / 40, k2, (3 / 40) * k1), y))
    k4 = rhs(_fma(3 / 5, h, t), _fma(h, _fma(6 / 5, k3, _fma(3 / 10, k1, (-9 / 10) * k2)), y))
    k5 = rhs(t + h, _fma(h, _fma(35 / 27, k4, _fma(-70 / 27, k3, _fma(5 / 2, k2, (-11 / 54) * k1))), y))
    k6 = rhs(_fma(7 / 8, h, t),
             _fma(h, _fma(253 / 4096, k5, _fma(44275 / 110592, k4, _fma(575 / 13824, k3, _fma(
                 1631 / 55296, k1, (175 / 512) * k2)))), y))
    return _fma(h, _fma(512 / 1771, k6, _fma(125 / 594, k4, _fma(37 / 378, k1, (250 / 621) * k3))), y)


_FIXABLE = [wl.V[v] for v in ("HOT_MASS", "HOT_OUTER_RADIUS", "DISK_MASS_GAS", "DISK_MASS_STELLAR",
                              "DISK_ANGULAR_MOMENTUM", "SPHEROID_MASS_GAS", "SPHEROID_MASS_STELLAR",
                              "SPHEROID_ANGULAR_MOMENTUM")]


def _one_step_batch(kind, n):
    """Intervals from 2^-10 to 2^-4 Gyr, the long ones a large part of what changes fast, from times whose sums with
    them are exact."""
    physics = gp.physics_params()
    if kind == "box":
        physics, b = wl.closed_box()[:2]
        b = wl.NodeBatch(*(np.repeat(a[..., :1], n, axis=-1) for a in (b.y, b.node_par, b.t_start, b.t_end, b.h_step)))
    else:
        b = (wl.satellite_halos if kind == "satellite" else wl.isolated_halos)(n, seed=47, params=physics)
    if kind == "test":
        physics = gp.physics_params(physicsMode=gp.PHYSICS_TEST)
    h = np.round(np.geomspace(2.0 ** -10, 2.0 ** -4, n) * 2.0 ** 20) / 2.0 ** 20
    t0 = np.round(b.t_start * 2.0 ** 30) / 2.0 ** 30
    assert ((t0 + h) - t0 == h).all()
    return physics, b, t0, h


@pytest.mark.parametrize("kind,operators", [("isolated", k) for k in range(16)] + [("satellite", k) for k in range(16)] +
                         [("box", None), ("test", None)])
def test_four_waves_compute_the_derivative_of_one_lane(torch_cuda, kind, operators):
    """One accepted step (tolerances that accept any) against the same step put together on the host from derivatives
    that rhs_device computes, one lane to a node: equal to the last bit.  Nodes that the step leaves negative where
    the post-step fixes apply, or not finite, are left out."""
    torch = torch_cuda
    from galacticus_amd.evolver import NodeEvolverBatched
    n = 70
    physics, b, t0, h = _one_step_batch(kind, n)
    if operators is not None:
        physics[gp.P["nodeOperators"]] = operators
    d = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    par = d(b.node_par)
    single = NodeEvolverBatched(n, physics, synthetic_cie_table())

    def rhs(t, y):
        bad = ~np.isfinite(y)
        k = single.rhs_device(d(t), d(np.where(bad, 1.0, y)), par).cpu().numpy()
        lost.update(np.nonzero((bad | ~np.isfinite(k)).any(axis=0))[0].tolist())
        return np.where(np.isfinite(k), k, 0.0)

    lost = set()
    expected = _cash_karp_step(rhs, t0, b.y, h)
    keep = (expected[_FIXABLE] >= 0.0).all(axis=0)
    keep[list(lost)] = False
    y, h_step, status, _, counters = _evolve(torch, physics, {"odeToleranceAbsolute": 1.0e12,
                                                              "odeToleranceRelative": 1.0e12},
                                             b.y, b.node_par, t0, t0 + h, np.full(n, -1.0))
    changed = (expected != b.y)[:, keep].any(axis=1).sum()
    print(kind, operators, "nodes compared", int(keep.sum()), "variables that change", int(changed), flush=True)
    assert keep.sum() >= n // 2
    assert (status == 0).all() and (counters.numpy()[:, keep] == np.array([[1], [1], [6]])).all()
    assert np.array_equal(y.numpy()[:, keep], expected[:, keep])


def test_autotune_takes_no_memory_and_runs_nothing(torch_cuda):
    """With one launch shape there is nothing to time: a leading dimension whose copies no device holds is accepted,
    and the arrays stay as they are.  What cannot be evolved is refused."""
    import ctypes
    torch = torch_cuda
    from galacticus_amd import _lib
    from galacticus_amd.evolver import NodeEvolverBatched
    b = wl.isolated_halos(64, seed=1)
    ev = NodeEvolverBatched(64, gp.physics_params(), synthetic_cie_table())
    arrays = [torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in (b.y, b.node_par, b.t_start, b.t_end, b.h_step)]
    before = [a.clone() for a in arrays]
    blocks = ctypes.c_int(), ctypes.c_int()
    pointers = [ctypes.c_void_p(a.data_ptr()) for a in arrays]
    call = lambda n, ld, p: ev.L.gal_ode_batch_autotune(ev.handle, n, ld, *p, None, None, None,
                                                        ctypes.byref(blocks[0]), ctypes.byref(blocks[1]))
    ev.set_launch(64, 4, 1)
    assert call(64, 2 ** 31 - 1, pointers) == _lib.GAL_OK
    torch.cuda.synchronize()
    assert (blocks[0].value, blocks[1].value) == (64, 1) and ev.launch() == (64, 1, 2)
    assert all(torch.equal(a, o) for a, o in zip(arrays, before))
    for n, ld, p in ((0, 64, pointers), (65, 65, pointers), (64, 63, pointers), (64, 64, [None] + pointers[1:])):
        assert call(n, ld, p) == -1        # GAL_E_INVALID
