"""Supports of many particle radii: the forms an untuned handle picks for them
against the ones sph_set_tuning asks for, bit for bit, forwards and backwards,
and one step against the CPU oracle (cells, order and neighbours exactly,
density to the 2e-6 that its sums of some thousand terms in another precision
keep elsewhere)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ratio,side,scenes", [(6.2, 12, 1), (6.3, 12, 1), (8.0, 9, 3), (12.0, 13, 1), (7.0, 52, 1)])
def test_wide_rows_agree_in_every_form(ratio, side, scenes):
    from simplefluid_amd import engine as E
    r = 0.005
    rng = np.random.default_rng(side)
    g = np.stack(np.meshgrid(*[np.arange(side)] * 3, indexing="ij"), -1).reshape(-1, 3) * (2.0 * r) + 2.0 * r
    x = np.concatenate([g + rng.uniform(-0.2 * r, 0.2 * r, g.shape) for _ in range(scenes)]).astype(np.float32)
    v = rng.normal(0.0, 0.2, x.shape).astype(np.float32)
    seed = rng.normal(0.0, 1e-4, x.shape).astype(np.float32)
    p = E.make_params(kernel_radius=ratio * r, particle_radius=r, pressure_stiffness=5.0)
    got = []
    for form in (None, dict(), dict(force_staged=1, density_staged=1, density_block=64, force_block=128)):
        e = E.BatchEngine([p] * scenes, [len(g)] * scenes)
        e.set_particles(x, v)
        e.make_ready()
        if form is not None:
            e.set_tuning(**form)
        else:
            t = e.get_tuning()
            assert t["split"] == (ratio < 6.25) and not t["force_staged"] and not t["density_staged"]
        e.rollout_forward(4, 2)
        got.append((e.get_particles(), e.get_velocity()) + tuple(e.rollout_backward(seed)))
        e.synchronize()
        e.close()
    assert all(np.isfinite(a).all() for a in got[0])
    for other in got[1:]:
        for a, b in zip(got[0], other):
            assert np.array_equal(a, b)


@pytest.mark.parametrize("ratio", [8.0, 12.0])
def test_wide_rows_step_agrees_with_the_oracle(ratio):
    import oracle
    from simplefluid_amd import engine as E
    r = 0.005
    rng = np.random.default_rng(2)
    g = np.stack(np.meshgrid(*[np.arange(14)] * 3, indexing="ij"), -1).reshape(-1, 3) * (2.0 * r) + 2.0 * r
    x = (g + rng.uniform(-0.2 * r, 0.2 * r, g.shape)).astype(np.float32)
    p = E.make_params(kernel_radius=ratio * r, particle_radius=r, pressure_stiffness=5.0)
    e = E.Engine(p)
    e.set_particles(x)
    e.make_ready()
    e.debug_keep_acc(True)
    e.advance_steps(1)
    d = e.debug_step_outputs(acc=True)
    off, lst = e.debug_neighbors()
    o = oracle.Oracle(oracle.from_params(p, e.debug_constants()["xsub"]), threads=4)
    o.record_neighbors(True)
    o.set_state(x.astype(np.float64))
    o.step()
    q = o.step_debug()
    ooff, olst = o.neighbors()
    assert np.array_equal(d["key"], q["key"]) and np.array_equal(d["perm"], q["perm"])
    assert np.array_equal(off, ooff) and np.array_equal(lst, olst)
    assert (np.abs(d["rho"] - q["rho"]) / q["rho"]).max() <= 2e-6
    e.close()
