"""The forms of density and force that a handle no one has tuned takes by its
size, against the ones sph_set_tuning asks for, bit for bit, one particle to
each side of the line."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [(1 << 17) - 1, 1 << 17])
def test_untuned_forms_equal_the_asked_for_ones(n):
    from simplefluid_amd import engine as E
    rng = np.random.default_rng(n)
    x = rng.uniform(0.01, 0.6, (n, 3)).astype(np.float32)
    v = rng.normal(0.0, 0.3, x.shape).astype(np.float32)
    g = rng.normal(0.0, 1.0, x.shape).astype(np.float32)
    got = []
    for form in (None, dict(), dict(force_staged=1, density_staged=1)):
        e = E.Engine(E.make_params())
        e.set_particles(x, v)
        e.make_ready()
        if form is not None:
            e.set_tuning(**form)
        e.advance_steps(2)
        rho = e.get_density()
        e.rollout_forward(2, 2)
        got.append((rho, e.get_particles(), e.get_velocity()) + tuple(e.rollout_backward(g)))
        e.synchronize()
        e.close()
    for other in got[1:]:
        for a, b in zip(got[0], other):
            assert np.array_equal(a, b)
