"""The scenes of crowded particles that the small handles' form is compared on
elsewhere: "dense" has rows of more than 64 candidates and lists of more than
one round, "denser" lists longer than their 128 places, which then run the
other forms' walks.  All forms agree bit for bit, forwards and backwards."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name,n,stiffness,box,lo,hi,seed,more_than",
                         [("dense", 9000, 1e-3, 0.3, 0.05, 0.22, 2, 65), ("denser", 6000, 1e-4, 0.2, 0.06, 0.14, 3, 129)])
def test_crowded_scenes_overflow_what_they_say(name, n, stiffness, box, lo, hi, seed, more_than):
    from simplefluid_amd import engine as E
    x = np.random.default_rng(seed).uniform(lo, hi, (n, 3)).astype(np.float32)
    g = np.random.default_rng(1).normal(0.0, 1.0, x.shape).astype(np.float32)
    got = []
    for form in (None, dict(), dict(force_staged=1, density_staged=1)):
        e = E.Engine(E.make_params(pressure_stiffness=stiffness, box_max=(box,) * 3))
        e.set_particles(x)
        e.make_ready()
        if form is not None:
            e.set_tuning(**form)
        assert e.get_tuning()["split"] == (form is None)
        e.advance_steps(1)
        off, _ = e.debug_neighbors()
        longest = int(np.diff(off.astype(np.int64)).max())
        # The particle itself is counted and has no place in its list.
        assert longest > more_than, f"{name}: {longest} neighbours at most, the scene tests nothing"
        e.rollout_forward(2, 1)
        got.append((e.get_particles(), e.get_velocity()) + tuple(e.rollout_backward(g)))
        e.close()
    for other in got[1:]:
        for a, b in zip(got[0], other):
            assert np.array_equal(a, b), name
