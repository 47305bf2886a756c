"""The small-handle form of the reverse pass against the forms sph_set_tuning
asks for, bit for bit, where it can go wrong: tiles of one particle and one
over, rows of more candidates than one and two mask words hold, lists of more
than one round and longer than they may be, ragged scenes of a batch (tiles of
64 against sums over 256), and segments of one step and of several.  (The
other forms are checked against central differences and the CPU oracle
elsewhere.)"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

FORMS = (dict(), dict(force_staged=1, density_staged=1))


def cloud(seed, n, lo, hi):
    return np.random.default_rng(seed).uniform(lo, hi, (n, 3)).astype(np.float32)


def scenes(E):
    out = {f"n{n}": ([E.make_params()], [cloud(n, n, 0.2, 0.25)]) for n in (1, 65, 257)}
    out["dense"] = ([E.make_params(pressure_stiffness=1e-3, box_max=(0.3, 0.3, 0.3))], [cloud(2, 9000, 0.05, 0.22)])
    out["denser"] = ([E.make_params(pressure_stiffness=1e-4, box_max=(0.2, 0.2, 0.2))], [cloud(3, 6000, 0.06, 0.14)])
    out["walls"] = ([E.make_params(box_max=(0.2, 0.2, 0.2))], [cloud(4, 5000, 0.005, 0.195)])
    out["attractive"] = ([E.make_params(use_attractive_pressure=1)], [cloud(5, 5000, 0.2, 0.5)])
    ns = (1, 0, 64, 300, 2000, 513)
    out["batch"] = ([E.make_params(pressure_stiffness=20.0 + 10 * i) for i in range(len(ns))],
                    [cloud(7 + i, n, 0.1, 0.3) for i, n in enumerate(ns)])
    return out


@pytest.mark.parametrize("name", ["n1", "n65", "n257", "dense", "denser", "walls", "attractive", "batch"])
@pytest.mark.parametrize("every", [1, 3])
def test_small_handles_reverse_pass_equals_the_others(name, every):
    from simplefluid_amd import engine as E
    params, pos = scenes(E)[name]
    x = np.concatenate(pos)
    rng = np.random.default_rng(1)
    v = rng.normal(0.0, 0.3, x.shape).astype(np.float32)
    g = rng.normal(0.0, 1.0, x.shape).astype(np.float32)
    got = []
    for form in (None,) + FORMS:
        e = E.Engine(params[0]) if len(params) == 1 else E.BatchEngine(params, [len(p) for p in pos])
        e.set_particles(x, v)
        e.make_ready()
        if form is not None:
            e.set_tuning(**form)
        e.rollout_forward(4, every)
        first = e.rollout_backward(g)
        again = e.rollout_backward(g)  # every segment recomputed
        for a, b in zip(first, again):
            assert np.array_equal(a, b), name
        got.append(first)
        e.synchronize()
        e.close()
    assert all(np.isfinite(a).all() for a in got[0]), name
    for other in got[1:]:
        for a, b in zip(got[0], other):
            assert np.array_equal(a, b), (name, np.abs(a - b).max())
