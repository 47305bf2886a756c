"""The small-handle form of the density and force passes against the forms
sph_set_tuning asks for, bit for bit, where it can go wrong: tiles of one
particle and one over, rows of more candidates than one and two mask words
hold, rows wider than their copy, lists longer than they may be, scenes of a
batch that share a tile's width, and a CFL step.  (The other forms are checked
against the CPU oracle elsewhere.)"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

FORMS = (dict(), dict(force_staged=1, density_staged=1, density_block=64, force_block=128))


def cloud(seed, n, lo, hi):
    return np.random.default_rng(seed).uniform(lo, hi, (n, 3)).astype(np.float32)


def scenes(E):
    box = dict(gravity=(0.0, -9.81, 0.0))
    out = {}
    for n in (1, 63, 64, 65, 129):
        out[f"n{n}"] = ([E.make_params(**box)], [cloud(n, n, 0.2, 0.25)], 0)
    # Rows of up to two mask words, and of more; lists past 64 neighbours.
    out["dense"] = ([E.make_params(pressure_stiffness=1e-3, box_max=(0.3, 0.3, 0.3))], [cloud(2, 9000, 0.05, 0.22)], 0)
    out["denser"] = ([E.make_params(pressure_stiffness=1e-4, box_max=(0.2, 0.2, 0.2))], [cloud(3, 6000, 0.06, 0.14)], 0)
    # Wide x cells and rows, short columns: waves that span columns and planes.
    out["wide"] = ([E.make_params(box_max=(0.14, 0.5, 0.5))], [cloud(4, 15000, 0.005, 0.13)], 1)
    out["sparse"] = ([E.make_params()], [cloud(5, 3000, 0.01, 0.99)], 0)
    # As many tiles as the form takes.
    out["most"] = ([E.make_params()], [cloud(6, 40960, 0.05, 0.5)], 0)
    # A batch of ragged scenes, an empty one among them.
    ns = (1, 0, 64, 333, 2000, 65)
    out["batch"] = ([E.make_params(pressure_stiffness=20.0 + 10 * i) for i in range(len(ns))],
                    [cloud(7 + i, n, 0.1, 0.3) for i, n in enumerate(ns)], 0)
    out["cfl"] = ([E.make_params(cfl_number=0.3)], [cloud(20, 5000, 0.2, 0.45)], 0)
    out["attractive"] = ([E.make_params(use_attractive_pressure=1)], [cloud(21, 5000, 0.2, 0.5)], 2)
    return out


@pytest.mark.parametrize("name", ["n1", "n63", "n64", "n65", "n129", "dense", "denser", "wide", "sparse", "most",
                                  "batch", "cfl", "attractive"])
def test_small_handles_form_equals_the_others(name):
    from simplefluid_amd import engine as E
    params, pos, xsub = scenes(E)[name]
    x = np.concatenate(pos)
    v = np.random.default_rng(1).normal(0.0, 0.3, x.shape).astype(np.float32)
    got = []
    for form in (None,) + FORMS:
        e = E.Engine(params[0]) if len(params) == 1 else E.BatchEngine(params, [len(p) for p in pos])
        e.set_cell_subdivision(xsub)
        e.set_particles(x, v)
        e.make_ready()
        if form is not None:
            e.set_tuning(**form)
        e.debug_keep_acc(True)
        e.advance_steps(2)
        d = e.debug_step_outputs(acc=True)
        off, lst = e.debug_neighbors()
        got.append((d["rho"], d["acc"], off, lst, e.get_particles(), e.get_velocity()))
        e.synchronize()
        e.close()
    if name in ("dense", "denser"):
        assert np.diff(got[0][2].astype(np.int64)).max() > 65, "every list fits: the scene tests nothing"
    for other in got[1:]:
        for a, b in zip(got[0], other):
            assert np.array_equal(a, b), name


@pytest.mark.parametrize("name", ["n1", "dense", "denser"])
def test_spare_buffers_give_way(name):
    """The neighbour lists and second mask words are left out where a memory
    cap has no room for them, and given back to an allocation that needs the
    room; the steps stay the same bit for bit either way, in every form."""
    from simplefluid_amd import engine as E
    params, pos, xsub = scenes(E)[name]
    x = pos[0]

    def run(limit, form, rollout):
        e = E.Engine(params[0])
        e.set_device_memory_limit(limit)
        e.set_cell_subdivision(xsub)
        e.set_particles(x)
        e.make_ready()
        if form is not None:
            e.set_tuning(**form)
        e.advance_steps(2)
        used = e.device_memory_used()
        if rollout:
            e.rollout_forward(2)
        e.advance_steps(2)
        out = (e.get_particles(), e.get_velocity(), used, e.device_memory_used())
        e.close()
        return out

    spares = len(x) * (9 * 4 + 128 * 2 + 4)
    for form in (None,) + FORMS:
        full = run(0, form, False)
        bare = run(full[2] - spares, form, False)
        assert bare[2] == full[2] - spares
        taped = run(0, form, True)
        tight = run(taped[3] - 4, form, True)
        assert tight[3] == taped[3] - spares
        for a, b in ((full, bare), (taped, tight)):
            assert np.array_equal(a[0], b[0]) and np.array_equal(a[1], b[1]), (name, form)
