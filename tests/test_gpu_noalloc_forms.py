"""sph_step_noalloc in the form it takes beyond the split form's size, at rows
wider than a wave's copy, and with rows and neighbour lists longer than their
fixed room, where it has no other copy of them: each call equals the first step
of a handle bit for bit, with the scratch full of another call's data."""
import ctypes as C

import numpy as np
import pytest

from test_zz_no_alloc import Hip

pytestmark = pytest.mark.gpu


def scene(name, E):
    rng = np.random.default_rng(len(name))

    def cloud(n, lo, hi):
        return rng.uniform(lo, hi, (n, 3)).astype(np.float32)

    def lattice(side, ratio):
        g = np.stack(np.meshgrid(*[np.arange(side)] * 3, indexing="ij"), -1).reshape(-1, 3) * 0.01 + 0.02
        return E.make_params(kernel_radius=ratio * 0.005, particle_radius=0.005), g.astype(np.float32)

    if name == "most split tiles":
        return E.make_params(), cloud(40960, 0.05, 0.5)
    if name == "one tile more":
        return E.make_params(), cloud(40961, 0.05, 0.5)
    if name == "most particles":
        return E.make_params(), cloud(65536, 0.05, 0.55)
    # Rows of up to 64 candidates and of more, lists of more than 64 and 128.
    if name == "long rows":
        return E.make_params(pressure_stiffness=1e-3, box_max=(0.3,) * 3), cloud(9000, 0.05, 0.22)
    if name == "long lists":
        return E.make_params(pressure_stiffness=1e-4, box_max=(0.2,) * 3), cloud(6000, 0.06, 0.14)
    if name == "long rows, many tiles":
        return E.make_params(pressure_stiffness=1e-4, box_max=(0.4,) * 3), cloud(60000, 0.05, 0.3)
    return {"support of 6.2 radii": lambda: lattice(20, 6.2), "support of 6.3 radii": lambda: lattice(20, 6.3),
            "support of 12 radii": lambda: lattice(30, 12.0)}[name]()


@pytest.mark.parametrize("name", ["most split tiles", "one tile more", "most particles", "long rows", "long lists",
                                  "long rows, many tiles", "support of 6.2 radii", "support of 6.3 radii",
                                  "support of 12 radii"])
def test_noalloc_step_equals_the_handles(name):
    from simplefluid_amd import engine as E
    L = E.load_library()
    hip = Hip(L)
    p, x = scene(name, E)
    v = np.random.default_rng(1).normal(0.0, 0.2, x.shape).astype(np.float32)
    dev = [hip.upload(a) for a in (x, v, np.full_like(x, np.nan), np.full_like(v, np.nan))]
    # Another scene's call first: what it leaves in the scratch is not this one's.
    q, y = scene("most particles" if len(x) < 65536 else "long lists", E)
    other = hip.upload(y)
    out = hip.alloc(2 * y.nbytes)
    rc = L.sph_step_noalloc(C.byref(q), other, None, out, C.c_void_p(out.value + y.nbytes), len(y), None)
    assert rc == E.SPH_OK
    rc = L.sph_step_noalloc(C.byref(p), dev[0], dev[1], dev[2], dev[3], len(x), None)
    assert rc == E.SPH_OK, L.sph_last_error(None)
    hip.ok(L.hipDeviceSynchronize(), "hipDeviceSynchronize")
    e = E.Engine(p)
    e.set_particles(x, v)
    e.make_ready()
    e.advance_steps(1)
    off, _ = e.debug_neighbors()
    longest = np.diff(off.astype(np.int64)).max()
    xg, vg = e.get_particles(), e.get_velocity()
    e.close()
    xa, va = hip.download(dev[2], x.shape), hip.download(dev[3], v.shape)
    for ptr in dev + [other, out]:
        hip.ok(L.hipFree(ptr), "hipFree")
    if name.startswith("long"):
        # A list holds 128 neighbours beside the particle itself.
        assert longest > (129 if "lists" in name else 65), f"{longest} neighbours: the scene tests nothing"
    assert np.array_equal(xa, xg) and np.array_equal(va, vg)
