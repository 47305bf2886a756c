"""Autotuned shapes are shared by a process's handles of one size bucket; how
a handle sorts is its own, whichever handle was tuned first."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,first", [(50000, "radix"), (50000, "cell"), (100000, "cell"), (100000, "radix")])
def test_autotune_leaves_the_sort_mode(n, first):
    from simplefluid_amd import engine as E
    modes = [E.SORT_RADIX, E.SORT_CELL_COUNT]
    x = np.random.default_rng(n).uniform(0.02, 0.6, (n, 3)).astype(np.float32)
    got = []
    for mode in modes if first == "radix" else modes[::-1]:
        e = E.Engine(E.make_params())
        e.set_particles(x)
        e.make_ready()
        e.set_sort_mode(mode)
        e.autotune()
        assert e.get_sort_mode() == mode
        e.advance_steps(2)
        got.append((e.get_particles(), e.get_velocity()))
        e.close()
    for a, b in zip(*got):
        assert np.array_equal(a, b)
