"""Downloads at the sizes where their path changes: one word, words past the
last 16 bytes, the last size that goes in one piece and the first that goes
in several, and many pieces with a ragged last one.  What was uploaded comes
back bit for bit, also while another handle's download runs on another
thread."""
import ctypes
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

READ = 3400  # particles whose order one block restores
SMALL = (1 << 19) // 3  # particles whose 3n words are the most one piece takes


def upload(n, seed):
    from simplefluid_amd import engine as E
    rng = np.random.default_rng(seed)
    x = rng.uniform(0.1, 0.9, (n, 3)).astype(np.float32)
    v = rng.normal(0.0, 1.0, (n, 3)).astype(np.float32)
    e = E.Engine(E.make_params())
    e.set_particles(x, v)
    e.make_ready()
    return e, x, v


@pytest.mark.parametrize("n", [1, 2, 3, 85, READ, READ + 1, SMALL, SMALL + 1, 700_001, 3_000_000])
def test_downloads_return_what_was_uploaded(n):
    e, x, v = upload(n, n)
    for _ in range(2):
        assert np.array_equal(e.get_particles(), x)
        assert np.array_equal(e.get_velocity(), v)
    e.close()


def test_downloads_on_two_threads():
    held = [upload(400_000 + 7 * i, i) for i in range(2)]
    bad = []

    def read(e, x, v):
        for _ in range(5):
            if not (np.array_equal(e.get_particles(), x) and np.array_equal(e.get_velocity(), v)):
                bad.append(len(x))

    threads = [threading.Thread(target=read, args=h) for h in held]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad
    for e, _, _ in held:
        e.close()


@pytest.mark.parametrize("n", [READ, READ + 1, 300_000])
def test_nothing_is_handed_over_where_the_error_flag_is_raised(n):
    """1,200 particles in one cell, more than the cell-count sort ranks: the
    read reports it and leaves the caller's array alone, on each path."""
    from simplefluid_amd import engine as E
    e, x, _ = upload(n, n)
    x[:1200] = np.nan
    e.set_particles(x)
    e.make_ready()
    e.advance_steps(1)
    out = np.full((n, 3), 7.0, np.float32)
    rc = e._L.sph_get_particles(e._h, out.ctypes.data_as(ctypes.c_void_p))
    assert rc == E.SPH_E_DEVICE and (out == 7.0).all()
    e.close()
