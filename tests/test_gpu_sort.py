"""The cell-count sort at its edges, against numpy's stable sort of the same
keys: tiles fuller than the LDS list, cells whose chain of runs is longer than
the sort follows, all tile sizes, partial last tiles, and grids of more
tiles than a block sums itself.  Permutation, sorted keys and cell table are
whole numbers and compared exactly."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def scenes():
    rng = np.random.default_rng(9)

    def params(E, box, h=0.02):
        # A step too short to move anything: the order changes, the cells don't.
        return E.make_params(kernel_radius=h, particle_radius=h / 4, box_max=box, dt=1e-12, gravity=(0, 0, 0))

    out = {}
    # 12,000 particles in 64 cells (one tile, more members than the LDS list).
    out["one_tile"] = lambda E: (params(E, (0.08, 0.08, 0.08)), rng.uniform(0.006, 0.074, (12000, 3)), 1)
    # 700 particles of one cell, every other particle of the upload: as many
    # links of one particle each.
    def pile(E):
        a = rng.uniform(0.2, 0.8, (1400, 3))
        a[::2] = np.array([0.503, 0.503, 0.503]) + rng.uniform(0.0, 0.002, (700, 3))
        return params(E, (1.0, 1.0, 1.0)), a, 4
    out["long_chain"] = pile
    # The same with a full tile around it.
    def pile_in_full_tile(E):
        a = rng.uniform(0.006, 0.074, (9000, 3))
        a[::15] = np.array([0.05, 0.05, 0.05]) + rng.uniform(0.0, 0.002, (600, 3))
        return params(E, (0.08, 0.08, 0.08)), a, 1
    out["long_chain_full_tile"] = pile_in_full_tile
    # One cell in all; a few particles; one more than a wave's run of links.
    out["one_cell"] = lambda E: (params(E, (0.0199, 0.0199, 0.0199)), rng.uniform(0.005, 0.0149, (79, 3)), 1)
    # 1,025 cells: a last tile of one cell.
    out["last_tile_of_one"] = lambda E: (params(E, (0.999 * 41 * 0.02, 0.999 * 5 * 0.02, 0.999 * 5 * 0.02)),
                                         rng.uniform(0.0, 1.0, (3000, 3)) * (0.8, 0.09, 0.09) + 0.005, 1)
    # Between 2^19 and 2^20 cells (tiles of 512) ...
    out["middle"] = lambda E: (params(E, (1.4, 1.1, 1.3)), rng.uniform(0.1, 1.0, (20000, 3)), 4)
    # ... more than 2^20 (tiles of 1024, four cells per thread) ...
    out["narrow"] = lambda E: (params(E, (2.0, 1.1, 1.3)), rng.uniform(0.1, 1.0, (20000, 3)), 4)
    # ... and more than 6144 tiles (their sums are scanned by their own kernel).
    out["scanned_tiles"] = lambda E: (params(E, (3.0, 3.0, 3.0)), rng.uniform(0.01, 2.99, (30000, 3)), 4)
    return out


@pytest.mark.parametrize("name", list(scenes()))
def test_cell_sort_is_stable_and_its_table_exact(name):
    from simplefluid_amd import engine as E
    p, pos, xsub = scenes()[name](E)
    pos = np.ascontiguousarray(pos, np.float32)
    e = E.Engine(p)
    e.set_cell_subdivision(xsub)
    e.set_particles(pos)
    e.make_ready()
    # The upload's order, then twice the order the step before left.
    for _ in range(3):
        e.advance_steps(1)
        d = e.debug_step_outputs()
        order = np.argsort(d["key"], kind="stable")
        assert np.array_equal(d["perm"], order), name
        assert np.array_equal(d["sorted_key"], d["key"][order])
        start, end = e.debug_cells()
        cells = start.size
        count = np.bincount(d["key"], minlength=cells)
        first = np.cumsum(count) - count
        full = count > 0
        assert np.array_equal(end > 0, full)
        assert np.array_equal(start[full], first[full]) and np.array_equal(end[full], (first + count)[full])
    e.synchronize()
    e.close()
